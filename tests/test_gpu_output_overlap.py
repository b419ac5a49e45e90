"""GPU: outputs that share memory with an input.  Every entry reads all inputs before it writes any output, whichever
rows the output is written to and however the sum is cut."""
import numpy as np
import pytest

import stkfmm_amd as S
from oracle import oracle as O
from tests.gpu_util import FP64_TOL, MIXED_TOL, host, say, to_dev, zeros

pytestmark = pytest.mark.gpu

UK = S.UKER.STOKES_VEL  # three values in, three out


def check(got, ref, prec, same=None):
    l2, mx = O.max_error(got, ref)
    tol = MIXED_TOL if prec else FP64_TOL
    assert l2 < tol and mx < tol, (l2, mx)
    if same is not None:  # the same pair sums as with an output of its own
        l2, mx = O.max_error(got, same)
        assert l2 < FP64_TOL and mx < FP64_TOL, (l2, mx)


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("tune", [None, dict(max_src_per_item=4096), dict(max_src_per_item=4096, broadcast=1),
                                  dict(max_src_per_item=128)], ids=["untuned", "lds", "scalar", "split"])
@pytest.mark.parametrize("n", [1000, 6000])  # (6,000: several source chunks)
@pytest.mark.parametrize("how", ["slice", "range"])
def test_one_group_into_rows_of_its_field(how, n, tune, prec):
    """The last n rows of a field, updated in place through a permutation: as arrays of their own (slice), and as a
    range of the whole arrays (range)."""
    say(f"overlap one group {how} n={n} prec={prec} tune={tune}")
    rng = np.random.default_rng(n)
    m = n + 5000
    x, f = rng.random((m, 3)), rng.normal(size=(m, 3))
    ref = f.copy()
    ref[5000:] += O.direct(int(UK), x[5000:], f[5000:], x[5000:])
    d_x, d_f = to_dev(x), to_dev(f)
    own = d_f.clone()
    if how == "slice":
        perm = to_dev(np.arange(5000, m, dtype=np.int32))
        plan = S.Plan(UK, prec, n, n, [0], [n], None, [0, 1], [0], [n], tune)
        args = d_x[5000:], d_f[5000:], d_x[5000:]
    else:
        perm = to_dev(np.arange(m, dtype=np.int32))
        plan = S.Plan(UK, prec, m, m, [5000], [m], None, [0, 1], [5000], [m], tune)
        args = d_x, d_f, d_x
    plan.execute(*args, own, perm=perm)
    plan.execute(*args, d_f, perm=perm)
    check(host(d_f), ref, prec, host(own))


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("bc", [0, 1], ids=["lds", "scalar"])
@pytest.mark.parametrize("per", [60, 300])  # items a tile: one, several
@pytest.mark.parametrize("permuted", [False, True])
def test_groups_in_place(permuted, per, bc, prec):
    """Many groups, each summed over another group's points: in place, and through a permutation that sends the
    results to rows behind the ones that are read first."""
    say(f"overlap groups permuted={permuted} per={per} bc={bc} prec={prec}")
    rng = np.random.default_rng(per)
    g = 300
    n = g * per
    x, f = rng.random((n, 3)), rng.normal(size=(n, 3))
    tb = np.arange(g) * per
    sb = tb[(np.arange(g) * 7 + 150) % g]
    u = np.concatenate([O.direct(int(UK), x[s:s + per], f[s:s + per], x[t:t + per]) for t, s in zip(tb, sb)])
    perm = rng.permutation(n).astype(np.int32) if permuted else np.arange(n, dtype=np.int32)
    ref = f.copy()
    ref[perm] += u
    d_x, d_f, d_perm = to_dev(x), to_dev(f), to_dev(perm) if permuted else None
    own = d_f.clone()
    plan = S.Plan(UK, prec, n, n, tb, tb + per, None, np.arange(g + 1), sb, sb + per,
                  dict(max_src_per_item=128, broadcast=bc))
    plan.execute(d_x, d_f, d_x, own, perm=d_perm)
    plan.execute(d_x, d_f, d_x, d_f, perm=d_perm)
    check(host(d_f), ref, prec, host(own))


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
def test_columns_of_one_tensor(prec):
    """Coordinates, values and results interleaved in one tensor."""
    say(f"overlap columns prec={prec}")
    n = 900
    rng = np.random.default_rng(n)
    t = rng.random((n, 9))
    ref = t.copy()
    ref[:, 6:] += O.direct(int(UK), t[:, :3], t[:, 3:6], t[:, :3])
    for groups in (1, 30):
        d = to_dev(t)
        tb = np.arange(groups) * (n // groups)
        plan = S.Plan(UK, prec, n, n, tb, tb + n // groups, None, np.arange(groups + 1), [0] * groups, [n] * groups)
        plan.execute(d[:, :3], d[:, 3:6], d[:, :3], d[:, 6:])
        check(host(d), ref, prec)


@pytest.mark.parametrize("no_alloc", [False, True])
@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("ns,nt", [(6000, 6000), (50, 600_000)])
def test_device_entry_over_its_sources(ns, nt, prec, no_alloc):
    """Source charges that are the first doubles of the output; the second size's outputs exceed the partial-sum
    array of the device entry."""
    say(f"overlap device ns={ns} nt={nt} prec={prec} no_alloc={no_alloc}")
    rng = np.random.default_rng(ns)
    src, trg, first = rng.random((ns, 3)), rng.random((nt, 3)), rng.normal(size=(nt, 4))
    ref = first + O.direct(int(S.UKER.LAPLACE_PGRAD), src, first.reshape(-1)[:ns].reshape(ns, 1).copy(), trg)
    out = to_dev(first)
    val = out.view(-1)[:ns].view(ns, 1)
    S.p2p_device(S.KERNEL.LapPGrad, S.PPKERNEL.SLS2T, to_dev(src), val, to_dev(trg), out, precision=S.PREC(prec),
                 no_alloc=no_alloc)
    check(host(out), ref, prec)


@pytest.mark.parametrize("kernel", [S.KERNEL.Stokes, S.KERNEL.RPY])
@pytest.mark.parametrize("ns,nt", [(300, 400), (5000, 5000)])
def test_wall_over_its_sources(kernel, ns, nt):
    """Wall images whose source values are the first doubles of the output."""
    say(f"overlap wall kernel={int(kernel)} ns={ns} nt={nt}")
    ks, kt = (3, 3) if kernel == S.KERNEL.Stokes else (4, 6)
    rng = np.random.default_rng(ns + ks)
    x, t, first = rng.random((ns, 3)), rng.random((nt, 3)), rng.normal(size=(nt, kt))
    x[:, 2] *= 0.5
    t[:, 2] *= 0.5
    if kernel == S.KERNEL.RPY:
        first.reshape(-1)[:ks * ns].reshape(ns, ks)[:, 3] = rng.uniform(1e-3, 5e-3, ns)
    val = first.reshape(-1)[:ks * ns].reshape(ns, ks).copy()
    u = O.wall(int(kernel), x, val, t)
    _, cond = O.max_error(O.wall(int(kernel), x[::-1], val[::-1], t), u)  # the images' own conditioning
    out, own = to_dev(first), zeros(nt, kt)
    S.wall_device(kernel, to_dev(x), out.view(-1)[:ks * ns].view(ns, ks), to_dev(t), out)
    S.wall_device(kernel, to_dev(x), to_dev(val), to_dev(t), own)
    bound = max(4 * cond, FP64_TOL)
    l2, mx = O.max_error(host(own), u)
    assert l2 < bound and mx < bound, (l2, mx, cond)
    l2, mx = O.max_error(host(out), first + host(own))
    assert l2 < FP64_TOL and mx < FP64_TOL, (l2, mx)
