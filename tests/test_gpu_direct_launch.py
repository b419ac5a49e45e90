"""GPU: direct sums in one launch (p2p_direct.hpp) against the item-kernel plan of the same group and the
oracle, at the edges of tiles, units, chunks and lane splits."""
import numpy as np
import pytest

import stkfmm_amd as S
from oracle import oracle as O
from tests.conftest import source_values
from tests.gpu_util import FP64_TOL, host, say, to_dev, zeros

pytestmark = pytest.mark.gpu

# one target, one source; a tile and a wave more or less; tails of each lane split; few targets against many
# sources (chunks) and the reverse; more units than one round of workgroups
SIZES = [(1, 1), (1, 300), (63, 65), (64, 64), (65, 129), (513, 17), (1000, 1000), (4100, 130), (30000, 3),
         (70, 9001), (2500, 12345)]


NO_DL = (S.KERNEL.LapQPGradGrad, S.KERNEL.Stokes, S.KERNEL.RPY, S.KERNEL.StokesRegVel, S.KERNEL.StokesRegVelOmega)


def layout(x, soa):
    """A device tensor over x with rows and columns in either order."""
    return to_dev(np.ascontiguousarray(x.T)).T if soa else to_dev(x)


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("uk", list(S.UKER))
def test_one_launch_matches_items_and_oracle(uk, prec):
    ks, kt = S.uker_dims(uk)
    for n, (ns, nt) in enumerate(SIZES):
        say(f"direct uk={uk.name} prec={prec} ns={ns} nt={nt}")
        rng = np.random.default_rng(100 + n)
        pad = 7 if n % 2 else 0  # the group is a part of the arrays
        src = rng.random((ns + 2 * pad, 3))
        trg = rng.random((nt + 2 * pad, 3))
        k = min(nt, ns, 5)
        trg[pad:pad + k] = src[pad:pad + k]  # coincident pairs
        val = source_values(int(uk), ns + 2 * pad, rng)
        perm = rng.permutation(nt + 2 * pad).astype(np.int32)
        soa = n % 3 == 0
        d_src, d_val, d_trg, d_perm = layout(src, soa), layout(val, soa), layout(trg, not soa), to_dev(perm)
        got = []
        for tune in (None, dict(max_src_per_item=512)):
            plan = S.Plan(uk, prec, ns + 2 * pad, nt + 2 * pad, [pad], [pad + nt], None, [0, 1], [pad], [pad + ns], tune)
            out = zeros(nt + 2 * pad, kt)
            v1, v2 = (d_val[:, :4], d_val[:, 4:]) if uk == S.UKER.STOKES_PVEL_FUSED else (d_val, None)
            for _ in range(2):  # adds
                plan.execute(d_src, v1, d_trg, out, src_value2=v2, perm=d_perm)
            got.append(host(out)[perm] / 2)
        # the same pairs (in mixed mode with the same FP32 sums) in another FP64 order
        l2, mx = O.max_error(got[0][pad:pad + nt], got[1][pad:pad + nt])
        assert l2 < FP64_TOL and mx < FP64_TOL, (ns, nt, l2, mx)
        assert not got[0][:pad].any() and not got[0][pad + nt:].any()
        if prec == 0:
            ref = O.direct(int(uk), src[pad:pad + ns], val[pad:pad + ns], trg[pad:pad + nt])
            l2, mx = O.max_error(got[0][pad:pad + nt], ref)
            assert l2 < FP64_TOL and mx < FP64_TOL, (ns, nt, l2, mx)


@pytest.mark.parametrize("kernel,p2p", [(k, p) for k in S.KERNEL for p in S.PPKERNEL
                                        if not (p == S.PPKERNEL.DLS2T and k in NO_DL)])
def test_direct_entry_matches_items_mixed(kernel, p2p):
    """The direct-sum entry (one target per lane below 32,768 targets) in mixed mode."""
    uk = S.get_uker(kernel, p2p)
    ks, kt = S.uker_dims(uk)
    for n, (ns, nt) in enumerate(SIZES + [(900, 33001)]):
        say(f"direct entry {kernel.name} {p2p.name} ns={ns} nt={nt}")
        rng = np.random.default_rng(300 + n)
        src, trg = to_dev(rng.random((ns, 3))), to_dev(rng.random((nt, 3)))
        val = to_dev(source_values(int(uk), ns, rng))
        out, ref = zeros(nt, kt), zeros(nt, kt)
        S.p2p_device(kernel, p2p, src, val, trg, out, precision=S.PREC.MIXED)
        tune = dict(targets_per_lane=1 if nt < 32768 else 2, max_src_per_item=512)
        S.Plan(uk, 1, ns, nt, [0], [nt], None, [0, 1], [0], [ns], tune).execute(src, val, trg, ref)
        l2, mx = O.max_error(host(out), host(ref))
        assert l2 < FP64_TOL and mx < FP64_TOL, (ns, nt, l2, mx)


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
def test_one_launch_nonfinite_and_overflow(prec):
    """A NaN source, a NaN target and (mixed) a pair too close for FP32: as the item-kernel plan."""
    uk, ns, nt = S.UKER.STOKES_PVEL, 700, 200
    say(f"direct nonfinite prec={prec}")
    rng = np.random.default_rng(5)
    for what in ("close", "nan target", "nan source"):
        src, trg = rng.random((ns, 3)), rng.random((nt, 3))
        val = source_values(int(uk), ns, rng)
        trg[3] = src[600] + 1e-14
        if what == "nan target":
            trg[5, 1] = np.nan
        if what == "nan source":
            src[650, 2] = np.nan
        got = []
        for tune in (None, dict(max_src_per_item=512)):
            plan = S.Plan(uk, prec, ns, nt, [0], [nt], None, [0, 1], [0], [ns], tune)
            out = zeros(nt, 4)
            plan.execute(to_dev(src), to_dev(val), to_dev(trg), out)
            got.append(host(out))
        assert np.array_equal(np.isfinite(got[0]), np.isfinite(got[1])), what
        ok = np.isfinite(got[0]).all(axis=1)
        ok[3] = ok[3] and prec == 0  # (mixed: the overflowed target's FP64 part differs in extent)
        if ok.any():
            l2, mx = O.max_error(got[0][ok], got[1][ok])
            assert l2 < FP64_TOL and mx < FP64_TOL, (what, l2, mx)
        if what == "close":
            ref = O.direct(int(uk), src, val, trg[3:4])
            assert np.abs(got[0][3] - ref[0]).max() <= (1e-12 if prec == 0 else 1e-6) * np.abs(ref[0]).max()


def test_output_over_an_input():
    """f += K f: everything is read before anything is written, in every direct entry."""
    n = 700  # one source chunk
    rng = np.random.default_rng(8)
    x, f = rng.random((n, 3)), rng.normal(size=(n, 3))
    ref = f + O.direct(int(S.UKER.STOKES_VEL), x, f, x)
    d_x = to_dev(x)
    plan = S.Plan(S.UKER.STOKES_VEL, 0, n, n, [0], [n], None, [0, 1], [0], [n])
    for name, call in (("entry", lambda v: S.p2p_device(S.KERNEL.Stokes, S.PPKERNEL.SLS2T, d_x, v, d_x, v)),
                       ("no-alloc", lambda v: S.p2p_device(S.KERNEL.Stokes, S.PPKERNEL.SLS2T, d_x, v, d_x, v,
                                                           no_alloc=True)),
                       ("plan", lambda v: plan.execute(d_x, v, d_x, v))):
        say(f"direct in place {name}")
        d_f = to_dev(f)
        call(d_f)
        l2, mx = O.max_error(host(d_f), ref)
        assert l2 < FP64_TOL and mx < FP64_TOL, (name, l2, mx)
    z = x.copy()
    z[:, 2] *= 0.5
    d_z, d_f = to_dev(z), to_dev(f)
    S.wall_device(S.KERNEL.Stokes, d_z, d_f, d_z, d_f)
    l2, mx = O.max_error(host(d_f), f + O.wall(int(S.KERNEL.Stokes), z, f, z))
    assert l2 < FP64_TOL and mx < FP64_TOL, ("wall", l2, mx)


@pytest.mark.parametrize("ns,nt,same", [(16384, 16384, False), (16384, 32767, False), (16384, 32768, False),
                                        (23170, 23170, True), (23171, 23171, True)])
@pytest.mark.parametrize("uk", [0, 8, 13, 15])
def test_fp64_sums_where_ordered_points_begin(uk, ns, nt, same):
    """One launch below 2^29 pairs, ordered points from there: the untuned plan and the device entry against the
    item kernels on the points as given."""
    uk = S.UKER(uk)
    say(f"direct or ordered uk={uk.name} ns={ns} nt={nt}")
    ks, kt = S.uker_dims(uk)
    rng = np.random.default_rng(ns + nt)
    src = rng.random((ns, 3))
    d_src = layout(src, not same)
    d_trg = d_src if same else layout(rng.random((nt, 3)) ** 2, False)
    d_val = layout(source_values(int(uk), ns, rng), True)
    v1, v2 = (d_val[:, :4], d_val[:, 4:]) if uk == S.UKER.STOKES_PVEL_FUSED else (d_val, None)
    perm = rng.permutation(nt).astype(np.int32)
    d_perm = to_dev(perm)
    got = []
    for tune in (dict(max_src_per_item=4096), None):
        plan = S.Plan(uk, 0, ns, nt, [0], [nt], None, [0, 1], [0], [ns], tune)
        out = zeros(nt, kt)
        for _ in range(2):  # adds
            plan.execute(d_src, v1, d_trg, out, src_value2=v2, perm=d_perm)
        got.append(host(out)[perm] / 2)
    out = zeros(nt, kt)
    S.uker_device(uk, d_src.contiguous(), d_val.contiguous(), d_trg.contiguous(), out)
    got.append(host(out))
    for g in got[1:]:
        l2, mx = O.max_error(g, got[0])
        assert l2 < FP64_TOL and mx < FP64_TOL, (l2, mx)
