"""GPU: how the item kernels hand out their work list -- queues, workgroups, items that write the output themselves --
does not change a bit of the result."""
import numpy as np
import pytest

import stkfmm_amd as S
from oracle import oracle as O
from tests.conftest import source_values
from tests.gpu_util import FP64_TOL, host, say, to_dev, zeros

pytestmark = pytest.mark.gpu


# one item; fewer items than queues; more items than waves of the launch; groups of odd sizes (cut tiles, lane
# splits), with one and with several items a tile
@pytest.mark.parametrize("bc", [0, 1], ids=["lds", "scalar"])
@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("groups,uk", [(1, 0), (7, 15), (40, 7), (9001, 2)])
def test_queues_give_the_same_bits(groups, uk, prec, bc):
    uk = S.UKER(uk)
    say(f"queues groups={groups} uk={uk.name} prec={prec} bc={bc}")
    rng = np.random.default_rng(groups)
    cnt = rng.integers(1, 6 if groups > 1000 else 300, groups)
    tb = np.concatenate([[0], np.cumsum(cnt)])
    ns, nt = 500, int(tb[-1])
    sb = rng.integers(0, 200, groups)
    se = sb + rng.integers(0, 300, groups)  # empty source lists too
    src, trg, val = rng.random((ns, 3)), rng.random((nt, 3)), source_values(int(uk), ns, rng)
    d_src, d_trg, d_val = to_dev(src), to_dev(trg), to_dev(val)
    perm = to_dev(rng.permutation(nt).astype(np.int32))
    first = rng.random((nt, S.uker_dims(uk)[1]))
    out = []
    for tune in (dict(), dict(persistent=2), dict(queues=2), dict(queues=8), dict(queues=65), dict(queues=256),
                 dict(queues=8, waves_per_cu=1), dict(waves_per_cu=1)):
        plan = S.Plan(uk, prec, ns, nt, tb[:-1], tb[1:], None, np.arange(groups + 1), sb, se,
                      dict(targets_per_lane=2, broadcast=bc, max_src_per_item=128, **tune))
        o = to_dev(first)
        for _ in range(2):  # adds; the counters are reset
            plan.execute(d_src, d_val, d_trg, o, perm=perm)
        out.append(host(o))
    for o in out[1:]:
        assert np.array_equal(o, out[0])
    if prec == 0 and groups <= 40:
        ref = np.zeros_like(first)
        for g in range(groups):
            if se[g] > sb[g]:
                ref[tb[g]:tb[g + 1]] = O.direct(int(uk), src[sb[g]:se[g]], val[sb[g]:se[g]], trg[tb[g]:tb[g + 1]])
        got = (out[0] - first)[host(perm)] / 2
        l2, mx = O.max_error(got, ref)
        assert l2 < FP64_TOL and mx < FP64_TOL, (l2, mx)


# total work below and above each step of the default FP64 item size (192 .. 512 sources), against items of 512
@pytest.mark.parametrize("groups,per", [(1, 191), (30, 193), (3000, 500), (9000, 900), (20000, 1300)])
@pytest.mark.parametrize("uk", [2, 15])
def test_default_fp64_items(uk, groups, per):
    uk = S.UKER(uk)
    say(f"default items uk={uk.name} groups={groups} sources={per}")
    rng = np.random.default_rng(per)
    ns, nt = 2000, groups * 2
    sb = rng.integers(0, ns - per, groups)
    src, trg, val = rng.random((ns, 3)), rng.random((nt, 3)), source_values(int(uk), ns, rng)
    out = []
    for tune in (None, dict(max_src_per_item=512)):
        plan = S.Plan(uk, 0, ns, nt, np.arange(0, nt, 2), np.arange(0, nt, 2) + 2, None, np.arange(groups + 1), sb,
                      sb + per, tune)
        o = zeros(nt, S.uker_dims(uk)[1])
        plan.execute(to_dev(src), to_dev(val), to_dev(trg), o)
        out.append(host(o))
    l2, mx = O.max_error(out[0], out[1])
    assert l2 < FP64_TOL and mx < FP64_TOL, (l2, mx)
