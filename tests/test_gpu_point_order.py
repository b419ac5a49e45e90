"""GPU: plans that order their points, against the same plan unordered, at the edges of the ordering's blocks and
grid levels; and the reduction of partial sums at the edges of its grouping."""
import numpy as np
import pytest

import stkfmm_amd as S
from oracle import oracle as O
from tests.conftest import source_values
from tests.gpu_util import FP64_TOL, host, say, to_dev, zeros

pytestmark = pytest.mark.gpu


def sums(uk, n_src, n_trg, groups, tune, src, val, trg, perm=None):
    tb, te, sb, se = (list(map(int, x)) for x in zip(*groups))
    plan = S.Plan(uk, 0, n_src, n_trg, tb, te, None, list(range(len(groups) + 1)), sb, se, tune)
    out = zeros(n_trg, S.uker_dims(uk)[1])
    v1, v2 = (val[:, :4], val[:, 4:]) if uk == S.UKER.STOKES_PVEL_FUSED else (val, None)
    plan.execute(src, v1, trg, out, src_value2=v2, perm=perm)
    plan.execute(src, v1, trg, out, src_value2=v2, perm=perm)  # adds
    return host(out) / 2


# (the second of two groups takes 7 sources and 17 targets) one block and one more; each level's last size and
# the next; many runs of blocks; level 4
@pytest.mark.parametrize("ns,nt", [(1, 1), (519, 530), (520, 529), (4103, 4114), (4104, 81), (32776, 147),
                                   (137, 100001), ((1 << 18) + 8, 87)])
@pytest.mark.parametrize("uk", [2, 8, 13])
def test_ordered_as_unordered(uk, ns, nt):
    uk = S.UKER(uk)
    say(f"ordered uk={uk.name} ns={ns} nt={nt}")
    rng = np.random.default_rng(ns + nt)
    src, trg = rng.random((ns, 3)), rng.random((nt, 3)) ** 2
    val = to_dev(source_values(int(uk), ns, rng))
    perm = to_dev(rng.permutation(nt).astype(np.int32))
    # two groups, the second with a source range and targets of its own
    groups = [(0, nt, 0, ns)] if ns < 2 else [(0, nt - 17, 0, ns - 7), (nt - 17, nt, ns - 7, ns)]
    ref, got = (sums(uk, ns, nt, groups, dict(sort_points=o, targets_per_lane=2, max_src_per_item=2048),
                     to_dev(src), val, to_dev(trg), perm) for o in (0, 1))
    l2, mx = O.max_error(got, ref)
    assert l2 < FP64_TOL and mx < FP64_TOL, (l2, mx)


# below and from the tile count that sums four components side by side; outputs that do not divide by four
@pytest.mark.parametrize("tiles", [1, 2047, 2048, 2051])
@pytest.mark.parametrize("uk", [0, 5, 10, 15])
def test_reduction_of_many_tiles(uk, tiles):
    uk = S.UKER(uk)
    say(f"reduce uk={uk.name} tiles={tiles}")
    rng = np.random.default_rng(tiles)
    ns, per = 700, 3
    src, trg = rng.random((ns, 3)), rng.random((per * tiles, 3))
    sval = source_values(int(uk), ns, rng)
    groups = [(per * g, per * g + per, 0, ns) for g in range(tiles)]
    got = sums(uk, ns, per * tiles, groups, dict(max_src_per_item=100), to_dev(src), to_dev(sval), to_dev(trg))
    l2, mx = O.max_error(got, O.direct(int(uk), src, sval, trg))
    assert l2 < FP64_TOL and mx < FP64_TOL, (l2, mx)
