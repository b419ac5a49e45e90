"""GPU: the FP64 adjoint on both sides of the sizes where its targets per lane change (one, two, four at 256 compute
units: 8 tiles of targets and sources per unit)."""
import numpy as np
import pytest

import stkfmm_amd as S
from oracle import oracle as O
from tests.conftest import source_values
from tests.gpu_util import host, say, to_dev

pytestmark = pytest.mark.gpu


# 4,133 targets are 65, 33 or 17 tiles; 62 and 63, 120 and 121 tiles of sources
@pytest.mark.parametrize("uk", [2, 6, 7, 8, 11, 13])
@pytest.mark.parametrize("ns,nt", [(3_968, 4_133), (3_969, 4_133), (7_680, 4_133), (7_681, 4_133), (64, 1_023),
                                   (65, 1_024), (2_000, 4_096)])
def test_fp64_adjoint_where_targets_per_lane_change(uk, ns, nt):
    say(f"vjp layout uker={uk} ns={ns} nt={nt}")
    rng = np.random.default_rng(ns + uk)
    src = rng.random((ns, 3))
    trg = np.concatenate([src[:9], rng.random((nt - 9, 3))])
    v = source_values(uk, ns, rng)
    w = rng.normal(size=(nt, O.trg_dim(uk)))
    ref = O.direct_vjp(uk, src, v, trg, w)
    for need in ((True, True, True), (False, True, False)):
        got = S.vjp_device(uk, to_dev(src), to_dev(v), to_dev(trg), to_dev(w), precision=0, need=need)
        for g, r, name in zip(got, ref, ("g_src_value", "g_src_coord", "g_trg_coord")):
            if g is not None:
                l2, mx = O.max_error(host(g), r)
                assert l2 < 1e-11 and mx < 1e-11, (name, l2, mx)
