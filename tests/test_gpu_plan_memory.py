"""GPU: device memory of untuned FP64 plans of one group, which order their points in copies of the arrays."""
import numpy as np
import pytest

import stkfmm_amd as S
from oracle import oracle as O
from tests.gpu_util import FP64_TOL, host, say, to_dev, torch, zeros

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pad_src,pad_trg", [(20_000_000, 0), (0, 20_000_000), (0, 0)])
def test_a_range_of_long_arrays_takes_memory_for_itself(pad_src, pad_trg):
    """25,000 points of arrays of 20 million: no copies of the arrays (640 MB and more); of their own: the same sums."""
    n = 25_000
    say(f"plan memory pad_src={pad_src} pad_trg={pad_trg}")
    t = torch()
    rng = np.random.default_rng(n)
    src, trg, val = rng.random((n, 3)), rng.random((n, 3)), rng.normal(size=(n, 1))
    arrays = [zeros(n + pad, k) for pad, k in ((pad_src, 3), (pad_src, 1), (pad_trg, 3))]
    for a, x in zip(arrays, (src, val, trg)):
        a[-n:] = to_dev(x)
    free = t.cuda.mem_get_info()[0]
    plan = S.Plan(S.UKER.LAPLACE_P, 0, n + pad_src, n + pad_trg, [pad_trg], [n + pad_trg], None, [0, 1], [pad_src],
                  [n + pad_src])
    used = free - t.cuda.mem_get_info()[0]
    assert used < 200e6, used
    out = zeros(n + pad_trg, 1)
    plan.execute(arrays[0], arrays[1], arrays[2], out)
    l2, mx = O.max_error(host(out[-n:]), O.direct(int(S.UKER.LAPLACE_P), src, val, trg))
    assert l2 < FP64_TOL and mx < FP64_TOL, (l2, mx)
    assert not pad_trg or not host(out[:pad_trg].any())
