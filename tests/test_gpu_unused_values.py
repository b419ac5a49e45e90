"""GPU: second source values of a micro-kernel that has none are ignored, whatever they are."""
import numpy as np
import pytest

import stkfmm_amd as S
from tests.gpu_util import host, say, to_dev, zeros

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 9), (5,), (5, 3, 3)])
def test_second_values_are_ignored(shape):
    say(f"unused second values {shape}")
    rng = np.random.default_rng(1)
    x, v = to_dev(rng.random((5, 3))), to_dev(rng.normal(size=(5, 3)))
    plan = S.Plan(S.UKER.STOKES_VEL, 0, 5, 5, [0], [5], None, [0, 1], [0], [5])
    ref, out = zeros(5, 3), zeros(5, 3)
    plan.execute(x, v, x, ref)
    plan.execute(x, v, x, out, src_value2=to_dev(np.zeros(shape)))
    assert np.array_equal(host(out), host(ref))
