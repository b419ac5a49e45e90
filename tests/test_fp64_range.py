"""How close and how far two points may be in the FP64 pair forms (stkfmm_amd/csrc/ukernels*.hpp, compiled for the
CPU): every micro-kernel over separations of 2^-143 (9e-44) to 2^145 (4e43).  The pair forms are homogeneous, so scaling
a pair by a power of two scales every output by one exactly, unless an intermediate leaves the range of a double."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_ukernels_host import host_pair

# source values with the dimension of a length (from this index on), which scale with the separation
LENGTHS = {7: 3, 9: 3, 10: 3, 11: 3, 13: 3, 14: 3, 16: 3, 18: 3, 20: 3, 24: 3}


def scaled(uk, r, f, m):
    g = f.copy()
    if uk in LENGTHS:
        g[LENGTHS[uk]:] *= 2.0 ** m
    return host_pair(uk, 0, r * 2.0 ** m, g)


@pytest.mark.parametrize("uk", range(25))
def test_fp64_forms_scale_exactly(uk):
    rng = np.random.default_rng(900 + uk)
    for _ in range(20):
        r = rng.uniform(0.6, 1.0, 3) * rng.choice([-1.0, 1.0], 3) / 2
        f = rng.uniform(0.5, 1.0, O.src_dim(uk))
        one, two = scaled(uk, r, f, 0), scaled(uk, r, f, 1)
        power = np.log2(np.abs(one / two)).round()  # of 1/r in each output
        for m in (-143, -100, 100, 145):
            assert np.array_equal(scaled(uk, r, f, m), one * 2.0 ** (-m * power)), m
