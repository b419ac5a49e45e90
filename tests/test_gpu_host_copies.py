"""GPU: host-pointer sums on both sides of the 1 MiB (131,072 doubles) up to which kernels and above which the copy
engines move a call's inputs, and its results."""
import numpy as np
import pytest

import stkfmm_amd as S
from oracle import oracle as O
from tests.conftest import source_values
from tests.gpu_util import FP64_TOL, MIXED_TOL, say

pytestmark = pytest.mark.gpu

SL, DL = S.PPKERNEL.SLS2T, S.PPKERNEL.DLS2T
CASES = [
    (S.KERNEL.LapPGrad, SL, 0, 32_000, 1_024),  # 131,072 doubles in
    (S.KERNEL.LapPGrad, SL, 0, 32_000, 1_025),
    (S.KERNEL.PVelGrad, SL, 0, 50, 8_192),      # 131,072 doubles out
    (S.KERNEL.PVelGrad, SL, 0, 50, 8_193),
    (S.KERNEL.PVelGrad, SL, 1, 50, 8_193),
    (S.KERNEL.PVelGrad, SL, 0, 16_000, 9_000),  # both above
    (S.KERNEL.PVelGrad, DL, 1, 50, 8_192),      # a plan, which adds
    (S.KERNEL.PVelGrad, DL, 1, 50, 8_193),
    (S.KERNEL.LapPGrad, SL, 0, 23_200, 23_200),  # a plan that orders the points
    (S.KERNEL.LapPGrad, SL, 1, 16_384, 16_384),
]


@pytest.mark.parametrize("kernel,p2p,prec,ns,nt", CASES)
def test_host_sums_around_the_copy_switch(kernel, p2p, prec, ns, nt):
    """Twice with other data into prefilled outputs: a stale workspace would show."""
    uk = S.get_uker(kernel, p2p)
    for seed in (1, 2):
        say(f"host copies {kernel.name} {p2p.name} prec={prec} ns={ns} nt={nt} seed={seed}")
        rng = np.random.default_rng(seed)
        src, trg, val = rng.random((ns, 3)), rng.random((nt, 3)), source_values(int(uk), ns, rng)
        first = rng.normal(size=(nt, S.uker_dims(uk)[1]))
        out = first.copy()
        S.evaluate_kernel(kernel, 1, p2p, src, val, trg, out, precision=S.PREC(prec))
        tol = MIXED_TOL if prec else FP64_TOL
        l2, mx = O.max_error(out - first, O.direct(int(uk), src, val, trg))
        assert l2 < tol and mx < tol, (l2, mx)


@pytest.mark.parametrize("kernel,kt", [(S.KERNEL.Stokes, 3), (S.KERNEL.RPY, 6)])
def test_host_walls_around_the_copy_switch(kernel, kt):
    ks = 3 if kernel == S.KERNEL.Stokes else 4
    for nt in (131_072 // kt, 131_072 // kt + 1):
        say(f"host copies wall {kernel.name} nt={nt}")
        rng = np.random.default_rng(nt)
        x, f, t = rng.random((40, 3)), rng.normal(size=(40, ks)), rng.random((nt, 3))
        if ks == 4:
            f[:, 3] = rng.uniform(1e-3, 5e-3, 40)
        out = np.zeros((nt, kt))
        for _ in range(2):
            S.wall_evaluate(kernel, x, f, t, out)
        ref = O.wall(int(kernel), x, f, t)
        _, cond = O.max_error(O.wall(int(kernel), x[::-1], f[::-1], t), ref)
        l2, mx = O.max_error(out / 2, ref)
        bound = max(4 * cond, FP64_TOL)
        assert l2 < bound and mx < bound, (l2, mx, cond)
