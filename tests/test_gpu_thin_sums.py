"""GPU: direct sums of few sources and many targets on both sides of the line from which the item kernels take them."""
import numpy as np
import pytest

import stkfmm_amd as S
from oracle import oracle as O
from tests.conftest import source_values
from tests.gpu_util import FP64_TOL, host, say, to_dev, torch, zeros

pytestmark = pytest.mark.gpu


def problem(uk, ns, nt):
    rng = np.random.default_rng(ns)
    t = torch()
    g = t.Generator(device="cuda:0").manual_seed(nt)
    trg = t.rand((nt, 3), dtype=t.float64, device="cuda:0", generator=g)
    return to_dev(rng.random((ns, 3))), to_dev(source_values(int(uk), ns, rng)), trg


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("kernel", [S.KERNEL.LapPGrad, S.KERNEL.RPY, S.KERNEL.PVelGrad])
@pytest.mark.parametrize("ns,nt", [(8192, 524_287), (8192, 524_288), (16_000, 268_500)])
def test_entry_and_plan_match_items(kernel, ns, nt, prec):
    """The device entry, twice into one output, and the untuned plan against the item kernels."""
    uk = S.get_uker(kernel, S.PPKERNEL.SLS2T)
    kt = S.uker_dims(uk)[1]
    say(f"thin {kernel.name} ns={ns} nt={nt} prec={prec}")
    src, val, trg = problem(uk, ns, nt)

    def plan(tune):
        o = zeros(nt, kt)
        S.Plan(uk, prec, ns, nt, [0], [nt], None, [0, 1], [0], [ns], tune).execute(src, val, trg, o)
        return host(o)

    out = zeros(nt, kt)
    for _ in range(2):
        S.p2p_device(kernel, S.PPKERNEL.SLS2T, src, val, trg, out, precision=S.PREC(prec))
    # (in mixed mode the FP32 sums are those of the same number of targets per lane: two in the entry, the kernel's
    # default in a plan)
    for name, got, ref in (("entry", host(out) / 2, plan(dict(targets_per_lane=2, max_src_per_item=4096))),
                           ("plan", plan(None), plan(dict(max_src_per_item=4096)))):
        l2, mx = O.max_error(got, ref)
        assert l2 < FP64_TOL and mx < FP64_TOL, (name, l2, mx)


def test_first_call_under_capture():
    """A first call of its shape inside a capture, where no plan can be made: replays equal the eager call."""
    kernel, uk, ns, nt = S.KERNEL.Stokes, S.UKER.STOKES_VEL, 8200, 524_300
    say(f"thin capture ns={ns} nt={nt}")
    t = torch()
    src, val, trg = problem(uk, ns, nt)
    out = zeros(nt, 3)
    warm = zeros(10, 3)
    S.p2p_device(kernel, S.PPKERNEL.SLS2T, src[:10], val[:10], trg[:10], warm)
    host(warm)
    graph = t.cuda.CUDAGraph()
    with t.cuda.graph(graph):
        S.p2p_device(kernel, S.PPKERNEL.SLS2T, src, val, trg, out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        got = host(out)
        eager = zeros(nt, 3)
        S.p2p_device(kernel, S.PPKERNEL.SLS2T, src, val, trg, eager)
        l2, mx = O.max_error(got, host(eager))
        assert l2 < FP64_TOL and mx < FP64_TOL, (l2, mx)
