// direct_layout_host.cpp -- test harness: the host rules of the direct sums (p2p_direct_layout.hpp,
// p2p_internal.hpp) behind C functions, so tests/test_direct_layout.py can check them without a GPU.  Built by
// stkfmm_amd/csrc/Makefile.  Not part of the library.
#include "../../stkfmm_amd/csrc/p2p_direct_layout.hpp"

using namespace stkp2p;

// direct_out_overlaps of views given as (first byte address, row stride, component stride) in x[3]
extern "C" int direct_overlaps_host(const unsigned long long *sc, const unsigned long long *v1,
                                    const unsigned long long *v2, const unsigned long long *tc,
                                    const unsigned long long *out, int perm, long long out_rows, int n_src,
                                    int n_trg, int ks, int ks1, int kt) {
    static const int some_perm = 0;
    const auto in = [](const unsigned long long *x) {
        return DArr{(const double *)(uintptr_t)x[0], (long long)x[1], (long long)x[2]};
    };
    DirectArgs a{};
    a.sc = in(sc);
    a.v1 = in(v1);
    a.v2 = in(v2);
    a.tc = in(tc);
    a.out = OArr{(double *)(uintptr_t)out[0], (long long)out[1], (long long)out[2]};
    a.perm = perm ? &some_perm : nullptr;
    a.n_src = n_src;
    a.n_trg = n_trg;
    return direct_out_overlaps(a, out_rows, ks, ks1, kt);
}

// the cut of an n_src x n_trg sum of micro-kernel outputs kt (mixed mode: FP32 runs of `run` sources) on n_cu CUs, T
// targets per lane: out = {units, chunks, chunk_tiles, waves, unit, ls, tail_begin, tail_ls}
extern "C" void direct_layout_host(int prec, int T, int kt, int run, int n_src, int n_trg, int n_cu, int *out) {
    const DirectLayout l = direct_layout(prec, T, direct_cost(prec, kt), kt, run, n_src, n_trg, n_cu);
    const int v[8] = {l.units, l.chunks, l.chunk_tiles, l.waves, l.unit, l.ls, l.tail_begin, l.tail_ls};
    for (int k = 0; k < 8; ++k)
        out[k] = v[k];
}

extern "C" int direct_items_pay_host(long long n_src, long long n_trg) { return direct_items_pay(n_src, n_trg); }

// threads of the launches over the targets: the sum's along x, the reduction's
extern "C" void direct_threads_host(int prec, int T, int kt, int max_waves, int n_src, int n_trg, long long *out) {
    DirectCost cost = direct_cost(prec, kt);
    if (max_waves > 0)
        cost.max_waves = max_waves;
    const DirectLayout l = direct_layout(prec, T, cost, kt, 16, n_src, n_trg, 256);
    out[0] = (long long)l.units * kWave * l.waves;
    out[1] = direct_reduce_blocks(n_trg) * 256LL;
}

extern "C" int direct_sizes_host(int n_src, int n_trg) { return direct_sizes(n_src, n_trg); }
