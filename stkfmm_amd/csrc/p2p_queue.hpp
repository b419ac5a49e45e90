// p2p_queue.hpp -- how a wave of the item kernels obtains its next work item, and where its sums go.
//
// Persistent mode: the plan's items are split into n_queues queues (one per XCD by default).  A wave
// starts on queue blockIdx.x % n_queues -- workgroups are dispatched to the XCDs round-robin, so
// that is the queue of the wave's own XCD, whose items share sources in that XCD's L2 -- and takes
// items with one atomic per item.  When its queue is empty it moves to the next queue, and after
// it has found every queue empty it exits: at most n_queues moves, so every wave reaches the exit.
// Counters may overshoot their queue's length; the host resets them before each launch.
// Otherwise (counter null): one workgroup per item, item = blockIdx.x.
#pragma once

#include <hip/hip_runtime.h>

#include "p2p_internal.hpp"
#include "ukernels.hpp"

namespace stkp2p {

struct ItemCursor {
    int q;
    int moves;
    bool first;
    __device__ explicit ItemCursor(const ItemArgs &a)
        : q(a.counter ? (int)(blockIdx.x % (unsigned)a.n_queues) : 0), moves(0), first(true) {}
};

// next item of this wave (uniform across the wave), or -1 when there is none left
__device__ inline int next_item(const ItemArgs &a, ItemCursor &c, int lane) {
    if (!a.counter) {
        if (!c.first)
            return -1;
        c.first = false;
        return (int)blockIdx.x < a.n_items ? (int)blockIdx.x : -1;
    }
    for (;;) {
        int v = 0;
        if (lane == 0)
            v = atomicAdd(a.counter + c.q, 1);
        v = __builtin_amdgcn_readfirstlane(v);
        const int it = a.q_ptr[c.q] + v;
        if (it < a.q_ptr[c.q + 1])
            return it;
        if (++c.moves >= a.n_queues)
            return -1;
        c.q = (c.q + 1 == a.n_queues) ? 0 : c.q + 1;
    }
}

// A finished item's sums (before post(), in the item's level frame) of its target slots slot0 + tstride t,
// by the lanes that hold them (mine): into its partial slot for the reduction, or, when the item is its
// tile's only one, straight into the output with the reduction's own operations (out += scale * sum) --
// no partial sums to write and read again, and no reduction where every tile is such.  Surface lists (one
// leaf's points against its surface) are all such tiles: the four PVel lists of a 262,144-point tree, mixed,
// 1.65 -> 1.58 ms.
template <class K, int PREC, int T>
__device__ __forceinline__ void write_sums(const Item &item, const double (&out)[T][K::KT], int slot0, int tstride,
                                           bool mine) {
    constexpr int KT = K::KT, TT = kWave * T;
    // the kernels' first argument, read here again: held in scalar registers over the pair loops, the output's
    // description costs them up to 20 spills (4M RPY U-list FP64 +1 %)
    typedef const __attribute__((address_space(4))) ItemArgs *Args;
    Args a = (Args)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    const bool whole = a->whole_out && (item.lsplit & kItemWhole);
    double *dst = a->partial + (long long)item.slot * KT * TT;
    if (!whole) {
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            const double osc = ((PREC == 0) ? 1.0 : ldexp(1.0, K::deg(k) * item.level)) * post_for<K, PREC>(k);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int i = slot0 + tstride * t;
                if (mine && i < item.trg_count)
                    dst[(long long)k * TT + i] = out[t][k] * osc;
            }
        }
    } else {
        double *const out_p = a->out.p;
        const long long out_s = a->out.s, out_fs = a->out.fs;
        const int *const perm = a->perm;
        const double scale = a->scale;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int i = slot0 + tstride * t;
            if (!mine || i >= item.trg_count)
                continue;
            const long long row = item.trg_begin + i;
            double *o = out_p + (perm ? (long long)perm[row] : row) * out_s;
#pragma unroll
            for (int k = 0; k < KT; ++k) {
                const double osc = ((PREC == 0) ? 1.0 : ldexp(1.0, K::deg(k) * item.level)) * post_for<K, PREC>(k);
                o[k * out_fs] += scale * (out[t][k] * osc);
            }
        }
    }
}

} // namespace stkp2p
