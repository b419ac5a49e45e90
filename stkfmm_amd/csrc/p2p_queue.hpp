// p2p_queue.hpp -- how a wave of the item kernels obtains its next work item, and where its sums go.
//
// Persistent mode: the plan's items are split into n_queues queues (one by default; one per XCD:
// workgroups are dispatched to the XCDs round-robin, so queue blockIdx.x % 8 is the wave's own XCD's, whose items
// share sources in that XCD's L2).  A wave takes an item with one atomic on its queue's counter.  When the
// queue is empty it looks at all others at once and moves on to the next that is not; when none is, it exits.
// Counters only grow and may overshoot their queue's length, so a queue seen empty stays so: at most n_queues
// moves, and every wave reaches the exit.  The host resets them before each launch.
// Otherwise (counter null): one workgroup per item, item = blockIdx.x.
//
// An atomic's round trip is some microseconds when all waves of a launch meet on one counter, and so is each of the
// loads that follow it in a chain (item, targets).  So the first item of a single queue is item blockIdx.x without
// an atomic (the queue then goes on at gridDim.x), the next one is asked for before the finished one is written
// out, and its record read before the sums are stored.  Waves of short items spent two thirds of their time so
// and in the chain of loads and stores of write_sums: the four PVel lists around a 262,144-point tree's surfaces,
// mixed, 1.557 -> 1.376 ms; U-lists of 65,536 points 1.1 to 1.4 times faster (Stokeslet 0.201 -> 0.154 ms FP64,
// 0.175 -> 0.133 mixed), of 262,144 points 1-5 % (PVel 1.025 -> 0.988 ms FP64).
#pragma once

#include <hip/hip_runtime.h>

#include "p2p_internal.hpp"
#include "ukernels.hpp"

namespace stkp2p {

struct ItemCursor {
    int q;
    __device__ explicit ItemCursor(const ItemArgs &a)
        : q((a.counter && a.n_queues > 1) ? (int)(blockIdx.x % (unsigned)a.n_queues) : 0) {}
};

// asks for the wave's next item: lane 0's result is the ticket
__device__ __forceinline__ int request_item(const ItemArgs &a, const ItemCursor &c, int lane) {
    int ticket = 0;
    if (a.counter && lane == 0)
        ticket = atomicAdd(a.counter + c.q, 1);
    return ticket;
}

// the first item of this wave (uniform across the wave), or -1
__device__ __forceinline__ int take_item(const ItemArgs &a, ItemCursor &c, int lane, int ticket);
__device__ __forceinline__ int first_item(const ItemArgs &a, ItemCursor &c, int lane) {
    if (a.counter && a.n_queues > 1)
        return take_item(a, c, lane, request_item(a, c, lane));
    return (int)blockIdx.x < a.n_items ? (int)blockIdx.x : -1;
}

// the item asked for (uniform across the wave), or -1 when there is none left
__device__ __forceinline__ int take_item(const ItemArgs &a, ItemCursor &c, int lane, int ticket) {
    if (!a.counter)
        return -1;
    if (a.n_queues == 1) {
        const long long it = (long long)gridDim.x + __builtin_amdgcn_readfirstlane(ticket);
        return it < a.n_items ? (int)it : -1;
    }
    for (;;) {
        const int it = a.q_ptr[c.q] + __builtin_amdgcn_readfirstlane(ticket);
        if (it < a.q_ptr[c.q + 1])
            return it;
        int to = -1;
        for (int d0 = 1; to < 0 && d0 < a.n_queues; d0 += kWave) {
            bool open = false;
            int q = c.q + d0 + lane;
            q -= (q >= a.n_queues) ? a.n_queues : 0;
            if (d0 + lane < a.n_queues)
                open = __hip_atomic_load(a.counter + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
                       a.q_ptr[q + 1] - a.q_ptr[q];
            const unsigned long long m = __ballot(open);
            if (m)
                to = c.q + d0 + __builtin_ctzll(m);
        }
        if (to < 0)
            return -1;
        c.q = to - ((to >= a.n_queues) ? a.n_queues : 0);
        ticket = request_item(a, c, lane);
    }
}

// A finished item's sums (before post(), in the item's level frame) of its target slots slot0 + tstride t,
// by the lanes that hold them (mine): into its partial slot for the reduction, or, when the item is its
// tile's only one, straight into the output with the reduction's own operations (out += scale * sum) --
// no partial sums to write and read again, and no reduction where every tile is such.  Surface lists (one
// leaf's points against its surface) are all such tiles: the four PVel lists of a 262,144-point tree, mixed,
// 1.65 -> 1.58 ms.
// The loads of as many targets as fit kWriteLoads values are in flight together (the output could overlap the
// permutation for all the compiler knows, so that it would keep each load behind the store before it); between:
// called after they are issued, before the sums are stored.
constexpr int kWriteLoads = 16;
template <class K, int PREC, int T, class Between>
__device__ __forceinline__ void write_sums(const Item &item, const double (&out)[T][K::KT], int slot0, int tstride,
                                           bool mine, Between between) {
    constexpr int KT = K::KT, TT = kWave * T;
    // the kernels' first argument, read here again: held in scalar registers over the pair loops, the output's
    // description costs them up to 20 spills (4M RPY U-list FP64 +1 %)
    typedef const __attribute__((address_space(4))) ItemArgs *Args;
    Args a = (Args)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    const bool whole = a->whole_out && (item.lsplit & kItemWhole);
    if (!whole) {
        double *dst = a->partial + (long long)item.slot * KT * TT;
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
        between();
    } else {
        constexpr int B = (T * KT <= kWriteLoads) ? T : 1; // targets a batch
        double *const out_p = a->out.p;
        const long long out_s = a->out.s, out_fs = a->out.fs;
        const int *const perm = a->perm;
        const double scale = a->scale;
#pragma unroll
        for (int t0 = 0; t0 < T; t0 += B) {
            double *o[B];
            double old[B][KT];
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int i = slot0 + tstride * (t0 + b);
                const bool ok = mine && i < item.trg_count;
                long long row = item.trg_begin + (ok ? i : 0);
                if (perm) {
                    row = perm[row];
                    // waited for here: where the two ways meet, the wait would be for everything in flight
                    asm volatile("" : "+v"(row));
                }
                o[b] = out_p + row * out_s;
#pragma unroll
                for (int k = 0; k < KT; ++k)
                    old[b][k] = ok ? o[b][k * out_fs] : 0.0;
            }
            if (t0 + B >= T)
                between();
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int i = slot0 + tstride * (t0 + b);
                if (!mine || i >= item.trg_count)
                    continue;
#pragma unroll
                for (int k = 0; k < KT; ++k) {
                    const double osc =
                        ((PREC == 0) ? 1.0 : ldexp(1.0, K::deg(k) * item.level)) * post_for<K, PREC>(k);
                    o[b][k * out_fs] = old[b][k] + scale * (out[t0 + b][k] * osc);
                }
            }
        }
    }
}

} // namespace stkp2p
