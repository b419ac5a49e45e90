// p2p_direct_layout.hpp -- how a direct sum is cut into workgroups (host side of p2p_direct.hpp).
#pragma once

#include "p2p_internal.hpp"

namespace stkp2p {

constexpr int kDirectWaves = 8; // waves per workgroup, at most
constexpr long long kMaxGridThreads = 1LL << 32; // of a launch, along each axis: below this

struct DirectLayout {
    int T;           // targets per lane
    int ls;          // log2 lanes per target
    int unit;        // targets per workgroup, 64*T >> ls
    int units;       // workgroups over the targets (blockIdx.x)
    int tail_begin;  // mixed: first target of the partly filled tile whose lanes split the runs, ...
    int tail_ls;     // ... and its log2 lanes per target (0: no such tile; it is then the last unit)
    int chunks;      // source chunks (blockIdx.y)
    int chunk_tiles; // 64-source tiles per chunk
    int waves;       // waves per workgroup
};

// The cheapest cut by a model of one CU, in cycles: a wave of a workgroup stages a source tile (kStage)
// and evaluates its 64 sources with 64*T >> ls pairs each, 64 lanes at a time (about 50 + 15 KT cycles
// a pair and lane in FP64, 50 + 8 KT in mixed mode); a CU holds ceil(workgroups / CUs) workgroups on
// four SIMDs, and fewer than about three waves on a SIMD run at the latency of their dependency chain
// (kAlone).  The partial sums of c chunks cost a second launch and their reads, kReduce + c kChunk, and kValue
// a value where there are many: the array holds kDirectPartial values, so that a sum of some 10^5 targets still
// comes in whole rounds of workgroups (16,000 x 100,000 LapPGrad, 782 units on 256 CUs, in four chunks: FP64
// 1,196 -> 1,060 us, mixed 998 -> 857; 120,000^2 without allocation, in three, 10.4 -> 9.0 ms FP64).  Fitted
// to a sweep of ls, chunks and waves over 11 shapes in each precision; the cut taken is within 15 % of
// the sweep's best (for instance 8192^2 LapPGrad FP64 54 us, best 53; 9,000 x 1,000 PVel 19 us, best 18).
struct DirectCost {
    double pair;   // cycles of a pair in one lane
    int max_waves; // waves per workgroup, at most: half of kDirectWaves where registers leave two or three
                   // waves per SIMD (more than six outputs: 120-156 VGPRs), so that workgroups pack
    int overlap;   // workgroups of a CU whose set-up (targets, the waves' sums) overlaps others' pairs
};
inline DirectCost direct_cost(int prec, int kt) {
    return DirectCost{prec == 0 ? 50.0 + 15.0 * kt : 50.0 + 8.0 * kt, kt > 6 ? kDirectWaves / 2 : kDirectWaves,
                      kt <= 4 ? 4 : (kt <= 6 ? 1 : 2)};
}
inline DirectLayout direct_layout(int prec, int T, const DirectCost &cost, int kt, int run, int n_src, int n_trg,
                                  int n_cu) {
    const int TT = kWave * T;
    const long long stiles = ((long long)n_src + kSrcTile - 1) / kSrcTile;
    DirectLayout best{};
    double best_t = -1.0;
    const int ls_max = (prec == 0) ? 4 : (run >= 64 ? 0 : (run == 32 ? 1 : 2));
    const double kStage = 800.0, kSetup = 4000.0, kReduce = 8000.0, kChunk = 250.0, kValue = 0.01, kFew = 131072.0, kAlone = 3.0;
    for (int ls = 0; ls <= ls_max; ++ls) {
        DirectLayout l{};
        l.T = T;
        l.ls = ls;
        l.unit = TT >> ls;
        if (prec != 0) {
            const int rem = n_trg % TT;
            l.tail_ls = rem ? tile_lsplit(rem, TT) : 0;
            l.tail_begin = l.tail_ls ? n_trg - rem : n_trg;
            l.units = (l.tail_begin + l.unit - 1) / l.unit + (l.tail_ls ? 1 : 0);
        } else {
            l.tail_begin = n_trg;
            l.units = (n_trg + l.unit - 1) / l.unit;
        }
        for (int c = 1; c <= stiles; c = (c < 8) ? c + 1 : c + c / 4) {
            if (c > 1 && ((long long)c * n_trg * kt > kDirectPartial || c > 65535))
                break;
            l.chunk_tiles = (int)((stiles + c - 1) / c);
            l.chunks = (int)((stiles + l.chunk_tiles - 1) / l.chunk_tiles);
            l.waves = cost.max_waves;
            while (l.waves > 1 && l.waves / 2 >= l.chunk_tiles)
                l.waves /= 2;
            while (l.waves > 1 && (long long)l.units * kWave * l.waves >= kMaxGridThreads)
                l.waves /= 2;
            if ((long long)l.units * kWave * l.waves >= kMaxGridThreads)
                continue;
            const double rounds = (double)((l.chunk_tiles + l.waves - 1) / l.waves);
            const double wave_t = rounds * (kStage + (kWave >> ls) * T * cost.pair);
            const long long wgs = ((long long)l.units * l.chunks + n_cu - 1) / n_cu;
            const double per_simd = (double)(wgs * l.waves) / 4.0; // waves a SIMD has to run
            const double t = kSetup * (double)((wgs + cost.overlap - 1) / cost.overlap) +
                             wave_t * ((per_simd > kAlone ? per_simd : kAlone) + 0.25) +
                             (l.chunks > 1 ? kReduce + kChunk * l.chunks : 0.0) +
                             ((long long)c * n_trg > kFew ? kValue * l.chunks * kt * n_trg : 0.0);
            if (best_t < 0.0 || t < best_t) {
                best_t = t;
                best = l;
            }
        }
    }
    return best;
}

// the layout of micro-kernel uk's direct sum, T targets per lane
inline DirectLayout direct_layout_uk(int uk, int prec, int T, int n_src, int n_trg, int n_cu) {
    DirectCost cost = direct_cost(prec, uker_kt(uk));
    // regularised force and torque with the rotation, and the fused PVel: as more than six outputs (152 and 160
    // VGPRs; 16,000 x 50,000 of the first 1.97 -> 1.62 ms, with the chunks above)
    if (prec == 0 && (uk == 20 || uk == 13))
        cost.max_waves = kDirectWaves / 2;
    return direct_layout(prec, T, cost, uker_kt(uk), uker_run(uk), n_src, n_trg, n_cu);
}

} // namespace stkp2p
