// p2p_direct.hpp -- one target group against one source range (a direct sum) in one launch, or one and a reduction.
//
// The item kernels give a 64*T-target tile and 512 or more sources to one wave, and a second launch
// sums the waves' partial results.  A small sum then has a handful of waves on 256 CUs (1,000 x
// 1,000: 32), each a serial chain of 512 sources.  Here a workgroup of W waves owns a unit of targets
// and shares out the source tiles (64 sources) among its waves: wave w stages and evaluates tiles w,
// w + W, ... from LDS of its own (no barrier inside the loop; the next tile's loads are in flight
// while one is evaluated), the waves' sums meet in LDS at the end, and the caller's output is written
// by the same launch.  A unit is 64*T >> ls targets: 2^ls lanes share a target and split each tile's
// sources between them, which gives a sum of few targets enough workgroups.  Where CUs would idle all the
// same, or the last round of workgroups be nearly empty, the sources are cut into chunks as well (blockIdx.y), whose
// partial results [chunk][KT][n_trg] direct_reduce_kernel adds up in a second launch: 8192^2 in 8 chunks, 3,001 x
// 2,503 in 6, 1,000^2 in one.  The layout is the cheapest by the cost model of direct_layout
// (p2p_direct_layout.hpp).  Measured on MI355X, whole calls on resident points,
// item kernel + reduce -> this kernel (+ reduction): LapPGrad FP64 8192^2 95 -> 52 us (705 -> 1290 Gpair/s; bound by its
// FP64 issue from there, 45 us), Stokeslet mixed 3,001 x 2,503 82 -> 16 us of GPU time; 24 Ker_t blocks of
// different sizes on host arrays 3.7 -> 1.2 ms (no work list to build and upload for a new size).
//
// FP64: lane part sub takes sources sub, sub + 2^ls, ... of a tile.  Mixed mode keeps the item
// kernel's FP32 partial sums, source by source: runs of MixedFlush<K> consecutive sources of a tile
// are summed in FP32 by one lane and added to its FP64 accumulator, so lanes share a target by whole
// runs; the last, partly filled 64*T tile of targets is the exception, as there (its lanes split the
// runs source by source, tile_lsplit).  Every pair takes the coincidence mask: the points come in the
// caller's order, so a unit's targets span the whole cloud and no tile would be clear of their box.
#pragma once

#include <hip/hip_runtime.h>

#include "p2p_clear.hpp"
#include "p2p_direct_layout.hpp"
#include "p2p_internal.hpp"
#include "p2p_mixed.hpp"
#include "ukernels.hpp"

namespace stkp2p {

// LDS of one wave, in doubles: FP64 [3 + KL][64] (coordinates and staged values); mixed [3][64] FP64
// coordinates and [64] rows of KLP FP32 values (16-byte quads, pitch not a multiple of 4 quads)
template <class K, int PREC> struct DirectLds {
    static constexpr int KL = StagedCount<K, PREC>::value;
    static constexpr int KLQ = (KL + 3) / 4;
    static constexpr int KLP = 4 * ((KLQ % 4 == 0) ? KLQ + 1 : KLQ);
    static constexpr int WORDS = (PREC == 0) ? (3 + KL) * kSrcTile : 3 * kSrcTile + kSrcTile * KLP / 2;
};

// pairs of a source and its wall image (wall_pairs.hpp), which take the heights over the wall as well
template <class K, class = void> struct IsWallPair { static constexpr bool value = false; };
template <class K> struct IsWallPair<K, decltype((void)K::WALL)> { static constexpr bool value = K::WALL; };

// LDS written by some lanes of a wave is read by others of the same wave only: the LDS keeps a wave's
// accesses in order, so it is enough that the compiler does
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// How the lanes of a workgroup hold its targets: a lane each, several lanes a target, or (FP64) either
enum class Lanes { own, shared, any };

// One workgroup's part of the sum.  In mixed mode each form of the source loop is a body of its own: side by side in
// one, they keep a set of the FP64 accumulators in registers each (two targets per lane, LapPGradGrad 167 VGPRs,
// apart 128; PVelLaplacian 150, 123; traction 152, 125; PVelGrad 240, 172: a wave less per SIMD than the item
// kernels).  16,000 x 33,000: LapPGradGrad 516 -> 483 us, traction 543 -> 515, RegFTVelOmega 966 -> 861; 16,000 x
// 260,000 PVelGrad 8.6 -> 7.2 ms; 8192^2 Stokeslet 50 -> 49 us.
template <int UK, int PREC, int T, Lanes LANES>
__device__ __forceinline__ void direct_unit(const DirectArgs &a, double *smem) {
    using K = typename UkerOf<UK>::type;
    using L = DirectLds<K, PREC>;
    constexpr int KL = L::KL, KLP = L::KLP, KT = K::KT, KS = K::KS, KS1 = K::KS1, TT = kWave * T;
    constexpr int NA = AccCount<K, PREC>::value;
    constexpr int RUN = (PREC == 0) ? kSrcTile : MixedFlush<K>::value;
    // a run's first source on its own where the item kernels take it so: its products then start the
    // sums, which decides which of them is rounded (f/r + r b: one FMA of either product)
    constexpr bool PEEL = MixedPeel<K>::value && RUN == kMixedAccBlock;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int W = (int)blockDim.x >> 6;
    double *const sm = smem + wave * L::WORDS;
    float *const rows = reinterpret_cast<float *>(sm + 3 * kSrcTile);

    // this workgroup's targets, and how its lanes share them
    int ls = LANES == Lanes::own ? 0 : a.ls, tb = (int)blockIdx.x * a.unit, te = tb + min(a.unit, a.n_trg - tb);
    bool runs = PREC != 0; // lanes share a target by whole FP32 runs
    if (LANES == Lanes::own) {
        te = min(te, a.tail_begin);
    } else if (PREC != 0 && a.tail_ls > 0) {
        if ((int)blockIdx.x == (int)gridDim.x - 1) {
            ls = a.tail_ls;
            tb = a.tail_begin;
            te = a.n_trg;
            runs = false;
        } else {
            te = min(te, a.tail_begin);
        }
    }
    const int slots = kWave >> ls; // target slots of a wave
    const int sub = lane >> (6 - ls), slot = lane & (slots - 1);

    double tx[T], ty[T], tz[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const long long i = tb + min(slot + slots * t, te - tb - 1);
        tx[t] = a.tc.p[i * a.tc.s];
        ty[t] = a.tc.p[i * a.tc.s + a.tc.fs];
        tz[t] = a.tc.p[i * a.tc.s + 2 * a.tc.fs];
    }
    double acc[T][NA];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int k = 0; k < NA; ++k)
            acc[t][k] = 0.0;

    // runs start at g0, g0 + gs, ... of a tile; a lane takes sources j0, j0 + js, ... of each
    const int g0 = runs ? sub * RUN : 0, gs = runs ? RUN << ls : RUN;
    const int j0 = runs ? 0 : sub, js = runs ? 1 : 1 << ls;
    const int n_tiles = (a.n_src + kSrcTile - 1) / kSrcTile;
    const int st0 = (int)blockIdx.y * a.chunk_tiles, st1 = min(st0 + a.chunk_tiles, n_tiles);

    double c[3], vin[KS];
    auto fetch = [&](int st) {
        const long long s = min((long long)st * kSrcTile + lane, (long long)a.n_src - 1);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            c[d] = a.sc.p[s * a.sc.s + d * a.sc.fs];
#pragma unroll
        for (int k = 0; k < KS; ++k)
            vin[k] = (k < KS1) ? a.v1.p[s * a.v1.s + k * a.v1.fs] : a.v2.p[s * a.v2.s + (k - KS1) * a.v2.fs];
    };
    auto pair64 = [&](int j) {
        const double sx = sm[j], sy = sm[kSrcTile + j], sz = sm[2 * kSrcTile + j];
        double f[KL];
#pragma unroll
        for (int k = 0; k < KL; ++k)
            f[k] = sm[(3 + k) * kSrcTile + j];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            if constexpr (IsWallPair<K>::value)
                K::eval_wall(acc[t], tx[t] - sx, ty[t] - sy, tz[t] - sz, tz[t] + sz, tz[t], f);
            else
                eval_acc<K, PREC, true>(acc[t], tx[t] - sx, ty[t] - sy, tz[t] - sz, f);
        }
    };
    float part[T][KT];
    auto pair32 = [&](auto j) { // (generic: instantiated in mixed mode only)
        const double sx = sm[j], sy = sm[kSrcTile + j], sz = sm[2 * kSrcTile + j];
        float f[KL];
#pragma unroll
        for (int k = 0; k < KL; ++k)
            f[k] = rows[j * KLP + k];
#pragma unroll
        for (int t = 0; t < T; ++t)
            eval_pair<K, true>(part[t], (float)(tx[t] - sx), (float)(ty[t] - sy), (float)(tz[t] - sz), f);
    };
    auto clear_runs = [&]() {
        // a start the compiler knows folds into the first source's products (see PEEL); runs of several
        // blocks carry their sums from block to block in the item kernel, where none is known
        float z = -0.0f;
        if constexpr (RUN != kMixedAccBlock)
            asm volatile("" : "+v"(z));
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int k = 0; k < KT; ++k)
                part[t][k] = z;
    };
    auto flush_runs = [&]() {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int k = 0; k < KT; ++k)
                acc[t][k] += (double)part[t][k];
    };

    int st = st0 + wave;
    if (st < st1)
        fetch(st);
    for (; st < st1; st += W) {
        const int n = min(kSrcTile, a.n_src - st * kSrcTile);
        double vst[KL];
        stage_for<K, PREC>(vin, vst);
        if constexpr (IsWallPair<K>::value)
            K::stage_height(c[2], vst);
        wave_lds_fence(); // every lane has read the previous tile
#pragma unroll
        for (int d = 0; d < 3; ++d)
            sm[d * kSrcTile + lane] = c[d];
        if constexpr (PREC == 0) {
#pragma unroll
            for (int k = 0; k < KL; ++k)
                sm[(3 + k) * kSrcTile + lane] = vst[k];
        } else {
            float row[KLP];
#pragma unroll
            for (int k = 0; k < KLP; ++k)
                row[k] = (k < KL) ? (float)vst[k < KL ? k : 0] : 0.0f;
            float4 *dst = reinterpret_cast<float4 *>(rows + lane * KLP);
#pragma unroll
            for (int q = 0; q < KLP / 4; ++q)
                dst[q] = make_float4(row[4 * q], row[4 * q + 1], row[4 * q + 2], row[4 * q + 3]);
        }
        wave_lds_fence();
        if (st + W < st1)
            fetch(st + W);
        if constexpr (PREC == 0) {
            if (ls == 0 && n == kSrcTile) {
#pragma unroll 2
                for (int j = 0; j < kSrcTile; ++j)
                    pair64(j);
            } else {
#pragma unroll 2
                for (int j = j0; j < n; j += js)
                    pair64(j);
            }
        } else {
            if constexpr (LANES == Lanes::own) {
                for (int g = 0; g < n; g += RUN) {
                    const int e = min(g + RUN, n);
                    clear_runs();
                    int j = g;
                    if constexpr (PEEL)
                        pair32(j++);
#pragma unroll 2
                    for (; j < e; ++j)
                        pair32(j);
                    flush_runs();
                }
            } else {
                for (int g = g0; g < n; g += gs) {
                    const int e = min(g + RUN, n);
                    clear_runs();
                    int j = g + j0;
                    if constexpr (PEEL) {
                        if (j < e)
                            pair32(j);
                        j += js;
                    }
#pragma unroll 2
                    for (; j < e; j += js)
                        pair32(j);
                    flush_runs();
                }
            }
        }
    }

    if constexpr (PREC != 0) {
        // targets whose FP32 sums overflowed: this lane's pairs again in FP64 (p2p_redo.hpp)
        bool fin[T], all = true;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            fin[t] = true;
#pragma unroll
            for (int k = 0; k < KT; ++k)
                fin[t] = fin[t] && __builtin_isfinite(acc[t][k]);
            all = all && fin[t];
        }
        if (!__builtin_expect(__all(all), 1)) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                if (fin[t])
                    continue;
#pragma unroll
                for (int k = 0; k < KT; ++k)
                    acc[t][k] = 0.0;
                for (int q = st0 + wave; q < st1; q += W) {
                    const int n = min(kSrcTile, a.n_src - q * kSrcTile);
                    for (int g = g0; g < n; g += gs)
                        for (int j = g + j0; j < min(g + RUN, n); j += js) {
                            const long long s = (long long)q * kSrcTile + j;
                            double in[KS], v64[StagedCount<K, 0>::value];
#pragma unroll
                            for (int k = 0; k < KS; ++k)
                                in[k] = (k < KS1) ? a.v1.p[s * a.v1.s + k * a.v1.fs]
                                                  : a.v2.p[s * a.v2.s + (k - KS1) * a.v2.fs];
                            stage_for<K, 0>(in, v64);
                            eval_pair<K, true>(acc[t], tx[t] - a.sc.p[s * a.sc.s], ty[t] - a.sc.p[s * a.sc.s + a.sc.fs],
                                               tz[t] - a.sc.p[s * a.sc.s + 2 * a.sc.fs], v64);
                        }
                }
                // to the power of 2 the mixed form accumulates at (exact), which post_for expects
#pragma unroll
                for (int k = 0; k < KT; ++k)
                    if constexpr (PostsByPrecision<K>::value)
                        acc[t][k] *= post_for<K, 0>(k) / post_for<K, 1>(k);
            }
        }
    }

    // lanes of one target (they differ in the high lane bits), then the waves through LDS, KG
    // components at a time
    for (int off = slots; off < kWave; off <<= 1)
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int k = 0; k < NA; ++k)
                acc[t][k] += __shfl_xor(acc[t][k], off);
    double out[T][KT];
#pragma unroll
    for (int t = 0; t < T; ++t)
        finish_acc<K, PREC>(acc[t], out[t]);
    constexpr int KG0 = L::WORDS / TT, KG = KG0 < KT ? KG0 : KT;
    static_assert(KG >= 1, "the waves' sums fit the staging memory");
    const int lgu = 6 - ls + (T == 2 ? 1 : 0); // log2 of the unit's target slots
#pragma unroll
    for (int k0 = 0; k0 < KT; k0 += KG) {
        __syncthreads(); // every wave has left the memory to be written
        if (sub == 0) {
#pragma unroll
            for (int q = 0; q < KG; ++q)
                if (k0 + q < KT)
#pragma unroll
                    for (int t = 0; t < T; ++t)
                        smem[(wave * KG + q) * TT + slot + slots * t] = out[t][k0 + q < KT ? k0 + q : 0];
        }
        __syncthreads();
        const int nk = (KT - k0 < KG) ? KT - k0 : KG;
        // consecutive threads write consecutive doubles: of the (usually contiguous) output rows, or of a
        // component's partial sums
        for (int e = threadIdx.x; e < nk << lgu; e += blockDim.x) {
            const int i = a.two_phase ? e & ((1 << lgu) - 1) : e / nk;
            const int q = a.two_phase ? e >> lgu : e - nk * i, k = k0 + q;
            if (tb + i >= te)
                continue;
            double v = 0.0;
            for (int w = 0; w < W; ++w)
                v += smem[(w * KG + q) * TT + i];
            v *= post_for<K, PREC>(k);
            if (!a.two_phase) {
                const long long o = a.perm ? (long long)a.perm[tb + i] : tb + i;
                double *const p = a.out.p + o * a.out.s + k * a.out.fs;
                *p = a.store ? a.scale * v : *p + a.scale * v;
            } else {
                a.partial[((long long)blockIdx.y * KT + k) * a.n_trg + tb + i] = v;
            }
        }
    }
}

// waves per SIMD asked of the compiler: four where that takes a few registers off and no spills, so that two
// workgroups of eight waves share a CU
template <int UK, int PREC> struct DirectMinWaves {
    static constexpr int value = (UK == 11 && PREC == 0) ? 4 : 1;
};

template <int UK, int PREC, int T>
__global__ void __launch_bounds__(kWave *kDirectWaves)
__attribute__((amdgpu_waves_per_eu(DirectMinWaves<UK, PREC>::value))) p2p_direct_kernel(DirectArgs a) {
    extern __shared__ __align__(16) double smem[];
    if constexpr (PREC == 0)
        direct_unit<UK, PREC, T, Lanes::any>(a, smem);
    else if (a.ls == 0 && (a.tail_ls == 0 || blockIdx.x + 1 < gridDim.x))
        direct_unit<UK, PREC, T, Lanes::own>(a, smem);
    else
        direct_unit<UK, PREC, T, Lanes::shared>(a, smem);
}

template <int UK, int PREC, int T>
hipError_t launch_direct_one(const DirectArgs &a, const DirectLayout &l, hipStream_t s) {
    using L = DirectLds<typename UkerOf<UK>::type, PREC>;
    static_assert(L::WORDS * sizeof(double) * kDirectWaves <= 65536, "LDS of a workgroup");
    hipLaunchKernelGGL((p2p_direct_kernel<UK, PREC, T>), dim3(l.units, l.chunks), dim3(kWave * l.waves),
                       sizeof(double) * L::WORDS * l.waves, s, a);
    return hipGetLastError();
}

// FP64 runs direct_fp64_targets targets per lane; mixed mode one or two
template <int UK>
hipError_t launch_direct_uk(int prec, int T, const DirectArgs &a, const DirectLayout &l, hipStream_t s) {
    constexpr int T64 = direct_fp64_targets(UkerOf<UK>::type::KT);
    if (prec == 0)
        return T == T64 ? launch_direct_one<UK, 0, T64>(a, l, s) : hipErrorInvalidValue;
    return T == 2 ? launch_direct_one<UK, 1, 2>(a, l, s)
                  : (T == 1 ? launch_direct_one<UK, 1, 1>(a, l, s) : hipErrorInvalidValue);
}

} // namespace stkp2p
