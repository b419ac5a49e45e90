// wall.hip -- the no-slip wall image system of StkWallFMM (Lib/src/StkWallFMM.cpp:154-292) as one direct
// sum of source-and-image pairs (wall_pairs.hpp) in the direct kernel (p2p_direct.hpp).
//
// User coordinates: the wall is the plane z = 0; the image of a source at (x, y, z) is (x, y, -z)
// (the reference's setPoints, :40-80, shifts z to [0.5, 1) and places the image at 1 - z).
// Bound by FP64 issue: 65,536 sources and targets, FP64, constituent sums (7 and 10 direct sums, ordered
// points) -> source-and-image pairs: Stokes 24.3 -> 6.7 ms, RPY 49.9 -> 13.5 ms; 30,555 x 1,360 RPY 1.09 ->
// 0.15 ms.  The Stokes pair's 42 FP64 operations, two reciprocal square roots (16 cycles each) and two masks
// take about 6.2 ms at one operation per 4.2 cycles and SIMD.
#include <hip/hip_runtime.h>

#include "p2p_direct.hpp"
#include "p2p_internal.hpp"
#include "wall_pairs.hpp"

namespace stkp2p {

template <int UK, int T>
static hipError_t launch_wall_t(DirectArgs &a, const DirectCost &cost, int n_cu, hipStream_t s) {
    const DirectLayout l = direct_layout(0, T, cost, UkerOf<UK>::type::KT, kSrcTile, a.n_src, a.n_trg, n_cu);
    direct_args_layout(a, l);
    const hipError_t e = launch_direct_one<UK, 0, T>(a, l, s);
    return e != hipSuccess ? e : launch_direct_reduce(a, l.chunks, UkerOf<UK>::type::KT, s);
}

hipError_t launch_wall(bool rpy, DirectArgs a, int n_cu, hipStream_t s) {
    return rpy ? launch_wall_t<26, 1>(a, DirectCost{500.0, kDirectWaves, 2}, n_cu, s)
               : launch_wall_t<25, 2>(a, DirectCost{250.0, kDirectWaves, 2}, n_cu, s);
}

} // namespace stkp2p
