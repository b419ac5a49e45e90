// p2p_mixed.hpp -- how the mixed-mode kernels group the sources of a target's FP32 partial sums.
#pragma once

#include "p2p_internal.hpp"

namespace stkp2p {

// sources per FP32 partial sum in mixed mode (a multiple of kMixedAccBlock that divides the 64-source
// tile): MIXED_ACC_SOURCES of the micro-kernel, else kMixedAccBlock.  The item kernels choose their path
// (masked / clear / far) per kMixedAccBlock sources all the same.
template <class K, class = void> struct MixedFlush { static constexpr int value = kMixedAccBlock; };
template <class K> struct MixedFlush<K, decltype((void)K::MIXED_ACC_SOURCES)> {
    static constexpr int value = K::MIXED_ACC_SOURCES;
    static_assert(value % kMixedAccBlock == 0 && kSrcTile % value == 0, "MIXED_ACC_SOURCES");
};

// the mixed-mode source loop takes each block's first source on its own (MIXED_PEEL of the
// micro-kernel, else not): measured on MI355X, same box, twice each: the fused PVel U-list 7.870 ->
// 7.830 ms, the RPY U-list 39.98 -> 39.78 ms, the single-layer PVel FMM lists 6.84 -> 6.80 ms (X
// list -1.3 %, W list +0.4 %), but the ordered Stokeslet instances 34.54 -> 34.86 ms
template <class K, class = void> struct MixedPeel { static constexpr bool value = false; };
template <class K> struct MixedPeel<K, decltype((void)K::MIXED_PEEL)> {
    static constexpr bool value = K::MIXED_PEEL;
};

} // namespace stkp2p
