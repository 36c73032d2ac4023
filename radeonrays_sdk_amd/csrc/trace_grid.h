// trace_grid.h — grid and piece sizes of a query, as plain arithmetic (no
// HIP), so that the host test compiles the same rules.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace rr {

constexpr uint32_t kTraceBlock = 256;  // threads of a traversal workgroup

// Rays per piece for n rays over `blocks` workgroups: the tuned value, cut to
// half an even share (a multiple of 32, rounded down), so that waves whose
// rays end early find more to take (524,288 rays of a camera, closest hit:
// 65,536-triangle soup 331 -> 235 us, 1M-triangle terrain 253 -> 211).
// Rounded up, a wave started with up to three quarters of its share just
// above a multiple: 524,289 rays inside a soup of 4,096 large triangles 836
// us against 684 (start of the range: 524,288 rays 688), inside the
// 65,536-triangle soup 413 against 347, 1.1M rays there 727 against 631.
// The cut ends at 64: smaller pieces cost more in atomics than they balance
// (480,000 rays in pieces of 32: 3,000-triangle soup, camera 108 -> 125 us;
// and 4M rays there in pieces of 64 330 -> 374).  With fewer rays than that
// for each wave, all of them (32 or 64).
inline uint32_t PieceRays(uint64_t n, uint32_t blocks, uint32_t tuned) {
    const uint64_t waves = (uint64_t)blocks * (kTraceBlock / 64);
    const uint64_t half = n / (2 * waves) / 32 * 32;
    const uint64_t least = std::min<uint64_t>(64, ((n + waves - 1) / waves + 31) / 32 * 32);
    return (uint32_t)std::min<uint64_t>(tuned, std::max(half, least));
}

}  // namespace rr
