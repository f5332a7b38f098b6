// What every tile kernel shares: which tile a workgroup computes, and buffer descriptors.
#pragma once
#include "common.hpp"

namespace maize {
namespace mt256 {

constexpr uint32_t OOB = 0x80000000u;   // OR-ed into an offset: >= num_records, reads as zero
typedef __attribute__((address_space(3))) char* lds_ptr;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

// Maps the linear workgroup id to a tile so that (a) the workgroups that land
// on one XCD (ids congruent mod 8) form a contiguous run of tiles and (b) a
// run covers a compact block of the tile grid, so an XCD's L2 sees few
// distinct A row panels and B column panels.
__device__ __forceinline__ uint32_t xcd_run(uint32_t pid, uint32_t total) {
    const uint32_t per = (total + 7u) / 8u;
    const uint32_t tall = (total % 8u) ? (total % 8u) : 8u;
    const uint32_t xcd = pid % 8u, local = pid / 8u;
    return xcd < tall ? xcd * per + local : tall * per + (xcd - tall) * (per - 1u) + local;
}
__device__ __forceinline__ void tile_of(uint32_t id, uint32_t tm, uint32_t tn, uint32_t* tile_m, uint32_t* tile_n) {
    // Sweeps of 4 tile rows: the 32 tiles an XCD works on at a time form a 4 x 8 block (12 operand panels through its
    // L2, the least a rectangle of 32 tiles needs).  Same-box A/B, 4096^3 / 8192^3 NT: 4 rows 87.6-88.2 / 661-662 us,
    // 8 rows (8 x 4, also 12 panels) 88.3-88.4 / 663 us, 2 or 16 rows (18 panels) 89.6-90.6 / 677-680 us.
    constexpr uint32_t GM = 4;
    const uint32_t group = id / (GM * tn);
    const uint32_t first = group * GM;
    const uint32_t gsz = (tm - first) < GM ? (tm - first) : GM;
    const uint32_t in = id % (GM * tn);
    *tile_m = first + in % gsz;
    *tile_n = in / gsz;
}

}  // namespace mt256
}  // namespace maize
