// dhip_txrec.hpp -- the 16-byte record of the mixed-precision PCG's tagged exchange: what a row publishes
// in one generation (r, w, s as float bits) and when a reader may take it.  Only a 64-bit half of a 128-bit access is
// single-copy atomic, so each half carries the generation: 16 bits of it, as w is split over the
// halves and leaves 16 in each.
//
//   {r, w_lo16 | gen16 << 16, s, w_hi16 | gen16 << 16}
//
// 16 bits tell the generations apart that a slot can hold.  Slots are double buffered by the generation's parity and
// every row is written and read in every generation, so a reader that waits for generation g finds halves of g - 2
// (which it took before) or of g; before generations 1 and 2 the slots are cleared, and 0 is neither's tag.
#pragma once

#include <cstdint>

namespace dhip {

template <class R>
__host__ __device__ __forceinline__ R txm_pack(uint32_t r, uint32_t w, uint32_t s, uint32_t g) {
    return R{r, (w & 0xffffu) | g << 16, s, (w >> 16) | g << 16};
}

template <class R>
__host__ __device__ __forceinline__ bool txm_ready(const R &v, uint32_t g) {
    return (((v[1] ^ (g << 16)) | (v[3] ^ (g << 16))) >> 16) == 0;
}

// the bits of w (r and s are words 0 and 2)
template <class R>
__host__ __device__ __forceinline__ uint32_t txm_w(const R &v) {
    return (v[1] & 0xffffu) | v[3] << 16;
}

}  // namespace dhip
