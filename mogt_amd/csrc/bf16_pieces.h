// fp32 values as three bf16 pieces x = x1 + x2 + x3 (split_gemm.hip), written
// four consecutive elements at a time, the pieces `plane` elements apart.
#pragma once

#include "common.h"

namespace mogt {

// Each piece is the remainder rounded to nearest, so x1 + x2 + x3 == x while
// the last piece is a normal bf16 number.  Values that are not finite, or
// whose first piece would round up to infinity, have no remainder / a
// truncated first piece.
__device__ __forceinline__ void bf16_pieces(float x, bf16_t& p1, bf16_t& p2, bf16_t& p3) {
    const uint32_t u = __float_as_uint(x);
    p1 = f32_to_bf16(x);
    if ((u & 0x7f800000u) == 0x7f800000u) {   // inf, NaN
        p2 = p3 = 0;
        return;
    }
    if ((p1 & 0x7f80u) == 0x7f80u) p1 = static_cast<bf16_t>(u >> 16);
    const float r1 = x - bf16_to_f32(p1);
    p2 = f32_to_bf16(r1);
    p3 = f32_to_bf16(r1 - bf16_to_f32(p2));
}

__device__ __forceinline__ void store_pieces4(const float (&v)[4], bf16_t* dst, int64_t plane) {
    Pack<bf16_t, 4> a, b, c;
#pragma unroll
    for (int e = 0; e < 4; ++e) bf16_pieces(v[e], a.v[e], b.v[e], c.v[e]);
    *reinterpret_cast<Pack<bf16_t, 4>*>(dst) = a;
    *reinterpret_cast<Pack<bf16_t, 4>*>(dst + plane) = b;
    *reinterpret_cast<Pack<bf16_t, 4>*>(dst + 2 * plane) = c;
}

}  // namespace mogt
