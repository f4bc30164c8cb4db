// wave_sum.hpp — sums of 64 values per lane over a wavefront (the blending gradients).
#pragma once

#include "common.hpp"

namespace tdgs {

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

// (x + y) after v_permlane32_swap / v_permlane16_swap of x and y: lanes whose bit 5 (resp. 4)
// is clear get x summed with its partner lane's x, the others y with the partner's y. The
// empty asm on the second result keeps the compiler from folding the two results of the
// swap into one (this toolchain compiles a plain r[0] + r[1] to r[0] + r[0]).
__device__ __forceinline__ float halve_swap32(float x, float y) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y),
                                                    false, false);
    uint32_t hi = r[1];
    asm volatile("" : "+v"(hi));
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ float halve_swap16(float x, float y) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y),
                                                    false, false);
    uint32_t hi = r[1];
    asm volatile("" : "+v"(hi));
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, hi);
}

// x[i] = (x[i] + y[i]) halved at lane distance 8 or 4 (D): lanes whose bit D is clear get x[i] summed
// with lane ^ D's x[i], the others y[i] with lane ^ D's y[i]. A DPP add writes only the lanes of the
// 4-lane banks its bank_mask names and leaves the others, so each half is one add with the rotation
// that reaches its partner (row_ror:n reads lane - n of the row) and no select: 8.4 issue cycles a
// pair, against 10.5 for two selects and a DPP add and 11 for a permlane swap and an add (measured
// at eight wavefronts per SIMD). A DPP read, or a permlane swap, needs two wait states after the
// write of its register, which the compiler does not see inside the block: hence the s_nop around it.
// (x early-clobbered: it is written before y is read, and would share y's register where the
// compiler knows the two to hold one value.)
template <int D>
__device__ __forceinline__ void halve_dpp(float (&x)[8], const float (&y)[8]) {
#define TDGS_HALF(I, CTRL, BANKS) "v_add_f32_dpp %" #I ", %" #I ", %" #I " " CTRL " row_mask:0xf bank_mask:" BANKS "\n"
#define TDGS_OTHER(I, J, CTRL, BANKS) "v_add_f32_dpp %" #I ", %" #J ", %" #J " " CTRL " row_mask:0xf bank_mask:" BANKS "\n"
#define TDGS_HALVE(CX, BX, CY, BY)                                                                          \
    asm("s_nop 1\n" TDGS_HALF(0, CX, BX) TDGS_HALF(1, CX, BX) TDGS_HALF(2, CX, BX) TDGS_HALF(3, CX, BX)       \
            TDGS_HALF(4, CX, BX) TDGS_HALF(5, CX, BX) TDGS_HALF(6, CX, BX) TDGS_HALF(7, CX, BX)               \
                TDGS_OTHER(0, 8, CY, BY) TDGS_OTHER(1, 9, CY, BY) TDGS_OTHER(2, 10, CY, BY)                   \
                    TDGS_OTHER(3, 11, CY, BY) TDGS_OTHER(4, 12, CY, BY) TDGS_OTHER(5, 13, CY, BY)             \
                        TDGS_OTHER(6, 14, CY, BY) TDGS_OTHER(7, 15, CY, BY) "s_nop 1"                        \
        : "+&v"(x[0]), "+&v"(x[1]), "+&v"(x[2]), "+&v"(x[3]), "+&v"(x[4]), "+&v"(x[5]), "+&v"(x[6]), "+&v"(x[7])      \
        : "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(y[4]), "v"(y[5]), "v"(y[6]), "v"(y[7]))
    static_assert(D == 8 || D == 4, "a distance inside a row, of whole banks");
    if constexpr (D == 8) TDGS_HALVE("row_ror:8", "0x3", "row_ror:8", "0xc");
    else TDGS_HALVE("row_ror:12", "0x5", "row_ror:4", "0xa");
#undef TDGS_HALVE
#undef TDGS_OTHER
#undef TDGS_HALF
}

// Sums 64 values per lane over the wavefront by recursive halving: at the step of lane
// distance D each lane keeps the half of its values whose index has the lane's bit D,
// adds the partner lane's copy of that half and passes on the other half. Six steps, the
// cheapest on the most values (8 and 4 by masked DPP adds: 48 of the 63 sums; then 32 and 16 by
// permlane swaps, 2 and 1 by selects and DPP), leave in lane l the wavefront sum of v[l]. v is
// destroyed.
__device__ __forceinline__ float wave_transpose_sum64(float (&v)[64]) {
    const int lane = __lane_id();
    // value index i = 16 r + 8 d3 + 4 d2 + c: the pairs (i, i + 8), eight of them at a time
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float x[8], y[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            x[k] = v[16 * r + k];
            y[k] = v[16 * r + 8 + k];
        }
        halve_dpp<8>(x, y);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[16 * r + k] = x[k];
    }
    // the pairs (i, i + 4) of two r at a time
#pragma unroll
    for (int r = 0; r < 4; r += 2) {
        float x[8], y[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            x[k] = v[16 * (r + k / 4) + k % 4];
            y[k] = v[16 * (r + k / 4) + 4 + k % 4];
        }
        halve_dpp<4>(x, y);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[16 * (r + k / 4) + k % 4] = x[k];
    }
    float w[8];   // w[4 h + c]: index 16 h + c, h = 0, 1 (after the distance 32)
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = halve_swap32(v[16 * (k / 4) + k % 4], v[16 * (k / 4) + 32 + k % 4]);
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = halve_swap16(w[k], w[k + 4]);
    const bool b1 = lane & 2, b0 = lane & 1;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float send = b1 ? w[i] : w[i + 2], keep = b1 ? w[i + 2] : w[i];
        w[i] = keep + dpp_f32<0x4e>(send);                        // quad_perm [2,3,0,1]
    }
    const float send = b0 ? w[0] : w[1], keep = b0 ? w[1] : w[0];
    return keep + dpp_f32<0xb1>(send);                            // quad_perm [1,0,3,2]
}

}  // namespace tdgs
