// quad16.hpp - lane-quad transposes of 16-bit values for GEMM epilogues that store whole row pieces
// from the MFMA's column-per-lane accumulators.
#pragma once

#include "common.hpp"

namespace cb {

// 16-bit 4 x 4 transpose across the lane quad (qi = lane % 4): on entry the lane holds rows
// 0..3 of its column as p01 = rows 0, 1 and p23 = rows 2, 3; on exit d0, d1 hold row qi, columns
// 0..3 of the quad.  Step 1 trades 2-row halves with lane qi ^ 2, step 2 single values with qi ^ 1;
// the lane-dependent choices are selects and per-lane byte selectors of v_perm_b32 (sel_*), not
// branches.
struct Quad16Sel {
    bool hi2;
    u32 s_send, s_d0, s_d1;
};

__device__ __forceinline__ Quad16Sel quad16_sel(const int qi)
{
    const bool odd = qi & 1;
    Quad16Sel q;
    q.hi2 = qi & 2;
    q.s_send = odd ? 0x05040100u : 0x07060302u;  // perm(second, first): lo / hi halves of both
    q.s_d0 = odd ? 0x03020504u : 0x05040100u;    // perm(r2, first)
    q.s_d1 = odd ? 0x03020706u : 0x07060100u;    // perm(r2, second)
    return q;
}

__device__ __forceinline__ void quad_transpose16(const u32 p01, const u32 p23, const Quad16Sel& q, u32& d0, u32& d1)
{
    const u32 recv = (u32)__builtin_amdgcn_mov_dpp((int)(q.hi2 ? p01 : p23), 0x4E, 0xF, 0xF, false);
    // first: column qi & 1, second: column (qi & 1) + 2, both for the lane pair's two rows
    const u32 first = q.hi2 ? recv : p01, second = q.hi2 ? p23 : recv;
    const u32 r2 = (u32)__builtin_amdgcn_mov_dpp((int)__builtin_amdgcn_perm(second, first, q.s_send), 0xB1, 0xF,
                                                     0xF, false);
    d0 = __builtin_amdgcn_perm(r2, first, q.s_d0);
    d1 = __builtin_amdgcn_perm(r2, second, q.s_d1);
}

// Two values rounded to bf16 (round to nearest even) in one dword, the first in the low half.
__device__ __forceinline__ u32 pack_bf16x2(const float a, const float b)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(u32, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

}  // namespace cb
