// fp32 activations split exactly into three bf16 parts, as "planes" in the
// order the W8 MFMA GEMM (gemm_w8f.hip) reads them, and the helpers with which
// the kernels that produce activations write them.
//
// x = hi + mid + lo: the top, middle and low 8 significand bits (each
// subtraction is exact by Sterbenz's lemma and the last remainder has at most 8
// significant bits), so a part times an int8 weight is exact in fp32.
//
// Layout: [row block of 32][K / 16][part][512 values]: the 32 x 16 fragment of
// one MFMA operand, 1 KB, lane l's 8 values (row l % 32, K values 8 (l / 32) ..)
// at byte 16 l. The parts of one fragment follow each other.
#pragma once

#include "pio_common.hpp"

namespace pio {

constexpr int WF_FRAG = 3 * 1024;   // bytes of a fragment's three parts

inline size_t wf_planes_bytes(int64_t M, int64_t K) { return (size_t)((M + 31) / 32 * 32 * K * 6); }

// Byte of (row m, k) in the hi plane; the mid and lo parts 1024 and 2048 further on.
__device__ __forceinline__ int64_t wf_plane_at(int m, int k, int K) {
    return ((int64_t)(m >> 5) * (K >> 4) + (k >> 4)) * WF_FRAG + ((((k >> 3) & 1) * 32 + (m & 31)) << 4) + ((k & 7) << 1);
}

// The parts of two values, packed (the first in the low half).
__device__ __forceinline__ void wf_split3_pair(float a, float c, int& h, int& m, int& l) {
    const float a1 = a - __uint_as_float(__float_as_uint(a) & 0xFFFF0000u);
    const float c1 = c - __uint_as_float(__float_as_uint(c) & 0xFFFF0000u);
    const float a2 = a1 - __uint_as_float(__float_as_uint(a1) & 0xFFFF0000u);
    const float c2 = c1 - __uint_as_float(__float_as_uint(c1) & 0xFFFF0000u);
    h = (int)__builtin_amdgcn_perm(__float_as_uint(c), __float_as_uint(a), 0x07060302u);
    m = (int)__builtin_amdgcn_perm(__float_as_uint(c1), __float_as_uint(a1), 0x07060302u);
    l = (int)__builtin_amdgcn_perm(__float_as_uint(c2), __float_as_uint(a2), 0x07060302u);
}

// SwiGLU of the prompt's MLP.
__device__ __forceinline__ float wf_silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// Values k .. k + 3 of row m (k % 4 == 0) into the planes of a [..][K] matrix.
__device__ __forceinline__ void wf_put4(int8_t* planes, int m, int k, int K, float4 v) {
    int2 h, d, l;
    wf_split3_pair(v.x, v.y, h.x, d.x, l.x);
    wf_split3_pair(v.z, v.w, h.y, d.y, l.y);
    int8_t* p = planes + wf_plane_at(m, k, K);
    *(int2*)p = h;
    *(int2*)(p + 1024) = d;
    *(int2*)(p + 2048) = l;
}
__device__ __forceinline__ void wf_put2(int8_t* planes, int m, int k, int K, float a, float b) {
    int h, d, l;
    wf_split3_pair(a, b, h, d, l);
    int8_t* p = planes + wf_plane_at(m, k, K);
    *(int*)p = h;
    *(int*)(p + 1024) = d;
    *(int*)(p + 2048) = l;
}

// Row of block b when one block writes one row's planes: blocks run on XCD
// b % 8, and the 8 rows whose 16-byte pieces share a 128-byte line go to one
// XCD, so that its L2 completes the line. Grid: wf_row_blocks(M); rows >= M idle.
__device__ __forceinline__ int wf_row_of_block(int b) { return 64 * (b >> 6) + 8 * (b & 7) + ((b >> 3) & 7); }
inline int wf_row_blocks(int M) { return (M + 63) / 64 * 64; }

}  // namespace pio
