// rope_math.h -- what the RoPE kernels share: the inverse frequencies as a
// kernel argument, fp16 cos/sin of an fp32 angle, the LDS layout of a token's
// cos/sin row, and their store form.
#pragma once

#include "mi_device.h"
#include "rope_sincos.h"

// Stores of the in-place RoPE and fused Q/K-norm + RoPE kernels: write-through
// ("nt sc1", st8_stream_wt) measured 1-3 points faster than plain non-temporal
// where each store instruction's pieces are whole 128-byte lines -- the halves of
// heads of 128, 256, 512 -- and far slower where they are not, each line then being
// written through in parts: T = 4096 in place, 32 + 32 heads of 80 33.3 -> 20.0 us
// without it, 32 + 8 of 80 20.8 -> 12.6, 14 + 2 of 64 with a bias 6.3 -> 4.9.
#ifndef MI_WT_ROPE
#define MI_WT_ROPE 1
#endif
#ifndef MI_WT_QKNR
#define MI_WT_QKNR 1
#endif

namespace mi {

constexpr int kMaxHalf = 256;  // head_dim <= 512

// Whether the halves of a head of 16 * CPH elements are whole 128-byte lines
// (CPH = 0, any other head_dim: no).
template <int CPH>
constexpr bool whole_lines() { return CPH > 0 && CPH % 8 == 0; }

// LDS position of element i of a half-row of n entries (n a multiple of 8),
// for lanes that each read the 8 entries c*8 .. c*8+7 as two 16-byte LDS
// reads: entries 0-3 of every lane's group sit together in the first n/2
// slots and entries 4-7 in the second, so lane c reads slots 4c .. 4c+3 and
// n/2 + 4c .. n/2 + 4c+3.  Eight consecutive lanes then cover 32 distinct
// banks per read; with the plain layout (lane c at 8c) lanes c and c+4 fall
// on the same banks and every read took a second pass (rocprof
// LdsBankConflict 0.97 conflicts per access).
__device__ __forceinline__ int quad_split(int i, int n) {
    return ((i & 4) ? (n >> 1) : 0) + ((i >> 3) << 2) + (i & 3);
}

// Host-computed inverse frequencies travel by value in the kernel arguments, as
// many as the head has, or as the next of a few sizes: a kernel with 1 KB of
// arguments took the host 4.3 us to launch, one with few 2.9.
template <int NF>
struct InvFreqN {
    float v[NF];
};

// fp16 cos/sin of an fp32 angle, equal to half(RN32(exact)) (see file header).
// |ang| <= 2^20: the fp32 Cody-Waite form, re-evaluated in fp64 when a value
// lies within rope_guard_width of an fp16 rounding boundary; larger angles
// (positions beyond 2^20 / inv_freq) go straight to the fp64 form
// (rope_sincos_any: Cody-Waite to 2^24, Payne-Hanek above), which covers
// every fp32 angle -- so every int64 position -- with no range limit.
__device__ __forceinline__ bool near_half_boundary(float v) {
    const float d = rope_guard_width(v);
    return to_half(v - d) != to_half(v + d);
}

__device__ __forceinline__ void cos_sin_half(float ang, half_t& hc, half_t& hs) {
    float s, c;
    rope_sincos_f32(ang, &s, &c);
    if (!rope_sincos_f32_ok(ang) || near_half_boundary(c) || near_half_boundary(s)) {
        double sd, cd;
        rope_sincos_any(ang, &sd, &cd);
        c = static_cast<float>(cd);
        s = static_cast<float>(sd);
    }
    hc = to_half(c);
    hs = to_half(s);
}

}  // namespace mi
