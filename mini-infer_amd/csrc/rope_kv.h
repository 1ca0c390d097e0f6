// rope_kv.h -- RoPE of a token's Q and K in place, with K's rotated rows and
// V's rows also written into the paged KV cache: one workgroup of 256 lanes
// per token.  The body of rope_kv_scatter_kernel (rope.hip) and of the one-launch
// decoder step (chain_step.hip).
#pragma once

#include "mi_kernels.h"
#include "rope_math.h"

namespace mi {

constexpr int kMaxKvSegs = 8;
struct KvSegs {
    int n;
    int64_t off[kMaxKvSegs], B[kMaxKvSegs], S[kMaxKvSegs], mb[kMaxKvSegs];
    const int* bt[kMaxKvSegs];
    const int* sl[kMaxKvSegs];
    const int* sp[kMaxKvSegs];
};

// Everything a launch needs but the inverse frequencies.
struct RopeKv {
    half_t *q, *k;
    const half_t* v;
    int Hq, Hkv, hd;
    const int64_t* positions;
    const half_t *bq, *bk, *bv, *wq, *wk;
    float eps, w_bias;
    half_t *k_cache, *v_cache;
    int64_t layer, num_blocks, bs;
    KvSegs sg;
};

// Checks a call of the one-launch attention pre-processing and fills its device
// arguments (rope.hip); slots: the larger of a token's (head, slice) units and its
// V vectors.  MI_OK, or the entry points' status for the call.
int rope_kv_plan(void* q, void* k, const void* v, const void* q_bias, const void* k_bias,
                 const void* v_bias, const void* q_weight, const void* k_weight, float eps,
                 int add_one, const int64_t* positions, const float* inv_freq_host, int64_t T,
                 int64_t Hq, int64_t Hkv, int64_t head_dim, void* k_cache, void* v_cache,
                 int64_t layer, int64_t num_blocks, int64_t block_size,
                 const mi_kv_segment* segments, int num_segments, bool wide, RopeKv& a,
                 int64_t& slots);

// The token's cache row, in elements from the cache's start (-1: not
// scattered), as launch_paged_kv_scatter places it
// (src/kernels/model_utils_kernel.cu:108-164); token indices and segment sizes
// fit 32 bits (T <= kMaxGridX).
__device__ __forceinline__ int64_t kv_row(const RopeKv& a, int64_t tok, int64_t hd) {
    const KvSegs& sg = a.sg;
    const int itok = static_cast<int>(tok);
    for (int i = 0; i < sg.n; ++i) {
        const int r = itok - static_cast<int>(sg.off[i]);
        const int S = static_cast<int>(sg.S[i]);
        if (r < 0 || r >= static_cast<int>(sg.B[i]) * S) continue;
        const int b = static_cast<int>(static_cast<uint32_t>(r) / static_cast<uint32_t>(S));
        const int64_t pos = static_cast<int64_t>(sg.sp[i][b]) + (r - b * S);
        const int len = sg.sl[i][b];
        if (pos < 0 || pos >= len) break;
        // 0 <= pos < len and bs < 2^31: 32-bit division
        const int blk = static_cast<int>(static_cast<uint32_t>(pos) / static_cast<uint32_t>(a.bs));
        if (blk >= sg.mb[i]) break;
        const int64_t phys = sg.bt[i][b * sg.mb[i] + blk];
        if (phys >= 0 && phys < a.num_blocks)
            return ((a.layer * a.num_blocks + phys) * a.Hkv * a.bs + (pos - blk * a.bs)) * hd;
        break;
    }
    return -1;
}

// Lane j takes the (head, slice) units j, j + 256, ... (P of them, P * 256 >=
// units) of the token -- x[i..i+7] and x[h+i..h+i+7] of a head -- and V's 16-byte
// vectors j, j + 256, ...; every load is issued before the cos/sin row is built
// (once per token, in LDS), and the cache slot's dependent scalar lookups overlap
// them.  BIAS: the projection bias is added first, rounded to fp16 as the
// reference's launch_add_bias stores it.  NORM: the per-head Q/K RMSNorm first --
// the CPH = hd / 16 lanes of a head sum their squares by DPP, the normalised
// value is rounded to fp16 where the reference stores it, and the rotation takes
// it from registers.  CPH at compile time (shifts for the lane -> (head, slice)
// split: 0.3-0.4 us less than CPH = 0 at Qwen2.5's shapes, T = 6064); CPH = 0:
// head_dim known at run time (no norm).  Rows are written through to
// memory ("nt sc1") where their pieces are whole lines.
// P = 2 (32 + 8 heads of 128, 320 units, T = 1048 in two segments): 13.5 us with the
// gather before it, against 19.7 for RoPE and two scatters after it.
// LPT: lanes per token -- 256, or 64 or 128 for tokens of so few units, so that a
// workgroup takes four or two (14 + 2 heads of 64, 64 units, T = 4096: 8.4 -> 5.9 us);
// cs: the token's 2 * kMaxHalf floats.  live = false: a token past the last,
// which touches no memory but takes the barrier.
template <bool BIAS, bool NORM, int CPH, int P, int LPT = 256>
__device__ __forceinline__ void rope_kv_token(const RopeKv& a, const float* inv, int64_t tok,
                                              bool live, float* cs) {
    static_assert(LPT == 256 || P == 1, "several tokens per workgroup take one slot per lane");
    static_assert(!(BIAS && NORM), "no model adds a QKV bias before a Q/K norm");
    static_assert(!NORM || (CPH >= 1 && CPH <= 32), "the norm needs head_dim / 16 at compile time");
    // written through (rope_math.h); with several units per lane the stores' wait
    // states would queue behind one another (T = 1, 320 units: 3.2 -> 2.7 us)
    constexpr bool WT = (NORM ? MI_WT_QKNR : MI_WT_ROPE) && whole_lines<CPH>() && P == 1;
    const int half = CPH ? CPH * 8 : a.hd >> 1;
    const int cph = CPH ? CPH : half >> 3;  // 16-byte slices per half head
    const int Hq = a.Hq, Hkv = a.Hkv;
    const int units = live ? (Hq + Hkv) * cph : 0;
    const int vecs = live && a.sg.n > 0 ? Hkv * (half >> 2) : 0;  // no segment: V not read
    const int tid = threadIdx.x & (LPT - 1);

    h8 x1[P], x2[P], b1[P], b2[P];
    half_t* hp[P];
    int h[P], c[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int u = tid + p * 256;
        x1[p] = x2[p] = b1[p] = b2[p] = h8(0);
        hp[p] = nullptr;
        h[p] = c[p] = 0;
        if (u < units) {
            if constexpr (CPH != 0) {
                h[p] = u / CPH;
                c[p] = u & (CPH - 1);
            } else {
                h[p] = small_div(u, 1.0f / static_cast<float>(cph));  // units < 2^22: exact
                c[p] = u - h[p] * cph;
            }
            const bool is_q = h[p] < Hq;
            hp[p] = is_q ? a.q + (tok * Hq + h[p]) * (2 * half)
                         : a.k + (tok * Hkv + (h[p] - Hq)) * (2 * half);
            x1[p] = ld8_stream(hp[p] + c[p] * 8);
            x2[p] = ld8_stream(hp[p] + half + c[p] * 8);
            if constexpr (BIAS) {  // a few KB every token re-reads: plain loads
                const half_t* bp = is_q ? a.bq + h[p] * (2 * half) : a.bk + (h[p] - Hq) * (2 * half);
                b1[p] = ld8(bp + c[p] * 8);
                b2[p] = ld8(bp + half + c[p] * 8);
            }
            if constexpr (NORM) {  // the norm weights [hd], as the biases
                const half_t* wp = is_q ? a.wq : a.wk;
                b1[p] = ld8(wp + c[p] * 8);
                b2[p] = ld8(wp + half + c[p] * 8);
            }
        }
    }
    h8 vv[P], vb[BIAS ? P : 1];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int vj = tid + p * 256;
        vv[p] = h8(0);
        if (BIAS) vb[BIAS ? p : 0] = h8(0);
        if (vj < vecs) {
            vv[p] = ld8_stream(a.v + tok * Hkv * (2 * half) + vj * 8);
            if constexpr (BIAS) vb[p] = ld8(a.bv + vj * 8);
        }
    }
    const float fpos = live ? static_cast<float>(a.positions[tok]) : 0.0f;
    const int64_t dst_base = live ? kv_row(a, tok, 2 * half) : -1;
    if (tid < half) {
        half_t hc, hs;
        cos_sin_half(fpos * inv[tid], hc, hs);
        const int li = quad_split(tid, half);
        cs[li] = (float)hc;
        cs[kMaxHalf + li] = (float)hs;
    }
    __syncthreads();

#pragma unroll
    for (int p = 0; p < P; ++p) {
        float rrms = 1.0f;
        if constexpr (NORM) {  // every lane takes part in the DPP sum (idle lanes add zeros)
            float ss = pair_sumsq(x1[p], x2[p]);
            ss = group_sum<CPH ? CPH : 1>(ss);
            rrms = rsqrtf(ss / static_cast<float>(CPH * 16) + a.eps);
        }
        if (tid + p * 256 >= units) continue;
        // quad_split layout: entries 0-3 of slice c at c*4, 4-7 at half/2 + c*4
        typedef float f4 __attribute__((ext_vector_type(4)));
        const f4 c_lo = *reinterpret_cast<const f4*>(&cs[c[p] * 4]);
        const f4 c_hi = *reinterpret_cast<const f4*>(&cs[(half >> 1) + c[p] * 4]);
        const f4 s_lo = *reinterpret_cast<const f4*>(&cs[kMaxHalf + c[p] * 4]);
        const f4 s_hi = *reinterpret_cast<const f4*>(&cs[kMaxHalf + (half >> 1) + c[p] * 4]);
        h8 y1, y2;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float cv = e < 4 ? c_lo[e & 3] : c_hi[e & 3];
            const float sv = e < 4 ? s_lo[e & 3] : s_hi[e & 3];
            float xa = (float)x1[p][e], xb = (float)x2[p][e];
            if constexpr (BIAS) {
                xa = (float)to_half(xa + (float)b1[p][e]);
                xb = (float)to_half(xb + (float)b2[p][e]);
            }
            if constexpr (NORM) {  // the normalised value as the reference stores it (fp16)
                xa = (float)to_half(xa * rrms * ((float)b1[p][e] + a.w_bias));
                xb = (float)to_half(xb * rrms * ((float)b2[p][e] + a.w_bias));
            }
            y1[e] = to_half(fp32_rounded(xa * cv - xb * sv));
            y2[e] = to_half(fp32_rounded(xb * cv + xa * sv));
        }
        st8_out<WT>(hp[p] + c[p] * 8, y1);
        st8_out<WT>(hp[p] + half + c[p] * 8, y2);
        if (h[p] >= Hq && dst_base >= 0) {
            half_t* kd = a.k_cache + dst_base + static_cast<int64_t>(h[p] - Hq) * a.bs * (2 * half);
            st8_out<WT>(kd + c[p] * 8, y1);
            st8_out<WT>(kd + half + c[p] * 8, y2);
        }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int vj = tid + p * 256;
        if (vj < vecs && dst_base >= 0) {
            if constexpr (BIAS) {
#pragma unroll
                for (int e = 0; e < 8; ++e) vv[p][e] = to_half((float)vv[p][e] + (float)vb[p][e]);
            }
            const int per_head = half >> 2;
            int vh;
            if constexpr (CPH != 0)
                vh = vj / (CPH * 2);
            else
                vh = small_div(vj, 1.0f / static_cast<float>(per_head));
            const int vd = (vj - vh * per_head) * 8;
            st8_out<WT>(a.v_cache + dst_base + static_cast<int64_t>(vh) * a.bs * (2 * half) + vd, vv[p]);
        }
    }
}

// The tokens of workgroup `block` (256 / LPT of them); cs: 256 / LPT * 2 * kMaxHalf
// floats.
template <bool BIAS, bool NORM, int CPH, int P, int LPT>
__device__ __forceinline__ void rope_kv_block(const RopeKv& a, const float* inv, int64_t block,
                                              int64_t T, float* cs) {
    if constexpr (LPT == 256) {
        rope_kv_token<BIAS, NORM, CPH, P>(a, inv, block, true, cs);
    } else {
        const int g = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / LPT);
        const int64_t tok = block * (256 / LPT) + g;
        rope_kv_token<BIAS, NORM, CPH, P, LPT>(a, inv, tok, tok < T, cs + g * 2 * kMaxHalf);
    }
}

}  // namespace mi
