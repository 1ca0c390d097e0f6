// chain_step.hip -- the decoder step's row-wise stages in one launch
// (chain_step.h): embedding gather + input norm, residual add + post-attention
// norm, residual add + final norm (src/model/transformer_model.cpp:561-660).
//
// HBM-bound.  As separate launches the residual stream is written and read
// back between them: 11 D elements a token move (13 with the norms of the
// blocks' outputs: those re-read what they wrote).  Held in registers it is
// written once: 7 D (9 D).  One workgroup of 256 lanes per token, lane j on
// 16-byte vectors j, j + 256, ...; every load of the row and of the weights is
// issued first.  The three sums of squares share one barrier, since the second
// and third residual need no norm's result; with the blocks' outputs
// normalised first (DOUBLE) those two sums join the first barrier and the two
// residuals' take a second.
// Measured in place of the separate launches, a whole step of
// mi_decoder_chain_run: T = 6064, D = 3584 222 -> 189 us (this launch 51 us, 5.9
// TB/s), T = 1048, D = 4096 60.6 -> 50.7, T = 24, D = 2560, DOUBLE 31.1 -> 21.6
// (two launches in place of six).
#include "chain_step.h"

#include "mi_device.h"
#include "mi_host.h"

namespace mi {
namespace {

struct RowArgs {
    const int64_t* ids;
    const half_t* table;
    half_t *hidden, *normed, *post, *fin, *attn, *mlp;
    const half_t *w_in, *w_post, *w_fin, *w_attn, *w_mlp;
    int64_t D, vocab;
    float scale, eps, w_bias;
};

// Opaque copies of x.
template <int N>
__device__ __forceinline__ void launder(h8 (&x)[N]) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int j = 0; j < N; ++j) {
        u32x4 u = __builtin_bit_cast(u32x4, x[j]);
        asm volatile("" : "+v"(u));
        x[j] = __builtin_bit_cast(h8, u);
    }
}

template <int VPT, bool DOUBLE>
__global__ __launch_bounds__(256) void chain_rows_kernel(RowArgs r) {
    __shared__ float slots[(256 / kWave) * 3];
    __shared__ float slots2[(256 / kWave) * 2];
    const int64_t t = blockIdx.x;
    const int64_t nv = r.D >> 3;
    const int64_t row = t * r.D;
    const float Df = static_cast<float>(r.D);
    // loads: attn and mlp do not wait for the token id
    h8 a[VPT], m[VPT], h[VPT];
    int64_t at[VPT];
    bool ok[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int64_t c = threadIdx.x + j * 256;
        ok[j] = c < nv;
        at[j] = (ok[j] ? c : nv - 1) * 8;  // unconditional loads; idle lanes masked below
    }
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        a[j] = ld8_stream(r.attn + row + at[j]);
        m[j] = ld8_stream(r.mlp + row + at[j]);
    }
    const int64_t id = r.ids[t];
    const bool valid = id >= 0 && (r.vocab <= 0 || id < r.vocab);
    const half_t* src = r.table + (valid ? id : 0) * r.D;
#pragma unroll
    for (int j = 0; j < VPT; ++j) h[j] = ld8(src + at[j]);
    // the output norms' weights: with the rows where latency counts (DOUBLE has
    // two reductions in a row), else after the reduction, from the caches, for
    // the registers (82 -> 73: [1048, 4096] 43.9 -> 41.6 us up to the final norm)
    h8 wi[VPT], wp[VPT], wf[VPT];
    auto load_weights = [&] {
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            wi[j] = ld8(r.w_in + at[j]);
            wp[j] = ld8(r.w_post + at[j]);
            wf[j] = ld8(r.w_fin + at[j]);
        }
    };
    h8 wa[DOUBLE ? VPT : 1], wm[DOUBLE ? VPT : 1];
    if constexpr (DOUBLE) {
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            wa[j] = ld8(r.w_attn + at[j]);
            wm[j] = ld8(r.w_mlp + at[j]);
        }
        load_weights();
    }
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        if (!(valid && ok[j])) h[j] = h8(0);
        if (!ok[j]) {
            a[j] = h8(0);
            m[j] = h8(0);
        }
    }
    if (r.scale != 1.0f) {
#pragma unroll
        for (int j = 0; j < VPT; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) h[j][k] = to_half((float)h[j][k] * r.scale);
    }
    auto squares = [&](const h8(&x)[VPT]) {
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < VPT; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float f = (float)x[j][k];
                ss = fmaf(f, f, ss);
            }
        return ss;
    };
    // x += y, rounded to fp16 as the residual is stored
    auto add = [&](const h8(&x)[VPT], const h8(&y)[VPT], h8(&o)[VPT]) {
#pragma unroll
        for (int j = 0; j < VPT; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) o[j][k] = to_half((float)x[j][k] + (float)y[j][k]);
    };
    auto norm1 = [&](const h8& x, const h8& w, float rrms) {
        h8 o;
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = to_half((float)x[k] * rrms * ((float)w[k] + r.w_bias));
        return o;
    };
    h8 h1[VPT];
    float ss[3], rr[3];
    ss[0] = squares(h);
    if constexpr (!DOUBLE) {
        add(h, a, h1);
        add(h1, m, m);  // m: the second residual from here on
        ss[1] = squares(h1);
        ss[2] = squares(m);
        block_sum_n<3>(ss, slots);
#pragma unroll
        for (int i = 0; i < 3; ++i) rr[i] = rsqrtf(ss[i] / Df + r.eps);
    } else {
        ss[1] = squares(a);
        ss[2] = squares(m);
        block_sum_n<3>(ss, slots);
        rr[0] = rsqrtf(ss[0] / Df + r.eps);
        const float ra = rsqrtf(ss[1] / Df + r.eps), rm = rsqrtf(ss[2] / Df + r.eps);
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            a[j] = norm1(a[j], wa[j], ra);
            m[j] = norm1(m[j], wm[j], rm);
            if (ok[j]) {
                st8_stream(r.attn + row + at[j], a[j]);
                st8_stream(r.mlp + row + at[j], m[j]);
            } else {  // the weight a clamped lane read is another lane's
                a[j] = h8(0);
                m[j] = h8(0);
            }
        }
        add(h, a, h1);
        add(h1, m, m);
        float s2[2] = {squares(h1), squares(m)};
        block_sum_n<2>(s2, slots2);
        rr[1] = rsqrtf(s2[0] / Df + r.eps);
        rr[2] = rsqrtf(s2[1] / Df + r.eps);
    }
    // opaque copies, so that the fp32 values of the sums above are not kept
    // live beside the fp16 ones until here
    launder(h);
    launder(h1);
    launder(m);
    if constexpr (!DOUBLE) load_weights();
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        if (!ok[j]) continue;
        st8_stream(r.normed + row + at[j], norm1(h[j], wi[j], rr[0]));
        st8_stream(r.post + row + at[j], norm1(h1[j], wp[j], rr[1]));
        st8_stream(r.hidden + row + at[j], m[j]);
        st8_stream(r.fin + row + at[j], norm1(m[j], wf[j], rr[2]));
    }
}

}  // namespace

int chain_rows(const ChainRows& c, void* stream) {
    if (c.T <= 0 || c.T > kMaxGridX || c.D <= 0 || c.D % 8 != 0 || c.D > 4 * 2048)
        return MI_ERR_UNSUPPORTED;
    const bool dbl = c.w_attn != nullptr;
    const void* rows[] = {c.table, c.hidden, c.normed, c.post_normed, c.final_normed, c.attn, c.mlp,
                          c.w_in, c.w_post, c.w_final, c.w_attn, c.w_mlp};
    for (const void* p : rows)
        if (!aligned16(p)) return MI_ERR_UNSUPPORTED;
    RowArgs r;
    r.ids = c.ids;
    r.table = static_cast<const half_t*>(c.table);
    r.hidden = static_cast<half_t*>(c.hidden);
    r.normed = static_cast<half_t*>(c.normed);
    r.post = static_cast<half_t*>(c.post_normed);
    r.fin = static_cast<half_t*>(c.final_normed);
    r.attn = static_cast<half_t*>(c.attn);
    r.mlp = static_cast<half_t*>(c.mlp);
    r.w_in = static_cast<const half_t*>(c.w_in);
    r.w_post = static_cast<const half_t*>(c.w_post);
    r.w_fin = static_cast<const half_t*>(c.w_final);
    r.w_attn = static_cast<const half_t*>(c.w_attn);
    r.w_mlp = static_cast<const half_t*>(c.w_mlp);
    r.D = c.D;
    r.vocab = c.vocab;
    r.scale = c.scale;
    r.eps = c.eps;
    r.w_bias = c.add_one ? 1.0f : -0.0f;  // -0: w + bias == w, signed zeros kept
    const dim3 g(static_cast<unsigned>(c.T)), b(256);
    const hipStream_t s = as_stream(stream);
    switch (ceil_div(c.D / 8, 256)) {
#define MI_ROWS_CASE(V)                                            \
    case V:                                                        \
        if (dbl) chain_rows_kernel<V, true><<<g, b, 0, s>>>(r);    \
        else chain_rows_kernel<V, false><<<g, b, 0, s>>>(r);       \
        break;
        MI_ROWS_CASE(1)
        MI_ROWS_CASE(2)
        MI_ROWS_CASE(3)
        MI_ROWS_CASE(4)
#undef MI_ROWS_CASE
        default: return MI_ERR_UNSUPPORTED;
    }
    return launch_status();
}

}  // namespace mi
