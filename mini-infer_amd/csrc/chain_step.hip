// chain_step.hip -- the decoder step's row-wise stages in one launch
// (chain_step.h): embedding gather + input norm, residual add + post-attention
// norm, residual add + final norm (src/model/transformer_model.cpp:561-660).
//
// HBM-bound.  As separate launches the residual stream is written and read
// back between them: 11 D elements a token move (13 with the norms of the
// blocks' outputs: those re-read what they wrote).  Held in registers it is
// written once: 7 D (9 D).  One workgroup of 256 lanes per token, lane j on
// 16-byte vectors j, j + lanes, ...; every load of the row and of the weights is
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
#include "rope_kv.h"
#include "softmax_stream.h"

namespace mi {
namespace {

struct RowArgs {
    const int64_t* ids;
    const half_t* table;
    half_t *hidden, *normed, *post, *fin, *attn, *mlp;
    const half_t *w_in, *w_post, *w_fin, *w_attn, *w_mlp;
    int64_t D, vocab;
    float scale, eps, w_bias;
    int lanes;  // of the 256: rms_row_kernel's for rows of D, so that the norms of the
                // blocks' outputs and of the residuals have its bits, and
                // rms_small_kernel's (D <= 512: one vector per lane in both).  The
                // gather + norm kernel has 256: where these are fewer and hold several
                // vectors each, the input norm may be an fp16 ulp from its
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

// Token t of the rows, by one workgroup; slots: 5 floats per wave.
template <int VPT, bool DOUBLE>
__device__ __forceinline__ void chain_row(const RowArgs& r, int64_t t, float* slots) {
    float* slots2 = slots + (256 / kWave) * 3;
    const int64_t nv = r.D >> 3;
    const int64_t row = t * r.D;
    const float Df = static_cast<float>(r.D);
    // loads: attn and mlp do not wait for the token id
    h8 a[VPT], m[VPT], h[VPT];
    int64_t at[VPT];
    bool ok[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int64_t c = threadIdx.x + j * r.lanes;
        ok[j] = c < nv && static_cast<int>(threadIdx.x) < r.lanes;
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

template <int VPT, bool DOUBLE>
__global__ __launch_bounds__(256) void chain_rows_kernel(RowArgs r) {
    __shared__ float slots[(256 / kWave) * 5];
    chain_row<VPT, DOUBLE>(r, blockIdx.x, slots);
}

// Checks the rows and fills their device arguments.
bool rows_plan(const ChainRows& c, RowArgs& r) {
    if (c.T <= 0 || c.T > kMaxGridX || c.D <= 0 || c.D % 8 != 0 || c.D > 4 * 2048)
        return false;
    const void* rows[] = {c.table, c.hidden, c.normed, c.post_normed, c.final_normed, c.attn, c.mlp,
                          c.w_in, c.w_post, c.w_final, c.w_attn, c.w_mlp};
    for (const void* p : rows)
        if (!aligned16(p)) return false;
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
    const int64_t chunks = c.D / 8, vpt = ceil_div(chunks, 256);
    r.lanes = static_cast<int>(ceil_div(ceil_div(chunks, vpt), kWave) * kWave);
    r.D = c.D;
    r.vocab = c.vocab;
    r.scale = c.scale;
    r.eps = c.eps;
    r.w_bias = c.add_one ? 1.0f : -0.0f;  // -0: w + bias == w, signed zeros kept
    return true;
}

// ---------------------------------------------------------------------------
// The whole step in one launch.  With few tokens each stage is a few microseconds
// of latency on a GPU mostly idle, and every launch costs the host about 3 us; with
// many, each launch ends in a round of workgroups that leaves most of it idle, and
// the sampling step, bound by its exchange, leaves HBM idle throughout.  The
// workgroups of one grid take the stages' shares, each running that stage's own
// kernel body: first the sampling chunks (they wait for one another, so all must
// be resident), then a workgroup per token for RoPE + cache and one for the rows,
// then the activation's tiles.  No stage reads what another writes.
// Only for a caller that has every stage's input before the call: in a model that
// runs, a GEMM between the stages makes each from the one before, and its layer
// calls the stages one by one.
// Measured as called, against rows, RoPE + cache, activation and sampling as four
// launches: T = 1 17.7 -> 8.2 us (5.9 since the Python call is native), T = 24 (Gemma
// norms) 25.6 -> 9.9 (9.2), T = 1048 44.0 -> 36.3 (36.1), T = 6064 196.8 -> 181.9
// (181.4, 6.3 TB/s of what the step has to move).
// ---------------------------------------------------------------------------
struct ActArgs {
    const half_t *gate, *up;
    half_t* out;
    int64_t nvec;
};
struct SampleArgs {
    const half_t* x;
    half_t* y;
    unsigned char* ws;
    int32_t* out;
    int64_t N, V;
    int poll_limit, splits, R, local, u, ragged;
};
enum RopeKind { kRopePlain = 0, kRopeBias = 1, kRopeNorm = 2 };
template <int NF>
struct StepArgs {
    SampleArgs sample;
    RowArgs rows;
    ActArgs act;
    int n_sample, n_tokens;       // workgroups of the first roles
    int vpt, rope, slots, gelu;  // which body each role runs
    RopeKv kv;
    InvFreqN<NF> inv;
};

// 16-byte vectors per lane and operand: T = 6064 181.9 us with 1, 182.9 with 2, 187.1
// with 4; T = 1048 36.3 / 37.2 / 39.0.
constexpr int kActVecs = 1;

template <bool GELU>
__device__ __forceinline__ void act_block(const ActArgs& a, int64_t block) {
    const int64_t base = block * (256 * kActVecs) + threadIdx.x;
    h8 g[kActVecs], u[kActVecs];
#pragma unroll
    for (int j = 0; j < kActVecs; ++j) {
        const int64_t v = base + j * 256;
        if (v < a.nvec) {
            g[j] = ld8_stream(a.gate + v * 8);
            u[j] = ld8_stream(a.up + v * 8);
        }
    }
#pragma unroll
    for (int j = 0; j < kActVecs; ++j) {
        const int64_t v = base + j * 256;
        if (v < a.nvec) {
            h8 o;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float f = (float)g[j][k], w = (float)u[j][k];
                o[k] = to_half(GELU ? (float)to_half(gelu_tanh(f)) * w : silu_mul(f, w));
            }
            st8_stream(a.out + v * 8, o);
        }
    }
}

template <int CPH, int P, int NF>
__device__ __forceinline__ void step_rope(const StepArgs<NF>& a, int64_t tok, float* cs) {
    if (a.rope == kRopeNorm)
        rope_kv_token<false, true, CPH, P>(a.kv, a.inv.v, tok, true, cs);
    else if (a.rope == kRopeBias)
        rope_kv_token<true, false, CPH, P>(a.kv, a.inv.v, tok, true, cs);
    else
        rope_kv_token<false, false, CPH, P>(a.kv, a.inv.v, tok, true, cs);
}

// NF = 64: heads of 64 and 128; NF = 128: heads of 256.  The sampling chunks have
// to be resident together, so the registers are held to 6 waves per SIMD (1536
// workgroups; 5 where the rows take two reductions, which would spill).
template <int NF, bool DOUBLE>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(DOUBLE ? 5 : 6))) void chain_step_kernel(
    StepArgs<NF> args) {
    // read where it lies, in the kernel-argument block (the one argument, at its
    // offset 0): through its name, a struct of this many uses is first copied
    // into scratch memory
    const StepArgs<NF>& a = *(const StepArgs<NF>*)__builtin_amdgcn_kernarg_segment_ptr();
    __shared__ __attribute__((aligned(16))) float cs[2 * kMaxHalf];
    __shared__ float slots[(256 / kWave) * 5];
    int b = blockIdx.x;
    if (b < a.n_sample) {
        const SampleArgs& s = a.sample;
#define MI_STEP_SAMPLE(U, RAGGED, ONE)                                                          \
    softmax_argmax_block<U, RAGGED, ONE>(b, s.x, s.y, s.ws, s.N, s.V, s.poll_limit, s.out, s.splits, \
                                         s.R, s.local)
        if (s.ragged) {
            if (s.u == 2) MI_STEP_SAMPLE(2, true, true);
            else MI_STEP_SAMPLE(4, true, true);
        } else {
            if (s.u == 2) MI_STEP_SAMPLE(2, false, true);
            else MI_STEP_SAMPLE(4, false, true);
        }
#undef MI_STEP_SAMPLE
        return;
    }
    b -= a.n_sample;
    if (b < a.n_tokens) {
        if constexpr (NF == 128) {
            if (a.slots <= 256) step_rope<16, 1>(a, b, cs);
            else step_rope<16, 2>(a, b, cs);
        } else if (a.kv.hd == 64) {
            if (a.slots <= 256) step_rope<4, 1>(a, b, cs);
            else step_rope<4, 2>(a, b, cs);
        } else {
            if (a.slots <= 256) step_rope<8, 1>(a, b, cs);
            else step_rope<8, 2>(a, b, cs);
        }
        return;
    }
    b -= a.n_tokens;
    if (b < a.n_tokens) {
        if (a.vpt == 1) chain_row<1, DOUBLE>(a.rows, b, slots);
        else chain_row<2, DOUBLE>(a.rows, b, slots);
        return;
    }
    b -= a.n_tokens;
    if (a.gelu) act_block<true>(a.act, b);
    else act_block<false>(a.act, b);
}

template <int NF, bool DOUBLE>
int step_go(const ChainStep& c, StepArgs<NF>& a, hipStream_t s) {
    const int64_t R = ceil_div(c.N, kXcds) * kXcds;  // 0: a step without sampling
    // every sampling chunk resident at once: at the softmax's own chunk size, or
    // the larger one
    const int64_t cap =
        resident_workgroups(reinterpret_cast<const void*>(chain_step_kernel<NF, DOUBLE>), 256);
    if (R * a.sample.splits > cap && a.sample.u < 4) {
        a.sample.u = 4;
        a.sample.splits = static_cast<int>(ceil_div(c.vocab + (a.sample.ragged ? 7 : 0), 2048 * 4));
    }
    const int64_t n_sample = R * a.sample.splits;
    if (n_sample > cap) return MI_ERR_UNSUPPORTED;
    a.sample.R = static_cast<int>(R);
    a.n_sample = static_cast<int>(n_sample);
    a.n_tokens = static_cast<int>(c.rows.T);
    for (int i = 0; i < NF; ++i) a.inv.v[i] = i < c.head_dim / 2 ? c.inv_freq_host[i] : 0.0f;
    const int64_t grid = n_sample + 2 * c.rows.T + ceil_div(a.act.nvec, 256 * kActVecs);
    if (grid > kMaxGridX) return MI_ERR_UNSUPPORTED;
    chain_step_kernel<NF, DOUBLE><<<dim3(static_cast<unsigned>(grid)), dim3(256), 0, s>>>(a);
    return launch_status();
}

template <int NF>
int step_plan(const ChainStep& c, const RowArgs& rows, const RopeKv& kv, int64_t slots,
              const StreamPlan& sp, hipStream_t s) {
    StepArgs<NF> a;
    a.rows = rows;
    a.kv = kv;
    a.slots = static_cast<int>(slots);
    a.vpt = static_cast<int>(ceil_div(c.rows.D / 8, 256));
    a.rope = c.q_weight ? kRopeNorm : c.q_bias ? kRopeBias : kRopePlain;
    a.gelu = c.gelu;
    a.act = ActArgs{static_cast<const half_t*>(c.gate), static_cast<const half_t*>(c.up),
                    static_cast<half_t*>(c.act_out), c.act_n / 8};
    a.sample = SampleArgs{static_cast<const half_t*>(c.logits),
                          static_cast<half_t*>(c.probs),
                          static_cast<unsigned char*>(c.workspace),
                          c.next_tokens,
                          c.N,
                          c.vocab,
                          sp.poll_limit,
                          sp.splits,
                          0,
                          sp.local,
                          sp.u,
                          sp.ragged ? 1 : 0};
    return c.rows.w_attn ? step_go<NF, true>(c, a, s) : step_go<NF, false>(c, a, s);
}

}  // namespace

int chain_step(const ChainStep& c, void* stream) {
    if (c.rows.T <= 0 || c.rows.D > 2 * 2048) return MI_ERR_UNSUPPORTED;
    if (c.head_dim != 64 && c.head_dim != 128 && c.head_dim != 256) return MI_ERR_UNSUPPORTED;
    if (c.act_n <= 0 || c.act_n % 8 != 0 || !aligned16(c.gate) || !aligned16(c.up) ||
        !aligned16(c.act_out))
        return MI_ERR_UNSUPPORTED;
    RowArgs rows;
    if (!rows_plan(c.rows, rows)) return MI_ERR_UNSUPPORTED;
    RopeKv kv;
    int64_t slots = 0;
    if (rope_kv_plan(c.q, c.k, c.v, c.q_bias, c.k_bias, c.v_bias, c.q_weight, c.k_weight, c.qk_eps,
                     /*add_one=*/0, c.positions, c.inv_freq_host, c.rows.T, c.Hq, c.Hkv, c.head_dim,
                     c.k_cache, c.v_cache, c.layer, c.num_blocks, c.block_size, c.segments,
                     c.num_segments, /*wide=*/true, kv, slots) != MI_OK ||
        slots > 512)
        return MI_ERR_UNSUPPORTED;
    // Where the launches apart are faster: without the sampling to hide, large
    // batches (T = 764, Gemma norms 40.9 -> 38.5 us in two launches instead of four,
    // but T = 5464 138.9 against 142.2); tokens of few units, which RoPE + cache by
    // itself takes several of per workgroup (14 + 2 heads of 64: T = 2830 37.7 -> 34.3,
    // but T = 5430 56.5 against 58.8).
    if ((c.N == 0 && c.rows.T > 1024) || (slots <= 128 && c.rows.T > 4096)) return MI_ERR_UNSUPPORTED;
    StreamPlan sp{};
    if (c.N > 0 && !softmax_argmax_plan(c.logits, c.probs, c.next_tokens, c.N, c.vocab, c.workspace,
                                        c.workspace_bytes, sp))
        return MI_ERR_UNSUPPORTED;
    const hipStream_t s = as_stream(stream);
    return c.head_dim == 256 ? step_plan<128>(c, rows, kv, slots, sp, s)
                             : step_plan<64>(c, rows, kv, slots, sp, s);
}

int chain_rows(const ChainRows& c, void* stream) {
    RowArgs r;
    if (!rows_plan(c, r)) return MI_ERR_UNSUPPORTED;
    const bool dbl = c.w_attn != nullptr;
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
