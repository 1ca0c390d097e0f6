// softmax_stream.h -- the one-launch split-row softmax (and its fused greedy
// argmax): a workgroup's share of it, which softmax_stream_kernel (softmax.hip) and
// the one-launch decoder step (chain_step.hip) run.
#pragma once

#include "argmax_key.h"
#include "mi_device.h"
#include "row_exchange.h"

// Softmax stores: plain non-temporal (1 = write-through "nt sc1"; measured neutral).
#ifndef MI_WT_SM
#define MI_WT_SM 0
#endif

namespace mi {

// exp(x - m) for every element of a row against one m, with m * log2(e)
// formed once: one fma and the exp per element instead of a subtract, a
// multiply and the exp (the VALU work sits on the critical path before and
// after a one-launch row's exchange: 9.5 -> 8.9 us at [64, 152064]).
constexpr float kLog2e = 1.4426950408889634f;
__device__ __forceinline__ float exp_shifted(float x, float m_log2e) {
    return __builtin_amdgcn_exp2f(fmaf(x, kLog2e, -m_log2e));
}

// Fold one loaded value group into the lane's online (m, s).
template <int VEC>
__device__ __forceinline__ void fold(const float (&v)[VEC], float& m, float& s) {
    float vm = v[0];
#pragma unroll
    for (int k = 1; k < VEC; ++k) vm = fmaxf(vm, v[k]);
    const float mn = fmaxf(m, vm);
    if (mn == -INFINITY) return;  // nothing but -inf so far
    float acc = s * fast_exp(m - mn);
    const float mnl = mn * kLog2e;
#pragma unroll
    for (int k = 0; k < VEC; ++k) acc += exp_shifted(v[k], mnl);
    s = acc;
    m = mn;
}

// Accumulate elements [begin, end) of a row into this lane's (m, s).  Loads
// are issued kStatUnroll groups at a time, before the math that consumes them.
constexpr int kStatUnroll = 4;
template <int VEC>
__device__ __forceinline__ void lane_stats(const half_t* xr, int64_t begin, int64_t end, float& m,
                                           float& s) {
    const int64_t step = static_cast<int64_t>(blockDim.x) * VEC;
    for (int64_t i0 = begin + static_cast<int64_t>(threadIdx.x) * VEC; i0 < end;
         i0 += step * kStatUnroll) {
        float v[kStatUnroll][VEC];
#pragma unroll
        for (int j = 0; j < kStatUnroll; ++j) {
            const int64_t i = i0 + j * step;
            if (i < end) {
                if constexpr (VEC == 8) {
                    const h8 h = ld8(xr + i);
#pragma unroll
                    for (int k = 0; k < 8; ++k) v[j][k] = (float)h[k];
                } else {
                    v[j][0] = (float)xr[i];
                }
            } else {
#pragma unroll
                for (int k = 0; k < VEC; ++k) v[j][k] = -INFINITY;
            }
        }
#pragma unroll
        for (int j = 0; j < kStatUnroll; ++j) fold<VEC>(v[j], m, s);
    }
}

// Vector form for split rows: [begin, end) is walked in tiles of 2048 * U
// elements (U vectors per lane), all loads of a tile issued first.  The
// tile's lane maximum comes from packed fp16 max (which passes over NaN, as
// fmaxf does), then one exp per element against it, and one online merge
// per tile -- not a rescale per vector.  Out-of-range slots hold -inf, whose
// exp is 0.  RAGGED: xr is the row's window `win`, [begin, end) positions in
// it.
template <int U, bool RAGGED = false>
__device__ __forceinline__ void tile_stats(const half_t* xr, int64_t begin, int64_t end, float& m,
                                           float& s, const RowWindow* win = nullptr) {
    constexpr int64_t kTile = 256 * 8 * U;
    for (int64_t t0 = begin; t0 < end; t0 += kTile) {
        h8 a[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int64_t i = t0 + (threadIdx.x + j * 256) * 8;
            a[j] = i < end ? ld8(xr + i) : h8(-__builtin_huge_valf16());
        }
        if constexpr (RAGGED) {
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const int64_t i = t0 + (threadIdx.x + j * 256) * 8;
                if (i < end && win->partial(static_cast<int>(i >> 3)))
                    win->mask(static_cast<int>(i >> 3), a[j]);
            }
        }
        h2 m2 = h2(-__builtin_huge_valf16());
#pragma unroll
        for (int j = 0; j < U; ++j) {
#pragma unroll
            for (int k = 0; k < 8; k += 2) m2 = __builtin_elementwise_max(m2, h2{a[j][k], a[j][k + 1]});
        }
        const float mt = (float)__builtin_elementwise_max(m2.x, m2.y);
        if (!(mt > -INFINITY)) continue;  // nothing but -inf (or NaN) in this lane's tile
        float st = 0.0f;
        const float mtl = mt * kLog2e;
#pragma unroll
        for (int j = 0; j < U; ++j) {
#pragma unroll
            for (int k = 0; k < 8; ++k) st += exp_shifted((float)a[j][k], mtl);
        }
        const float mn = fmaxf(m, mt);
        s = s * fast_exp(m - mn) + st * fast_exp(mt - mn);
        m = mn;
    }
}

// Workgroup-wide merge of per-lane (m, s): max first, then rescaled sums.
// (A one-barrier form -- wave (max, sum) pairs folded after a single barrier
// -- measured no faster at [64, 152064].)  `slots` needs one float per wave.
__device__ __forceinline__ void block_merge(float& m, float& s, float* slots) {
    const float M = block_max(m, slots);
    const float part = (m == -INFINITY) ? 0.0f : s * fast_exp(m - M);
    __syncthreads();  // slots are reused by the sum
    s = block_sum(part, slots);
    m = M;
}

// ---------------------------------------------------------------------------
// One-launch split rows (row records: mi_softmax_ws_f16, or stream 0; x != y):
// each workgroup holds an 8192-element chunk of a row in registers, publishes
// the chunk's (max, sum), and reads every chunk's pair of its row to finish --
// one launch, one read of x, no atomics on a contended address.  The grid is
// `chunks per row` x R row slots, all resident; slot r handles rows r, r + R,
// ... in rounds (one round when every row fits), and issues its next row's
// loads before it polls for the current row's statistics.
//
// Workspace (zero before first use; every call leaves it valid for the
// next): row slot r owns a fixed record at r * kRowRecordBytes -- a 64-bit
// epoch word (128-byte header), then two sets of kOnePassMaxSplits slots of
// two 64-bit words {tag << 32 | bits(max)}, {tag << 32 | bits(sum)}, and a
// mirror of both sets (row_exchange.h: each word is published into the XCD's
// L2 and through to memory; polls read the L2 copy first).  A call
// reads the slot's epoch E; round k publishes into set k & 1 with tag = the
// low 32 bits of E + 1 + k and polls the set until every chunk's pair carries
// that tag.  Because slots are fixed per (row slot, chunk) whatever the
// call's shape, and an epoch only grows (64 bits: it cannot wrap), a slot
// left by an earlier call never carries the tag a later call waits for --
// short of a slot left unwritten for 2^32 of its epochs and read again at
// exactly a multiple of 2^32 later:
//   * the chunk-0 workgroup raises the epoch to E + K (atomic max) after the
//     last (K-th) round, when every workgroup of the slot has published it --
//     so every one of them has already read E;
//   * a workgroup whose polling runs out (kPollLimit polls or kPollTicks of
//     the 100 MHz constant clock, whichever comes first; not expected when
//     the grid fits the GPU) computes that row's statistics itself from x and
//     raises the epoch to E + K + 1 at once, past every tag the launch writes
//     for the slot.  A workgroup that starts after that reads the higher
//     epoch, its tags match nobody's, and it takes the same fallback for its
//     rows: slower, still correct.  A workgroup that has fallen back once
//     stops polling for its remaining rounds (its row-mates may be out of
//     step with it for good), so a late start costs at most one poll bound
//     per workgroup, not one per round.  Polling is bounded: no workgroup
//     can wait forever.
// A workgroup publishes round k + 2 into a set only after it has seen every
// chunk's round k + 1 pair, which its row-mates publish after they have read
// round k: no pair is overwritten before it is read.  Each 64-bit word is
// stored and loaded whole, so a tag always travels with its value.
// The grid is 1-D and places every chunk of a row slot on one XCD
// (chunk_of), so the L2 copy normally serves the polls.
// ---------------------------------------------------------------------------
constexpr int kOnePassMaxSplits = 64;
#ifndef MI_SOFTMAX_ONEPASS_U
#define MI_SOFTMAX_ONEPASS_U 4
#endif
constexpr int kOnePassU = MI_SOFTMAX_ONEPASS_U;     // vectors per lane
constexpr int64_t kOnePassChunk = 2048 * kOnePassU;  // elements per workgroup
// header, then two sets of slots (alternated by round) and their mirror; a
// slot is the chunk's tagged (max, sum) pair, plus its tagged argmax key (two
// words) in the fused softmax + argmax pass
constexpr int64_t kRowRecordBytes = kRecordHeaderBytes + 4 * kOnePassMaxSplits * 16;
constexpr int64_t kRowRecordBytesAM = kRecordHeaderBytes + 4 * kOnePassMaxSplits * 32;
template <bool AM>
constexpr int64_t record_bytes() { return AM ? kRowRecordBytesAM : kRowRecordBytes; }

__device__ __forceinline__ uint64_t tagged(uint32_t tag, float v) {
    return (static_cast<uint64_t>(tag) << 32) | __builtin_bit_cast(uint32_t, v);
}

// The pieces of a one-launch chunk workgroup.
// The lane's (max, sum) over its vectors: packed fp16 maximum, one exp per
// element.
template <int U>
__device__ __forceinline__ void chunk_lane_stats(const h8 (&a)[U], float& m, float& s) {
    h2 m2 = h2(-__builtin_huge_valf16());
#pragma unroll
    for (int j = 0; j < U; ++j) {
#pragma unroll
        for (int k = 0; k < 8; k += 2) m2 = __builtin_elementwise_max(m2, h2{a[j][k], a[j][k + 1]});
    }
    m = (float)__builtin_elementwise_max(m2.x, m2.y);
    s = 0.0f;
    if (m > -INFINITY) {
        const float ml = m * kLog2e;
#pragma unroll
        for (int j = 0; j < U; ++j) {
#pragma unroll
            for (int k = 0; k < 8; ++k)
                s += exp_shifted((float)a[j][k], ml);
        }
    } else {
        m = -INFINITY;  // NaN-free lane maximum of an all -inf (or NaN) lane
    }
}
// Thread 0 publishes the chunk's pair (and, AM, its argmax key) into slot
// `split` of `slots` (SW = 2 or 4 words per slot) and of its mirror
// (`mirror` words on).
template <bool AM>
__device__ __forceinline__ void chunk_publish(uint64_t* slots, int64_t mirror, int split,
                                              uint32_t tag, float m, float s, uint64_t key) {
    constexpr int SW = AM ? 4 : 2;
    if (threadIdx.x == 0) {
        uint64_t w[SW];
        w[0] = tagged(tag, m);
        w[1] = tagged(tag, s);
        if constexpr (AM) {
            const uint64_t t = static_cast<uint64_t>(tag) << 32;
            w[2] = t | (key >> 32);
            w[3] = t | (key & 0xffffffffu);
        }
        uint64_t* p = slots + SW * split;
#pragma unroll
        for (int i = 0; i < SW; ++i) local_store(&p[i], w[i]);
#pragma unroll
        for (int i = 0; i < SW; ++i) device_store(&p[mirror + i], w[i]);
    }
}
// Wave 0 (the caller calls it there) polls the row's `splits` slots (lane j
// reads chunk j) until all carry `tag`, at most poll_limit rounds -- the L2
// copy (local) for up to kLocalPollTicks, then the mirror `mirror` words on
// at device scope (row_exchange.h) -- and leaves
// the row's (M, S) in row_stats[0..1] (AM with want_key: its best key in
// *row_key, the key words polled too; without, only the pair words, half
// the bytes per poll: 12.9 -> 12.0 us at [64, 152064]) and row_stats[2] = 0,
// or row_stats[2] = 1 when polling ran out.  The caller's barrier publishes
// them.
// Polls of one phase (LOCAL: the L2 copy, else the device-scope mirror) of
// `set` (workgroup-uniform) until every chunk's slot carries `tag`, `it`
// reaches poll_limit or the clock passes t0 + ticks; lane j < splits reads
// slot j.  Returns whether every slot was seen.
template <bool AM, bool LOCAL>
__device__ __forceinline__ bool poll_phase(const uint64_t* set, int splits, uint32_t tag,
                                           bool want_key, int& it, int poll_limit, uint64_t t0,
                                           uint64_t ticks, float& mj, float& sj, uint64_t& kj) {
    constexpr int SW = AM ? 4 : 2;
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t off = static_cast<uint32_t>(lane) * (SW * 8);
    for (; it < poll_limit; ++it) {
        if (it > 0 && __builtin_amdgcn_s_memrealtime() - t0 > ticks) return false;
        bool mine = true;
        if (lane < splits) {
            // chunk 0 alone writes the index, so only it reads the key words
            uint64_t w[SW];
            if (AM && want_key)
                load_slot<LOCAL, SW>(set, off, w);
            else
                load_slot<LOCAL, 2>(set, off, reinterpret_cast<uint64_t(&)[2]>(w));
            mine = static_cast<uint32_t>(w[0] >> 32) == tag && static_cast<uint32_t>(w[1] >> 32) == tag;
            mj = __builtin_bit_cast(float, static_cast<uint32_t>(w[0]));
            sj = __builtin_bit_cast(float, static_cast<uint32_t>(w[1]));
            if constexpr (AM) {
                if (want_key) {
                    mine = mine && static_cast<uint32_t>(w[2] >> 32) == tag &&
                           static_cast<uint32_t>(w[3] >> 32) == tag;
                    kj = (w[2] << 32) | (w[3] & 0xffffffffu);
                }
            }
        }
        if (__all(mine)) return true;
        __builtin_amdgcn_s_sleep(2);
    }
    return false;
}

template <bool AM>
__device__ __forceinline__ void row_poll(const uint64_t* slots, int64_t mirror, bool local,
                                         int splits, uint32_t tag, int poll_limit,
                                         float* row_stats, uint64_t* row_key, bool want_key) {
    const int lane = threadIdx.x & (kWave - 1);
    float mj = -INFINITY, sj = 0.0f;
    uint64_t kj = 0;
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    int it = 0;
    bool all = local && poll_phase<AM, true>(slots, splits, tag, want_key, it, poll_limit, t0,
                                             kLocalPollTicks, mj, sj, kj);
    if (!all)
        all = poll_phase<AM, false>(slots + mirror, splits, tag, want_key, it, poll_limit, t0,
                                    kPollTicks, mj, sj, kj);
    if (all) {
        if (lane >= splits) {
            mj = -INFINITY;
            sj = 0.0f;
            kj = 0;
        }
        const float M = group_max<kWave>(mj);
        const float S = group_sum<kWave>(mj == -INFINITY ? 0.0f : sj * fast_exp(mj - M));
        if (AM && want_key) kj = wave_max_u64(kj);
        if (lane == 0) {
            row_stats[0] = M;
            row_stats[1] = S;
            row_stats[2] = 0.0f;
            if (AM && want_key) *row_key = kj;
        }
    } else if (lane == 0) {
        row_stats[2] = 1.0f;
    }
}
// The row's statistics from x itself (the fallback when polling runs out; x
// is not written: y != x).  Barriers: called by the whole workgroup.
template <bool RAGGED>
__device__ __forceinline__ void row_stats_from_x(const half_t* xr, int64_t D, float& M, float& S,
                                                 float* slots) {
    float fm = -INFINITY, fs = 0.0f;
    if constexpr (RAGGED)
        lane_stats<1>(xr, 0, D, fm, fs);
    else
        tile_stats<2>(xr, 0, D, fm, fs);
    __syncthreads();  // slots reused
    block_merge(fm, fs, slots);
    __syncthreads();  // every wave has read slots before a later round writes them
    M = fm;
    S = fs;
}
// The persistent kernel's per-lane view of its chunk: the same in every
// round, so one 32-bit byte offset (rows are < 2^31 bytes) and a valid flag
// per vector, against a row base that is uniform across the workgroup.
template <int U>
__device__ __forceinline__ void lane_load(const half_t* row, uint32_t lo, const bool (&ok)[U],
                                          h8 (&a)[U]) {
    const char* base = reinterpret_cast<const char*>(row) + lo;
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const half_t* p = reinterpret_cast<const half_t*>(base + j * 256 * 16);
        a[j] = ok[j] ? ld8_stream(p) : h8(-__builtin_huge_valf16());
    }
}
// RAGGED: row is the row's window, v0 the lane's first vector in it.
template <int U, bool RAGGED>
__device__ __forceinline__ void lane_store(const h8 (&a)[U], half_t* row, uint32_t lo,
                                           const bool (&ok)[U], float M, float inv,
                                           const RowWindow& win, int v0) {
    // y = exp(x - M) / S = exp2(x log2(e) - (M log2(e) + log2(S))): the division folded into
    // the exponent's constant c, one fma and the exp per element ([512, 131072] 46.4 -> 46.0
    // us; c carries the same rounding as M log2(e) alone, well under an fp16 ulp of y)
    const float c = M * kLog2e - __builtin_amdgcn_logf(inv);
    char* base = reinterpret_cast<char*>(row) + lo;
#pragma unroll
    for (int j = 0; j < U; ++j) {
        if (ok[j]) {
            h8 o;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                o[k] = to_half(__builtin_amdgcn_exp2f(fmaf((float)a[j][k], kLog2e, -c)));
            half_t* p = reinterpret_cast<half_t*>(base + j * 256 * 16);
            if constexpr (RAGGED)
                win.store(v0 + j * 256, p, o);
            else
                st8_out<MI_WT_SM>(p, o);
        }
    }
}

// How the one-launch softmax + argmax cuts a call's rows (softmax.hip): u vectors
// per lane, splits chunks per row.  False when the call does not take that form.
struct StreamPlan {
    int u, splits, poll_limit, local;
    bool ragged;
};
bool softmax_argmax_plan(const void* logits, const void* probs, const void* out, int64_t N,
                         int64_t V, const void* workspace, int64_t workspace_bytes, StreamPlan& p);

// A workgroup's share of the fused softmax + greedy argmax, for a kernel that
// runs it beside other work.
template <int U, bool RAGGED, bool ONE>
__device__ __forceinline__ void softmax_argmax_block(int block, const half_t* x, half_t* y,
                                                     unsigned char* ws, int64_t N, int64_t D,
                                                     int poll_limit, int32_t* out, int splits,
                                                     int R, int local) {
    constexpr bool AM = true;
#include "softmax_stream_body.h"
}

}  // namespace mi
