// softmax.hip -- row softmax for gfx950, fp16 in/out, fp32 math.
//
// Arithmetic follows the reference (src/kernels/softmax_kernel.cu:26-58):
// m = max(x), S = sum(exp(x - m)), y = half(exp(x - m) * (1 / S)).
//
// Design (HBM-bound: 4 bytes/element):
//   * Each lane keeps an online (max, sum) pair over its 16-byte vectors,
//     rescaling the sum when the max grows, so statistics need ONE read of x
//     (the reference makes separate max and sum passes, then a third to write).
//   * Many rows (N >= 512; N >= 256 up to 65536): whole rows, in registers
//     where they fit (softmax_reg_kernel), else one workgroup per row whose
//     write pass re-reads the row through L2.
//   * Few long rows (the LM-head case, 64 x 152064), and many rows longer
//     than 32768 (N >= 512, or N >= 256 up to 65536): one workgroup per row
//     would light up few CUs or re-read the row, so each row is cut into
//     8192-element chunks.  With row records -- a caller workspace, or on
//     stream 0 a region the library holds -- and y != x, one launch
//     (softmax_stream_kernel, below): a resident grid of chunk workgroups
//     holds the chunks in registers and exchanges their (max, sum) through
//     tagged per-row records, walking the rows in rounds when they are more
//     than the grid holds, with the next row's loads in flight during each
//     exchange.  Otherwise many rows take a workgroup per row, and few rows
//     two launches with `splits` chunks:
//     Kernel 1 writes a (max, sum) pair per chunk to a small stream-ordered
//     workspace (8 bytes per chunk), from tiles whose loads are all issued
//     first (one HBM wait per tile), a packed fp16 lane maximum and one exp
//     per element;
//     kernel 2, on the same grid, merges the row's pairs (each lane folds
//     every 64th chunk, then wave reductions, no barrier) and writes its
//     chunk.  Its re-read of the chunk misses L2, which does not carry
//     data across kernel launches on this multi-XCD GPU (FETCH_SIZE counts
//     the full 2 bytes/element again); it is served from the 256 MB
//     Infinity Cache when the logits are still resident there, else HBM.
#include <atomic>
#include <map>
#include <mutex>

#include "argmax_key.h"
#include "mi_device.h"
#include "mi_host.h"
#include "row_exchange.h"
#include "softmax_stream.h"

namespace mi {
namespace {

constexpr int kSplitMaxRows = 512;  // below this many rows, split each row
#ifndef MI_SOFTMAX_REG_ROWS
#define MI_SOFTMAX_REG_ROWS 256
#endif
constexpr int kMaxSplits = 1024;    // chunk pairs of a row, folded by one wave
#ifndef MI_SOFTMAX_TARGET_WGS
#define MI_SOFTMAX_TARGET_WGS 2048
#endif
constexpr int64_t kSplitTargetWgs = MI_SOFTMAX_TARGET_WGS;

// y = exp(x - m) * inv over [begin, end): the last use of x and the only
// write of y, both streamed.
template <int VEC, bool RAGGED = false>
__device__ __forceinline__ void write_range(const half_t* xr, half_t* yr, int64_t begin,
                                            int64_t end, float m, float inv,
                                            const RowWindow* win = nullptr) {
    const int64_t step = static_cast<int64_t>(blockDim.x) * VEC;
    for (int64_t i0 = begin + static_cast<int64_t>(threadIdx.x) * VEC; i0 < end;
         i0 += step * kStatUnroll) {
        if constexpr (VEC == 8) {
            h8 h[kStatUnroll];
#pragma unroll
            for (int j = 0; j < kStatUnroll; ++j) {
                const int64_t i = i0 + j * step;
                if (i < end) h[j] = ld8_stream(xr + i);
            }
#pragma unroll
            for (int j = 0; j < kStatUnroll; ++j) {
                const int64_t i = i0 + j * step;
                if (i < end) {
                    h8 o;
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        o[k] = to_half(exp_shifted((float)h[j][k], m * kLog2e) * inv);
                    if constexpr (RAGGED)
                        win->store(static_cast<int>(i >> 3), yr + i, o);
                    else
                        st8_out<MI_WT_SM>(yr + i, o);
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < kStatUnroll; ++j) {
                const int64_t i = i0 + j * step;
                if (i < end) yr[i] = to_half(exp_shifted((float)xr[i], m * kLog2e) * inv);
            }
        }
    }
}

// Register-resident rows (16-byte vectors, D <= G * VPT * 8): G lanes per
// row -- G <= 64: 256 / G rows per workgroup and DPP-only reductions;
// G = 128, 256 or 1024: one row per workgroup and one LDS exchange per
// reduction -- with VPT vectors per lane.  x is read once: a packed fp16
// lane maximum, the row maximum, one exp per element (kept in registers when
// VPT <= 4, recomputed at the write otherwise), the row sum, then the scaled
// write.  Lanes past the row hold -inf, whose exp is 0.  No lane returns
// early, so every group reduction sees all of its lanes.
// RAGGED: rows walked through their aligned windows (RowWindow), bound by HBM
// like the aligned rows but for the two partial granules of each row.  Against
// the 2-byte kernel that such rows took before (one element per lane, the row
// read twice): [57344, 511] 137 -> 24.7 us (aligned 512: 20.6), [17108, 1203]
// 90 -> 16.7, [28672, 2047] 173 -> 44.2, [14336, 1001] 79 -> 13.4.  Plain
// instead of streaming stores here: 16.7 -> 19.4 us at 1203; the partial
// vectors element by element: 16.8 -> 17.7.
template <int G, int VPT, bool RAGGED>
__global__ __launch_bounds__(G > 64 ? G : 256) void softmax_reg_kernel(const half_t* x,
                                                                        half_t* y, int64_t N,
                                                                        int64_t D) {
    constexpr int kThreads = G > 64 ? G : 256;
    constexpr int kRows = kThreads / G;
    constexpr bool kKeepExp = VPT <= 4;
    __shared__ float smax[kThreads / kWave], ssum[kThreads / kWave];
    const int gl = threadIdx.x & (G - 1);
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kRows + threadIdx.x / G;
    const bool live = row < N;
    const RowWindow win(x + row * D, D);  // RAGGED
    const int64_t nv = RAGGED ? win.nv : D >> 3;
    const int64_t off = row * D - (RAGGED ? win.shift : 0);
    const half_t* xr = x + off;
    h8 a[VPT];
    // vector j of this lane: a uniform base per j (xr + j * G * 8) plus the
    // lane's 32-bit byte offset (with the forced recompute below, 8-vector
    // rows went from 90-115 to 78-88 VGPRs)
    const uint32_t lo = static_cast<uint32_t>(gl) * 16u;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int64_t v = gl + j * G;
        const char* base = reinterpret_cast<const char*>(xr + static_cast<int64_t>(j) * G * 8);
        a[j] = live && v < nv ? ld8_stream(reinterpret_cast<const half_t*>(base + lo))
                              : h8(-__builtin_huge_valf16());
    }
    if constexpr (RAGGED) {
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const int v = gl + j * G;
            if (v < nv && win.partial(v)) win.mask(v, a[j]);
        }
    }
    h2 m2 = h2(-__builtin_huge_valf16());
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
#pragma unroll
        for (int k = 0; k < 8; k += 2) m2 = __builtin_elementwise_max(m2, h2{a[j][k], a[j][k + 1]});
    }
    float m = (float)__builtin_elementwise_max(m2.x, m2.y);
    if constexpr (G <= 64)
        m = group_max<G>(m);
    else
        m = block_max(m, smax);
    float e[kKeepExp ? VPT : 1][8];
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float t = exp_shifted((float)a[j][k], m * kLog2e);
            if constexpr (kKeepExp) e[j][k] = t;
            s += t;
        }
    }
    if constexpr (G <= 64)
        s = group_sum<G>(s);
    else
        s = block_sum(s, ssum);
    const float inv = 1.0f / s;
    // Recomputing the exps (VPT > 4): an opaque copy of m keeps the compiler
    // from reusing the sum loop's exps, which would hold 8 * VPT fp32 values
    // live instead of the 4 * VPT registers of fp16 data.
    float mw = m;
    if constexpr (!kKeepExp) asm volatile("" : "+v"(mw));
    half_t* yr = y + off;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int64_t v = gl + j * G;
        if (live && v < nv) {
            h8 o;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float t =
                    kKeepExp ? e[kKeepExp ? j : 0][k] : exp_shifted((float)a[j][k], mw * kLog2e);
                o[k] = to_half(t * inv);
            }
            half_t* p = reinterpret_cast<half_t*>(
                reinterpret_cast<char*>(yr + static_cast<int64_t>(j) * G * 8) + lo);
            if constexpr (RAGGED)
                win.store(static_cast<int>(v), p, o);
            else
                st8_out<MI_WT_SM>(p, o);
        }
    }
}

// Launch shape for softmax_reg_kernel: the fewest lanes per row (8, 16, 32,
// 64, then 128, 256 or 1024 as whole workgroups) that hold the row in at most
// 3 vectors each (of 8 to 64 lanes) or 4, else 1024 lanes with up to 8.  (3
// against 4 in a wave: [57344, 512] 20.7 -> 20.05 us, [14336, 1001] 13.2 -> 12.3,
// [20000, 256] 5.04 -> 4.69, [500, 1000] 2.99 -> 2.72, [17108, 1203] level; 2:
// 18.7 at 1203.)  128 lanes stop at
// kPairMax vectors, where 256 lanes would leave 3/8 of their slots idle:
// [20000, 2100] (263 vectors) 41.9 -> 31.1 us, but [20000, 3000] (375) 40.6
// against 42.3 us with 128.  (More than 4 vectors per lane of a single wave:
// 47.5 against 44.2 us at [28672, 2047].)  Returns false when the row needs
// more than 1024 x 8 vectors.
constexpr int kWaveVpt = 3;
constexpr int kRegVpt = 4;
constexpr int64_t kPairMax = 320;
// At most 8 vectors per lane (rows <= 1024 x 8 x 8 = 65536).  12 fit in
// 110 VGPRs but measured mixed: [256, 98304] 51% -> 57%, [300, 70000]
// 45% -> 36% (idle lanes and a 17%-full second round); 16 or more spill.
constexpr int kRegVptMax = 8;
bool reg_shape(int64_t nv, int& G, int& VPT) {
    static const int kG[] = {8, 16, 32, 64, 128, 256, 1024};
    G = 0;
    for (int g : kG) {
        if (nv <= (g == 128 ? kPairMax : static_cast<int64_t>(g <= 64 ? kWaveVpt : kRegVpt) * g)) {
            G = g;
            break;
        }
    }
    if (G == 0) {
        if (nv > 1024 * kRegVptMax) return false;
        G = 1024;
    }
    VPT = static_cast<int>(ceil_div(nv, G));
    if (VPT > 4) VPT = 8;
    return true;
}

template <int G, bool RAGGED>
void launch_reg(const half_t* x, half_t* y, int64_t N, int64_t D, int VPT, hipStream_t s) {
    constexpr int kThreads = G > 64 ? G : 256;
    const dim3 g(static_cast<unsigned>(ceil_div(N, kThreads / G))), b(kThreads);
    switch (VPT) {
#define MI_REG_CASE(V) \
    case V: softmax_reg_kernel<G, V, RAGGED><<<g, b, 0, s>>>(x, y, N, D); break;
        MI_REG_CASE(1)
        MI_REG_CASE(2)
        MI_REG_CASE(3)
        MI_REG_CASE(4)
        default:  // only 1024 lanes hold more (reg_shape)
            if constexpr (G == 1024) softmax_reg_kernel<G, 8, RAGGED><<<g, b, 0, s>>>(x, y, N, D);
#undef MI_REG_CASE
    }
}

template <bool RAGGED>
int launch_reg_rows(const half_t* x, half_t* y, int64_t N, int64_t D, int G, int VPT,
                    hipStream_t s) {
    switch (G) {
        case 8: launch_reg<8, RAGGED>(x, y, N, D, VPT, s); break;
        case 16: launch_reg<16, RAGGED>(x, y, N, D, VPT, s); break;
        case 32: launch_reg<32, RAGGED>(x, y, N, D, VPT, s); break;
        case 64: launch_reg<64, RAGGED>(x, y, N, D, VPT, s); break;
        case 128: launch_reg<128, RAGGED>(x, y, N, D, VPT, s); break;
        case 256: launch_reg<256, RAGGED>(x, y, N, D, VPT, s); break;
        default: launch_reg<1024, RAGGED>(x, y, N, D, VPT, s); break;
    }
    return launch_status();
}

template <int VEC>
__global__ __launch_bounds__(1024) void softmax_row_kernel(const half_t* x, half_t* y, int64_t D) {
    __shared__ float slots[1024 / kWave];
    const int64_t row = blockIdx.x;
    const half_t* xr = x + row * D;
    half_t* yr = y + row * D;
    float m = -INFINITY, s = 0.0f;
    lane_stats<VEC>(xr, 0, D, m, s);
    block_merge(m, s, slots);
    write_range<VEC>(xr, yr, 0, D, m, 1.0f / s);
}

// VEC = 8: U vectors per lane per tile (tile_stats); VEC = 1: lane_stats.
// RAGGED (VEC = 8): chunks of the row's window, the last one to its end.
template <int VEC, int U, bool RAGGED = false>
__global__ __launch_bounds__(256) void softmax_partial_kernel(const half_t* x, float* ws,
                                                              int64_t D, int64_t chunk) {
    __shared__ float slots[256 / kWave];
    const int split = blockIdx.x, splits = gridDim.x;
    const int64_t row = blockIdx.y;
    const int64_t b = split * chunk;
    const int64_t e = b + chunk < D ? b + chunk : D;
    float m = -INFINITY, s = 0.0f;
    if constexpr (RAGGED) {
        const RowWindow win(x + row * D, D);
        tile_stats<U, true>(x + row * D - win.shift, b, split + 1 == splits ? win.len() : b + chunk,
                            m, s, &win);
    } else if constexpr (VEC == 8)
        tile_stats<U>(x + row * D, b, e, m, s);
    else
        lane_stats<VEC>(x + row * D, b, e, m, s);
    block_merge(m, s, slots);
    if (threadIdx.x == 0) {
        float* p = ws + (row * splits + split) * 2;
        p[0] = m;
        p[1] = s;
    }
}

template <int VEC, bool RAGGED = false>
__global__ __launch_bounds__(256) void softmax_finish_kernel(const half_t* x, half_t* y,
                                                             const float* __restrict__ ws,
                                                             int64_t D, int64_t chunk) {
    const int split = blockIdx.x, splits = gridDim.x;
    const int64_t row = blockIdx.y;
    const int lane = threadIdx.x & (kWave - 1);
    // Every wave merges the row's pairs itself: lane j folds chunks j, j + 64, ...
    float m = -INFINITY, s = 0.0f;
    for (int j = lane; j < splits; j += kWave) {
        const float* p = ws + (row * splits + j) * 2;
        const float mj = p[0], sj = p[1];
        if (mj == -INFINITY) continue;
        const float mn = fmaxf(m, mj);
        s = s * fast_exp(m - mn) + sj * fast_exp(mj - mn);
        m = mn;
    }
    const float M = group_max<kWave>(m);
    const float S = group_sum<kWave>(m == -INFINITY ? 0.0f : s * fast_exp(m - M));
    const int64_t b = split * chunk;
    const int64_t e = b + chunk < D ? b + chunk : D;
    if constexpr (RAGGED) {
        const RowWindow win(x + row * D, D);
        const int64_t off = row * D - win.shift;
        write_range<VEC, true>(x + off, y + off, b, split + 1 == splits ? win.len() : b + chunk, M,
                               1.0f / S, &win);
    } else {
        write_range<VEC>(x + row * D, y + row * D, b, e, M, 1.0f / S);
    }
}

// softmax_stream.h: the one-launch split rows
template <int U, bool AM, bool RAGGED, bool ONE>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(AM ? 5 : 1))) void softmax_stream_kernel(
    const half_t* x, half_t* y, unsigned char* ws, int64_t N, int64_t D, int poll_limit, int32_t* out,
    int splits, int R, int local) {
    const int block = blockIdx.x;
#include "softmax_stream_body.h"
}

constexpr int kPollLimit = 1 << 16;
std::atomic<int> g_poll_limit{kPollLimit};  // mi_softmax_test_poll_limit

// kStream: many rows long enough that chunking them beats a workgroup per
// row; with row records and y != x they run as softmax_stream_kernel,
// otherwise as kRow.
enum class Plan { kRow, kTwoPass, kStream };

#ifndef MI_SOFTMAX_STREAM
#define MI_SOFTMAX_STREAM 1
#endif
#ifndef MI_SOFTMAX_STREAM_MIN_D
#define MI_SOFTMAX_STREAM_MIN_D 32769
#endif
bool stream_shape(int64_t D) {
    return MI_SOFTMAX_STREAM && D >= MI_SOFTMAX_STREAM_MIN_D &&
           D <= kOnePassMaxSplits * kOnePassChunk;
}

// Few long rows are split into chunks: aim at ~2048 workgroups (a 19.5 MB
// read-and-reduce measured flat at 5.0-5.5 us from 1216 to 4800 workgroups)
// with chunks of a whole number of tiles -- 4096 elements (two vectors per
// lane) when that still gives >= 1024 workgroups, else 2048.  (Keeping a
// whole row in one workgroup's registers instead measured 2x slower at
// [64, 152064]: a single CU sustains only ~12 GB/s, so 64 busy CUs cannot
// feed HBM.)
int64_t split_tile(int64_t N, int64_t D) { return N * ceil_div(D, 4096) >= 1024 ? 4096 : 2048; }

Plan plan(int64_t N, int64_t D, int64_t& splits, int64_t& chunk) {
    splits = 1;
    chunk = D;
    if (N >= kSplitMaxRows || D < 8192) return stream_shape(D) ? Plan::kStream : Plan::kRow;
    // 256 rows or more that register rows hold (D <= 1024 x 8 x 8): one
    // 1024-lane workgroup per row beat splitting them (measured at [256,
    // 32000] 45% -> 49%, [256, 65536] 49% -> 56%, [384, 16384] 39% -> 47%)
    if (N >= MI_SOFTMAX_REG_ROWS && D <= 1024 * kRegVptMax * 8)
        return stream_shape(D) ? Plan::kStream : Plan::kRow;
    const int64_t tile = split_tile(N, D);
    int64_t sp = ceil_div(kSplitTargetWgs, N);
    if (sp > kMaxSplits) sp = kMaxSplits;
    int64_t tiles = (ceil_div(D, sp) + tile / 2) / tile;  // nearest whole number of tiles
    if (tiles < 1) tiles = 1;
    chunk = tiles * tile;
    splits = ceil_div(D, chunk);
    return Plan::kTwoPass;
}

// Workspace of the two-pass split plan: one (max, sum) pair per chunk.
int64_t twopass_bytes(int64_t N, int64_t D) {
    int64_t splits, chunk;
    if (plan(N, D, splits, chunk) != Plan::kTwoPass) return 0;
    return N * splits * 2 * static_cast<int64_t>(sizeof(float));
}

// mi_softmax_ws_f16's workspace for split rows: the one-pass records of
// every possible row (fixed, so any call shape finds its rows' records in the
// same place), then the two-pass pairs (in-place or unaligned calls).
constexpr int64_t kOnePassRegion = kSplitMaxRows * kRowRecordBytes;
int64_t workspace_bytes(int64_t N, int64_t D) {
    int64_t splits, chunk;
    if (plan(N, D, splits, chunk) == Plan::kStream) return kOnePassRegion;
    const int64_t two = twopass_bytes(N, D);
    return two > 0 ? kOnePassRegion + two : 0;
}

#ifndef MI_SOFTMAX_ONEPASS
#define MI_SOFTMAX_ONEPASS 1
#endif
#ifndef MI_SOFTMAX_REG
#define MI_SOFTMAX_REG 1
#endif

// What a workspace handed to softmax_checked holds.
enum class Ws {
    kPairs,             // the two-pass (max, sum) pairs only (allocating entry point)
    kRecordsThenPairs,  // workspace_bytes() layout (mi_softmax_ws_f16)
    kRecords,           // the one-pass row records only (library-held, stream 0)
};

// Vectors per lane of the one-launch chunks: kOnePassU (8192 elements), or
// half that when the larger chunks would leave fewer than
// MI_SOFTMAX_SMALL_CHUNK_WGS workgroups in the launch (measured +1.4 to +2.2
// points at [200, 32000], [100, 40000], [32, 152064]; 2048 cost [64, 152064]
// 6 points, as its 38 smaller chunks per row no longer fit in one round).
#ifndef MI_SOFTMAX_SMALL_CHUNK_WGS
#define MI_SOFTMAX_SMALL_CHUNK_WGS 1024
#endif
int onelaunch_u(int64_t N, int64_t D) {
    constexpr int kSmall = kOnePassU / 2;
    if (N * ceil_div(D, kOnePassChunk) < MI_SOFTMAX_SMALL_CHUNK_WGS &&
        ceil_div(D, 2048 * kSmall) <= kOnePassMaxSplits)
        return kSmall;
    return kOnePassU;
}
template <bool AM, bool RAGGED, bool ONE>
const void* stream_kernel(int u) {
    return u == kOnePassU
               ? reinterpret_cast<const void*>(softmax_stream_kernel<kOnePassU, AM, RAGGED, ONE>)
               : reinterpret_cast<const void*>(softmax_stream_kernel<kOnePassU / 2, AM, RAGGED, ONE>);
}
// one: the single-round kernel (ragged rows)
const void* onelaunch_kernel(int u, bool am, bool ragged, bool one) {
    if (!ragged) return am ? stream_kernel<true, false, false>(u) : stream_kernel<false, false, false>(u);
    if (one) return am ? stream_kernel<true, true, true>(u) : stream_kernel<false, true, true>(u);
    return am ? stream_kernel<true, true, false>(u) : stream_kernel<false, true, false>(u);
}

// The one-launch form of a row: whole 16-byte vectors at D % 8 == 0 and
// aligned bases, else the row's window, up to 7 elements longer.
bool onelaunch_ragged(const void* x, const void* y, int64_t D) {
    return !(D % 8 == 0 && aligned16(x) && aligned16(y));
}
int64_t onelaunch_len(int64_t D, bool ragged) { return ragged ? D + 7 : D; }

// The one-launch grid: `splits` chunks per row, R row slots (a multiple of
// kXcds, so that chunk_of keeps each slot's chunks on one XCD; slots past
// N - 1 exit at once), 1-D.  `local`: whether polls start on the L2 copy.
struct OneLaunchGrid {
    int u, splits, R, local;
    bool one;
    unsigned blocks() const { return static_cast<unsigned>(splits) * static_cast<unsigned>(R); }
};
OneLaunchGrid onelaunch_grid(int64_t N, int64_t D, bool am, bool ragged) {
    OneLaunchGrid g;
    const int64_t len = onelaunch_len(D, ragged);
    g.u = onelaunch_u(N, len);
    g.splits = static_cast<int>(ceil_div(len, 2048 * g.u));
    // row slots that stay resident next to each other (at most the records;
    // at least 20 = 1280 resident workgroups / 64 chunks)
    auto slots = [&](bool one) {
        const int64_t cap = resident_workgroups(onelaunch_kernel(g.u, am, ragged, one), 256) / g.splits;
        return cap < kSplitMaxRows ? cap : int64_t{kSplitMaxRows};
    };
    // every row in one round when a whole number of groups of that many
    // slots fits (slots past N - 1 idle), else the largest whole number of
    // groups that does (rows in rounds)
    const int64_t all = ceil_div(N < kSplitMaxRows ? N : kSplitMaxRows, kXcds) * kXcds;
    g.one = ragged && N <= all && all <= slots(true);
    if (g.one) {
        g.R = static_cast<int>(all);
    } else {
        const int64_t cap = slots(false);
        const int64_t up = ceil_div(N < cap ? N : cap, kXcds) * kXcds;
        g.R = static_cast<int>(up <= cap ? up : cap / kXcds * kXcds);
    }
    g.local = exchange_test_mode().load() == 0 ? 1 : 0;
    return g;
}

// Whether [N, D] runs as the one-launch form given row records: a split or
// kStream shape, y != x (the fallback re-reads x), rows of x and y with the
// same window, at most 64 chunks per row.
bool onelaunch_ok(const void* x, const void* y, int64_t N, int64_t D, bool am = false) {
    int64_t splits, chunk;
    if (!MI_SOFTMAX_ONEPASS || plan(N, D, splits, chunk) == Plan::kRow) return false;
    if (x == y || !same_window(x, y)) return false;
    const bool ragged = onelaunch_ragged(x, y, D);
    const int64_t len = onelaunch_len(D, ragged);
    const int u = onelaunch_u(N, len);
    const int64_t sp1 = ceil_div(len, 2048 * u);
    return sp1 <= kOnePassMaxSplits &&
           resident_workgroups(onelaunch_kernel(u, am, ragged, false), 256) / sp1 >= 1;
}

// One launch of softmax_stream_kernel (onelaunch_ok holds).
template <bool AM>
int launch_stream(const half_t* x, half_t* y, unsigned char* rec, int32_t* out, int64_t N,
                  int64_t D, hipStream_t s) {
    const bool ragged = onelaunch_ragged(x, y, D);
    const OneLaunchGrid g = onelaunch_grid(N, D, AM, ragged);
    const dim3 gr(g.blocks()), b(256);
#define MI_STREAM(UU, RR, ONE)                                                                  \
    softmax_stream_kernel<UU, AM, RR, ONE><<<gr, b, 0, s>>>(x, y, rec, N, D, g_poll_limit.load(), \
                                                            out, g.splits, g.R, g.local)
    const bool large = g.u == kOnePassU;
    if (!ragged) {
        if (large) MI_STREAM(kOnePassU, false, false);
        else MI_STREAM(kOnePassU / 2, false, false);
    } else if (g.one) {
        if (large) MI_STREAM(kOnePassU, true, true);
        else MI_STREAM(kOnePassU / 2, true, true);
    } else {
        if (large) MI_STREAM(kOnePassU, true, false);
        else MI_STREAM(kOnePassU / 2, true, false);
    }
#undef MI_STREAM
    return launch_status();
}

int softmax_checked(const void* x, void* y, int64_t N, int64_t D, void* ws, int64_t ws_bytes,
                    Ws layout, void* stream) {
    if (N < 0 || D < 0 || ws_bytes < 0) return MI_ERR_INVALID_ARGUMENT;
    if (N == 0 || D == 0) return MI_OK;
    if (!x || !y) return MI_ERR_INVALID_ARGUMENT;
    if (N > kMaxGridX) return MI_ERR_UNSUPPORTED;
    if (!product_fits({N, D, 2})) return MI_ERR_INVALID_ARGUMENT;
    const int64_t bytes = N * D * 2;
    if (x != y && overlaps(x, bytes, y, bytes)) return MI_ERR_ALIASING;
    int64_t splits, chunk;
    const Plan p = plan(N, D, splits, chunk);
    bool onelaunch = layout != Ws::kPairs && onelaunch_ok(x, y, N, D);
    // many long ragged rows need no workspace (a workgroup per row): the
    // one-launch form only with a usable one
    if (onelaunch && p == Plan::kStream && onelaunch_ragged(x, y, D) &&
        (!ws || ws_bytes < kOnePassRegion || reinterpret_cast<uintptr_t>(ws) % 16 != 0 ||
         overlaps(ws, kOnePassRegion, x, bytes) || overlaps(ws, kOnePassRegion, y, bytes)))
        onelaunch = false;
    if (layout == Ws::kRecords && p == Plan::kTwoPass && !onelaunch)
        return MI_ERR_UNSUPPORTED;  // no pairs to fall back on (callers check onelaunch_ok)
    const int64_t need = p == Plan::kRow ? 0
                         : p == Plan::kStream ? (onelaunch ? kOnePassRegion : 0)
                         : layout == Ws::kPairs ? twopass_bytes(N, D)
                         : layout == Ws::kRecords ? kOnePassRegion
                                                  : workspace_bytes(N, D);
    if (need > 0) {
        if (!ws || ws_bytes < need) return MI_ERR_INVALID_ARGUMENT;
        if (overlaps(ws, need, x, bytes) || overlaps(ws, need, y, bytes)) return MI_ERR_ALIASING;
        if (layout != Ws::kPairs && reinterpret_cast<uintptr_t>(ws) % 16 != 0)
            return MI_ERR_INVALID_ARGUMENT;
    }
    const auto* xh = static_cast<const half_t*>(x);
    auto* yh = static_cast<half_t*>(y);
    const hipStream_t s = as_stream(stream);
    const bool vec = D % 8 == 0 && aligned16(x) && aligned16(y);
    if (p == Plan::kRow || (p == Plan::kStream && !onelaunch)) {
        // rows through their aligned windows: up to 7 elements of a
        // neighbour at each end
        const bool ragged = !vec && same_window(x, y);
        const int64_t nv = ragged ? ceil_div(D + 7, 8) : D / 8;
        int G = 0, VPT = 0;
        if (MI_SOFTMAX_REG && (vec || ragged) && reg_shape(nv, G, VPT) &&
            ceil_div(N, (G > 64 ? G : 256) / G) <= kMaxGridX)
            return ragged ? launch_reg_rows<true>(xh, yh, N, D, G, VPT, s)
                          : launch_reg_rows<false>(xh, yh, N, D, G, VPT, s);
        const int64_t want = ceil_div(D, vec ? 8 : 1);
        const int threads = static_cast<int>(ceil_div(want < 1024 ? want : 1024, kWave) * kWave);
        if (vec)
            softmax_row_kernel<8><<<dim3(static_cast<unsigned>(N)), dim3(threads), 0, s>>>(xh, yh, D);
        else
            softmax_row_kernel<1><<<dim3(static_cast<unsigned>(N)), dim3(threads), 0, s>>>(xh, yh, D);
        return launch_status();
    }
    if (onelaunch)
        return launch_stream<false>(xh, yh, static_cast<unsigned char*>(ws), nullptr, N, D, s);
    auto* part = reinterpret_cast<float*>(static_cast<unsigned char*>(ws) +
                                          (layout == Ws::kRecordsThenPairs ? kOnePassRegion : 0));
    const dim3 g(static_cast<unsigned>(splits), static_cast<unsigned>(N));
    if (vec) {
        if (split_tile(N, D) == 4096)
            softmax_partial_kernel<8, 2><<<g, dim3(256), 0, s>>>(xh, part, D, chunk);
        else
            softmax_partial_kernel<8, 1><<<g, dim3(256), 0, s>>>(xh, part, D, chunk);
        softmax_finish_kernel<8><<<g, dim3(256), 0, s>>>(xh, yh, part, D, chunk);
    } else if (same_window(x, y) && D <= kMaxWindowRow) {
        if (split_tile(N, D) == 4096)
            softmax_partial_kernel<8, 2, true><<<g, dim3(256), 0, s>>>(xh, part, D, chunk);
        else
            softmax_partial_kernel<8, 1, true><<<g, dim3(256), 0, s>>>(xh, part, D, chunk);
        softmax_finish_kernel<8, true><<<g, dim3(256), 0, s>>>(xh, yh, part, D, chunk);
    } else {
        softmax_partial_kernel<1, 1><<<g, dim3(256), 0, s>>>(xh, part, D, chunk);
        softmax_finish_kernel<1><<<g, dim3(256), 0, s>>>(xh, yh, part, D, chunk);
    }
    return launch_status();
}

// ---------------------------------------------------------------------------
// Allocation-free entry (mi_softmax_noalloc_f16): the same plans and kernels
// as mi_softmax_ws_f16, with the workspace taken from a file-scope device
// array (`scratch`, below) instead of the caller or the runtime.  Its host
// address comes from hipGetSymbolAddress once per device; it is zero from
// the library's load (the row records must start at zero) and then left to
// each call, which leaves it valid for the next.
// ---------------------------------------------------------------------------
constexpr int64_t kNoAllocPairBytes = 256 * 1024;  // two-pass (max, sum) pairs
constexpr int64_t kScratchBytes = kOnePassRegion + kNoAllocPairBytes;

}  // namespace
}  // namespace mi

// 2,424,832 bytes per GPU, held from the library's load until the process
// ends.  Host code never passes this name to a kernel or a copy: it is a
// host-side stand-in; the device address comes from hipGetSymbolAddress.
// It starts at zero, as the row records must: an object of static storage
// with no initializer is zero-initialized, and in the code object it is
// .bss, which the loader zero-fills on each device when it loads the code.
static __device__ __align__(256) unsigned char scratch[mi::kScratchBytes];

namespace mi {
namespace {

// This device's address of `scratch` (nullptr with *err set when the
// runtime cannot give it), looked up on the device's first call.  Nothing
// is launched here (the array is zero from load; each call leaves it valid
// for the next), so a first call under graph capture records only the
// softmax itself.
void* scratch_for_current_device(int* err) {
    static std::mutex mu;
    static std::map<int, void*> ptrs;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        *err = taken(e);
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(mu);
    auto it = ptrs.find(dev);
    if (it != ptrs.end()) return it->second;
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
        *err = taken(e != hipSuccess ? e : hipErrorInvalidSymbol);
        return nullptr;
    }
    ptrs[dev] = ptr;
    return ptr;
}

}  // namespace
}  // namespace mi

extern "C" int mi_softmax_noalloc_f16(const void* x, void* y, int64_t N, int64_t D,
                                      void* stream) {
    if (N < 0 || D < 0) return MI_ERR_INVALID_ARGUMENT;
    if (N == 0 || D == 0) return MI_OK;
    if (!x || !y) return MI_ERR_INVALID_ARGUMENT;
    const int64_t need = mi::workspace_bytes(N, D);
    if (need > mi::kScratchBytes) return MI_ERR_UNSUPPORTED;  // beyond the array
    if (need == 0)
        return mi::softmax_checked(x, y, N, D, nullptr, 0, mi::Ws::kRecordsThenPairs, stream);
    int err = MI_OK;
    void* ptr = mi::scratch_for_current_device(&err);
    if (!ptr) return err;
    return mi::softmax_checked(x, y, N, D, ptr, mi::kScratchBytes, mi::Ws::kRecordsThenPairs,
                               stream);
}

extern "C" int64_t mi_softmax_workspace_bytes(int64_t N, int64_t D) {
    if (N <= 0 || D <= 0) return 0;
    return mi::workspace_bytes(N, D);
}

extern "C" int mi_softmax_ws_f16(const void* x, void* y, int64_t N, int64_t D, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
    return mi::softmax_checked(x, y, N, D, workspace, workspace_bytes,
                               mi::Ws::kRecordsThenPairs, stream);
}

// Fused softmax + greedy argmax: [fused row records | softmax workspace |
// argmax workspace]; the one-launch fused kernel when the shape takes the
// one-launch softmax, else the two entry points in turn on their parts, each
// 16-byte aligned.
namespace {
constexpr int64_t kFusedRegion = mi::kSplitMaxRows * mi::kRowRecordBytesAM;
static_assert(kFusedRegion % 16 == 0, "the parts are 16-byte aligned");
// (the softmax's pairs are 8 bytes each, an odd number of them for some shapes)
int64_t fused_argmax_offset(int64_t N, int64_t V) {
    return kFusedRegion + mi::ceil_div(mi::workspace_bytes(N, V), 16) * 16;
}
}  // namespace

extern "C" int64_t mi_softmax_argmax_workspace_bytes(int64_t N, int64_t V) {
    if (N <= 0 || V <= 0) return 0;
    return fused_argmax_offset(N, V) + mi_greedy_argmax_workspace_bytes(N, V);
}

namespace {
int softmax_argmax_check(const void* logits, const void* probs, const void* out, int64_t N,
                         int64_t V, const void* workspace, int64_t workspace_bytes) {
    if (N < 0 || V < 0 || workspace_bytes < 0) return MI_ERR_INVALID_ARGUMENT;
    if (N == 0 || V == 0) return MI_OK;
    if (!logits || !probs || !out || !workspace) return MI_ERR_INVALID_ARGUMENT;
    if (N > 65535) return MI_ERR_UNSUPPORTED;  // the argmax grid's rows
    if (!mi::product_fits({N, V, 2})) return MI_ERR_INVALID_ARGUMENT;
    const int64_t need = mi_softmax_argmax_workspace_bytes(N, V);
    if (workspace_bytes < need || reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
        return MI_ERR_INVALID_ARGUMENT;
    const int64_t bytes = N * V * 2;
    if (logits != probs && mi::overlaps(logits, bytes, probs, bytes)) return MI_ERR_ALIASING;
    if (mi::overlaps(workspace, need, logits, bytes) || mi::overlaps(workspace, need, probs, bytes) ||
        mi::overlaps(out, N * 4, logits, bytes) || mi::overlaps(out, N * 4, probs, bytes) ||
        mi::overlaps(out, N * 4, workspace, need))
        return MI_ERR_ALIASING;
    return MI_OK;
}
}  // namespace

bool mi::softmax_argmax_plan(const void* logits, const void* probs, const void* out, int64_t N,
                             int64_t V, const void* workspace, int64_t workspace_bytes,
                             StreamPlan& p) {
    if (softmax_argmax_check(logits, probs, out, N, V, workspace, workspace_bytes) != MI_OK ||
        N <= 0 || V <= 0 || N > kSplitMaxRows || !onelaunch_ok(logits, probs, N, V, true))
        return false;
    p.ragged = onelaunch_ragged(logits, probs, V);
    const int64_t len = onelaunch_len(V, p.ragged);
    p.u = onelaunch_u(N, len);
    p.splits = static_cast<int>(ceil_div(len, 2048 * p.u));
    p.poll_limit = g_poll_limit.load();
    p.local = exchange_test_mode().load() == 0 ? 1 : 0;
    return true;
}

extern "C" int mi_softmax_argmax_ws_f16(const void* logits, void* probs, int32_t* out, int64_t N,
                                        int64_t V, void* workspace, int64_t workspace_bytes,
                                        void* stream) {
    const int st0 = softmax_argmax_check(logits, probs, out, N, V, workspace, workspace_bytes);
    if (st0 != MI_OK || N == 0 || V == 0) return st0;
    auto* ws = static_cast<unsigned char*>(workspace);
    const hipStream_t s = mi::as_stream(stream);
    if (mi::onelaunch_ok(logits, probs, N, V, true))
        return mi::launch_stream<true>(static_cast<const mi::half_t*>(logits),
                                       static_cast<mi::half_t*>(probs), ws, out, N, V, s);
    // separately: argmax first (in place, softmax would overwrite the logits)
    const int64_t sw = mi::workspace_bytes(N, V);
    unsigned char* aw = ws + fused_argmax_offset(N, V);
    const int st = mi_greedy_argmax_ws_f16(logits, N, V, out, aw,
                                           mi_greedy_argmax_workspace_bytes(N, V), stream);
    if (st != MI_OK) return st;
    return mi_softmax_ws_f16(logits, probs, N, V, sw > 0 ? ws + kFusedRegion : nullptr, sw,
                             stream);
}

extern "C" int mi_softmax_f16(const void* x, void* y, int64_t N, int64_t D, void* stream) {
    const int64_t need = (N > 0 && D > 0) ? mi::twopass_bytes(N, D) : 0;
    const hipStream_t s = mi::as_stream(stream);
    // Long split rows on the default stream (every caller in the reference
    // passes 0): one launch, with row records the library holds for stream 0.
    if (x && y && N > 0 && D > 0 && N <= mi::kMaxGridX && mi::onelaunch_ok(x, y, N, D)) {
        void* rec = mi::default_stream_region(mi::kRegionSoftmax, mi::kOnePassRegion, s);
        if (rec)
            return mi::softmax_checked(x, y, N, D, rec, mi::kOnePassRegion, mi::Ws::kRecords,
                                       stream);
    }
    if (need == 0) return mi::softmax_checked(x, y, N, D, nullptr, 0, mi::Ws::kPairs, stream);
    if (!x || !y) return MI_ERR_INVALID_ARGUMENT;
    // Otherwise two launches with a stream-ordered workspace from the
    // device's default pool (concurrent calls on other streams get their
    // own; a fresh pool allocation is not zeroed, which the two-pass form
    // does not need).
    void* ws = nullptr;
    const hipError_t e = hipMallocAsync(&ws, static_cast<size_t>(need), s);
    if (e != hipSuccess) return mi::taken(e);
    const int st = mi::softmax_checked(x, y, N, D, ws, need, mi::Ws::kPairs, stream);
    const int released = mi::taken(hipFreeAsync(ws, s));
    return st != MI_OK ? st : released;
}

extern "C" int mi_softmax_test_poll_limit(int limit) {
    if (limit < 0) return MI_ERR_INVALID_ARGUMENT;
    return mi::g_poll_limit.exchange(limit);
}
