// softmax_stream_body.h -- the statements of one workgroup of the one-launch
// split-row softmax, included into the function that runs them with U, AM,
// RAGGED, ONE and `block` (the workgroup's index in the splits x R grid), x, y, ws,
// N, D, poll_limit, out, splits, R, local in scope.  Text and not a function for
// softmax_stream_kernel's sake: inlined from one, its U = 4 form measured 9.5
// instead of 9.0 us at [64, 152064].
//
// 64 VGPRs, so 8 workgroups per CU (per-lane 32-bit offsets, not 64-bit
// indices: 68 VGPRs and 7 workgroups per CU with them measured 5-10 points
// lower; amdgpu_waves_per_eu(8) also measured ~8 points lower at the same
// 64 VGPRs); wave 0 publishes and polls.
// U vectors per lane: chunks of 2048 * U elements.  AM: the fused softmax +
// greedy argmax pass -- each chunk also forms its best argmax key from the
// registers it already holds, publishes it with its (max, sum), and chunk 0
// writes the row's index to `out` (the fallback scans the row from x).
// (AM: its kernel is held to 5 waves per SIMD, <= 96 VGPRs, so that 1216 chunk workgroups
// of [64, 152064] stay resident at once; the compiler otherwise settles at
// 98 and the grid needs a second round.)
// RAGGED: chunks of the row's aligned window (RowWindow) -- rows of a slot are
// R (a multiple of 8) apart, so one window shape serves all its rounds.
// Against the 2-byte two-launch forms: [64, 151643] 32.1 -> 9.9 us (softmax),
// 37.1 -> 11.0 (with the argmax); aligned [64, 152064] 9.0 / 10.2.
// ONE: every row in one round, so no next row's registers and no conditions
// kept across rounds.  softmax_stream_kernel takes it for ragged rows, 44-68
// VGPRs against 73-96 and, with AM, spills: [64, 151643] softmax + argmax 14.2 ->
// 11.0 us, [200, 32001] softmax 10.2 -> 8.2; aligned rows, which have no such
// conditions, measured slower with it there ([64, 152064] 9.0 -> 9.6 and 10.2 ->
// 11.1 us).  The one-launch step, whose chunks are all resident, takes no other.
    constexpr int64_t kChunk = 2048 * U;
    constexpr int SW = AM ? 4 : 2;
    __shared__ float slots[256 / kWave];
    __shared__ float row_stats[3];  // M, S, fallback flag
    __shared__ uint64_t epoch_sh;
    __shared__ uint64_t kslots[AM ? 256 / kWave : 1];  // per-wave keys (AM)
    __shared__ uint64_t row_key;                        // the row's best key (AM)
    // 1-D grid of splits x R (R a multiple of kXcds): a row slot's chunks
    // share one XCD (row_exchange.h); slots past N-1 have no rows
    int split, slot;
    chunk_of(block, splits, split, slot);
    const int64_t r0 = slot;
    if (r0 >= N) return;  // workgroup-uniform, before any barrier
    unsigned char* rec = ws + r0 * record_bytes<AM>();
    uint64_t* epoch = reinterpret_cast<uint64_t*>(rec);
    uint64_t* sets = reinterpret_cast<uint64_t*>(rec + kRecordHeaderBytes);
    constexpr int64_t kMirror = 2 * SW * kOnePassMaxSplits;  // words from a set to its mirror
    const int64_t K = ONE ? 1 : (N - r0 + R - 1) / R;  // rounds of this row slot (>= 1)
    RowWindow win(x + r0 * D, D);  // RAGGED
    const int64_t shift = RAGGED ? win.shift : 0;
    const int64_t len = RAGGED ? win.nv * 8 : D;
    const int64_t b = split * kChunk;
    const int64_t e = b + kChunk < len ? b + kChunk : len;
    const uint32_t lo = static_cast<uint32_t>(b + threadIdx.x * 8) * 2;
    const int v0 = static_cast<int>(b >> 3) + static_cast<int>(threadIdx.x);
    bool ok[U];
#pragma unroll
    for (int j = 0; j < U; ++j) ok[j] = b + (threadIdx.x + j * 256) * 8 < e;

    if (threadIdx.x == 0)
        epoch_sh = __hip_atomic_load(epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    h8 a[U], n[ONE ? 1 : U];
    lane_load<U>(x + r0 * D - shift, lo, ok, a);
    bool gave_up = false;  // workgroup-uniform: set after the first fallback
    for (int64_t k = 0; k < K; ++k) {
        const int64_t row = r0 + k * R;
        // The guard is always true (256 lanes); written out, it keeps the
        // statistics in a block of their own, which measured 64 VGPRs with
        // no spill against 80 without it.
        if constexpr (RAGGED) {
            // workgroup-uniform: the row's first or last vector.  (win made
            // opaque in each round: its conditions otherwise stay in
            // registers across the rounds, some 250 of them)
            if constexpr (!ONE) asm volatile("" : "+s"(win.shift), "+s"(win.last));
            if (split == 0 || e == len) {
#pragma unroll
                for (int j = 0; j < U; ++j)
                    if (ok[j]) win.mask(v0 + j * 256, a[j]);
            }
        }
        float m = -INFINITY, s = 0.0f;
        if (threadIdx.x < 256) chunk_lane_stats<U>(a, m, s);
        if constexpr (AM) {
            // vectors past the row hold -inf (lane_load), whose key is 0
            const uint64_t kw = wave_max_u64(lane_best_key<U, RAGGED>(a, b, static_cast<int>(shift)));
            if ((threadIdx.x & (kWave - 1)) == 0) kslots[threadIdx.x / kWave] = kw;
        }
        block_merge(m, s, slots);  // barriers: epoch_sh (first round) and kslots visible after
        uint64_t key = 0;
        if constexpr (AM) {
#pragma unroll
            for (int w = 0; w < 256 / kWave; ++w) key = max_u64(key, kslots[w]);
        }
        const uint64_t E = epoch_sh;
        const uint32_t tag = static_cast<uint32_t>(E + 1 + k);
        uint64_t* set = sets + (k & 1) * (SW * kOnePassMaxSplits);
        chunk_publish<AM>(set, kMirror, split, tag, m, s, key);
        if constexpr (!ONE) {
            if (k + 1 < K) lane_load<U>(x + (row + R) * D - shift, lo, ok, n);
        }
        if (gave_up) {
            if (threadIdx.x == 0) row_stats[2] = 1.0f;
        } else if (threadIdx.x < kWave) {
            // only chunk 0 writes the index, so only it polls the key words
            row_poll<AM>(set, kMirror, local != 0, splits, tag, poll_limit, row_stats, &row_key,
                         split == 0);
        }
        __syncthreads();
        float M = row_stats[0], S = row_stats[1];
        const bool fallback = row_stats[2] != 0.0f;
        gave_up = gave_up || fallback;
        if (fallback) row_stats_from_x<RAGGED>(x + row * D, D, M, S, slots);
        if constexpr (AM) {
            if (split == 0) {  // workgroup-uniform: chunk_best has barriers
                uint64_t rk = row_key;
                if (fallback) {
                    rk = RAGGED ? chunk_best<1, 8>(x + row * D, 0, D, kslots)
                                : chunk_best<8, 4>(x + row * D, 0, D, kslots);
                    __syncthreads();  // kslots are written again by the next round
                }
                if (threadIdx.x == 0) out[row] = key_index(rk);
            }
        }
        if (threadIdx.x == 0 && (fallback || (split == 0 && k + 1 == K)))
            __hip_atomic_fetch_max(epoch, fallback ? E + K + 1 : E + K, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        if constexpr (RAGGED && !ONE) asm volatile("" : "+s"(win.shift), "+s"(win.last));
        lane_store<U, RAGGED>(a, y + row * D - shift, lo, ok, M, 1.0f / S, win, v0);
        if constexpr (!ONE) {
            if (k + 1 < K) {
#pragma unroll
                for (int j = 0; j < U; ++j) a[j] = n[j];
            }
        }
    }
