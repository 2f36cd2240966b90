// Paged attention of the 32-bit path on the matrix cores' 32-bit instruction (v_mfma_f32_16x16x4_f32): every kind of row,
// every head size that is a multiple of four up to 256; nothing is rounded to fewer bits.
//
// The keys of a request are cut into segments of 64 from its position 0 on.  A wave takes one segment for a tile of 16 query
// rows that share a key head (the query heads of that group times as many tokens as fit): scores, their maximum, the
// weights exp(s - maximum), their sum and the weighted values of the segment.  Segments are folded in ascending order,
// maximum by maximum.  A segment that a row sees nothing of leaves the fold as it was, so the result for a position depends
// neither on how its request was cut into steps nor on what else is in the batch, bit for bit.  Two ways to fold:
//   whole   a workgroup of four waves owns a tile and walks its segments, four a round, which meet in LDS;
//   split   where few tiles stand before many keys every wave leaves its segment in memory and a second kernel folds.
//
// Nothing is staged: a lane loads 16 bytes of its key's row and of its values' rows, which are its operands of four
// instructions (the weights leave the first product in the layout that the second takes them in), half a segment ahead.
// Bound by the matrix cores with many tokens and by the chain of loads with few.  Before this kernel a wave walked all keys
// of one query head, a key a lane: a step of 8 tokens at contexts up to 512 (16 heads over 8 of 128) 472 us, a prompt of
// 700 tokens 660 us.
#include <cfloat>

#include "common.hpp"

typedef float af_f32x4 __attribute__((ext_vector_type(4)));

#define AF_SEGMENT 64

// The token tile `slot` of a step whose requests bring q_len[s] tokens, `tile` tokens a tile: its request and its first token
// there.  Requests without context are padding and have none.  The last tiles of a request, which see most keys, come first.
__device__ __forceinline__ bool af_find_tile(int slot, const int* __restrict__ q_len, const int* __restrict__ ctx_len,
                                             int num_seqs, int tile, int& seq, int& first) {
    const int lane = threadIdx.x % PL_WAVE;
    int before = 0;
    for (int base = 0; base < num_seqs; base += PL_WAVE) {
        const int s = base + lane;
        const int mine = s < num_seqs && q_len[s] > 0 && ctx_len[s] > 0 ? (q_len[s] + tile - 1) / tile : 0;
        int through = mine;
#pragma unroll
        for (int off = 1; off < PL_WAVE; off <<= 1) {
            const int other = __shfl_up(through, off, PL_WAVE);
            if (lane >= off) through += other;
        }
        const int total = __builtin_amdgcn_readfirstlane(__shfl(through, PL_WAVE - 1, PL_WAVE));
        if (slot < before + total) {
            const int at = slot - before;
            const int l = __ffsll(static_cast<unsigned long long>(__ballot(at >= through - mine && at < through))) - 1;
            seq = __builtin_amdgcn_readfirstlane(base + l);
            first = __builtin_amdgcn_readfirstlane((__shfl(through, l, PL_WAVE) - 1 - at) * tile);
            return true;
        }
        before += total;
    }
    return false;
}

// One segment joins what lies before it.
__device__ __forceinline__ void af_fold(float& m, float& l, float& kept, float& joins, float seg_m, float seg_l) {
    const float top = fmaxf(m, seg_m);
    kept = expf(m - top);               // (exp(-inf) = 0: nothing before)
    joins = expf(seg_m - top);
    l = fmaf(l, kept, seg_l * joins);   // (spelled out: the two kernels that fold have to round alike)
    m = top;
}

// What the read-out is multiplied by once every segment has joined: one over the denominator, a sink's term in it, and the gate.
__device__ __forceinline__ float af_finish(float m, float l, int row, int head, const float* sinks, const PlAttentionMore& more) {
    float scale = 1.f;
    if (sinks != nullptr) {
        const float sink = sinks[head], top = fmaxf(m, sink);
        scale = expf(m - top);
        l = fmaf(l, scale, expf(sink - top));
    }
    if (!(l > 0.f) && l == l) return 0.f;           // (no key seen; a sum that is no number stays none)
    return scale / l * (more.gate != nullptr ? pl_head_gate(more, row, head) : 1.f);
}

// DT: stretches of 64 values of a head.  FULL: the head has all 64 DT of them.
template <int DT, bool FULL>
__global__ void __launch_bounds__(4 * PL_WAVE, DT <= 2 ? 2 : 1)
attention_f32_kernel(const float* __restrict__ q, int q_stride, float* __restrict__ out, const int* __restrict__ q_start,
                     const int* __restrict__ q_len, const int* __restrict__ ctx_len, int num_seqs,
                     const int* __restrict__ block_table, int max_blocks, int block_size, const float* k_pool,
                     const float* v_pool, int nq, int nkv, int d, float scale, int window, const float* __restrict__ sinks,
                     const float* __restrict__ slopes, PlAttentionMore more, int group, int tokens, int head_tiles, int shares,
                     float* __restrict__ part_acc, float* __restrict__ part_ml, int max_segments) {
    constexpr int PITCH = 64 * DT + 4;
    __shared__ __attribute__((aligned(16))) float seg_acc[4][16 * PITCH];
    __shared__ float seg_ml[4][16][2];

    const int lane = threadIdx.x % PL_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PL_WAVE);
    const int r = lane % 16, c = lane / 16;
    int work = blockIdx.x;
    const int share = work % shares;
    work /= shares;
    const int head_tile = work % head_tiles;
    work /= head_tiles;
    const int kvh = work % nkv;
    int seq, q0;
    if (!af_find_tile(work / nkv, q_len, ctx_len, num_seqs, tokens, seq, q0)) return;      // (the whole workgroup)

    // the lane's query row
    const int count = q_len[seq], start = ctx_len[seq] - count, row0 = q_start[seq];
    const int token = q0 + (group <= 16 ? r / group : 0);
    const int in_group = group <= 16 ? r % group : head_tile * 16 + r;
    const bool live = (group <= 16 ? r / group < tokens : in_group < group) && token < count;
    const int head = kvh * group + (live ? in_group : 0);
    const int row = row0 + (live ? token : q0);
    const int pos = live ? start + token : -1;
    const int first = live ? pl_first_visible(pos, window) : 0;
    const float slope = slopes != nullptr ? slopes[head] : 0.f;
    af_f32x4 qv[4 * DT];
#pragma unroll
    for (int m = 0; m < 4 * DT; ++m) {
        const int col = 16 * m + 4 * c;
        qv[m] = af_f32x4{0.f, 0.f, 0.f, 0.f};
        if (live && (FULL || col < d))
            qv[m] = *reinterpret_cast<const af_f32x4*>(q + static_cast<size_t>(row) * q_stride + static_cast<size_t>(head) * d + col);
    }

    // the tile's segments: those of the kept keys in front of the window, then the window's
    const int low = start + q0, high = start + min(q0 + tokens, count) - 1;
    const int from = pl_first_visible(low, window) / AF_SEGMENT;
    const int front = more.keep > 0 ? min((more.keep + AF_SEGMENT - 1) / AF_SEGMENT, from) : 0;
    const int segments = front + high / AF_SEGMENT - from + 1;
    const int* table = block_table + static_cast<size_t>(seq) * max_blocks;

    // whole: what the thread folds, four values of each stretch of 64 of row threadIdx.x / 16
    float fold_m = -INFINITY, fold_l = 0.f;
    af_f32x4 folded[DT];
#pragma unroll
    for (int j = 0; j < DT; ++j) folded[j] = af_f32x4{0.f, 0.f, 0.f, 0.f};

    for (int base = share * 4; base < segments; base += shares * 4) {
        const int index = base + wave;
        const int seg = index < front ? index : from + index - front;
        float top = -INFINITY, sum = 0.f;
        af_f32x4 acc[4 * DT];
#pragma unroll
        for (int i = 0; i < 4 * DT; ++i) acc[i] = af_f32x4{0.f, 0.f, 0.f, 0.f};
        if (index < segments) {
            const int key0 = seg * AF_SEGMENT;
            int slot = -1;                                   // of key key0 + lane
            if (key0 + lane <= high) {
                const int blk = table[(key0 + lane) / block_size];
                if (blk >= 0) slot = blk * block_size + (key0 + lane) % block_size;
            }
            // 16 keys a tile.  A key that is not there is read from the pool's first row and its score replaced; its
            // values are cleared below.
            af_f32x4 buf[2][4 * DT];
            auto ask_keys = [&](int kt, af_f32x4 (&b)[4 * DT]) {
                const int s = __shfl(slot, kt * 16 + r, PL_WAVE);
                const float* at = k_pool + (static_cast<size_t>(max(s, 0)) * nkv + kvh) * d;
#pragma unroll
                for (int m = 0; m < 4 * DT; ++m) {
                    const int col = 16 * m + 4 * c;
                    b[m] = *reinterpret_cast<const af_f32x4*>(at + (FULL || col < d ? col : 0));
                }
            };
            auto ask_values = [&](int kt, af_f32x4 (&b)[4 * DT]) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int s = __shfl(slot, kt * 16 + c * 4 + t, PL_WAVE);
                    const float* at = v_pool + (static_cast<size_t>(max(s, 0)) * nkv + kvh) * d;
#pragma unroll
                    for (int j = 0; j < DT; ++j) {
                        const int col = 64 * j + 4 * r;
                        b[t * DT + j] = *reinterpret_cast<const af_f32x4*>(at + (FULL || col < d ? col : 0));
                    }
                }
            };
            af_f32x4 score[4];                               // [tile of 16 keys][key 4 c + t]: one of the lane's row
            ask_keys(0, buf[0]);
            ask_keys(1, buf[1]);
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                __builtin_amdgcn_sched_barrier(0);
                af_f32x4 (&b)[4 * DT] = buf[kt % 2];
                af_f32x4 even = {0.f, 0.f, 0.f, 0.f}, odd = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int m = 0; m < 4 * DT; ++m) {
                    if (!FULL) {                             // (columns past the head's: the query's are zeros)
#pragma unroll
                        for (int i = 0; i < 4; ++i) b[m][i] = 16 * m + 4 * c < d ? b[m][i] : 0.f;
                    }
#pragma unroll
                    for (int i = 0; i < 4; i += 2) {
                        even = __builtin_amdgcn_mfma_f32_16x16x4f32(b[m][i], qv[m][i], even, 0, 0, 0);
                        odd = __builtin_amdgcn_mfma_f32_16x16x4f32(b[m][i + 1], qv[m][i + 1], odd, 0, 0, 0);
                    }
                }
                score[kt] = even + odd;
                if (kt < 2) ask_keys(kt + 2, b);
                else ask_values(kt - 2, b);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int key = key0 + kt * 16 + c * 4 + t;
                    const bool there = __shfl(slot, kt * 16 + c * 4 + t, PL_WAVE) >= 0;
                    float s = score[kt][t] * scale;
                    if (more.cap > 0.f) s = more.cap * tanhf(s / more.cap);
                    s -= slope * static_cast<float>(pos - key);
                    const bool seen = there && key <= pos && (key >= first || key < more.keep);
                    score[kt][t] = seen ? s : -INFINITY;
                    top = fmaxf(top, score[kt][t]);
                }
            }
            top = fmaxf(top, __shfl_xor(top, 16, PL_WAVE));
            top = fmaxf(top, __shfl_xor(top, 32, PL_WAVE));
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    // (a score of -inf is a key that the row does not see, or one that weighs nothing)
                    score[kt][t] = score[kt][t] == -INFINITY ? 0.f : expf(score[kt][t] - top);
                    sum += score[kt][t];
                }
            sum += __shfl_xor(sum, 16, PL_WAVE);
            sum += __shfl_xor(sum, 32, PL_WAVE);
            if (sum != sum) top = fmaxf(top, -FLT_MAX);     // (scores that are all NaN: not a segment without keys)
            // Values of keys that are not there count as zeros.  Keys that some rows of the tile see and others do not meet
            // weights of zero there, which has to give zero: an infinity or a NaN among such a segment's values stays out
            // of the products and joins the rows that see it one by one.
            const bool ragged = key0 + AF_SEGMENT - 1 > low || key0 < pl_first_visible(high, window);
            bool odd_values = false;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                __builtin_amdgcn_sched_barrier(0);
                af_f32x4 (&b)[4 * DT] = buf[kt % 2];
                if (ragged) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const bool there = __shfl(slot, kt * 16 + c * 4 + t, PL_WAVE) >= 0;
#pragma unroll
                        for (int j = 0; j < DT; ++j)
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const float v = b[t * DT + j][i];
                                const bool plain = fabsf(v) < INFINITY;
                                odd_values |= there && !plain;
                                b[t * DT + j][i] = there && plain ? v : 0.f;
                            }
                    }
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int j = 0; j < DT; ++j)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            acc[j * 4 + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[t * DT + j][i], score[kt][t], acc[j * 4 + i], 0, 0, 0);
                if (kt < 2) ask_values(kt + 2, b);
            }
            if (__any(odd_values)) {
#pragma clang loop unroll(disable)
                for (int k = 0; k < AF_SEGMENT; ++k) {
                    const int s = __shfl(slot, k, PL_WAVE), key = key0 + k;
                    float weight = 0.f;
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const float of = __shfl(score[e / 4][e % 4], k % 16 / 4 * 16 + r, PL_WAVE);
                        if (k / 16 * 4 + k % 4 == e) weight = of;
                    }
                    const bool seen = s >= 0 && key <= pos && (key >= first || key < more.keep);
                    const float* at = v_pool + (static_cast<size_t>(max(s, 0)) * nkv + kvh) * d;
#pragma unroll
                    for (int j = 0; j < DT; ++j)
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const int col = 64 * j + 16 * c + e;
                            const float v = at[FULL || col < d ? col : 0];
                            if (seen && !(fabsf(v) < INFINITY)) acc[j * 4 + e % 4][e / 4] = fmaf(weight, v, acc[j * 4 + e % 4][e / 4]);
                        }
                }
            }
        }
        // The lane holds, of its row, 16 values of every stretch of 64: value 64 j + 16 c + 4 e + i is acc[4 j + i][e].
        if (part_acc != nullptr) {
            if (index < segments && live && seg < max_segments) {
                const size_t at = (static_cast<size_t>(row) * nq + head) * max_segments + seg;
                if (c == 0) {
                    part_ml[2 * at] = top;
                    part_ml[2 * at + 1] = sum;
                }
#pragma unroll
                for (int j = 0; j < DT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int col = 64 * j + 16 * c + 4 * e;
                        if (FULL || col < d)
                            *reinterpret_cast<af_f32x4*>(part_acc + at * d + col) =
                                af_f32x4{acc[4 * j][e], acc[4 * j + 1][e], acc[4 * j + 2][e], acc[4 * j + 3][e]};
                    }
            }
            continue;
        }
        __syncthreads();                                     // (everybody has folded the round before)
        if (c == 0) {
            seg_ml[wave][r][0] = top;
            seg_ml[wave][r][1] = sum;
        }
#pragma unroll
        for (int j = 0; j < DT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                *reinterpret_cast<af_f32x4*>(&seg_acc[wave][r * PITCH + 64 * j + 16 * c + 4 * e]) =
                    af_f32x4{acc[4 * j][e], acc[4 * j + 1][e], acc[4 * j + 2][e], acc[4 * j + 3][e]};
        __syncthreads();
        const int mine = threadIdx.x / 16;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float seg_m = seg_ml[s][mine][0];
            if (seg_m == -INFINITY) continue;
            float kept, joins;
            af_fold(fold_m, fold_l, kept, joins, seg_m, seg_ml[s][mine][1]);
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                const af_f32x4 a = *reinterpret_cast<const af_f32x4*>(&seg_acc[s][mine * PITCH + 64 * j + threadIdx.x % 16 * 4]);
#pragma unroll
                for (int i = 0; i < 4; ++i) folded[j][i] = fmaf(folded[j][i], kept, a[i] * joins);
            }
        }
    }
    if (part_acc != nullptr) return;

    // (the row that the thread folded; lane r of its wave holds what is known of row r)
    const int mine = threadIdx.x / 16;
    const int my_row = __shfl(row, mine, PL_WAVE), my_head = __shfl(head, mine, PL_WAVE);
    if (!__shfl(static_cast<int>(live), mine, PL_WAVE)) return;
    const float by = af_finish(fold_m, fold_l, my_row, my_head, sinks, more);
    float* to = out + (static_cast<size_t>(my_row) * nq + my_head) * d;
#pragma unroll
    for (int j = 0; j < DT; ++j) {
        const int col = 64 * j + threadIdx.x % 16 * 4;
        if (FULL || col < d) *reinterpret_cast<af_f32x4*>(to + col) = by == 0.f ? af_f32x4{0.f, 0.f, 0.f, 0.f} : folded[j] * by;
    }
}

// A wave a token and head: the segments that it sees, in ascending order.
__global__ void __launch_bounds__(PL_WAVE)
attention_f32_merge_kernel(float* __restrict__ out, const int* __restrict__ positions, const float* __restrict__ part_acc,
                           const float* __restrict__ part_ml, int max_segments, int nq, int d, int window,
                           const float* __restrict__ sinks, PlAttentionMore more) {
    const int row = blockIdx.x, head = blockIdx.y;
    const int pos = positions[row];
    if (pos < 0) return;
    const int first = pl_first_visible(pos, window), from = first / AF_SEGMENT;
    const int front = more.keep > 0 ? min((min(more.keep, first) + AF_SEGMENT - 1) / AF_SEGMENT, from) : 0;
    const int segments = front + pos / AF_SEGMENT - from + 1;
    const size_t base = (static_cast<size_t>(row) * nq + head) * max_segments;
    const int col = threadIdx.x * 4;
    float* const to = out + (static_cast<size_t>(row) * nq + head) * d + col;
    if (pos / AF_SEGMENT >= max_segments) {             // (a context longer than the launch was told: there is no room with its last segments)
        if (col < d) *reinterpret_cast<af_f32x4*>(to) = af_f32x4{NAN, NAN, NAN, NAN};
        return;
    }
    float m = -INFINITY, l = 0.f;
    af_f32x4 a = {0.f, 0.f, 0.f, 0.f};
    constexpr int AHEAD = 4;
    for (int i0 = 0; i0 < segments; i0 += AHEAD) {
        float seg_m[AHEAD], seg_l[AHEAD];
        af_f32x4 part[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int i = min(i0 + u, segments - 1);
            const size_t at = base + (i < front ? i : from + i - front);
            seg_m[u] = part_ml[2 * at];
            seg_l[u] = part_ml[2 * at + 1];
            part[u] = *reinterpret_cast<const af_f32x4*>(part_acc + at * d + min(col, d - 4));
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (i0 + u >= segments || seg_m[u] == -INFINITY) continue;
            float kept, joins;
            af_fold(m, l, kept, joins, seg_m[u], seg_l[u]);
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = fmaf(a[i], kept, part[u][i] * joins);
        }
    }
    const float by = af_finish(m, l, row, head, sinks, more);
    if (col < d) *reinterpret_cast<af_f32x4*>(to) = by == 0.f ? af_f32x4{0.f, 0.f, 0.f, 0.f} : a * by;
}

// Whether the kernel takes heads of this size over these tensors (all rows are then whole groups of four aligned values).
extern "C" int pl_paged_attention_f32_applies(const void* q, int q_stride, const void* out, const void* k_pool, const void* v_pool, int d) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(k_pool) |
                           reinterpret_cast<uintptr_t>(v_pool);
    return d > 0 && d <= 256 && d % 4 == 0 && q_stride % 4 == 0 && bits % 16 == 0;
}

// Request s of the first `num_seqs` brings the rows q_start[s] .. q_start[s] + q_len[s] - 1 at the positions that end in
// ctx_len[s] - 1.  `part_acc` [n, nq, max_segments, d] and `part_ml` [n, nq, max_segments, 2]: room for the segments of every
// row where they are folded by a second kernel (rows at positions behind them come out as NaN); null: folded in the first.
extern "C" int pl_paged_attention_f32(const float* q, int q_stride, float* out, const int* positions, const int* q_start,
                                      const int* q_len, const int* ctx_len, int num_seqs, const int* block_table, int max_blocks,
                                      int block_size, const float* k_pool, const float* v_pool, int n, int nq, int nkv, int d,
                                      float scale, int window, const float* sinks, const float* slopes, float cap, int keep,
                                      const float* gate, int gate_stride, float* part_acc, float* part_ml, int max_segments,
                                      hipStream_t stream) {
    PL_REQUIRE(cap >= 0.f && keep >= 0 && (gate == nullptr || gate_stride >= nq), "attention: a cap of %g, %d first keys kept, gates in rows of %d",
               static_cast<double>(cap), keep, gate_stride);
    PL_REQUIRE(keep == 0 || window >= 0, "attention: first keys kept beside blocks of positions");
    PL_REQUIRE(pl_paged_attention_f32_applies(q, q_stride, out, k_pool, v_pool, d), "attention in 32-bit: heads of %d, query rows of %d", d, q_stride);
    PL_REQUIRE(nq > 0 && nkv > 0 && nq % nkv == 0 && nq <= 65535, "attention: %d query heads over %d key heads", nq, nkv);
    PL_REQUIRE(block_size > 0 && max_blocks > 0 && q_stride >= nq * d && num_seqs >= 0,
               "attention: block size %d, %d blocks a row, query stride %d", block_size, max_blocks, q_stride);
    PL_REQUIRE((part_acc == nullptr) == (part_ml == nullptr) && (part_acc == nullptr || max_segments > 0), "attention: room for %d segments", max_segments);
    if (n <= 0 || num_seqs == 0) return 0;
    const PlAttentionMore more{cap, keep, gate, gate_stride};
    const int group = nq / nkv;
    const int tokens = group <= 16 ? 16 / group : 1, head_tiles = pl_ceil_div(group, 16);
    const int slots = n < n / tokens + num_seqs ? n : n / tokens + num_seqs;
    const int shares = part_acc != nullptr ? pl_ceil_div(max_segments, 4) : 1;
    const long blocks = static_cast<long>(slots) * nkv * head_tiles * shares;
    PL_REQUIRE(blocks < (1L << 31), "attention: %ld workgroups are more than one launch covers", blocks);
#define PL_AF_LAUNCH(DT, FULL)                                                                                           \
    attention_f32_kernel<DT, FULL><<<static_cast<unsigned>(blocks), 4 * PL_WAVE, 0, stream>>>(                           \
        q, q_stride, out, q_start, q_len, ctx_len, num_seqs, block_table, max_blocks, block_size, k_pool, v_pool, nq,    \
        nkv, d, scale, window, sinks, slopes, more, group, tokens, head_tiles, shares, part_acc, part_ml, max_segments)
    if (d == 64) PL_AF_LAUNCH(1, true);
    else if (d < 64) PL_AF_LAUNCH(1, false);
    else if (d == 128) PL_AF_LAUNCH(2, true);
    else if (d < 128) PL_AF_LAUNCH(2, false);
    else if (d == 256) PL_AF_LAUNCH(4, true);
    else PL_AF_LAUNCH(4, false);
#undef PL_AF_LAUNCH
    PL_CHECK_LAUNCH("attention_f32");
    if (part_acc != nullptr) {
        attention_f32_merge_kernel<<<dim3(n, nq), PL_WAVE, 0, stream>>>(out, positions, part_acc, part_ml, max_segments, nq, d, window, sinks, more);
        PL_CHECK_LAUNCH("attention_f32_merge");
    }
    return 0;
}
