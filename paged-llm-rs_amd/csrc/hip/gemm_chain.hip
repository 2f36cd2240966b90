// The products behind a layer's attention for few rows (n <= 64), bfloat16 weights in strips, as ONE launch:
//
//   stage 0  mid    = stream + rows . w_out^T                 (the mixer's output projection)
//   stage 1  hidden = act(norm2(mid) . gate^T) * (norm2(mid) . up^T)
//   stage 2  out    = mid + hidden . w_down^T
//   stage 3  after  = norm1'(out) . w_after^T                 (the next layer's first projection; optional)
//   stage 4  the next layer's attention of single tokens over it (optional, for few workgroups; attention_decode.hpp)
//
// A launch of its own takes a stage 5.2 us (one row of a stream of 1,024; weights of 4 to 12 MB that memory gives in
// 0.8 to 2.3 us): the boundary between two kernels, weights that are asked for only then, and the drain.  Here the
// workgroups of all stages are in one grid, 16 columns each.  A workgroup asks for its weights first, into registers, and
// then looks for its input; so the weights of a stage travel while the stages before it work, and what is left between
// two stages is one trip of the rows through memory.  It keeps its weights for all its tiles of 16 rows, and a stage begins with a
// tile as soon as the stage before is done with that tile; from 17 rows on the tiles of rows are dealt to two workgroups
// (one / two, us a layer: 24 rows 23.2 / 21.2, 64 rows 36.3 / 30.5; one for each tile of rows 64 rows 33.1).  Four products of the 0.6B shape, 28
// layers, weights from memory, us a layer, four launches / one: 1 row 20.8 / 15.0, 8 rows 22.8 / 15.9, 15 rows 25.3 / 18.5, 16 rows 24.8 / 18.4,
// 32 rows 26.2 / 21.4, 48 rows 29.2 / 27.3, 64 rows 31.0 / 28.6.
//
// With the next layer's attention as the last stage, what is left of its launch (11.5 us of one token, 12.3 of eight, positions, pages and keys one
// behind the other, and the boundary) is what stands behind its rows of q: one trip, the arithmetic of keys that are there, the meeting of the shares.
// When a stage's workgroups have their rows and end, us from the launch's begin (one token, medians): output projection 4.2, 5.7; gate/up 7.5, 8.9;
// down 10.7, 11.3; q/k/v 12.5, 13.8; attention 15.2, 19.4 (keys weighed 17.1, shares written 18.6).  A layer of a step, chain and attention apart /
// together: one token at 512 26.2 / 21, eight 28.2 / 25.
//
// How a stage learns that its rows are there.  What the stages leave begins as words of all ones (PL_MISSING), and every word
// is written once, past the XCD's L2 (relaxed atomics of device scope, as in pl_share): a word that differs is the value.
// A result that happens to be all ones (a NaN, or a pair of them) is written as another NaN.  There is no counter: one that all
// workgroups of a stage add to costs 2 us a stage (20.8 us a layer, no gain at all).
// The rows between stages lie in the order in which the next stage's lanes load them ("laid", see cn_laid): 8 rows as
// [row][column] cost 18.5 us a layer where 15.6 were taken laid, since a load then touches a line a row twice.
//
// Nothing waits for ever.  A workgroup looks `looks` times for a tile of rows, and once more at all of them; if its rows are not there by then (workgroups are started in the order
// of their numbers, what they wait for before them or, where the attention stands in front, beside them on the other half of the chip; but another launch may hold the compute units they need), it finds
// out which places of the earlier stages are missing, stage by stage, works them out, and then its own: the same arithmetic, so the same bits to the same words, whoever writes
// them first.  Workgroups that miss the same begin at unlike places and look again behind each, so what is missing is dealt out among them (us a
// launch in which nobody may wait, 0.6B shape: 1 row 48, 8 rows 100; each by itself working all earlier stages out 1,250).  What is known to be there is taken without a
// look, so that way ends whatever anybody else does.
//
// Beside others on the chip (us a step of eight tokens at a context of 512, launches apart / chains): alone 1,093 / 811, two streams 1,365 / 1,060, three
// 1,665 / 1,662, four 2,010 / 3,000, where the attention's workgroups wait on half of the chip for each of them (chains without attention 2,080); one
// token alone 985 / 676, four streams 1,475 / 1,300; two prompts of 64 rows in two processes 1,690 / 1,890, where one alone is 1,208 / 1,107.  From three processes on
// the hardware gives the chip, compute die by compute die, to some of them at a time: then chains wait for workgroups that are not on it (four processes of eight
// tokens each, all their steps in two seconds 1,575 / 1,240 to 1,770; three of 64 rows 1,845 / 700).
//
// The arithmetic is gemm_skinny's for one tile of rows, to the same bits: K in as many stretches as that launch has waves (a
// wave here takes up to four of them, each an accumulator of its own), the stretches' tiles added in their order.  As there, the norms in front
// of stages 1 and 3 are taken from the 32-bit stream below CN_HANDED rows, and from there on handed forward: the stage that adds
// into the stream leaves bf16(stream * gain) and the sums of squares of its 16 columns.  (Of more than 32 rows over many columns the launches apart are
// another kernel, which adds its sums in another order: then a result here is the neighbouring bfloat16 now and then.)
#include "attention_decode.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

#define CN_ADD 0        // y = old + x . w^T, 32-bit
#define CN_ADD_HANDS 1  // the same, and what the next norm's product takes of it
#define CN_GATED 2      // y = act(norm(x) . gate^T) * (norm(x) . up^T), bfloat16
#define CN_STORE 3      // y = norm(x) . w^T, bfloat16
#define CN_GATED_TAKES 4    // the same of rows that a CN_ADD_HANDS left
#define CN_STORE_TAKES 5
#define CN_ATTEND 6     // the next layer's attention of single tokens, over the rows that CN_STORE left
#define CN_STAGES 5
#define CN_WAVES 4
#define CN_STRETCHES 16     // of K, at most
#define CN_ROWS 64
#define CN_HANDED 16        // rows from which on norms are handed forward
#define CN_RUN 4            // sums of squares a lane adds up: sixteen lanes a row, a stream of 1,024

struct cn_stage_t {
    const void* x;          // CN_ADD*: bfloat16 rows; CN_GATED, CN_STORE: the 32-bit stream, laid; *_TAKES: bfloat16 rows, laid
    const bf16_t* w;        // in strips
    void* y;
    const float* old;       // CN_ADD*
    const float* gain;      // of the norm in front (CN_GATED, CN_STORE) or behind (CN_ADD_HANDS)
    const float* squares;   // *_TAKES: [n, K / 16]
    bf16_t* hand_x;         // CN_ADD_HANDS: [n, N], laid, ...
    float* hand_squares;    // ... and [n, N / 16]
    float eps;
    int N, K;               // columns of y
    int per, stretches;     // K steps of a stretch; stretches of K
    int kind;
    int first, tiles;       // its workgroups: tiles of 16 columns times parts
    int parts;              // workgroups that the tiles of 16 rows are dealt to
    int x_laid, old_laid, y_laid;
    int y_missing;          // rows that another stage waits for, but not laid
};
struct cn_chain_t {
    cn_stage_t s[CN_STAGES];
    int stages, n, act, looks;
};
// The next layer's attention (ad_attend's arguments).
struct cn_attend_t {
    const bf16_t* q;
    int q_stride;
    bf16_t* out;
    float *part_acc, *part_ml;
    const int *positions, *seq_of, *block_table;
    int max_blocks, block_size;
    bf16_t *k_pool, *v_pool;
    int nq, nkv, d;
    float scale_log2e;
    int window, splits, g;
    uint32_t splits_magic;
    ad_fuse_t fuse;
    int* arrivals;
};
struct cn_nothing_t {};
template <bool ATTENDS>
using cn_attend_of = typename std::conditional<ATTENDS, cn_attend_t, cn_nothing_t>::type;
// (where a kernel's second argument stands)
constexpr size_t CN_ATTEND_AT = (sizeof(cn_chain_t) + alignof(cn_attend_t) - 1) / alignof(cn_attend_t) * alignof(cn_attend_t);
#define CN_HEADS 2          // query heads a workgroup of the attention
#define CN_KEYS 8           // keys a lane group asks for at once (as in a launch of its own of at most a workgroup a compute unit, to the same bits)
#define CN_ATTEND_LOOKS 128 // after which a workgroup of the attention sees to its token's row itself (some 0.15 ms; with 64 and 256 four streams took the same or more)
#define CN_SHARE 256        // keys of a share of the context, at most: two rounds

// Where value (row, col) of a laid [n, width] tensor stands: 16 rows after 16 rows, in these K step by K step of 32 columns, in the order of the
// lanes that load it (8 columns a group, 16 bytes a load: 32-bit rows in two halves).
__device__ __forceinline__ uint32_t cn_laid(int row, int col, int n, int width, bool wide) {
    const int begin = row / 16 * 16, rows = min(16, n - begin);
    const int step = col / 32, group = col % 32 / 8;
    return begin * width
           + (wide ? ((step * 8 + col % 8 / 4 * 4 + group) * rows + row % 16) * 4 + col % 4 : ((step * 4 + group) * rows + row % 16) * 8 + col % 8);
}

// Two neighbouring columns' values, four lanes apart, as the even column's word.
__device__ __forceinline__ uint32_t cn_pair(float f) {
    const uint32_t half = bf16_bits_from_float(f);
    return half | static_cast<uint32_t>(__shfl_down(half, 4, PL_WAVE)) << 16;
}

// One tile of 16 columns of one stage, all rows.  V stretches of K a wave, of at most S K steps of 32.  trust: this workgroup knows that the rows
// are there.  FULL: every stretch of the 4 V has S steps (asking that of each load costs 8 rows 1.4 us a layer).  Returns whether the tile is done (false: its rows were not there in time), the same for
// all threads.
template <int KIND, int V, int S, bool FULL>
__device__ __forceinline__ bool cn_tile(const cn_chain_t& a, const cn_stage_t& s, int stage, int place, bool trust, float* red, float* ssq_lds,
                                        int* late) {
    const int tile = s.parts == 1 ? place : place / s.parts, part = place - tile * s.parts;
    constexpr bool ADD = KIND == CN_ADD || KIND == CN_ADD_HANDS;
    constexpr bool GATED = KIND == CN_GATED || KIND == CN_GATED_TAKES;
    constexpr bool NORM = KIND == CN_GATED || KIND == CN_STORE;
    constexpr bool TAKES = KIND == CN_GATED_TAKES || KIND == CN_STORE_TAKES;
    constexpr int BT = GATED ? 2 : 1;
    constexpr int PARTS = NORM ? 2 : 1;        // loads of 16 bytes for a lane's 8 values
    const int lane = threadIdx.x % PL_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PL_WAVE);
    const int c = lane % 16, g = lane / 16;
    const int K = s.K, steps = K / 32;
    const bool asks = stage > 0 && !trust;

    // the weights first: they come from memory and depend on nothing (steps that a stretch does not have are read past a
    // buffer's end, which gives zeros, and so are rows that are not there)
    auto step_of = [&](int u) { return FULL ? wave * V * S + u : (wave * V + u / S) * s.per + u % S; };
    auto is_step = [&](int u) { return FULL || (u % S < s.per && step_of(u) < steps); };
    bf16x8 w[BT][V * S];
    float gn[NORM ? S : 1][8];
#pragma unroll
    for (int b = 0; b < BT; ++b) {
        const __amdgpu_buffer_rsrc_t strip =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(s.w) + static_cast<size_t>(b * (s.N / 16) + tile) * 16 * K, 0, 32u * K, 0x00027000);
#pragma unroll
        for (int u = 0; u < V * S; ++u)
            w[b][u] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(strip, is_step(u) ? lane * 16u : CN_NOWHERE, is_step(u) ? step_of(u) * 1024 : 0, 0));
    }
    if constexpr (NORM) {
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const f32x8 v = *reinterpret_cast<const f32x8*>(s.gain + (is_step(u) ? step_of(u) : 0) * 32 + g * 8);
#pragma unroll
            for (int e = 0; e < 8; ++e) gn[u][e] = v[e];
        }
    }
    // the element of a tile that this thread finishes
    const int t = threadIdx.x;
    const int tile_row = t / 64 * 4 + t % 4, col = tile * 16 + t / 4 % 16;
    float hand_gain = 0.f;
    if constexpr (KIND == CN_ADD_HANDS) hand_gain = s.gain[col];

    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(s.x), 0, static_cast<uint32_t>(a.n) * K * (NORM ? 4 : 2), 0x00027000);

    for (int row0 = part * 16, turn = 0; row0 < a.n; row0 += s.parts * 16, turn ^= 1) {
        const int tile_rows = min(16, a.n - row0);
        const int row = row0 + tile_row;
        const bool mine = row < a.n;
        float* const tiles = red + turn * (CN_STRETCHES * 256);        // (two of them in turn, and of `late`: a barrier a tile of rows, behind which a
                                                                       // wave may be in the next tile while another has not read this one's)
        float* const squares = ssq_lds + turn * (CN_WAVES * 16);
        // where the lane's values of K step k stand: at `lane_at` + begin + k * stride
        const uint32_t begin = row0 * K * (NORM ? 4 : 2), second = NORM ? 64 * tile_rows : 0;
        const uint32_t stride = s.x_laid ? (NORM ? 128 : 64) * tile_rows : 64;
        const uint32_t lane_at = c >= tile_rows ? CN_NOWHERE : s.x_laid ? (g * tile_rows + c) * 16 : (c * K + g * 8) * 2;
        auto load = [&](int u, int h, auto policy) {
            return __builtin_amdgcn_raw_buffer_load_b128(rows, is_step(u) ? lane_at : CN_NOWHERE, begin + h * second + (is_step(u) ? step_of(u) * stride : 0),
                                                         decltype(policy)::value);
        };

        // One piece of the wave's rows is looked at until it is there (all of them would be KBs a look, by every workgroup), then
        // all are loaded and looked at: once in any case, and as often again as looks are left.
        bool there = true;
        int left = a.looks;
        if (asks) {
            there = false;
            for (; left > 0 && !there; --left) {
                asm volatile("" ::: "memory");
                const cn_words4 p = load(0, 0, cn_past_l2_t{});
                there = __all(max(max(p[0], p[1]), max(p[2], p[3])) != PL_MISSING);
                if (!there) __builtin_amdgcn_s_sleep(1);
            }
        }
        cn_words4 raw[V * S][PARTS];
        uint32_t old = 0, sums[TAKES ? CN_RUN : 1];
        for (int again = 0; again <= left; ++again) {
            asm volatile("" ::: "memory");
            if constexpr (ADD) old = mine ? cn_word(s.old + (s.old_laid ? cn_laid(row, col, a.n, s.N, true) : row * s.N + col)) : 0u;
            if constexpr (TAKES) {
                // the sixteen threads of a row add up a run of its sums of squares each
                const int count = K / 16, run = pl_ceil_div(count, 16), from = t / 4 % 16 * run;
#pragma unroll
                for (int j = 0; j < CN_RUN; ++j)
                    sums[j] = mine && j < run && from + j < count ? cn_word(s.squares + static_cast<size_t>(row) * count + from + j) : 0u;
            }
            // (the first time through L2, which the workgroups of an XCD share: what a load that came too early has left there is
            // seen to be missing, and then read past L2)
            if (stage == 0 || (asks && again == 0)) {
#pragma unroll
                for (int u = 0; u < V * S; ++u)
#pragma unroll
                    for (int h = 0; h < PARTS; ++h) raw[u][h] = load(u, h, cn_cached_t{});
            } else {
#pragma unroll
                for (int u = 0; u < V * S; ++u)
#pragma unroll
                    for (int h = 0; h < PARTS; ++h) raw[u][h] = load(u, h, cn_past_l2_t{});
            }
            if (!asks) break;
            uint32_t most = old;
            if constexpr (TAKES)
#pragma unroll
                for (int j = 0; j < CN_RUN; ++j) most = max(most, sums[j]);
#pragma unroll
            for (int u = 0; u < V * S; ++u)
#pragma unroll
                for (int e = 0; e < 4 * PARTS; ++e) most = max(most, raw[u][e / 4][e % 4]);
            there = __all(most != PL_MISSING);
            if (there) break;
            __builtin_amdgcn_s_sleep(1);
        }
        if (!there && lane == 0) late[turn] = 1;

        f32x4 acc[BT][V];
#pragma unroll
        for (int b = 0; b < BT; ++b)
#pragma unroll
            for (int v = 0; v < V; ++v) acc[b][v] = f32x4{0.f, 0.f, 0.f, 0.f};
        float ssq = 0.f;
#pragma unroll
        for (int u = 0; u < S; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const int k = v * S + u;
                bf16x8 x;
                if constexpr (NORM) {
                    f32x8 scaled;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float xv = __uint_as_float(raw[k][e / 4][e % 4]);
                        ssq = fmaf(xv, xv, ssq);
                        scaled[e] = xv * gn[u][e];
                    }
                    x = __builtin_convertvector(scaled, bf16x8);
                } else {
                    x = __builtin_bit_cast(bf16x8, raw[k][0]);
                }
#pragma unroll
                for (int b = 0; b < BT; ++b)
                    acc[b][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w[b][k], acc[b][v], 0, 0, 0);
            }
#pragma unroll
        for (int b = 0; b < BT; ++b)
#pragma unroll
            for (int v = 0; v < V; ++v) *reinterpret_cast<f32x4*>(tiles + ((wave * V + v) * BT + b) * 256 + lane * 4) = acc[b][v];
        if constexpr (NORM) {
            ssq += __shfl_xor(ssq, 16, PL_WAVE);
            ssq += __shfl_xor(ssq, 32, PL_WAVE);
            if (g == 0) squares[wave * 16 + c] = ssq;
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(late[turn])) return false;

        float val[BT];
#pragma unroll
        for (int b = 0; b < BT; ++b) {
            val[b] = 0.f;
#pragma unroll
            for (int k = 0; k < CN_WAVES * V; ++k)
                if (FULL || k < s.stretches) val[b] += tiles[(k * BT + b) * 256 + t];
        }
        if constexpr (NORM || TAKES) {
            float total = 0.f;
            if constexpr (NORM) {
#pragma unroll
                for (int k = 0; k < CN_WAVES; ++k) total += squares[k * 16 + tile_row];
            } else {
#pragma unroll
                for (int j = 0; j < CN_RUN; ++j) total += __uint_as_float(sums[j]);
                total += __shfl_xor(total, 4, PL_WAVE);
                total += __shfl_xor(total, 8, PL_WAVE);
                total += __shfl_xor(total, 16, PL_WAVE);
                total += __shfl_xor(total, 32, PL_WAVE);
            }
            const float rinv = 1.f / sqrtf(total / static_cast<float>(K) + s.eps);
#pragma unroll
            for (int b = 0; b < BT; ++b) val[b] *= rinv;
        }
        if constexpr (ADD) {
            float updated = 0.f;
            if (mine) updated = __uint_as_float(old) + val[0];
            if (mine) cn_leave(static_cast<float*>(s.y) + (s.y_laid ? cn_laid(row, col, a.n, s.N, true) : row * s.N + col), cn_value(updated));
            if constexpr (KIND == CN_ADD_HANDS) {
                uint32_t pair = cn_pair(updated * hand_gain);
                pair = pair == PL_MISSING ? 0x7fff7fffu : pair;
                if (mine && col % 2 == 0) cn_leave(s.hand_x + cn_laid(row, col, a.n, s.N, false), pair);
                float sq = updated * updated;
                sq += __shfl_xor(sq, 4, PL_WAVE);
                sq += __shfl_xor(sq, 8, PL_WAVE);
                sq += __shfl_xor(sq, 16, PL_WAVE);
                sq += __shfl_xor(sq, 32, PL_WAVE);
                if (mine && col % 16 == 0) cn_leave(s.hand_squares + static_cast<size_t>(row) * (s.N / 16) + tile, cn_value(sq));
            }
        } else {
            uint32_t pair = cn_pair(GATED ? pl_activate<false>(val[0], a.act) * val[BT - 1] : val[0]);
            if ((s.y_laid || s.y_missing) && pair == PL_MISSING) pair = 0x7fff7fffu;
            if (mine && col % 2 == 0)
                cn_leave(static_cast<bf16_t*>(s.y) + (s.y_laid ? cn_laid(row, col, a.n, s.N, false) : row * s.N + col), pair);
        }
    }
    return true;
}

template <int KIND, int V, int S>
__device__ __forceinline__ bool cn_form(const cn_chain_t& a, const cn_stage_t& s, int stage, int place, bool trust, float* red, float* ssq_lds, int* late) {
    if (s.per == S && s.K == CN_WAVES * V * S * 32) return cn_tile<KIND, V, S, true>(a, s, stage, place, trust, red, ssq_lds, late);
    return cn_tile<KIND, V, S, false>(a, s, stage, place, trust, red, ssq_lds, late);
}
// Stretches of K in the kernel's unrolled forms (cn_stretches has how many there are).
template <int KIND>
__device__ __forceinline__ bool cn_add(const cn_chain_t& a, const cn_stage_t& s, int stage, int place, bool trust, float* red, float* ssq_lds, int* late) {
    if (s.stretches <= CN_WAVES) return cn_form<KIND, 1, 8>(a, s, stage, place, trust, red, ssq_lds, late);
    if (s.stretches <= CN_WAVES * 2) return cn_form<KIND, 2, 8>(a, s, stage, place, trust, red, ssq_lds, late);
    if constexpr (KIND == CN_ADD) return cn_form<KIND, 3, 8>(a, s, stage, place, trust, red, ssq_lds, late);
    return cn_form<KIND, 4, 6>(a, s, stage, place, trust, red, ssq_lds, late);
}

// A place of a stage (tile of columns, part of the rows) whose results in rows row0 to row1 are not all there, the first from `from` on, so that workgroups
// that miss the same begin with unlike ones; -1: all are there.
template <bool HANDED>
__device__ __forceinline__ int cn_missing_place(const __attribute__((address_space(4))) cn_chain_t& a, int stage, int from, int row0, int row1, float* lds) {
    const auto& s = a.s[stage];
    const int tiles = s.N / 16;
    int first = INT_MAX;
    // (`each` words of a tile's row; a look is a trip to memory, so eight are on their way together)
    auto look = [&](int each, auto at) {
        const int step = PL_WAVE * CN_WAVES / each, turns = pl_ceil_div(tiles, step);
#pragma unroll 8
        for (int i = 0; i < (row1 - row0) * turns; ++i) {
            const int row = row0 + i / turns, tile = min(i % turns * step + static_cast<int>(threadIdx.x) / each, tiles - 1);
            const uint32_t word = cn_word(reinterpret_cast<const float*>(at(row, tile, threadIdx.x % each)));
            const int turned = tile * s.parts + row / 16 % s.parts - from;
            first = word == PL_MISSING ? min(first, turned < 0 ? turned + s.tiles : turned) : first;
        }
    };
    if (s.kind == CN_ADD || s.kind == CN_ADD_HANDS) {
        look(16, [&](int row, int tile, int i) { return static_cast<const float*>(s.y) + cn_laid(row, tile * 16 + i, a.n, s.N, true); });
    } else {
        look(8, [&](int row, int tile, int i) {
            const int col = tile * 16 + i * 2;
            return static_cast<const bf16_t*>(s.y) + (s.y_laid ? cn_laid(row, col, a.n, s.N, false) : row * s.N + col);
        });
    }
    if (HANDED && s.kind == CN_ADD_HANDS) {
        look(8, [&](int row, int tile, int i) { return s.hand_x + cn_laid(row, tile * 16 + i * 2, a.n, s.N, false); });
        look(1, [&](int row, int tile, int) { return s.hand_squares + static_cast<size_t>(row) * tiles + tile; });
    }
    int* const least = reinterpret_cast<int*>(lds);
    if (threadIdx.x == 0) *least = INT_MAX;
    __syncthreads();
    if (first != INT_MAX) atomicMin(least, first);
    __syncthreads();
    const int found = __builtin_amdgcn_readfirstlane(*least);
    __syncthreads();
    return found == INT_MAX ? -1 : (found + from) % s.tiles;
}

// 256 registers a lane, two workgroups a compute unit: without attention the first 512 workgroups hold their weights at once (64 + 192 + 64 of the
// first three stages of the 0.6B shape and most of the 256 of the last).  With it, its workgroups have those places before the last stage's: one token's
// 64 leave 128 of the 256 a place, the 256 of four or eight tokens none until earlier workgroups end.
template <bool HANDED, bool ATTENDS>
__global__ void __launch_bounds__(PL_WAVE * CN_WAVES, 2) gemm_chain_kernel(cn_chain_t a, cn_attend_of<ATTENDS>) {
    __shared__ __attribute__((aligned(16))) float red[2 * CN_STRETCHES * 256];      // [stretch][gate, up][256] partial tiles
    __shared__ float ssq_lds[2 * CN_WAVES * 16];
    __shared__ int late[2];     // (one a turn of cn_tile; the attention takes the first)
    cn_touch_arguments(sizeof(cn_chain_t) + (ATTENDS ? sizeof(cn_attend_t) : 0));
    auto stage_of = [](const auto& a) {
        int stage = 0;
#pragma unroll
        for (int i = 1; i < CN_STAGES; ++i) {
            const int at = static_cast<int>(blockIdx.x) - a.s[i].first;
            if (i < a.stages && at >= 0 && at < a.s[i].tiles) stage = i;
        }
        return stage;
    };
    if (threadIdx.x == 0) late[0] = late[1] = 0;
    __syncthreads();
    int p = stage_of(a), q = static_cast<int>(blockIdx.x) - a.s[p].first;
    bool trust = false, own = true;     // (own: place q of stage p is the workgroup's, and not one that it works out because it is missing)
    while (true) {
        p = __builtin_amdgcn_readfirstlane(p);
        q = __builtin_amdgcn_readfirstlane(q);
        const cn_stage_t& s = a.s[p];
        bool done;
        if (ATTENDS && s.kind == CN_ATTEND) {
            if constexpr (ATTENDS) {
                // (read here, where they are needed: as values kept from the kernel's beginning on they spill)
                const __attribute__((address_space(4))) char* args = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
                asm volatile("" : "+s"(args));
                cn_attend_t next;
                __builtin_memcpy(&next, (const void*)(args + CN_ATTEND_AT), sizeof(next));
                const int n = ((const __attribute__((address_space(4))) cn_chain_t*)args)->n;
                const int token = q / next.nkv, split = token / n;
                done = ad_attend<16, CN_HEADS, CN_KEYS, CN_WAVES, 0, true>(
                    next.q, next.q_stride, next.out, next.part_acc, next.part_ml, next.positions, next.seq_of, nullptr, 0, 0, next.block_table,
                    next.max_blocks, next.block_size, next.k_pool, next.v_pool, next.nq, next.nkv, next.d, next.scale_log2e, next.window, next.splits, 1,
                    next.g, next.splits_magic, next.fuse, next.arrivals, ad_extras_t<0>{}, q - token * next.nkv, token - split * n, split, red,
                    ad_rows_t{!trust, min(a.looks, CN_ATTEND_LOOKS), late});
            }
        } else if constexpr (HANDED) {
            if (s.kind == CN_ADD) done = cn_add<CN_ADD>(a, s, p, q, trust, red, ssq_lds, late);
            else if (s.kind == CN_ADD_HANDS) done = cn_add<CN_ADD_HANDS>(a, s, p, q, trust, red, ssq_lds, late);
            else if (s.kind == CN_GATED_TAKES) done = cn_form<CN_GATED_TAKES, 1, 8>(a, s, p, q, trust, red, ssq_lds, late);
            else done = cn_form<CN_STORE_TAKES, 1, 8>(a, s, p, q, trust, red, ssq_lds, late);
        } else {
            if (s.kind == CN_ADD) done = cn_add<CN_ADD>(a, s, p, q, trust, red, ssq_lds, late);
            else if (s.kind == CN_GATED) done = cn_form<CN_GATED, 1, 8>(a, s, p, q, trust, red, ssq_lds, late);
            else done = cn_form<CN_STORE, 1, 8>(a, s, p, q, trust, red, ssq_lds, late);
        }
        if (done && own) return;
        // The rows were not there in time: what the earlier stages have not left yet, stage by stage, then the workgroup's own once more.  (What the
        // workgroup has written is where its loads past L2 find it before it goes on.)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) {
            int zero;
            asm volatile("v_mov_b32 %0, 0" : "=v"(zero));       // (as a constant it is kept through the kernel, and something else spilt)
            late[0] = late[1] = zero;
        }
        __syncthreads();
        // (its arguments read here, where they are needed: as values kept from the kernel's beginning on they spill)
        const __attribute__((address_space(4))) cn_chain_t* args = (const __attribute__((address_space(4))) cn_chain_t*)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(args));
        const int stage = stage_of(*args), place = static_cast<int>(blockIdx.x) - args->s[stage].first;
        int row0 = 0, row1 = args->n;
        if (ATTENDS && stage == CN_STAGES - 1 && !trust && (own || done)) {
            // The attention begins with its token's row of the projection, for which what that reads may be there: its workgroups stand in the grid
            // before the projection's, and several launches of them side by side can fill the chip.
            p = stage - 1;
            row0 = place / ((const __attribute__((address_space(4))) cn_attend_t*)((const __attribute__((address_space(4))) char*)args + CN_ATTEND_AT))->nkv % row1;
            row1 = row0 + 1;
        } else if (!trust) {
            trust = true;
            p = 0;
        }
        for (q = -1; p < stage; ++p) {
            q = cn_missing_place<HANDED>(*args, p, place % args->s[p].tiles, row0, row1, red);
            if (q >= 0) break;
        }
        own = q < 0;
        if (own) q = place;
    }
}

// How gemm_skinny's launches for one tile of rows cut K (launch_unr and launch_one in gemm_skinny.hpp): the stretches, 0 where they are
// more, or longer, than this kernel takes.
static int cn_stretches(int K, int kind) {
    const int steps = K / 32;
    if (steps <= CN_WAVES * 8) return CN_WAVES;
    if (kind != CN_ADD && kind != CN_ADD_HANDS) return 0;
    const int least = pl_ceil_div(steps, 8);
    if (least <= 8) return least < 5 ? 5 : least;
    const int many = max(9, kind == CN_ADD_HANDS ? pl_ceil_div(steps, 6) : least);
    return many <= (kind == CN_ADD_HANDS ? 16 : 12) ? many : 0;
}

// Whether the products of so many rows are this launch's: a stream of `width`, an output projection of inner width `inner`, a feed-forward of `ff`,
// and (0: none) `after` columns behind the next norm.
extern "C" int pl_gemm_chain_applies(int n, int width, int inner, int ff, int after) {
    return n > 0 && n <= CN_ROWS && width > 0 && width % 32 == 0 && inner > 0 && inner % 32 == 0 && ff > 0 && ff % 32 == 0 && after >= 0 && after % 16 == 0
           && ff <= (1 << 20) && after <= (1 << 20) && width / 16 <= 16 * CN_RUN
           && cn_stretches(width, CN_STORE) && cn_stretches(inner, CN_ADD) && cn_stretches(ff, CN_ADD);
}

// The 32-bit words that one launch leaves between its stages, all ones before it: mid [n, width], hidden [n, ff] in bfloat16, out [n, width], from CN_HANDED
// rows on the two norms handed forward, rows [n, width] in bfloat16 and sums [n, width / 16] each, and, where the launch goes on to the next layer's
// attention, the rows [n, after] in bfloat16 in between.  `out` begins at word out_at.
static size_t cn_room(int n, int width, int ff, int attended, size_t* out_at) {
    const size_t stream = static_cast<size_t>(n) * width, handed = n >= CN_HANDED ? stream / 2 + stream / 16 : 0;
    if (out_at) *out_at = stream + static_cast<size_t>(n) * ff / 2;
    return 2 * stream + static_cast<size_t>(n) * ff / 2 + 2 * handed + static_cast<size_t>(n) * attended / 2;
}
extern "C" long pl_gemm_chain_room(int n, int width, int ff, int attended) { return static_cast<long>(cn_room(n, width, ff, attended, nullptr)); }
extern "C" long pl_gemm_chain_out(int n, int width, int ff) {
    size_t at = 0;
    cn_room(n, width, ff, 0, &at);
    return static_cast<long>(at);
}

// Whether a step's attention of single tokens (one a request, nq over nkv heads of d, so many shares of a context of up to `bound`) may be the last stage of
// a chain.  At most a workgroup a compute unit: they stand in the grid before the workgroups that they wait for, and so leave these half of the
// chip.  (512 of them filled it, and none of those began before all looks were in vain.)  At most two rounds of keys a workgroup: it has one in
// registers when its rows come, and asks for a further one only when that is taken (us a step, last stage / a launch of its own, 0.6B shape: 1 token at a
// context of 512 693 / 785, 4 tokens 728 / 815, 8 tokens 815 / 871, at contexts up to 1,000 958 / 972; 16 tokens, four rounds, at 512 1,044 / 1,072, at
// 1,000 1,321 / 1,263; 32 tokens, eight rounds, 1,524 / 1,309).
extern "C" int pl_gemm_chain_attends(int n, int nq, int nkv, int d, int splits, int bound) {
    return n > 0 && n < CN_HANDED && nkv > 0 && nq % nkv == 0 && nq / nkv <= CN_HEADS && d > 64 && d <= 128 && d % 16 == 0 && splits >= 1
           && splits <= AD_MERGE_AT_ONCE && bound > 0 && pl_ceil_div(bound, splits) <= CN_SHARE
           && static_cast<long>(nkv) * n * splits <= pl_compute_units();
}

// stream: [n, width] 32-bit, rows or (stream_laid) as an earlier chain left it.  rows: bfloat16 [n, inner].  The weights in strips: w_out [width, inner],
// w_gated [2 ff, width] (gate rows first), w_down [width, ff], w_next [after, width] or null.  room: cn_room words of all ones; its `out`
// [n, width] takes the updated stream, laid with a w_next and in rows without.  next: bfloat16 [n, after].  looks: how often a
// workgroup looks for its rows before it works them out itself.  attend: the next layer's attention, or null.
static int chain_launch(const float* stream, int stream_laid, const void* rows, void* room, void* next, const void* w_out,
                             const void* w_gated, const void* w_down, const void* w_next, const float* gain2, float eps2, const float* gain_next,
                             float eps_next, int n, int width, int inner, int ff, int after, int act, int looks, cn_attend_t* attend, hipStream_t stream_) {
    if (n == 0) return 0;
    PL_REQUIRE(pl_gemm_chain_applies(n, width, inner, ff, after), "chain of products: %d rows, a stream of %d, inner widths %d and %d, %d columns behind it", n, width, inner, ff, after);
    PL_REQUIRE(stream && rows && room && w_out && w_gated && w_down && gain2, "chain of products: an operand is missing");
    PL_REQUIRE((w_next != nullptr) == (after > 0) && (next != nullptr) == (after > 0 && !attend) && (!attend || after > 0) && (gain_next != nullptr) == (after > 0),
               "chain of products: %d columns behind the chain", after);
    PL_REQUIRE(act >= PL_ACT_SILU && act <= PL_ACT_RELU2, "chain of products: activation code %d", act);
    PL_REQUIRE(looks >= 0, "chain of products: %d looks", looks);
    for (const void* p : {static_cast<const void*>(stream), rows, static_cast<const void*>(room), w_out, w_gated, w_down, w_next, static_cast<const void*>(gain2),
                          static_cast<const void*>(gain_next), static_cast<const void*>(next)})
        PL_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "chain of products: an operand begins in the middle of 16 bytes");
    const bool handed = n >= CN_HANDED, follows = after > 0;
    size_t out_at = 0;
    const size_t room_words = cn_room(n, width, ff, 0, &out_at);
    const size_t words = static_cast<size_t>(n) * width;
    float* const mid = static_cast<float*>(room);
    float* const hidden = mid + words;
    float* const out = mid + out_at;
    // (only there with handed norms)
    bf16_t* const mid_x = reinterpret_cast<bf16_t*>(out + words);
    float* const mid_squares = out + words + words / 2;
    bf16_t* const out_x = reinterpret_cast<bf16_t*>(mid_squares + words / 16);
    float* const out_squares = mid_squares + words / 16 + words / 2;
    cn_chain_t a{};
    a.n = n;
    a.act = act;
    a.looks = looks;
    a.stages = attend ? 5 : follows ? 4 : 3;
    cn_stage_t& project = a.s[0];
    project.x = rows; project.w = static_cast<const bf16_t*>(w_out); project.y = mid; project.old = stream;
    project.N = width; project.K = inner; project.kind = handed ? CN_ADD_HANDS : CN_ADD;
    project.old_laid = stream_laid ? 1 : 0; project.y_laid = 1;
    project.gain = gain2; project.hand_x = mid_x; project.hand_squares = mid_squares;
    cn_stage_t& gated = a.s[1];
    gated.x = handed ? static_cast<const void*>(mid_x) : mid; gated.w = static_cast<const bf16_t*>(w_gated); gated.y = hidden; gated.gain = gain2; gated.eps = eps2;
    gated.squares = mid_squares; gated.N = ff; gated.K = width; gated.kind = handed ? CN_GATED_TAKES : CN_GATED;
    gated.x_laid = 1; gated.y_laid = 1;
    cn_stage_t& down = a.s[2];
    down.x = hidden; down.w = static_cast<const bf16_t*>(w_down); down.y = out; down.old = mid;
    down.N = width; down.K = ff; down.kind = handed && follows ? CN_ADD_HANDS : CN_ADD;
    down.x_laid = 1; down.old_laid = 1; down.y_laid = follows ? 1 : 0;
    down.gain = gain_next; down.hand_x = out_x; down.hand_squares = out_squares;
    cn_stage_t& last = a.s[3];
    last.x = handed ? static_cast<const void*>(out_x) : out; last.w = static_cast<const bf16_t*>(w_next); last.y = next; last.gain = gain_next; last.eps = eps_next;
    last.squares = out_squares; last.N = after; last.K = width; last.kind = handed ? CN_STORE_TAKES : CN_STORE;
    last.x_laid = 1;
    if (attend) {
        last.y = mid + room_words;
        last.y_missing = 1;
        attend->q = reinterpret_cast<const bf16_t*>(last.y);
        attend->q_stride = after;
    }
    int grid = 0;
    for (int i = 0; i < (follows ? 4 : 3); ++i) {
        cn_stage_t& s = a.s[i];
        if (i == 3 && attend) {
            // The attention's workgroups before those of the projection that they wait for: behind them they began 9 us into the launch and were
            // still asking for pages, keys and values when their rows came, at 14 (a step of one token 785 us, so 693).
            a.s[4].kind = CN_ATTEND;
            a.s[4].first = grid;
            a.s[4].tiles = attend->nkv * n * attend->splits;
            grid += a.s[4].tiles;
        }
        s.stretches = cn_stretches(s.K, s.kind);
        s.per = pl_ceil_div(s.K / 32, s.stretches);
        s.first = grid;
        s.parts = n > 16 ? 2 : 1;
        s.tiles = s.N / 16 * s.parts;
        grid += s.tiles;
    }
    if (attend) {
        gemm_chain_kernel<false, true><<<grid, PL_WAVE * CN_WAVES, 0, stream_>>>(a, *attend);
    } else if (handed) {
        gemm_chain_kernel<true, false><<<grid, PL_WAVE * CN_WAVES, 0, stream_>>>(a, cn_nothing_t{});
    } else {
        gemm_chain_kernel<false, false><<<grid, PL_WAVE * CN_WAVES, 0, stream_>>>(a, cn_nothing_t{});
    }
    PL_CHECK_LAUNCH("gemm_chain");
    return 0;
}

extern "C" int pl_gemm_chain(const float* stream, int stream_laid, const void* rows, void* room, void* next, const void* w_out,
                             const void* w_gated, const void* w_down, const void* w_next, const float* gain2, float eps2, const float* gain_next,
                             float eps_next, int n, int width, int inner, int ff, int after, int act, int looks, hipStream_t stream_) {
    return chain_launch(stream, stream_laid, rows, room, next, w_out, w_gated, w_down, w_next, gain2, eps2, gain_next, eps_next, n, width, inner, ff, after, act,
                        looks, nullptr, stream_);
}

// The same, and behind the next layer's projection [q | k | v] of `after` = (nq + 2 nkv) d columns, which stays in the room, that layer's attention: as
// pl_paged_attention_decode with fuse_mode 1 or 2 and no lengths, extras or second kernel (splits > 1: with arrivals).
extern "C" int pl_gemm_chain_attend(const float* stream, int stream_laid, const void* rows, void* room, const void* w_out, const void* w_gated,
                                    const void* w_down, const void* w_next, const float* gain2, float eps2, const float* gain_next, float eps_next, int n,
                                    int width, int inner, int ff, int after, int act, int looks, void* out, float* part_acc, float* part_ml,
                                    const int* positions, const int* seq_of, const int* block_table, int max_blocks, int block_size, void* k_pool,
                                    void* v_pool, int nq, int nkv, int d, float scale, int window, int splits, int fuse_mode, const void* q_gain,
                                    const void* k_gain, int gain_dtype, float eps, const float* cos_table, const float* sin_table, int rot, int* arrivals,
                                    hipStream_t stream_) {
    if (n == 0) return 0;
    PL_REQUIRE(pl_gemm_chain_attends(n, nq, nkv, d, splits, 1), "chain with attention: %d tokens, %d over %d heads of %d, %d shares", n, nq, nkv, d, splits);
    PL_REQUIRE(after == (nq + 2 * nkv) * d && out && positions && seq_of && block_table && k_pool && v_pool && block_size > 0 && max_blocks > 0,
               "chain with attention: rows of %d values, block size %d, %d blocks a row", after, block_size, max_blocks);
    PL_REQUIRE(splits == 1 || (part_acc && part_ml && arrivals), "chain with attention: %d shares without a workspace", splits);
    PL_REQUIRE(fuse_mode == 1 || fuse_mode == 2, "chain with attention: fuse mode %d", fuse_mode);
    PL_REQUIRE(rot >= 0 && rot <= d && rot % 16 == 0, "chain with attention: a rotated width of %d of a head of %d is not fused", rot, d);
    PL_REQUIRE((q_gain == nullptr) == (k_gain == nullptr), "chain with attention: one of the two gains is missing");
    PL_REQUIRE(!q_gain || gain_dtype == PL_DTYPE_F32 || gain_dtype == PL_DTYPE_BF16, "chain with attention: gain dtype code %d", gain_dtype);
    PL_REQUIRE((cos_table == nullptr) == (sin_table == nullptr) && (cos_table || rot == 0), "chain with attention: rotation tables");
    for (const void* p : {static_cast<const void*>(k_pool), static_cast<const void*>(v_pool), q_gain, k_gain, static_cast<const void*>(cos_table),
                          static_cast<const void*>(sin_table)})
        PL_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "chain with attention: an operand begins in the middle of 16 bytes");
    cn_attend_t attend{nullptr, 0, static_cast<bf16_t*>(out), part_acc, part_ml, positions, seq_of, block_table, max_blocks, block_size,
                       static_cast<bf16_t*>(k_pool), static_cast<bf16_t*>(v_pool), nq, nkv, d, scale * 1.4426950408889634f, window, splits, nq / nkv,
                       static_cast<uint32_t>((0x100000000ull + splits - 1) / static_cast<unsigned>(splits)),
                       ad_fuse_t{q_gain, k_gain, gain_dtype, eps, cos_table, sin_table, rot, fuse_mode}, arrivals};
    return chain_launch(stream, stream_laid, rows, room, nullptr, w_out, w_gated, w_down, w_next, gain2, eps2, gain_next, eps_next, n, width, inner, ff, after,
                        act, looks, &attend, stream_);
}
