// The products behind a layer's attention for few rows (n <= 15), bfloat16 weights in strips, as ONE launch:
//
//   stage 0  mid    = stream + rows . w_out^T                 (the mixer's output projection)
//   stage 1  hidden = act(norm2(mid) . gate^T) * (norm2(mid) . up^T)
//   stage 2  out    = mid + hidden . w_down^T
//   stage 3  after  = norm1'(out) . w_after^T                 (the next layer's first projection; optional)
//
// A launch of its own takes a stage 5.2 us (one row of a stream of 1,024; weights of 4 to 12 MB that memory gives in
// 0.8 to 2.3 us): the boundary between two kernels, weights that are asked for only then, and the drain.  Here the
// workgroups of all stages are in one grid, 16 columns each.  A workgroup asks for its weights first, into registers, and
// then looks for its input; so the weights of a stage travel while the stages before it work, and what is left between
// two stages is one trip of the rows through memory.  Four products of the 0.6B shape, 28 layers, weights from memory, us
// a layer, four launches / one: 1 row 20.8 / 14.7, 8 rows 22.9 / 15.6, 15 rows 25.3 / 18.3.
//
// How a stage learns that its rows are there.  mid, out and hidden begin as words of all ones (PL_MISSING), and every word
// is written once, past the XCD's L2 (relaxed atomics of device scope, as in pl_share): a word that differs is the value.
// A result that happens to be all ones (a NaN, or a pair of them) is written as another NaN.  There is no counter: one that all
// workgroups of a stage add to costs 2 us a stage (20.8 us a layer, no gain at all).
// mid, hidden and out lie in the order in which the next stage's lanes load them ("laid", see cn_laid): 8 rows as
// [row][column] cost 18.5 us a layer, since a load then touches a line a row twice.
//
// Nothing waits for ever.  A workgroup looks `looks` times; if its rows are not there by then (workgroups are started in the order
// of their numbers, earlier stages first, but another launch may hold the compute units they need), it works out all
// earlier stages' tiles itself, in their order, and then its own: the same arithmetic, so the same bits to the same words, whoever writes
// them first.  What it wrote itself it takes without a look, so that way ends whatever anybody else does.
//
// The arithmetic is gemm_skinny's for one tile of rows, to the same bits: K in as many stretches as that launch has waves (a
// wave here takes up to three of them, each an accumulator of its own), the stretches' tiles added in their order.
#include "common.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define CN_ADD 0        // y = old + x . w^T, 32-bit
#define CN_GATED 1      // y = act(norm(x) . gate^T) * (norm(x) . up^T), bfloat16
#define CN_STORE 2      // y = norm(x) . w^T, bfloat16
#define CN_STAGES 4
#define CN_WAVES 4
#define CN_STEPS 8      // K steps of 32 that a stretch of K has at most
#define CN_STRETCHES 3  // stretches a wave takes at most
#define CN_ROWS 15
#define PL_MISSING 0xffffffffu
#define CN_PAST_L2 16   // cache policy of a buffer load: device scope (sc1)
#define CN_NOWHERE 0x7ff00000u

struct cn_stage_t {
    const void* x;          // CN_ADD: bfloat16 rows; otherwise the 32-bit stream, laid
    const bf16_t* w;        // in strips
    void* y;
    const float* old;       // CN_ADD
    const float* gain;
    float eps;
    int N, K;               // columns of y
    int per, stretches;     // K steps of a stretch; stretches of K
    int kind;
    int first, tiles;       // its workgroups
    int x_laid, old_laid, y_laid;
};
struct cn_chain_t {
    cn_stage_t s[CN_STAGES];
    int stages, n, act, looks;
};

// Where value (row, col) of a laid [n, width] tensor stands: K step by K step of 32 columns, in the order of the lanes that load
// it (8 columns a group, 16 bytes a load: 32-bit rows in two halves).
__host__ __device__ static inline size_t cn_laid(int row, int col, int n, bool wide) {
    const size_t step = col / 32, group = col % 32 / 8;
    return wide ? ((step * 8 + col % 8 / 4 * 4 + group) * n + row) * 4 + col % 4 : ((step * 4 + group) * n + row) * 8 + col % 8;
}

// One tile of 16 columns of one stage.  trust: the rows were written by this workgroup.  Returns whether the tile is done
// (false: its rows were not there in time), the same for all threads.
template <int KIND, int V>
__device__ __forceinline__ bool cn_tile(const cn_chain_t& a, const cn_stage_t& s, int stage, int tile, bool trust, float* red, float* ssq_lds,
                                        int* late) {
    constexpr int BT = KIND == CN_GATED ? 2 : 1;
    constexpr bool NORM = KIND != CN_ADD;
    constexpr int PARTS = NORM ? 2 : 1;        // loads of 16 bytes for a lane's 8 values
    const int lane = threadIdx.x % PL_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PL_WAVE);
    const int c = lane % 16, g = lane / 16;
    const int K = s.K, steps = K / 32;
    const bool asks = stage > 0 && !trust;

    // the weights first: they come from memory and depend on nothing
    int step[V * CN_STEPS];                    // (-1: none)
    bf16x8 w[BT][V * CN_STEPS];
    float gn[NORM ? CN_STEPS : 1][8];
#pragma unroll
    for (int u = 0; u < V * CN_STEPS; ++u) {
        const int at = (wave * V + u / CN_STEPS) * s.per + u % CN_STEPS;
        step[u] = u % CN_STEPS < s.per && at < steps ? at : -1;
    }
#pragma unroll
    for (int b = 0; b < BT; ++b) {
        const bf16_t* strip = s.w + static_cast<size_t>(b * (s.N / 16) + tile) * 16 * K + lane * 8;
#pragma unroll
        for (int u = 0; u < V * CN_STEPS; ++u) w[b][u] = *reinterpret_cast<const bf16x8*>(strip + static_cast<size_t>(max(step[u], 0)) * 512);
    }
    if constexpr (NORM) {
#pragma unroll
        for (int u = 0; u < CN_STEPS; ++u) {
            const f32x8 v = *reinterpret_cast<const f32x8*>(s.gain + max(step[u], 0) * 32 + g * 8);
#pragma unroll
            for (int e = 0; e < 8; ++e) gn[u][e] = v[e];
        }
    }

    // where the lane's values of each step stand (rows and steps that are not there: past the buffer's end, which gives zeros)
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(s.x), 0, static_cast<uint32_t>(a.n) * K * (NORM ? 4 : 2), 0x00027000);
    const uint32_t second = NORM ? 4 * 16 * a.n : 0;
    uint32_t at[V * CN_STEPS];
#pragma unroll
    for (int u = 0; u < V * CN_STEPS; ++u)
        at[u] = c >= a.n || step[u] < 0 ? CN_NOWHERE
                : !s.x_laid             ? (static_cast<uint32_t>(c) * K + step[u] * 32 + g * 8) * 2
                                        : ((static_cast<uint32_t>(step[u]) * (NORM ? 8 : 4) + g) * a.n + c) * 16;

    // the element that this thread finishes
    const int t = threadIdx.x;
    const int row = t / 64 * 4 + t % 4, col = tile * 16 + t / 4 % 16;
    const bool mine = row < a.n;

    // One piece of the wave's rows is looked at until it is there (all of them would be n KB a look, by every workgroup), then
    // all are loaded and looked at.
    bool there = true;
    if (asks) {
        there = false;
        for (int look = 0; look < a.looks && !there; ++look) {
            asm volatile("" ::: "memory");
            const u32x4 p = __builtin_amdgcn_raw_buffer_load_b128(rows, at[0], 0, CN_PAST_L2);
            there = __all(max(max(p[0], p[1]), max(p[2], p[3])) != PL_MISSING);
            if (!there) __builtin_amdgcn_s_sleep(1);
        }
    }
    u32x4 raw[V * CN_STEPS][PARTS];
    uint32_t old = 0;
    for (int look = 0; look <= a.looks; ++look) {
        asm volatile("" ::: "memory");
        if (KIND == CN_ADD)
            old = mine ? __hip_atomic_load(reinterpret_cast<const uint32_t*>(s.old) + (s.old_laid ? cn_laid(row, col, a.n, true) : static_cast<size_t>(row) * s.N + col),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                       : 0u;
        // (the first time through L2, which the workgroups of an XCD share: what a load that came too early has left there is
        // seen to be missing, and then read past L2)
        if (stage == 0 || (asks && look == 0)) {
#pragma unroll
            for (int u = 0; u < V * CN_STEPS; ++u)
#pragma unroll
                for (int h = 0; h < PARTS; ++h) raw[u][h] = __builtin_amdgcn_raw_buffer_load_b128(rows, at[u] + h * second, 0, 0);
        } else {
#pragma unroll
            for (int u = 0; u < V * CN_STEPS; ++u)
#pragma unroll
                for (int h = 0; h < PARTS; ++h) raw[u][h] = __builtin_amdgcn_raw_buffer_load_b128(rows, at[u] + h * second, 0, CN_PAST_L2);
        }
        if (!asks) break;
        uint32_t most = old;
#pragma unroll
        for (int u = 0; u < V * CN_STEPS; ++u)
#pragma unroll
            for (int e = 0; e < 4 * PARTS; ++e) most = max(most, raw[u][e / 4][e % 4]);
        there = __all(most != PL_MISSING);
        if (there) break;
        __builtin_amdgcn_s_sleep(1);
    }
    if (!there && lane == 0) *late = 1;

    f32x4 acc[BT][V];
#pragma unroll
    for (int b = 0; b < BT; ++b)
#pragma unroll
        for (int v = 0; v < V; ++v) acc[b][v] = f32x4{0.f, 0.f, 0.f, 0.f};
    float ssq = 0.f;
#pragma unroll
    for (int u = 0; u < CN_STEPS; ++u)
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const int k = v * CN_STEPS + u;
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
            // (a step past the stretch multiplies nothing, whatever the weights in its place are)
#pragma unroll
            for (int b = 0; b < BT; ++b)
                acc[b][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, step[k] >= 0 ? w[b][k] : bf16x8{}, acc[b][v], 0, 0, 0);
        }
#pragma unroll
    for (int b = 0; b < BT; ++b)
#pragma unroll
        for (int v = 0; v < V; ++v) *reinterpret_cast<f32x4*>(red + ((wave * V + v) * BT + b) * 256 + lane * 4) = acc[b][v];
    if constexpr (NORM) {
        ssq += __shfl_xor(ssq, 16, PL_WAVE);
        ssq += __shfl_xor(ssq, 32, PL_WAVE);
        if (g == 0) ssq_lds[wave * 16 + c] = ssq;
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(*late)) return false;

    float val[BT];
#pragma unroll
    for (int b = 0; b < BT; ++b) {
        val[b] = 0.f;
#pragma unroll
        for (int k = 0; k < CN_WAVES * V; ++k)
            if (k < s.stretches) val[b] += red[(k * BT + b) * 256 + t];
    }
    if constexpr (NORM) {
        float total = 0.f;
#pragma unroll
        for (int k = 0; k < CN_WAVES; ++k) total += ssq_lds[k * 16 + row];
        const float rinv = 1.f / sqrtf(total / static_cast<float>(K) + s.eps);
#pragma unroll
        for (int b = 0; b < BT; ++b) val[b] *= rinv;
    }
    if constexpr (KIND == CN_ADD) {
        uint32_t bits = __float_as_uint(__uint_as_float(old) + val[0]);
        bits = bits == PL_MISSING ? 0x7fc00000u : bits;
        if (mine)
            __hip_atomic_store(static_cast<uint32_t*>(s.y) + (s.y_laid ? cn_laid(row, col, a.n, true) : static_cast<size_t>(row) * s.N + col), bits,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        const float r = KIND == CN_GATED ? pl_activate<false>(val[0], a.act) * val[BT - 1] : val[0];
        // two neighbouring columns, four lanes apart, are a word
        const uint32_t half = bf16_bits_from_float(r);
        uint32_t pair = half | static_cast<uint32_t>(__shfl_down(half, 4, PL_WAVE)) << 16;
        if (s.y_laid && pair == PL_MISSING) pair = 0x7fff7fffu;
        if (mine && col % 2 == 0)
            __hip_atomic_store(reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(s.y) + (s.y_laid ? cn_laid(row, col, a.n, false) : static_cast<size_t>(row) * s.N + col)),
                               pair, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return true;
}

// 256 registers a lane, two workgroups a compute unit: the first 512 workgroups hold their weights at once (64 + 192 + 64 of the
// first three stages of the 0.6B shape and most of the 256 of the last).
__global__ void __launch_bounds__(PL_WAVE * CN_WAVES, 2) gemm_chain_kernel(cn_chain_t a) {
    __shared__ float red[CN_WAVES * CN_STRETCHES * 256];      // [stretch][gate, up][256] partial tiles
    __shared__ float ssq_lds[CN_WAVES * 16];
    __shared__ int late;
    int stage = 0;
    while (stage + 1 < a.stages && static_cast<int>(blockIdx.x) >= a.s[stage + 1].first) ++stage;
    const int tile = static_cast<int>(blockIdx.x) - a.s[stage].first;
    if (threadIdx.x == 0) late = 0;
    __syncthreads();
    int p = stage, q = tile;
    bool trust = false;
    while (true) {
        p = __builtin_amdgcn_readfirstlane(p);
        q = __builtin_amdgcn_readfirstlane(q);
        const cn_stage_t& s = a.s[p];
        bool done;
        if (s.kind == CN_ADD) {
            if (s.stretches <= CN_WAVES) done = cn_tile<CN_ADD, 1>(a, s, p, q, trust, red, ssq_lds, &late);
            else if (s.stretches <= CN_WAVES * 2) done = cn_tile<CN_ADD, 2>(a, s, p, q, trust, red, ssq_lds, &late);
            else done = cn_tile<CN_ADD, 3>(a, s, p, q, trust, red, ssq_lds, &late);
        } else if (s.kind == CN_GATED) {
            done = cn_tile<CN_GATED, 1>(a, s, p, q, trust, red, ssq_lds, &late);
        } else {
            done = cn_tile<CN_STORE, 1>(a, s, p, q, trust, red, ssq_lds, &late);
        }
        if (done && p == stage && q == tile) return;
        // The rows were not there in time: all tiles of the earlier stages, then the workgroup's own once more.  (What the
        // workgroup has written is where its loads past L2 find it before the next tile begins.)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) late = 0;
        __syncthreads();
        if (!trust) {
            trust = true;
            p = 0;
            q = 0;
        } else if (++q == s.tiles) {
            ++p;
            q = 0;
        }
        if (p == stage) q = tile;
    }
}

// How gemm_skinny's launch for up to 16 rows cuts K (launch_unr in gemm_skinny.hpp): the stretches, 0 where they are more
// than this kernel takes.
static int cn_stretches(int K, bool norm) {
    const int steps = K / 32;
    if (steps <= CN_WAVES * CN_STEPS) return CN_WAVES;
    if (norm) return 0;
    const int least = pl_ceil_div(steps, CN_STEPS);
    if (least <= 8) return least < 5 ? 5 : least;
    const int many = least < 9 ? 9 : least;
    return many <= CN_WAVES * CN_STRETCHES ? many : 0;
}

// Whether the products of so many rows are this launch's: a stream of `width`, an output projection of inner width `inner`, a feed-forward of `ff`,
// and (0: none) `after` columns behind the next norm.
extern "C" int pl_gemm_chain_applies(int n, int width, int inner, int ff, int after) {
    return n > 0 && n <= CN_ROWS && width > 0 && width % 32 == 0 && inner > 0 && inner % 32 == 0 && ff > 0 && ff % 32 == 0 && after >= 0 && after % 16 == 0
           && width <= (1 << 20) && ff <= (1 << 20) && after <= (1 << 20)
           && cn_stretches(width, true) && cn_stretches(inner, false) && cn_stretches(ff, false);
}

// stream: [n, width] 32-bit, rows or (stream_laid) as an earlier chain left it.  rows: bfloat16 [n, inner].  The weights in strips: w_out [width, inner],
// w_gated [2 ff, width] (gate rows first), w_down [width, ff], w_next [after, width] or null.  mid [n, width] and out [n, width] 32-bit and hidden [n, ff]
// bfloat16 are all ones before; out comes laid with a w_next and in rows without.  next: bfloat16 [n, after].  looks: how often a workgroup
// looks for its rows before it works them out itself.
extern "C" int pl_gemm_chain(const float* stream, int stream_laid, const void* rows, float* mid, void* hidden, float* out, void* next, const void* w_out,
                             const void* w_gated, const void* w_down, const void* w_next, const float* gain2, float eps2, const float* gain_next,
                             float eps_next, int n, int width, int inner, int ff, int after, int act, int looks, hipStream_t stream_) {
    if (n == 0) return 0;
    PL_REQUIRE(pl_gemm_chain_applies(n, width, inner, ff, after), "chain of products: %d rows, a stream of %d, inner widths %d and %d, %d columns behind it", n, width, inner, ff, after);
    PL_REQUIRE(stream && rows && mid && hidden && out && w_out && w_gated && w_down && gain2, "chain of products: an operand is missing");
    PL_REQUIRE((w_next != nullptr) == (after > 0) && (next != nullptr) == (after > 0) && (gain_next != nullptr) == (after > 0),
               "chain of products: %d columns behind the chain", after);
    PL_REQUIRE(act >= PL_ACT_SILU && act <= PL_ACT_RELU2, "chain of products: activation code %d", act);
    PL_REQUIRE(looks >= 0, "chain of products: %d looks", looks);
    for (const void* p : {static_cast<const void*>(stream), rows, static_cast<const void*>(mid), static_cast<const void*>(hidden), static_cast<const void*>(out), w_out, w_gated,
                          w_down, w_next, static_cast<const void*>(gain2), static_cast<const void*>(gain_next), static_cast<const void*>(next)})
        PL_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "chain of products: an operand begins in the middle of 16 bytes");
    cn_chain_t a{};
    a.n = n;
    a.act = act;
    a.looks = looks;
    a.s[0] = {rows, static_cast<const bf16_t*>(w_out), mid, stream, nullptr, 0.f, width, inner, 0, 0, CN_ADD, 0, 0, 0, stream_laid ? 1 : 0, 1};
    a.s[1] = {mid, static_cast<const bf16_t*>(w_gated), hidden, nullptr, gain2, eps2, ff, width, 0, 0, CN_GATED, 0, 0, 1, 0, 1};
    a.s[2] = {hidden, static_cast<const bf16_t*>(w_down), out, mid, nullptr, 0.f, width, ff, 0, 0, CN_ADD, 0, 0, 1, 1, after > 0 ? 1 : 0};
    a.s[3] = {out, static_cast<const bf16_t*>(w_next), next, nullptr, gain_next, eps_next, after, width, 0, 0, CN_STORE, 0, 0, 1, 0, 0};
    a.stages = after > 0 ? 4 : 3;
    int grid = 0;
    for (int i = 0; i < a.stages; ++i) {
        cn_stage_t& s = a.s[i];
        s.stretches = cn_stretches(s.K, s.kind != CN_ADD);
        s.per = pl_ceil_div(s.K / 32, s.stretches);
        s.first = grid;
        s.tiles = s.N / 16;
        grid += s.tiles;
    }
    gemm_chain_kernel<<<grid, PL_WAVE * CN_WAVES, 0, stream_>>>(a);
    PL_CHECK_LAUNCH("gemm_chain");
    return 0;
}
