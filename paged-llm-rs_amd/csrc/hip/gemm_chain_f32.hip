// The products behind a layer's attention for few rows (n <= 16) of the 32-bit path as ONE launch: the stages of gemm_chain.hip, and its way for a stage
// to learn that its rows are there (values that all ones words wait for, bounded looks, workgroups whose rows do not come share what is missing: 108 us a launch
// of 8 rows in which nobody may wait, 5,800 when each worked all of it out).
//
//   stage 0  mid    = stream + rows . w_out^T
//   stage 1  hidden = act(norm2(mid) . gate^T) * (norm2(mid) . up^T)
//   stage 2  out    = mid + hidden . w_down^T
//   stage 3  after  = norm1'(out) . w_after^T                 (the next layer's first projection; optional)
//
// Bound by the weights' bytes (63 MB a layer of the 0.6B shape, which memory gives in some 12 us) and by three trips of the rows between the stages.
// Apart the stages are six launches, two norms among them: 42.5 us a layer at 8 rows of the 0.6B shape, this one 29; a decoding step of 8 tokens
// 1,860 us before, 1,624 now.  Half of a layer's weights fit into the registers of the workgroups that the chip holds, and those of the last two stages are asked for
// when earlier workgroups leave; stage 2's workgroups in the grid before stage 1's, so that theirs are among the first half, took 1,647.
//
// The arithmetic is that of the launches apart, to the same bits: K in the parts of gemm_f32.hip (at most 16, by K alone), a part one chain of matrix
// instructions, the parts added in ascending order; a norm's squares in the order of add_rmsnorm_quads_kernel.
//
// A workgroup is eight waves, each two parts of K.  The two products that add into the stream have few columns and go to workgroups of 8: an
// instruction then takes 8 columns of two parts (SHARE 2 of gemm_f32.hip) for 8 rows of x, a second time for the rows from 8 on, with the weights kept.
// The two behind norms take 16 columns (8 of gate and the same 8 of up) and all rows.
#include "gemm_chain.hpp"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define CF_ADD 0        // y = old + x . w^T
#define CF_GATED 1      // y = act(norm(x) . gate^T) * (norm(x) . up^T)
#define CF_STORE 2      // y = norm(x) . w^T
#define CF_STAGES 4
#define CF_WAVES 8
#define CF_PARTS 16     // of K (gemm_f32.hip)
#define CF_ROWS 16
#define CF_DEEPEST 3072         // K of a product that adds
#define CF_WIDEST 1024          // and of one behind a norm
#define CF_FOURS (CF_WIDEST / 4 + 4)        // sums of four squares a row, one row's in other banks than the next's

struct cf_stage_t {
    const float* x;
    const float* w;
    float* y;
    const float* old;       // CF_ADD
    const float* gain;      // of the norm in front
    float eps;
    int N, K;               // columns of y
    int part_len;
    int kind;
    int first, tiles;       // its workgroups
    int x_laid, old_laid, y_laid;
};
struct cf_chain_t {
    cf_stage_t s[CF_STAGES];
    int stages, n, act, looks;
};

// Rows between stages lie four columns after four columns, in these row by row: what the lanes of a load ask for is one stretch.
__device__ __forceinline__ uint32_t cf_place(int row, int col, int n, int width, int laid) {
    return laid ? (col / 4 * n + row) * 4 + col % 4 : row * width + col;
}

// num / den, correctly rounded, with `inverse` the correctly rounded 1 / den (Markstein's division: the quotient's remainder, exact in a fused
// multiply-add, corrects it).  `plain`: den or its inverse is not of ordinary size; and a remainder needs room below num.
__device__ __forceinline__ float cf_quotient(float num, float den, float inverse, bool plain) {
    if (plain || fabsf(num) < 0x1p-80f) return num / den;
    const float q = num * inverse;
    return fmaf(fmaf(-q, den, num), inverse, q);
}

struct cf_lds_t {
    float parts[2][CF_PARTS][CF_ROWS * 16];         // [turn][part][row][column of w]
    float gain[CF_WIDEST];
    float denom[CF_ROWS];
    int least;
    int late[2];        // (by turn as the parts: behind a tile's barrier a wave may be in the next tile while another has not read this one's)
};

// One tile of one stage, all rows; S steps of 16 k a part at most, FULL: every part has them.  trust: this workgroup knows that the rows are there.  Returns
// whether the tile is done (false: its rows were not there in time), the same for all threads.
template <int KIND, int S, bool FULL>
__device__ __forceinline__ bool cf_tile(const cf_chain_t& a, const cf_stage_t& s, int stage, int tile, bool trust, cf_lds_t& lds) {
    constexpr bool ADD = KIND == CF_ADD, GATED = KIND == CF_GATED;
    constexpr int SHARE = ADD ? 2 : 1, V = 2 / SHARE;           // parts an instruction takes; chains a wave
    constexpr int STEPS = S > 8 ? S / 2 : S;                    // of x at a time: the weights of twelve leave no registers for more
    constexpr int COLS = 16 / SHARE, ROWS = 16 / SHARE, OUT = GATED ? COLS / 2 : COLS;
    const int lane = threadIdx.x % PL_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PL_WAVE);
    const int r = lane % 16, c = lane / 16;
    const int K = s.K, n = a.n, n0 = tile * OUT;
    const bool asks = stage > 0 && !trust;

    auto k_of = [&](int v, int u) { return (ADD ? wave * 2 + r / 8 : wave * 2 + v) * s.part_len + u * 16 + c * 4; };
    auto is_step = [&](int v, int u) { return FULL || (u * 16 < s.part_len && k_of(v, u) < K); };

    // the weights first: they come from memory and depend on nothing
    const int wr = GATED && r >= OUT ? s.N + r - OUT : r % COLS;
    const __amdgpu_buffer_rsrc_t weights = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(s.w) + static_cast<size_t>(n0) * K, 0,
                                                                            4u * ((GATED ? s.N : 0) + OUT) * K, 0x00027000);
    const uint32_t w_at = 4u * (wr * K + k_of(0, 0));
    cn_words4 w[V][S];
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
        for (int u = 0; u < S; ++u)
            w[v][u] = __builtin_amdgcn_raw_buffer_load_b128(weights, is_step(v, u) ? w_at : CN_NOWHERE, 4 * (v * s.part_len + u * 16), 0);
    // (the norm's gains wait in LDS)
    if constexpr (!ADD)
        for (int k = threadIdx.x; k < K; k += CF_WAVES * PL_WAVE) lds.gain[k] = s.gain[k];

    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(s.x), 0, 4u * n * K, 0x00027000);
    const int t = threadIdx.x, at_row = t / OUT, at_col = t % OUT, col = n0 + at_col;      // the element that this thread finishes

    for (int row0 = 0, turn = 0; row0 < n; row0 += ROWS, turn ^= 1) {
        const int x_row = row0 + r % ROWS;
        const bool mine = at_row < ROWS && row0 + at_row < n;
        const uint32_t x_at = x_row < n ? 4u * cf_place(x_row, k_of(0, 0), n, K, s.x_laid) : CN_NOWHERE, each = s.x_laid ? 4 * n : 4;
        auto load = [&](int v, int u, auto policy) {
            return __builtin_amdgcn_raw_buffer_load_b128(rows, is_step(v, u) ? x_at : CN_NOWHERE, (v * s.part_len + u * 16) * each, decltype(policy)::value);
        };
        bool there = true;
        int left = a.looks;
        if (asks) {         // (one piece of the wave's rows until it is there, then all of them: once in any case, and as often again as looks are left)
            there = false;
            for (; left > 0 && !there; --left) {
                asm volatile("" ::: "memory");
                const cn_words4 p = load(0, 0, cn_past_l2_t{});
                there = __all(max(max(p[0], p[1]), max(p[2], p[3])) != PL_MISSING);
                if (!there) __builtin_amdgcn_s_sleep(1);
            }
        }
        f32x4 acc[V];
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] = f32x4{0.f, 0.f, 0.f, 0.f};
        uint32_t old = 0;
#pragma unroll
        for (int half = 0; half < S / STEPS; ++half) {
            cn_words4 x[V][STEPS];
            for (int again = 0; again <= left; ++again) {
                asm volatile("" ::: "memory");
                if (ADD && half == 0) old = mine ? cn_word(s.old + cf_place(row0 + at_row, col, n, s.N, s.old_laid)) : 0u;
                // (the first time through L2, which the workgroups of an XCD share; what a load that came too early has left there is seen to be missing)
                if (stage == 0 || (asks && again == 0)) {
#pragma unroll
                    for (int v = 0; v < V; ++v)
#pragma unroll
                        for (int u = 0; u < STEPS; ++u) x[v][u] = load(v, half * STEPS + u, cn_cached_t{});
                } else {
#pragma unroll
                    for (int v = 0; v < V; ++v)
#pragma unroll
                        for (int u = 0; u < STEPS; ++u) x[v][u] = load(v, half * STEPS + u, cn_past_l2_t{});
                }
                if (!asks) break;
                uint32_t most = old;
#pragma unroll
                for (int v = 0; v < V; ++v)
#pragma unroll
                    for (int u = 0; u < STEPS; ++u)
#pragma unroll
                        for (int e = 0; e < 4; ++e) most = max(most, x[v][u][e]);
                there = __all(most != PL_MISSING);
                if (there) break;
                __builtin_amdgcn_s_sleep(1);
            }
            if (!there) {
                left = 0;       // (of the second half too)
                if (lane == 0) lds.late[turn] = 1;
            }

            if constexpr (!ADD) {
                // x / sqrt(mean of squares + eps) * gain: sums of four squares to LDS, a wave a row adds them up as the norm kernel's workgroup does
                float* const fours = &lds.parts[0][0][0];           // [row][CF_FOURS] (free until the products' tiles come)
#pragma unroll
                for (int v = 0; v < V; ++v)
#pragma unroll
                    for (int u = 0; u < S; ++u) {
                        float four = 0.f;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float f = __uint_as_float(x[v][u][e]);
                            four += f * f;
                        }
                        if (is_step(v, u)) fours[r * CF_FOURS + k_of(v, u) / 4] = four;
                    }
                __syncthreads();
                if (__builtin_amdgcn_readfirstlane(lds.late[turn])) return false;
                for (int row = wave; row < n; row += CF_WAVES) {
                    float total = 0.f;
#pragma unroll
                    for (int q = 0; q < CF_WIDEST / 256; ++q) {
                        const int quad = q * PL_WAVE + lane;
                        total += wave_sum(quad * 4 < K ? fours[row * CF_FOURS + quad] : 0.f);
                    }
                    if (lane == 0) lds.denom[row] = sqrtf(total / static_cast<float>(K) + s.eps);
                }
                __syncthreads();
                const float denom = lds.denom[r], inverse = 1.f / denom;
                const bool plain = !(denom > 0x1p-40f && denom < 0x1p40f);
#pragma unroll
                for (int v = 0; v < V; ++v)
#pragma unroll
                    for (int u = 0; u < S; ++u) {
                        const f32x4 g = *reinterpret_cast<const f32x4*>(&lds.gain[is_step(v, u) ? k_of(v, u) : 0]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[v][u][e] = __float_as_uint(cf_quotient(__uint_as_float(x[v][u][e]), denom, inverse, plain) * g[e]);
                    }
            }

#pragma unroll
            for (int u = 0; u < STEPS; ++u)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int v = 0; v < V; ++v)
                        acc[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[v][half * STEPS + u][q]), __uint_as_float(x[v][u][q]), acc[v], 0, 0, 0);
        }
        // (a lane holds four columns of one row of x; with two parts an instruction, the blocks that mix them are nobody's)
        if (!ADD || c / 2 == r / 8) {
#pragma unroll
            for (int v = 0; v < V; ++v)
                *reinterpret_cast<f32x4*>(&lds.parts[turn][wave * 2 + (ADD ? r / 8 : v)][r % ROWS * COLS + c * 4 % COLS]) = acc[v];
        }
        __syncthreads();
        if (ADD && __builtin_amdgcn_readfirstlane(lds.late[turn])) return false;

        if (mine) {
            const int used = FULL ? CF_PARTS : pl_ceil_div(K, s.part_len);
            float sum = 0.f, up = 0.f;
#pragma unroll
            for (int p = 0; p < CF_PARTS; ++p) {
                if (FULL || p < used) {
                    sum += lds.parts[turn][p][at_row * COLS + at_col];
                    if (GATED) up += lds.parts[turn][p][at_row * COLS + OUT % COLS + at_col];
                }
            }
            if (ADD) sum = __uint_as_float(old) + sum;
            if (GATED) sum = pl_activate<true>(sum, a.act) * up;
            float* const to = s.y + cf_place(row0 + at_row, col, n, s.N, s.y_laid);
            cn_leave(to, s.y_laid ? cn_value(sum) : __float_as_uint(sum));
        }
    }
    return true;
}

template <int KIND, int S>
__device__ __forceinline__ bool cf_form(const cf_chain_t& a, const cf_stage_t& s, int stage, int tile, bool trust, cf_lds_t& lds) {
    if (s.K == CF_PARTS * S * 16) return cf_tile<KIND, S, true>(a, s, stage, tile, trust, lds);
    return cf_tile<KIND, S, false>(a, s, stage, tile, trust, lds);
}

// A tile of a stage whose results are not all there, the first from `from` on, so that workgroups that miss the same begin with unlike ones; -1: all are
// there.
__device__ __forceinline__ int cf_missing_tile(const __attribute__((address_space(4))) cf_chain_t& a, int stage, int from, cf_lds_t& lds) {
    const auto& s = a.s[stage];
    const int shift = s.kind == CF_STORE ? 4 : 3;       // (columns of a tile)
    int first = INT_MAX;
    const int turns = pl_ceil_div(s.N, CF_WAVES * PL_WAVE);
#pragma unroll 8        // (a look is a trip to memory: eight are on their way together)
    for (int i = 0; i < a.n * turns; ++i) {
        const int row = i / turns, col = min(i % turns * (CF_WAVES * PL_WAVE) + static_cast<int>(threadIdx.x), s.N - 1);
        const uint32_t word = cn_word(s.y + cf_place(row, col, a.n, s.N, s.y_laid));
        const int turned = (col >> shift) - from;
        first = word == PL_MISSING ? min(first, turned < 0 ? turned + s.tiles : turned) : first;
    }
    int* const least = &lds.least;
    if (threadIdx.x == 0) *least = INT_MAX;
    __syncthreads();
    if (first != INT_MAX) atomicMin(least, first);
    __syncthreads();
    const int found = __builtin_amdgcn_readfirstlane(*least);
    __syncthreads();
    return found == INT_MAX ? -1 : (found + from) % s.tiles;
}

// 128 registers a lane: two workgroups a compute unit, half of a layer's weights in registers at once.  (Two values do not fit: 12 bytes of
// scratch a lane.)
__global__ void __launch_bounds__(PL_WAVE * CF_WAVES, 4) gemm_chain_f32_kernel(cf_chain_t a) {
    __shared__ __attribute__((aligned(16))) cf_lds_t lds;
    cn_touch_arguments(sizeof(cf_chain_t));
    auto stage_of = [](const auto& a) {
        int stage = 0;
#pragma unroll
        for (int i = 1; i < CF_STAGES; ++i)
            if (i < a.stages && static_cast<int>(blockIdx.x) >= a.s[i].first) stage = i;
        return stage;
    };
    if (threadIdx.x < 2) lds.late[threadIdx.x] = 0;
    __syncthreads();
    int p = stage_of(a), q = static_cast<int>(blockIdx.x) - a.s[p].first;
    bool trust = false, own = true;     // (own: tile q of stage p is the workgroup's, and not one that it works out because it is missing)
    while (true) {
        p = __builtin_amdgcn_readfirstlane(p);
        q = __builtin_amdgcn_readfirstlane(q);
        const cf_stage_t& s = a.s[p];
        bool done;
        if (s.kind == CF_GATED) done = cf_form<CF_GATED, 4>(a, s, p, q, trust, lds);
        else if (s.kind == CF_STORE) done = cf_form<CF_STORE, 4>(a, s, p, q, trust, lds);
        else if (s.part_len <= 64) done = cf_form<CF_ADD, 4>(a, s, p, q, trust, lds);
        else if (s.part_len <= 128) done = cf_form<CF_ADD, 8>(a, s, p, q, trust, lds);
        else done = cf_form<CF_ADD, 12>(a, s, p, q, trust, lds);
        if (done && own) return;
        // The rows were not there in time: what the earlier stages have not left yet, stage by stage, then the workgroup's own tile once more.  (What the
        // workgroup has written is where its loads past L2 find it before it goes on.)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) {
            int zero;
            asm volatile("v_mov_b32 %0, 0" : "=v"(zero));       // (as a constant it is kept through the kernel, and something else spilt)
            lds.late[0] = lds.late[1] = zero;
        }
        __syncthreads();
        // (its arguments read here, where they are needed: as values kept from the kernel's beginning on they spill)
        const __attribute__((address_space(4))) cf_chain_t* args = (const __attribute__((address_space(4))) cf_chain_t*)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(args));
        const int stage = stage_of(*args), tile = static_cast<int>(blockIdx.x) - args->s[stage].first;
        if (!trust) {
            trust = true;
            p = 0;
        }
        for (q = -1; p < stage; ++p) {
            q = cf_missing_tile(*args, p, tile % args->s[p].tiles, lds);
            if (q >= 0) break;
        }
        own = q < 0;
        if (own) q = tile;
    }
}

// Whether the products of so many rows are this launch's: a stream of `width`, an output projection of inner width `inner`, a feed-forward of `ff`, and
// (0: none) `after` columns behind the next norm.  (The width's lower end: the norm kernel's workgroups have 256 threads from there on.)
extern "C" int pl_gemm_chain_f32_applies(int n, int width, int inner, int ff, int after) {
    return n > 0 && n <= CF_ROWS && width >= 512 && width <= CF_WIDEST && width % 64 == 0 && inner > 0 && inner <= CF_DEEPEST && inner % 64 == 0
           && ff > 0 && ff <= CF_DEEPEST && ff % 64 == 0 && after >= 0 && after % 16 == 0 && after <= (1 << 20);
}

// The words that one launch leaves between its stages, all ones before it: mid [n, width], hidden [n, ff] and out [n, width], which begins at word out.
extern "C" long pl_gemm_chain_f32_room(int n, int width, int ff) { return static_cast<long>(n) * (2 * static_cast<long>(width) + ff); }
extern "C" long pl_gemm_chain_f32_out(int n, int width, int ff) { return static_cast<long>(n) * (static_cast<long>(width) + ff); }

// As pl_gemm_chain (gemm_chain.hip), everything 32-bit and the weights as stored: w_out [width, inner], w_gated [2 ff, width] (gate rows first), w_down
// [width, ff], w_next [after, width] or null.
extern "C" int pl_gemm_chain_f32(const float* stream, int stream_laid, const float* rows, float* room, float* next, const float* w_out, const float* w_gated,
                                 const float* w_down, const float* w_next, const float* gain2, float eps2, const float* gain_next, float eps_next, int n,
                                 int width, int inner, int ff, int after, int act, int looks, hipStream_t stream_) {
    if (n == 0) return 0;
    PL_REQUIRE(pl_gemm_chain_f32_applies(n, width, inner, ff, after), "chain of products: %d rows, a stream of %d, inner widths %d and %d, %d columns behind it", n,
               width, inner, ff, after);
    PL_REQUIRE(stream && rows && room && w_out && w_gated && w_down && gain2, "chain of products: an operand is missing");
    PL_REQUIRE((w_next != nullptr) == (after > 0) && (next != nullptr) == (after > 0) && (gain_next != nullptr) == (after > 0),
               "chain of products: %d columns behind the chain", after);
    PL_REQUIRE(act >= PL_ACT_SILU && act <= PL_ACT_RELU2, "chain of products: activation code %d", act);
    PL_REQUIRE(looks >= 0, "chain of products: %d looks", looks);
    for (const float* p : {stream, rows, static_cast<const float*>(room), w_out, w_gated, w_down, w_next, gain2, gain_next, static_cast<const float*>(next)})
        PL_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "chain of products: an operand begins in the middle of 16 bytes");
    const bool follows = after > 0;
    float* const mid = room;
    float* const hidden = mid + static_cast<size_t>(n) * width;
    float* const out = room + pl_gemm_chain_f32_out(n, width, ff);
    cf_chain_t a{};
    a.n = n;
    a.act = act;
    a.looks = looks;
    a.stages = follows ? 4 : 3;
    //                x       w        y      old     gain     eps   N      K      part first tiles, (set below)   kind         x, old, y laid
    a.s[0] = cf_stage_t{rows, w_out, mid, stream, nullptr, 0.f, width, inner, 0, CF_ADD, 0, 0, 0, stream_laid ? 1 : 0, 1};
    a.s[1] = cf_stage_t{mid, w_gated, hidden, nullptr, gain2, eps2, ff, width, 0, CF_GATED, 0, 0, 1, 0, 1};
    a.s[2] = cf_stage_t{hidden, w_down, out, mid, nullptr, 0.f, width, ff, 0, CF_ADD, 0, 0, 1, 1, follows ? 1 : 0};
    a.s[3] = cf_stage_t{out, w_next, next, nullptr, gain_next, eps_next, after, width, 0, CF_STORE, 0, 0, 1, 0, 0};
    int grid = 0;
    for (int i = 0; i < a.stages; ++i) {
        cf_stage_t& s = a.s[i];
        s.part_len = pl_ceil_div(pl_ceil_div(s.K, CF_PARTS), 64) * 64;      // (gemm_f32.hip's)
        s.first = grid;
        s.tiles = s.N / (s.kind == CF_STORE ? 16 : 8);
        grid += s.tiles;
    }
    gemm_chain_f32_kernel<<<grid, PL_WAVE * CF_WAVES, 0, stream_>>>(a);
    PL_CHECK_LAUNCH("gemm_chain (32-bit)");
    return 0;
}
