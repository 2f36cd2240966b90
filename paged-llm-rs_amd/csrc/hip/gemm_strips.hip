// y[M, N] = silu(x . gate^T) * (x . up^T) for many rows of bfloat16, 32-bit sums, out of weights in strips
// (kernels.weights_in_strips), on the matrix cores.
//
// A strip tile is 16 rows of w by 32 k as the lanes of a wave take them, so the weights go from memory straight into the
// registers that multiply them, two stages of 64 k ahead, and pass LDS by: the four waves of a workgroup own different columns and
// all of its rows of x, which alone go through LDS (registers, two stages of LDS, 16-byte pieces permuted by their row against bank
// conflicts).  A wave's tile of 32 CT columns by 32 RT rows then reads LDS once for CT matrix instructions, where a tile whose operands both
// come through LDS (gemm_tiled.hip) reads it once an instruction.  v_mfma_f32_32x32x16_bf16, A = w: rows 0 .. 15 of A are a strip of gate,
// 16 .. 31 the strip of up that belongs to it, so a lane holds gate and up of the same columns.
//
// Reads of LDS, loads and stores into LDS are dealt between the matrix instructions one by one: asked for together in front of them
// they kept the matrix cores waiting for what LDS gives a compute unit in turn (a stage of 64 k by 128 rows by 256 columns 0.71 us, 0.54 so;
// its instructions alone 0.43).  The loop is bound by the matrix cores at 70 to 85% of their rate while the operands come out of L2, by the
// 64 bytes a clock that a compute unit takes in at the small tiles, and with few rows before wide weights by the weights' trip from memory.
// Beside it a workgroup pays some 5 us for its launch, its first loads and its tile's way out.
//
// us, library's product and activation kernel / this one (before: gemm_tiled up to 1,024 rows of width 1,024, in brackets): 3,072 columns of
// 1,024: 100 rows 15.8 / 9.4 (17.2), 300 17.6 / 9.8 (16.6), 512 21 / 12.3 (17.5), 1,024 25 / 18 (25), 2,048 37 / 28 (41), 4,096 64 / 51;
// 12,288 columns of 4,096: 65 rows 57 / 45, 575 125 / 112, 1,024 175 / 168, and 2,048 294 / 332: the library's.
#include "common.hpp"

typedef __bf16 gs_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 gs_bf16x2 __attribute__((ext_vector_type(2)));
typedef float gs_f32x16 __attribute__((ext_vector_type(16)));
typedef float gs_f32x4 __attribute__((ext_vector_type(4)));
typedef float gs_f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t gs_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t gs_u32x2 __attribute__((ext_vector_type(2)));

#define GS_BK 64           // K a stage
#define GS_BAND 16         // row tiles that are walked before the next column tile's

__device__ __forceinline__ uint32_t gs_pack2(float lo, float hi) {
    const gs_f32x2 pair = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, gs_bf16x2));
}

// silu(g), the division by the hardware's reciprocal (1 ulp of 32 bits; what leaves is bfloat16)
__device__ __forceinline__ float gs_silu(float g) { return g * __builtin_amdgcn_rcpf(1.f + __expf(-g)); }

template <int V>
struct GsInt {
    static constexpr int value = V;
};

// The workgroup's tile.  Workgroups go to the eight XCDs in turn; an XCD gets tiles that follow each other, the row tiles of one column
// tile first, so that its L2 reads a row of w once.
__device__ __forceinline__ void gs_tile(int at, int row_tiles, int col_tiles, int& row_tile, int& col_tile) {
    const int total = row_tiles * col_tiles, each = total / 8, rest = total % 8;
    const int xcd = at % 8;
    const int work = xcd * each + min(xcd, rest) + at / 8;
    const int band = work / (GS_BAND * col_tiles), in_band = work - band * GS_BAND * col_tiles;
    const int rows = min(GS_BAND, row_tiles - band * GS_BAND);
    row_tile = band * GS_BAND + in_band % rows;
    col_tile = in_band / rows;
}

constexpr int gs_out_cols(int CT) { return 4 * 16 * CT; }
// bytes between two rows of the tile on its way out
constexpr int gs_pitch(int CT) { return gs_out_cols(CT) * 2 + 16; }
constexpr int gs_lds_bytes(int CT, int RT) {
    const int in = 2 * 32 * RT * GS_BK * 2, out = 32 * RT * gs_pitch(CT);
    return in > out ? in : out;
}

// CT, RT: a wave's tiles of 32 rows of w (16 of gate, 16 of up) and of 32 rows of x.  N a multiple of 16, K of 64; rows and columns past the
// matrices are read from their last and not stored.
template <int CT, int RT, int PER_SIMD>
__global__ void __launch_bounds__(256, PER_SIMD)
gemm_strips_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ strips, bf16_t* __restrict__ y, int M, int N, int K,
                   int row_tiles, int col_tiles) {
    constexpr int ROWS = 32 * RT, STAGE = ROWS * GS_BK * 2;
    extern __shared__ __attribute__((aligned(16))) char gs_lds[];          // two stages of x [row][64], then the tile on its way out
    int row_tile, col_tile;
    gs_tile(blockIdx.x, row_tiles, col_tiles, row_tile, col_tile);
    const int m0 = row_tile * ROWS;
    const int tid = threadIdx.x, lane = tid % PL_WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / PL_WAVE);
    const int r32 = lane % 32, h = lane / 32;
    constexpr int COLS = 16 * CT;                                          // output columns a wave
    const int n_wave = (col_tile * 4 + wave) * COLS;                       // the wave's first

    const int last_strip = N / 16 - 1;                                     // of gate
    uint32_t w_at[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int strip = min(n_wave / 16 + c, last_strip) + (r32 < 16 ? 0 : N / 16);
        w_at[c] = static_cast<uint32_t>(strip) * static_cast<uint32_t>(K) * 32u + h * 256 + r32 % 16 * 16;
    }
    uint32_t x_at[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
        x_at[i] = static_cast<uint32_t>(min(m0 + tid / 8 + 32 * i, M - 1)) * static_cast<uint32_t>(K) * 2u + tid % 8 * 16;
    char* const put_at = gs_lds + tid / 8 * 128 + ((tid % 8) ^ (tid / 8 % 8)) * 16;
    int b_at[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) b_at[kk] = r32 * 128 + (((2 * kk + h) ^ (r32 % 8)) * 16);

    const int stages = K / GS_BK;
    gs_bf16x8 w[2][4][CT], b[2][RT];
    gs_u32x4 xr[2][RT];
    gs_f32x16 acc[CT][RT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[c][t][i] = 0.f;

    // (past the end the last stage is asked for again)
    auto ask_w = [&](auto set, auto kk, int s, int c) {
        const char* from = reinterpret_cast<const char*>(strips) + static_cast<size_t>(min(s, stages - 1)) * 2048 + kk.value * 512;
        w[set.value][kk.value][c] = *reinterpret_cast<const gs_bf16x8*>(from + w_at[c]);
    };
    auto ask_x = [&](auto set, int s, int i) {
        const char* from = reinterpret_cast<const char*>(x) + static_cast<size_t>(min(s, stages - 1)) * 128;
        xr[set.value][i] = *reinterpret_cast<const gs_u32x4*>(from + x_at[i]);
    };
    auto put_x = [&](auto set, int s, int i) {
        *reinterpret_cast<gs_u32x4*>(put_at + (s % 2) * STAGE + i * 32 * 128) = xr[set.value][i];
    };
    auto read_b = [&](auto set, int s, int kk, int t) {
        b[set.value][t] = *reinterpret_cast<const gs_bf16x8*>(gs_lds + (s % 2) * STAGE + b_at[kk] + t * 32 * 128);
    };
    auto meet = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto slice = [&](auto set, auto kk, int s) {
        constexpr int KK = decltype(kk)::value, SET = decltype(set)::value;
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                const int m = c * RT + t;
                if (KK == 3 && m == 1) meet();
                if (m >= 1 && m <= RT) {
                    if constexpr (KK < 3) read_b(GsInt<(KK + 1) % 2>{}, s, KK + 1, m - 1);
                    else read_b(GsInt<0>{}, s + 1, 0, m - 1);
                }
                if (KK == 1 && c == (CT > 1 ? 1 : 0)) put_x(GsInt<1 - SET>{}, s + 1, t);
                __builtin_amdgcn_sched_barrier(0);
                acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[SET][KK][c], b[KK % 2][t], acc[c][t], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (KK == 2 && c == 0) ask_x(GsInt<1 - SET>{}, s + 3, t);
                if (t == RT - 1) ask_w(set, kk, s + 2, c);
                if (CT == 1 && t == RT - 1) {
                    if constexpr (KK < 3) read_b(GsInt<(KK + 1) % 2>{}, s, KK + 1, t);
                    else read_b(GsInt<0>{}, s + 1, 0, t);
                }
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto stage = [&](auto set, int s) {
        slice(set, GsInt<0>{}, s);
        slice(set, GsInt<1>{}, s);
        slice(set, GsInt<2>{}, s);
        slice(set, GsInt<3>{}, s);
    };
    auto ask_all = [&](auto set, int s) {
#pragma unroll
        for (int i = 0; i < RT; ++i) ask_x(set, s, i);
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            ask_w(set, GsInt<0>{}, s, c);
            ask_w(set, GsInt<1>{}, s, c);
            ask_w(set, GsInt<2>{}, s, c);
            ask_w(set, GsInt<3>{}, s, c);
        }
    };
    ask_all(GsInt<0>{}, 0);
    ask_all(GsInt<1>{}, 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RT; ++i) put_x(GsInt<0>{}, 0, i);
#pragma unroll
    for (int i = 0; i < RT; ++i) ask_x(GsInt<0>{}, 2, i);
    meet();
#pragma unroll
    for (int t = 0; t < RT; ++t) read_b(GsInt<0>{}, 0, 0, t);
    int s = 0;
    for (; s + 1 < stages; s += 2) {
        stage(GsInt<0>{}, s);
        stage(GsInt<1>{}, s + 1);
    }
    if (s < stages) stage(GsInt<0>{}, s);
    __syncthreads();

    // The tile leaves through LDS in whole rows.  acc[c][t][4 j + i]: row 32 t + r32, row of A 8 j + 4 h + i
    constexpr int PITCH = gs_pitch(CT), LANES = 4 * COLS / 8;              // (lanes of a row)
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        char* at_row = gs_lds + (32 * t + r32) * PITCH + wave * COLS * 2;
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = gs_silu(acc[c][t][4 * j + i]) * acc[c][t][4 * (j + 2) + i];
                const gs_u32x2 packed = {gs_pack2(v[0], v[1]), gs_pack2(v[2], v[3])};
                *reinterpret_cast<gs_u32x2*>(at_row + (16 * c + 8 * j + 4 * h) * 2) = packed;
            }
    }
    __syncthreads();
    const int n0 = col_tile * 4 * COLS;
    for (int i = tid; i < ROWS * LANES; i += 256) {
        const int r = i / LANES, piece = i % LANES;
        if (m0 + r < M && n0 + piece * 8 < N)
            *reinterpret_cast<gs_u32x4*>(y + static_cast<size_t>(m0 + r) * N + n0 + piece * 8) =
                *reinterpret_cast<const gs_u32x4*>(gs_lds + r * PITCH + piece * 16);
    }
}

template <int CT, int RT, int PER_SIMD>
static int gs_launch(const void* x, const void* strips, void* y, int M, int N, int K, hipStream_t stream) {
    constexpr int lds = gs_lds_bytes(CT, RT);
    static_assert(lds <= 64 * 1024, "a workgroup's LDS");
    const int row_tiles = pl_ceil_div(M, 32 * RT), col_tiles = pl_ceil_div(N, gs_out_cols(CT));
    gemm_strips_kernel<CT, RT, PER_SIMD><<<row_tiles * col_tiles, 256, lds, stream>>>(
        static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(strips), static_cast<bf16_t*>(y), M, N, K, row_tiles, col_tiles);
    PL_CHECK_LAUNCH("gemm_strips");
    return 0;
}

// The tiles there are, and what one costs a compute unit: us for the tile itself and for 64 k, as timed one tile a compute unit
// (K of 1,024 and of 3,072).  A launch is taken to last as long as the compute unit with most tiles: that is the order of the shapes in all
// of 40 timed products (65 to 4,096 rows of 1,024, 4,096 and 5,120) but for differences of a few per cent.
struct GsShape {
    int ct, rt;
    float tile, stage;
};
static const GsShape GS_SHAPES[] = {{1, 2, 3.0f, 0.25f}, {1, 4, 2.9f, 0.37f}, {2, 3, 5.2f, 0.425f}, {2, 4, 5.8f, 0.54f}, {3, 4, 9.0f, 0.755f}};

static int gs_pick(int M, int N, int K) {
    int best = 0;
    float least = 0.f;
    for (int i = 0; i < 5; ++i) {
        const GsShape& s = GS_SHAPES[i];
        const long tiles = static_cast<long>(pl_ceil_div(M, 32 * s.rt)) * pl_ceil_div(N, gs_out_cols(s.ct));
        const float cost = static_cast<float>((tiles + pl_compute_units() - 1) / pl_compute_units()) * (s.tile + K / GS_BK * s.stage);
        if (i == 0 || cost < least) best = i, least = cost;
    }
    return best;
}

// Whether a shape is served: N (of gate) a multiple of 16, K of 64, and offsets of 32 bits into x and into the weights.
extern "C" int pl_gemm_strips_apply(int M, int N, int K) {
    return M > 0 && N > 0 && K > 0 && N % 16 == 0 && K % GS_BK == 0 && static_cast<long long>(M) * K < (1ll << 31) &&
           2ll * N * K < (1ll << 31) && static_cast<long long>(pl_ceil_div(M, 64)) * pl_ceil_div(N, 64) < (1ll << 30);
}

// x: bfloat16 [M, K].  strips: bfloat16 [2 N, K], gate rows first, in strips.  y: bfloat16 [M, N].  All aligned to 16 bytes.
extern "C" int pl_gemm_strips(const void* x, const void* strips, void* y, int M, int N, int K, hipStream_t stream) {
    PL_REQUIRE(pl_gemm_strips_apply(M, N, K), "product out of strips: %d rows, %d columns, inner width %d", M, N, K);
    PL_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(strips) | reinterpret_cast<uintptr_t>(y)) % 16 == 0,
               "product out of strips: rows that are not aligned to 16 bytes");
    switch (gs_pick(M, N, K)) {
        case 0: return gs_launch<1, 2, 2>(x, strips, y, M, N, K, stream);
        case 1: return gs_launch<1, 4, 2>(x, strips, y, M, N, K, stream);
        case 2: return gs_launch<2, 3, 2>(x, strips, y, M, N, K, stream);
        case 3: return gs_launch<2, 4, 1>(x, strips, y, M, N, K, stream);
        default: return gs_launch<3, 4, 1>(x, strips, y, M, N, K, stream);
    }
}
