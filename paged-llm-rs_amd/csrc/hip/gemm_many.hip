// y[M, N] = x[M, K] . w[N, K]^T for many rows of bfloat16, 32-bit sums, on the matrix cores, with what stands around the product fused into it:
// the norm in front of it (what an earlier product left of it), the gated activation, the sum into the residual stream and the norm behind that.
//
// A workgroup of four waves owns 32 RT rows of x and 128 CT rows of w; a wave all of the former and a quarter of the latter, as tiles of
// v_mfma_f32_32x32x16_bf16 with A = w: a lane then holds, for one row of x, groups of four neighbouring columns.  K is walked 64 a stage, two stages
// and more asked for ahead.  The rows of x go through registers and two stages of LDS, their 16-byte pieces permuted by their row against bank
// conflicts.  The weights in strips (kernels.weights_in_strips: 16 rows by 32 k as the lanes of a wave take them) go from memory straight into the
// registers that multiply them, and pass LDS by: it is read once for CT matrix instructions, where a tile whose operands are shared by two waves each
// (gemm_tiled.hip) reads it once an instruction.  Weights in rows, as they are stored, go through LDS as x does, a wave's through a part of
// its own (100 and 2,048 rows, 3,072 gated columns of 1,024: 9.8 and 28.3 us, 9.0 and 27.5 in strips).
//
// Reads of LDS, loads and stores into LDS are dealt between the matrix instructions one by one: asked for together in front of them
// they kept the matrix cores waiting for what LDS gives a compute unit in turn (a stage of 64 k by 128 rows by 256 columns 0.71 us, 0.54 so;
// its instructions alone 0.43).  The loop is bound by the matrix cores at 70 to 85% of their rate while the operands come out of L2, by the
// 64 bytes a clock that a compute unit takes in at the small tiles, and with few rows before wide weights by the weights' trip from memory.
// Beside it a workgroup pays some 5 us for its launch, its first loads and its tile's way out.
//
// us, before (the library's product and the kernels around it; gemm_tiled for gated columns up to 1,024 rows) / this one.  Gated, 3,072 columns
// of 1,024: 100 rows 17 / 9.4, 512 17.5 / 12.3, 1,024 25 / 18, 2,048 37 / 28, 4,096 64 / 51; 12,288 of 4,096: 65 rows 57 / 45, 575 125 / 112, and
// 2,048 294 / 332: the library's.  Added into the stream with the norm behind it, 1,024 columns: of 2,048, 512 rows 13.7 / 13.2, 2,048 22.5 / 16.7; of
// 3,072, 2,048 rows 26.6 / 21.1.  Plain, 4,096 columns of 1,024: 300 rows 10 / 7.5, 1,024 13.3 / 12.3, 2,048 20.3 / 20.8.
#include "common.hpp"
#include "head_rows.hpp"

typedef __bf16 gm_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 gm_bf16x2 __attribute__((ext_vector_type(2)));
typedef float gm_f32x16 __attribute__((ext_vector_type(16)));
typedef float gm_f32x4 __attribute__((ext_vector_type(4)));
typedef float gm_f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t gm_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t gm_u32x2 __attribute__((ext_vector_type(2)));

#define GM_STORE 0         // y (bfloat16) = result
#define GM_SWIGLU 1        // w is [gate | up], N rows each: y (bfloat16) = silu(gate) * up
#define GM_ADD 2           // y (32-bit, the residual stream) += result
#define GM_STORE32 3       // y (32-bit) = result
#define GM_HEADS 4         // rows [q | k | v] of heads of 128: q normed and turned into y (bfloat16 [M, N]), k (the same) and v into the pages (GmHeads)

#define GM_BK 64           // K a stage
#define GM_STRIPE 64       // columns of the stream whose squares are one number of a norm handed forward
#define GM_BAND 16         // row tiles that are walked before the next column tile's

// Norms on both sides of a product (kernels.HandedNorm).
struct GmNorms {
    const float* taken;        // [M, taken_count]: sums of squares of the rows of the stream that x is bfloat16(row * gain) of; the
    int taken_count;           // (a multiple of four) result is scaled by 1 / sqrt(their sum / K + eps); null: x is what it is
    float eps;
    const float* gain;         // [N] of the norm behind the updated stream (GM_ADD): left behind are
    bf16_t* rows;              // [M, N] bfloat16(y * gain) and
    float* sums;               // [M, N / 64] the sums of squares of every 64 columns of y; null: no norm
};
#define GM_TAKEN_MOST 64

// What GM_HEADS does with its rows: qk_norm_rope_kv_write_128_kernel's work, on the tile on its way out (heads of 128 rotated whole or not at all).
struct GmHeads {
    const void *q_gain, *k_gain;       // [128] or null
    int gain_dtype;
    float eps;
    const float *cos_table, *sin_table;        // [positions, 64] or null
    const int *positions, *seq_of, *block_table;
    int max_blocks, block_size;
    bf16_t *k_pool, *v_pool;
    int nq, nkv;
};

// Grouped: the rows are dealt to groups (experts), every group with a weight matrix of its own, one behind the other in w.  A tile of 128 rows belongs to one
// group (`tile_group`; the tiles in use come first, and how many they are stands behind the last of all); row r of the tiles reads row gather[r] of x (null: row r itself; negative: a row of
// padding, which reads row 0 and whose result nobody looks at) and writes row r of y.
struct GmGroups {
    const int* tile_group;     // [row tiles + 1]
    const int* gather;         // [row tiles * 128] or null
    long long w_stride;        // elements between two groups' matrices
    int x_pitch, y_pitch;      // elements between two rows of x and of y
    int last, N_last, K_last;  // one group, `last` (-1: none), may have a matrix of other sizes: w_last, [N_last (2 N_last with GM_SWIGLU), K_last]
    const bf16_t* w_last;
};

__device__ __forceinline__ uint32_t gm_pack2(float lo, float hi) {
    const gm_f32x2 pair = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, gm_bf16x2));
}

// silu(g), the division by the hardware's reciprocal (1 ulp of 32 bits; what leaves is bfloat16)
__device__ __forceinline__ float gm_silu(float g) { return g * __builtin_amdgcn_rcpf(1.f + __expf(-g)); }

template <int V>
struct GmInt {
    static constexpr int value = V;
};

// The workgroup's tile.  Workgroups go to the eight XCDs in turn; an XCD gets tiles that follow each other, the row tiles of one column
// tile first, so that its L2 reads a row of w once.
__device__ __forceinline__ void gm_tile(int at, int row_tiles, int col_tiles, int& row_tile, int& col_tile) {
    const int total = row_tiles * col_tiles, each = total / 8, rest = total % 8;
    const int xcd = at % 8;
    const int work = xcd * each + min(xcd, rest) + at / 8;
    const int band = work / (GM_BAND * col_tiles), in_band = work - band * GM_BAND * col_tiles;
    const int rows = min(GM_BAND, row_tiles - band * GM_BAND);
    row_tile = band * GM_BAND + in_band % rows;
    col_tile = in_band / rows;
}

constexpr int gm_out_cols(int CT, int epi) { return 4 * (epi == GM_SWIGLU ? 16 : 32) * CT; }
constexpr bool gm_is_32(int epi) { return epi == GM_ADD || epi == GM_STORE32; }
// bytes between two rows of the tile on its way out
constexpr int gm_pitch(int CT, int epi) { return gm_out_cols(CT, epi) * (gm_is_32(epi) ? 4 : 2) + 16; }
// ... and of the LDS of a workgroup: two stages of x (and of weights in rows), or the tile on its way out, and 1 / rms of its rows (with GM_HEADS also
// their positions and places in the pages)
constexpr int gm_lds_bytes(int CT, int RT, int epi, bool strips) {
    const int in = 2 * 32 * RT * GM_BK * 2 + (strips ? 0 : 4 * 2 * 32 * CT * GM_BK * 2), out = 32 * RT * gm_pitch(CT, epi);
    return (in > out ? in : out) + 32 * RT * (epi == GM_HEADS ? 12 : 4);
}

// CT, RT: a wave's tiles of 32 rows of w (with GM_SWIGLU 16 of gate, 16 of up) and of 32 rows of x.  N a multiple of 16, K of 64; rows and columns past the
// matrices are read from their last and not stored.
// STRIPS: the weights in strips; otherwise in rows as they are stored, which go through registers and LDS as the rows of x do, each wave's
// through a part of LDS of its own.  The sums are the same, k after k: the layout changes no bit.
template <int CT, int RT, int PER_SIMD, int EPI, bool TAKES, bool STRIPS, bool GROUPED = false>
__global__ void __launch_bounds__(256, PER_SIMD)
gemm_many_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ weights, void* __restrict__ y_, int M, int N, int K,
                   int row_tiles, int col_tiles, GmNorms norms, GmGroups groups, GmHeads heads) {
    static_assert(!GROUPED || (RT == 4 && !TAKES && !STRIPS && EPI != GM_ADD), "groups' tiles are of 128 rows");
    constexpr int ROWS = 32 * RT, STAGE = ROWS * GM_BK * 2;
    extern __shared__ __attribute__((aligned(16))) char gm_lds[];          // two stages of x [row][64], then the tile on its way out
    int row_tile, col_tile;
    if constexpr (GROUPED) {
        row_tiles = groups.tile_group[row_tiles];                          // those that are used: the XCDs share them evenly
        if (static_cast<int>(blockIdx.x) >= row_tiles * col_tiles) return; // (the whole workgroup)
    }
    gm_tile(blockIdx.x, row_tiles, col_tiles, row_tile, col_tile);
    const int m0 = row_tile * ROWS;
    const int tid = threadIdx.x, lane = tid % PL_WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / PL_WAVE);
    const int r32 = lane % 32, h = lane / 32;
    constexpr int COLS = gm_out_cols(CT, EPI) / 4;                         // output columns a wave
    const int n_wave = (col_tile * 4 + wave) * COLS;                       // the wave's first
    int x_pitch = K, y_pitch = N;
    if constexpr (GROUPED) {
        const int group = groups.tile_group[row_tile];
        if (group == groups.last) {
            weights = groups.w_last;
            N = groups.N_last;
            K = groups.K_last;
        } else {
            weights += static_cast<long long>(group) * groups.w_stride;
        }
        if (col_tile * 4 * COLS >= N) return;                              // (this group has fewer columns than another)
        x_pitch = groups.x_pitch;
        y_pitch = groups.y_pitch;
    }

    const int last_strip = N / 16 - 1;                                     // (of gate alone)
    auto strip_of = [&](int c, int half) {                                 // the strip of either half of an instruction's 32 rows
        return EPI == GM_SWIGLU ? min(n_wave / 16 + c, last_strip) + half * (N / 16) : min(n_wave / 16 + 2 * c + half, last_strip);
    };
    // bytes from the weights' first: a lane's operands in strips; its pieces of rows 0 .. 7 of either half
    uint32_t w_at[CT][STRIPS ? 1 : 2];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        if constexpr (STRIPS) {
            w_at[c][0] = static_cast<uint32_t>(strip_of(c, r32 / 16)) * static_cast<uint32_t>(K) * 32u + h * 256 + r32 % 16 * 16;
        } else {
#pragma unroll
            for (int half = 0; half < 2; ++half)
                w_at[c][half] = (static_cast<uint32_t>(strip_of(c, half)) * 16u + lane / 8) * static_cast<uint32_t>(K) * 2u + lane % 8 * 16;
        }
    }
    uint32_t x_at[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        int row = min(m0 + tid / 8 + 32 * i, M - 1);
        if constexpr (GROUPED) {
            if (groups.gather != nullptr) row = max(groups.gather[row], 0);
        }
        x_at[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(x_pitch) * 2u + tid % 8 * 16;
    }
    char* const w_lds = gm_lds + 2 * STAGE + wave * 2 * CT * 4096;         // the wave's weights in rows: two stages of [32 CT][64]
    char* const put_w_at = w_lds + lane / 8 * 128 + ((lane % 8) ^ (lane / 8)) * 16;
    char* const put_at = gm_lds + tid / 8 * 128 + ((tid % 8) ^ (tid / 8 % 8)) * 16;
    int b_at[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) b_at[kk] = r32 * 128 + (((2 * kk + h) ^ (r32 % 8)) * 16);

    const int stages = K / GM_BK;
    // w: weights on their way or, in strips, the operands [set][k / 16 in the stage][c]; in rows the pieces [set][rows / 8][c], whose operands are a
    gm_bf16x8 w[2][4][CT], a[2][CT], b[2][RT];
    gm_u32x4 xr[2][RT];
    gm_f32x16 acc[CT][RT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[c][t][i] = 0.f;

    // (past the end the last stage is asked for again)
    auto ask_w = [&](auto set, auto kk, int s, int c) {
        constexpr int KK = decltype(kk)::value;
        const char* from = reinterpret_cast<const char*>(weights) + static_cast<size_t>(min(s, stages - 1)) * (STRIPS ? 2048 : 128);
        if constexpr (STRIPS) w[set.value][KK][c] = *reinterpret_cast<const gm_bf16x8*>(from + KK * 512 + w_at[c][0]);
        else w[set.value][KK][c] = *reinterpret_cast<const gm_bf16x8*>(from + static_cast<size_t>(KK % 2) * 16 * K + w_at[c][KK / 2]);
    };
    auto put_w = [&](auto set, auto kk, int s, int c) {
        *reinterpret_cast<gm_bf16x8*>(put_w_at + (s % 2) * CT * 4096 + c * 4096 + kk.value * 1024) = w[set.value][kk.value][c];
    };
    auto read_a = [&](auto set, int s, int kk, int c) {
        a[set.value][c] = *reinterpret_cast<const gm_bf16x8*>(w_lds + (s % 2) * CT * 4096 + c * 4096 + b_at[kk]);
    };
    auto ask_x = [&](auto set, int s, int i) {
        const char* from = reinterpret_cast<const char*>(x) + static_cast<size_t>(min(s, stages - 1)) * 128;
        xr[set.value][i] = *reinterpret_cast<const gm_u32x4*>(from + x_at[i]);
    };
    auto put_x = [&](auto set, int s, int i) {
        *reinterpret_cast<gm_u32x4*>(put_at + (s % 2) * STAGE + i * 32 * 128) = xr[set.value][i];
    };
    auto read_b = [&](auto set, int s, int kk, int t) {
        b[set.value][t] = *reinterpret_cast<const gm_bf16x8*>(gm_lds + (s % 2) * STAGE + b_at[kk] + t * 32 * 128);
    };
    auto meet = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // 16 k.  The next 16's operands are read, and what else there is to do is done, an instruction of it between two of the matrix cores'.
    // (The weights in rows: a stage's are laid down in LDS by the wave that reads them, a quarter a slice, while the stage before is multiplied.)
    auto slice = [&](auto set, auto kk, int s) {
        constexpr int KK = decltype(kk)::value, SET = decltype(set)::value;
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                const int m = c * RT + t;
                if (KK == 3 && m == 1) meet();
                if (m >= 1 && m <= RT) {
                    if constexpr (KK < 3) read_b(GmInt<(KK + 1) % 2>{}, s, KK + 1, m - 1);
                    else read_b(GmInt<0>{}, s + 1, 0, m - 1);
                }
                if constexpr (!STRIPS) {
                    // (the last quarter is written in front of the first read of what it is a part of)
                    if (t == 0) put_w(GmInt<1 - SET>{}, kk, s + 1, c);
                    if (c == CT - 1 && t >= RT - CT && t < RT) {
                        if constexpr (KK < 3) read_a(GmInt<(KK + 1) % 2>{}, s, KK + 1, t - RT + CT);
                        else read_a(GmInt<0>{}, s + 1, 0, t - RT + CT);
                    }
                }
                if (KK == 1 && c == (CT > 1 ? 1 : 0)) put_x(GmInt<1 - SET>{}, s + 1, t);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (STRIPS) acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[SET][KK][c], b[KK % 2][t], acc[c][t], 0, 0, 0);
                else acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[KK % 2][c], b[KK % 2][t], acc[c][t], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (KK == 2 && c == 0) ask_x(GmInt<1 - SET>{}, s + 3, t);
                if (t == RT - 1) {
                    if constexpr (STRIPS) ask_w(set, kk, s + 2, c);
                    else ask_w(GmInt<1 - SET>{}, kk, s + 3, c);
                }
                if (CT == 1 && t == RT - 1) {
                    if constexpr (KK < 3) read_b(GmInt<(KK + 1) % 2>{}, s, KK + 1, t);
                    else read_b(GmInt<0>{}, s + 1, 0, t);
                }
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto stage = [&](auto set, int s) {
        slice(set, GmInt<0>{}, s);
        slice(set, GmInt<1>{}, s);
        slice(set, GmInt<2>{}, s);
        slice(set, GmInt<3>{}, s);
    };
    auto ask_all = [&](auto set, int s) {
#pragma unroll
        for (int i = 0; i < RT; ++i) ask_x(set, s, i);
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            ask_w(set, GmInt<0>{}, s, c);
            ask_w(set, GmInt<1>{}, s, c);
            ask_w(set, GmInt<2>{}, s, c);
            ask_w(set, GmInt<3>{}, s, c);
        }
    };
    // where the tile's rows stand, a thread a row (its page is asked for behind the first stages and looked at when the tile leaves)
    int row_pos = -1, row_seq = 0, row_page = -1;
    if constexpr (EPI == GM_HEADS) {
        if (tid < ROWS && m0 + tid < M) {
            row_pos = heads.positions[m0 + tid];
            row_seq = heads.seq_of[m0 + tid];
        }
    }
    // the sums of squares of the tile's rows, four lanes a row, asked for first
    constexpr int PASSES = (ROWS + 63) / 64;
    gm_f32x4 sums[TAKES ? PASSES : 1][GM_TAKEN_MOST / 16];
    if constexpr (TAKES) {
#pragma unroll
        for (int q = 0; q < PASSES; ++q) {
            const float* from = norms.taken + static_cast<size_t>(min(m0 + 64 * q + tid / 4, M - 1)) * norms.taken_count + tid % 4 * 4;
#pragma unroll
            for (int i = 0; i < GM_TAKEN_MOST / 16; ++i) {
                sums[q][i] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
                if (16 * i + tid % 4 * 4 < norms.taken_count) sums[q][i] = *reinterpret_cast<const gm_f32x4*>(from + 16 * i);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    ask_all(GmInt<0>{}, 0);
    ask_all(GmInt<1>{}, 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (EPI == GM_HEADS) {
        if (row_pos >= 0) row_page = heads.block_table[static_cast<size_t>(row_seq) * heads.max_blocks + row_pos / heads.block_size];
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) put_x(GmInt<0>{}, 0, i);
#pragma unroll
    for (int i = 0; i < RT; ++i) ask_x(GmInt<0>{}, 2, i);
    if constexpr (!STRIPS) {
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            put_w(GmInt<0>{}, GmInt<0>{}, 0, c);
            put_w(GmInt<0>{}, GmInt<1>{}, 0, c);
            put_w(GmInt<0>{}, GmInt<2>{}, 0, c);
            put_w(GmInt<0>{}, GmInt<3>{}, 0, c);
            ask_w(GmInt<0>{}, GmInt<0>{}, 2, c);
            ask_w(GmInt<0>{}, GmInt<1>{}, 2, c);
            ask_w(GmInt<0>{}, GmInt<2>{}, 2, c);
            ask_w(GmInt<0>{}, GmInt<3>{}, 2, c);
        }
    }
    float* const scales = reinterpret_cast<float*>(gm_lds + gm_lds_bytes(CT, RT, EPI, STRIPS) - ROWS * 4);
    int* const places = reinterpret_cast<int*>(scales) - 2 * ROWS;         // (GM_HEADS) [row]: its position and its row of the pages, or -1
    if constexpr (TAKES) {
#pragma unroll
        for (int q = 0; q < PASSES; ++q) {
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < GM_TAKEN_MOST / 16; ++i) sum += (sums[q][i][0] + sums[q][i][1]) + (sums[q][i][2] + sums[q][i][3]);
            sum += __shfl_xor(sum, 1, PL_WAVE);
            sum += __shfl_xor(sum, 2, PL_WAVE);
            if (tid % 4 == 0 && 64 * q + tid / 4 < ROWS) scales[64 * q + tid / 4] = 1.f / sqrtf(sum / K + norms.eps);
        }
    }
    meet();
#pragma unroll
    for (int t = 0; t < RT; ++t) read_b(GmInt<0>{}, 0, 0, t);
    if constexpr (!STRIPS) {
#pragma unroll
        for (int c = 0; c < CT; ++c) read_a(GmInt<0>{}, 0, 0, c);
    }
    int s = 0;
    for (; s + 1 < stages; s += 2) {
        stage(GmInt<0>{}, s);
        stage(GmInt<1>{}, s + 1);
    }
    if (s < stages) stage(GmInt<0>{}, s);
    constexpr int PITCH = gm_pitch(CT, EPI), OUT_COLS = 4 * COLS;
    const int n0 = col_tile * OUT_COLS;
    // (32-bit results: a thread's four columns are the same in all of its rows)
    constexpr bool IS_32 = gm_is_32(EPI);
    constexpr int LANES = OUT_COLS / (IS_32 ? 4 : 8), STEP = 256 / LANES, AHEAD = 8;          // lanes of a row, rows a pass
    const int col = n0 + tid % LANES * 4;
    gm_f32x4 old[AHEAD];
    auto ask_old = [&](int r0) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int row = m0 + r0 + i * STEP + tid / LANES;
            old[i] = *reinterpret_cast<const gm_f32x4*>(static_cast<const float*>(y_) + static_cast<size_t>(min(row, M - 1)) * N + min(col, N - 4));
        }
    };
    if constexpr (EPI == GM_ADD) ask_old(0);
    if constexpr (EPI == GM_HEADS) {
        if (tid < ROWS) {
            places[2 * tid] = row_pos;
            places[2 * tid + 1] = row_page >= 0 ? row_page * heads.block_size + row_pos % heads.block_size : -1;
        }
    }
    __syncthreads();

    // The tile leaves through LDS in whole rows.  acc[c][t][4 j + i]: row 32 t + r32, row of A 8 j + 4 h + i
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        char* at_row = gm_lds + (32 * t + r32) * PITCH + wave * COLS * (IS_32 ? 4 : 2);
        const float scale = TAKES ? scales[32 * t + r32] : 1.f;
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int j = 0; j < (EPI == GM_SWIGLU ? 2 : 4); ++j) {
                gm_f32x4 v;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = acc[c][t][4 * j + i] * scale;
                    if constexpr (EPI == GM_SWIGLU) v[i] = gm_silu(v[i]) * (acc[c][t][4 * (j + 2) + i] * scale);
                }
                const int at = (EPI == GM_SWIGLU ? 16 : 32) * c + 8 * j + 4 * h;
                if constexpr (IS_32) {
                    *reinterpret_cast<gm_f32x4*>(at_row + at * 4) = v;
                } else {
                    const gm_u32x2 packed = {gm_pack2(v[0], v[1]), gm_pack2(v[2], v[3])};
                    *reinterpret_cast<gm_u32x2*>(at_row + at * 2) = packed;
                }
            }
    }
    __syncthreads();
    if constexpr (EPI == GM_HEADS) {
        // 16 lanes a head's row; the angles of four rows are asked for together.  Bound by the vector instructions, some 140 a row and 9 cycles apart where a wave
        // is alone on its SIMD (128 rows by 256 columns 8 us, 128 by 128 two a compute unit 5): the shapes are chosen with that.  us, the product and the
        // stand-alone kernel / this one, 16 heads over 8 of a width of 1,024: 300 rows 12.3 / 10.3, 1,024 21.8 / 17.0, 2,048 30.3 / 27.2.
        static_assert(EPI != GM_HEADS || (ROWS * LANES) % (4 * 256) == 0, "whole groups of four rows a thread");
        const int chunk = tid % 16;
        const bool gain = heads.q_gain != nullptr, turn = heads.cos_table != nullptr;
        float gq[8], gk[8];
        if (gain) {
            hr_load_gain(heads.q_gain, heads.gain_dtype, chunk, gq);
            hr_load_gain(heads.k_gain, heads.gain_dtype, chunk, gk);
        }
        for (int i0 = tid; i0 < ROWS * LANES; i0 += 4 * 256) {
            float cs[4][8], sn[4][8];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int r = (i0 + 256 * u) / LANES;
                if (turn) {
                    const size_t at = static_cast<size_t>(max(places[2 * r], 0)) * 64 + (chunk & 7) * 8;
                    hr_load8(heads.cos_table + at, cs[u]);
                    hr_load8(heads.sin_table + at, sn[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int r = (i0 + 256 * u) / LANES, head = n0 / 128 + (i0 + 256 * u) % LANES / 16;
                const bool is_q = head < heads.nq, is_k = !is_q && head < heads.nq + heads.nkv;
                hr_u32x4 v = *reinterpret_cast<const hr_u32x4*>(gm_lds + r * PITCH + (i0 + 256 * u) % LANES * 16);
                if (is_q || is_k) v = hr_prepare(v, gain, is_q ? gq : gk, heads.eps, turn, cs[u], sn[u], chunk < 8);
                const int place = places[2 * r + 1];
                bf16_t* to = static_cast<bf16_t*>(y_) + static_cast<size_t>(m0 + r) * N + head * 128;
                bool there = m0 + r < M && places[2 * r] >= 0 && head * 128 < N;
                if (!is_q) {
                    there = there && place >= 0;               // (never written through a hole in the table)
                    to = (is_k ? heads.k_pool : heads.v_pool) + (static_cast<size_t>(max(place, 0)) * heads.nkv + head - heads.nq - (is_k ? 0 : heads.nkv)) * 128;
                }
                if (there) *reinterpret_cast<hr_u32x4*>(to + chunk * 8) = v;
            }
        }
    } else if constexpr (!IS_32) {
        bf16_t* y = static_cast<bf16_t*>(y_);
        for (int i = tid; i < ROWS * LANES; i += 256) {
            const int r = i / LANES, piece = i % LANES;
            if (m0 + r < M && n0 + piece * 8 < N)
                *reinterpret_cast<gm_u32x4*>(y + static_cast<size_t>(m0 + r) * y_pitch + n0 + piece * 8) =
                    *reinterpret_cast<const gm_u32x4*>(gm_lds + r * PITCH + piece * 16);
        }
    } else {
        static_assert(!IS_32 || (256 % LANES == 0 && LANES % 16 == 0 && ROWS % (STEP * AHEAD) == 0), "whole passes");
        const bool hands = EPI == GM_ADD && norms.gain != nullptr;
        gm_f32x4 gain = {0.f, 0.f, 0.f, 0.f};
        if (hands) gain = *reinterpret_cast<const gm_f32x4*>(norms.gain + min(col, N - 4));
        for (int r0 = 0; r0 < ROWS; r0 += STEP * AHEAD) {
            if (EPI == GM_ADD && r0 > 0) ask_old(r0);
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) {
                const int r = r0 + i * STEP + tid / LANES, row = m0 + r;
                const bool there = row < M && col < N;
                gm_f32x4 v = *reinterpret_cast<const gm_f32x4*>(gm_lds + r * PITCH + tid % LANES * 16);
                if constexpr (EPI == GM_ADD) v += old[i];
                const size_t to = static_cast<size_t>(row) * y_pitch + col;
                if (there) *reinterpret_cast<gm_f32x4*>(static_cast<float*>(y_) + to) = v;
                if (hands) {
                    const float square = hr_sum16(there ? (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]) : 0.f);
                    if (there) {
                        const gm_u32x2 packed = {gm_pack2(v[0] * gain[0], v[1] * gain[1]), gm_pack2(v[2] * gain[2], v[3] * gain[3])};
                        *reinterpret_cast<gm_u32x2*>(norms.rows + to) = packed;
                        if (tid % 16 == 0) norms.sums[static_cast<size_t>(row) * (N / GM_STRIPE) + col / GM_STRIPE] = square;
                    }
                }
            }
        }
    }
}

struct GmProduct {
    const void *x, *weights;
    bool strips;
    void* y;
    int M, N, K;
    GmNorms norms;
    GmHeads heads;
};

template <int CT, int RT, int PER_SIMD, int EPI, bool TAKES, bool STRIPS>
static int gm_launch_one(const GmProduct& g, hipStream_t stream) {
    constexpr int lds = gm_lds_bytes(CT, RT, EPI, STRIPS);
    static_assert(lds <= 160 * 1024, "a workgroup's LDS");
    const int row_tiles = pl_ceil_div(g.M, 32 * RT), col_tiles = pl_ceil_div(g.N, gm_out_cols(CT, EPI));
    if constexpr (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_many_kernel<CT, RT, PER_SIMD, EPI, TAKES, STRIPS>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        PL_REQUIRE(e == hipSuccess, "product of many rows: %d bytes of LDS refused: %s", lds, hipGetErrorString(e));
    }
    gemm_many_kernel<CT, RT, PER_SIMD, EPI, TAKES, STRIPS><<<row_tiles * col_tiles, 256, lds, stream>>>(
        static_cast<const bf16_t*>(g.x), static_cast<const bf16_t*>(g.weights), g.y, g.M, g.N, g.K, row_tiles, col_tiles, g.norms, GmGroups{}, g.heads);
    PL_CHECK_LAUNCH("gemm_many");
    return 0;
}

template <int CT, int RT, int PER_SIMD, int EPI>
static int gm_launch(const GmProduct& g, hipStream_t stream) {
    if constexpr (!gm_is_32(EPI)) {
        if (g.norms.taken != nullptr)
            return g.strips ? gm_launch_one<CT, RT, PER_SIMD, EPI, true, true>(g, stream) : gm_launch_one<CT, RT, PER_SIMD, EPI, true, false>(g, stream);
    }
    return g.strips ? gm_launch_one<CT, RT, PER_SIMD, EPI, false, true>(g, stream) : gm_launch_one<CT, RT, PER_SIMD, EPI, false, false>(g, stream);
}

// The tiles there are, and what one costs a compute unit: us for 64 k, and for the tile itself by what is done with it, as timed one tile a
// compute unit (K of 1,024 and of 3,072).  A launch is taken to last as long as the compute unit with most tiles: that is the order of the
// shapes in all of 40 timed products (65 to 4,096 rows of 1,024, 4,096 and 5,120) but for differences of a few per cent.  (32-bit
// results of the largest tile would not fit into LDS.)
//
// The order is the same for weights in rows, which take more LDS: {2, 3} then has a compute unit to itself, as its 32-bit results have out of strips, where it and the smaller
// ones are two a unit otherwise.  Over 68 products (65 to 3,072 rows of 1,024 to 4,096, weights from memory) the shape taken lost 0.7% to the fastest on average and 4% at most out
// of strips, 1.0% and 4% in rows; 32-bit results of very many columns 7% and, past 64 rows in rows, 14% at most (65,536 columns of 2,048, 65 rows out of strips: 60 us, 56 with {1, 4}).
// More registers for a {2, 3} that is alone changed nothing (29 products within 2.5% either way).
struct GmShape {
    int ct, rt;
    float stage, tile[5];      // (by epilogue)
};
static const GmShape GM_SHAPES[] = {{1, 2, 0.25f, {1.5f, 3.0f, 4.0f, 2.5f, 4.0f}},
                                    {1, 4, 0.37f, {2.2f, 2.9f, 8.0f, 4.0f, 7.0f}},
                                    {2, 3, 0.425f, {3.0f, 5.2f, 10.f, 5.0f, 10.f}},
                                    {2, 4, 0.54f, {4.0f, 5.8f, 14.f, 6.0f, 18.f}},
                                    {3, 4, 0.755f, {6.0f, 9.0f, 0.f, 0.f, 22.f}}};

static int gm_pick(int M, int N, int K, int epilogue) {
    int best = 0;
    float least = 0.f;
    for (int i = 0; i < (gm_is_32(epilogue) ? 4 : 5); ++i) {
        const GmShape& s = GM_SHAPES[i];
        const long tiles = static_cast<long>(pl_ceil_div(M, 32 * s.rt)) * pl_ceil_div(N, gm_out_cols(s.ct, epilogue));
        const float cost = static_cast<float>((tiles + pl_compute_units() - 1) / pl_compute_units()) * (s.tile[epilogue] + K / GM_BK * s.stage);
        if (i == 0 || cost < least) best = i, least = cost;
    }
    return best;
}

template <int EPI>
static int gm_shaped(const GmProduct& g, hipStream_t stream) {
    switch (gm_pick(g.M, g.N, g.K, EPI)) {
        case 0: return gm_launch<1, 2, 2, EPI>(g, stream);
        case 1: return gm_launch<1, 4, 2, EPI>(g, stream);
        case 2: return gm_launch<2, 3, 2, EPI>(g, stream);
        case 3: return gm_launch<2, 4, 1, EPI>(g, stream);
        default:
            if constexpr (!gm_is_32(EPI)) return gm_launch<3, 4, 1, EPI>(g, stream);
    }
    return -1;
}

// Whether a shape is served: N (of gate alone for epilogue 1) a multiple of 16, K of 64, and offsets of 32 bits into x and into the weights.
extern "C" int pl_gemm_many_applies(int M, int N, int K, int epilogue) {
    return M > 0 && N > 0 && K > 0 && N % 16 == 0 && K % GM_BK == 0 && static_cast<long long>(M) * K < (1ll << 31) &&
           (epilogue == GM_SWIGLU ? 2ll : 1ll) * N * K < (1ll << 31) && static_cast<long long>(pl_ceil_div(M, 64)) * pl_ceil_div(N, 64) < (1ll << 30);
}

// x: bfloat16 [M, K].  weights: bfloat16 [N, K], or [2 N, K], gate rows first, for epilogue 1; in strips or as they are.
// epilogue 0: y (bfloat16 [M, N]) = result.  1: y = silu(gate) * up.  2: y (32-bit [M, N]) += result.  3: y (32-bit) = result.  All aligned to 16 bytes.
// taken [M, taken_count] (epilogues 0 and 1; a multiple of four, up to 64): the sums of a norm handed forward, whose rows x are.  gain [N], rows [M, N],
// sums [M, N / 64] (epilogue 2, N a multiple of 64): the norm behind the sum, handed forward.
extern "C" int pl_gemm_many(const void* x, const void* weights, int in_strips, void* y, int M, int N, int K, int epilogue, const float* taken, int taken_count,
                              float eps, const float* gain, void* rows, float* sums, hipStream_t stream) {
    PL_REQUIRE(epilogue >= GM_STORE && epilogue <= GM_STORE32 && pl_gemm_many_applies(M, N, K, epilogue),
               "product of many rows: %d rows, %d columns, inner width %d, epilogue %d", M, N, K, epilogue);
    PL_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weights) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(gain) |
                reinterpret_cast<uintptr_t>(rows)) % 16 == 0, "product of many rows: rows that are not aligned to 16 bytes");
    PL_REQUIRE(taken == nullptr || (!gm_is_32(epilogue) && taken_count > 0 && taken_count <= GM_TAKEN_MOST && taken_count % 4 == 0 && reinterpret_cast<uintptr_t>(taken) % 16 == 0), "product of many rows: %d sums of a norm, epilogue %d",
               taken_count, epilogue);
    PL_REQUIRE((gain == nullptr) == (rows == nullptr) && (gain == nullptr) == (sums == nullptr) && (gain == nullptr || (epilogue == GM_ADD && N % GM_STRIPE == 0)),
               "product of many rows: a norm handed forward by epilogue %d", epilogue);
    const GmProduct g{x, weights, in_strips != 0, y, M, N, K, GmNorms{taken, taken_count, eps, gain, static_cast<bf16_t*>(rows), sums}, GmHeads{}};
    if (epilogue == GM_STORE) return gm_shaped<GM_STORE>(g, stream);
    if (epilogue == GM_SWIGLU) return gm_shaped<GM_SWIGLU>(g, stream);
    if (epilogue == GM_ADD) return gm_shaped<GM_ADD>(g, stream);
    return gm_shaped<GM_STORE32>(g, stream);
}

// The projection [q | k | v] of heads of 128 and what stands between it and attention (see GmHeads).  x, weights: as pl_gemm_many, N = (nq + 2 nkv) 128.  y: bfloat16
// [M, N], of which the queries are written; rows at negative positions are not.  taken: as pl_gemm_many.
extern "C" int pl_gemm_many_heads(const void* x, const void* weights, int in_strips, void* y, int M, int K, const float* taken, int taken_count,
                                  float taken_eps, const void* q_gain, const void* k_gain, int gain_dtype, float eps, const float* cos_table,
                                  const float* sin_table, const int* positions, const int* seq_of, const int* block_table, int max_blocks, int block_size,
                                  void* k_pool, void* v_pool, int nq, int nkv, hipStream_t stream) {
    const int N = (nq + 2 * nkv) * 128;
    PL_REQUIRE(nq > 0 && nkv > 0 && nq <= (1 << 16) && nkv <= (1 << 16) && pl_gemm_many_applies(M, N, K, GM_STORE), "heads of many rows: %d rows, %d and %d heads, inner width %d",
               M, nq, nkv, K);
    PL_REQUIRE(block_size > 0 && max_blocks > 0, "heads of many rows: block size %d, %d blocks a row", block_size, max_blocks);
    PL_REQUIRE((q_gain == nullptr) == (k_gain == nullptr) && (cos_table == nullptr) == (sin_table == nullptr), "heads of many rows: one of the two gains or tables is missing");
    PL_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weights) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(k_pool) |
                reinterpret_cast<uintptr_t>(v_pool) | reinterpret_cast<uintptr_t>(q_gain) | reinterpret_cast<uintptr_t>(k_gain) |
                reinterpret_cast<uintptr_t>(cos_table) | reinterpret_cast<uintptr_t>(sin_table)) % 16 == 0, "heads of many rows: rows that are not aligned to 16 bytes");
    PL_REQUIRE(taken == nullptr || (taken_count > 0 && taken_count <= GM_TAKEN_MOST && taken_count % 4 == 0 && reinterpret_cast<uintptr_t>(taken) % 16 == 0),
               "heads of many rows: %d sums of a norm", taken_count);
    const GmProduct g{x, weights, in_strips != 0, y, M, N, K, GmNorms{taken, taken_count, taken_eps, nullptr, nullptr, nullptr},
                      GmHeads{q_gain, k_gain, gain_dtype, eps, cos_table, sin_table, positions, seq_of, block_table, max_blocks, block_size,
                              static_cast<bf16_t*>(k_pool), static_cast<bf16_t*>(v_pool), nq, nkv}};
    return gm_shaped<GM_HEADS>(g, stream);
}

template <int CT, int PER_SIMD, int EPI>
static int gm_launch_grouped(const GmProduct& g, const GmGroups& groups, int row_tiles, int columns, hipStream_t stream) {
    constexpr int lds = gm_lds_bytes(CT, 4, EPI, false);
    static_assert(lds <= 160 * 1024, "a workgroup's LDS");
    const int col_tiles = pl_ceil_div(columns, gm_out_cols(CT, EPI));
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_many_kernel<CT, 4, PER_SIMD, EPI, false, false, true>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    PL_REQUIRE(e == hipSuccess, "grouped product of many rows: %d bytes of LDS refused: %s", lds, hipGetErrorString(e));
    gemm_many_kernel<CT, 4, PER_SIMD, EPI, false, false, true><<<row_tiles * col_tiles, 256, lds, stream>>>(
        static_cast<const bf16_t*>(g.x), static_cast<const bf16_t*>(g.weights), g.y, g.M, g.N, g.K, row_tiles, col_tiles, g.norms, groups, GmHeads{});
    PL_CHECK_LAUNCH("gemm_many_grouped");
    return 0;
}

// Whether the grouped form takes these sizes (those of the last group too, where it has its own).
extern "C" int pl_gemm_many_grouped_applies(int row_tiles, int x_rows, int N, int K, int x_pitch) {
    return row_tiles > 0 && row_tiles <= (1 << 22) && x_rows > 0 && N > 0 && K > 0 && N % 16 == 0 && K % GM_BK == 0 && 2ll * N * K < (1ll << 31) &&
           static_cast<long long>(x_rows) * x_pitch < (1ll << 31) && static_cast<long long>(row_tiles) * pl_ceil_div(N, 64) < (1ll << 30);
}

// The product over rows dealt to groups (see GmGroups).  x: bfloat16 [x_rows, x_pitch], read through `gather` ([row_tiles * 128]) or, with gather null, in
// place (x_rows >= row_tiles * 128).  w: bfloat16, group g's matrix at w + g * w_stride: [N, K], or [2 N, K] with the gate rows first for epilogue 1.
// y: [row_tiles * 128, y_pitch], bfloat16 for epilogue 1 (silu(gate) * up), 32-bit for epilogue 3.  last >= 0: that group's matrix is w_last, of N_last and
// K_last in the places of N and K, under the same rules.  likely_tiles: how many of the tiles will likely be used (the shape goes by it).
// us, gemm_tiled / this one, 28 tiles of 36 used: 1,536 gated columns of 1,024 50 / 32, 1,024 of 1,536 in 32 bits 26.6 / 22.6.
extern "C" int pl_gemm_many_grouped(const void* x, const void* w, void* y, const int* tile_group, const int* gather, long long w_stride, int row_tiles,
                                    int likely_tiles, int x_rows, int N, int K, int epilogue, int x_pitch, int y_pitch, int last, const void* w_last, int N_last,
                                    int K_last, hipStream_t stream) {
    PL_REQUIRE((epilogue == GM_SWIGLU || epilogue == GM_STORE32) && pl_gemm_many_grouped_applies(row_tiles, x_rows, N, K, x_pitch) &&
                   (last < 0 || (w_last != nullptr && pl_gemm_many_grouped_applies(row_tiles, x_rows, N_last, K_last, x_pitch))),
               "grouped product of many rows: %d tiles, %d columns, inner width %d, epilogue %d", row_tiles, N, K, epilogue);
    PL_REQUIRE(x_pitch >= K && y_pitch >= N && x_pitch % 8 == 0 && y_pitch % 8 == 0 && (last < 0 || (x_pitch >= K_last && y_pitch >= N_last)),
               "grouped product of many rows: rows of %d and %d for an inner width of %d and %d columns", x_pitch, y_pitch, K, N);
    PL_REQUIRE(tile_group != nullptr && (gather != nullptr || x_rows >= row_tiles * 128), "grouped product of many rows: %d rows for %d tiles", x_rows, row_tiles);
    PL_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(w_last)) % 16 == 0 &&
                   w_stride % 8 == 0, "grouped product of many rows: rows that are not aligned to 16 bytes");
    const GmProduct g{x, w, false, y, row_tiles * 128, N, K, GmNorms{}, GmHeads{}};
    const GmGroups groups{tile_group, gather, w_stride, x_pitch, y_pitch, last, N_last, K_last, static_cast<const bf16_t*>(w_last)};
    const int columns = last >= 0 && N_last > N ? N_last : N;
    int best = 0;
    float least = 0.f;
    for (int i = 1; i < (epilogue == GM_STORE32 ? 4 : 5); ++i) {
        const GmShape& s = GM_SHAPES[i];
        if (s.rt != 4) continue;
        const long tiles = static_cast<long>(likely_tiles) * pl_ceil_div(columns, gm_out_cols(s.ct, epilogue));
        const float cost = static_cast<float>((tiles + pl_compute_units() - 1) / pl_compute_units()) * (s.tile[epilogue] + K / GM_BK * s.stage);
        if (best == 0 || cost < least) best = i, least = cost;
    }
    if (epilogue == GM_SWIGLU) {
        if (best == 1) return gm_launch_grouped<1, 2, GM_SWIGLU>(g, groups, row_tiles, columns, stream);
        if (best == 3) return gm_launch_grouped<2, 1, GM_SWIGLU>(g, groups, row_tiles, columns, stream);
        return gm_launch_grouped<3, 1, GM_SWIGLU>(g, groups, row_tiles, columns, stream);
    }
    if (best == 1) return gm_launch_grouped<1, 2, GM_STORE32>(g, groups, row_tiles, columns, stream);
    return gm_launch_grouped<2, 1, GM_STORE32>(g, groups, row_tiles, columns, stream);
}
