// y[n, N] = x[n, K] . w[N, K]^T of 32-bit operands on the matrix cores' 32-bit instruction (v_mfma_f32_16x16x4_f32): the
// product of the true 32-bit path.  Operands, products and sums are 32-bit; nothing is rounded to fewer bits.
//
// A row's result does not depend on what else is in the batch, bit for bit, whichever of the kernels below runs: K is cut
// into at most 16 parts by K alone, a part is one chain of matrix instructions from its first k to its last, and the parts
// are added in ascending order.  (Inside 16 consecutive k an instruction takes k, k + 4, k + 8, k + 12: the four
// consecutive values a lane holds are its operands of four instructions.)
#include "common.hpp"

#define PL_F32_PARTS 16

typedef float f32x4 __attribute__((ext_vector_type(4)));

// The length of a part: whole double steps of the tiled kernel, whole rounds of the kernel for few rows.
static inline int f32_part_len(int K) { return pl_ceil_div(pl_ceil_div(K, PL_F32_PARTS), 64) * 64; }

// The values k .. k + 3 of a row of K; past its end whatever stands at the end (f32_end clears it).  VEC: rows and K are
// multiples of four values and the base is aligned.
template <bool VEC>
__device__ __forceinline__ f32x4 f32_load4(const float* row, int k, int K) {
    if (VEC) return *reinterpret_cast<const f32x4*>(row + min(k, K - 4));
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = row[min(k + i, K - 1)];
    return v;
}

__device__ __forceinline__ f32x4 f32_end(f32x4 v, int k, int K) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = k + i < K ? v[i] : 0.f;
    return v;
}

// 16 k of TM tiles of 16 columns of w against TN tiles of 16 rows of x.
template <int TM, int TN>
__device__ __forceinline__ void f32_multiply(const f32x4 (&a)[TM], const f32x4 (&b)[TN], f32x4 (&acc)[TM][TN]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][q], b[j][q], acc[i][j], 0, 0, 0);
}

__device__ __forceinline__ void f32_store4(float* to, f32x4 v, int col, int N, bool whole) {
    if (whole) {
        if (col < N) *reinterpret_cast<f32x4*>(to) = v;
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (col + q < N) to[q] = v[q];
    }
}

// ---- few rows ----------------------------------------------------------------------------------------------------------------
// Bound by the weights' bytes.  A workgroup of sixteen waves owns 16 columns and TN x 16 rows of x; a wave takes one part
// of K straight from memory in the instruction's layout, 64 k a round, and the parts meet in LDS (a row tile a blockIdx.y).
// VEC: rows are made of aligned groups of four values.
//
// With at most 8 rows of x half of the instruction's 16 would be copies.  SHARE 2 gives that half to another part of K: a wave takes
// two parts of 8 columns, rows 0 .. 7 of its operands from one part and 8 .. 15 from the next, and of the result keeps the two
// blocks of 8 x 8 whose operands belong together (each element the same chain as before); SHARE 4 four parts of 4 columns
// for at most 4 rows.  A product has two or four times as many workgroups of fewer waves, and reads no row of x twice.
//
// GATED: w is [gate | up], N rows each; half of a workgroup's columns are columns of gate, the other half the same of up, and
// y[n, N] = act(x . gate^T) * (x . up^T), each sum and then the pair as the product and the activation kernel would make them.
template <int TN, bool VEC, int SHARE, bool GATED>
__global__ void __launch_bounds__(PL_F32_PARTS / SHARE * PL_WAVE)
gemm_f32_few_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ y, int n, int N, int K,
                    int ldx, int ldy, long sx, long sw, long sy, int part_len, int act) {
    static_assert(SHARE == 1 || TN == 1, "parts share the instruction of one tile of rows");
    static_assert(!GATED || SHARE < 4, "four columns of gate and of up make a store");
    constexpr int ROUND = TN > 2 ? 2 : 4;                               // steps of 16 k asked for together
    constexpr int COLS = 16 / SHARE, ROWS = TN * 16 / SHARE, OUT = GATED ? COLS / 2 : COLS;    // (OUT: columns of y)
    __shared__ __attribute__((aligned(16))) float parts[PL_F32_PARTS][ROWS][COLS];       // [part][row of x][column of w]
    x += blockIdx.z * sx;
    w += blockIdx.z * sw;
    y += blockIdx.z * sy;
    const int lane = threadIdx.x % PL_WAVE, wave = threadIdx.x / PL_WAVE;
    const int r = lane % 16, c = lane / 16;
    const int n0 = blockIdx.x * OUT, m0 = blockIdx.y * ROWS;
    const float* wr = w + (static_cast<size_t>(min(n0 + r % OUT, N - 1)) + (GATED && r % COLS >= OUT ? N : 0)) * K;
    const float* xr[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) xr[j] = x + static_cast<size_t>(min(m0 + (j * 16 + r) % ROWS, n - 1)) * ldx;

    // (the wave's first part; a lane's own begins `mine` behind it and ends at `end`)
    const int first = wave * SHARE * part_len, last = min(K, first + part_len);
    const int mine = r / COLS * part_len, end = SHARE == 1 ? K : min(K, first + mine + part_len);
    if (first < last) {
        f32x4 acc[1][TN];
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[0][j] = zero;
        f32x4 a[ROUND][1], b[ROUND][TN];
        auto ask = [&](int u, int k) {
            a[u][0] = f32_load4<VEC>(wr, k + mine + c * 4, K);
#pragma unroll
            for (int j = 0; j < TN; ++j) b[u][j] = f32_load4<VEC>(xr[j], k + mine + c * 4, K);
        };
        auto clear = [&](int u, int k) {
            a[u][0] = f32_end(a[u][0], k + mine + c * 4, end);
#pragma unroll
            for (int j = 0; j < TN; ++j) b[u][j] = f32_end(b[u][j], k + mine + c * 4, end);
        };
#pragma unroll
        for (int u = 0; u < ROUND; ++u) ask(u, first + u * 16);
        int k = first;
        for (; k + ROUND * 16 < last; k += ROUND * 16) {
            // (two steps' registers, a row's 128 bytes, are filled again as soon as they are multiplied; every load is
            // unconditional, since a load in a branch would make the compiler wait for all that are on their way, and nothing past
            // the part is asked for)
#pragma unroll
            for (int u = 0; u < ROUND; u += 2) {
#pragma unroll
                for (int e = u; e < u + 2; ++e) {
                    if (SHARE > 1) clear(e, k + e * 16);
                    f32_multiply<1, TN>(a[e], b[e], acc);
                }
#pragma unroll
                for (int e = u; e < u + 2; ++e) ask(e, k + (ROUND + e) * 16);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int u = 0; u < ROUND; ++u) {
            if (k + u * 16 < last) {
                clear(u, k + u * 16);
                f32_multiply<1, TN>(a[u], b[u], acc);
            }
        }
        // (a lane holds four columns of one row of x; the other blocks mix two parts)
        if (c * 4 / COLS == r / COLS) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
                *reinterpret_cast<f32x4*>(&parts[wave * SHARE + r / COLS][(j * 16 + r) % ROWS][c * 4 % COLS]) = acc[0][j];
        }
    }
    __syncthreads();
    const int used = (K + part_len - 1) / part_len;
    const int row = threadIdx.x * 4 / OUT, at = threadIdx.x * 4 % OUT, col = n0 + at;         // four columns of one row
    if (row < ROWS && m0 + row < n) {
        f32x4 sum = {0.f, 0.f, 0.f, 0.f}, up = {0.f, 0.f, 0.f, 0.f};
        for (int p = 0; p < used; ++p) {
            sum += *reinterpret_cast<const f32x4*>(&parts[p][row][at]);
            if (GATED) up += *reinterpret_cast<const f32x4*>(&parts[p][row][OUT % COLS + at]);
        }
        if (GATED)
#pragma unroll
            for (int q = 0; q < 4; ++q) sum[q] = pl_activate<true>(sum[q], act) * up[q];
        const bool whole = N % 4 == 0 && ldy % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
        f32_store4(y + static_cast<size_t>(m0 + row) * ldy + col, sum, col, N, whole);
    }
}

// ---- many rows ---------------------------------------------------------------------------------------------------------------
// Bound by the matrix cores: a workgroup of four waves, two by two, owns TILE rows of x and TILE columns; 32 k a stage through
// four stages of LDS, filled three steps ahead by loads that write LDS themselves (global_load_lds_dwordx4: a wave's load is
// eight whole 128-byte pieces of rows).  Lane l of a load brings piece (l % 8) ^ (row % 8) of its row into slot l % 8, so that
// the lanes that read one piece of eight rows find it in different banks.  What a step costs beside its products (1,024 cycles
// at tiles of 64) is its barrier and what the addresses and the loads take to issue: with one workgroup a compute unit 1,024 x
// 2,048 takes 41 us where the products alone take 27; 2,048 rows of 4,096 x 1,024 run at 113 TFLOP/s, and 104 to 125 in the
// library's product.  Tiles of 128 run as fast as tiles of 64 there and leave more of the chip idle elsewhere, and operands
// straight from L2 into registers (no LDS) half as fast: a compute unit's L1 then gives out each line twice.
#define F32_BK 32
#define F32_STAGES 4

// The workgroup's tile, of row_tiles x col_tiles.  Workgroups go to the eight XCDs in turn: an XCD gets every eighth column of tiles,
// the rows of x first, so that a row of w is read into one L2 only; the tiles of the columns left over are dealt out in
// runs, so that no XCD has more than one of them more than another.  (With those as whole columns too 16 heads of 1,500 rows by 128 by 192,
// two columns of tiles, ran on two of the eight XCDs: 55 us, 19 so; 64 by 128 24 and 9.9.  With runs of all tiles 400 rows of 8,192 x
// 4,096 took 257 us, 241 so.)
__device__ __forceinline__ bool f32_tile(int row_tiles, int col_tiles, int& row_tile, int& col_tile) {
    const int whole = col_tiles / 8 * 8, in_whole = whole * row_tiles;
    int at = blockIdx.x;
    if (at < in_whole) {
        col_tile = at % 8 + at / 8 / row_tiles * 8;
        row_tile = at / 8 % row_tiles;
        return true;
    }
    at -= in_whole;             // (a multiple of eight: the XCDs' turns begin anew)
    at = at % 8 * ((gridDim.x - in_whole) / 8) + at / 8;
    row_tile = at % row_tiles;
    col_tile = whole + at / row_tiles;
    return col_tile < col_tiles;
}

// 16 bytes a lane from `offset` bytes behind `base` (the same for the wave) to LDS, lane after lane from byte `to` on.  Assembly,
// so that the compiler does not count the load and make every later read of LDS wait for all of them.
__device__ __forceinline__ void f32_load_to_lds(const void* base, uint32_t offset, uint32_t to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(offset), "s"(base) : "memory", "m0");
}

// K a multiple of 64 (two steps).
template <int TILE>
__global__ void __launch_bounds__(256)
gemm_f32_tiled_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ y, int n, int N, int K,
                      int ldx, int ldy, long sx, long sw, long sy, int part_len, int row_tiles, int col_tiles) {
    constexpr int TM = TILE / 32, TN = TM;                      // tiles of 16 a wave: columns, rows
    constexpr int STAGE = 2 * TILE * F32_BK, LOADS = TILE / 16;
    extern __shared__ __attribute__((aligned(16))) float f32_lds[];         // [stage][rows of x, then columns of w][32]
    int row_tile, col_tile;
    if (!f32_tile(row_tiles, col_tiles, row_tile, col_tile)) return;        // (the whole workgroup)
    const int m0 = row_tile * TILE, n0 = col_tile * TILE;
    const int lane = threadIdx.x % PL_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PL_WAVE);
    const int r = lane % 16, c = lane / 16;
    y += blockIdx.z * sy;
    const float* x0 = x + blockIdx.z * sx + static_cast<size_t>(m0) * ldx;
    const float* w0 = w + blockIdx.z * sw + static_cast<size_t>(n0) * K;

    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const float*)f32_lds));
    uint32_t offset[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (wave + 4 * i) * 8 + lane / 8;          // of the stage: rows of x for i < TN, columns of w behind them
        const int piece = (lane % 8 ^ row % 8) * 4;
        offset[i] = 4u * (i < TN ? static_cast<uint32_t>(min(row, n - 1 - m0)) * ldx + piece
                                 : static_cast<uint32_t>(min(row - TILE, N - 1 - n0)) * K + piece);
    }
    const int steps = K / F32_BK;
    auto ask = [&](int step) {              // (past the end: the last step again, so that the counts stay)
        const int k = min(step, steps - 1) * F32_BK;
        const uint32_t to = lds0 + (static_cast<uint32_t>(step) % F32_STAGES * STAGE + wave * 8 * F32_BK) * 4u;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) f32_load_to_lds((i < TN ? x0 : w0) + k, offset[i], to + i * 32 * F32_BK * 4u);
    };
    int a_at[2], b_at[2];                   // this lane's operands in a stage, for either half of a step
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int slot = ((c + 4 * h) ^ r % 8) * 4;
        a_at[h] = (TILE + wave % 2 * TM * 16 + r) * F32_BK + slot;
        b_at[h] = (wave / 2 * TN * 16 + r) * F32_BK + slot;
    }
    // The operands of a step are read out of LDS one step early, while the step before is multiplied: two sets of registers
    // that take turns.
    f32x4 a[2][2][TM], b[2][2][TN];         // [set][half of the step]
    auto read = [&](int set, int step) {
        const float* at = f32_lds + static_cast<uint32_t>(step) % F32_STAGES * STAGE;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < TM; ++i) a[set][h][i] = *reinterpret_cast<const f32x4*>(at + a_at[h] + i * 16 * F32_BK);
#pragma unroll
            for (int j = 0; j < TN; ++j) b[set][h][j] = *reinterpret_cast<const f32x4*>(at + b_at[h] + j * 16 * F32_BK);
        }
    };
    f32x4 acc[TM][TN], total[TM][TN];
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) total[i][j] = zero;
    // One step.  The loads of the step after this one have landed in this wave (one later step's may be on their way); after
    // the barrier every wave's have, and every wave has multiplied the step before, whose stage is filled next.
    auto one_step = [&](int set, int step) {
        __builtin_amdgcn_s_waitcnt(0x0F70 | LOADS);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        ask(step + 3);
        read(set ^ 1, step + 1);
        __builtin_amdgcn_sched_barrier(0);
        f32_multiply<TM, TN>(a[set][0], b[set][0], acc);
        f32_multiply<TM, TN>(a[set][1], b[set][1], acc);
        __builtin_amdgcn_sched_barrier(0);
    };
    ask(0);
    ask(1);
    ask(2);
    __builtin_amdgcn_s_waitcnt(0x0F70 | 2 * LOADS);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0);
    const int part_steps = part_len / F32_BK;
    for (int s0 = 0; s0 < steps; s0 += part_steps) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = zero;
        const int stop = min(steps, s0 + part_steps);           // (both are even)
        for (int s = s0; s < stop; s += 2) {
            one_step(0, s);
            one_step(1, s + 1);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) total[i][j] += acc[i][j];
    }
    // (the loads asked for past the end still write LDS: they have to have landed before the workgroup ends)
    __builtin_amdgcn_s_waitcnt(0x0F70);
    const bool whole = N % 4 == 0 && ldy % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int row = m0 + (wave / 2 * TN + j) * 16 + r;
        if (row >= n) continue;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int col = n0 + (wave % 2 * TM + i) * 16 + c * 4;
            f32_store4(y + static_cast<size_t>(row) * ldy + col, total[i][j], col, N, whole);
        }
    }
}

// ---- many rows, any K ----------------------------------------------------------------------------------------------------------
// The same where K is no multiple of 64 or rows are not aligned groups of four values: a step's operands come through registers,
// asked for two steps ahead, into two stages of LDS that take turns.  What lies past K counts as zeros, which leave a chain as it is.
// Bound by the matrix cores and the barrier a step, and by the loads' issue where they are of one value (VEC false): 1,500 rows of 4,096 x
// 1,026 81 TFLOP/s, of 4,096 x 4,128 110; the kernel for few rows, which took them before, 21 and 57.
template <int TILE, bool VEC>
__global__ void __launch_bounds__(256)
gemm_f32_ragged_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ y, int n, int N, int K,
                       int ldx, int ldy, long sx, long sw, long sy, int part_len, int row_tiles, int col_tiles) {
    constexpr int TM = TILE / 32, TN = TM;                      // tiles of 16 a wave: columns, rows
    constexpr int STAGE = 2 * TILE * F32_BK, WIDE = VEC ? 4 : 1, LANES = F32_BK / WIDE, LOADS = STAGE / 256 / WIDE;
    __shared__ __attribute__((aligned(16))) float lds[2 * STAGE];           // [stage][rows of x, then columns of w][32]
    int row_tile, col_tile;
    if (!f32_tile(row_tiles, col_tiles, row_tile, col_tile)) return;        // (the whole workgroup)
    const int m0 = row_tile * TILE, n0 = col_tile * TILE;
    const int lane = threadIdx.x % PL_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PL_WAVE);
    const int r = lane % 16, c = lane / 16;
    y += blockIdx.z * sy;

    const int kk = threadIdx.x % LANES * WIDE, first = threadIdx.x / LANES;
    const float* from[LOADS];                                   // rows first + i * 8 WIDE of the stage
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = first + i * 8 * WIDE;
        from[i] = i < LOADS / 2 ? x + blockIdx.z * sx + static_cast<size_t>(min(m0 + row, n - 1)) * ldx
                                : w + blockIdx.z * sw + static_cast<size_t>(min(n0 + row - TILE, N - 1)) * K;
    }
    float* const to = lds + first * F32_BK + ((kk / 4) ^ first % 8) * 4 + kk % 4;
    f32x4 wide[VEC ? LOADS : 1];
    float narrow[VEC ? 1 : LOADS];
    auto ask = [&](int step) {
        const int k = step * F32_BK + kk;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            if (VEC) wide[i] = f32_load4<VEC>(from[i], k, K);
            else narrow[i] = from[i][min(k, K - 1)];
        }
    };
    auto put = [&](int step) {
        const int k = step * F32_BK + kk;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            float* at = to + step % 2 * STAGE + i * 8 * WIDE * F32_BK;
            if (VEC) *reinterpret_cast<f32x4*>(at) = f32_end(wide[i], k, K);
            else *at = k < K ? narrow[i] : 0.f;
        }
    };
    int a_at[2], b_at[2];                   // this lane's operands in a stage, for either half of a step
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int slot = ((c + 4 * h) ^ r % 8) * 4;
        a_at[h] = (TILE + wave % 2 * TM * 16 + r) * F32_BK + slot;
        b_at[h] = (wave / 2 * TN * 16 + r) * F32_BK + slot;
    }
    f32x4 acc[TM][TN], total[TM][TN];
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) total[i][j] = zero;
    ask(0);
    put(0);
    ask(1);
    __syncthreads();
    const int steps = (K + F32_BK - 1) / F32_BK, part_steps = part_len / F32_BK;
    for (int s0 = 0; s0 < steps; s0 += part_steps) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = zero;
        const int stop = min(steps, s0 + part_steps);
        for (int s = s0; s < stop; ++s) {
            const float* stage = lds + s % 2 * STAGE;
            f32x4 a[2][TM], b[2][TN];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int i = 0; i < TM; ++i) a[h][i] = *reinterpret_cast<const f32x4*>(stage + a_at[h] + i * 16 * F32_BK);
#pragma unroll
                for (int j = 0; j < TN; ++j) b[h][j] = *reinterpret_cast<const f32x4*>(stage + b_at[h] + j * 16 * F32_BK);
            }
            put(s + 1);                     // (everybody has read that stage before the last barrier)
            ask(s + 2);
            __builtin_amdgcn_sched_barrier(0);
            f32_multiply<TM, TN>(a[0], b[0], acc);
            f32_multiply<TM, TN>(a[1], b[1], acc);
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) total[i][j] += acc[i][j];
    }
    const bool whole = N % 4 == 0 && ldy % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int row = m0 + (wave / 2 * TN + j) * 16 + r;
        if (row >= n) continue;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int col = n0 + (wave % 2 * TM + i) * 16 + c * 4;
            f32_store4(y + static_cast<size_t>(row) * ldy + col, total[i][j], col, N, whole);
        }
    }
}

namespace {

struct F32Product {
    const float *x, *w;
    float* y;
    int n, N, K, ldx, ldy, batch;
    long sx, sw, sy;
};

template <int TN, bool VEC, int SHARE = 1, bool GATED = false>
void launch_few(const F32Product& g, hipStream_t stream, int act = 0) {
    const dim3 grid(pl_ceil_div(g.N, 16 / SHARE / (GATED ? 2 : 1)), pl_ceil_div(g.n, TN * 16 / SHARE), g.batch);
    gemm_f32_few_kernel<TN, VEC, SHARE, GATED><<<grid, PL_F32_PARTS / SHARE * PL_WAVE, 0, stream>>>(
        g.x, g.w, g.y, g.n, g.N, g.K, g.ldx, g.ldy, g.sx, g.sw, g.sy, f32_part_len(g.K), act);
}

template <int TILE>
void launch_tiled(const F32Product& g, hipStream_t stream) {
    constexpr size_t lds = sizeof(float) * F32_STAGES * 2 * TILE * F32_BK;
    static_assert(lds <= 64 * 1024, "a workgroup's LDS");
    const int row_tiles = pl_ceil_div(g.n, TILE), col_tiles = pl_ceil_div(g.N, TILE);
    const dim3 grid(pl_ceil_div(col_tiles * row_tiles, 8) * 8, 1, g.batch);
    gemm_f32_tiled_kernel<TILE><<<grid, 256, lds, stream>>>(g.x, g.w, g.y, g.n, g.N, g.K, g.ldx, g.ldy, g.sx, g.sw, g.sy,
                                                            f32_part_len(g.K), row_tiles, col_tiles);
}

template <int TILE, bool VEC>
void launch_ragged(const F32Product& g, hipStream_t stream) {
    const int row_tiles = pl_ceil_div(g.n, TILE), col_tiles = pl_ceil_div(g.N, TILE);
    const dim3 grid(pl_ceil_div(col_tiles * row_tiles, 8) * 8, 1, g.batch);
    gemm_f32_ragged_kernel<TILE, VEC><<<grid, 256, 0, stream>>>(g.x, g.w, g.y, g.n, g.N, g.K, g.ldx, g.ldy, g.sx, g.sw, g.sy,
                                                                f32_part_len(g.K), row_tiles, col_tiles);
}

}  // namespace

// `batch` products, their operands and results sx, sw and sy values apart.  Which kernel: up to 16 rows the one for few rows,
// whose workgroups hold all rows and read every weight once; against many columns its 16 columns a workgroup reads the rows
// too often from nine rows on, and from 17 rows on earlier (us, few / tiles of 32: 16 rows, 6,144 x 1,024 12.2 / 12.8, 151,936 x
// 1,024 172 / 141; 32 rows, 4,096 x 1,024 10.2 / 13.1, 6,144 x 1,024 17.0 / 12.9; 64 rows, 4,096 x 1,024 14.1 / 13.2).
// Parts share the instruction where 16 columns a workgroup leave half of the chip idle (us, sixteen parts a workgroup / shared:
// 1,024 x 3,072, 1 row 10.0 / 6.1, 4 rows 11.0 / 6.3, 8 rows 12.4 / 9.1; 1,024 x 2,048, 8 rows 8.9 / 6.9).  Wider ones read x
// too often then (8 rows, 4,096 x 1,024 6.6 / 7.4, 151,936 x 1,024 125 / 164), unless there is one row (4,096 x 1,024 6.3 / 5.7,
// 6,144 x 1,024 9.0 / 7.3, 151,936 x 1,024 113 / 101).
// Tiles of 64 rows by 64 columns or of 32 by 32: the shorter estimate for the compute unit with most of them, a small tile
// costing 1.15 times as much for what it does (700 rows, tiles of 64 / 32: 1,024 x 2,048 43.7 / 34.7, 4,096 x 1,024 62.3 /
// 59.5; 2,048 rows, 1,024 x 2,048 76.7 / 87.6, 4,096 x 1,024 152 / 178).
// Where the tiled kernel does not apply: rows of aligned groups stay with the kernel for few rows while its workgroups are no more than the
// compute units (us, few / ragged tiles of 32: 200 rows, 1,000 x 1,040 12.7 / 15.6, 300 rows 20.5 / 20.0, 700 rows 30.5 / 26.6; 64 rows,
// 4,096 x 4,128 46.0 / 55.9, 96 rows 77.6 / 67.0; 17 rows, 151,936 x 1,028 240 / 162), others only up to 16 rows (17 rows, 4,096 x
// 1,026 19.9 / 17.3, 64 rows 29.9 / 17.5, 1,500 rows 610 / 187).  Ragged tiles of 64 cost a small tile's quarter of 0.83, and another
// quarter of a tile to begin with (tiles of 64 / 32: 200 rows, 4,096 x 1,026 38.5 / 34.6, 700 rows 77.3 / 84.8, 1,500 rows 156 / 187;
// 700 rows, 3,072 x 1,000 65.2 / 59.5, 1,500 rows 107 / 114).  On the vector units, before the matrix instruction was used: 700 and
// 1,500 rows of 4,096 x 1,026 189 and 218.
int pl_gemm_f32(const float* x, const float* w, float* y, int n, int N, int K, int ldx, int ldy, int batch, long sx,
                long sw, long sy, hipStream_t stream) {
    const F32Product g{x, w, y, n, N, K, ldx, ldy, batch, sx, sw, sy};
    const bool vec = K % 4 == 0 && ldx % 4 == 0 && sx % 4 == 0 && sw % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(w) % 16 == 0;
    // (a row of a tile is addressed by 32 bits from the tile's first)
    const bool tiles = vec && K % 64 == 0 && K < (1 << 22) && ldx < (1 << 22);
    const long units = pl_compute_units();
    const auto busiest = [&](int tile) {
        return (static_cast<long>(pl_ceil_div(n, tile)) * pl_ceil_div(N, tile) * batch + units - 1) / units * tile * tile;
    };
    const long few_workgroups = static_cast<long>(pl_ceil_div(n, n <= 32 ? 32 : 64)) * pl_ceil_div(N, 16) * batch;
    const bool few = n <= 8 || (n <= 16 && N < 32768) || (tiles && n <= 32 && N <= 4096) || (vec && !tiles && few_workgroups <= units);
    PL_REQUIRE(static_cast<long>(pl_ceil_div(n, 32)) * (pl_ceil_div(N, 32) + 8) < (1L << 31) && pl_ceil_div(n, 64) <= 65535,
               "gemm: %d x %d results are more than one launch covers", n, N);
    if (few) {
        const bool idle = static_cast<long>(pl_ceil_div(N, 16)) * batch * 2 <= units;
        if (!vec) launch_few<1, false>(g, stream);          // (up to 16 rows)
        else if (n == 1 || (n <= 4 && idle)) launch_few<1, true, 4>(g, stream);
        else if (n <= 8 && idle) launch_few<1, true, 2>(g, stream);
        else if (n <= 16) launch_few<1, true>(g, stream);
        else if (n <= 32) launch_few<2, true>(g, stream);
        else launch_few<4, true>(g, stream);
    } else if (tiles) {
        if (busiest(64) * 20 <= busiest(32) * 23) launch_tiled<64>(g, stream);
        else launch_tiled<32>(g, stream);
    } else if ((busiest(64) + 1000) * 20 <= busiest(32) * 24) {
        if (vec) launch_ragged<64, true>(g, stream);
        else launch_ragged<64, false>(g, stream);
    } else {
        if (vec) launch_ragged<32, true>(g, stream);
        else launch_ragged<32, false>(g, stream);
    }
    PL_CHECK_LAUNCH("gemm_f32");
    return 0;
}

// y[n, I] = act(x . gate^T) * (x . up^T), w [gate | up] of I rows each: one launch instead of two for up to 16 rows whose product
// is the kernel for few rows; the same bits as pl_gemm_f32 and then pl_swiglu.
static bool f32_gated_applies(const void* x, const void* w, int n, int I, int K) {
    return n >= 1 && n <= 16 && (n <= 8 || I < 16384) && I >= 1 && I < (1 << 30) && K >= 4 && K % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(w) % 16 == 0;
}

extern "C" int pl_gemm_f32_gated_applies(const void* x, const void* w, int n, int I, int K) { return f32_gated_applies(x, w, n, I, K) ? 1 : 0; }

extern "C" int pl_gemm_f32_gated(const float* x, const float* w, float* y, int n, int I, int K, int act, hipStream_t stream) {
    PL_REQUIRE(f32_gated_applies(x, w, n, I, K), "gated product: %d rows, %d x %d", n, I, K);
    PL_REQUIRE(act >= PL_ACT_SILU && act <= PL_ACT_RELU2, "gated product: activation code %d", act);
    const F32Product g{x, w, y, n, I, K, K, I, 1, 0, 0, 0};
    if (n == 1) launch_few<1, true, 2, true>(g, stream, act);
    else launch_few<1, true, 1, true>(g, stream, act);
    PL_CHECK_LAUNCH("gemm_f32 (gated)");
    return 0;
}
