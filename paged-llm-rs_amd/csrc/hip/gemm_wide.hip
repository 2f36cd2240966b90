// y[n, N] = x[n, K] . w[N, K]^T for up to 32 rows of bfloat16 over very many columns, out of weights in strips (gemm_skinny.hpp has the
// layout: a wave's load of a K step is one contiguous kilobyte), 32-bit sums and results: the projection onto the vocabulary of a
// wide model.
//
// Bound by the weights' trip from memory.  A workgroup of eight waves owns 128 columns; the waves split K, each asks for the weights of its
// steps and the rows of x that they meet (which come from L2) four steps ahead, straight into the matrix instruction's layout, and their
// partial tiles are added in order through LDS.  128 columns a workgroup, because the rows of x travel once for each: 24 rows against 151,936 x
// 5,120 take 281 us (5.5 TB/s), with 64 columns 308, with 32 377; the library 334.  (24 rows, 4,096: 249, library 267; 2,048: 125, streamed
// 144; 9 rows, 5,120: 264, library 309.  With 64 rows the rows' trip costs more than the library's product takes, and below these widths
// the streamed product and the one for few rows are faster: 24 rows, 1,024: 73, 64; 9 rows, 4,096: 236, 215.)  A row's result depends on K
// alone, not on how many rows there are.
#include "common.hpp"

typedef __bf16 gw_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gw_f32x4 __attribute__((ext_vector_type(4)));

#define GW_WAVES 8
#define GW_TILES 8              // tiles of 16 columns a workgroup
#define GW_DEPTH 4              // steps on their way

// MT: tiles of 16 rows.
template <int MT>
__global__ void __launch_bounds__(64 * GW_WAVES, 2)
gemm_wide_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ strips, float* __restrict__ y, int n, int N, int K) {
    extern __shared__ __attribute__((aligned(16))) float gw_red[];          // [wave][tile of columns][tile of rows][256]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int steps = K / 32, each = (steps + GW_WAVES - 1) / GW_WAVES;
    const int first = wave * each, count = min(each, steps - first);        // (the wave's steps)
    const int strip0 = blockIdx.x * GW_TILES, last_strip = N / 16 - 1;
    gw_f32x4 acc[GW_TILES][MT];
#pragma unroll
    for (int b = 0; b < GW_TILES; ++b)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[b][m] = gw_f32x4{0.f, 0.f, 0.f, 0.f};
    if (count > 0) {
        // (bases that are the same for the wave, and 32-bit offsets in bytes: the weights' is the lane's place in a strip's tile)
        const char* wb[GW_TILES];
#pragma unroll
        for (int b = 0; b < GW_TILES; ++b)
            wb[b] = reinterpret_cast<const char*>(strips + (static_cast<size_t>(min(strip0 + b, last_strip)) * steps + first) * 512);
        const char* xb = reinterpret_cast<const char*>(x + first * 32);
        uint32_t x_at[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) x_at[m] = 2u * (static_cast<uint32_t>(min(m * 16 + c, n - 1)) * K + g * 8);
        // (the waves begin at different places of their stretches: with a K that is a power of two these lie at the same place of a memory's
        // pages, and together they would ask the same channels)
        const int turn = wave * count / GW_WAVES;
        gw_bf16x8 a[GW_DEPTH][MT], w[GW_DEPTH][GW_TILES];
        auto ask = [&](int slot, int step) {
            const int within = min(step, count - 1) + turn;                          // (past the end the last step again)
            const uint32_t t = static_cast<uint32_t>(within < count ? within : within - count);
#pragma unroll
            for (int b = 0; b < GW_TILES; ++b) w[slot][b] = *reinterpret_cast<const gw_bf16x8*>(wb[b] + t * 1024u + lane * 16u);
#pragma unroll
            for (int m = 0; m < MT; ++m) a[slot][m] = *reinterpret_cast<const gw_bf16x8*>(xb + (x_at[m] + t * 64u));
        };
#pragma unroll
        for (int d = 0; d < GW_DEPTH; ++d) ask(d, d);
        for (int t = 0; t < count; t += GW_DEPTH) {
#pragma unroll
            for (int d = 0; d < GW_DEPTH; ++d) {
                __builtin_amdgcn_sched_barrier(0);
                if (t + d < count) {
#pragma unroll
                    for (int b = 0; b < GW_TILES; ++b)
#pragma unroll
                        for (int m = 0; m < MT; ++m) acc[b][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][m], w[d][b], acc[b][m], 0, 0, 0);
                }
                ask(d, t + d + GW_DEPTH);
            }
        }
    }
#pragma unroll
    for (int b = 0; b < GW_TILES; ++b)
#pragma unroll
        for (int m = 0; m < MT; ++m) *reinterpret_cast<gw_f32x4*>(gw_red + ((wave * GW_TILES + b) * MT + m) * 256 + lane * 4) = acc[b][m];
    __syncthreads();
    // a lane held rows 4 (lane / 16) + i of column lane % 16; a thread finishes a column of some rows, neighbours neighbouring columns
    constexpr int COLS = 16 * GW_TILES, ROWS = 64 * GW_WAVES / COLS;
    static_assert(64 * GW_WAVES % COLS == 0 && 16 % ROWS == 0, "whole rows a pass");
    const int col = threadIdx.x % COLS, b = col / 16;
    if (strip0 + b > last_strip) return;
#pragma unroll
    for (int r0 = 0; r0 < 16 * MT; r0 += ROWS) {
        const int row = r0 + threadIdx.x / COLS;
        if (row >= n) break;
        const float* at = gw_red + (b * MT + row / 16) * 256 + (row % 16 / 4 * 16 + col % 16) * 4 + row % 4;
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < GW_WAVES; ++k) sum += at[k * GW_TILES * MT * 256];
        y[static_cast<size_t>(row) * N + strip0 * 16 + col] = sum;
    }
}

template <int MT>
static int launch_wide(const void* x, const void* strips, float* y, int n, int N, int K, hipStream_t stream) {
    const size_t lds = sizeof(float) * GW_WAVES * GW_TILES * MT * 256;
    if (lds > 48 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_wide_kernel<MT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 static_cast<int>(lds));
        PL_REQUIRE(e == hipSuccess, "wide product: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
    }
    gemm_wide_kernel<MT><<<pl_ceil_div(N / 16, GW_TILES), 64 * GW_WAVES, lds, stream>>>(
        static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(strips), y, n, N, K);
    PL_CHECK_LAUNCH("gemm_wide");
    return 0;
}

// x [n, K] bfloat16, strips: w [N, K] in strips; y [n, N] 32-bit.
extern "C" int pl_gemm_wide(const void* x, const void* strips, float* y, int n, int N, int K, hipStream_t stream) {
    PL_REQUIRE(n >= 0 && n <= 32, "wide product: %d rows, it takes up to 32", n);
    PL_REQUIRE(N > 0 && N % 16 == 0 && K > 0 && K % 32 == 0 && K <= (1 << 22), "wide product: %d columns, inner width %d", N, K);
    PL_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(strips) % 16 == 0, "wide product: operands that are not aligned");
    if (n == 0) return 0;
    return n <= 16 ? launch_wide<1>(x, strips, y, n, N, K, stream) : launch_wide<2>(x, strips, y, n, N, K, stream);
}
