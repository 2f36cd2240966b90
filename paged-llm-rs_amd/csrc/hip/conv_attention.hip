// What an attention layer with short convolutions does between its projections and the attention
// kernels: for every token and head, the convolution over the projected rows (with the request's
// carried history), the norm over a head of q and k, the rotation of the first `rot` values of a head
// (value i with value i + rot/2, angle position * freq[i]), and then q into the query buffer and k
// and v into the request's pages.  Heads are stored in rows of Dp values, zeros behind a head's own
// size, so that queries, keys and values of different sizes share the attention kernels' one head size.
// Convolution, norm, angles and rotation are 32-bit; a value is rounded once, when it is stored.
#include "common.hpp"

struct ConvQkArgs {
    const float* rows;        // [n, stride]: the projections, q | k | v from column `off`
    int stride, off;
    const float* conv_w;      // [taps, H*D + G*D + G*V]: a tap's filter values of all channels side by side
    int taps;
    float* state;             // [slots, state_stride], the history at hist_off: [taps - 1][channels]
    long state_stride;
    int hist_off;
    const float* q_gain;      // [D]
    const float* k_gain;      // [D]
    float eps;
    const float* freq;        // [rot / 2], or null
    int rot;
    const int* positions;
    const int* seq_of;
    const int* q_start;
    const int* state_slots;
    const int* block_table;
    int max_blocks, block_size;
    void* q_out;              // [n, H * Dp]
    void* k_pool;             // [pages * block_size, G * Dp]
    void* v_pool;
    int H, G, D, V, Dp;
};

// A step of one token a request: a wave a token and head, all of them at once.  The wave that convolves a request's channels is the only
// one that reads their history, and moves it on as well.  Bound by its chain of trips (position, request, slot, history): everything
// that does not wait for the slot is asked for in front of it, the taps together (TAPS known; otherwise up to 16), and the angles
// are worked out meanwhile.  Two tokens of 16 over 8 heads of 128, four taps: 4.0 us, and 7.7 with the taps one by one, beside a launch of
// 3.8 for the history.
template <typename T, int NI, int TAPS>
__global__ __launch_bounds__(64) void conv_qk_prepare_single_kernel(ConvQkArgs a) {
    __shared__ float head[64 * NI];
    constexpr int MOST = TAPS > 0 ? TAPS : 16;
    const int t = blockIdx.x, which = blockIdx.y, lane = threadIdx.x;
    const int pos = a.positions[t];
    const int s = a.seq_of[t];
    if (pos < 0) return;
    const int H = a.H, G = a.G, D = a.D, V = a.V, Dp = a.Dp;
    const int channels = H * D + G * D + G * V, taps = TAPS > 0 ? TAPS : a.taps;
    const int kind = which < H ? 0 : (which < H + G ? 1 : 2);               // a query head, a key head or a value head
    const int index = kind == 0 ? which : (kind == 1 ? which - H : which - H - G);
    const int width = kind == 2 ? V : D;
    const int c0 = kind == 0 ? index * D : (kind == 1 ? H * D + index * D : H * D + G * D + index * V);
    const int half = a.rot / 2;
    const int slot = a.state_slots[s];
    const int page = kind == 0 ? 0 : a.block_table[static_cast<size_t>(s) * a.max_blocks + pos / a.block_size];
    const float* gains = kind == 0 ? a.q_gain : a.k_gain;
    float u[MOST][NI], w[MOST][NI], gain[NI], turn[NI];
    int at[NI];                         // (past the head's end: its last value again, which is cleared)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int e = lane + 64 * i;
        at[i] = c0 + min(e, width - 1);
        const float now = a.rows[static_cast<size_t>(t) * a.stride + a.off + at[i]];
#pragma unroll
        for (int j = 0; j < MOST; ++j)
            if (j < taps) {
                w[j][i] = a.conv_w[j * channels + at[i]];
                if (j == taps - 1) u[j][i] = now;
            }
        gain[i] = kind != 2 ? gains[min(e, width - 1)] : 0.f;
        turn[i] = kind != 2 && e < a.rot ? a.freq[e < half ? e : e - half] : 0.f;
    }
    if (slot < 0) return;
    float* hist = a.state + static_cast<size_t>(slot) * a.state_stride + a.hist_off;
#pragma unroll
    for (int j = 0; j + 1 < MOST; ++j)
#pragma unroll
        for (int i = 0; i < NI; ++i)
            if (j < taps - 1) u[j][i] = hist[static_cast<size_t>(j) * channels + at[i]];
    float cs[NI], sn[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        cs[i] = 1.f;
        sn[i] = 0.f;
        if (kind != 2 && lane + 64 * i < a.rot) sincosf(static_cast<float>(pos) * turn[i], &sn[i], &cs[i]);
    }
    float x[NI], ss = 0.f;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        x[i] = 0.f;
#pragma unroll
        for (int j = 0; j < MOST; ++j)
            if (j < taps) x[i] += w[j][i] * u[j][i];
        if (lane + 64 * i < width) {
#pragma unroll
            for (int j = 0; j + 1 < MOST; ++j)
                if (j < taps - 1) hist[static_cast<size_t>(j) * channels + at[i]] = u[j + 1][i];
        } else {
            x[i] = 0.f;
        }
        ss = fmaf(x[i], x[i], ss);          // (written out, so that it is rounded as in the kernels of longer portions)
    }
    if (kind != 2) {
        ss = wave_sum(ss);
        const float inv = 1.f / sqrtf(ss / static_cast<float>(D) + a.eps);
#pragma unroll
        for (int i = 0; i < NI; ++i) x[i] = x[i] * inv * gain[i];
        if (a.rot > 0) {
#pragma unroll
            for (int i = 0; i < NI; ++i) head[lane + 64 * i] = x[i];
            __syncthreads();
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int e = lane + 64 * i;
                if (e < a.rot) x[i] = e < half ? x[i] * cs[i] - head[e + half] * sn[i] : x[i] * cs[i] + head[e - half] * sn[i];
            }
        }
    }
    if (page < 0) return;
    const size_t row = static_cast<size_t>(page) * a.block_size + pos % a.block_size;
    T* dst = kind == 0 ? static_cast<T*>(a.q_out) + (static_cast<size_t>(t) * H + index) * Dp
                       : static_cast<T*>(kind == 1 ? a.k_pool : a.v_pool) + (row * G + index) * Dp;
#pragma unroll
    for (int i = 0; i < NI; ++i)
        if (lane + 64 * i < Dp) dst[lane + 64 * i] = from_float<T>(x[i]);
}

// Few tokens of portions: a wave a token and head.
template <typename T>
__global__ __launch_bounds__(64) void conv_qk_prepare_heads_kernel(ConvQkArgs a) {
    __shared__ float head[256];
    const int t = blockIdx.x, which = blockIdx.y, lane = threadIdx.x;
    const int pos = a.positions[t];
    if (pos < 0) return;
    const int s = a.seq_of[t];
    const int slot = a.state_slots[s];
    if (slot < 0) return;
    const int H = a.H, G = a.G, D = a.D, V = a.V, Dp = a.Dp;
    const int channels = H * D + G * D + G * V;
    // which head this wave prepares: a query head, a key head or a value head
    const int kind = which < H ? 0 : (which < H + G ? 1 : 2);
    const int index = kind == 0 ? which : (kind == 1 ? which - H : which - H - G);
    const int width = kind == 2 ? V : D;
    const int c0 = kind == 0 ? index * D : (kind == 1 ? H * D + index * D : H * D + G * D + index * V);
    const float* hist = a.state + static_cast<size_t>(slot) * a.state_stride + a.hist_off;
    const int r = t - a.q_start[s];

    float ss = 0.f;
    for (int e = lane; e < width; e += 64) {
        const int c = c0 + e;
        float acc = 0.f;
        for (int jt = 0; jt < a.taps; ++jt) {
            const int back = a.taps - 1 - jt;
            const int src = r - back;
            const float u = src >= 0 ? a.rows[static_cast<size_t>(t - back) * a.stride + a.off + c]
                                     : hist[static_cast<size_t>(a.taps - 1 + src) * channels + c];
            acc += a.conv_w[jt * channels + c] * u;
        }
        head[e] = acc;
        ss += acc * acc;
    }
    if (kind != 2) {
        ss = wave_sum(ss);
        const float inv = 1.f / sqrtf(ss / static_cast<float>(D) + a.eps);
        const float* gain = kind == 0 ? a.q_gain : a.k_gain;
        for (int e = lane; e < width; e += 64) head[e] = head[e] * inv * gain[e];
    }
    __syncthreads();

    T* dst;
    if (kind == 0) {
        dst = static_cast<T*>(a.q_out) + (static_cast<size_t>(t) * H + index) * Dp;
    } else {
        const int page = a.block_table[static_cast<size_t>(s) * a.max_blocks + pos / a.block_size];
        if (page < 0) return;
        const size_t row = static_cast<size_t>(page) * a.block_size + pos % a.block_size;
        dst = static_cast<T*>(kind == 1 ? a.k_pool : a.v_pool) + (row * G + index) * Dp;
    }
    const int half = a.rot / 2;
    for (int e = lane; e < Dp; e += 64) {
        float x = 0.f;
        if (e < width) {
            x = head[e];
            if (kind != 2 && e < a.rot) {
                const int i = e < half ? e : e - half;
                float sn, cs;
                sincosf(static_cast<float>(pos) * a.freq[i], &sn, &cs);
                x = e < half ? head[e] * cs - head[e + half] * sn : head[e] * cs + head[e - half] * sn;
            }
        }
        dst[e] = from_float<T>(x);
    }
}

// Many tokens (prompt portions): one workgroup a token; its waves take the token's heads (query, key and value heads alike) in turn, and
// the angles' cosines and sines are worked out once for the token.  A wave needs nobody else for a head: a lane holds NI of its values,
// asks for all taps of them together (TAPS known) and finds the ones to turn them with in the wave's own LDS.  Bound by the chain of a
// head's work (3,000 tokens, four taps, 16 query heads over 8 of 128: 36 us for 49 MB of rows, read four times over through the caches, and 25 MB written).  With
// the loads one by one and two barriers a round of four heads it took 75 us.
template <typename T, int NI, int TAPS>
__global__ __launch_bounds__(256) void conv_qk_prepare_kernel(ConvQkArgs a) {
    __shared__ float heads[4][64 * NI];
    __shared__ float cs[128], sn[128];
    const int t = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const int pos = a.positions[t];
    if (pos < 0) return;
    const int s = a.seq_of[t];
    const int slot = a.state_slots[s];
    if (slot < 0) return;
    const int H = a.H, G = a.G, D = a.D, V = a.V, Dp = a.Dp;
    const int channels = H * D + G * D + G * V, taps = TAPS > 0 ? TAPS : a.taps;
    const float* hist = a.state + static_cast<size_t>(slot) * a.state_stride + a.hist_off;
    const int r = t - a.q_start[s];
    const int half = a.rot / 2;
    for (int i = threadIdx.x; i < half; i += 256) sincosf(static_cast<float>(pos) * a.freq[i], &sn[i], &cs[i]);
    int page_row = -1;
    {
        const int page = a.block_table[static_cast<size_t>(s) * a.max_blocks + pos / a.block_size];
        if (page >= 0) page_row = page * a.block_size + pos % a.block_size;
    }
    const auto tap_row = [&](int jt) {
        const int back = taps - 1 - jt, src = r - back;
        return src >= 0 ? a.rows + static_cast<size_t>(t - back) * a.stride + a.off : hist + static_cast<size_t>(taps - 1 + src) * channels;
    };
    float* head = heads[wave];
    __syncthreads();
    for (int which = wave; which < H + 2 * G; which += 4) {
        const int kind = which < H ? 0 : (which < H + G ? 1 : 2);
        const int index = kind == 0 ? which : (kind == 1 ? which - H : which - H - G);
        const int width = kind == 2 ? V : D;
        const int c0 = kind == 0 ? index * D : (kind == 1 ? H * D + index * D : H * D + G * D + index * V);
        float x[NI];
        int at[NI];                     // (past the head's end: its last value again, which is cleared)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            x[i] = 0.f;
            at[i] = c0 + min(lane + 64 * i, width - 1);
        }
        if constexpr (TAPS > 0) {
            float u[TAPS][NI], w[TAPS][NI];
#pragma unroll
            for (int jt = 0; jt < TAPS; ++jt) {
                const float* row = tap_row(jt);
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    u[jt][i] = row[at[i]];
                    w[jt][i] = a.conv_w[jt * channels + at[i]];
                }
            }
#pragma unroll
            for (int jt = 0; jt < TAPS; ++jt)
#pragma unroll
                for (int i = 0; i < NI; ++i) x[i] += w[jt][i] * u[jt][i];
        } else {
            for (int jt = 0; jt < taps; ++jt) {
                const float* row = tap_row(jt);
#pragma unroll
                for (int i = 0; i < NI; ++i) x[i] += a.conv_w[jt * channels + at[i]] * row[at[i]];
            }
        }
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if (lane + 64 * i >= width) x[i] = 0.f;
            ss += x[i] * x[i];
        }
        if (kind != 2) {
            ss = wave_sum(ss);
            const float inv = 1.f / sqrtf(ss / static_cast<float>(D) + a.eps);
            const float* gain = kind == 0 ? a.q_gain : a.k_gain;
#pragma unroll
            for (int i = 0; i < NI; ++i) x[i] = x[i] * inv * gain[min(lane + 64 * i, width - 1)];
            if (a.rot > 0) {
#pragma unroll
                for (int i = 0; i < NI; ++i) head[lane + 64 * i] = x[i];
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const int e = lane + 64 * i;
                    if (e < a.rot) {
                        const int k = e < half ? e : e - half;
                        x[i] = e < half ? x[i] * cs[k] - head[e + half] * sn[k] : x[i] * cs[k] + head[e - half] * sn[k];
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        if (kind != 0 && page_row < 0) continue;
        T* dst = kind == 0 ? static_cast<T*>(a.q_out) + (static_cast<size_t>(t) * H + index) * Dp
                           : static_cast<T*>(kind == 1 ? a.k_pool : a.v_pool) + (static_cast<size_t>(page_row) * G + index) * Dp;
#pragma unroll
        for (int i = 0; i < NI; ++i)
            if (lane + 64 * i < Dp) dst[lane + 64 * i] = from_float<T>(x[i]);
    }
}

template <typename T, int NI>
static void launch_conv_qk(const ConvQkArgs& a, int n, hipStream_t stream) {
    if (a.taps == 4) conv_qk_prepare_kernel<T, NI, 4><<<n, 256, 0, stream>>>(a);
    else conv_qk_prepare_kernel<T, NI, 0><<<n, 256, 0, stream>>>(a);
}

template <typename T>
static void launch_conv_qk(const ConvQkArgs& a, int n, hipStream_t stream) {
    if (a.Dp <= 64) launch_conv_qk<T, 1>(a, n, stream);
    else if (a.Dp <= 128) launch_conv_qk<T, 2>(a, n, stream);
    else launch_conv_qk<T, 4>(a, n, stream);
}

template <typename T, int NI>
static void launch_conv_qk_single(const ConvQkArgs& a, const dim3& grid, hipStream_t stream) {
    if (a.taps == 4) conv_qk_prepare_single_kernel<T, NI, 4><<<grid, 64, 0, stream>>>(a);
    else conv_qk_prepare_single_kernel<T, NI, 0><<<grid, 64, 0, stream>>>(a);
}

template <typename T>
static void launch_conv_qk_single(const ConvQkArgs& a, const dim3& grid, hipStream_t stream) {
    if (a.Dp <= 64) launch_conv_qk_single<T, 1>(a, grid, stream);
    else if (a.Dp <= 128) launch_conv_qk_single<T, 2>(a, grid, stream);
    else launch_conv_qk_single<T, 4>(a, grid, stream);
}

// single: every request of the step brings one token, and the history moves on in the same launch (conv_history is then not called).
extern "C" int pl_conv_qk_prepare(const float* rows, int stride, int off, const float* conv_w, int taps,
                                  float* state, long state_stride, int hist_off,
                                  const float* q_gain, const float* k_gain, float eps, const float* freq, int rot,
                                  const int* positions, const int* seq_of, const int* q_start, const int* state_slots,
                                  const int* block_table, int max_blocks, int block_size,
                                  void* q_out, void* k_pool, void* v_pool, int dtype,
                                  int n, int H, int G, int D, int V, int Dp, int single, hipStream_t stream) {
    PL_REQUIRE(n >= 0 && H > 0 && G > 0 && H % G == 0, "conv_qk_prepare: rows %d, %d query heads over %d key heads", n, H, G);
    PL_REQUIRE(D > 0 && V > 0 && Dp >= D && Dp >= V && Dp <= 256, "conv_qk_prepare: heads of %d and %d in rows of %d (up to 256)", D, V, Dp);
    PL_REQUIRE(taps >= 1 && taps <= 16, "conv_qk_prepare: %d taps", taps);
    PL_REQUIRE(rot >= 0 && rot % 2 == 0 && rot <= D && (rot == 0 || freq != nullptr), "conv_qk_prepare: a rotation over %d of %d values", rot, D);
    PL_REQUIRE(block_size > 0 && max_blocks > 0, "conv_qk_prepare: pages of %d, tables of %d", block_size, max_blocks);
    if (n == 0) return 0;
    ConvQkArgs a{rows, stride, off, conv_w, taps, state, state_stride, hist_off, q_gain, k_gain, eps, freq, rot,
                 positions, seq_of, q_start, state_slots, block_table, max_blocks, block_size, q_out, k_pool, v_pool,
                 H, G, D, V, Dp};
    // (steps of few tokens are bound by the chain of one token's work, which a wave a head keeps shortest;
    // large steps by what they compute and read, where the angles once a token and the heads in rounds pay)
    const bool few = n < 512 && H + 2 * G <= 65535;
    const dim3 grid(n, H + 2 * G);
    PL_REQUIRE(!single || H + 2 * G <= 65535, "conv_qk_prepare: %d heads", H + 2 * G);
    if (single && dtype == PL_DTYPE_F32)
        launch_conv_qk_single<float>(a, grid, stream);
    else if (single && dtype == PL_DTYPE_BF16)
        launch_conv_qk_single<bf16_t>(a, grid, stream);
    else if (dtype == PL_DTYPE_F32) {
        if (few) conv_qk_prepare_heads_kernel<float><<<grid, 64, 0, stream>>>(a);
        else launch_conv_qk<float>(a, n, stream);
    } else if (dtype == PL_DTYPE_BF16) {
        if (few) conv_qk_prepare_heads_kernel<bf16_t><<<grid, 64, 0, stream>>>(a);
        else launch_conv_qk<bf16_t>(a, n, stream);
    }
    else
        PL_REQUIRE(false, "conv_qk_prepare: dtype code %d", dtype);
    PL_CHECK_LAUNCH("conv_qk_prepare");
    return 0;
}
