// The state space whose decay and step size come with the token (kind ssd of the scans): per head, with
// dt = softplus(x1 + dt_bias) and a = e^A_log,
//     S_t = e^(-a dt_t) S_(t-1) + dt_t B_t x_t^T   (N x V),     y_t = S_t^T C_t + D x_t .
// q, k and v of the scan's arguments are C, B and x; C and B have G heads, head h reads head h / (H / G).
//
// Linear attention with a fixed decay a head (kind retention) is the same recurrence with e^(-a dt) = decay, dt = 1 in front of
// B x^T and no D: the chunked kernels serve it too (p1 holds the decays), retention_step is its kernel for few tokens.
// Its q and k turn with their positions: retention_turn does that to a step's rows in front of the chunked kernels,
// retention_step to what it reads.
//
// ssd_step: requests of few tokens, token by token, the state read and written once, 16 bytes a lane.
//
// ssd_chunked: requests of many tokens in chunks of 64.  With b_t the sum of -a dt over a chunk's tokens up to t,
//     y_t = sum_{u<=t} e^(b_t - b_u) dt_u (C_t . B_u) x_u + e^(b_t) S_0^T C_t + D x_t ,
// so a chunk adds sum_u e^(b_L - b_u) dt_u B_u x_u^T to the state (`summary`, every chunk at once), the states
// before the chunks follow by a short walk (`carry`), and a chunk's read-outs are three small products (`output`,
// every chunk at once).  The products run on the matrix cores in 32-bit (v_mfma_f32_32x32x2_f32: 32-bit operands, 32-bit
// multiply-add).  The sums b are kept in 64-bit: decays of a chunk may be anything from 1 to 0 beside each other, what
// enters an exponential is a difference of two sums, and a small difference of large sums would lose its digits in 32.
//
// The matrix instruction, D[32 x 32] += A[32 x 2] B[2 x 32]: lane l gives A[l % 32][l / 32] and B[l / 32][l % 32]
// and holds, in register r, D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].  The order of the inner index is free as long as A and
// B agree: the two halves of a wave take runs of four, 8 q + 4 (l / 32) + e for e = 0 .. 3, so that an operand whose
// rows lie along the inner index is read 16 bytes a lane.
#include "recurrent.hpp"

typedef float ssd_f32x16 __attribute__((ext_vector_type(16)));
typedef float ssd_f32x4 __attribute__((ext_vector_type(4)));

#define SSD_CHUNK 64

__device__ __forceinline__ ssd_f32x16 ssd_mfma(float a, float b, ssd_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// ---- few tokens ----------------------------------------------------------------------------------------

// A workgroup of four waves owns 64 columns of a head's state for one request.  A thread holds R rows of four columns:
// rows (4 wave + lane / 16) R .. + R - 1, columns 4 (lane % 16) .. + 3.  ALIGNED: k, q and v may be read 16 bytes at a time.
template <int R, bool ALIGNED>
__global__ __launch_bounds__(256) void ssd_step_kernel(ScanArgs a) {
    __shared__ ssd_f32x4 part[4][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = blockIdx.y, s = blockIdx.z;
    const int slot = a.state_slots[s];
    const int count = a.q_len[s];
    if (slot < 0 || count <= 0 || (a.below > 0 && count >= a.below)) return;
    const int start = a.q_start[s];
    const int N = a.D, V = a.V, H = a.H;
    const int g = h / (H / a.G);
    const int n0 = (4 * wave + (lane >> 4)) * R;
    const int v0 = blockIdx.x * 64 + 4 * (lane & 15);
    const bool owns = v0 < V;                                   // (V is a multiple of 4)
    float* Sg = a.state + static_cast<size_t>(slot) * a.state_stride + a.s_off + static_cast<size_t>(h) * N * V;
    ssd_f32x4 S[R];
#pragma unroll
    for (int i = 0; i < R; ++i)
        S[i] = (owns && n0 + i < N) ? *reinterpret_cast<const ssd_f32x4*>(Sg + static_cast<size_t>(n0 + i) * V + v0) : ssd_f32x4{0.f, 0.f, 0.f, 0.f};
    const float rate = expf(a.p1[h]), bias = a.p2[h], skip = a.p3[h];
    for (int t = 0; t < count; ++t) {
        const float* row = a.qkv + static_cast<size_t>(start + t) * a.qkv_stride;
        const float* kr = row + a.k_off + g * N;
        const float* qr = row + a.q_off + g * N;
        float k[R], q[R];
        if (ALIGNED && R % 4 == 0) {                            // (N is a multiple of 4 then)
#pragma unroll
            for (int i = 0; i < R; i += 4) {
                const bool in = n0 + i < N;
                const ssd_f32x4 kk = in ? *reinterpret_cast<const ssd_f32x4*>(kr + n0 + i) : ssd_f32x4{0.f, 0.f, 0.f, 0.f};
                const ssd_f32x4 qq = in ? *reinterpret_cast<const ssd_f32x4*>(qr + n0 + i) : ssd_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    k[(i + e) % R] = kk[e];
                    q[(i + e) % R] = qq[e];
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < R; ++i) {
                k[i] = n0 + i < N ? kr[n0 + i] : 0.f;
                q[i] = n0 + i < N ? qr[n0 + i] : 0.f;
            }
        }
        ssd_f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (owns) {
            const float* vr = row + a.v_off + h * V + v0;
            if (ALIGNED) v = *reinterpret_cast<const ssd_f32x4*>(vr);
            else v = ssd_f32x4{vr[0], vr[1], vr[2], vr[3]};
        }
        const float dt = softplus_f(a.gates[static_cast<size_t>(start + t) * a.gates_stride + a.g1_off + h] + bias);
        const float keep = expf(-rate * dt);
        ssd_f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const float kd = k[i] * dt;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                S[i][e] = keep * S[i][e] + kd * v[e];
                o[e] += S[i][e] * q[i];
            }
        }
#pragma unroll
        for (int off = 16; off < 64; off <<= 1)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] += __shfl_xor(o[e], off, 64);
        if (lane < 16) part[wave][lane] = o;
        __syncthreads();
        if (wave == 0 && lane < 16 && owns) {
            ssd_f32x4 y = part[0][lane];
#pragma unroll
            for (int w = 1; w < 4; ++w)
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] += part[w][lane][e];
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] += skip * v[e];
            *reinterpret_cast<ssd_f32x4*>(a.out + static_cast<size_t>(start + t) * (H * V) + h * V + v0) = y;
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
        if (owns && n0 + i < N) *reinterpret_cast<ssd_f32x4*>(Sg + static_cast<size_t>(n0 + i) * V + v0) = S[i];
}

// How q and k of a head turn: values i and i + dims / 2 by position * freq[i], cosine and sine times `amplitude`, i < dims / 2;
// k times `k_scale` behind that.
struct HalfTurn {
    const float* freq;
    const int* positions;
    int dims;
    float amplitude, k_scale;
};

// Pair i of q and k (values i and i + dims / 2), turned.
struct TurnedPair {
    float q0, q1, k0, k1;
};
__device__ __forceinline__ TurnedPair turn_pair(const float* q, const float* k, int i, int half, float cs, float sn, float k_scale) {
    const float q0 = q[i], q1 = q[i + half], k0 = k[i], k1 = k[i + half];
    return {q0 * cs - q1 * sn, q1 * cs + q0 * sn, (k0 * cs - k1 * sn) * k_scale, (k1 * cs + k0 * sn) * k_scale};
}
__device__ __forceinline__ void half_angle(const HalfTurn& turn, int position, int i, float& cs, float& sn) {
    sincosf(static_cast<float>(position) * turn.freq[i], &sn, &cs);
    cs *= turn.amplitude;
    sn *= turn.amplitude;
}

// As ssd_step_kernel, a workgroup 64 columns of a head's state for one request; every token's q and k are turned into LDS first
// (`turns`: they have not been turned yet).
template <int R>
__global__ __launch_bounds__(256) void retention_step_kernel(ScanArgs a, HalfTurn turn, int turns) {
    __shared__ ssd_f32x4 part[4][16];
    __shared__ __attribute__((aligned(16))) float qs[16 * R], ks[16 * R];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = blockIdx.y, s = blockIdx.z;
    const int slot = a.state_slots[s];
    const int count = a.q_len[s];
    if (slot < 0 || count <= 0 || (a.below > 0 && count >= a.below)) return;
    const int start = a.q_start[s];
    const int N = a.D, V = a.V, H = a.H;
    const int n0 = (4 * wave + (lane >> 4)) * R;
    const int v0 = blockIdx.x * 64 + 4 * (lane & 15);
    const bool owns = v0 < V;                                   // (V is a multiple of 4)
    float* Sg = a.state + static_cast<size_t>(slot) * a.state_stride + a.s_off + static_cast<size_t>(h) * N * V;
    ssd_f32x4 S[R];
#pragma unroll
    for (int i = 0; i < R; ++i)
        S[i] = (owns && n0 + i < N) ? *reinterpret_cast<const ssd_f32x4*>(Sg + static_cast<size_t>(n0 + i) * V + v0) : ssd_f32x4{0.f, 0.f, 0.f, 0.f};
    const float keep = a.p1[h];
    const int half = turns ? turn.dims / 2 : 0;
    const float k_scale = turns ? turn.k_scale : 1.f;
    for (int i = N + tid; i < 16 * R; i += 256) qs[i] = ks[i] = 0.f;
    for (int t = 0; t < count; ++t) {
        const float* row = a.qkv + static_cast<size_t>(start + t) * a.qkv_stride;
        const float* kr = row + a.k_off + h * N;
        const float* qr = row + a.q_off + h * N;
        ssd_f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (owns) {
            const float* vr = row + a.v_off + h * V + v0;
            v = ssd_f32x4{vr[0], vr[1], vr[2], vr[3]};
        }
        if (tid < half) {
            float cs, sn;
            half_angle(turn, turn.positions[start + t], tid, cs, sn);
            const TurnedPair p = turn_pair(qr, kr, tid, half, cs, sn, k_scale);
            qs[tid] = p.q0;
            qs[tid + half] = p.q1;
            ks[tid] = p.k0;
            ks[tid + half] = p.k1;
        } else if (tid + half < N) {
            qs[tid + half] = qr[tid + half];
            ks[tid + half] = kr[tid + half] * k_scale;
        }
        __syncthreads();
        float k[R], q[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            k[i] = ks[n0 + i];
            q[i] = qs[n0 + i];
        }
        ssd_f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                S[i][e] = keep * S[i][e] + k[i] * v[e];
                o[e] += S[i][e] * q[i];
            }
#pragma unroll
        for (int off = 16; off < 64; off <<= 1)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] += __shfl_xor(o[e], off, 64);
        if (lane < 16) part[wave][lane] = o;
        __syncthreads();
        if (wave == 0 && lane < 16 && owns) {
            ssd_f32x4 y = part[0][lane];
#pragma unroll
            for (int w = 1; w < 4; ++w)
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] += part[w][lane][e];
            *reinterpret_cast<ssd_f32x4*>(a.out + static_cast<size_t>(start + t) * (H * V) + h * V + v0) = y;
        }
        // (nobody writes `part` again before the next token's first barrier, which the first wave reaches behind its reads)
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
        if (owns && n0 + i < N) *reinterpret_cast<ssd_f32x4*>(Sg + static_cast<size_t>(n0 + i) * V + v0) = S[i];
}

// A workgroup a token: q and k of every head, turned in place.
__global__ __launch_bounds__(256) void retention_turn_kernel(float* __restrict__ rows, int stride, int q_off, int k_off, int H, int N, HalfTurn turn) {
    __shared__ float cosine[128], sine[128];
    const int t = blockIdx.x;
    const int position = turn.positions[t];
    if (position < 0) return;
    const int half = turn.dims / 2, each = N - half;             // pairs, then the values that do not turn
    for (int i = threadIdx.x; i < half; i += 256) half_angle(turn, position, i, cosine[i], sine[i]);
    __syncthreads();
    float* row = rows + static_cast<size_t>(t) * stride;
    for (int e = threadIdx.x; e < H * each; e += 256) {
        const int h = e / each, i = e - h * each;
        float* q = row + q_off + h * N;
        float* k = row + k_off + h * N;
        if (i < half) {
            const TurnedPair p = turn_pair(q, k, i, half, cosine[i], sine[i], turn.k_scale);
            q[i] = p.q0;
            q[i + half] = p.q1;
            k[i] = p.k0;
            k[i + half] = p.k1;
        } else {
            k[i + half] *= turn.k_scale;
        }
    }
}

// The other recurrences, token by token (kinds lightning, mlstm and delta): a workgroup of four waves owns 64 columns of a head's
// state for one request, as above.  Bound by the chain of a token: state and rows on their way together, one round through
// LDS for the read-out (delta: two more, for the unit vectors and for what the memory says to the key).  A wave with a
// column of the state a lane (the scan kernel) asks for D rows one after the other and adds them up alone: 20 to 25 us for one token of
// two requests (8 heads of 128 by 128, 4 of 128 by 256), and 5.5 here.
template <int R, int KIND>
__global__ __launch_bounds__(256) void state_step_kernel(ScanArgs a) {
    __shared__ ssd_f32x4 part[4][16], memory[4][16];
    __shared__ __attribute__((aligned(16))) float qs[16 * R], ks[16 * R];
    __shared__ float sums[2][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = blockIdx.y, s = blockIdx.z;
    const int slot = a.state_slots[s];
    const int count = a.q_len[s];
    if (slot < 0 || count <= 0 || (a.below > 0 && count >= a.below)) return;
    const int start = a.q_start[s];
    const int N = a.D, V = a.V, H = a.H, g = h / (H / a.G), tiles = gridDim.x;
    const int n0 = (4 * wave + (lane >> 4)) * R;
    const int v0 = blockIdx.x * 64 + 4 * (lane & 15);
    const bool owns = v0 < V;                                   // (V is a multiple of 4)
    float* slot_state = a.state + static_cast<size_t>(slot) * a.state_stride;
    float* Sg = slot_state + a.s_off + static_cast<size_t>(h) * N * V;
    ssd_f32x4 S[R];
#pragma unroll
    for (int i = 0; i < R; ++i)
        S[i] = (owns && n0 + i < N) ? *reinterpret_cast<const ssd_f32x4*>(Sg + static_cast<size_t>(n0 + i) * V + v0) : ssd_f32x4{0.f, 0.f, 0.f, 0.f};
    // (every tile of columns has a copy of the normaliser and of the maximum of its own: see the scan kernel)
    float* ng = slot_state + a.n_off + (static_cast<size_t>(h) * tiles + blockIdx.x) * N + tid;
    float* mg = slot_state + a.m_off + h * tiles + blockIdx.x;
    float nv = 0.f, m = 0.f;
    if (KIND == PL_SCAN_MLSTM) {
        if (tid < N) nv = *ng;
        m = *mg;
    }
    const float c1 = KIND == PL_SCAN_DELTA ? expf(a.p1[h]) : a.p1[h], c2 = KIND == PL_SCAN_LIGHTNING ? 0.f : a.p2[h];
    const float q_scale = 1.f / sqrtf(static_cast<float>(N));
    for (int i = N + tid; i < 16 * R; i += 256) qs[i] = ks[i] = 0.f;
    for (int t = 0; t < count; ++t) {
        const float* row = a.qkv + static_cast<size_t>(start + t) * a.qkv_stride;
        ssd_f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (owns) {
            const float* vr = row + a.v_off + h * V + v0;
            v = ssd_f32x4{vr[0], vr[1], vr[2], vr[3]};
        }
        float q = 0.f, k = 0.f, x1 = 0.f, x2 = 0.f;
        if (tid < N) {
            q = row[a.q_off + g * N + tid];
            k = row[a.k_off + g * N + tid];
        }
        if (KIND != PL_SCAN_LIGHTNING) {
            const float* gates = a.gates + static_cast<size_t>(start + t) * a.gates_stride;
            x1 = gates[a.g1_off + h];
            x2 = gates[a.g2_off + h];
        }
        if (KIND == PL_SCAN_LIGHTNING) {
            q = silu_f(q);
            k = silu_f(k);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = silu_f(v[e]);
        }
        if (KIND == PL_SCAN_MLSTM) q *= q_scale;
        if (KIND == PL_SCAN_DELTA) {
            const float qq = wave_sum(q * q), kk = wave_sum(k * k);
            if (lane == 0) {
                sums[0][wave] = qq;
                sums[1][wave] = kk;
            }
        }
        if (tid < N) {
            qs[tid] = q;
            ks[tid] = k;
        }
        __syncthreads();
        float kr[R], qr[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            kr[i] = ks[n0 + i];
            qr[i] = qs[n0 + i];
        }
        float keep = c1, add = 1.f, below = 0.f;
        if (KIND == PL_SCAN_MLSTM) {
            const float gi = a.cap * tanhf((x1 + c1) / a.cap), gf = logsigmoid_f(a.cap * tanhf((x2 + c2) / a.cap));
            const float top = fmaxf(gf + m, gi);
            keep = expf(gf + m - top);
            add = expf(gi - top);
            m = top;
            below = expf(-top);
            nv = keep * nv + add * k;
            const float nq = wave_sum(nv * q);
            if (lane == 0) sums[0][wave] = nq;
        }
        if (KIND == PL_SCAN_DELTA) {
            const float qq = sums[0][0] + sums[0][1] + sums[0][2] + sums[0][3], kk = sums[1][0] + sums[1][1] + sums[1][2] + sums[1][3];
            const float by_q = 1.f / sqrtf(qq + 1e-6f) * q_scale, by_k = 1.f / sqrtf(kk + 1e-6f);
            keep = expf(-c1 * softplus_f(x2 + c2));
            ssd_f32x4 says = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < R; ++i) {
                kr[i] *= by_k;
                qr[i] *= by_q;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    S[i][e] *= keep;
                    says[e] += S[i][e] * kr[i];
                }
            }
#pragma unroll
            for (int off = 16; off < 64; off <<= 1)
#pragma unroll
                for (int e = 0; e < 4; ++e) says[e] += __shfl_xor(says[e], off, 64);
            if (lane < 16) memory[wave][lane] = says;
            __syncthreads();
            const float beta = sigmoid_f(x1);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float said = 0.f;
#pragma unroll
                for (int w = 0; w < 4; ++w) said += memory[w][lane & 15][e];
                v[e] = beta * (v[e] - said);
            }
            keep = 1.f;
        }
        ssd_f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= add;
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                S[i][e] = keep * S[i][e] + kr[i] * v[e];
                o[e] += S[i][e] * qr[i];
            }
#pragma unroll
        for (int off = 16; off < 64; off <<= 1)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] += __shfl_xor(o[e], off, 64);
        if (lane < 16) part[wave][lane] = o;
        __syncthreads();
        if (wave == 0 && lane < 16 && owns) {
            ssd_f32x4 y = part[0][lane];
#pragma unroll
            for (int w = 1; w < 4; ++w)
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] += part[w][lane][e];
            if (KIND == PL_SCAN_MLSTM) {
                const float nq = sums[0][0] + sums[0][1] + sums[0][2] + sums[0][3];
                const float by = 1.f / (fmaxf(fabsf(nq), below) + 1e-6f);
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] *= by;
            }
            *reinterpret_cast<ssd_f32x4*>(a.out + static_cast<size_t>(start + t) * (H * V) + h * V + v0) = y;
        }
        // (what the first wave reads here, `part` and mlstm's `sums`, is written again behind the next token's first barrier, which
        // the first wave reaches behind its reads; delta's `sums` were read by everybody before this token's last barrier)
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
        if (owns && n0 + i < N) *reinterpret_cast<ssd_f32x4*>(Sg + static_cast<size_t>(n0 + i) * V + v0) = S[i];
    if (KIND == PL_SCAN_MLSTM) {
        if (tid < N) *ng = nv;
        if (tid == 0) *mg = m;
    }
}

template <int KIND>
static void launch_step(const ScanArgs& a, int seqs, hipStream_t stream) {
    const dim3 grid(pl_ceil_div(a.V, 64), a.H, seqs);
    if (a.D <= 32) state_step_kernel<2, KIND><<<grid, 256, 0, stream>>>(a);
    else if (a.D <= 64) state_step_kernel<4, KIND><<<grid, 256, 0, stream>>>(a);
    else if (a.D <= 128) state_step_kernel<8, KIND><<<grid, 256, 0, stream>>>(a);
    else state_step_kernel<16, KIND><<<grid, 256, 0, stream>>>(a);
}

// The kernel above needs whole aligned quads of columns.  False: it does not apply, and nothing was launched.
bool pl_state_step(int kind, const ScanArgs& a, int seqs, hipStream_t stream) {
    if (a.V % 4 != 0 || a.state_stride % 4 != 0 || a.s_off % 4 != 0 || reinterpret_cast<uintptr_t>(a.state) % 16 != 0 ||
        reinterpret_cast<uintptr_t>(a.out) % 16 != 0)
        return false;
    if (kind == PL_SCAN_LIGHTNING) launch_step<PL_SCAN_LIGHTNING>(a, seqs, stream);
    else if (kind == PL_SCAN_MLSTM) launch_step<PL_SCAN_MLSTM>(a, seqs, stream);
    else if (kind == PL_SCAN_DELTA) launch_step<PL_SCAN_DELTA>(a, seqs, stream);
    else return false;
    return true;
}

// ---- many tokens -----------------------------------------------------------------------------------------

struct SsdArgs {
    ScanArgs a;
    float* U;        // [chunks, H, N, V]  a chunk's weighted sum of B x^T
    float* Sin;      // [chunks, H, N, V]  the state before a chunk
    float* ends;     // [chunks, H]        b at the chunk's end
    // the matrix memory's, null for the others
    float* Uk;       // [chunks, H, N]     a chunk's weighted sum of B, for the normaliser
    float* nin;      // [chunks, H, N]     the normaliser before a chunk
    float* tops;     // [chunks, H, 2]     b at the chunk's end plus the largest w_t - b_t; the running maximum before the chunk
};

// A request's chunks have numbers of their own among all chunks of the step: requests lie one behind the
// other in the step's rows, so q_start / 64 + (index of the request) + (chunk in the request) is unique.
__device__ __forceinline__ int ssd_chunk(const ScanArgs& a, int s, int c) { return a.q_start[s] / SSD_CHUNK + s + c; }

// By one wave, all its lanes: the running sums b (64-bit) and the step sizes of a chunk's L <= 64 tokens; the sum
// over the chunk comes back.  Lanes past the chunk hold the last sum and a step of zero.  The matrix memory has in the
// place of the step size the log weight of a token's write less b (64-bit; -inf past the chunk).
template <int KIND>
__device__ __forceinline__ double ssd_gates(const ScanArgs& a, int h, int row0, int L, int lane, double& b, double& dt) {
    dt = KIND == PL_SCAN_MLSTM ? -INFINITY : 0.0;
    if (KIND == PL_SCAN_RETENTION || KIND == PL_SCAN_LIGHTNING) {
        const double each = log(static_cast<double>(a.p1[h]));
        if (lane < L) dt = 1.0;
        b = each * (min(lane, L - 1) + 1);
        return each * L;
    }
    double sum = 0.0;
    if (KIND == PL_SCAN_MLSTM) {
        if (lane < L) {
            const float* gates = a.gates + static_cast<size_t>(row0 + lane) * a.gates_stride;
            dt = a.cap * tanhf((gates[a.g1_off + h] + a.p1[h]) / a.cap);
            sum = logsigmoid_f(a.cap * tanhf((gates[a.g2_off + h] + a.p2[h]) / a.cap));
        }
    } else {
        if (lane < L) dt = softplus_f(a.gates[static_cast<size_t>(row0 + lane) * a.gates_stride + a.g1_off + h] + a.p2[h]);
        sum = -static_cast<double>(expf(a.p1[h])) * dt;
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double other = __shfl_up(sum, off, 64);
        if (lane >= off) sum += other;
    }
    b = sum;
    if (KIND == PL_SCAN_MLSTM) dt -= b;
    return __shfl(sum, L - 1, 64);
}

// What the rows hold becomes q, k and v: linear attention takes them through silu, the matrix memory scales its queries.
template <int KIND>
__device__ __forceinline__ float ssd_kv(float x) { return KIND == PL_SCAN_LIGHTNING ? silu_f(x) : x; }
template <int KIND>
__device__ __forceinline__ float ssd_q(float x, float scale) { return KIND == PL_SCAN_MLSTM ? x * scale : ssd_kv<KIND>(x); }

// (Retention and lightning: one decay a head, p1, and steps of one.  The matrix memory, mlstm: with w_t the log weight of token
// t's write and m the maximum that holds its exponentials, m_t = b_t + max(m_0, max_{u<=t} (w_u - b_u)), which is the very
// sequence that the token-by-token form walks through, every exponent is at or below zero:
//     y_t = (sum_{u<=t} e^(w_u - b_u - c_t) (q_t . k_u) v_u + e^(m_0 - c_t) S_0^T q_t) / max(|n . q|, e^(-m_t)),  c_t = m_t - b_t,
// with n . q the same sum without v_u and S_0.)

// summary: a wave a tile of 32 rows of N (and the tile four further on, where N has more than 128), 64 columns of V.
// Both operands come straight from memory, a token a row: 128 bytes a half wave.
template <int KIND>
__global__ __launch_bounds__(256) void ssd_summary_kernel(SsdArgs sa) {
    const ScanArgs& a = sa.a;
    __shared__ float weight[SSD_CHUNK];
    const int N = a.D, V = a.V, H = a.H;
    const int tiles = (V + 63) / 64;
    const int c = blockIdx.x, h = blockIdx.y / tiles, vt = blockIdx.y % tiles, s = blockIdx.z;
    const int slot = a.state_slots[s], count = a.q_len[s];
    if (slot < 0 || count < a.below || c * SSD_CHUNK >= count) return;
    const int L = min(SSD_CHUNK, count - c * SSD_CHUNK), row0 = a.q_start[s] + c * SSD_CHUNK;
    const size_t idx = static_cast<size_t>(ssd_chunk(a, s, c)) * H + h;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int g = h / (H / a.G);
    const bool two = vt * 64 + 32 < V;               // whether the second 32 columns exist
    const int va = min(vt * 64 + l32, V - 1), vb = min(vt * 64 + 32 + l32, V - 1);
    float xa[SSD_CHUNK / 2], xb[SSD_CHUNK / 2];
    const float* rows = a.qkv + static_cast<size_t>(row0) * a.qkv_stride;
    // (every load before the first silu: one behind a branch would be waited for alone)
#pragma unroll
    for (int k = 0; k < SSD_CHUNK / 2; ++k) {
        const float* x = rows + static_cast<size_t>(min(2 * k + half, L - 1)) * a.qkv_stride + a.v_off + h * V;
        xa[k] = x[va];
        xb[k] = x[vb];
    }
    if (wave == 0) {
        double b, dt;
        const double end = ssd_gates<KIND>(a, h, row0, L, lane, b, dt);
        if (KIND == PL_SCAN_MLSTM) {
            double top = dt;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) top = fmax(top, __shfl_xor(top, off, 64));
            weight[lane] = expf(static_cast<float>(dt - top));
            if (vt == 0 && lane == 0) {
                // (their sum: either may be hundreds where it is small, and rounded alone would leave its rounding in the state)
                sa.tops[2 * idx] = static_cast<float>(end + top);
                // the maximum that the request's first chunk starts from: the carry reads it here, not in the slot it writes
                if (c == 0) sa.tops[2 * idx + 1] = a.state[static_cast<size_t>(slot) * a.state_stride + a.m_off + h * tiles];
            }
        } else {
            weight[lane] = expf(static_cast<float>(end - b)) * static_cast<float>(dt);  // (zero past the chunk's tokens)
        }
        if (vt == 0 && lane == 0) sa.ends[idx] = static_cast<float>(end);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SSD_CHUNK / 2; ++k) {
        const float w = weight[2 * k + half];
        xa[k] = ssd_kv<KIND>(xa[k]) * w;
        xb[k] = ssd_kv<KIND>(xb[k]) * w;
    }
    float* U = sa.U + idx * N * V;
    for (int n0 = wave * 32; n0 < N; n0 += 128) {
        const int n = min(n0 + l32, N - 1);
        float ka[SSD_CHUNK / 2];
#pragma unroll
        for (int k = 0; k < SSD_CHUNK / 2; ++k)
            ka[k] = rows[static_cast<size_t>(min(2 * k + half, L - 1)) * a.qkv_stride + a.k_off + g * N + n];
        if (KIND == PL_SCAN_LIGHTNING) {
#pragma unroll
            for (int k = 0; k < SSD_CHUNK / 2; ++k) ka[k] = ssd_kv<KIND>(ka[k]);
        }
        if (KIND == PL_SCAN_MLSTM && vt == 0) {
            float sum = 0.f;
#pragma unroll
            for (int k = 0; k < SSD_CHUNK / 2; ++k) sum += weight[2 * k + half] * ka[k];
            sum += __shfl_xor(sum, 32, 64);
            if (half == 0 && n0 + l32 < N) sa.Uk[idx * N + n0 + l32] = sum;
        }
        ssd_f32x16 da, db;
#pragma unroll
        for (int r = 0; r < 16; ++r) da[r] = db[r] = 0.f;
#pragma unroll
        for (int k = 0; k < SSD_CHUNK / 2; ++k) {
            da = ssd_mfma(ka[k], xa[k], da);
            if (two) db = ssd_mfma(ka[k], xb[k], db);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = n0 + 8 * (r >> 2) + 4 * half + (r & 3);
            if (row >= N) continue;
            if (vt * 64 + l32 < V) U[static_cast<size_t>(row) * V + vt * 64 + l32] = da[r];
            if (vt * 64 + 32 + l32 < V) U[static_cast<size_t>(row) * V + vt * 64 + 32 + l32] = db[r];
        }
    }
}

// summary_pair, the same for two tiles of 64 columns of V a workgroup, four waves each; of a tile, a wave 32 rows of N (and the 32 four further on, where N
// has more than 128).  Both operands go through LDS, a token a row, so that a value is read and activated once a workgroup; rows there are
// 16 values longer than they hold.  What it is bound by: the trip to memory, the activation (silu of linear attention: an exponential and a
// division a value) and the trip back, one behind the other.  42 chunks of 8 heads of 128 by 128: 26.4 us (34.4 with every wave
// reading and activating all of v and a workgroup for each 64 columns and each chunk that there might be), of 4 heads of 128 by 256
// (matrix memory) 24.7 (24.5); 25 chunks of the first 17.8 (28.7).
#define SSD_SUMMARY_PAD 16
template <int KIND>
__global__ __launch_bounds__(512) void ssd_summary_pair_kernel(SsdArgs sa, int seqs, int aligned) {
    const ScanArgs& a = sa.a;
    __shared__ float weight[SSD_CHUNK];
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int T = 512, COLS = 128, XP = COLS + SSD_SUMMARY_PAD;
    const int N = a.D, V = a.V, H = a.H;
    const int tiles = (V + COLS - 1) / COLS;
    const int h = blockIdx.y / tiles, vt = blockIdx.y % tiles;
    ChunkPlace place;
    if (!find_chunk(a, seqs, blockIdx.x, place)) return;
    const int c = place.c, s = place.s;
    const int L = min(SSD_CHUNK, place.count - c * SSD_CHUNK), row0 = place.first_row + c * SSD_CHUNK;
    const size_t idx = static_cast<size_t>(place.first_row / SSD_CHUNK + s + c) * H + h;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int g = h / (H / a.G);
    const int Nq = (N + 31) / 32 * 32, KP = Nq + SSD_SUMMARY_PAD;
    float* Xs = lds;                                  // [64][XP]
    float* Ks = lds + SSD_CHUNK * XP;                 // [64][KP]
    const float* rows = a.qkv + static_cast<size_t>(row0) * a.qkv_stride;
    const float* v_at = rows + a.v_off + h * V;
    const float* k_at = rows + a.k_off + g * N;
    // four neighbouring columns from column i on of a row's `width`, zeros past it
    auto load4 = [&](const float* row, int i, int width) {
        if (aligned && i + 3 < width) return *reinterpret_cast<const ssd_f32x4*>(row + i);
        ssd_f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = i + j < width ? row[i + j] : 0.f;
        return v;
    };
    // (tokens past the chunk: its last again, under a weight of zero)
    ssd_f32x4 x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int e = tid + i * T, t = e / (COLS / 4), col = vt * COLS + 4 * (e % (COLS / 4));
        x[i] = load4(v_at + static_cast<size_t>(min(t, L - 1)) * a.qkv_stride, col, V);
    }
    for (int e0 = 0; e0 < SSD_CHUNK * Nq / 4; e0 += 4 * T) {
        ssd_f32x4 kv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = min(e0 + tid + i * T, SSD_CHUNK * Nq / 4 - 1), t = e / (Nq / 4);
            kv[i] = load4(k_at + static_cast<size_t>(min(t, L - 1)) * a.qkv_stride, 4 * (e - t * (Nq / 4)), N);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = e0 + tid + i * T;
            if (e >= SSD_CHUNK * Nq / 4) continue;
            const int t = e / (Nq / 4), n = 4 * (e - t * (Nq / 4));
            if (KIND == PL_SCAN_LIGHTNING) {
#pragma unroll
                for (int j = 0; j < 4; ++j) kv[i][j] = ssd_kv<KIND>(kv[i][j]);
            }
            *reinterpret_cast<ssd_f32x4*>(Ks + t * KP + n) = kv[i];
        }
    }
    if (wave == 0) {
        double b, dt;
        const double end = ssd_gates<KIND>(a, h, row0, L, lane, b, dt);
        if (KIND == PL_SCAN_MLSTM) {
            double top = dt;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) top = fmax(top, __shfl_xor(top, off, 64));
            weight[lane] = expf(static_cast<float>(dt - top));
            if (vt == 0 && lane == 0) {
                // (their sum: either may be hundreds where it is small, and rounded alone would leave its rounding in the state)
                sa.tops[2 * idx] = static_cast<float>(end + top);
                // the maximum that the request's first chunk starts from: the carry reads it here, not in the slot it writes
                if (c == 0) sa.tops[2 * idx + 1] = a.state[static_cast<size_t>(a.state_slots[s]) * a.state_stride + a.m_off + h * ((V + 63) / 64)];
            }
        } else {
            weight[lane] = expf(static_cast<float>(end - b)) * static_cast<float>(dt);  // (zero past the chunk's tokens)
        }
        if (vt == 0 && lane == 0) sa.ends[idx] = static_cast<float>(end);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int e = tid + i * T, t = e / (COLS / 4), col = 4 * (e % (COLS / 4));
        const float w = weight[t];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[i][j] = ssd_kv<KIND>(x[i][j]) * w;
        *reinterpret_cast<ssd_f32x4*>(Xs + t * XP + col) = x[i];
    }
    __syncthreads();
    if (KIND == PL_SCAN_MLSTM && vt == 0) {
        for (int n = tid; n < N; n += T) {
            float even = 0.f, odd = 0.f;
#pragma unroll 8
            for (int t = 0; t < SSD_CHUNK; t += 2) {
                even += weight[t] * Ks[t * KP + n];
                odd += weight[t + 1] * Ks[(t + 1) * KP + n];
            }
            sa.Uk[idx * N + n] = even + odd;
        }
    }
    float* U = sa.U + idx * N * V;
    const int v0 = 64 * (wave >> 2);                  // the wave's first column of the workgroup's
    if (vt * COLS + v0 >= V) return;
    const bool two = vt * COLS + v0 + 32 < V;         // whether its second 32 columns exist
    for (int n0 = (wave & 3) * 32; n0 < N; n0 += 128) {
        ssd_f32x16 da, db;
#pragma unroll
        for (int r = 0; r < 16; ++r) da[r] = db[r] = 0.f;
        const float* kr = Ks + half * KP + n0 + l32;
        const float* xr = Xs + half * XP + v0 + l32;
#pragma unroll
        for (int k = 0; k < SSD_CHUNK / 2; ++k) {
            const float kk = kr[2 * k * KP];
            da = ssd_mfma(kk, xr[2 * k * XP], da);
            if (two) db = ssd_mfma(kk, xr[2 * k * XP + 32], db);
        }
        const int va = vt * COLS + v0 + l32;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = n0 + 8 * (r >> 2) + 4 * half + (r & 3);
            if (row >= N) continue;
            if (va < V) U[static_cast<size_t>(row) * V + va] = da[r];
            if (va + 32 < V) U[static_cast<size_t>(row) * V + va + 32] = db[r];
        }
    }
}

// carry: the state before every chunk, and the request's state after its last; a thread an element, the sums of the next
// chunks on their way while the ones before are taken in.
template <int KIND>
__global__ __launch_bounds__(256) void ssd_carry_kernel(SsdArgs sa) {
    const ScanArgs& a = sa.a;
    const int N = a.D, V = a.V, H = a.H;
    const int h = blockIdx.y, s = blockIdx.z;
    const int slot = a.state_slots[s], count = a.q_len[s];
    if (slot < 0 || count < a.below) return;
    const int chunks = (count + SSD_CHUNK - 1) / SSD_CHUNK;
    const int e = blockIdx.x * 256 + threadIdx.x;
    // the normaliser's N values ride along in the threads behind the matrix's
    const bool element = e < N * V, of_n = KIND == PL_SCAN_MLSTM && e >= N * V && e < N * (V + 1);
    if (!element && !of_n) return;
    const size_t NV = static_cast<size_t>(N) * V;
    const int tiles = (V + 63) / 64;       // (n and m have a copy a tile of columns in the slot; all are equal)
    float* slot_state = a.state + static_cast<size_t>(slot) * a.state_stride;
    const int en = e - N * V;
    float* at = of_n ? slot_state + a.n_off + static_cast<size_t>(h) * tiles * N + en : slot_state + a.s_off + h * NV + e;
    const size_t first = static_cast<size_t>(ssd_chunk(a, s, 0)) * H + h;
    const float* __restrict__ U = of_n ? sa.Uk + first * N + en : sa.U + first * NV + e;
    float* __restrict__ Sin = of_n ? sa.nin + first * N + en : sa.Sin + first * NV + e;
    const float* __restrict__ ends = sa.ends + first;
    const size_t step = (of_n ? N : NV) * H;
    float S = *at;
    float m = KIND == PL_SCAN_MLSTM ? sa.tops[2 * first + 1] : 0.f;
    constexpr int AHEAD = 8;
    for (int c0 = 0; c0 < chunks; c0 += AHEAD) {
        float u[AHEAD], keep[AHEAD], most[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int c = min(c0 + i, chunks - 1);
            u[i] = U[c * step];
            keep[i] = ends[static_cast<size_t>(c) * H];
            most[i] = KIND == PL_SCAN_MLSTM ? sa.tops[2 * (first + static_cast<size_t>(c) * H)] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            if (c0 + i < chunks) {
                Sin[(c0 + i) * step] = S;
                if (KIND == PL_SCAN_MLSTM) {
                    if (c0 + i > 0 && e == 0) sa.tops[2 * (first + static_cast<size_t>(c0 + i) * H) + 1] = m;
                    const float kept = keep[i] + m;
                    m = fmaxf(kept, most[i]);
                    S = expf(kept - m) * S + expf(most[i] - m) * u[i];
                } else {
                    S = expf(keep[i]) * S + u[i];
                }
            }
    }
    *at = S;
    if (of_n)
        for (int t = 1; t < tiles; ++t) at[static_cast<size_t>(t) * N] = S;
    if (KIND == PL_SCAN_MLSTM && e < tiles) slot_state[a.m_off + h * tiles + e] = m;
}

// output: the read-outs of one chunk, head and tile of 64 columns.  Four waves; wave 2 ti + j owns the tokens 32 ti .. + 31 and, of the
// scores, the earlier tokens 32 j .. + 31, of the read-outs, the columns 32 j .. + 31.
// LDS: C [64][P], B [64][P] (behind the scores' barrier the weighted scores [64][68] lie in its place), b, step sizes, two numbers a token.
template <int KIND>
__global__ __launch_bounds__(256, 2) void ssd_output_kernel(SsdArgs sa, int aligned) {
    const ScanArgs& a = sa.a;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int N = a.D, V = a.V, H = a.H;
    const int tiles = (V + 63) / 64;
    const int c = blockIdx.x, h = blockIdx.y / tiles, vt = blockIdx.y % tiles, s = blockIdx.z;
    const int slot = a.state_slots[s], count = a.q_len[s];
    if (slot < 0 || count < a.below || c * SSD_CHUNK >= count) return;
    const int L = min(SSD_CHUNK, count - c * SSD_CHUNK), row0 = a.q_start[s] + c * SSD_CHUNK;
    const size_t idx = static_cast<size_t>(ssd_chunk(a, s, c)) * H + h;
    const int g = h / (H / a.G);
    const int Np = (N + 7) & ~7, P = Np + 4;
    constexpr int PA = SSD_CHUNK + 4;
    // mlstm: bd holds c_t, dtd the w_u - b_u, before_w what multiplies S_0^T q_t, below what the read-out is divided by
    double* bd = reinterpret_cast<double*>(lds);
    double* dtd = bd + SSD_CHUNK;
    float* before_w = lds + 4 * SSD_CHUNK;
    float* below = before_w + SSD_CHUNK;
    float* Cs = below + SSD_CHUNK;
    const float q_scale = 1.f / sqrtf(static_cast<float>(N));
    float* Bs = Cs + SSD_CHUNK * P;
    float* As = Bs;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int ti = wave >> 1, tj = wave & 1;
    const float* rows = a.qkv + static_cast<size_t>(row0) * a.qkv_stride;

    // ---- what waits for nothing: C and B into LDS, the columns of x into registers, the first rows of S_0 ----
    if (aligned) {
        const int quads = Np / 4;
        for (int e = tid; e < SSD_CHUNK * quads; e += 256) {
            const int t = e / quads, i = 4 * (e - t * quads);
            ssd_f32x4 cv = {0.f, 0.f, 0.f, 0.f}, bv = cv;
            if (t < L && i < N) {
                const float* row = rows + static_cast<size_t>(t) * a.qkv_stride + g * N + i;
                cv = *reinterpret_cast<const ssd_f32x4*>(row + a.q_off);
                bv = *reinterpret_cast<const ssd_f32x4*>(row + a.k_off);
            }
            if (KIND == PL_SCAN_LIGHTNING || KIND == PL_SCAN_MLSTM) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    cv[j] = ssd_q<KIND>(cv[j], q_scale);
                    bv[j] = ssd_kv<KIND>(bv[j]);
                }
            }
            *reinterpret_cast<ssd_f32x4*>(Cs + t * P + i) = cv;
            *reinterpret_cast<ssd_f32x4*>(Bs + t * P + i) = bv;
        }
    } else {
        for (int e = tid; e < SSD_CHUNK * Np; e += 256) {
            const int t = e / Np, i = e - t * Np;
            const bool in = t < L && i < N;
            const float* row = rows + static_cast<size_t>(in ? t : 0) * a.qkv_stride + g * N + (in ? i : 0);
            Cs[t * P + i] = in ? ssd_q<KIND>(row[a.q_off], q_scale) : 0.f;
            Bs[t * P + i] = in ? ssd_kv<KIND>(row[a.k_off]) : 0.f;
        }
    }
    const int v = vt * 64 + 32 * tj + l32, vc = min(v, V - 1);
    const bool columns = vt * 64 + 32 * tj < V && 32 * ti < L;      // (the same for the wave) it has read-outs to give
    float x[SSD_CHUNK / 2];                                           // x of token 8 q + 4 half + e in x[4 q + e]
#pragma unroll
    for (int k = 0; k < SSD_CHUNK / 2; ++k) {
        x[k] = 0.f;
        if (columns && (k < 16 || ti == 1)) {
            const int u = 8 * (k >> 2) + 4 * half + (k & 3);
            x[k] = rows[static_cast<size_t>(min(u, L - 1)) * a.qkv_stride + a.v_off + h * V + vc];
        }
    }
    const float* S0 = sa.Sin + idx * N * V + vc;
    auto ask = [&](int n0, float (&s0)[32]) {                         // rows n0 .. n0 + 63 of S_0, the wave's columns
#pragma unroll
        for (int k = 0; k < 32; ++k) {
            const int n = n0 + 8 * (k >> 2) + 4 * half + (k & 3);
            s0[k] = S0[static_cast<size_t>(min(n, N - 1)) * V];
        }
    };
    float s0[32];
    if (columns) ask(0, s0);
    if (wave == 0) {
        double b, dt;
        ssd_gates<KIND>(a, h, row0, L, lane, b, dt);
        if (KIND == PL_SCAN_MLSTM) {
            const double m0 = sa.tops[2 * idx + 1];
            double top = fmax(m0, dt);
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const double other = __shfl_up(top, off, 64);
                if (lane >= off) top = fmax(top, other);
            }
            before_w[lane] = expf(static_cast<float>(m0 - top));
            below[lane] = static_cast<float>(-(b + top));               // -m_t, until the weighted scores are there
            b = top;
        } else {
            before_w[lane] = expf(static_cast<float>(b));
        }
        bd[lane] = b;
        dtd[lane] = dt;
    }
    __syncthreads();

    // ---- the scores C_t . B_u of a tile of 32 by 32 (the tile of later tokens against earlier ones is all hidden) ----
    const bool scored = tj <= ti && 32 * ti < L;
    ssd_f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    if (scored) {
        const float* ca = Cs + (32 * ti + l32) * P + 4 * half;
        const float* ba = Bs + (32 * tj + l32) * P + 4 * half;
        for (int q = 0; q < Np; q += 8) {
            const ssd_f32x4 cv = *reinterpret_cast<const ssd_f32x4*>(ca + q), bv = *reinterpret_cast<const ssd_f32x4*>(ba + q);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = ssd_mfma(cv[e], bv[e], acc);
        }
        const int u = 32 * tj + l32;
        const double bu = bd[u], du = dtd[u];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int t = 32 * ti + 8 * (r >> 2) + 4 * half + (r & 3);
            const float w = KIND == PL_SCAN_MLSTM ? expf(static_cast<float>(du - bd[t]))
                                                  : expf(static_cast<float>(bd[t] - bu)) * static_cast<float>(du);
            acc[r] = (u <= t && t < L) ? acc[r] * w : 0.f;
        }
    }
    __syncthreads();                                                  // nobody reads B any more
    if (scored) {
#pragma unroll
        for (int r = 0; r < 16; ++r) As[(32 * ti + 8 * (r >> 2) + 4 * half + (r & 3)) * PA + 32 * tj + l32] = acc[r];
    }
    // ---- S_0^T C_t, times e^(b_t) ----
    // (in two chains, and the chunk's own part below in one of its own: half the roundings, each of its part's size.  Linear attention
    // with heads of 256, against 64 bits: 1.2e-7 to 1.5e-7; everything in one chain 1.5e-7 to 2.5e-7)
    ssd_f32x16 y, y2;
#pragma unroll
    for (int r = 0; r < 16; ++r) y[r] = y2[r] = 0.f;
    if (columns) {
        const float* ca = Cs + (32 * ti + l32) * P + 4 * half;
        for (int n0 = 0; n0 < Np; n0 += 64) {
            float now[32];
#pragma unroll
            for (int k = 0; k < 32; ++k) now[k] = s0[k];
            if (n0 + 64 < Np) ask(n0 + 64, s0);
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if (n0 + 8 * q < Np) {
                    const ssd_f32x4 cv = *reinterpret_cast<const ssd_f32x4*>(ca + n0 + 8 * q);   // (zeros past N)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (q % 2 == 0) y = ssd_mfma(cv[e], now[4 * q + e], y);
                        else y2 = ssd_mfma(cv[e], now[4 * q + e], y2);
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) y[r] = (y[r] + y2[r]) * before_w[32 * ti + 8 * (r >> 2) + 4 * half + (r & 3)];
    }
    __syncthreads();                                                  // the weighted scores are written
    if (KIND == PL_SCAN_MLSTM) {
        // n . q of a token, by four lanes: the weighted scores' sum and e^(m_0 - c_t) (n_0 . q_t)
        const int t = tid >> 2, part = tid & 3;
        float sum = 0.f, dot = 0.f;
        if (t < L) {
            const float* n0 = sa.nin + idx * N;
            for (int u = part; u <= t; u += 4) sum += As[t * PA + u];
            for (int i = part; i < N; i += 4) dot += n0[i] * Cs[t * P + i];
        }
        sum += before_w[t] * dot;
        sum += __shfl_xor(sum, 1, 64);
        sum += __shfl_xor(sum, 2, 64);
        if (part == 0) below[t] = 1.f / (fmaxf(fabsf(sum), expf(below[t])) + 1e-6f);
        __syncthreads();
    }
    if (!columns) return;
    // ---- the weighted scores times x, and D x ----
    if (KIND == PL_SCAN_LIGHTNING) {
#pragma unroll
        for (int k = 0; k < SSD_CHUNK / 2; ++k)
            if (k < 16 || ti == 1) x[k] = ssd_kv<KIND>(x[k]);
    }
    ssd_f32x16 own;
#pragma unroll
    for (int r = 0; r < 16; ++r) own[r] = 0.f;
    {
        const float* sc = As + (32 * ti + l32) * PA + 4 * half;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (q < 4 || ti == 1) {
                const ssd_f32x4 av = *reinterpret_cast<const ssd_f32x4*>(sc + 8 * q);
#pragma unroll
                for (int e = 0; e < 4; ++e) own = ssd_mfma(av[e], x[4 * q + e], own);
            }
        }
    }
    const float skip = KIND == PL_SCAN_SSD ? a.p3[h] : 0.f;
    float* out = a.out + static_cast<size_t>(row0) * (H * V) + h * V;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int t = 32 * ti + 8 * (r >> 2) + 4 * half + (r & 3);
        // (token t's own x is the one this lane holds in the same place of its half of the chunk)
        if (t >= L || v >= V) continue;
        float o = y[r] + own[r];
        if (KIND == PL_SCAN_SSD) o += skip * (ti == 0 ? x[r] : x[16 + r]);
        if (KIND == PL_SCAN_MLSTM) o *= below[t];
        out[static_cast<size_t>(t) * (H * V) + v] = o;
    }
}

// output_pair: the read-outs of one chunk, head and two tiles of 64 columns.  Eight waves; wave 4 ti + j owns the tokens 32 ti .. + 31 and, of the
// scores, the earlier tokens 32 j .. + 31 (j < 2), of the read-outs, the columns 32 j .. + 31.  Bound by its chain (rows, scores, what the
// state gives, what the chunk gives; three barriers), so waves without scores do the state's part meanwhile, and two workgroups share a
// compute unit.  Two tiles a workgroup make the scores once for both: 42 chunks of 8 heads of 128 by 128 44.6 us (50.8 with a tile a
// workgroup and one for each chunk that there might be), of 4 heads of 128 by 256 (matrix memory) 40.8 (49.3), 25 chunks of the first 27.6 (40.7);
// one tile a workgroup with the same order of loads 56.7, 52.9 and 30.8.
// LDS: C [64][P], B [64][P] (behind the scores' barrier the weighted scores [64][68] lie in its place), b, step sizes, two numbers a token.
template <int KIND>
__global__ __launch_bounds__(512, 4) void ssd_output_pair_kernel(SsdArgs sa, int seqs, int aligned) {
    const ScanArgs& a = sa.a;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int T = 512;
    const int N = a.D, V = a.V, H = a.H;
    const int tiles = (V + 128 - 1) / (128);
    const int h = blockIdx.y / tiles, vt = blockIdx.y % tiles;
    ChunkPlace place;
    if (!find_chunk(a, seqs, blockIdx.x, place)) return;
    const int c = place.c, s = place.s;
    const int L = min(SSD_CHUNK, place.count - c * SSD_CHUNK), row0 = place.first_row + c * SSD_CHUNK;
    const size_t idx = static_cast<size_t>(place.first_row / SSD_CHUNK + s + c) * H + h;
    const int g = h / (H / a.G);
    const int Np = (N + 7) & ~7, P = Np + 4;
    constexpr int PA = SSD_CHUNK + 4;
    // mlstm: bd holds c_t, dtd the w_u - b_u, before_w what multiplies S_0^T q_t, below what the read-out is divided by
    double* bd = reinterpret_cast<double*>(lds);
    double* dtd = bd + SSD_CHUNK;
    float* before_w = lds + 4 * SSD_CHUNK;
    float* below = before_w + SSD_CHUNK;
    float* Cs = below + SSD_CHUNK;
    const float q_scale = 1.f / sqrtf(static_cast<float>(N));
    float* Bs = Cs + SSD_CHUNK * P;
    float* As = Bs;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int ti = wave / (4), tj = wave % (4);
    const float* rows = a.qkv + static_cast<size_t>(row0) * a.qkv_stride;

    // ---- what waits for nothing: C and B into LDS, the first rows of S_0 into registers ----
    // (every load is unconditional, from an address that is valid in any case: one in a branch would be waited for alone)
    const int v = vt * 128 + 32 * tj + l32, vc = min(v, V - 1);
    const bool columns = vt * 128 + 32 * tj < V && 32 * ti < L;      // (the same for the wave) it has read-outs to give
    // (32-bit offsets from bases that are the same for the wave: an address a load would take two registers)
    const char* S0 = reinterpret_cast<const char*>(sa.Sin + idx * N * V);
    auto ask = [&](int n0, float (&s0)[16]) {                         // rows n0 .. n0 + 31 of S_0, the wave's columns
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int n = n0 + 8 * (k >> 2) + 4 * half + (k & 3);
            s0[k] = *reinterpret_cast<const float*>(S0 + 4u * static_cast<uint32_t>(min(n, N - 1) * V + vc));
        }
    };
    float s_even[16], s_odd[16];
    if (aligned) {
        const int quads = Np / 4, all = SSD_CHUNK * quads;
        for (int e0 = 0; e0 < all; e0 += 4 * T) {
            ssd_f32x4 cv[4], bv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int e = min(e0 + tid + k * T, all - 1), t = e / quads, i = min(4 * (e - t * quads), N - 4);
                const float* row = rows + static_cast<size_t>(min(t, L - 1)) * a.qkv_stride + g * N + i;
                cv[k] = *reinterpret_cast<const ssd_f32x4*>(row + a.q_off);
                bv[k] = *reinterpret_cast<const ssd_f32x4*>(row + a.k_off);
            }
            if (e0 == 0) {
                ask(0, s_even);
                ask(32, s_odd);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int e = e0 + tid + k * T, t = e / quads, i = 4 * (e - t * quads);
                if (e >= all) continue;
                const bool in = t < L && i < N;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    cv[k][j] = in ? ssd_q<KIND>(cv[k][j], q_scale) : 0.f;
                    bv[k][j] = in ? ssd_kv<KIND>(bv[k][j]) : 0.f;
                }
                *reinterpret_cast<ssd_f32x4*>(Cs + t * P + i) = cv[k];
                *reinterpret_cast<ssd_f32x4*>(Bs + t * P + i) = bv[k];
            }
        }
    } else {
        ask(0, s_even);
        ask(32, s_odd);
        for (int e = tid; e < SSD_CHUNK * Np; e += T) {
            const int t = e / Np, i = e - t * Np;
            const bool in = t < L && i < N;
            const float* row = rows + static_cast<size_t>(in ? t : 0) * a.qkv_stride + g * N + (in ? i : 0);
            Cs[t * P + i] = in ? ssd_q<KIND>(row[a.q_off], q_scale) : 0.f;
            Bs[t * P + i] = in ? ssd_kv<KIND>(row[a.k_off]) : 0.f;
        }
    }
    const char* x_at = reinterpret_cast<const char*>(rows + a.v_off + h * V);
    const int last_x = min(L, 32 * ti + 32) - 1;
    float x[SSD_CHUNK / 2];                                           // x of token 8 q + 4 half + e in x[4 q + e]
    auto ask_x = [&]() {                                              // (behind the scores, whose registers it takes)
#pragma unroll
        for (int k = 0; k < SSD_CHUNK / 2; ++k) {
            const int u = 8 * (k >> 2) + 4 * half + (k & 3);          // (the tokens behind its own a wave of the first half does not use)
            x[k] = *reinterpret_cast<const float*>(x_at + 4u * static_cast<uint32_t>(min(u, last_x) * a.qkv_stride + vc));
        }
    };
    if (wave == 0) {
        double b, dt;
        ssd_gates<KIND>(a, h, row0, L, lane, b, dt);
        if (KIND == PL_SCAN_MLSTM) {
            const double m0 = sa.tops[2 * idx + 1];
            double top = fmax(m0, dt);
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const double other = __shfl_up(top, off, 64);
                if (lane >= off) top = fmax(top, other);
            }
            before_w[lane] = expf(static_cast<float>(m0 - top));
            below[lane] = static_cast<float>(-(b + top));               // -m_t, until the weighted scores are there
            b = top;
        } else {
            before_w[lane] = expf(static_cast<float>(b));
        }
        bd[lane] = b;
        dtd[lane] = dt;
    }
    __syncthreads();

    // ---- the scores C_t . B_u of a tile of 32 by 32 (the tile of later tokens against earlier ones is all hidden) ----
    const bool scored = tj <= ti && 32 * ti < L;
    // (in two chains, and the chunk's own part below in one of its own: half the roundings, each of its part's size.  Linear attention
    // with heads of 256, against 64 bits: 1.2e-7 to 1.5e-7; everything in one chain 1.5e-7 to 2.5e-7)
    ssd_f32x16 y, y2;
#pragma unroll
    for (int r = 0; r < 16; ++r) y[r] = y2[r] = 0.f;
    auto state_part = [&]() {                                         // S_0^T C_t, times e^(b_t)
        const float* ca = Cs + (32 * ti + l32) * P + 4 * half;
        auto take = [&](int n0, const float (&s0)[16]) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (n0 + 8 * q < Np) {
                    const ssd_f32x4 cv = *reinterpret_cast<const ssd_f32x4*>(ca + n0 + 8 * q);   // (zeros past N)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (q % 2 == 0) y = ssd_mfma(cv[e], s0[4 * q + e], y);
                        else y2 = ssd_mfma(cv[e], s0[4 * q + e], y2);
                    }
                }
            }
        };
        for (int n0 = 0; n0 < Np; n0 += 64) {                         // (past N the last row again)
            take(n0, s_even);
            ask(n0 + 64, s_even);
            take(n0 + 32, s_odd);
            ask(n0 + 96, s_odd);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) y[r] = (y[r] + y2[r]) * before_w[32 * ti + 8 * (r >> 2) + 4 * half + (r & 3)];
    };
    if (columns && !scored) {
        ask_x();
        state_part();
    }
    ssd_f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    if (scored) {
        const float* ca = Cs + (32 * ti + l32) * P + 4 * half;
        const float* ba = Bs + (32 * tj + l32) * P + 4 * half;
        for (int q = 0; q < Np; q += 8) {
            const ssd_f32x4 cv = *reinterpret_cast<const ssd_f32x4*>(ca + q), bv = *reinterpret_cast<const ssd_f32x4*>(ba + q);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = ssd_mfma(cv[e], bv[e], acc);
        }
        const int u = 32 * tj + l32;
        const double bu = bd[u], du = dtd[u];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int t = 32 * ti + 8 * (r >> 2) + 4 * half + (r & 3);
            const float w = KIND == PL_SCAN_MLSTM ? expf(static_cast<float>(du - bd[t]))
                                                  : expf(static_cast<float>(bd[t] - bu)) * static_cast<float>(du);
            acc[r] = (u <= t && t < L) ? acc[r] * w : 0.f;
        }
    }
    __syncthreads();                                                  // nobody reads B any more
    if (scored) {
#pragma unroll
        for (int r = 0; r < 16; ++r) As[(32 * ti + 8 * (r >> 2) + 4 * half + (r & 3)) * PA + 32 * tj + l32] = acc[r];
    }
    if (columns && scored) {
        ask_x();
        state_part();
    }
    __syncthreads();                                                  // the weighted scores are written
    if (KIND == PL_SCAN_MLSTM) {
        // n . q of a token, by four lanes: the weighted scores' sum and e^(m_0 - c_t) (n_0 . q_t)
        const int t = tid >> 2, part = tid & 3;
        float sum = 0.f, dot = 0.f;
        if (t < L) {                                                  // (of a second tile's threads, none)
            const float* n0 = sa.nin + idx * N;
            for (int u = part; u <= t; u += 4) sum += As[t * PA + u];
            for (int i = part; i < N; i += 4) dot += n0[i] * Cs[t * P + i];
        }
        if (t < SSD_CHUNK) sum += before_w[t] * dot;
        sum += __shfl_xor(sum, 1, 64);
        sum += __shfl_xor(sum, 2, 64);
        if (part == 0 && t < SSD_CHUNK) below[t] = 1.f / (fmaxf(fabsf(sum), expf(below[t])) + 1e-6f);
        __syncthreads();
    }
    if (!columns) return;
    // ---- the weighted scores times x, and D x ----
    if (KIND == PL_SCAN_LIGHTNING) {
#pragma unroll
        for (int k = 0; k < SSD_CHUNK / 2; ++k)
            if (k < 16 || ti == 1) x[k] = ssd_kv<KIND>(x[k]);
    }
    ssd_f32x16 own;
#pragma unroll
    for (int r = 0; r < 16; ++r) own[r] = 0.f;
    {
        const float* sc = As + (32 * ti + l32) * PA + 4 * half;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (q < 4 || ti == 1) {
                const ssd_f32x4 av = *reinterpret_cast<const ssd_f32x4*>(sc + 8 * q);
#pragma unroll
                for (int e = 0; e < 4; ++e) own = ssd_mfma(av[e], x[4 * q + e], own);
            }
        }
    }
    const float skip = KIND == PL_SCAN_SSD ? a.p3[h] : 0.f;
    float* out = a.out + static_cast<size_t>(row0) * (H * V) + h * V;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int t = 32 * ti + 8 * (r >> 2) + 4 * half + (r & 3);
        // (token t's own x is the one this lane holds in the same place of its half of the chunk)
        if (t >= L || v >= V) continue;
        float o = y[r] + own[r];
        if (KIND == PL_SCAN_SSD) o += skip * (ti == 0 ? x[r] : x[16 + r]);
        if (KIND == PL_SCAN_MLSTM) o *= below[t];
        out[static_cast<size_t>(t) * (H * V) + v] = o;
    }
}

static bool ssd_aligned(const ScanArgs& a) {
    return ((a.qkv_stride | a.q_off | a.k_off | a.v_off | a.D) & 3) == 0 && reinterpret_cast<uintptr_t>(a.qkv) % 16 == 0;
}

// Whether ssd_step serves a state of V columns with slots `state_stride` floats apart (the scan kernel does otherwise).
extern "C" int pl_ssd_step_applies(int V, long state_stride) { return V % 4 == 0 && state_stride % 4 == 0 ? 1 : 0; }

// The requests that bring fewer than `below` tokens (0: all), token by token.
extern "C" int pl_ssd_step(const float* qkv, int qkv_stride, int q_off, int k_off, int v_off, const float* gates, int gates_stride,
                           int g_off, const float* a_log, const float* dt_bias, const float* skip, float* state, long state_stride,
                           float* out, const int* q_start, const int* q_len, const int* state_slots, int seqs, int H, int G, int N,
                           int V, int below, hipStream_t stream) {
    PL_REQUIRE(H > 0 && G > 0 && H % G == 0 && H <= 65535 && seqs >= 0 && seqs <= 65535, "ssd_step: %d heads over %d groups, %d requests", H, G, seqs);
    PL_REQUIRE(N > 0 && N <= 256 && V > 0 && pl_ssd_step_applies(V, state_stride) && reinterpret_cast<uintptr_t>(state) % 16 == 0 &&
               reinterpret_cast<uintptr_t>(out) % 16 == 0, "ssd_step: a state of %d by %d a head, slots of %ld floats", N, V, state_stride);
    PL_REQUIRE(gates != nullptr && a_log != nullptr && dt_bias != nullptr && skip != nullptr, "ssd_step: constants of the heads are missing");
    if (seqs == 0) return 0;
    const ScanArgs a{qkv, qkv_stride, q_off, k_off, v_off, gates, gates_stride, g_off, 0, a_log, dt_bias, skip, 0.f, state, state_stride,
                     0, 0, 0, out, q_start, q_len, state_slots, H, G, N, V, below};
    const dim3 grid(pl_ceil_div(V, 64), H, seqs);
    const bool aligned = ssd_aligned(a);
#define SSD_STEP(R)                                                              \
    do {                                                                         \
        if (aligned) ssd_step_kernel<R, true><<<grid, 256, 0, stream>>>(a);      \
        else ssd_step_kernel<R, false><<<grid, 256, 0, stream>>>(a);             \
    } while (0)
    if (N <= 16) SSD_STEP(1);
    else if (N <= 32) SSD_STEP(2);
    else if (N <= 64) SSD_STEP(4);
    else if (N <= 128) SSD_STEP(8);
    else SSD_STEP(16);
#undef SSD_STEP
    PL_CHECK_LAUNCH("ssd_step");
    return 0;
}

template <int KIND>
static int launch_chunk_pairs(const SsdArgs& sa, int rows, int seqs, int max_q_len, hipStream_t stream) {
    const ScanArgs& a = sa.a;
    const int N = a.D, V = a.V;
    const dim3 grid(chunk_bound(rows, max_q_len, seqs), a.H * pl_ceil_div(V, 128));
    const auto room = [](const void* kernel, size_t lds) {
        return lds <= 48 * 1024 ? hipSuccess : hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    };
    const size_t lds_s = SSD_CHUNK * (128 + pl_ceil_div(N, 32) * 32 + 2 * SSD_SUMMARY_PAD) * sizeof(float);
    hipError_t e = room(reinterpret_cast<const void*>(&ssd_summary_pair_kernel<KIND>), lds_s);
    PL_REQUIRE(e == hipSuccess, "ssd_chunked: %zu bytes of LDS refused: %s", lds_s, hipGetErrorString(e));
    const bool aligned = ssd_aligned(a);
    ssd_summary_pair_kernel<KIND><<<grid, 512, lds_s, stream>>>(sa, seqs, aligned && V % 4 == 0 ? 1 : 0);
    PL_CHECK_LAUNCH("ssd_chunked (summary)");
    ssd_carry_kernel<KIND><<<dim3(pl_ceil_div(N * (KIND == PL_SCAN_MLSTM ? V + 1 : V), 256), a.H, seqs), 256, 0, stream>>>(sa);
    PL_CHECK_LAUNCH("ssd_chunked (carry)");
    const int P = ((N + 7) & ~7) + 4;
    const size_t lds = (6 * SSD_CHUNK + SSD_CHUNK * static_cast<size_t>(P) + SSD_CHUNK * static_cast<size_t>(P > SSD_CHUNK + 4 ? P : SSD_CHUNK + 4)) * sizeof(float);
    e = room(reinterpret_cast<const void*>(&ssd_output_pair_kernel<KIND>), lds);
    PL_REQUIRE(e == hipSuccess, "ssd_chunked: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
    ssd_output_pair_kernel<KIND><<<grid, 512, lds, stream>>>(sa, seqs, aligned ? 1 : 0);
    PL_CHECK_LAUNCH("ssd_chunked (output)");
    return 0;
}

template <int KIND>
static int launch_chunks(const SsdArgs& sa, int rows, int seqs, int max_q_len, int dealt, hipStream_t stream) {
    const ScanArgs& a = sa.a;
    const int N = a.D, V = a.V, tiles = pl_ceil_div(V, 64);
    // (The same bits either way; which steps are dealt, and the times of both, is where the caller chooses.)
    if (dealt && V > 64) return launch_chunk_pairs<KIND>(sa, rows, seqs, max_q_len, stream);
    const dim3 grid(pl_ceil_div(max_q_len, SSD_CHUNK), a.H * tiles, seqs);
    ssd_summary_kernel<KIND><<<grid, 256, 0, stream>>>(sa);
    PL_CHECK_LAUNCH("ssd_chunked (summary)");
    ssd_carry_kernel<KIND><<<dim3(pl_ceil_div(N * (KIND == PL_SCAN_MLSTM ? V + 1 : V), 256), a.H, seqs), 256, 0, stream>>>(sa);
    PL_CHECK_LAUNCH("ssd_chunked (carry)");
    const int P = ((N + 7) & ~7) + 4;
    const size_t lds = (6 * SSD_CHUNK + SSD_CHUNK * static_cast<size_t>(P) + SSD_CHUNK * static_cast<size_t>(P > SSD_CHUNK + 4 ? P : SSD_CHUNK + 4)) * sizeof(float);
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&ssd_output_kernel<KIND>), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        PL_REQUIRE(e == hipSuccess, "ssd_chunked: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
    }
    ssd_output_kernel<KIND><<<grid, 256, lds, stream>>>(sa, ssd_aligned(a) ? 1 : 0);
    PL_CHECK_LAUNCH("ssd_chunked (output)");
    return 0;
}

// The requests that bring at least `from` tokens, in chunks of 64; `rows`: what the step's requests bring together at most.  U, Sin: room
// for (rows / 64 + requests + 1) chunks of H * N * V floats; ends: of H.  dealt: a workgroup for each chunk that the rows can hold, two tiles
// of 64 columns each where V has them, instead of the longest request's chunks for every request.
extern "C" int pl_ssd_chunked(const float* qkv, int qkv_stride, int q_off, int k_off, int v_off, const float* gates, int gates_stride,
                              int g_off, const float* a_log, const float* dt_bias, const float* skip, float* state, long state_stride,
                              float* out, const int* q_start, const int* q_len, const int* state_slots, int rows, int seqs, int max_q_len, int dealt, int H,
                              int G, int N, int V, int from, float* U, float* Sin, float* ends, hipStream_t stream) {
    PL_REQUIRE(H > 0 && G > 0 && H % G == 0 && N > 0 && N <= 256 && V > 0 && from >= 1, "ssd_chunked: %d heads of %d by %d over %d groups, from %d tokens", H, N, V, G, from);
    PL_REQUIRE(gates != nullptr && a_log != nullptr && dt_bias != nullptr && skip != nullptr && U != nullptr && Sin != nullptr && ends != nullptr,
               "ssd_chunked: constants of the heads or room for the chunks' sums are missing");
    const int tiles = pl_ceil_div(V, 64);
    PL_REQUIRE(static_cast<long long>(H) * tiles <= 65535 && seqs >= 0 && seqs <= 65535, "ssd_chunked: %d heads of %d columns, %d requests", H, V, seqs);
    if (seqs == 0 || max_q_len < from) return 0;
    const SsdArgs sa{{qkv, qkv_stride, q_off, k_off, v_off, gates, gates_stride, g_off, 0, a_log, dt_bias, skip, 0.f, state, state_stride,
                      0, 0, 0, out, q_start, q_len, state_slots, H, G, N, V, from}, U, Sin, ends, nullptr, nullptr, nullptr};
    return launch_chunks<PL_SCAN_SSD>(sa, rows, seqs, max_q_len, dealt, stream);
}

// Retention: S = decay S + k v^T, o = S^T q, q and k turning with their positions (HalfTurn; freq null: not at all).
// The rows of q and k in `rows` turn in place.
extern "C" int pl_retention_turn(float* rows, int stride, int q_off, int k_off, int n, int H, int N, const float* freq, int dims,
                                 float amplitude, float k_scale, const int* positions, hipStream_t stream) {
    PL_REQUIRE(n >= 0 && H > 0 && N > 0 && N <= 256 && dims >= 0 && dims % 2 == 0 && dims <= N && (dims == 0 || freq != nullptr) && positions != nullptr,
               "retention_turn: %d heads of %d values, %d of which turn", H, N, dims);
    PL_REQUIRE(q_off >= 0 && k_off >= 0 && q_off + H * N <= stride && k_off + H * N <= stride, "retention_turn: q and k at %d and %d of rows of %d", q_off, k_off, stride);
    if (n == 0) return 0;
    retention_turn_kernel<<<n, 256, 0, stream>>>(rows, stride, q_off, k_off, H, N, HalfTurn{freq, positions, dims, amplitude, k_scale});
    PL_CHECK_LAUNCH("retention_turn");
    return 0;
}

// The requests that bring fewer than `below` tokens (0: all), token by token.  turns: q and k of these rows have not been turned.
extern "C" int pl_retention_step(const float* qkv, int qkv_stride, int q_off, int k_off, int v_off, const float* decay, const float* freq,
                                 int dims, float amplitude, float k_scale, int turns, const int* positions, float* state, long state_stride,
                                 float* out, const int* q_start, const int* q_len, const int* state_slots, int seqs, int H, int N, int V,
                                 int below, hipStream_t stream) {
    PL_REQUIRE(H > 0 && H <= 65535 && seqs >= 0 && seqs <= 65535, "retention_step: %d heads, %d requests", H, seqs);
    PL_REQUIRE(N > 0 && N <= 256 && V > 0 && pl_ssd_step_applies(V, state_stride) && reinterpret_cast<uintptr_t>(state) % 16 == 0 &&
               reinterpret_cast<uintptr_t>(out) % 16 == 0, "retention_step: a state of %d by %d a head, slots of %ld floats", N, V, state_stride);
    PL_REQUIRE(decay != nullptr && positions != nullptr && dims >= 0 && dims % 2 == 0 && dims <= N && (dims == 0 || freq != nullptr),
               "retention_step: %d of %d values turn", dims, N);
    if (seqs == 0) return 0;
    const ScanArgs a{qkv, qkv_stride, q_off, k_off, v_off, nullptr, 0, 0, 0, decay, nullptr, nullptr, 0.f, state, state_stride,
                     0, 0, 0, out, q_start, q_len, state_slots, H, H, N, V, below};
    const HalfTurn turn{freq, positions, dims, amplitude, k_scale};
    const dim3 grid(pl_ceil_div(V, 64), H, seqs);
    if (N <= 16) retention_step_kernel<1><<<grid, 256, 0, stream>>>(a, turn, turns);
    else if (N <= 32) retention_step_kernel<2><<<grid, 256, 0, stream>>>(a, turn, turns);
    else if (N <= 64) retention_step_kernel<4><<<grid, 256, 0, stream>>>(a, turn, turns);
    else if (N <= 128) retention_step_kernel<8><<<grid, 256, 0, stream>>>(a, turn, turns);
    else retention_step_kernel<16><<<grid, 256, 0, stream>>>(a, turn, turns);
    PL_CHECK_LAUNCH("retention_step");
    return 0;
}

// The requests that bring at least `from` tokens, in chunks of 64, q and k turned already; decays above zero.  Room as in pl_ssd_chunked.
extern "C" int pl_retention_chunked(const float* qkv, int qkv_stride, int q_off, int k_off, int v_off, const float* decay, float* state,
                                    long state_stride, float* out, const int* q_start, const int* q_len, const int* state_slots, int rows, int seqs,
                                    int max_q_len, int dealt, int H, int N, int V, int from, float* U, float* Sin, float* ends, hipStream_t stream) {
    PL_REQUIRE(H > 0 && N > 0 && N <= 256 && V > 0 && from >= 1, "retention_chunked: %d heads of %d by %d, from %d tokens", H, N, V, from);
    PL_REQUIRE(decay != nullptr && U != nullptr && Sin != nullptr && ends != nullptr, "retention_chunked: the decays or room for the chunks' sums are missing");
    PL_REQUIRE(static_cast<long long>(H) * pl_ceil_div(V, 64) <= 65535 && seqs >= 0 && seqs <= 65535, "retention_chunked: %d heads of %d columns, %d requests", H, V, seqs);
    if (seqs == 0 || max_q_len < from) return 0;
    const SsdArgs sa{{qkv, qkv_stride, q_off, k_off, v_off, nullptr, 0, 0, 0, decay, nullptr, nullptr, 0.f, state, state_stride,
                      0, 0, 0, out, q_start, q_len, state_slots, H, H, N, V, from}, U, Sin, ends, nullptr, nullptr, nullptr};
    return launch_chunks<PL_SCAN_RETENTION>(sa, rows, seqs, max_q_len, dealt, stream);
}

// Linear attention with a fixed decay a head and silu on q, k and v (kind lightning), and the matrix memory with exponential gates
// (kind mlstm): the requests of the step that bring at least `from` tokens; the others are the token-by-token kernel's.
// U, Sin: room for (rows / 64 + requests) chunks of H * D * V floats; Uk, nin: of H * D (mlstm); scal: of H * 4.
extern "C" int pl_recurrent_chunked(int kind, const float* qkv, int qkv_stride, int q_off, int k_off, int v_off,
                                    const float* gates, int gates_stride, int g1_off, int g2_off,
                                    const float* p1, const float* p2, float cap,
                                    float* state, long state_stride, int s_off, int n_off, int m_off,
                                    float* out, const int* q_start, const int* q_len, const int* state_slots,
                                    int rows, int seqs, int max_q_len, int dealt, int H, int D, int V, int from, int chunks,
                                    float* U, float* Uk, float* Sin, float* nin, float* scal, hipStream_t stream) {
    PL_REQUIRE(kind == PL_SCAN_LIGHTNING || kind == PL_SCAN_MLSTM, "recurrent_chunked: kind %d", kind);
    PL_REQUIRE(H > 0 && D > 0 && D <= 256 && V > 0 && from >= 1, "recurrent_chunked: %d heads of %d by %d, from %d tokens", H, D, V, from);
    PL_REQUIRE(p1 != nullptr && (kind == PL_SCAN_LIGHTNING || (gates != nullptr && p2 != nullptr && cap > 0.f)),
               "recurrent_chunked: the gates of kind %d are missing", kind);
    PL_REQUIRE(U != nullptr && Sin != nullptr && scal != nullptr && (kind == PL_SCAN_LIGHTNING || (Uk != nullptr && nin != nullptr)),
               "recurrent_chunked: no room for the chunks' sums");
    PL_REQUIRE(static_cast<long long>(H) * pl_ceil_div(V, 64) <= 65535 && seqs <= 65535, "recurrent_chunked: %d heads of %d columns, %d requests", H, V, seqs);
    if (seqs == 0 || max_q_len < from) return 0;
    const SsdArgs sa{{qkv, qkv_stride, q_off, k_off, v_off, gates, gates_stride, g1_off, g2_off, p1, p2, nullptr, cap, state, state_stride,
                      s_off, n_off, m_off, out, q_start, q_len, state_slots, H, H, D, V, from},
                     U, Sin, scal, Uk, nin, scal + static_cast<size_t>(chunks) * H};
    return kind == PL_SCAN_LIGHTNING ? launch_chunks<PL_SCAN_LIGHTNING>(sa, rows, seqs, max_q_len, dealt, stream)
                                     : launch_chunks<PL_SCAN_MLSTM>(sa, rows, seqs, max_q_len, dealt, stream);
}
