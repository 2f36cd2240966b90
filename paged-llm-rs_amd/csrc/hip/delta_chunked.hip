// Prompt portions through the gated delta rule in chunks of 64 tokens.  For one head, with decays g_t,
// G_t = g_1 ... g_t inside a chunk, and S_0 the state before the chunk, the rule
//     S_t = g_t S_(t-1) + k_t u_t^T ,   u_t = beta_t (v_t - g_t S_(t-1)^T k_t)
// unrolls to  S_t = G_t S_0 + sum_{s<=t} (G_t / G_s) k_s u_s^T , and the u of a chunk solve
//     (I + M) U = R ,  M[t][s] = beta_t (G_t / G_s) (k_t . k_s) for s < t ,  R_t = beta_t (v_t - G_t S_0^T k_t) .
// `prepare` (every chunk and head at once) makes k and q unit vectors, and computes T = (I + M)^-1 and
// Aq[t][s] = (G_t / G_s) (q_t . k_s) for s <= t.  `walk` (one workgroup for a request, a head and 16 columns of the
// state) then goes through the chunks in order:
//     R = beta (V - G K S) ;  U = T R ;  O = G Q S + Aq U ;  S = G_L S + (K weighted by G_L / G_s)^T U .
// Operands and sums are 32-bit, the products on the matrix cores (v_mfma_f32_16x16x4_f32); the sums of log decays are 64-bit.
//
// The instruction, D[16 x 16] += A[16 x 4] B[4 x 16]: lane l gives A[l % 16][l / 16] and B[l / 16][l % 16] and holds, in
// register t, D[4 (l / 16) + t][l % 16].  With r = l % 16, c = l / 16 everything here takes 16 of the inner index at a time as four
// instructions, the t-th of which multiplies the places 4 c + t: an operand whose rows lie along the inner index is four
// neighbouring values a lane, and a result is a right operand of the next product as it stands.
#include "recurrent.hpp"

typedef float dl_f32x4 __attribute__((ext_vector_type(4)));

#define DL_C 64                 // tokens of a chunk
#define DL_T 68                 // values from one row of a 64 x 64 matrix in LDS to the next

struct DeltaArgs {
    ScanArgs a;
    float* Kn;       // [chunks, H, 64, Dp]  k as unit vectors, rows of Dp = D rounded up to 64, zeros behind D
    float* Qn;       // [chunks, H, 64, Dp]  q as unit vectors times D^-1/2
    float* Kw;       // [chunks, H, Dp, 64]  k weighted by G_L / G_t, a token a column
    float* Tm;       // [chunks, H, 64, 64]  (I + M)^-1, the blocks of 16 x 16 on and below the diagonal
    float* Aq;       // [chunks, H, 64, 64]  the same blocks
    float* scal;     // [chunks, H, 2, 64]   G_t; beta_t
};

__device__ __forceinline__ int delta_chunk_number(const ScanArgs& a, int s, int c) { return a.q_start[s] / DL_C + s + c; }

__device__ __forceinline__ dl_f32x4 dl_read4(const float* p) { return *reinterpret_cast<const dl_f32x4*>(p); }

// D += A B over 16 of the inner index.
__device__ __forceinline__ dl_f32x4 dl_multiply(const dl_f32x4& a, const dl_f32x4& b, dl_f32x4 d) {
#pragma unroll
    for (int t = 0; t < 4; ++t) d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], d, 0, 0, 0);
    return d;
}

// A workgroup of four waves a chunk and head; wave w owns the tokens 16 w .. + 15.  The two products of 64 x 64 x D take some
// 3 us, the inverse another 2: its diagonal blocks by forward substitution, a column a lane, the others as products,
// T_ij = -T_ii sum_k M_ik T_kj, a block row after the other.  (On the vector units with the whole inverse a column a thread: 111 us for
// two prompts of 1,500 tokens and eight heads of 128.)
__global__ __launch_bounds__(256) void delta_prepare_kernel(DeltaArgs da, int Dp, int seqs) {
    const ScanArgs& a = da.a;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int D = a.D, H = a.H;
    const int h = blockIdx.y;
    ChunkPlace place;
    if (seqs > 0) {
        if (!find_chunk(a, seqs, blockIdx.x, place)) return;
    } else {
        place = {static_cast<int>(blockIdx.z), static_cast<int>(blockIdx.x), a.q_len[blockIdx.z], a.q_start[blockIdx.z]};
        if (a.state_slots[place.s] < 0 || place.count < a.below || place.c * DL_C >= place.count) return;
    }
    const int c_at = place.c, s = place.s, n = place.count;
    const int L = min(DL_C, n - c_at * DL_C), row0 = place.first_row + c_at * DL_C;
    const int g = h / (H / a.G);
    const size_t idx = static_cast<size_t>(place.first_row / DL_C + s + c_at) * H + h;
    const int P = Dp + 4;
    double* bd = reinterpret_cast<double*>(lds);        // [64] b_t, the sum of log decays
    double* nrm = bd + DL_C;                            // [2][64]
    float* be = lds + 6 * DL_C;                         // [64] beta_t
    float* qs = be + DL_C;                              // [64][P]
    float* ks = qs + DL_C * P;                          // [64][P]
    float* M = qs;                                      // [64][DL_T], where q lay
    float* T = ks;                                      // [64][DL_T], where k lay
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, c = lane >> 4;
    for (int e = tid; e < DL_C * Dp; e += 256) {
        const int t = e / Dp, i = e - t * Dp;
        float q = 0.f, k = 0.f;
        if (t < L && i < D) {
            const float* row = a.qkv + static_cast<size_t>(row0 + t) * a.qkv_stride;
            q = row[a.q_off + g * D + i];
            k = row[a.k_off + g * D + i];
        }
        qs[t * P + i] = q;
        ks[t * P + i] = k;
    }
    if (wave == 0) {
        float beta = 0.f;
        double sum = 0.0;
        if (lane < L) {
            const float* row = a.gates + static_cast<size_t>(row0 + lane) * a.gates_stride;
            beta = sigmoid_f(row[a.g1_off + h]);
            sum = -static_cast<double>(expf(a.p1[h])) * static_cast<double>(softplus_f(row[a.g2_off + h] + a.p2[h]));
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double other = __shfl_up(sum, off, 64);
            if (lane >= off) sum += other;
        }
        bd[lane] = sum;
        be[lane] = beta;
        da.scal[idx * 2 * DL_C + lane] = expf(static_cast<float>(sum));
        da.scal[idx * 2 * DL_C + DL_C + lane] = beta;
    }
    __syncthreads();
    {
        // four lanes a row of q and one of k
        const int t = tid >> 2, part = tid & 3;
        // (a norm's rounding would stand in all of its row: 64-bit sums)
        double qq = 0.0, kk = 0.0;
        for (int i = part; i < Dp; i += 4) {
            const double q = qs[t * P + i], k = ks[t * P + i];
            qq += q * q;
            kk += k * k;
        }
        qq += __shfl_xor(qq, 1, 64);
        kk += __shfl_xor(kk, 1, 64);
        qq += __shfl_xor(qq, 2, 64);
        kk += __shfl_xor(kk, 2, 64);
        if (part == 0) {
            nrm[t] = 1.0 / sqrt((qq + 1e-6) * D);
            nrm[DL_C + t] = 1.0 / sqrt(kk + 1e-6);
        }
    }
    __syncthreads();
    const double end = bd[L - 1];
    float* Kn = da.Kn + idx * DL_C * Dp;
    float* Qn = da.Qn + idx * DL_C * Dp;
    for (int e = tid; e < DL_C * Dp; e += 256) {
        const int t = e / Dp, i = e - t * Dp;
        const float q = static_cast<float>(qs[t * P + i] * nrm[t]), k = static_cast<float>(ks[t * P + i] * nrm[DL_C + t]);
        qs[t * P + i] = q;
        ks[t * P + i] = k;
        Qn[e] = q;
        Kn[e] = k;
    }
    __syncthreads();
    float* Kw = da.Kw + idx * DL_C * Dp;
    {
        const float w = lane < L ? expf(static_cast<float>(end - bd[lane])) : 0.f;
        for (int i = wave; i < Dp; i += 4) Kw[i * DL_C + lane] = ks[lane * P + i] * w;
    }
    // k_t . k_u and q_t . k_u for the wave's tokens t and the blocks of tokens u up to its own
    dl_f32x4 kk[4], qk[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) kk[j] = qk[j] = dl_f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < Dp; i += 64) {                  // (64 of D a chain, the chains added)
        dl_f32x4 kc[4], qc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) kc[j] = qc[j] = dl_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int at = i + 16 * e + 4 * c;
            const dl_f32x4 ka = dl_read4(ks + (16 * wave + r) * P + at), qa = dl_read4(qs + (16 * wave + r) * P + at);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j <= wave) {
                    const dl_f32x4 kb = dl_read4(ks + (16 * j + r) * P + at);
                    kc[j] = dl_multiply(ka, kb, kc[j]);
                    qc[j] = dl_multiply(qa, kb, qc[j]);
                }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            kk[j] += kc[j];
            qk[j] += qc[j];
        }
    }
    __syncthreads();                                    // q and k are done with
    float* Aq = da.Aq + idx * DL_C * DL_C;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (j <= wave) {
            const int u = 16 * j + r;
            const double bu = bd[u];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * wave + 4 * c + e;
                const float w = (u <= t && t < L) ? expf(static_cast<float>(bd[t] - bu)) : 0.f;
                M[t * DL_T + u] = u < t ? be[t] * w * kk[j][e] : 0.f;
                Aq[t * DL_C + u] = w * qk[j][e];
            }
        }
    __syncthreads();
    // the diagonal blocks: T[t][j] = [t == j] - sum_{s < t} M[t][s] T[s][j], a column a lane
    if (lane < 16) {
        float col[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            float val = t == lane ? 1.f : 0.f;
#pragma unroll
            for (int u = 0; u < t; ++u) val -= M[(16 * wave + t) * DL_T + 16 * wave + u] * col[u];
            col[t] = val;
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) T[(16 * wave + t) * DL_T + 16 * wave + lane] = col[t];
    }
    __syncthreads();
#pragma unroll
    for (int i = 1; i < 4; ++i) {
        if (wave < i) {                                 // block (i, wave)
            dl_f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < i; ++k)
                if (k >= wave) {
                    dl_f32x4 b;
#pragma unroll
                    for (int t = 0; t < 4; ++t) b[t] = T[(16 * k + 4 * c + t) * DL_T + 16 * wave + r];
                    x = dl_multiply(dl_read4(M + (16 * i + r) * DL_T + 16 * k + 4 * c), b, x);
                }
            dl_f32x4 y = {0.f, 0.f, 0.f, 0.f};
            y = dl_multiply(dl_read4(T + (16 * i + r) * DL_T + 16 * i + 4 * c), x, y);
#pragma unroll
            for (int t = 0; t < 4; ++t) T[(16 * i + 4 * c + t) * DL_T + 16 * wave + r] = -y[t];
        }
        __syncthreads();
    }
    float* Tm = da.Tm + idx * DL_C * DL_C;
    for (int e = tid; e < DL_C * DL_C; e += 256) {
        const int t = e / DL_C, u = e % DL_C;
        if (u / 16 <= t / 16) Tm[e] = T[t * DL_T + u];
    }
}

// One workgroup of four waves: a request, a head, 16 columns of the state; the chunks in order.  Wave w owns the tokens 16 w .. + 15 of a
// chunk and the rows 16 RT w .. of the state, which stay in its registers; what it needs of a chunk (its rows of K, Q, T and
// Aq, its rows of the weighted K, its values) goes from memory straight into registers in the instruction's layout, and is
// asked for again, for the next chunk, as soon as it is multiplied.  What the waves give each other (S, R and U, a column of the state
// a row in LDS) costs a barrier each.  A chunk takes its 128 matrix instructions a wave (1.7 us for heads of 128) and three barriers.  (With tiles of
// 8 columns on the vector units and every operand through LDS: 313 us for two prompts of 1,500 tokens and eight heads of 128.)
template <int RT>
__global__ __launch_bounds__(256) void delta_walk_kernel(DeltaArgs da) {
    constexpr int Dp = 64 * RT, PS = Dp + 4, KT = 4 * RT;           // KT: stretches of 16 rows of the state
    __shared__ __attribute__((aligned(16))) float Ss[16 * PS], Rs[16 * DL_T], Us[16 * DL_T];       // [column][row of S; token]
    const ScanArgs& a = da.a;
    const int D = a.D, V = a.V, H = a.H;
    const int h = blockIdx.x % H, s = blockIdx.x / H;
    const int slot = a.state_slots[s], n = a.q_len[s];
    if (slot < 0 || n < a.below) return;
    const int chunks = (n + DL_C - 1) / DL_C, start = a.q_start[s];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, c = lane >> 4;
    const int v = blockIdx.y * 16 + r;
    const bool owns = v < V;
    float* Sg = a.state + static_cast<size_t>(slot) * a.state_stride + a.s_off + static_cast<size_t>(h) * D * V + (owns ? v : 0);
    const size_t first = static_cast<size_t>(delta_chunk_number(a, s, 0)) * H + h;

    dl_f32x4 S[RT];                                                 // rows 16 (RT wave + i) + 4 c + t, column r
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int d = 16 * (RT * wave + i) + 4 * c + t;
            S[i][t] = owns && d < D ? Sg[static_cast<size_t>(d) * V] : 0.f;
        }

    dl_f32x4 K[KT], Q[KT], Kw[RT][4], T[4], A[4], value, decay, beta;
    float gl;
    const dl_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    auto ask_rows = [&](int ch) {                                   // (past the last chunk: the last one again)
        const size_t at = (first + static_cast<size_t>(min(ch, chunks - 1)) * H) * DL_C * Dp + (16 * wave + r) * Dp + 4 * c;
#pragma unroll
        for (int i = 0; i < KT; ++i) {
            K[i] = dl_read4(da.Kn + at + 16 * i);
            Q[i] = dl_read4(da.Qn + at + 16 * i);
        }
    };
    auto ask_tokens = [&](int ch) {
        const int now = min(ch, chunks - 1), L = min(DL_C, n - now * DL_C), row0 = start + now * DL_C;
        const size_t idx = first + static_cast<size_t>(now) * H;
        const float* scal = da.scal + idx * 2 * DL_C;
        decay = dl_read4(scal + 16 * wave + 4 * c);
        beta = dl_read4(scal + DL_C + 16 * wave + 4 * c);
        gl = scal[L - 1];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int row = 16 * wave + 4 * c + t;
            value[t] = a.qkv[static_cast<size_t>(row0 + min(row, L - 1)) * a.qkv_stride + a.v_off + h * V + (owns ? v : 0)];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const size_t at = idx * DL_C * DL_C + (16 * wave + r) * DL_C + 16 * min(j, wave) + 4 * c;
            T[j] = dl_read4(da.Tm + at);
        }
    };
    auto ask_mixed = [&](int ch) {
        const size_t idx = first + static_cast<size_t>(min(ch, chunks - 1)) * H;
#pragma unroll
        for (int j = 0; j < 4; ++j) A[j] = dl_read4(da.Aq + idx * DL_C * DL_C + (16 * wave + r) * DL_C + 16 * min(j, wave) + 4 * c);
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) Kw[i][j] = dl_read4(da.Kw + idx * DL_C * Dp + (16 * (RT * wave + i) + r) * DL_C + 16 * j + 4 * c);
    };
    ask_rows(0);
    ask_tokens(0);
    ask_mixed(0);
#pragma unroll
    for (int i = 0; i < RT; ++i) *reinterpret_cast<dl_f32x4*>(Ss + r * PS + 16 * (RT * wave + i) + 4 * c) = S[i];
    __syncthreads();
    for (int ch = 0; ch < chunks; ++ch) {
        const int L = min(DL_C, n - ch * DL_C), row0 = start + ch * DL_C;
        // K S and Q S of the wave's tokens
        dl_f32x4 ks[2] = {zero, zero}, qs[2] = {zero, zero};        // (two chains each: half the roundings of one)
#pragma unroll
        for (int i = 0; i < KT; ++i) {
            const dl_f32x4 b = dl_read4(Ss + r * PS + 16 * i + 4 * c);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                ks[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(K[i][t], b[t], ks[i & 1], 0, 0, 0);
                qs[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(Q[i][t], b[t], qs[i & 1], 0, 0, 0);
            }
        }
        const dl_f32x4 ksum = ks[0] + ks[1], qsum = qs[0] + qs[1];
        ask_rows(ch + 1);
        __builtin_amdgcn_sched_barrier(0);
        dl_f32x4 R;
#pragma unroll
        for (int t = 0; t < 4; ++t) R[t] = beta[t] * ((owns && 16 * wave + 4 * c + t < L ? value[t] : 0.f) - decay[t] * ksum[t]);
        *reinterpret_cast<dl_f32x4*>(Rs + r * DL_T + 16 * wave + 4 * c) = R;
        __syncthreads();
        dl_f32x4 U = zero;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j <= wave) U = dl_multiply(T[j], dl_read4(Rs + r * DL_T + 16 * j + 4 * c), U);
        const dl_f32x4 before = decay * qsum;
        const float keep = gl;
        ask_tokens(ch + 1);
        __builtin_amdgcn_sched_barrier(0);
        *reinterpret_cast<dl_f32x4*>(Us + r * DL_T + 16 * wave + 4 * c) = U;
        __syncthreads();
        // (the chunk's own part is summed by itself: its roundings are of its own size, not of the state's)
        dl_f32x4 O = zero, grown[RT];
#pragma unroll
        for (int i = 0; i < RT; ++i) grown[i] = zero;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const dl_f32x4 b = dl_read4(Us + r * DL_T + 16 * j + 4 * c);
            if (j <= wave) O = dl_multiply(A[j], b, O);
#pragma unroll
            for (int i = 0; i < RT; ++i) grown[i] = dl_multiply(Kw[i][j], b, grown[i]);
        }
        O += before;
#pragma unroll
        for (int i = 0; i < RT; ++i) S[i] = keep * S[i] + grown[i];
        ask_mixed(ch + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < RT; ++i) *reinterpret_cast<dl_f32x4*>(Ss + r * PS + 16 * (RT * wave + i) + 4 * c) = S[i];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int row = 16 * wave + 4 * c + t;
            if (owns && row < L) a.out[static_cast<size_t>(row0 + row) * (H * V) + h * V + v] = O[t];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int d = 16 * (RT * wave + i) + 4 * c + t;
            if (owns && d < D) Sg[static_cast<size_t>(d) * V] = S[i][t];
        }
}

static int launch_delta(const DeltaArgs& da, int rows, int seqs, int max_q_len, int dealt, hipStream_t stream) {
    const ScanArgs& a = da.a;
    const int Dp = pl_ceil_div(a.D, 64) * 64, P = Dp + 4;
    const size_t lds_p = (7 * DL_C + 2 * static_cast<size_t>(DL_C) * (P > DL_T ? P : DL_T)) * sizeof(float);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_prepare_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       static_cast<int>(lds_p));
    PL_REQUIRE(e == hipSuccess, "delta_chunked: %zu bytes of LDS refused: %s", lds_p, hipGetErrorString(e));
    // (dealt: a workgroup for each chunk that the rows can hold; otherwise the longest's chunks for every request)
    if (dealt) delta_prepare_kernel<<<dim3(chunk_bound(rows, max_q_len, seqs), a.H), 256, lds_p, stream>>>(da, Dp, seqs);
    else delta_prepare_kernel<<<dim3(pl_ceil_div(max_q_len, DL_C), a.H, seqs), 256, lds_p, stream>>>(da, Dp, 0);
    PL_CHECK_LAUNCH("delta_chunked (prepare)");
    // the workgroups of one head read the same chunks: with heads and requests along x they share a chiplet's cache wherever those are a
    // multiple of the eight chiplets
    const dim3 grid(static_cast<unsigned>(a.H) * seqs, pl_ceil_div(a.V, 16));
    if (Dp == 64) delta_walk_kernel<1><<<grid, 256, 0, stream>>>(da);
    else if (Dp == 128) delta_walk_kernel<2><<<grid, 256, 0, stream>>>(da);
    else if (Dp == 192) delta_walk_kernel<3><<<grid, 256, 0, stream>>>(da);
    else delta_walk_kernel<4><<<grid, 256, 0, stream>>>(da);
    PL_CHECK_LAUNCH("delta_chunked (walk)");
    return 0;
}

// The requests of the step that bring at least `from` tokens.  Kn, Qn, Kw: room for (rows / 64 + requests) chunks of
// H * 64 * (D rounded up to 64) floats; Tm, Aq: of H * 64 * 64; scal: of H * 2 * 64.
extern "C" int pl_delta_chunked(const float* qkv, int qkv_stride, int q_off, int k_off, int v_off,
                                const float* gates, int gates_stride, int g1_off, int g2_off,
                                const float* a_log, const float* dt_bias,
                                float* state, long state_stride, float* out,
                                const int* q_start, const int* q_len, const int* state_slots,
                                int rows, int seqs, int max_q_len, int dealt, int H, int G, int D, int V, int from,
                                float* Kn, float* Qn, float* Kw, float* Tm, float* Aq, float* scal, hipStream_t stream) {
    PL_REQUIRE(H > 0 && G > 0 && H % G == 0 && D > 0 && D <= 256 && V > 0 && from >= 1,
               "delta_chunked: %d heads over %d of q and k, %d by %d, from %d tokens", H, G, D, V, from);
    PL_REQUIRE(gates != nullptr && a_log != nullptr && dt_bias != nullptr, "delta_chunked: the gates are missing");
    PL_REQUIRE(Kn != nullptr && Qn != nullptr && Kw != nullptr && Tm != nullptr && Aq != nullptr && scal != nullptr, "delta_chunked: no room for the chunks");
    PL_REQUIRE(seqs >= 0 && seqs <= 65535 && H <= 65535, "delta_chunked: %d requests, %d heads", seqs, H);
    PL_REQUIRE(static_cast<long long>(seqs) * H <= 0x7fffffffLL && V <= 16 * 65535, "delta_chunked: %d requests, %d heads of %d", seqs, H, V);
    if (seqs == 0 || max_q_len < from) return 0;
    DeltaArgs da{{qkv, qkv_stride, q_off, k_off, v_off, gates, gates_stride, g1_off, g2_off, a_log, dt_bias, nullptr, 0.f, state,
                  state_stride, 0, 0, 0, out, q_start, q_len, state_slots, H, G, D, V, from},
                 Kn, Qn, Kw, Tm, Aq, scal};
    return launch_delta(da, rows, seqs, max_q_len, dealt, stream);
}
