// Shared by the kernels of the mixers that carry a matrix of state: what a launch is told, and the
// gates' functions, all 32-bit.
#pragma once

#include "common.hpp"

#define PL_SCAN_LIGHTNING 0
#define PL_SCAN_MLSTM 1
#define PL_SCAN_DELTA 2
#define PL_SCAN_SSD 3
#define PL_SCAN_RETENTION 4

struct ScanArgs {
    const float* qkv;         // rows holding q, k and v (for the delta rule: already convolved and activated)
    int qkv_stride, q_off, k_off, v_off;
    const float* gates;       // rows holding the two pre-activations of the gates (mlstm: i, f; delta: beta, a); ssd: the step size's, from g1_off
    int gates_stride, g1_off, g2_off;
    const float* p1;          // lightning, retention: decay a head; mlstm: bias of i; delta, ssd: A_log
    const float* p2;          // mlstm: bias of f; delta, ssd: dt_bias
    const float* p3;          // ssd: what a head's v counts in its own read-out
    float cap;                // mlstm: the cap of the gates' pre-activations
    float* state;             // [slots, state_stride]
    long state_stride;
    int s_off, n_off, m_off;  // where S [H, D, V], n [H, tiles, D] and m [H, tiles] start inside a slot (tiles of 64
                              // columns of V: every tile's wave keeps a copy of n and m of its own)
    float* out;               // [rows, H * V]
    const int* q_start;
    const int* q_len;
    const int* state_slots;
    int H, G, D, V;           // heads, heads of q and k (G divides H), size of q and k, size of v
    int below;                // the token-by-token kernel takes requests of fewer tokens than this (0: all);
                              // the chunked kernels take the others
};

__device__ __forceinline__ float softplus_f(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float logsigmoid_f(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }
__device__ __forceinline__ float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float silu_f(float x) { return x / (1.f + expf(-x)); }

// A launch in chunks of 64 tokens has a workgroup for every chunk that the step's rows can hold, not for the chunks of the longest request
// times the requests (a padded step only knows that every row might be one request's): which request's chunk is number `at`
// among the chunks of the requests that the launch serves?  Called by all lanes of a wave; false: there is no such chunk.  (Three requests
// over 2,816 rows, 42 chunks, 16 workgroups each: 752 workgroups in the place of 2,112.  One that finds nothing to do costs a launch
// some 7 ns.)
struct ChunkPlace {
    int s, c, count, first_row;         // the request, the chunk of it, the request's tokens and first row
};
__device__ __forceinline__ bool find_chunk(const ScanArgs& a, int seqs, int at, ChunkPlace& place) {
    const int lane = threadIdx.x & 63;
    for (int base = 0; base < seqs; base += 64) {
        const int s = min(base + lane, seqs - 1);
        const int count = a.q_len[s], first_row = a.q_start[s];
        const bool served = base + lane < seqs && a.state_slots[s] >= 0 && count >= a.below;
        const int mine = served ? (count + 63) / 64 : 0;
        int through = mine;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int other = __shfl_up(through, off, 64);
            if (lane >= off) through += other;
        }
        const int total = __builtin_amdgcn_readfirstlane(__shfl(through, 63, 64));
        if (at < total) {
            const int l = __ffsll(static_cast<unsigned long long>(__ballot(at < through))) - 1;      // the first request that reaches it
            place.s = __builtin_amdgcn_readfirstlane(base + l);
            place.c = __builtin_amdgcn_readfirstlane(at - __shfl(through - mine, l, 64));
            place.count = __builtin_amdgcn_readfirstlane(__shfl(count, l, 64));
            place.first_row = __builtin_amdgcn_readfirstlane(__shfl(first_row, l, 64));
            return true;
        }
        at -= total;
    }
    return false;
}
// The workgroups such a launch needs: of `rows` rows, requests of up to `max_q_len` tokens.
static inline int chunk_bound(int rows, int max_q_len, int seqs) {
    const long long each = static_cast<long long>((max_q_len + 63) / 64) * seqs, all = rows / 64 + static_cast<long long>(seqs);
    return static_cast<int>(each < all ? each : all);
}

// The kernel for requests of few tokens that spreads a state over four waves (ssd.hip), for the kinds lightning, mlstm and delta.
bool pl_state_step(int kind, const ScanArgs& a, int seqs, hipStream_t stream);
