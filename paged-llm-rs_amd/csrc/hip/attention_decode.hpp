// One workgroup of the attention of single tokens in bfloat16 (attention_decode.hip has what the kernel is built around): in a launch of its own, or as
// the last stage of a chain of products (gemm_chain.hip), whose rows of q come while its keys and values are on their way.
#pragma once
#include "gemm_chain.hpp"


struct __attribute__((aligned(16))) u32x4 {
    uint32_t v[4];
};

__device__ __forceinline__ void unpack8(const u32x4& p, float* f) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = __uint_as_float(p.v[i] << 16);
        f[2 * i + 1] = __uint_as_float(p.v[i] & 0xffff0000u);
    }
}

template <int LPK>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
    for (int off = LPK / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, PL_WAVE);
    return v;
}

// What the kernel needs to normalise and rotate queries and the new key itself (a step in which every
// request brings one token): then no kernel of its own runs for that before attention.
struct ad_fuse_t {
    const void* q_gain;       // per-head norm gains, or null
    const void* k_gain;
    int gain_dtype;
    float eps;
    const float* cos_table;   // [max_pos, rot/2], or null
    const float* sin_table;
    int rot;                  // a multiple of 16
    int mode;                 // 0: q, k and v are ready; 1: q is raw; 2: q is raw, and the token's key and value
                              //    are taken raw from its row, used, and written into the cache
};

__device__ __forceinline__ void ad_load_gain8(const void* gain, int dtype, int at, float* out) {
    if (dtype == PL_DTYPE_F32) {
        struct __attribute__((aligned(16))) f4 { float v[4]; };
        const f4 a = *reinterpret_cast<const f4*>(static_cast<const float*>(gain) + at);
        const f4 b = *reinterpret_cast<const f4*>(static_cast<const float*>(gain) + at + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            out[i] = a.v[i];
            out[4 + i] = b.v[i];
        }
    } else {
        unpack8(*reinterpret_cast<const u32x4*>(static_cast<const bf16_t*>(gain) + at), out);
    }
}

// Sum over the LPK lanes of a key.  Sixteen lanes are a row of the wave's data-parallel primitives: the
// sum then runs on the vector unit alone (four rotations within the row), without a trip through LDS.
template <int LPK>
__device__ __forceinline__ float key_sum(float v) {
    if constexpr (LPK == 16) {
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf, 0xf, false));  // row_ror:8
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xf, 0xf, false));  // row_ror:4
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x122, 0xf, 0xf, false));  // row_ror:2
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x121, 0xf, 0xf, false));  // row_ror:1
        return v;
    } else {
        return group_sum<LPK>(v);
    }
}

// What a lane needs of the norm's gains and the rotation's angles for its eight elements of a head, asked
// for before anything else so that the norm waits for no load of its own.
struct ad_prep_t {
    float gain[8];
    float c[8], s[8];
};

__device__ __forceinline__ void ad_load_prep(ad_prep_t& p, const void* gain, const ad_fuse_t& f, int d, int dl, int pos) {
    const int at = min(dl * 8, d - 8);
    if (gain) ad_load_gain8(gain, f.gain_dtype, at, p.gain);
    const int half = f.rot / 2, hc = half / 8;
    if (f.cos_table && dl * 8 < f.rot) {
        const int ta = (dl < hc ? dl : dl - hc) * 8;
        ad_load_gain8(f.cos_table + static_cast<size_t>(pos) * half, PL_DTYPE_F32, ta, p.c);
        ad_load_gain8(f.sin_table + static_cast<size_t>(pos) * half, PL_DTYPE_F32, ta, p.s);
    }
}

// One head spread over LPK lanes, eight elements a lane: RMSNorm over the head, rotation by the
// token's position (the partner of an element lies rot/16 lanes away), rounding to bfloat16 as the
// stand-alone kernel stores it.  Every lane of the wave takes part in the exchanges.
template <int LPK>
__device__ __forceinline__ void ad_norm_rope8(float* x, bool with_gain, const ad_prep_t& p, const ad_fuse_t& f, int d, int dl) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = fmaf(x[i], x[i], ss);
    ss = key_sum<LPK>(ss);
    if (with_gain) {
        const float rinv = 1.f / sqrtf(ss / static_cast<float>(d) + f.eps);   // (as the stand-alone kernel computes it)
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = x[i] * rinv * p.gain[i];
    }
    const int half = f.rot / 2, hc = half / 8;
    const bool low = dl < hc;
    float px[8];
    if (LPK == 16 && hc == 8) {
        // a head of 128 rotated whole: the partner lies eight lanes on in the row of sixteen
#pragma unroll
        for (int i = 0; i < 8; ++i)
            px[i] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x[i]), 0x128, 0xf, 0xf, false));
    } else {
        const int lane = threadIdx.x % PL_WAVE;
        const int partner = min(max(lane + (low ? hc : -hc), 0), PL_WAVE - 1);
#pragma unroll
        for (int i = 0; i < 8; ++i) px[i] = __shfl(x[i], partner, PL_WAVE);
    }
    if (f.cos_table && dl * 8 < f.rot) {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = low ? x[i] * p.c[i] - px[i] * p.s[i] : x[i] * p.c[i] + px[i] * p.s[i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = to_float(from_float<bf16_t>(x[i]));
}

typedef __bf16 ad_bf16x2 __attribute__((ext_vector_type(2)));

// a . b over two bfloat16 pairs held in one word each, added to c in 32-bit (v_dot2c_f32_bf16)
__device__ __forceinline__ float ad_dot2(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(ad_bf16x2, a), __builtin_bit_cast(ad_bf16x2, b), c, false);
}

__device__ __forceinline__ uint32_t ad_pack2(float lo, float hi) {
    return static_cast<uint32_t>(bf16_bits_from_float(lo)) | (static_cast<uint32_t>(bf16_bits_from_float(hi)) << 16);
}

// The tokens of the requests with fewer than `short_limit` tokens, counted through the requests in their
// order: which row of the step is number `slot`?  (The requests' rows follow each other.)  A step of a long
// portion beside single tokens then has workgroups for the single tokens only: one for every row of the
// portion as well, each of which would leave at once, costs the launch some 7 ns apiece.  Every thread of the
// workgroup calls this with all lanes of its wave; false: there is no such token.
__device__ __forceinline__ bool ad_find_row(int slot, const int* __restrict__ q_len, int num_seqs, int short_limit,
                                            int& row) {
    const int lane = threadIdx.x % PL_WAVE;
    int rows_before = 0, short_before = 0;
    for (int base = 0; base < num_seqs; base += PL_WAVE) {
        const int s = base + lane;
        const int count = s < num_seqs ? q_len[s] : 0;
        const int few = count < short_limit ? count : 0;
        int rows_through = count, short_through = few;
#pragma unroll
        for (int off = 1; off < PL_WAVE; off <<= 1) {
            const int a = __shfl_up(rows_through, off, PL_WAVE), b = __shfl_up(short_through, off, PL_WAVE);
            if (lane >= off) {
                rows_through += a;
                short_through += b;
            }
        }
        // (uniform, and said to be: what follows from them stays in scalar registers)
        const int rows_here = __builtin_amdgcn_readfirstlane(__shfl(rows_through, PL_WAVE - 1, PL_WAVE));
        const int short_here = __builtin_amdgcn_readfirstlane(__shfl(short_through, PL_WAVE - 1, PL_WAVE));
        if (slot < short_before + short_here) {
            const bool mine = few > 0 && slot >= short_before + short_through - few && slot < short_before + short_through;
            const int l = __ffsll(static_cast<unsigned long long>(__ballot(mine))) - 1;   // one lane says so
            row = __builtin_amdgcn_readfirstlane(rows_before + __shfl(rows_through - count, l, PL_WAVE) +
                                                 (slot - short_before - __shfl(short_through - few, l, PL_WAVE)));
            return true;
        }
        rows_before += rows_here;
        short_before += short_here;
    }
    return false;
}

// The pages of a workgroup's stretch of keys are copied into LDS first, this many at most; a longer
// stretch looks its pages up in the table itself.
#define AD_PAGES_LDS 2048

// LPK: lanes a key (a power of two, LPK*8 >= d).  GT: query heads a workgroup serves.
// U: keys a lane group asks for at once.  WV: waves a workgroup.
// num_seqs > 0: blockIdx.y counts the tokens of the short requests (ad_find_row) and not the step's rows.
//
// The kernel's time with few tokens is the length of its chain of dependent trips to memory and the
// number of instructions a wave issues (four cycles each).  The chain is kept at three: the token's position and request (scalar loads); then, together, the pages of the
// workgroup's stretch (into LDS), the query row, the norm's gains, the rotation's angles and, when it is
// to be written, the token's own raw key and value; then keys and values, two rounds of them in flight
// at all times with nothing else between them in the queue of loads (page numbers come from LDS, so no
// round waits behind a table lookup).  Queries and the own key are normalised and rotated while the
// first two rounds are on their way.
// EX 1: the launch has sinks or distance slopes; without them (0) the kernel is compiled as if it knew neither, and takes
// the arguments it always took.  EX 2: it may also have a soft cap on the scores, first keys kept beside the window
// and a gate a head (PlAttentionMore).
// Kept keys stand in front of the window's in the numbering that splits and rounds go by: key number i is key
// i - (first - kept) of the request where i < first, and key i from `first` on.
template <int EX>
struct ad_extras_t {
    const float* sinks;
    const float* slopes;
    PlAttentionMore more;
};
template <>
struct ad_extras_t<1> {
    const float* sinks;
    const float* slopes;
};
template <>
struct ad_extras_t<0> {
    static constexpr const float* sinks = nullptr;
    static constexpr const float* slopes = nullptr;
};

struct ad_true_t { static constexpr bool value = true; };
struct ad_false_t { static constexpr bool value = false; };

#define AD_MERGE_AT_ONCE 8      // shares whose results are on their way together when they are put together

// Where a workgroup's rows of q come from another stage of the same launch (WAITS): whether it has to look for them, how often, and where
// it says that they did not come.
struct ad_rows_t {
    bool asks;
    int looks;
    int* late;
};

// One workgroup's part (bx: key head and tile of its query heads, by: token, bz: split).  Returns whether it is done (false, with WAITS: its rows were
// not there in time), the same for all threads.
template <int LPK, int GT, int U, int WV, int EX, bool WAITS>
__device__ __forceinline__ bool
ad_attend(const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out,
                              float* __restrict__ part_acc, float* __restrict__ part_ml,
                              const int* __restrict__ positions, const int* __restrict__ seq_of,
                              const int* __restrict__ q_len, int short_limit, int num_seqs,
                              const int* __restrict__ block_table, int max_blocks, int block_size,
                              bf16_t* __restrict__ k_pool, bf16_t* __restrict__ v_pool, int nq,
                              int nkv, int d, float scale_log2e, int window, int splits, int tiles, int g,
                              uint32_t splits_magic, ad_fuse_t fuse, int* __restrict__ arrivals, ad_extras_t<EX> extras,
          int bx, int by, int bz, float* lds, ad_rows_t rows_of) {
#define AD_DONE(done) return done
#include "attention_decode_body.hpp"
#undef AD_DONE
    return true;
}
