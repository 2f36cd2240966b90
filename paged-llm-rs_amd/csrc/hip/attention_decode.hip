// Paged attention for single tokens in bfloat16: a decoded token, or a token of
// a short prompt portion, reading the keys 0..position of its request through
// the block table.  The work is a stream of the request's keys and values
// through the chip, so the kernel is built around 16-byte loads that are all in
// flight together:
//
//   grid (kv head x query-head tile, token, split).  A workgroup of four or eight
//   waves owns one stretch of the context (split-KV) of one kv head and serves up to
//   GT of the query heads that share it, so keys and values are read once per
//   kv head, not once per query head.
//   A group of LPK lanes owns one key: each lane holds 8 of its values.  A wave
//   handles 64/LPK keys with one load instruction and four or eight such
//   instructions are issued back to back for keys and for values.
//   Softmax is online (running maximum and sum in 32-bit, base-2 exponentials
//   with log2(e) folded into the query scale).  The lane groups and waves keep
//   separate running states; a wave's are merged in its registers and the waves'
//   through LDS at the end; with more than one split the partial results go to a
//   workspace and a second kernel merges them.
#include "attention_decode.hpp"

template <int LPK, int GT, int U, int WV, int EX = 0>
__global__ void __launch_bounds__(64 * WV)
paged_attention_decode_kernel(const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out,
                              float* __restrict__ part_acc, float* __restrict__ part_ml,
                              const int* __restrict__ positions, const int* __restrict__ seq_of,
                              const int* __restrict__ q_len, int short_limit, int num_seqs,
                              const int* __restrict__ block_table, int max_blocks, int block_size,
                              bf16_t* __restrict__ k_pool, bf16_t* __restrict__ v_pool, int nq,
                              int nkv, int d, float scale_log2e, int window, int splits, int tiles, int g,
                              uint32_t splits_magic, ad_fuse_t fuse, int* __restrict__ arrivals, ad_extras_t<EX> extras) {
    extern __shared__ float lds[];
    constexpr bool WAITS = false;
    constexpr ad_rows_t rows_of{false, 0, nullptr};
    const int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
#define AD_DONE(done) return
#include "attention_decode_body.hpp"
#undef AD_DONE
}

// Merges the splits of one (token, query head): out = sum_s a_s 2^(m_s - M) / sum_s l_s 2^(m_s - M).
// For launches without room for their workgroups' arrivals.  One thread an output element; every load is asked for before
// any is used.
#define AD_MAX_SPLITS 64

template <int SP, bool EX = false>
__global__ void __launch_bounds__(256)
paged_attention_merge_kernel(const float* __restrict__ part_acc, const float* __restrict__ part_ml,
                             bf16_t* __restrict__ out, const int* __restrict__ positions,
                             const int* __restrict__ seq_of, const int* __restrict__ q_len, int short_limit,
                             int nq, int d, int splits, int n, int num_seqs, const float* __restrict__ sinks,
                             PlAttentionMore more) {
    const int per_token = nq * d;
    int t, rest;
    bool inside;
    if (num_seqs > 0) {      // blockIdx.y counts the tokens of the short requests, blockIdx.x a token's elements
        if (!ad_find_row(blockIdx.y, q_len, num_seqs, short_limit, t)) return;
        rest = blockIdx.x * blockDim.x + threadIdx.x;
        inside = rest < per_token;
        rest = min(rest, per_token - 1);
    } else {                 // blockIdx.y is the token
        t = blockIdx.y;
        rest = blockIdx.x * blockDim.x + threadIdx.x;
        inside = rest < per_token;
        rest = min(rest, per_token - 1);
    }
    // (a head size that is a power of two spares the kernel a division in front of its loads)
    const int h = (d & (d - 1)) == 0 ? rest >> (31 - __builtin_clz(static_cast<unsigned>(d))) : rest / d;
    const int dd = rest - h * d;
    const size_t base = (static_cast<size_t>(t) * nq + h) * splits;
    const int pos = positions[t];
    const int len = q_len ? q_len[seq_of[t]] : 0;
    float ms[SP], ls[SP], as[SP];
#pragma unroll
    for (int s = 0; s < SP; ++s) {
        const int sc = min(s, splits - 1);
        ms[s] = part_ml[(base + sc) * 2];
        ls[s] = part_ml[(base + sc) * 2 + 1];
        as[s] = part_acc[(base + sc) * d + dd];
    }
    if (!inside || pos < 0 || (q_len && len >= short_limit)) return;
    float big = -INFINITY;
#pragma unroll
    for (int s = 0; s < SP; ++s) big = fmaxf(big, s < splits ? ms[s] : -INFINITY);
    float sum = 0.f, a = 0.f;
#pragma unroll
    for (int s = 0; s < SP; ++s) {
        const float w = (s < splits && ms[s] != -INFINITY) ? exp2f(ms[s] - big) : 0.f;
        sum = fmaf(ls[s], w, sum);
        a = fmaf(as[s], w, a);
    }
    if (EX && sinks != nullptr) {
        const float sk = sinks[h] * 1.4426950408889634f;
        const float top = fmaxf(big, sk);
        const float keep = big == -INFINITY ? 0.f : exp2f(big - top);
        sum = sum * keep + exp2f(sk - top);
        a *= keep;
    }
    if (EX && more.gate != nullptr) a *= pl_head_gate(more, t, h);
    out[(static_cast<size_t>(t) * nq + h) * d + dd] = from_float<bf16_t>(sum > 0.f ? a / sum : 0.f);
}

#define AD_WAVES 4

template <int LPK, int GT, int U>
static int launch_decode_keys(const void* q, int q_stride, void* out, float* part_acc, float* part_ml,
                              const int* positions, const int* seq_of, const int* q_len, int short_limit, int num_seqs,
                              int short_rows, const int* block_table, int max_blocks, int block_size, void* k_pool,
                              void* v_pool, int n, int nq, int nkv, int d, float scale, int window, int splits,
                              const ad_fuse_t& fuse, int* arrivals, const float* sinks, const float* slopes,
                              const PlAttentionMore& more, hipStream_t stream) {
    constexpr int WV = AD_WAVES;
    const int g = nq / nkv;
    const int tiles = pl_ceil_div(g, GT);
    const size_t lds_bytes = (AD_PAGES_LDS + static_cast<size_t>(WV) * GT * 2 + static_cast<size_t>(WV) * GT * d) * sizeof(float);
    PL_REQUIRE(lds_bytes <= 160 * 1024, "decode attention: %zu bytes of LDS for head size %d", lds_bytes, d);
    const int extras = pl_has_more(more) ? 2 : (sinks != nullptr || slopes != nullptr ? 1 : 0);
    if (lds_bytes > 48 * 1024) {
        const void* kernel = extras == 2 ? reinterpret_cast<const void*>(&paged_attention_decode_kernel<LPK, GT, U, WV, 2>)
                             : extras == 1 ? reinterpret_cast<const void*>(&paged_attention_decode_kernel<LPK, GT, U, WV, 1>)
                                           : reinterpret_cast<const void*>(&paged_attention_decode_kernel<LPK, GT, U, WV, 0>);
        hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes));
        PL_REQUIRE(e == hipSuccess, "decode attention: %zu bytes of LDS refused: %s", lds_bytes, hipGetErrorString(e));
    }
    // rows of the grid: the step's rows, or, where fewer, the tokens that the short requests can bring
    const bool compact = q_len != nullptr && num_seqs > 0 && short_rows > 0 && short_rows < n;
    dim3 grid(nkv * tiles, compact ? short_rows : n, splits);
    PL_REQUIRE(n <= 65535 && splits <= 65535, "decode attention: %d tokens or %d splits are more than one launch covers", n, splits);
#define AD_LAUNCH(EX)                                                                                                  \
    paged_attention_decode_kernel<LPK, GT, U, WV, EX><<<grid, 64 * WV, lds_bytes, stream>>>(                           \
        static_cast<const bf16_t*>(q), q_stride, static_cast<bf16_t*>(out), part_acc, part_ml, positions, seq_of,      \
        q_len, short_limit, compact ? num_seqs : 0, block_table, max_blocks, block_size, static_cast<bf16_t*>(k_pool), \
        static_cast<bf16_t*>(v_pool), nq, nkv, d, scale * 1.4426950408889634f, window, splits, tiles, g,              \
        static_cast<uint32_t>((0x100000000ull + splits - 1) / static_cast<unsigned>(splits)), fuse, arrivals, with)
    if (extras == 2) {
        const ad_extras_t<2> with{sinks, slopes, more};
        AD_LAUNCH(2);
    } else if (extras == 1) {
        const ad_extras_t<1> with{sinks, slopes};
        AD_LAUNCH(1);
    } else {
        const ad_extras_t<0> with{};
        AD_LAUNCH(0);
    }
#undef AD_LAUNCH
    PL_CHECK_LAUNCH("paged_attention_decode");
    if (splits > 1 && arrivals == nullptr) {
        const dim3 mgrid = dim3(pl_ceil_div(nq * d, 256), compact ? short_rows : n);
#define AD_MERGE(SP)                                                                                              \
    do {                                                                                                          \
        if (sinks != nullptr || more.gate != nullptr)                                                             \
            paged_attention_merge_kernel<SP, true><<<mgrid, 256, 0, stream>>>(                                    \
                part_acc, part_ml, static_cast<bf16_t*>(out), positions, seq_of, q_len, short_limit, nq, d,       \
                splits, n, compact ? num_seqs : 0, sinks, more);                                                     \
        else                                                                                                      \
            paged_attention_merge_kernel<SP, false><<<mgrid, 256, 0, stream>>>(                                   \
                part_acc, part_ml, static_cast<bf16_t*>(out), positions, seq_of, q_len, short_limit, nq, d,       \
                splits, n, compact ? num_seqs : 0, nullptr, more);                                                     \
    } while (0)
        if (splits <= 4) AD_MERGE(4);
        else if (splits <= 8) AD_MERGE(8);
        else if (splits <= 16) AD_MERGE(16);
        else AD_MERGE(AD_MAX_SPLITS);
#undef AD_MERGE
        PL_CHECK_LAUNCH("paged_attention_merge");
    }
    return 0;
}

// Keys a lane group asks for a round (as many again are in flight for the round after).  With at most a
// workgroup a compute unit, what one workgroup has in flight has to keep its compute unit's path to memory
// busy: eight keys a round, which the registers of a lone wave a SIMD hold.  With more workgroups, four (two
// where a workgroup serves many query heads), so that several workgroups fit a compute unit.  The choice
// goes by the step's rows, not by the rows that get workgroups, so that a step computes the same bits
// however its launch is sized.

template <int LPK, int GT>
static int launch_decode(const void* q, int q_stride, void* out, float* part_acc, float* part_ml,
                         const int* positions, const int* seq_of, const int* q_len, int short_limit, int num_seqs,
                         int short_rows, const int* block_table, int max_blocks, int block_size, void* k_pool,
                         void* v_pool, int n, int nq, int nkv, int d, float scale, int window, int splits,
                         const ad_fuse_t& fuse, int* arrivals, const float* sinks, const float* slopes,
                              const PlAttentionMore& more, hipStream_t stream) {
    const long long workgroups = static_cast<long long>(nkv) * pl_ceil_div(nq / nkv, GT) * n * splits;
#define AD_KEYS_CALL(U)                                                                                            \
    return launch_decode_keys<LPK, GT, U>(q, q_stride, out, part_acc, part_ml, positions, seq_of, q_len,          \
                                          short_limit, num_seqs, short_rows, block_table, max_blocks, block_size,  \
                                          k_pool, v_pool, n, nq, nkv, d, scale, window, splits, fuse, arrivals, sinks, slopes, more, stream)
    if constexpr (GT <= 2) {
        if (workgroups <= pl_compute_units()) AD_KEYS_CALL(8);
        AD_KEYS_CALL(4);
    } else {
        AD_KEYS_CALL(2);
    }
#undef AD_KEYS_CALL
}

template <int LPK>
static int dispatch_gt(int gt, const void* q, int q_stride, void* out, float* part_acc, float* part_ml,
                       const int* positions, const int* seq_of, const int* q_len, int short_limit, int num_seqs,
                       int short_rows, const int* block_table, int max_blocks, int block_size, void* k_pool,
                       void* v_pool, int n, int nq, int nkv, int d, float scale, int window, int splits,
                       const ad_fuse_t& fuse, int* arrivals, const float* sinks, const float* slopes,
                              const PlAttentionMore& more, hipStream_t stream) {
#define AD_CALL(G)                                                                                              \
    return launch_decode<LPK, G>(q, q_stride, out, part_acc, part_ml, positions, seq_of, q_len, short_limit,   \
                                 num_seqs, short_rows, block_table, max_blocks, block_size, k_pool, v_pool, n, nq, nkv, d, scale,    \
                                 window, splits, fuse, arrivals, sinks, slopes, more, stream)
    switch (gt) {
        case 1: AD_CALL(1);
        case 2: AD_CALL(2);
        case 4: AD_CALL(4);
        default: AD_CALL(8);
    }
#undef AD_CALL
}

// The most shares whose workgroups meet in the kernel.
extern "C" int pl_paged_attention_decode_meets() { return AD_MERGE_AT_ONCE; }

// bfloat16 only.  With splits > 1 the workspace needs n*nq*splits*d floats (part_acc) and n*nq*splits*2 (part_ml).
// q_len (may be null) and short_limit leave the tokens of requests with q_len >= short_limit to the tiled kernel.
// With q_len: num_seqs, the requests whose rows follow each other in q from row 0 on, and short_rows, the most
// tokens that the other requests bring together (0: not known); where that is fewer than the step's rows the
// launch has workgroups for those tokens only.
// fuse_mode 0: the rows of q are ready and the cache holds every key up to each token's own.  1: the rows of q are
// the raw projection and are normalised (gains, eps) and rotated (tables, rot a multiple of 16) here.  2: as 1, and
// each token's key and value are taken raw from its row [q | k | v], used, and written into the cache; every
// request then has to bring exactly one token.
// `arrivals`: n * nq zeros, and zeros again behind the launch, for the shares' workgroups to meet at; null: the shares are put
// together by a second kernel, and so are more than AD_MERGE_AT_ONCE, which the last workgroup would fetch in several trips and in
// another order of sums (the 0.6B shape, one token at contexts up to 3,900 1,197 us a step against 1,273; 64 tokens the same either way).
extern "C" int pl_paged_attention_decode(const void* q, int q_stride, void* out, float* part_acc, float* part_ml,
                                         const int* positions, const int* seq_of, const int* q_len, int short_limit,
                                         int num_seqs, int short_rows,
                                         const int* block_table, int max_blocks, int block_size, void* k_pool,
                                         void* v_pool, int n, int nq, int nkv, int d, float scale, int window,
                                         int splits, int fuse_mode, const void* q_gain, const void* k_gain,
                                         int gain_dtype, float eps, const float* cos_table, const float* sin_table,
                                         int rot, const float* sinks, const float* slopes, float cap, int keep,
                                         const float* gate, int gate_stride, int* arrivals, hipStream_t stream) {
    const PlAttentionMore more{cap, keep, gate, gate_stride};
    PL_REQUIRE(cap >= 0.f && keep >= 0 && (gate == nullptr || gate_stride >= nq) && (keep == 0 || window >= 0),
               "decode attention: a cap of %g, %d first keys kept beside a window of %d, gates in rows of %d",
               static_cast<double>(cap), keep, window, gate_stride);
    PL_REQUIRE(fuse_mode == 0 || !pl_has_more(more), "decode attention: caps, kept keys and gates go with prepared queries");
    PL_REQUIRE(d > 0 && d <= 256 && d % 16 == 0, "decode attention: head size %d, which has to be a multiple of 16 up to 256", d);
    PL_REQUIRE(nq > 0 && nkv > 0 && nq % nkv == 0, "decode attention: %d query heads over %d key heads", nq, nkv);
    PL_REQUIRE(block_size > 0 && max_blocks > 0 && q_stride >= nq * d && q_stride % 8 == 0 && splits >= 1 && splits <= AD_MAX_SPLITS,
               "decode attention: block size %d, %d blocks a row, query stride %d, window %d, %d splits", block_size,
               max_blocks, q_stride, window, splits);
    PL_REQUIRE(splits == 1 || (part_acc && part_ml), "decode attention: %d splits without a workspace", splits);
    PL_REQUIRE(fuse_mode >= 0 && fuse_mode <= 2, "decode attention: fuse mode %d", fuse_mode);
    if (fuse_mode != 0) {
        PL_REQUIRE(rot >= 0 && rot <= d && rot % 16 == 0, "decode attention: a rotated width of %d of a head of %d is not fused", rot, d);
        PL_REQUIRE((q_gain == nullptr) == (k_gain == nullptr), "decode attention: one of the two gains is missing");
        PL_REQUIRE(!q_gain || gain_dtype == PL_DTYPE_F32 || gain_dtype == PL_DTYPE_BF16, "decode attention: gain dtype code %d", gain_dtype);
        PL_REQUIRE((cos_table == nullptr) == (sin_table == nullptr) && (cos_table || rot == 0), "decode attention: rotation tables");
        PL_REQUIRE(fuse_mode != 2 || (q_len == nullptr && q_stride >= (nq + 2 * nkv) * d),
                   "decode attention: the fused cache write is for steps of one token a request over rows [q | k | v]");
    }
    const ad_fuse_t fuse{q_gain, k_gain, gain_dtype, eps, cos_table, sin_table, rot, fuse_mode};
    if (n <= 0) return 0;
    if (splits > AD_MERGE_AT_ONCE) arrivals = nullptr;
    const int g = nq / nkv;
    const int gt = g >= 8 ? 8 : (g > 2 ? 4 : g);   // 1, 2, 4 or 8 query heads a workgroup; the rest are more tiles
    const int chunks = d / 8;
#define AD_LPK(L)                                                                                                  \
    return dispatch_gt<L>(gt, q, q_stride, out, part_acc, part_ml, positions, seq_of, q_len, short_limit,        \
                          num_seqs, short_rows, block_table, max_blocks, block_size, k_pool, v_pool, n, nq, nkv, d, scale, window,      \
                          splits, fuse, arrivals, sinks, slopes, more, stream)
    if (chunks <= 2) AD_LPK(2);
    if (chunks <= 4) AD_LPK(4);
    if (chunks <= 8) AD_LPK(8);
    if (chunks <= 16) AD_LPK(16);
    AD_LPK(32);
#undef AD_LPK
}
