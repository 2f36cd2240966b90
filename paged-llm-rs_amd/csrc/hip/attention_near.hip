// Attention of a step in which no request's context is longer than 128 tokens, from the raw projection on: per-head norm and rotation of q and k,
// the write of k and v into the pages, and the read-out, one launch for what takes two otherwise (bfloat16, heads of 128 rotated whole or not at all).
//
// A workgroup of eight waves is one request and query head.  What is new of the request it takes from the projection's rows, what was there before
// from the pages: all threads prepare rows (16 lanes a row of 128, as the stand-alone kernel does, so the pages get the same bits), which go to LDS, keys and
// queries in rows of 256 bytes (16-byte pieces permuted by their row against bank conflicts), values transposed.  A wave then takes 32 tokens and one or
// two tiles of 32 of the head's columns: S^T = K Q^T and O^T = V^T P^T (v_mfma_f32_32x32x16_bf16), P straight from the first product's registers, the
// keys of a step of the second in the order in which a lane holds them.  Every query head prepares its key head's keys again; the first of a group
// writes them.
//
// A weight of zero does not hide an infinite or NaN value, and the second product multiplies a tile's tokens with keys behind them: what comes out is then not finite, which is what a
// wave looks for.  It then takes the product again without such values and adds them value by value to the tokens that see their key, so a token is what it is with only the keys up to itself.
//
// Bound by its chain of trips (the request's numbers and pages; its rows) and the arithmetic of preparing rows, a vector instruction a wave every 4 to 5
// cycles.  us, a hundred in a row in a captured graph, the two kernels before / this one, 16 heads over 8: 37 fresh tokens 10.4 / 7.3, 128 15.1 / 12.7, eight requests of
// 10 15.6 / 5.6, 10 tokens behind 110 10.8 / 9.3; 64 heads over 8: 37 fresh tokens 10.6 / 7.4, eight requests of 10 19.1 / 10.1.  (0.1 to 0.2 of it look whether the result is
// finite; looking through the values as they are laid in LDS took 0.2 to 0.4.)
#include "common.hpp"
#include "head_rows.hpp"

typedef __bf16 an_bf16x8 __attribute__((ext_vector_type(8)));
typedef float an_f32x16 __attribute__((ext_vector_type(16)));
typedef hr_u32x4 an_u32x4;
typedef uint32_t an_u32x2 __attribute__((ext_vector_type(2)));

#define AN_KEYS 128                // of a context, at most
#define AN_D 128
#define AN_V_PITCH (AN_KEYS * 2 + 8)   // bytes between two columns of values

// Whether a value, its low 16 bits, is infinite or NaN.
__device__ __forceinline__ bool an_wild(uint32_t value) { return (value & 0x7f80u) == 0x7f80u; }

__global__ void __launch_bounds__(512, 1)
attention_near_kernel(const bf16_t* __restrict__ qkv, bf16_t* __restrict__ out, const void* __restrict__ q_gain, const void* __restrict__ k_gain,
                      int gain_dtype, float eps, const float* __restrict__ cos_table, const float* __restrict__ sin_table,
                      const int* __restrict__ q_start, const int* __restrict__ q_len, const int* __restrict__ ctx_len,
                      const int* __restrict__ block_table, int max_blocks, int block_size, bf16_t* __restrict__ k_pool,
                      bf16_t* __restrict__ v_pool, int nq, int nkv, float scale) {
    extern __shared__ __attribute__((aligned(16))) char an_lds[];
    char* const q_lds = an_lds;                                        // [token][128]
    char* const k_lds = an_lds + AN_KEYS * 256;                        // [key][128]
    char* const v_lds = an_lds + 2 * AN_KEYS * 256;                    // [column][key]
    const int seq = blockIdx.x, head = blockIdx.y, group = nq / nkv, kvh = head / group;
    const int tid = threadIdx.x, lane = tid % PL_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / PL_WAVE);
    const int chunk = tid % 16, slot = tid / 16;                       // eight values of one of 32 rows
    const int count = q_len[seq], ctx = ctx_len[seq], row0 = q_start[seq];
    // the pool's rows of keys `lane` and 64 + `lane` (negative: the page is missing), asked for beside the request's numbers
    int rows_of[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int key = 64 * u + lane, page = key / block_size;
        const int at = block_table[static_cast<size_t>(seq) * max_blocks + min(page, max_blocks - 1)];
        rows_of[u] = page < max_blocks && at >= 0 ? at * block_size + (key - page * block_size) : -1;
    }
    float gq[8], gk[8];
    const bool gain = q_gain != nullptr;
    if (gain) {
        hr_load_gain(q_gain, gain_dtype, chunk, gq);
        hr_load_gain(k_gain, gain_dtype, chunk, gk);
    }
    if (count <= 0 || ctx <= 0) return;                                // (padding; the whole workgroup)
    const size_t stride = static_cast<size_t>(nq + 2 * nkv) * AN_D;
    if (ctx > AN_KEYS || count > ctx) {                                // (more than the launch was told: none of it is right)
        for (int i = tid; i < count * (AN_D / 2); i += 512)
            *reinterpret_cast<uint32_t*>(out + static_cast<size_t>(row0 + i / (AN_D / 2)) * nq * AN_D + head * AN_D + i % (AN_D / 2) * 2) = 0x7fc07fc0u;
        return;
    }
    const int start = ctx - count;
    const bool writes = head % group == 0, low = chunk < 8;
    // which keys there are, one bit a key, and their rows (asked of the lanes that hold them: by whole waves)
    const unsigned long long there0 = __ballot(lane < ctx && rows_of[0] >= 0), there1 = __ballot(64 + lane < ctx && rows_of[1] >= 0);
    auto place = [&](int key) {
        const int a = __shfl(rows_of[0], key % 64, PL_WAVE), b = __shfl(rows_of[1], key % 64, PL_WAVE);
        return key >= ctx ? -1 : key < 64 ? a : b;
    };
    const int key_tiles = (ctx + 31) / 32;

    // values, two keys a thread, asked for first; those past the context or without a page are zeros (weights of zero meet them)
    an_u32x4 v[2][2];
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int key = 2 * (slot + 32 * w) + u, at = place(key);
            v[w][u] = an_u32x4{0, 0, 0, 0};
            if (at >= 0) {
                const bf16_t* from = key >= start ? qkv + (row0 + key - start) * stride + static_cast<size_t>(nq + nkv + kvh) * AN_D
                                                  : v_pool + (static_cast<size_t>(at) * nkv + kvh) * AN_D;
                v[w][u] = *reinterpret_cast<const an_u32x4*>(from + chunk * 8);
            }
        }
    // the request's own rows, 64 tokens at a time: queries and new keys
    for (int first = 0; first < count; first += 64) {
        an_u32x4 q[2], k[2];
        float c[2][8], sn[2][8];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (first + 32 * u + wave * 4 >= count) continue;          // (the whole wave, which has four of the rows)
            const int t = min(first + 32 * u + slot, count - 1);
            const bf16_t* row = qkv + (row0 + t) * stride + chunk * 8;
            q[u] = *reinterpret_cast<const an_u32x4*>(row + head * AN_D);
            k[u] = *reinterpret_cast<const an_u32x4*>(row + (nq + kvh) * AN_D);
            if (cos_table != nullptr) {
                const size_t at = static_cast<size_t>(start + t) * (AN_D / 2) + (chunk & 7) * 8;
                hr_load8(cos_table + at, c[u]);
                hr_load8(sin_table + at, sn[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (first + 32 * u + wave * 4 >= count) continue;
            const int t = first + 32 * u + slot, key = start + t, at = place(key);
            q[u] = hr_prepare(q[u], gain, gq, eps, cos_table != nullptr, c[u], sn[u], low);
            k[u] = hr_prepare(k[u], gain, gk, eps, cos_table != nullptr, c[u], sn[u], low);
            if (t < count) {
                *reinterpret_cast<an_u32x4*>(q_lds + t * 256 + (chunk ^ (t % 16)) * 16) = q[u];
                *reinterpret_cast<an_u32x4*>(k_lds + key * 256 + (chunk ^ (key % 16)) * 16) = k[u];
                if (writes && at >= 0) *reinterpret_cast<an_u32x4*>(k_pool + (static_cast<size_t>(at) * nkv + kvh) * AN_D + chunk * 8) = k[u];
            }
        }
    }
    // keys that were there before
    for (int first = 0; first < start; first += 32) {
        const int key = first + slot, at = place(key);
        an_u32x4 k = {0, 0, 0, 0};
        if (key < start && at >= 0) k = *reinterpret_cast<const an_u32x4*>(k_pool + (static_cast<size_t>(at) * nkv + kvh) * AN_D + chunk * 8);
        if (key < start) *reinterpret_cast<an_u32x4*>(k_lds + key * 256 + (chunk ^ (key % 16)) * 16) = k;
    }
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const int pair = slot + 32 * w;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int key = 2 * pair + u, at = place(key);
            if (writes && key >= start && at >= 0) *reinterpret_cast<an_u32x4*>(v_pool + (static_cast<size_t>(at) * nkv + kvh) * AN_D + chunk * 8) = v[w][u];
        }
        if (pair >= key_tiles * 16) continue;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t a = e % 2 ? v[w][0][e / 2] >> 16 : v[w][0][e / 2] & 0xffffu, b = e % 2 ? v[w][1][e / 2] >> 16 : v[w][1][e / 2] & 0xffffu;
            *reinterpret_cast<uint32_t*>(v_lds + (chunk * 8 + e) * AN_V_PITCH + pair * 4) = a | b << 16;
        }
    }
    __syncthreads();

    // a wave's 32 tokens and columns: two tiles of tokens by four of columns, or four by two pairs
    const bool many = count > 64;
    const int tile = many ? wave / 2 : wave / 4, r32 = lane % 32, h = lane / 32;
    if (tile * 32 >= count) return;
    const int token = tile * 32 + r32, pos = start + token;
    const int seen_tiles = min(key_tiles, (start + min(tile * 32 + 32, count) + 31) / 32);          // (behind them are keys that no token of the tile sees)
    an_bf16x8 q[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) q[kk] = *reinterpret_cast<const an_bf16x8*>(q_lds + token * 256 + ((2 * kk + h) ^ (token % 16)) * 16);
    an_f32x16 s[4];
    float top = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[kt][i] = 0.f;
        if (kt >= seen_tiles) continue;
        const int key = kt * 32 + r32;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
            const an_bf16x8 k = *reinterpret_cast<const an_bf16x8*>(k_lds + key * 256 + ((2 * kk + h) ^ (key % 16)) * 16);
            s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k, q[kk], s[kt], 0, 0, 0);
        }
        const uint32_t there = static_cast<uint32_t>((kt < 2 ? there0 : there1) >> (kt % 2 * 32));
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int of = 8 * (i / 4) + 4 * h + i % 4;                // the key of the tile
            s[kt][i] = kt * 32 + of <= pos && (there >> of & 1) ? s[kt][i] * (scale * 1.4426950408889634f) : -INFINITY;
            top = fmaxf(top, s[kt][i]);
        }
    }
    top = fmaxf(top, __shfl_xor(top, 32, PL_WAVE));
    const float base = top == -INFINITY ? 0.f : top;                   // (no key seen: all weights are zero)
    float sum = 0.f;
    an_bf16x8 p[4][2];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        if (kt >= seen_tiles) continue;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[kt][i] = __builtin_amdgcn_exp2f(s[kt][i] - base);
            sum += s[kt][i];
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const an_u32x4 packed = {hr_pack2(s[kt][8 * u], s[kt][8 * u + 1]), hr_pack2(s[kt][8 * u + 2], s[kt][8 * u + 3]),
                                     hr_pack2(s[kt][8 * u + 4], s[kt][8 * u + 5]), hr_pack2(s[kt][8 * u + 6], s[kt][8 * u + 7])};
            p[kt][u] = __builtin_bit_cast(an_bf16x8, packed);
        }
    }
    sum += __shfl_xor(sum, 32, PL_WAVE);
    const float by = sum > 0.f || sum != sum ? 1.f / sum : 0.f;
    for (int d = many ? wave % 2 * 2 : wave % 4, last = many ? d + 2 : d + 1; d < last; ++d) {
        an_f32x16 o;
#pragma unroll
        for (int i = 0; i < 16; ++i) o[i] = 0.f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            if (kt >= seen_tiles) continue;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                // (keys 8 (e / 4) + 4 h + e % 4 of this 16, as p holds them)
                const char* from = v_lds + (d * 32 + r32) * AN_V_PITCH + (kt * 32 + u * 16 + 4 * h) * 2;
                const an_u32x2 a = *reinterpret_cast<const an_u32x2*>(from), b = *reinterpret_cast<const an_u32x2*>(from + 16);
                o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(an_bf16x8, an_u32x4{a[0], a[1], b[0], b[1]}), p[kt][u], o, 0, 0, 0);
            }
        }
        // values that are not finite: taken out, and added key by key by the tokens that see it
        float finite = 0.f;                                            // (or NaN)
#pragma unroll
        for (int i = 0; i < 16; ++i) finite = fmaf(o[i], 0.f, finite);
        if (__ballot(token < count && finite != finite) != 0) {
            unsigned long long wild[2] = {0, 0};                       // one bit a key, as `there0` and `there1`
#pragma unroll
            for (int i = 0; i < 16; ++i) o[i] = 0.f;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                if (kt >= seen_tiles) continue;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const char* from = v_lds + (d * 32 + r32) * AN_V_PITCH + (kt * 32 + u * 16 + 4 * h) * 2;
                    const an_u32x2 a = *reinterpret_cast<const an_u32x2*>(from), b = *reinterpret_cast<const an_u32x2*>(from + 16);
                    an_u32x4 kept = {a[0], a[1], b[0], b[1]};
#pragma unroll
                    for (int e = 0; e < 8; ++e) {                      // (both halves of the wave: keys 4 apart)
                        const bool mine = an_wild(kept[e / 2] >> (e % 2 * 16));
                        const unsigned long long lanes = __ballot(mine);
                        const int key = kt % 2 * 32 + u * 16 + e / 4 * 8 + e % 4;
                        if (lanes & 0xffffffffull) wild[kt / 2] |= 1ull << key;
                        if (lanes >> 32) wild[kt / 2] |= 1ull << (key + 4);
                        if (mine) kept[e / 2] &= e % 2 ? 0xffffu : 0xffff0000u;
                    }
                    o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(an_bf16x8, kept), p[kt][u], o, 0, 0, 0);
                }
            }
#pragma unroll
            for (int half = 0; half < 2; ++half)
                for (unsigned long long left = wild[half]; left != 0; left &= left - 1) {
                    const int key = 64 * half + __ffsll(left) - 1, of = key % 32;
                    float weight = 0.f;                                // (held by one of the token's two lanes)
#pragma unroll
                    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                        for (int i = 0; i < 16; ++i)
                            if (kt < seen_tiles && kt == key / 32 && 8 * (i / 4) + 4 * h + i % 4 == of) weight = s[kt][i];
                    weight += __shfl_xor(weight, 32, PL_WAVE);
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const uint32_t value = *reinterpret_cast<const uint16_t*>(v_lds + (d * 32 + 8 * (i / 4) + 4 * h + i % 4) * AN_V_PITCH + key * 2);
                        if (key <= pos && an_wild(value)) o[i] += weight * __uint_as_float(value << 16);
                    }
                }
        }
        if (token < count) {
            bf16_t* to = out + static_cast<size_t>(row0 + token) * nq * AN_D + head * AN_D + d * 32 + 4 * h;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *reinterpret_cast<an_u32x2*>(to + 8 * j) = an_u32x2{hr_pack2(o[4 * j] * by, o[4 * j + 1] * by), hr_pack2(o[4 * j + 2] * by, o[4 * j + 3] * by)};
        }
    }
}

// Request s of the first `num_seqs` brings the rows q_start[s] .. q_start[s] + q_len[s] - 1 of qkv (raw projections [q | k | v]) at the positions that end in
// ctx_len[s] - 1; no context is longer than 128 (rows of longer ones come out as NaN).  gains: null, or of 128 values; cos_table null: nothing is turned.
extern "C" int pl_attention_near(const void* qkv, void* out, const void* q_gain, const void* k_gain, int gain_dtype, float eps, const float* cos_table,
                                 const float* sin_table, const int* q_start, const int* q_len, const int* ctx_len, int num_seqs, const int* block_table,
                                 int max_blocks, int block_size, void* k_pool, void* v_pool, int nq, int nkv, float scale, hipStream_t stream) {
    PL_REQUIRE(nq > 0 && nkv > 0 && nq % nkv == 0 && nq <= 65535 && block_size > 0 && max_blocks > 0 && num_seqs >= 0,
               "near attention: %d query heads over %d key heads, block size %d, %d blocks a row", nq, nkv, block_size, max_blocks);
    PL_REQUIRE((q_gain == nullptr) == (k_gain == nullptr) && (cos_table == nullptr) == (sin_table == nullptr), "near attention: one of the two gains or tables is missing");
    PL_REQUIRE((reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(k_pool) | reinterpret_cast<uintptr_t>(v_pool) |
                reinterpret_cast<uintptr_t>(cos_table) | reinterpret_cast<uintptr_t>(sin_table) | reinterpret_cast<uintptr_t>(q_gain) | reinterpret_cast<uintptr_t>(k_gain)) % 16 == 0, "near attention: rows that are not aligned to 16 bytes");
    if (num_seqs == 0) return 0;
    constexpr int lds = 2 * AN_KEYS * 256 + AN_D * AN_V_PITCH;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attention_near_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    PL_REQUIRE(e == hipSuccess, "near attention: %d bytes of LDS refused: %s", lds, hipGetErrorString(e));
    attention_near_kernel<<<dim3(num_seqs, nq), 512, lds, stream>>>(
        static_cast<const bf16_t*>(qkv), static_cast<bf16_t*>(out), q_gain, k_gain, gain_dtype, eps, cos_table, sin_table, q_start, q_len, ctx_len,
        block_table, max_blocks, block_size, static_cast<bf16_t*>(k_pool), static_cast<bf16_t*>(v_pool), nq, nkv, scale);
    PL_CHECK_LAUNCH("attention_near");
    return 0;
}
