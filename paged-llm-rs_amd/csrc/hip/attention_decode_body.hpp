// The body of one workgroup's part of the attention of single tokens: included as text by the kernel of its own launch (attention_decode.hip) and by the
// stage of a chain (ad_attend in attention_decode.hpp), with their template arguments and parameters by the same names, AD_DONE(done) for a return
// and WAITS.  As a function that both call it costs the launch of its own 6 to 18 registers a lane (two heads, eight keys: 250 to 256 and 5 of the others,
// one workgroup a compute unit where two fitted; alone that does not show, with a second engine beside it eight tokens took 1,440 us where it was 1,390, with
// three more 2,290 where it was 2,020).
    const float* const sinks = extras.sinks;
    const float* const slopes = extras.slopes;
    constexpr int KPW = PL_WAVE / LPK;  // keys a wave handles with one load
    constexpr int ROUND = WV * KPW * U;
    // lds: [AD_PAGES_LDS] page numbers, then [WV][GT][2] running max and sum, [WV][GT][d] accumulators
    int* pages_lds = reinterpret_cast<int*>(lds);
    float* ml = lds + AD_PAGES_LDS;               // [WV][GT][2]
    float* accs = ml + WV * GT * 2;               // [WV][GT][d]

    int t = by;
    if (num_seqs > 0 && !ad_find_row(by, q_len, num_seqs, short_limit, t)) AD_DONE(true);
    const int pos = positions[t];
    if (pos < 0) AD_DONE(true);
    const int seq = seq_of[t];
    if (q_len && q_len[seq] >= short_limit) AD_DONE(true);  // a long portion: the tiled kernel's

    // (g = nq / nkv and splits_magic = ceil(2^32 / splits) come from the launch: a division by a number that the
    // kernel learns only when it runs is some thirty instructions, and these stood in front of its first loads)
    const int kvh = tiles == 1 ? bx : bx / tiles;
    const int tile = tiles == 1 ? 0 : bx % tiles;
    const int h0 = kvh * g + tile * GT;               // first query head of this workgroup
    const int heads = min(GT, g - tile * GT);         // how many of the GT are real
    const int split = bz;

    const int lane = threadIdx.x % PL_WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PL_WAVE);  // the same for the whole wave: kept scalar
    const int sub = lane / LPK;   // which of the wave's keys
    const int dl = lane % LPK;    // which 8 values of the head
    const bool d_ok = dl * 8 < d;
    const int at8 = min(dl * 8, d - 8);

    // the stretch of keys of this split, in whole rounds of the workgroup
    const int first = pl_first_visible(pos, window);
    const int limit = fuse.mode == 2 ? pos : pos + 1;   // the token's own key is not in the cache yet
    int kept = 0;
    if constexpr (EX == 2) kept = min(extras.more.keep, first);
    auto key_at = [&](int i) { return EX == 2 && i < first ? i - (first - kept) : i; };
    const int total = max(limit - (first - kept), 0);
    // ceil(total / splits): the high half of (total + splits - 1) * ceil(2^32 / splits), exact below 2^32 / splits
    const int share = splits == 1 ? total : static_cast<int>(__umulhi(static_cast<uint32_t>(total + splits - 1), splits_magic));
    const int per_split = pl_ceil_div(share, ROUND) * ROUND;
    const int s_begin = first - kept + split * per_split;
    const int s_end = min(limit, s_begin + per_split);
    const int rounds = s_end > s_begin ? pl_ceil_div(s_end - s_begin, ROUND) : 0;

    const int* table = block_table + static_cast<size_t>(seq) * max_blocks;
    const size_t row_stride = static_cast<size_t>(nkv) * d;
    const size_t head_off = static_cast<size_t>(kvh) * d + at8;
    // floor(2^32 / block_size): the high half of j * bs_magic is j / block_size or one less
    const uint32_t bs_magic = block_size == 1 ? 0xffffffffu : static_cast<uint32_t>(0x100000000ull / static_cast<uint32_t>(block_size));
    auto page_of = [&](int j, int& w) -> int {          // which entry of the table holds key j, and its place in the page
        int bi = static_cast<int>(__umulhi(static_cast<uint32_t>(j), bs_magic));
        w = j - bi * block_size;
        const int low = w >= block_size ? 1 : 0;        // the estimate is the quotient or one less
        w -= low * block_size;
        return bi + low;
    };

    // ---- everything that does not wait for anything but the position, asked for at once ----
    int unused;
    // (the pages of the stretch: those of its kept keys, then those of its keys in the window; without kept keys the latter alone)
    int kept_first = 0, kept_pages = 0;
    if constexpr (EX == 2) {
        if (rounds > 0 && s_begin < first) {
            kept_first = page_of(key_at(s_begin), unused);
            kept_pages = page_of(key_at(min(s_end, first) - 1), unused) - kept_first + 1;
        }
    }
    const bool in_window = rounds > 0 && (EX != 2 || s_end > first);
    const int page_first = in_window ? page_of(EX == 2 ? max(s_begin, first) : s_begin, unused) : 0;
    const int page_count = (in_window ? page_of(s_end - 1, unused) - page_first + 1 : 0) + kept_pages;
    const bool pages_in_lds = page_count <= AD_PAGES_LDS;
    int page_got[AD_PAGES_LDS / (64 * WV) > 0 ? AD_PAGES_LDS / (64 * WV) : 1];
    constexpr int PAGE_TURNS = AD_PAGES_LDS / (64 * WV) > 0 ? AD_PAGES_LDS / (64 * WV) : 1;
    if (pages_in_lds) {
#pragma unroll
        for (int i = 0; i < PAGE_TURNS; ++i) {
            const int e = static_cast<int>(threadIdx.x) + i * 64 * WV;
            const int ee = min(e, max(page_count - 1, 0));
            page_got[i] = table[EX == 2 && ee < kept_pages ? kept_first + ee : page_first + ee - kept_pages];
        }
    }
    u32x4 qraw[GT];
    auto head_at = [&](int hq) { return static_cast<size_t>(h0 + min(hq, heads - 1)) * d + at8; };
    if constexpr (!WAITS) {
#pragma unroll
        for (int hq = 0; hq < GT; ++hq) qraw[hq] = *reinterpret_cast<const u32x4*>(q + static_cast<size_t>(t) * q_stride + head_at(hq));
    }
    // the token's own key and value (taken raw from its row by the first wave of the last split), and its page
    const bool own = fuse.mode == 2 && split == splits - 1 && wave == 0;
    u32x4 own_k = {{0u, 0u, 0u, 0u}}, own_v = {{0u, 0u, 0u, 0u}};
    int own_page = -1, own_within = 0;
    if (own) {
        if constexpr (!WAITS) {
            const bf16_t* row = q + static_cast<size_t>(t) * q_stride;
            own_k = *reinterpret_cast<const u32x4*>(row + static_cast<size_t>(nq + kvh) * d + at8);
            own_v = *reinterpret_cast<const u32x4*>(row + static_cast<size_t>(nq + nkv + kvh) * d + at8);
        }
        own_page = table[page_of(pos, own_within)];
    }
    ad_prep_t prep_q, prep_k;
    if (fuse.mode != 0) {
        ad_load_prep(prep_q, fuse.q_gain, fuse, d, dl, pos);
        if (own) {
            prep_k = prep_q;                                   // the same angles
            if (fuse.k_gain) ad_load_gain8(fuse.k_gain, fuse.gain_dtype, at8, prep_k.gain);
        }
    }
    if (pages_in_lds) {
#pragma unroll
        for (int i = 0; i < PAGE_TURNS; ++i) {
            const int e = static_cast<int>(threadIdx.x) + i * 64 * WV;
            if (e < page_count) pages_lds[e] = page_got[i];
        }
        __syncthreads();
    }

    // ---- keys and values: a round is U keys a lane group, two rounds are in flight ----
    // (a round that holds kept keys is told apart once, for the whole workgroup: the others pay nothing for them)
    auto in_front = [&](int round) { return EX == 2 && s_begin + round * ROUND < first; };
    auto ask_of = [&](auto front, int round, u32x4* kk, u32x4* vv, bool* ok) {
        constexpr bool FRONT = decltype(front)::value;
        const int base = s_begin + round * ROUND + wave * KPW * U;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = base + u * KPW + sub;
            const bool in = j < s_end;
            int w;
            const int i = in ? j : s_begin;                             // a key that exists in any case
            // (behind the rounds in front, s_begin itself may be a kept key: the first key of the window stands in for it)
            const int bi = page_of(FRONT ? key_at(i) : (EX == 2 ? max(i, first) : i), w);
            const int page = pages_in_lds ? pages_lds[FRONT && i < first ? bi - kept_first : bi - page_first + kept_pages] : table[bi];
            ok[u] = in && page >= 0;
            const size_t off = (static_cast<size_t>(max(page, 0)) * block_size + w) * row_stride + head_off;
            kk[u] = *reinterpret_cast<const u32x4*>(k_pool + off);
            vv[u] = *reinterpret_cast<const u32x4*>(v_pool + off);
        }
    };
    auto ask = [&](int round, u32x4* kk, u32x4* vv, bool* ok) {
        if constexpr (EX == 2) {
            if (in_front(round)) {
                ask_of(ad_true_t{}, round, kk, vv, ok);
                return;
            }
        }
        ask_of(ad_false_t{}, round, kk, vv, ok);
    };
    // (WAITS: one round in flight, since the registers of two do not fit beside the rest of that launch; of the second a word of every line
    // is asked for, so that it is in L2 when its turn comes)
    u32x4 ka[U], va[U], kb[WAITS ? 1 : U], vb[WAITS ? 1 : U];
    bool oka[U], okb[WAITS ? 1 : U];
    if (rounds > 0) ask(0, ka, va, oka);
    if constexpr (!WAITS)
        if (rounds > 1) ask(1, kb, vb, okb);
    uint32_t touched[WAITS ? 2 * U : 1];
    if constexpr (WAITS) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            touched[2 * u] = touched[2 * u + 1] = 0;
            const int j = s_begin + ROUND + wave * KPW * U + u * KPW + sub;
            if (j < s_end) {
                int w;
                const int bi = page_of(j, w);
                const int page = pages_in_lds ? pages_lds[bi - page_first] : table[bi];
                const size_t off = (static_cast<size_t>(max(page, 0)) * block_size + w) * row_stride + head_off;
                touched[2 * u] = *reinterpret_cast<const uint32_t*>(k_pool + off);
                touched[2 * u + 1] = *reinterpret_cast<const uint32_t*>(v_pool + off);
            }
        }
    }

    if constexpr (WAITS) {
        // the rows of q, which another stage of the launch leaves past L2
        const __amdgpu_buffer_rsrc_t row = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(q) + static_cast<size_t>(t) * q_stride, 0, 2u * q_stride, 0x00027000);
        auto load = [&](size_t at) {
            return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(row, static_cast<uint32_t>(at) * 2, 0, cn_past_l2_t::value));
        };
        auto most = [](const u32x4& p) { return max(max(p.v[0], p.v[1]), max(p.v[2], p.v[3])); };
        bool there = false;
        for (int look = 0; look <= rows_of.looks; ++look) {
            asm volatile("" ::: "memory");
            uint32_t all = 0;
#pragma unroll
            for (int hq = 0; hq < GT; ++hq) {
                qraw[hq] = load(head_at(hq));
                all = max(all, most(qraw[hq]));
            }
            if (own) {
                own_k = load(static_cast<size_t>(nq + kvh) * d + at8);
                own_v = load(static_cast<size_t>(nq + nkv + kvh) * d + at8);
                all = max(all, max(most(own_k), most(own_v)));
            }
            there = !rows_of.asks || __all(all != PL_MISSING);
            if (there) break;
            __builtin_amdgcn_s_sleep(1);
        }
#pragma unroll
        for (int i = 0; i < 2 * U; ++i) asm volatile("" ::"v"(touched[i]));
        if (!there && lane == 0) *rows_of.late = 1;
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(*rows_of.late)) AD_DONE(false);
    }

    // ---- while they are on their way: the queries, and the token's own key ----
    // The queries stay bfloat16 pairs (as the stand-alone kernel would have stored them): a score is four
    // two-element dot products a lane, and the scale multiplies the sum.
    u32x4 qp[GT];
#pragma unroll
    for (int hq = 0; hq < GT; ++hq) {
        const bool real = hq < heads && d_ok;
        if (fuse.mode != 0) {
            float x[8];
            unpack8(qraw[hq], x);
            if (!real) {
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = 0.f;
            }
            ad_norm_rope8<LPK>(x, fuse.q_gain != nullptr, prep_q, fuse, d, dl);
#pragma unroll
            for (int w = 0; w < 4; ++w) qp[hq].v[w] = ad_pack2(x[2 * w], x[2 * w + 1]);
        } else {
#pragma unroll
            for (int w = 0; w < 4; ++w) qp[hq].v[w] = real ? qraw[hq].v[w] : 0u;
        }
    }
    // (a penalty on the distance, where the layer has one: slope_h (pos - j) leaves the score, in the exponent's unit)
    const bool tilted = EX && slopes != nullptr;
    float tilt[EX ? GT : 1];
    int round_now = 0;            // (EX) the round that `consume` is given, for the distance of its keys
    // a soft cap, in the exponent's unit: c tanh(s / c) = c (1 - 2 / (2^(2 log2(e) s / c) + 1))
    float cap_in = 0.f, cap_out = 0.f;
    if constexpr (EX == 2) {
        if (extras.more.cap > 0.f) {
            cap_in = 2.f / extras.more.cap;
            cap_out = extras.more.cap * 1.4426950408889634f;
        }
    }
    if constexpr (EX != 0) {
#pragma unroll
        for (int hq = 0; hq < GT; ++hq) tilt[hq] = tilted ? slopes[h0 + min(hq, heads - 1)] * 1.4426950408889634f : 0.f;
    }
    float m[GT], l[GT], acc[GT][8];
#pragma unroll
    for (int hq = 0; hq < GT; ++hq) {
        m[hq] = -INFINITY;
        l[hq] = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[hq][i] = 0.f;
    }
    if (own) {
        // normalised and rotated here, written into the cache by one workgroup, and the first thing that
        // the running state of one lane group holds
        float kf[8], vf[8];
        unpack8(own_k, kf);
        unpack8(own_v, vf);
        if (!d_ok) {
#pragma unroll
            for (int i = 0; i < 8; ++i) kf[i] = vf[i] = 0.f;
        }
        ad_norm_rope8<LPK>(kf, fuse.k_gain != nullptr, prep_k, fuse, d, dl);
        u32x4 own_kp;
#pragma unroll
        for (int w = 0; w < 4; ++w) own_kp.v[w] = ad_pack2(kf[2 * w], kf[2 * w + 1]);
        if (tile == 0 && sub == 0 && d_ok && own_page >= 0) {
            const size_t off = (static_cast<size_t>(own_page) * block_size + own_within) * row_stride + static_cast<size_t>(kvh) * d + dl * 8;
            *reinterpret_cast<u32x4*>(k_pool + off) = own_kp;
            *reinterpret_cast<u32x4*>(v_pool + off) = own_v;
        }
#pragma unroll
        for (int hq = 0; hq < GT; ++hq) {
            float dot = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) dot = ad_dot2(qp[hq].v[w], own_kp.v[w], dot);
            dot = key_sum<LPK>(dot) * scale_log2e;
            if (sub == 0 && own_page >= 0) {
                m[hq] = dot;
                l[hq] = 1.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[hq][i] = vf[i];
            }
        }
    }

    // A key that does not exist (or whose page the request no longer holds) gets a score of minus
    // infinity by selection, whatever its row holds; its value is cleared, since a probability of zero
    // times a value that is not finite would not be zero.  Lanes past the head's width hold zero queries.
    // Values are taken two keys at a time: element i of both keys in one word against both probabilities
    // (rounded to bfloat16, as the matrix-core kernels round them), one instruction an element and head.
    static_assert(U % 2 == 0, "values are taken two keys at a time");
    auto consume = [&](u32x4* kraw, u32x4* vraw, const bool* ok) {
        float s[U][GT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int hq = 0; hq < GT; ++hq) {
                float dot = 0.f;
#pragma unroll
                for (int w = 0; w < 4; ++w) dot = ad_dot2(qp[hq].v[w], kraw[u].v[w], dot);
                dot = key_sum<LPK>(dot) * scale_log2e;
                if constexpr (EX == 2) {
                    if (cap_out > 0.f) dot = cap_out - 2.f * cap_out * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(dot * cap_in) + 1.f);
                }
                if constexpr (EX != 0) {
                    if (tilted) {
                        int key = s_begin + round_now * ROUND + wave * KPW * U + u * KPW + sub;
                        if constexpr (EX == 2) {
                            if (in_front(round_now)) key = key_at(key);
                        }
                        dot = fmaf(-tilt[hq], static_cast<float>(pos - key), dot);
                    }
                }
                s[u][hq] = ok[u] ? dot : -INFINITY;
            }
            const uint32_t keep = ok[u] ? 0xffffffffu : 0u;
#pragma unroll
            for (int w = 0; w < 4; ++w) vraw[u].v[w] &= keep;
        }
        float p[U][GT], corr[GT];
#pragma unroll
        for (int hq = 0; hq < GT; ++hq) {
            float m_new = m[hq];
#pragma unroll
            for (int u = 0; u < U; ++u) m_new = fmaxf(m_new, s[u][hq]);
            const float m_use = m_new == -INFINITY ? 0.f : m_new;   // nothing seen yet by this lane group: all weights zero
            corr[hq] = exp2f(m[hq] - m_use);
            float psum = 0.f;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                p[u][hq] = exp2f(s[u][hq] - m_use);
                psum += p[u][hq];
            }
            l[hq] = l[hq] * corr[hq] + psum;
            m[hq] = m_new;
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[hq][i] *= corr[hq];
        }
#pragma unroll
        for (int u = 0; u < U; u += 2) {
            uint32_t pp[GT];
#pragma unroll
            for (int hq = 0; hq < GT; ++hq) pp[hq] = ad_pack2(p[u][hq], p[u + 1][hq]);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                // (bytes 0..3 of the selector's second operand, 4..7 of its first)
                const uint32_t even = __builtin_amdgcn_perm(vraw[u + 1].v[w], vraw[u].v[w], 0x05040100u);
                const uint32_t odd = __builtin_amdgcn_perm(vraw[u + 1].v[w], vraw[u].v[w], 0x07060302u);
#pragma unroll
                for (int hq = 0; hq < GT; ++hq) {
                    acc[hq][2 * w] = ad_dot2(even, pp[hq], acc[hq][2 * w]);
                    acc[hq][2 * w + 1] = ad_dot2(odd, pp[hq], acc[hq][2 * w + 1]);
                }
            }
        }
    };
    if constexpr (WAITS) {
        static_assert(EX == 0, "no extras beside a chain");
        for (int r = 0; r < rounds; ++r) {
            consume(ka, va, oka);
            if (r + 1 < rounds) ask(r + 1, ka, va, oka);
        }
    } else
    for (int r = 0; r < rounds; r += 2) {
        if constexpr (EX != 0) round_now = r;
        consume(ka, va, oka);
        if (r + 2 < rounds) ask(r + 2, ka, va, oka);
        if (r + 1 < rounds) {
            if constexpr (EX != 0) round_now = r + 1;
            consume(kb, vb, okb);
            if (r + 3 < rounds) ask(r + 3, kb, vb, okb);
        }
    }

    // merge the lane groups of a wave in registers, then the waves through LDS
#pragma unroll
    for (int off = LPK; off < PL_WAVE; off <<= 1) {
#pragma unroll
        for (int hq = 0; hq < GT; ++hq) {
            const float mo = __shfl_xor(m[hq], off, PL_WAVE), lo = __shfl_xor(l[hq], off, PL_WAVE);
            const float mn = fmaxf(m[hq], mo);
            const float ca = mn == -INFINITY ? 0.f : exp2f(m[hq] - mn), cb = mn == -INFINITY ? 0.f : exp2f(mo - mn);
            l[hq] = l[hq] * ca + lo * cb;
            m[hq] = mn;
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[hq][i] = acc[hq][i] * ca + __shfl_xor(acc[hq][i], off, PL_WAVE) * cb;
        }
    }
    if (sub == 0) {
#pragma unroll
        for (int hq = 0; hq < GT; ++hq) {
            if (dl == 0) {
                ml[(wave * GT + hq) * 2] = m[hq];
                ml[(wave * GT + hq) * 2 + 1] = l[hq];
            }
            if (d_ok) {
#pragma unroll
                for (int i = 0; i < 8; ++i) accs[(static_cast<size_t>(wave) * GT + hq) * d + dl * 8 + i] = acc[hq][i];
            }
        }
    }
    auto finish = [&](int h, int dd, float big, float sum, float a) {
        float opened = 1.f;
        if constexpr (EX == 2) {
            if (extras.more.gate != nullptr) opened = pl_head_gate(extras.more, t, h);
        }
        if constexpr (EX != 0) {
            if (sinks != nullptr) {
                // a sink: one more term of the denominator, unscaled, with no value behind it
                const float sk = sinks[h] * 1.4426950408889634f;
                const float top = fmaxf(big, sk);
                const float keep = big == -INFINITY ? 0.f : exp2f(big - top);
                sum = sum * keep + exp2f(sk - top);
                a *= keep;
            }
        }
        out[(static_cast<size_t>(t) * nq + h) * d + dd] = from_float<bf16_t>(sum > 0.f ? a / sum * opened : 0.f);
    };
    __syncthreads();
    for (int idx = threadIdx.x; idx < heads * d; idx += blockDim.x) {
        const int hq = idx / d, dd = idx % d;
        float mw[WV], big = -INFINITY;
#pragma unroll
        for (int w = 0; w < WV; ++w) {
            mw[w] = ml[(w * GT + hq) * 2];
            big = fmaxf(big, mw[w]);
        }
        float sum = 0.f, a = 0.f;
#pragma unroll
        for (int w = 0; w < WV; ++w) {
            const float wt = mw[w] == -INFINITY ? 0.f : exp2f(mw[w] - big);
            sum = fmaf(ml[(w * GT + hq) * 2 + 1], wt, sum);
            a = fmaf(accs[(static_cast<size_t>(w) * GT + hq) * d + dd], wt, a);
        }
        const int h = h0 + hq;
        if (splits == 1) {
            finish(h, dd, big, sum, a);
        } else {
            const size_t pi = (static_cast<size_t>(t) * nq + h) * splits + split;
            if (arrivals != nullptr) {
                pl_share(part_acc + pi * d + dd, a);
                if (dd == 0) {
                    pl_share(part_ml + pi * 2, big);
                    pl_share(part_ml + pi * 2 + 1, sum);
                }
            } else {
                part_acc[pi * d + dd] = a;
                if (dd == 0) {
                    part_ml[pi * 2] = big;
                    part_ml[pi * 2 + 1] = sum;
                }
            }
        }
    }
    if (splits == 1 || arrivals == nullptr) AD_DONE(true);
    // The last of the shares to arrive puts them together, in their order whichever it is.
    pl_shares_written();
    __syncthreads();
    if (threadIdx.x == 0) pages_lds[0] = pl_arrive(arrivals + static_cast<size_t>(t) * nq + h0, splits) ? 1 : 0;
    __syncthreads();
    if (pages_lds[0] == 0) AD_DONE(true);
    for (int idx = threadIdx.x; idx < heads * d; idx += blockDim.x) {
        const int hq = idx / d, dd = idx % d, h = h0 + hq;
        const size_t base = (static_cast<size_t>(t) * nq + h) * splits;
        float ms[AD_MERGE_AT_ONCE], ls[AD_MERGE_AT_ONCE], as[AD_MERGE_AT_ONCE];
#pragma unroll
        for (int i = 0; i < AD_MERGE_AT_ONCE; ++i) {
            const size_t at = base + min(i, splits - 1);
            ms[i] = pl_shared(part_ml + at * 2);
            ls[i] = pl_shared(part_ml + at * 2 + 1);
            as[i] = pl_shared(part_acc + at * d + dd);
        }
        float big = -INFINITY, sum = 0.f, a = 0.f;
#pragma unroll
        for (int i = 0; i < AD_MERGE_AT_ONCE; ++i) big = fmaxf(big, i < splits ? ms[i] : -INFINITY);
#pragma unroll
        for (int i = 0; i < AD_MERGE_AT_ONCE; ++i) {
            const float w = (i < splits && ms[i] != -INFINITY) ? exp2f(ms[i] - big) : 0.f;
            sum = fmaf(ls[i], w, sum);
            a = fmaf(as[i], w, a);
        }
        finish(h, dd, big, sum, a);
    }
