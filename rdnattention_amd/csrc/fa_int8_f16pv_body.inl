// Body of the fa_fwd_int8_f16pv kernels (fa_fwd_int8_f16pv.hip), included into
// each of them: as a device function that the kernels call, the whole-row-tile
// kernel was compiled to other code (228 registers, not 245) and measured up to
// 1.5 % slower on causal GQA S = 3000, D = 128.  In scope: D, VTOK, SCORES,
// MODE (see Int8Mode) and the parameters p.
    constexpr bool SPLIT = MODE == Int8Mode::kSplit || MODE == Int8Mode::kRowMax;
    constexpr bool ALT = MODE == Int8Mode::kAlternate;
    constexpr bool ROWMAX = MODE == Int8Mode::kRowMax;
    using C = I8Cfg<D>;
    // K (and V) chunks that one group stages, and per thread of it
    constexpr int TASK = ALT ? 2 * C::HALF_TASK : C::HALF_TASK;
    constexpr int CT = (TASK + 255) / 256;
    __shared__ __attribute__((aligned(16))) int8_t sKs[2 * C::TILE_K];
    __shared__ __attribute__((aligned(16))) _Float16 sVs[2 * C::TILE_V];
    __shared__ __attribute__((aligned(16))) float sks[2][kI8BN]; // K scale of each key of a tile
    __shared__ __attribute__((aligned(16))) float sbk[2][kI8BN]; // -kI8Bias * that scale
    __shared__ __attribute__((aligned(16))) _Float16 sO[kI8Waves * 32 * C::LDO];

    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const int l32 = lane & 31;
    const int g = lane >> 5;
    const int grp = wave >> 2;
    const int rw = ALT ? wave & 3 : wave; // wave by its rows
    const int ugrp = ALT ? __builtin_amdgcn_readfirstlane(grp) : 0;
    // kAlternate: every row's running maximum, and group B's (m, l)
    __shared__ float sm_max[ALT ? 128 : 1];
    __shared__ float2 sm_ml[ALT ? 128 : 1];
    const int gtid = tid & 255;

    // Persistent: this workgroup walks its share of the row tiles (one per
    // workgroup of a one-tile-per-workgroup grid, see persistent_item). Every
    // group passes the same barriers per tile and leaves a tile only after its
    // last LDS read of K/V, so the next tile's prologue may overwrite them;
    // each wave's sO slot is its own.
    auto run_tile = [&](const int wg) {
        int hg, rt, split = 0;
        wg_tile(wg, p.n_head_groups, SPLIT ? p.n_row_tiles * p.splits : p.n_row_tiles, p.hg_chunk, hg, rt);
        if constexpr (SPLIT) {
            split_row_tile(p.n_row_tiles, rt, split);
        }
        const int per_b = p.Hkv * p.groups_per_kv;
        const int b = hg / per_b;
        const int rem = hg - b * per_b;
        const int kvh = rem / p.groups_per_kv;
        const int sub = rem - kvh * p.groups_per_kv;
        const int h = kvh * p.ratio + sub * p.G + (rw % p.G);
        const int wg_q0 = rt * p.rows_per_wg;
        const int q0 = wg_q0 + (rw / p.G) * 32;
        const int q = q0 + l32;
        const bool wave_active = q0 < p.Sq;
        const int q_hi = min(q0 + 31, p.Sq - 1);
        const int Sk = p.mask.sk;

        const int8_t* qbase = p.q + b * p.q_sb + h * p.q_sh;
        const int8_t* kbase = p.k + b * p.k_sb + kvh * p.k_sh;
        const int8_t* vbase = p.v + b * p.v_sb + kvh * p.v_sh;
        _Float16* obase = p.o + b * p.o_sb + h * p.o_sh;
        const float* ksbase = p.ksv ? p.ksv + ((int64_t)b * p.Hkv + kvh) * Sk : nullptr;
        const float* vtbase = VTOK ? p.vtok + ((int64_t)b * p.Hkv + kvh) * Sk : nullptr;

        // Q^T operand: lane holds Q[q][32s + 16g .. +15]
        i4 qreg[C::NS];
        float qs = p.q_scale;
        {
            const bool valid = q < p.Sq;
            const int8_t* qrow = qbase + (int64_t)(valid ? q : 0) * p.q_ss;
#pragma unroll
            for (int s = 0; s < C::NS; s++) {
                qreg[s] = valid ? *reinterpret_cast<const i4*>(qrow + 32 * s + 16 * g) : i4{};
            }
            if (p.qsv != nullptr && valid) {
                qs = p.qsv[((int64_t)b * p.Hq + h) * p.Sq + q];
            }
        }
        // s_j = t_j * qc with t_j = S_j * ks_j.  When every lane's qc is positive
        // the row max is taken over t (one multiply per score saved); otherwise t
        // is first scaled by qc in place and qeff = 1.
        const float qc = qs * p.scale_log2e;
        const bool qpos = !wave_any(!(qc > 0.0f));
        const float qeff = qpos ? qc : 1.0f;

        const int wg_q_hi = min(wg_q0 + p.rows_per_wg, p.Sq) - 1;
        int klo, khi;
        visible_key_range(p.mask, wg_q0, wg_q_hi, klo, khi);
        int t_begin = 0, n = 0;
        if (khi >= klo) {
            t_begin = klo / kI8BN;
            n = khi / kI8BN + 1 - t_begin;
        }
        if constexpr (SPLIT) {
            split_key_tiles(p.splits, split, t_begin, n);
        }
        // key tile i of this wave's sequence of ng tiles
        const int ng = ALT ? (n + 1 - ugrp) / 2 : n;
        auto tile_at = [&](int i) { return ALT ? t_begin + 2 * i + ugrp : t_begin + i; };
        int row_lo, row_hi;
        row_key_bounds(p.mask, q, row_lo, row_hi);
        // class of key tile t_begin + i for this wave's rows (0 skip, 1 no mask, 2 masked)
        const TileClasses tcls = wave_active ? tile_classes<kI8BN>(p.mask, q0, q_hi) : TileClasses{1, 0, 1, 0};

        f16x oacc[C::NDT];
#pragma unroll
        for (int dt = 0; dt < C::NDT; dt++) {
            oacc[dt] = f16x{};
        }
        // m_run: the scheme's exact running max; m_ref: the lagging reference
        // O and l are kept relative to (m_ref <= m_run)
        float m_run = -INFINITY, m_ref = -INFINITY, l_run = 0.0f;
        if constexpr (SPLIT && !ROWMAX) {
            if (q < p.Sq) {
                m_run = earlier_max(p, split, ((int64_t)b * p.Hq + h) * p.Sq + q);
            }
        }
        const i16x bias16 = SCORES || ALT ? i16x{} : (i16x{} + __float_as_int(kI8Bias));
        f16x tsc[2]; // scores of the current tile, dequantised by ks (t = S * ks)
        tsc[0] = f16x{};
        tsc[1] = f16x{};
        h8 pb[4]; // P^T operands of the four 16-key groups: integers 0..127 in fp16
#pragma unroll
        for (int u = 0; u < 4; u++) {
            pb[u] = h8{};
        }
        int cls_prev = 0;

        // ---- staging (one group's 32 rows of K and V per pair; ks by group A)
        i4 kreg[CT], vreg[CT];
        uint32_t coff_k[CT], coff_v[CT];
        int clk[CT], clv[CT];
#pragma unroll
        for (int it = 0; it < CT; it++) {
            const int e = gtid + it * 256;
            const bool ok = TASK % 256 == 0 || e < TASK;
            const int row = (ALT ? 0 : 32 * grp) + (ok ? e / C::KCH : 0);
            const int ch = ok ? e - (e / C::KCH) * C::KCH : 0;
            coff_k[it] = (uint32_t)((int64_t)row * p.k_ss + 16 * ch);
            coff_v[it] = (uint32_t)((int64_t)row * p.v_ss + 16 * ch);
            clk[it] = ok ? row * C::LDK + 16 * ch : -1;
            clv[it] = ok ? row * C::LDV + 16 * ch : -1;
        }
        float ksreg = 0.0f;
        float vsreg[CT]; // VTOK: the scale of each staged V row
        auto load_pair = [&](int x) {
            const int tk = tile_at(x), tv = ALT ? tile_at(x - 1) : t_begin + x - 1;
            const auto rk = make_rsrc(kbase + (int64_t)tk * kI8BN * p.k_ss,
                                      x < ng ? tile_bytes<kI8BN>(Sk - tk * kI8BN, (uint32_t)p.k_ss, D) : 0u);
            const auto rv = make_rsrc(vbase + (int64_t)tv * kI8BN * p.v_ss,
                                      (!ROWMAX && x >= 1 && x <= ng) ? tile_bytes<kI8BN>(Sk - tv * kI8BN, (uint32_t)p.v_ss, D) : 0u);
#pragma unroll
            for (int it = 0; it < CT; it++) {
                if constexpr (ALT && TASK % 256 == 0) { // pass it: 256 / KCH rows further on
                    kreg[it] = buffer_load_i4(rk, coff_k[0], (uint32_t)(it * (256 / C::KCH) * p.k_ss));
                    vreg[it] = buffer_load_i4(rv, coff_v[0], (uint32_t)(it * (256 / C::KCH) * p.v_ss));
                } else {
                    kreg[it] = buffer_load_i4(rk, coff_k[it]);
                    vreg[it] = buffer_load_i4(rv, coff_v[it]);
                }
                if constexpr (VTOK) {
                    const int key = tv * kI8BN + (ALT ? 0 : 32 * grp) + (gtid + it * 256) / C::KCH;
                    vsreg[it] = (x >= 1 && x <= ng && key < Sk) ? vtbase[key] : 0.0f;
                }
            }
            if ((ALT || grp == 0) && gtid < kI8BN && x < ng) {
                const int key = tk * kI8BN + gtid;
                ksreg = (ksbase != nullptr && key < Sk) ? ksbase[key] : p.k_scale;
            }
        };
        auto store_pair = [&](int x) {
            int8_t* sK = sKs + (ALT ? ugrp : x & 1) * C::TILE_K;
            _Float16* sV = sVs + (ALT ? ugrp : (x - 1) & 1) * C::TILE_V;
#pragma unroll
            for (int it = 0; it < CT; it++) {
                if (TASK % 256 == 0 || clk[it] >= 0) {
                    if (x < ng) {
                        *reinterpret_cast<i4*>(&sK[clk[it]]) = kreg[it];
                    }
                    if (!ROWMAX && x >= 1 && x <= ng) {
                        h8 lo, hi;
                        if constexpr (VTOK) {
                            i8x16_to_h8x2_scaled(vreg[it], vsreg[it], lo, hi);
                        } else {
                            i8x16_to_h8x2(vreg[it], lo, hi);
                        }
                        *reinterpret_cast<h8*>(&sV[clv[it]]) = lo;
                        *reinterpret_cast<h8*>(&sV[clv[it] + 8]) = hi;
                    }
                }
            }
            if ((ALT || grp == 0) && gtid < kI8BN && x < ng) {
                // ks rounded to 22 significant bits (relative change <= 2^-23),
                // so that kI8Bias ks = 3 2^22 ks is exact in fp32 and the
                // dequantisation fma returns S ks rounded once
                const float ks22 = __uint_as_float((__float_as_uint(ksreg) + 2u) & ~3u);
                sks[ALT ? ugrp : x & 1][gtid] = ks22;
                sbk[ALT ? ugrp : x & 1][gtid] = -kI8Bias * ks22;
            }
        };

        // M(i): S(i)^T = K(i) Q^T (int8 MFMA, i < n) then O^T += V(i-1)^T P(i-1)^T
        // (fp16 MFMA, i >= 1): one stream of MFMAs whose LDS operands are read
        // kI8OpDepth MFMAs ahead through a register ring.  The dequantisation
        // of S(i) rides on the P V MFMAs: 8 groups of 4 scores, group u after
        // P V MFMA 2u + 1, its K scales and biases read at MFMA 2u (at head
        // dim 64, 8 P V MFMAs: group u after MFMA u).  (With the
        // P V MFMAs first it ran after the last Q K^T MFMA, on the phase's
        // critical path.)
        auto mfma_stream = [&](auto do_pv_c, auto do_s_c, int i) {
            constexpr bool DO_PV = decltype(do_pv_c)::value;
            constexpr bool DO_S = decltype(do_s_c)::value;
            constexpr bool DQ = DO_S && !SCORES;
            constexpr int NSK = DO_S ? 2 * C::NS : 0;   // (st, kt)
            constexpr int NPV = DO_PV ? 4 * C::NDT : 0; // (u, dt)
            static_assert(!DO_PV || NPV == 16 || NPV == 8, "8 dequantisation groups over the P V MFMAs");
            constexpr int T = NSK + NPV;
            // kAlternate holds twice the staged chunks in registers
            constexpr int OPS = !ALT ? kI8OpDepth : VTOK && D == 128 ? 2 : 4;
            constexpr int DEPTH = T < OPS ? T : OPS;
            const int j16 = lane & 15;
            const _Float16* vrow = sVs + (ALT ? ugrp : (i - 1) & 1) * C::TILE_V + (4 * g + (j16 >> 2)) * C::LDV +
                                   16 * ((lane >> 4) & 1) + 4 * (j16 & 3);
            const int8_t* krow = sKs + (ALT ? ugrp : i & 1) * C::TILE_K + l32 * C::LDK + 16 * g;
            auto op = [&](int j) -> i4 {
                if (j < NSK) {
                    const int st = j >> 1, kt = j & 1;
                    return *reinterpret_cast<const i4*>(krow + kt * 32 * C::LDK + 32 * st);
                }
                const int jp = j - NSK, u = jp / C::NDT, dt = jp % C::NDT;
                const _Float16* base = vrow + (16 * u) * C::LDV + 32 * dt;
                h4 lo = lds_read_tr16(base);
                h4 hi = lds_read_tr16(base + 8 * C::LDV);
                return __builtin_bit_cast(i4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            };
            // SCORES: the raw int32 sums.  Otherwise each chain starts at the bit
            // pattern of kI8Bias, so the int32 result is the fp32 number
            // kI8Bias + S (exact: |S| <= 127^2 D < 2^22, the ulp there is 1)
            const i16x start = SCORES || ALT ? i16x{} : bias16;
            i16x acc0 = {}, acc1 = {};
            // dequantisation group u (keys 32 kt + 8 r4 + 4 g .. +3, kt = u / 4,
            // r4 = u % 4), one fma per score: t = (kI8Bias + S) ks - kI8Bias ks,
            // both terms exact (ks has 22 significant bits)
            const float* ksl = sks[ALT ? ugrp : i & 1];
            const float* bkl = sbk[ALT ? ugrp : i & 1];
            f4 gks = {}, gbk = {};
            auto dq_load = [&](int u) {
                const int o = 32 * (u >> 2) + 8 * (u & 3) + 4 * g;
                gks = *reinterpret_cast<const f4*>(&ksl[o]);
                gbk = *reinterpret_cast<const f4*>(&bkl[o]);
            };
            auto dq_apply = [&](int u) {
                const int kt = u >> 2, r4 = u & 3;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int32_t sv = kt == 0 ? acc0[4 * r4 + e] : acc1[4 * r4 + e];
                    // kAlternate: from 0 and converted, the same value (16 registers fewer)
                    tsc[kt][4 * r4 + e] =
                        ALT ? (float)sv * gks[e] : fmaf(__int_as_float(sv), gks[e], gbk[e]);
                }
            };
            i4 ring[DEPTH > 0 ? DEPTH : 1];
#pragma unroll
            for (int j = 0; j < DEPTH; j++) {
                ring[j] = op(j);
            }
#pragma unroll
            for (int j = 0; j < T; j++) {
                const i4 a = ring[j % DEPTH];
                if (j + DEPTH < T) {
                    ring[j % DEPTH] = op(j + DEPTH);
                }
                if (j < NSK) {
                    const int st = j >> 1;
                    if (j & 1) {
                        acc1 = mfma_32x32x32_i8(a, qreg[st], st == 0 ? start : acc1);
                    } else {
                        acc0 = mfma_32x32x32_i8(a, qreg[st], st == 0 ? start : acc0);
                    }
                } else {
                    const int jp = j - NSK, u = jp / C::NDT, dt = jp % C::NDT;
                    oacc[dt] = mfma_32x32x16_f16(__builtin_bit_cast(h8, a), pb[u], oacc[dt]);
                    if constexpr (DQ && NPV == 16) {
                        if (jp & 1) {
                            dq_apply(jp >> 1);
                        } else {
                            dq_load(jp >> 1);
                        }
                    } else if constexpr (DQ) {
                        dq_load(jp);
                        dq_apply(jp);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (DO_S && SCORES) {
                // the two S^T blocks of this tile: lane holds query q, keys
                // kt0 + 32 kt + 8 (e / 4) + 4 g + e % 4
                if (q < p.Sq) {
                    const int kt0 = (t_begin + i) * kI8BN;
                    int32_t* srow = p.scores + (((int64_t)b * p.Hq + h) * p.Sq + q) * Sk;
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const int k0 = kt0 + 8 * (e >> 2) + 4 * g + (e & 3);
                        if (k0 < Sk) {
                            srow[k0] = acc0[e];
                        }
                        if (k0 + 32 < Sk) {
                            srow[k0 + 32] = acc1[e];
                        }
                    }
                }
            } else if constexpr (DQ && !DO_PV) {
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    dq_load(u);
                    dq_apply(u);
                }
            }
        };
        auto phase_m = [&](int i) {
            if (!wave_active) {
                return;
            }
            const bool do_pv = !SCORES && !ROWMAX && i >= 1 && cls_prev != 0;
            const int cls_now = i < ng ? tile_class(tcls, tile_at(i)) : 0;
            using T_ = std::true_type;
            using F_ = std::false_type;
            if (do_pv && cls_now != 0) {
                mfma_stream(T_{}, T_{}, i);
            } else if (do_pv) {
                mfma_stream(T_{}, F_{}, i);
            } else if (cls_now != 0) {
                mfma_stream(F_{}, T_{}, i);
            }
            cls_prev = cls_now;
        };

        // V(i): exact running max over the 64-key block, P as integers 0..127
        // times the reference factor f; O and l are rescaled only when the
        // reference moves
        auto phase_v = [&](int i) {
            if (SCORES || !wave_active || cls_prev == 0) {
                return;
            }
            f16x (&t)[2] = tsc; // in place: a copy cost 16 moves per tile
            if (!qpos) {
#pragma unroll
                for (int kt = 0; kt < 2; kt++) {
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        t[kt][e] *= qc;
                    }
                }
            }
            if (cls_prev == 2) {
                const int kt0 = tile_at(i) * kI8BN;
                const int a = row_lo - kt0 - 4 * g;
                const int bnd = row_hi - kt0 - 4 * g;
#pragma unroll
                for (int kt = 0; kt < 2; kt++) {
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const int off = kt * 32 + 8 * (e >> 2) + (e & 3);
                        t[kt][e] = (off < a || off > bnd) ? -INFINITY : t[kt][e];
                    }
                }
            }
            float mx = t[0][0];
#pragma unroll
            for (int e = 1; e < 16; e++) {
                mx = fmaxf(mx, t[0][e]);
            }
#pragma unroll
            for (int e = 0; e < 16; e++) {
                mx = fmaxf(mx, t[1][e]);
            }
            mx = pair_max(mx) * qeff; // qeff > 0: -inf stays -inf
            m_run = fmaxf(m_run, mx);
            if constexpr (ALT) { // the other group's tile just before this one
                m_run = fmaxf(m_run, sm_max[rw * 32 + l32]);
                if (g == 0) {
                    sm_max[rw * 32 + l32] = m_run;
                }
            }
            if constexpr (ROWMAX) {
                return;
            }
            const bool move = m_run > m_ref + kI8RefThreshold; // false while m_run = -inf
            if (wave_any(move)) {
                const float alpha = move ? fast_exp2(m_ref - m_run) : 1.0f; // m_ref = -inf -> 0
                if (move) {
                    m_ref = m_run;
                }
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < C::NDT; dt++) {
                    oacc[dt] *= alpha;
                }
            }
            // m_ref = -inf only while m_run = -inf (no visible key yet: every p is 0)
            const _Float16 f16 = (_Float16)(m_ref == -INFINITY ? 1.0f : fast_exp2(m_run - m_ref));
            const float c0 = int8_exp_offset(m_run);
            const h2 fv = {f16, f16};
            float psum = 0.0f;
#pragma unroll
            for (int kt = 0; kt < 2; kt++) {
#pragma unroll
                for (int e = 0; e < 16; e += 2) {
                    // y = 127 p (<= 127); h = fp16(1 + y 2^-10) = 1 + round(y) 2^-10
                    // (one v_fma_mix per score: [1, 2) has ulp 2^-10 in fp16),
                    // then h f - f = pq f 2^-10, rounded once (one packed fma)
                    const float y0 = fast_exp2(fmaf(t[kt][e], qeff, c0));
                    const float y1 = fast_exp2(fmaf(t[kt][e + 1], qeff, c0));
                    psum += y0;
                    psum += y1;
                    const h2 hq = {(_Float16)fmaf(y0, kI8PScale, 1.0f), (_Float16)fmaf(y1, kI8PScale, 1.0f)};
                    const h2 pq = hq * fv - fv;
                    pb[kt * 2 + (e >> 3)][e & 7] = pq[0];
                    pb[kt * 2 + (e >> 3)][(e & 7) + 1] = pq[1];
                }
            }
            l_run = fmaf(psum, (float)f16, l_run);
        };

        if (n > 0) {
            load_pair(0);
            store_pair(0);
            load_pair(1);
        }
        if (ALT && grp == 0 && g == 0) {
            sm_max[rw * 32 + l32] = -INFINITY;
        }
        __syncthreads();
        if constexpr (ALT) {
            const int n2 = (n + 1) / 2; // steps of group A
            if (n > 0) {
                if (ugrp == 1) {
                    __syncthreads();
                }
                for (int i = 0; i < n2; i++) {
                    phase_m(i);
                    __syncthreads();
                    store_pair(i + 1); // K(i) and V(i - 1) were read in M(i) the last time
                    load_pair(i + 2);
                    phase_v(i);
                    __syncthreads();
                }
                phase_m(n2);
                __syncthreads();
                if (ugrp == 0) {
                    __syncthreads();
                }
            }
        } else if (n > 0) {
            if (grp == 0) {
                for (int i = 0; i < n; i++) {
                    phase_m(i);
                    __syncthreads();
                    store_pair(i + 1);
                    load_pair(i + 2);
                    phase_v(i);
                    __syncthreads();
                }
                phase_m(n);
                __syncthreads();
                __syncthreads();
            } else {
                store_pair(1);
                load_pair(2);
                __syncthreads();
                for (int i = 0; i < n; i++) {
                    phase_m(i);
                    __syncthreads();
                    store_pair(i + 2);
                    load_pair(i + 3);
                    phase_v(i);
                    __syncthreads();
                }
                phase_m(n);
                __syncthreads();
            }
        }

        if (SCORES || (!ALT && !wave_active)) {
            return;
        }
        if constexpr (ROWMAX) {
            if (g == 0 && q < p.Sq) {
                p.row_max[split * p.n_rows + ((int64_t)b * p.Hq + h) * p.Sq + q] = m_run;
            }
            return;
        }
        // O = O^T * v_scale / l (times the per-channel V scales of this kv head
        // when given), through this wave's sO slot
        float l = pair_sum(l_run);
        if constexpr (ALT) {
            // group B's O (relative to its own maximum) into group A's, through
            // LDS that nothing else reads after the last barrier
            constexpr int LDM = D + 4;
            static_assert(4 * 32 * LDM * 4 <= sizeof(sO) && 4 * 32 * C::LDO * 2 <= sizeof(sVs), "O fits");
            float* const so = reinterpret_cast<float*>(sO) + (rw * 32 + l32) * LDM + 4 * g;
            if (ugrp == 1 && wave_active) {
#pragma unroll
                for (int dt = 0; dt < C::NDT; dt++) {
#pragma unroll
                    for (int qq = 0; qq < 4; qq++) {
                        *reinterpret_cast<f4*>(so + 32 * dt + 8 * qq) = f4{oacc[dt][4 * qq], oacc[dt][4 * qq + 1],
                                                                           oacc[dt][4 * qq + 2], oacc[dt][4 * qq + 3]};
                    }
                }
                if (g == 0) {
                    sm_ml[rw * 32 + l32] = float2{m_ref, l};
                }
            }
            __syncthreads();
            if (ugrp == 0 && wave_active) {
                const float2 other = sm_ml[rw * 32 + l32];
                const float m = fmaxf(l > 0.0f ? m_ref : -INFINITY, other.y > 0.0f ? other.x : -INFINITY);
                const float wa = l > 0.0f ? fast_exp2(m_ref - m) : 0.0f;
                const float wb = other.y > 0.0f ? fast_exp2(other.x - m) : 0.0f;
                l = l * wa + other.y * wb;
#pragma unroll
                for (int dt = 0; dt < C::NDT; dt++) {
#pragma unroll
                    for (int qq = 0; qq < 4; qq++) {
                        const f4 x = *reinterpret_cast<const f4*>(so + 32 * dt + 8 * qq);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            oacc[dt][4 * qq + e] = oacc[dt][4 * qq + e] * wa + x[e] * wb;
                        }
                    }
                }
                const float f = l > 0.0f ? p.v_scale / (l * kI8PScale) : 0.0f;
                const float* vch = p.vch != nullptr ? p.vch + ((int64_t)b * p.Hkv + kvh) * D : nullptr;
                store_o_tile<D, C::LDO>(
                    oacc,
                    [&](int d0) {
                        return vch != nullptr ? f * *reinterpret_cast<const f4*>(vch + d0) : f4{f, f, f, f};
                    },
                    sVs + rw * 32 * C::LDO, obase, q0, p.Sq, p.o_ss, lane);
            }
            __syncthreads(); // before the next row tile's staging
            return;
        }
        if constexpr (SPLIT) {
            const float* vch = p.vch != nullptr ? p.vch + ((int64_t)b * p.Hkv + kvh) * D : nullptr;
            if (q < p.Sq) {
                const int64_t row = split * p.n_rows + ((int64_t)b * p.Hq + h) * p.Sq + q;
                const float f = p.v_scale / kI8PScale;
                store_partial(oacc, m_ref, l, g == 0, p.part_o, p.part_ml, row, D, 0, g, [&](int d0) {
                    return vch != nullptr ? f * *reinterpret_cast<const f4*>(vch + d0) : f4{f, f, f, f};
                });
            }
            return;
        }
        const float f = l > 0.0f ? p.v_scale / (l * kI8PScale) : 0.0f;
        const float* vch = p.vch != nullptr ? p.vch + ((int64_t)b * p.Hkv + kvh) * D : nullptr;
        store_o_tile<D, C::LDO>(
            oacc,
            [&](int d0) {
                return vch != nullptr ? f * *reinterpret_cast<const f4*>(vch + d0) : f4{f, f, f, f};
            },
            sO + wave * 32 * C::LDO, obase, q0, p.Sq, p.o_ss, lane);
    };
    for (int item = 0;; item++) {
        const int wg = persistent_item(blockIdx.x, gridDim.x, item, p.n_items);
        if (wg < 0) {
            break;
        }
        run_tile(wg);
    }
