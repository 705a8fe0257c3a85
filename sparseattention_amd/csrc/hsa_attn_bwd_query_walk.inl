// The query pass of the two-pass backward over one strip.
// Included into the kernel's body and into that of the second walk (hsa_attn_bwd_tile.h) with `p`, `unit`, `lane`,
// `lds`, `carry` and ODD defined.  (Text and not a function: inlined from a function the widest variants get
// other registers and spill more, B2 N2048 H8 D128 R64 74 -> 79 us for both passes.)
    using BT = BwdTile<T, D, DC>;
    constexpr bool PART = DC > 0;
    using M_ = Mma<T>;
    constexpr int KS = BT::KS, NJ = BT::NJ, RPI = BT::RPI, NLD = BT::NLD;
    constexpr int NKL = CAUSAL ? NBW + 1 : 2 * NBW + 1;
    constexpr int NKB = NKL + 2;  // leaf blocks, near tree block, far tree block
    float odd_scores = 0.f;       // part heads: NaN once a score or a product with dO is not finite
    BT bt;
    bt.init(lds, lane);
    const int r16 = bt.r16, g = bt.g, lrow = bt.lrow, lchk = bt.lchk;

    const int N = p.N, L = p.L, R = p.R, H = p.H;
    const int NB = N / TILE_Q, NS = NB / SB;
    const int h = unit % H;
    const int strip = (unit / H) % NS;
    const int b = unit / (H * NS);
    const int blk0 = strip * SB;
    const int qs = blk0 * TILE_Q;  // first query of the strip
    const int dh = PART ? p.dh : D;
    const size_t rs = (size_t)H * dh;
    const int pchk = PART ? min(lchk, dh / 8 - 1) : lchk;  // the piece this lane fetches
    const bool own_piece = !PART || 8 * lchk < dh;         // the piece exists: this lane stores it
    const uint16_t *Qb = p.q + ((size_t)b * N * H + h) * dh + 8 * pchk;
    const uint16_t *Gb = p.dout + ((size_t)b * N * H + h) * dh + 8 * pchk;
    const uint16_t *Kb = p.k + ((size_t)b * p.M * H + h) * dh + 8 * pchk;
    const uint16_t *Vb = p.v + ((size_t)b * p.M * H + h) * dh + 8 * pchk;
    uint16_t *dKb = p.dk + ((size_t)b * p.M * H + h) * dh + 8 * pchk;
    uint16_t *dVb = p.dv + ((size_t)b * p.M * H + h) * dh + 8 * pchk;

    // ---- tree slot constants (same slot layout as the forward kernel) -------------------------
    int t_lvl[NLD], t_add[NLD], t_xor[NLD], u_row[NLD];  // rows this lane fetches; u_row -1 = no such slot
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int sl = i * RPI + lrow;
        if (sl < 8) { t_lvl[i] = 1; t_add[i] = sl; t_xor[i] = 0; }
        else if (sl < 12) { t_lvl[i] = 2; t_add[i] = sl - 8; t_xor[i] = 0; }
        else if (sl < 14) { t_lvl[i] = 3; t_add[i] = sl - 12; t_xor[i] = 0; }
        else { t_lvl[i] = 4 + (sl - 14); t_add[i] = 0; t_xor[i] = 1; }
        const int ul = 6 + sl;
        u_row[i] = ul < L ? level_offset(N, ul) + ((qs >> ul) ^ 1) : -1;
    }
    auto near_row = [&](int i, int q0) {  // -1 = the slot's level does not exist
        return t_lvl[i] < L ? level_offset(N, t_lvl[i]) + (((q0 >> t_lvl[i]) + t_add[i]) ^ t_xor[i]) : -1;
    };
    auto slot_level = [](int sl, int &pl) {  // near slot -> level, position under the ancestor (-1: sibling slot)
        if (sl < 8) { pl = sl; return 1; }
        if (sl < 12) { pl = sl - 8; return 2; }
        if (sl < 14) { pl = sl - 12; return 3; }
        pl = -1;
        return 4 + (sl - 14);
    };
    // far block liveness in orientation 1 (lane = query r16, regs = slots 4g+i) and orientation 2
    // (lane = slot r16, regs = queries 4g+i): the same for every block of the strip
    float b1U[4], b2U[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int ul1 = 6 + 4 * g + i;
        b1U[i] = (ul1 < L && (!CAUSAL || ((qs >> ul1) & 1))) ? 0.f : NEG_INF;
        const int ul2 = 6 + r16;
        b2U[i] = (ul2 < L && (!CAUSAL || ((qs >> ul2) & 1))) ? 0.f : NEG_INF;
    }

    // ---- loads ------------------------------------------------------------------------------
    auto load_block = [&](const uint16_t *base, int row0, u32x4_t (&dst)[NLD]) {
        const uint16_t *ptr = base + (size_t)(row0 + lrow) * rs;
#pragma unroll
        for (int i = 0; i < NLD; ++i) dst[i] = *reinterpret_cast<const u32x4_t *>(ptr + (size_t)(i * RPI) * rs);
    };
    auto leaf_row0 = [&](int kb) {
        kb = kb < 0 ? 0 : (kb >= NB ? NB - 1 : kb);
        return kb * TILE_Q;
    };
    struct Stage {
        u32x4_t q[NLD], g[NLD], k[NLD], v[NLD], kt[NLD], vt[NLD];
    };
    auto request = [&](Stage &sg, int blk) {
        const int q0 = blk * TILE_Q;
        load_block(Qb, q0, sg.q);
        load_block(Gb, q0, sg.g);
        const int row0 = leaf_row0(blk - NBW + NKL - 1);  // the leaf block that enters with this query block
        load_block(Kb, row0, sg.k);
        load_block(Vb, row0, sg.v);
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int tr = near_row(i, q0);
            sg.kt[i] = *reinterpret_cast<const u32x4_t *>(Kb + (size_t)(tr < 0 ? q0 : tr) * rs);
            sg.vt[i] = *reinterpret_cast<const u32x4_t *>(Vb + (size_t)(tr < 0 ? q0 : tr) * rs);
        }
    };

    // everything the first block needs is requested before anything is consumed
    u32x4_t Kc[NKB][KS], Vc[NKB][KS];
    uint32_t odd_keys[ODD ? NKB : 1];
    Stage sg;
    {
        u32x4_t rKu[NLD], rVu[NLD], rKh[NKL][NLD], rVh[NKL][NLD];
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            rKu[i] = *reinterpret_cast<const u32x4_t *>(Kb + (size_t)(u_row[i] < 0 ? qs : u_row[i]) * rs);
            rVu[i] = *reinterpret_cast<const u32x4_t *>(Vb + (size_t)(u_row[i] < 0 ? qs : u_row[i]) * rs);
        }
#pragma unroll
        for (int c = 0; c + 1 < NKL; ++c) {
            load_block(Kb, leaf_row0(blk0 - NBW + c), rKh[c]);
            load_block(Vb, leaf_row0(blk0 - NBW + c), rVh[c]);
        }
        request(sg, blk0);
        bt.put(2, rKu);
        bt.put(3, rVu);
        bt.get(2, Kc[NKL + 1]);
        bt.get(3, Vc[NKL + 1]);
        if constexpr (ODD) odd_keys[NKL + 1] = bt.odd_keys(Kc[NKL + 1], Vc[NKL + 1], dh);
#pragma unroll
        for (int c = 0; c + 1 < NKL; ++c) {
            bt.put(2, rKh[c]);
            bt.put(3, rVh[c]);
            bt.get(2, Kc[c]);
            bt.get(3, Vc[c]);
            if constexpr (ODD) odd_keys[c] = bt.odd_keys(Kc[c], Vc[c], dh);
        }
    }
    // partial rows of the far block, summed over the strip
    f32x4 fk[NJ], fv[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) { fk[j] = f32x4{0.f, 0.f, 0.f, 0.f}; fv[j] = f32x4{0.f, 0.f, 0.f, 0.f}; }

#pragma unroll
    for (int it = 0; it < SB; ++it) {
        const int blk = blk0 + it;
        const int q0 = blk * TILE_Q;
        if (it > 0) request(sg, blk);
        // rows -> operand pieces
        u32x4_t Qf[KS], Gf[KS];
        bt.put(0, sg.q);
        bt.put(1, sg.g);
        bt.put(2, sg.k);
        bt.put(3, sg.v);
        bt.get(0, Qf);
        bt.get(1, Gf);
        uint32_t odd_q = 0, odd_g = 0;
        if constexpr (PART) {
            bt.clear_behind(Qf, dh);
            bt.clear_behind(Gf, dh);
        }
        if constexpr (ODD) {
            odd_q = bt.odd_rows(Qf);
            odd_g = bt.odd_rows(Gf);
        }
        bt.get(2, Kc[NKL - 1]);
        bt.get(3, Vc[NKL - 1]);
        if constexpr (ODD) odd_keys[NKL - 1] = bt.odd_keys(Kc[NKL - 1], Vc[NKL - 1], dh);
        bt.put(2, sg.kt);
        bt.put(3, sg.vt);
        bt.get(2, Kc[NKL]);
        bt.get(3, Vc[NKL]);
        if constexpr (ODD) odd_keys[NKL] = bt.odd_keys(Kc[NKL], Vc[NKL], dh);

        // liveness of the near block and of the leaf blocks for this query block
        int t_row[NLD];
#pragma unroll
        for (int i = 0; i < NLD; ++i) t_row[i] = near_row(i, q0);
        float b1T[4], b2T[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            {
                int pl;
                const int lvl = slot_level(4 * g + i, pl);
                const bool live = pl >= 0 ? (pl == ((r16 >> lvl) ^ 1) && (!CAUSAL || ((r16 >> lvl) & 1)))
                                          : (lvl < L && (!CAUSAL || ((q0 >> lvl) & 1)));
                b1T[i] = live ? 0.f : NEG_INF;
            }
            {
                int pl;
                const int lvl = slot_level(r16, pl);
                const int ql = 4 * g + i;
                const bool live = pl >= 0 ? (pl == ((ql >> lvl) ^ 1) && (!CAUSAL || ((ql >> lvl) & 1)))
                                          : (lvl < L && (!CAUSAL || ((q0 >> lvl) & 1)));
                b2T[i] = live ? 0.f : NEG_INF;
            }
        }
        float biasL[NKL][4];
#pragma unroll
        for (int c = 0; c < NKL; ++c) {
            const int dlt = TILE_Q * (c - NBW);
            const int kb = blk - NBW + c;
            const bool inside = kb >= 0 && kb < NB;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int kl = 4 * g + i;
                const int diff = dlt + kl - r16;
                const bool win = diff >= -R && diff <= (CAUSAL ? 0 : R);
                const bool sib = dlt == 0 && kl == (r16 ^ 1) && (!CAUSAL || (r16 & 1));
                const int cnt = (int)win + (int)sib;
                biasL[c][i] = (!inside || cnt == 0) ? NEG_INF : (cnt == 2 ? 1.0f : 0.0f);
            }
        }

        // ---- orientation 1: S^T, dP^T [key, query] ---------------------------------------------------
        float sc[NKB][4], dp[NKB][4];
        float mx = NEG_INF;
#pragma unroll
        for (int c = 0; c < NKB; ++c) {
            f32x4 a = {0.f, 0.f, 0.f, 0.f}, d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                a = M_::k32(Kc[c][ks], Qf[ks], a);
                d = M_::k32(Vc[c][ks], Gf[ks], d);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float bias = c < NKL ? biasL[c < NKL ? c : 0][i] : (c == NKL ? b1T[i] : b1U[i]);
                sc[c][i] = fmaf(a[i], p.scale_log2e, bias);
                dp[c][i] = d[i];
                if constexpr (PART && !ODD) odd_scores = fmaf(a[i], 0.f, fmaf(d[i], 0.f, odd_scores));
                if (ODD && bias == NEG_INF) {
                    sc[c][i] = NEG_INF;
                    dp[c][i] = 0.f;
                }
                mx = fmaxf(mx, sc[c][i]);
            }
        }
        if constexpr (PART && !ODD) asm volatile("" : "+v"(odd_scores));  // summed here, not when registers are short
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        if constexpr (ODD) mx = fmaxf(mx, -3.0e38f);  // every key -inf: weights of zero
        float den = 0.f;
#pragma unroll
        for (int c = 0; c < NKB; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sc[c][i] = __builtin_amdgcn_exp2f(sc[c][i] - mx);
                den += sc[c][i];
            }
        den += __shfl_xor(den, 16, 64);
        den += __shfl_xor(den, 32, 64);
        if constexpr (ODD) den = fmaxf(den, 1.0e-5f);  // (also where it is NaN)
        const float inv = 1.0f / den;
        float delta = 0.f;
#pragma unroll
        for (int c = 0; c < NKB; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sc[c][i] *= inv;  // P
                delta = fmaf(sc[c][i], dp[c][i], delta);
            }
        delta += __shfl_xor(delta, 16, 64);
        delta += __shfl_xor(delta, 32, 64);
        const float lse = mx + __builtin_amdgcn_logf(den);  // log2 domain: P = exp2(s' - lse)
        if (g == 0) {
            float *stp = p.stats + (((size_t)b * N + q0 + r16) * H + h) * 2;
            stp[0] = lse;
            stp[1] = delta;
        }

        // ---- dQ^T = sum_c K_c^T . dS_c^T ---------------------------------------------------------------
        {
            f32x4 acc[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < NKB; ++c) {
                u32x2_t KT[NJ];
                bt.transpose(Kc[c], KT);
                if constexpr (ODD)
                    if (odd_keys[c]) bt.clear_rows(KT, odd_keys[c]);
                float ds[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) ds[i] = sc[c][i] * (dp[c][i] - delta) * p.scale;
                typename BT::W dsw;
                dsw.set(ds);
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[j] = dsw.product(KT[j], acc[j]);
            }
            bt.put_result(0, acc, 1.0f);
            uint16_t *optr = p.dq + ((size_t)b * N * H + h) * dh + 8 * pchk + (size_t)(q0 + lrow) * rs;
#pragma unroll
            for (int i = 0; i < NLD; ++i)
                if (own_piece) *reinterpret_cast<u32x4_t *>(optr + (size_t)(i * RPI) * rs) = bt.get_row_piece(0, i);
        }

        // ---- orientation 2 for the tree blocks: dK^T, dV^T [channel, slot] ------------------------------
        u32x2_t QT[NJ], GT[NJ];
        bt.transpose(Qf, QT);
        bt.transpose(Gf, GT);
        if constexpr (ODD) {
            if (odd_q) bt.clear_rows(QT, odd_q);
            if (odd_g) bt.clear_rows(GT, odd_g);
        }
        float lse4[4], del4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lse4[i] = __shfl(lse, 4 * g + i, 64);
            del4[i] = __shfl(delta, 4 * g + i, 64);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int c = NKL + t;
            f32x4 a = {0.f, 0.f, 0.f, 0.f}, d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                a = M_::k32(Qf[ks], Kc[c][ks], a);   // S[query 4g+i, slot r16]
                d = M_::k32(Gf[ks], Vc[c][ks], d);   // dP[query, slot]
            }
            float pp[4], ds[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float bias = t == 0 ? b2T[i] : b2U[i];
                pp[i] = __builtin_amdgcn_exp2f(fmaf(a[i], p.scale_log2e, bias) - lse4[i]);
                ds[i] = pp[i] * (d[i] - del4[i]) * p.scale;
                if (ODD) bt.settle(bias == NEG_INF, odd_g, i, pp[i], ds[i]);
            }
            typename BT::W pk, dk;
            pk.set(pp);
            dk.set(ds);
            if (t == 0) {
                f32x4 tk[NJ], tv[NJ];
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    f32x4 z = {0.f, 0.f, 0.f, 0.f};
                    tk[j] = dk.product(QT[j], z);
                    tv[j] = pk.product(GT[j], z);
                }
                // A level-5 node collects from the two blocks under its sibling.  In a strip both
                // are this wavefront's: the even block parks its row, the odd block adds it and
                // the sum is final.  A strip of one block stores a partial row instead.
                bool five_final = false;
                if constexpr (SB > 1) {
                    if (r16 == 15) {
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            const int ch = 32 * (j >> 1) + 8 * g + 4 * (j & 1);
                            if (it & 1) {
                                const f32x4 ck = *reinterpret_cast<const f32x4 *>(carry + ch);
                                const f32x4 cv = *reinterpret_cast<const f32x4 *>(carry + D + ch);
                                tk[j] += ck;
                                tv[j] += cv;
                            } else {
                                *reinterpret_cast<f32x4 *>(carry + ch) = tk[j];
                                *reinterpret_cast<f32x4 *>(carry + D + ch) = tv[j];
                            }
                        }
                    }
                    five_final = (it & 1) != 0;
                } else if (r16 == 15 && 5 < L) {
                    const size_t po = ((((size_t)b * NB + blk) * H + h) * 2 + 1) * dh;
                    float *pkp = p.partial + po;
                    float *pvp = p.partial + (size_t)p.B * NB * H * 2 * dh + po;
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        const int ch = 32 * (j >> 1) + 8 * g + 4 * (j & 1);
                        if (PART && ch >= dh) continue;
                        *reinterpret_cast<f32x4 *>(pkp + ch) = tk[j];
                        *reinterpret_cast<f32x4 *>(pvp + ch) = tv[j];
                    }
                }
                // slots 0..14 (levels 1..4) are attended from inside the block only: rows written
                // directly, and so is the finished level-5 row
                bt.put_result(0, tk, 1.0f);
                bt.put_result(1, tv, 1.0f);
#pragma unroll
                for (int i = 0; i < NLD; ++i) {
                    const int sl = i * RPI + lrow;
                    if ((sl < 15 || five_final) && t_row[i] >= 0 && own_piece) {
                        *reinterpret_cast<u32x4_t *>(dKb + (size_t)t_row[i] * rs) = bt.get_row_piece(0, i);
                        *reinterpret_cast<u32x4_t *>(dVb + (size_t)t_row[i] * rs) = bt.get_row_piece(1, i);
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    fk[j] = dk.product(QT[j], fk[j]);
                    fv[j] = pk.product(GT[j], fv[j]);
                }
            }
        }

        // slide the leaf window by one block
#pragma unroll
        for (int c = 0; c + 1 < NKL; ++c) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) { Kc[c][ks] = Kc[c + 1][ks]; Vc[c][ks] = Vc[c + 1][ks]; }
            if constexpr (ODD) odd_keys[c] = odd_keys[c + 1];
        }
    }

    // levels >= 6: the strip's partial rows
    {
        const int lvl = 6 + r16;
        const int LF = L - 6;
        if (lvl < L) {
            float *far = p.partial + 2 * (size_t)p.B * NB * H * 2 * dh;
            const size_t po = ((((size_t)b * NS + strip) * H + h) * LF + (lvl - 6)) * dh;
            float *pkp = far + po;
            float *pvp = far + (size_t)p.B * NS * H * LF * dh + po;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int ch = 32 * (j >> 1) + 8 * g + 4 * (j & 1);
                if (PART && ch >= dh) continue;
                *reinterpret_cast<f32x4 *>(pkp + ch) = fk[j];
                *reinterpret_cast<f32x4 *>(pvp + ch) = fv[j];
            }
        }
    }
