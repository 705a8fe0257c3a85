// The key pass of the two-pass backward over one strip of leaf key blocks.
// Included into the kernel's body and into that of the second walk (hsa_attn_bwd_tile.h) with `p`, `unit`, `lane`,
// `lds` and ODD defined.  (Text and not a function: inlined from a function the widest variants get
// other registers and spill more, B2 N2048 H8 D128 R64 74 -> 79 us for both passes.)
    using BT = BwdTile<T, D, DC>;
    constexpr bool PART = DC > 0;
    const int dh = PART ? p.dh : D;
    using M_ = Mma<T>;
    constexpr int KS = BT::KS, NJ = BT::NJ, RPI = BT::RPI, NLD = BT::NLD;
    constexpr int NQB = CAUSAL ? NBW + 1 : 2 * NBW + 1;  // query blocks that reach a key block
    constexpr int QOFF = CAUSAL ? 0 : -NBW;              // first of them, relative to the key block
    float odd_scores = 0.f;
    BT bt;
    bt.init(lds, lane);
    const int r16 = bt.r16, g = bt.g, lrow = bt.lrow, lchk = bt.lchk;

    const int N = p.N, R = p.R, H = p.H;
    const int NB = N / TILE_Q, NS = NB / SB;
    const int h = unit % H;
    const int strip = (unit / H) % NS;
    const int b = unit / (H * NS);
    const int kb0 = strip * SB;
    const size_t rs = (size_t)H * dh;
    const int pchk = PART ? min(lchk, dh / 8 - 1) : lchk;  // the piece this lane fetches
    const bool own_piece = !PART || 8 * lchk < dh;         // the piece exists: this lane stores it
    const uint16_t *Qb = p.q + ((size_t)b * N * H + h) * dh + 8 * pchk;
    const uint16_t *Gb = p.dout + ((size_t)b * N * H + h) * dh + 8 * pchk;
    const uint16_t *Kb = p.k + ((size_t)b * p.M * H + h) * dh + 8 * pchk;
    const uint16_t *Vb = p.v + ((size_t)b * p.M * H + h) * dh + 8 * pchk;

    auto load_block = [&](const uint16_t *base, int row0, u32x4_t (&dst)[NLD]) {
        const uint16_t *ptr = base + (size_t)(row0 + lrow) * rs;
#pragma unroll
        for (int i = 0; i < NLD; ++i) dst[i] = *reinterpret_cast<const u32x4_t *>(ptr + (size_t)(i * RPI) * rs);
    };
    auto clampb = [&](int qb) { return qb < 0 ? 0 : (qb >= NB ? NB - 1 : qb); };
    // a query block in the forms the key pass needs
    struct QBlock {
        u32x4_t Qf[KS], Gf[KS];
        u32x2_t QT[NJ], GT[NJ];
        float lse4[4], del4[4];
        uint32_t odd_g;  // rows of dO with an infinity or a NaN
    };
    struct Stage {
        u32x4_t k[NLD], v[NLD], q[NLD], g[NLD];
        float lse4[4], del4[4];
    };
    auto request = [&](Stage &sg, int kb) {  // key block kb and the query block that enters with it
        load_block(Kb, kb * TILE_Q, sg.k);
        load_block(Vb, kb * TILE_Q, sg.v);
        const int qb = clampb(kb + QOFF + NQB - 1);
        load_block(Qb, qb * TILE_Q, sg.q);
        load_block(Gb, qb * TILE_Q, sg.g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float *stp = p.stats + (((size_t)b * N + qb * TILE_Q + 4 * g + i) * H + h) * 2;
            sg.lse4[i] = stp[0];
            sg.del4[i] = stp[1];
        }
    };
    auto absorb = [&](QBlock &qq, const u32x4_t (&rq)[NLD], const u32x4_t (&rg)[NLD], const float (&l4)[4],
                      const float (&d4)[4]) {
        bt.put(2, rq);
        bt.put(3, rg);
        bt.get(2, qq.Qf);
        bt.get(3, qq.Gf);
        if constexpr (PART) {
            bt.clear_behind(qq.Qf, dh);
            bt.clear_behind(qq.Gf, dh);
        }
        bt.transpose(qq.Qf, qq.QT);
        bt.transpose(qq.Gf, qq.GT);
        if constexpr (ODD) {
            qq.odd_g = bt.odd_rows(qq.Gf);
            if (const uint32_t odd_q = bt.odd_rows(qq.Qf)) bt.clear_rows(qq.QT, odd_q);
            if (qq.odd_g) bt.clear_rows(qq.GT, qq.odd_g);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            qq.lse4[i] = l4[i];
            qq.del4[i] = d4[i];
            // (a query of this block may have met an infinity in another strip)
            if constexpr (PART && !ODD) odd_scores = fmaf(l4[i], 0.f, fmaf(d4[i], 0.f, odd_scores));
        }
    };

    QBlock qblk[NQB];
    Stage st[SB];
    {
        // the query blocks carried into the first key block, then the first stage
        u32x4_t rq[NQB][NLD], rg[NQB][NLD];
        float l4[NQB][4], d4[NQB][4];
#pragma unroll
        for (int c = 0; c + 1 < NQB; ++c) {
            const int qb = clampb(kb0 + QOFF + c);
            load_block(Qb, qb * TILE_Q, rq[c]);
            load_block(Gb, qb * TILE_Q, rg[c]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float *stp = p.stats + (((size_t)b * N + qb * TILE_Q + 4 * g + i) * H + h) * 2;
                l4[c][i] = stp[0];
                d4[c][i] = stp[1];
            }
        }
        request(st[0], kb0);
#pragma unroll
        for (int c = 0; c + 1 < NQB; ++c) absorb(qblk[c], rq[c], rg[c], l4[c], d4[c]);
    }

#pragma unroll
    for (int it = 0; it < SB; ++it) {
        const int kb = kb0 + it;
        const int k0 = kb * TILE_Q;
        Stage &sg = st[it];
        u32x4_t Kf[KS], Vf[KS];
        bt.put(0, sg.k);
        bt.put(1, sg.v);
        bt.get(0, Kf);
        bt.get(1, Vf);
        if constexpr (ODD) {
            bt.clear_behind(Kf, dh);
            bt.clear_behind(Vf, dh);
        }
        absorb(qblk[NQB - 1], sg.q, sg.g, sg.lse4, sg.del4);
        if (it + 1 < SB) request(st[it + 1 < SB ? it + 1 : it], kb + 1);

        f32x4 tk[NJ], tv[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) { tk[j] = f32x4{0.f, 0.f, 0.f, 0.f}; tv[j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
#pragma unroll
        for (int c = 0; c < NQB; ++c) {
            const int qb = kb + QOFF + c;
            const bool inside = qb >= 0 && qb < NB;  // uniform
            const QBlock &qq = qblk[c];
            f32x4 a = {0.f, 0.f, 0.f, 0.f}, d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                a = M_::k32(qq.Qf[ks], Kf[ks], a);  // S[query 4g+i of block qb, key r16]
                d = M_::k32(qq.Gf[ks], Vf[ks], d);
            }
            float pp[4], ds[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int ql = 4 * g + i;
                const int diff = (kb - qb) * TILE_Q + r16 - ql;  // key - query
                const bool win = diff >= -R && diff <= (CAUSAL ? 0 : R);
                const bool sib = qb == kb && r16 == (ql ^ 1) && (!CAUSAL || (ql & 1));
                const int cnt = (int)win + (int)sib;
                const float bias = (!inside || cnt == 0) ? NEG_INF : (cnt == 2 ? 1.0f : 0.0f);
                pp[i] = __builtin_amdgcn_exp2f(fmaf(a[i], p.scale_log2e, bias) - qq.lse4[i]);
                ds[i] = pp[i] * (d[i] - qq.del4[i]) * p.scale;
                if constexpr (PART && !ODD) odd_scores = fmaf(a[i], 0.f, fmaf(d[i], 0.f, odd_scores));
                if (ODD) bt.settle(bias == NEG_INF, qq.odd_g, i, pp[i], ds[i]);
            }
            if constexpr (PART && !ODD) asm volatile("" : "+v"(odd_scores));
            typename BT::W pk, dk;
            pk.set(pp);
            dk.set(ds);
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                tk[j] = dk.product(qq.QT[j], tk[j]);
                tv[j] = pk.product(qq.GT[j], tv[j]);
            }
        }
        bt.put_result(0, tk, 1.0f);
        bt.put_result(1, tv, 1.0f);
        uint16_t *dKp = p.dk + ((size_t)b * p.M * H + h) * dh + 8 * pchk + (size_t)(k0 + lrow) * rs;
        uint16_t *dVp = p.dv + ((size_t)b * p.M * H + h) * dh + 8 * pchk + (size_t)(k0 + lrow) * rs;
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            if (!own_piece) continue;
            *reinterpret_cast<u32x4_t *>(dKp + (size_t)(i * RPI) * rs) = bt.get_row_piece(0, i);
            *reinterpret_cast<u32x4_t *>(dVp + (size_t)(i * RPI) * rs) = bt.get_row_piece(1, i);
        }
        // slide the query blocks by one
#pragma unroll
        for (int c = 0; c + 1 < NQB; ++c) qblk[c] = qblk[c + 1];
    }
