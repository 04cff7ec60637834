// The body of an FP64 stage kernel: one tile (included by stream_fp64.h in the
// kernels, which define FACE, C, HALO, GAUGE, the parameters and the LDS arrays).
{
    // (constant address space: scalar loads, so that every base is uniform)
    const auto *const tp = (const __attribute__((address_space(4))) Tile *)tiles + blockIdx.x;
    const auto *const bp = (const __attribute__((address_space(4))) DBlock *)blocks + tp->block;
    const Tile tl{tp->block, tp->q0, {tp->o[0], tp->o[1], tp->o[2]}, {tp->e[0], tp->e[1], tp->e[2]}, tp->lanetab,
                  HALO ? tp->stagetab_halo : tp->stagetab};
    const DBlock B{bp->offset, bp->q0, {bp->n[0], bp->n[1], bp->n[2]}, bp->bflag, {}, {}};
    StreamCtx<FACE, C, HALO, GAUGE> c;
    c.block = bp;
    c.s_tile = s_tile;
    c.s_dx = s_dx;
    c.s_dy = s_dy;
    c.s_keep = s_keep;
    c.K = (const __attribute__((address_space(4))) dgr::AxisConsts *)bconst + 3 * (size_t)tl.block;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        c.kc[a] = c.K[a].d1_60;
        c.kc[3 + a] = c.K[a].d2_180;
        c.kc[6 + a] = c.K[a].ko_pre;
    }
#pragma unroll
    for (int i = 0; i < 9; i++) asm volatile("" : "+s"(c.kc[i]));
    const int nx = B.n[0], ny = B.n[1], nz = B.n[2];
    const int ex = tl.e[0], ey = tl.e[1], ez = tl.e[2];
    c.ox = tl.o[0];
    c.oy = tl.o[1];
    c.oz = tl.o[2];
    c.ex1 = ex - 1;
    c.ey1 = ey - 1;
    c.ez1 = ez - 1;
    // tiles are at least 3 points deep along every axis of such a block, so a
    // point within 2 of a face lies in the tile that meets it
    const uint32_t bf = FACE ? B.bflag : 0u;
    c.lox = (bf & 1u) && c.ox == PW;
    c.hix = (bf & 2u) && c.ox + ex == nx - PW;
    c.loy = (bf & 4u) && c.oy == PW;
    c.hiy = (bf & 8u) && c.oy + ey == ny - PW;
    c.loz = (bf & 16u) && c.oz == PW;
    c.hiz = (bf & 32u) && c.oz + ez == nz - PW;
    c.boff0 = B.offset;
    c.boff = HALO ? 0 : B.offset;
    c.m = (uint32_t)((nx - 2 * PW) * (ny - 2 * PW) * (nz - 2 * PW));
    c.u0 = io.u0 + NV * B.q0;
    c.acc = io.acc + NV * B.q0;
    // (scalars by construction: a buffer whose base or size the compiler took for
    // a vector value would be accessed in a loop over its distinct values)
    auto uniform = [](bool on) {
        return (uint32_t)__builtin_amdgcn_readfirstlane(on ? (int)decltype(c)::ALL : 0);
    };
    c.from = io.stage == 3 ? c.acc : c.u0;
    c.first = io.stage == 0;
    c.n_from = uniform(io.stage > 0);
    c.n_acc = uniform(io.stage == 1 || io.stage == 2);
    c.n_u0 = uniform(io.stage == 0);
    c.n_next = uniform((uint32_t)io.stage < 3u);
    c.cacc = io.cacc;
    c.cnext = io.cnext;
    const int tid = threadIdx.x;
    c.tid = tid;
    // the pairs this thread stages; rows beyond a short tile's region read the
    // block's first points, and nobody reads those
    {
        constexpr int PASS = C::passes(HALO), CROSS = C::cross_passes(HALO);
#pragma unroll
        for (int q = 0; q < (PASS + 1) / 2; q++) c.spot[q] = 0;
#pragma unroll
        for (int q = 0; q < PASS; q++) {
            const uint32_t w = tabs[tl.stagetab + q * C::FT + tid];
            c.spot[q / 2] |= w << (16 * (q & 1));
            const int row = w / FRX, col = w - row * FRX, kk = row / RMAX, jj = row - kk * RMAX;
            const bool in_region = jj < ey + 2 * PW && kk < ez + 2 * PW;
            const int gi = c.ox - PW + col, gj = c.oy - PW + jj, gk = c.oz - PW + kk;
            if constexpr (HALO)
                c.goff[q] = (uint32_t)(halo_source(io.nbo + 27 * (size_t)tl.block, B, in_region, gi, gj, gk) * sizeof(double));
            else
                c.goff[q] = in_region ? (uint32_t)(gi + nx * (gj + ny * gk)) * (uint32_t)sizeof(double) : 0u;
        }
        c.goff_cross = (CROSS - 1) * C::FT + tid < C::cross(HALO) ? c.goff[CROSS - 1] : c.NOWHERE_AT_ALL;
    }
    c.template fetch_to<0, 2>();
    const int lt = tabs[tl.lanetab + tid];
    c.active = !(lt & LANE_SHADOW);
    const int p = lt & (LANE_SHADOW - 1);
    const int lx = p % ex, ly = (p / ex) % ey, lz = p / (ex * ey);
    c.at3 = lx | ly << 4 | lz << 8;
    c.cofs = (PW + lx) + FRX * (PW + ly) + FRXY * (PW + lz);
    const int ax = c.ox + lx, ay = c.oy + ly, az = c.oz + lz;
    c.li = c.active ? (uint32_t)(ax + nx * (ay + ny * az)) * (uint32_t)sizeof(double) : c.NOWHERE;
    c.lq = c.active ? ((uint32_t)tl.q0 + tabs[tl.lanetab + C::FT + tid]) * (uint32_t)sizeof(double) : c.NOWHERE;
    c.face = FACE && ((c.lox && lx == 0) || (c.hix && lx == ex - 1) || (c.loy && ly == 0) || (c.hiy && ly == ey - 1) ||
                      (c.loz && lz == 0) || (c.hiz && lz == ez - 1));
    // this thread's line: D_x rows first on the tile's z planes (all 13 of each),
    // then on its y rows of the other planes
    {
        c.x_wave = __builtin_amdgcn_readfirstlane(tid >> 6) < C::XWAVES;
        const int l = c.x_wave ? tid : tid - 64 * C::XWAVES;
        c.has_line = l < (c.x_wave ? C::XLINES : C::YLINES);
        if (c.x_wave) {
            const int o = l - RMAX * C::FZ, q = o / TMAX;
            const int kk = o < 0 ? PW + l / RMAX : q < PW ? q : q + C::FZ;
            const int jj = o < 0 ? l % RMAX : PW + o - TMAX * q;
            c.line = FRX * jj + FRXY * kk;
        } else {
            c.line = l % TMAX + FRXY * (l / TMAX);
        }
    }
    // sigma: sqrt(chi) * eps (rhs.cpp:356-360), or one number
    c.root = 1.0;
    c.eps_gauge = c.eps_other = io.prm.ko_sigma;
    if (io.prm.cako) {
        c.root = sqrt(c.template fld<1>());
        c.eps_gauge = io.prm.eps_gauge;
        c.eps_other = io.prm.eps_other;
    }
    asm volatile("" : "+s"(c.eps_gauge));
    asm volatile("" : "+s"(c.eps_other));
    if constexpr (FACE || GAUGE) {
        double x[3];
        c.coords(x);
        if constexpr (FACE) c.inv_r = inv_radius(x[0], x[1], x[2]);
        if constexpr (GAUGE) c.eta_v = io.prm.eta_func ? 0.0 : rit_eta(x[0], x[1], x[2], io.prm);
    }
    c.template bring<0>();
    __syncthreads();
    dgr::bssn_rhs_stream<GAUGE>(c);
}
