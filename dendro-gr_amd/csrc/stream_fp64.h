// The FP64 stage kernel: derivatives, equations, dissipation, boundary values
// and the Runge-Kutta stage update of one tile per workgroup, one point per
// thread, in the streaming order of bssn_rhs_stream.h (included by
// dgr_bssn.hip inside its namespace).
//
// Its live set (about 75 doubles) fits 256 registers, so a SIMD runs two waves
// and one wave's LDS and memory waits are the other's issue slots. Everything
// else follows from that budget:
//   * LDS: two region buffers, one D_x and one D_y plane set and eleven parked
//     values a thread: 79 KB for a 256-thread tile, two workgroups a CU. The
//     7-deep tile (384 threads, one workgroup a CU) has room for three buffers
//     and two sets, hence one barrier a phase;
//   * a right-hand side leaves the registers in the phase that completes it
//     (the stage update reads its inputs one phase ahead), so no 24-value
//     epilogue and no 49 KB of LDS for it;
//   * the point's addresses are 32-bit offsets from uniform bases, D_x / D_y
//     slots are packed in halves, the stencil constants sit in scalar registers.
// What bounds it: the L1's fills of the staged regions. A 7x7x5 tile reads 7.6
// values for each of its own, and with 8-byte loads of whole regions the texture
// address units were 84% busy while the vector units idled at 28%. So a
// region is read 16 bytes a lane, the corners no stencil reaches are left out,
// and the interior buffers lie in lane order (stage_table, StreamIO).
// Busy now, of a launch's cycles: 7x7x5 tiles (octree) the texture address units 76%,
// LDS 41%, the vector units 40%; 7x7x7 tiles 43-54%, 26-29% and 28-32%, their six waves
// on four SIMDs waiting 45% of their time (LDS, memory, the barrier); flagged tiles 24%,
// 22% and 31% on 288 KB of code, of which 3-4% of the fetches miss the 64 KB
// instruction cache (the others' 62 KB fit: 0.1%).
// Measured, a whole RK4 step with its padding copy, against the one-wave kernel
// this replaces (126 live doubles, 480 registers): 30.0 M points of uneven octree
// 95.6 -> 60.9 ms; 4096 blocks of 13^3 5.05 -> 3.57 ms (its stage alone 1.06 -> 0.77); the
// right-hand side of 200 ragged blocks, 28% of them flagged, 1.88 -> 0.99 ms;
// one 19^3 block with every face flagged 118 -> 83 us (1.12 ms and 115 us before
// D_x and D_y went along lines, SCfg::XLINES).

template <int FT_, int FZ_, bool DEEP_>
struct SCfg {
    static constexpr int FT = FT_;
    static constexpr int FZ = FZ_;
    // one barrier a phase: three region buffers and two D_x / D_y sets (below)
    static constexpr bool DEEP = DEEP_;
    static constexpr int NROW = RMAX * (FZ + 2 * PW);  // x rows of the staged region
    static constexpr int NBUF = FRX * NROW;
    // Staging: a thread reads two neighbouring doubles (16 bytes) of a row at a
    // time (stage_table). First what a variable without second derivatives
    // needs: NCROSS pairs, all of rows inside the tile along y and z and the
    // tile's own columns of rows outside along one of them; then what mixed
    // derivatives need besides: the rest of those rows, and the tile's columns
    // of rows outside along both. A row takes 7 pairs, or 8 with HALO, where no
    // pair may reach across the block's own first or last node.
    static constexpr int pairs(bool halo) { return halo ? 8 : 7; }
    static constexpr int NIN = TMAX * FZ, NONE = 2 * PW * (TMAX + FZ), NOUT = 4 * PW * PW;  // rows in, out once, out twice
    static constexpr int cross(bool halo) { return NIN * pairs(halo) + NONE * 4; }
    static constexpr int all(bool halo) { return cross(halo) + NONE * (pairs(halo) - 4) + NOUT * 4; }
    static constexpr int passes(bool halo) { return (all(halo) + FT - 1) / FT; }
    static constexpr int cross_passes(bool halo) { return (cross(halo) + FT - 1) / FT; }
    // D_x is evaluated along whole x rows of 7 points, D_y along whole y columns,
    // one a thread: D_y(D_x u) reads D_x on the tile's z planes (all region rows),
    // D_z(D_x u) on its y rows (all region planes). The first XWAVES waves take the
    // rows, the others the columns.
    static constexpr int XLINES = RMAX * FZ + TMAX * 2 * PW, YLINES = TMAX * (FZ + 2 * PW);
    static constexpr int XWAVES = (XLINES + 63) / 64;
    static_assert(YLINES <= FT - 64 * XWAVES, "a thread per line");
    static constexpr int NSDX = TMAX + FRX * (RMAX - 1) + FRXY * (FZ + 2 * PW - 1);
    static constexpr int NSDY = TMAX + FRX * (TMAX - 1) + FRXY * (FZ + 2 * PW - 1);
    static constexpr int RB = DEEP ? 3 : 2, DB = DEEP ? 2 : 1;
    static constexpr size_t LDS = sizeof(double) * (RB * NBUF + DB * (NSDX + NSDY) + dgr::kStreamKeep * FT);
};
using SWide = SCfg<CfgWide::FT, CfgWide::FZ, false>;
using SFull = SCfg<CfgFull::FT, CfgFull::FZ, true>;
static_assert(2 * SWide::LDS <= 160 * 1024, "two regular workgroups per CU");
static_assert(SFull::LDS <= 160 * 1024, "one 7x7x7 workgroup per CU");

// What a launch reads and writes. An RK4 step alternates two padded states,
// the caller's u and the plan's work state (see StageIO). u0 and the
// accumulator hold interior points only, in the order the kernel's threads
// take them, so that a wave reads and writes whole lines: variable v of a block
// with m interior points, the first of them numbered q0, starts at 24 q0 + v m;
// there its tiles follow each other (Tile::q0), each in the order of its
// lanes without those that repeat a point (the lane table's second half).
// The kernel's first parameter: StreamCtx::args() finds it by that place.
struct StreamIO {
    VarPtrs src;   // padded stage input
    VarPtrs dst;   // padded next state (right-hand side alone: the output)
    double *u0, *acc;
    RhsParams prm;
    double cacc, cnext;
    int stage;  // 0..3, or -1: the right-hand side alone
    int enforce;
    int *err;
    const int64_t *nbo;  // HALO: 27 neighbour offsets per block, as in StageIO
};

template <bool FACE, class C, bool HALO, bool GAUGE>
struct StreamCtx {
    static constexpr int FT = C::FT, NBUF = C::NBUF;
    static constexpr int PASS = C::passes(HALO), CROSS = C::cross_passes(HALO);
    // Variables in flight (1 to 3) once variable Q is staged, that is while phase
    // Q runs (one to three in the later phases measured the same to 1%)
    static constexpr int ahead(int q) { return q < 5 ? 2 : 1; }
    // the last variable fetched by then
    static constexpr int last(int q) {
        int l = 2;
        for (int k = 0; k <= q; k++) l = l < k + ahead(k) ? k + ahead(k) : l;
        return l < NV ? l : NV - 1;
    }
    const __attribute__((address_space(4))) dgr::AxisConsts *K;
    double *s_tile, *s_dx, *s_dy, *s_keep;
    // tile (uniform)
    uint64_t boff;
    // the stage update: the block's part of the interior buffers (from: what
    // `next` starts from), and the bytes each access may touch (0: none)
    double *u0, *acc, *from;
    uint32_t m;  // the block's interior points
    uint32_t n_from, n_acc, n_u0, n_next;
    double cacc, cnext;
    bool first;  // stage 0
    int ox, oy, oz, ex1, ey1, ez1;  // first point; extents - 1
    bool lox, hix, loy, hiy, loz, hiz;  // the tile meets a flagged face of its block
    double kc[9];  // interior stencil constants: 1/(60h), 1/(180h^2), KO prefactor per axis
    const __attribute__((address_space(4))) DBlock *block;  // read through scalar loads
    // this thread
    int tid, at3, cofs;  // at3: the point within its tile, four bits an axis
    // byte offsets of the point within its padded block and within its block's
    // part of an interior buffer; past any range on lanes that repeat a point
    // (those compute with zeros and store nothing)
    uint32_t li, lq;
    uint64_t boff0;  // the block's offset (boff is 0 with HALO)
    bool active, face;
    double inv_r, eta_v;
    double root;                  // dissipation: sigma = root * eps
    double eps_gauge, eps_other;  // (uniform)
    // staging: byte offsets of the pairs this thread reads (goff_cross: its last
    // one for a variable without second derivatives, past any range if it has
    // none there) and where they go, two halves a word
    uint32_t goff[PASS], goff_cross, spot[(PASS + 1) / 2];
    typedef double Pair __attribute__((ext_vector_type(2)));
    Pair pre[3][PASS];
    int line;        // where this thread's D_x row or D_y column starts in the region
    bool has_line;
    bool x_wave;     // (uniform) this wave's lines are rows
    // the current phase
    double d1[3], d2[6], kv, centre;
    // the stage update
    double r0[NV], r1[NV];  // step's start, accumulator (live from want to put)
    double out[NV];         // next values held for the constraints
    double *to[NV];         // where they go
    bool bad_metric;

    __device__ StreamCtx() {}

    __device__ __forceinline__ void pin(double &x) const { DGR_PIN(x); }

    // ---- staging -----------------------------------------------------------
    template <int Q>
    __device__ __forceinline__ void fetch() {
        constexpr int v = dgr::kStreamVar[Q];
        const __amdgpu_buffer_rsrc_t rs = buffer(args()->src.p[v] + boff, HALO ? 0xffffffe0u : ALL);
        constexpr int N = d2slot(v) >= 0 ? PASS : CROSS;
#pragma unroll
        for (int c = 0; c < N; c++) {
            const uint32_t off = d2slot(v) < 0 && c == CROSS - 1 ? goff_cross : goff[c];
            pre[Q % 3][c] = __builtin_bit_cast(Pair, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
        }
    }

    template <int Q, int TO>
    __device__ __forceinline__ void fetch_to() {
        if constexpr (Q <= TO) {
            fetch<Q>();
            fetch_to<Q + 1, TO>();
        }
    }
    // Variable Q into its region buffer
    template <int Q>
    __device__ __forceinline__ void bring() {
        if constexpr (Q < NV) {
            constexpr int N = d2slot(dgr::kStreamVar[Q]) >= 0 ? PASS : CROSS;
            double *t = s_tile + (Q % C::RB) * NBUF;
#pragma unroll
            for (int c = 0; c < N; c++) {
                const uint32_t w = c & 1 ? spot[c / 2] >> 16 : spot[c / 2] & 0xffffu;
                t[w] = pre[Q % 3][c].x;
                t[w + 1] = pre[Q % 3][c].y;
            }
            fetch_to<last(Q - 1) + 1, last(Q)>();
        }
    }

    // ---- stencils ----------------------------------------------------------
    template <int A>
    static constexpr int stride() { return A == 0 ? 1 : A == 1 ? FRX : FRXY; }
    template <int A>
    __device__ __forceinline__ bool lo() const { return A == 0 ? lox : A == 1 ? loy : loz; }
    template <int A>
    __device__ __forceinline__ bool hi() const { return A == 0 ? hix : A == 1 ? hiy : hiz; }
    template <int A>
    __device__ __forceinline__ int local() const { return (at3 >> (4 * A)) & 15; }

    // FACE: the N values next to a flagged face on the line through s along axis
    // A, from the face inwards; l is the distance from the face
    template <int A, int N, bool HI>
    __device__ __forceinline__ void edge(const double *s, int l, double *e) const {
        const double *p = s + (HI ? l : -l) * stride<A>();
#pragma unroll
        for (int k = 0; k < N; k++) e[k] = p[(HI ? -k : k) * stride<A>()];
    }
    // First derivatives of the tile's (up to 7) points along axis A from the 13
    // region values of the line at s: 13 LDS reads for 7 results, where a
    // stencil at a time reads 42
    template <int A>
    __device__ __forceinline__ void d1_line(const double *s, double *to) const {
        constexpr int ST = stride<A>();
        double u[RMAX], r[TMAX];
#pragma unroll
        for (int k = 0; k < RMAX; k++) u[k] = s[k * ST];
#pragma unroll
        for (int i = 0; i < TMAX; i++)
            r[i] = dgr::d1_of({{u[i], u[i + 1], u[i + 2], u[i + 4], u[i + 5], u[i + 6]}}, kc[A]);
        if constexpr (FACE) {
            const double by12 = K[A].d1_12;
            if (lo<A>()) {
                r[0] = dgr::d1_row<false, 0>(u + PW, by12);
                r[1] = dgr::d1_row<false, 1>(u + PW, by12);
                r[2] = dgr::d1_row<false, 2>(u + PW, by12);
            }
            if (hi<A>()) {
                // the last point's place is the tile's extent (4 to 7) less one
                auto at_end = [&](auto last) {
                    constexpr int N = decltype(last)::value;
                    const double e[5] = {u[PW + N], u[PW + N - 1], u[PW + N - 2], u[PW + N - 3], u[PW + N - 4]};
                    r[N] = dgr::d1_row<true, 0>(e, by12);
                    r[N - 1] = dgr::d1_row<true, 1>(e, by12);
                    r[N - 2] = dgr::d1_row<true, 2>(e, by12);
                };
                switch (last_point<A>()) {
                    case 3: at_end(std::integral_constant<int, 3>()); break;
                    case 4: at_end(std::integral_constant<int, 4>()); break;
                    case 5: at_end(std::integral_constant<int, 5>()); break;
                    default: at_end(std::integral_constant<int, 6>());
                }
            }
        }
#pragma unroll
        for (int i = 0; i < TMAX; i++) to[i * ST] = r[i];
    }

    // N first derivatives along axis A from their taps; s: where they were read,
    // l: the points' places within the tile along A (a tile with lo<A>() starts
    // on that face, one with hi<A>() ends on it). The closures of all N in one
    // stretch a face: their LDS reads wait together.
    template <int A, int N>
    __device__ __forceinline__ void D1(const dgr::Taps *u, const double *const *s, const int *l, double *r) const {
#pragma unroll
        for (int k = 0; k < N; k++) r[k] = dgr::d1_of(u[k], kc[A]);
        if constexpr (FACE) {
            double e[N][5];
            if (lo<A>()) {
#pragma unroll
                for (int k = 0; k < N; k++) edge<A, 5, false>(s[k], l[k], e[k]);
#pragma unroll
                for (int k = 0; k < N; k++) r[k] = dgr::d1_face<false>(e[k], r[k], l[k], K[A].d1_12);
            }
            if (hi<A>()) {
                const int last = last_point<A>();
#pragma unroll
                for (int k = 0; k < N; k++) edge<A, 5, true>(s[k], last - l[k], e[k]);
#pragma unroll
                for (int k = 0; k < N; k++) r[k] = dgr::d1_face<true>(e[k], r[k], last - l[k], K[A].d1_12);
            }
        }
    }
    template <int A>
    __device__ __forceinline__ int last_point() const { return A == 0 ? ex1 : A == 1 ? ey1 : ez1; }

    // What a variable needs along axis A at its own point: the dissipation, and
    // the first (FIRST) and second (SECOND) derivatives
    template <int A, bool FIRST, bool SECOND>
    __device__ __forceinline__ void own_axis(const dgr::Taps &u, const double *s, double &ko, double &first,
                                             double &second) const {
        ko = dgr::ko_of(u, centre, kc[6 + A]);
        if constexpr (FIRST) first = dgr::d1_of(u, kc[A]);
        if constexpr (SECOND) second = dgr::d2_of(u, centre, kc[3 + A]);
        if constexpr (FACE) {
            double e[6];
            if (lo<A>()) {
                const int l = local<A>();
                edge<A, 6, false>(s, l, e);
                ko = dgr::ko_face(e, ko, l, K[A]);
                if constexpr (FIRST) first = dgr::d1_face<false>(e, first, l, K[A].d1_12);
                if constexpr (SECOND) second = dgr::d2_face<false>(e, second, l, K[A].d2_12);
            }
            if (hi<A>()) {
                const int l = last_point<A>() - local<A>();
                edge<A, 6, true>(s, l, e);
                ko = dgr::ko_face(e, ko, l, K[A]);
                if constexpr (FIRST) first = dgr::d1_face<true>(e, first, l, K[A].d1_12);
                if constexpr (SECOND) second = dgr::d2_face<true>(e, second, l, K[A].d2_12);
            }
        }
    }

    // `before_wait` runs when the phase's derivatives are done, before the wait
    // for the next variable's region: memory operations issued there have the
    // staging and the barrier to complete in.
    //
    // Buffers. DEEP: phase Q stages variable Q+1 before its one barrier, which
    // publishes that region and Q's D_x / D_y; region buffer (Q+1)%3 and D_x / D_y
    // set Q&1 were last read in phase Q-2, before barrier Q-1, which every wave
    // has passed when it writes them. Otherwise: region buffer (Q+1)&1 was last
    // read in phase Q-1 and D_x / D_y in the last phase that had them, both
    // before the barrier that ended phase Q-1.
    template <int V, int Q, typename F>
    __device__ __forceinline__ void phase(F before_wait) {
        static_assert(dgr::kStreamVar[Q] == V, "phase order");
        const double *t = s_tile + (Q % C::RB) * NBUF;
        const double *s = t + cofs;
        double *dx = s_dx + (C::DEEP ? (Q & 1) * C::NSDX : 0), *dy = s_dy + (C::DEEP ? (Q & 1) * C::NSDY : 0);
        constexpr bool MIXED = d2slot(V) >= 0;
        dgr::Taps ux, uy, uz;
        auto own = [&] {
            ux = dgr::taps<1>(s);
            uy = dgr::taps<FRX>(s);
            uz = dgr::taps<FRXY>(s);
            centre = s[0];
        };
        if constexpr (MIXED) {
            // the mixed derivatives are D_y(D_x u), D_z(D_x u), D_z(D_y u)
            own();
            if (x_wave) {
                if (has_line) d1_line<0>(t + line, dx + line);
            } else {
                if (has_line) d1_line<1>(t + line + PW, dy + line);
            }
        } else {
            own();
        }
        {
            // sigma (ko_x + ko_y + ko_z) (rhs.cpp:434-489)
#pragma clang fp contract(off)
            double kx, ky, kz;
            own_axis<0, !MIXED, MIXED>(ux, s, kx, d1[0], d2[0]);
            own_axis<1, !MIXED, MIXED>(uy, s, ky, d1[1], d2[3]);
            own_axis<2, true, MIXED>(uz, s, kz, d1[2], d2[5]);
            kv = root * (is_gauge(V) ? eps_gauge : eps_other) * (kx + ky + kz);
            DGR_PIN(kv);
        }
        if constexpr (C::DEEP) bring<Q + 1>();
        if constexpr (d2slot(V) >= 0 || (C::DEEP && Q + 1 < NV)) __syncthreads();
        if constexpr (d2slot(V) >= 0) {
            const double *const cx = dx + (cofs - PW), *const cy = dy + (cofs - PW - FRX * PW);
            const dgr::Taps xy = dgr::taps<FRX>(cx), z[2] = {dgr::taps<FRXY>(cx), dgr::taps<FRXY>(cy)};
            d1[0] = cx[0];
            d1[1] = cy[0];
            const int ly = local<1>(), lz[2] = {local<2>(), local<2>()};
            const double *const czs[2] = {cx, cy};
            double rz[2];
            D1<1, 1>(&xy, &cx, &ly, &d2[1]);
            D1<2, 2>(z, czs, lz, rz);
            d2[2] = rz[0];
            d2[4] = rz[1];
#pragma unroll
            for (int k = 0; k < 6; k++) DGR_PIN(d2[k]);
        }
        DGR_PIN(d1[0]);
        DGR_PIN(d1[1]);
        DGR_PIN(d1[2]);
        DGR_PIN(centre);
        if constexpr (FACE) {
            if (face) {
                // bssn_bcs in place of the equations (rhs.cpp:511-631), the
                // dissipation added to it
#pragma clang fp contract(off)
                double x[3];
                coords(x);
                kv = -inv_r * (x[0] * d1[0] + x[1] * d1[1] + x[2] * d1[2] + BC_FALLOFF[V] * (centre - BC_ASYM[V])) + kv;
            }
        }
        before_wait();
        if constexpr (!C::DEEP && Q + 1 < NV) {
            bring<Q + 1>();
            __syncthreads();
        }
    }

    // ---- the point's fields and results -------------------------------------
    // Raw buffer accesses: a uniform base and a 32-bit byte offset a lane. An
    // access past `bytes` is dropped (a load gives 0), so what a stage does not
    // read or write (bytes = 0) and lanes that repeat a point (offset past any
    // range) need no branch, and the code from phase to phase is one stretch
    // whose loads in flight the compiler can count.
    static constexpr uint32_t ALL = 0x7fffffffu, NOWHERE = 0x80000000u;
    // (with HALO a variable may take all of the 32-bit range but its end)
    static constexpr uint32_t NOWHERE_AT_ALL = 0xfffffff0u;
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const double *p, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), 0, (int)bytes, 0x00020000);
    }
    static __device__ __forceinline__ double load(const double *p, uint32_t bytes, uint32_t off) {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(buffer(p, bytes), off, 0, 0));
    }
    static __device__ __forceinline__ void save(double *p, uint32_t bytes, uint32_t off, double x) {
        typedef unsigned int pair __attribute__((ext_vector_type(2)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(pair, x), buffer(p, bytes), off, 0, 0);
    }
    // The launch's pointer tables, read where they are needed: opaque to the
    // compiler, which otherwise loads all 48 pointers at the top and parks them
    // in vector lanes (350 of them, with 830 reads)
    typedef const StreamIO __attribute__((address_space(4))) ConstIO;
    static __device__ __forceinline__ ConstIO *args() {
        ConstIO *p = (ConstIO *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(p));
        return p;
    }
    // a parameter, likewise
    __device__ __forceinline__ double lam(int i) const { return args()->prm.lam[i]; }
    __device__ __forceinline__ double lamf(int i) const { return args()->prm.lamf[i]; }
    template <int V>
    __device__ __forceinline__ double fld() const { return load(args()->src.p[V] + boff0, ALL, li); }
    // N fields from variable V on: their addresses in one scalar load
    template <int V, int N>
    __device__ __forceinline__ void flds(double *f) const {
        ConstIO *a = args();
        const double *p[N];
#pragma unroll
        for (int k = 0; k < N; k++) p[k] = a->src.p[V + k];
#pragma unroll
        for (int k = 0; k < N; k++) f[k] = load(p[k] + boff0, ALL, li);
    }
    __device__ __forceinline__ double here() const { return centre; }
    __device__ __forceinline__ double eta() const { return eta_v; }
    template <int S>
    __device__ __forceinline__ void keep(double x) { s_keep[S * FT + tid] = x; }
    template <int S>
    __device__ __forceinline__ double take() const { return s_keep[S * FT + tid]; }
    template <int V>
    __device__ __forceinline__ double part(double x) const {
#pragma clang fp contract(off)
        return (FACE && face) ? kv : x + kv;
    }

    // Stage s of the step (U = {0, 1/2, 1/2, 1}, C = {1/6, 1/3, 1/3, 1/6}):
    // acc = (s ? acc : u0) + C[s] dt k; next = u0 + U[s+1] dt k, or acc at the
    // last. r0 is what `next` starts from (stage 0: the field f; 1, 2: the
    // saved u0; 3: the accumulator; right-hand side alone: 0 with cnext = 1).
    template <int V>
    __device__ __forceinline__ void want() {
        r0[V] = load(from + V * m, n_from, lq);
        r1[V] = load(acc + V * m, n_acc, lq);
    }
    template <int V, int N>
    __device__ __forceinline__ void wants() {
        want<V>();
        if constexpr (N > 1) wants<V + 1, N - 1>();
    }
    template <int V, int N>
    __device__ __forceinline__ void destinations() {
        ConstIO *a = args();
#pragma unroll
        for (int k = 0; k < N; k++) to[V + k] = a->dst.p[V + k] + boff0;
    }
    template <int V>
    __device__ __forceinline__ void put(double p, double x, double f) {
#pragma clang fp contract(off)
        const double k = (FACE && face) ? p : p + x;
        const double start = first ? f : r0[V];
        const double a = (first ? f : r1[V]) + cacc * k;
        const double next = start + cnext * k;
        save(u0 + V * m, n_u0, lq, start);
        save(acc + V * m, n_next, lq, a);
        if (slot14(V) >= 0) {
            out[V] = next;
            DGR_PIN(out[V]);
        } else {
            save(to[V], ALL, li, next);
        }
    }
    template <int V>
    __device__ __forceinline__ void store() { save(to[V], ALL, li, out[V]); }
    __device__ __forceinline__ void metric_done() {
        bad_metric = false;
        ConstIO *a = args();
        if (a->enforce) {
            const int e = enforce_metric(out, a->prm.chi_floor);
            bad_metric = e & 1;
            if (e && active) atomicOr(a->err, e);
        }
        destinations<0, 2>();
        destinations<12, 6>();
        store<0>(); store<1>(); store<12>(); store<13>(); store<14>(); store<15>(); store<16>(); store<17>();
    }
    __device__ __forceinline__ void curvature_done() {
        ConstIO *a = args();
        if (a->enforce && !bad_metric) {
            const int e = enforce_trace(out);
            if (e && active) atomicOr(a->err, e);
        }
        destinations<18, 6>();
        store<18>(); store<19>(); store<20>(); store<21>(); store<22>(); store<23>();
        if constexpr (!GAUGE) {
            double x[3];
            coords(x);
            const RhsParams prm = {.eta_central = args()->prm.eta_central, .eta_outer = args()->prm.eta_outer,
                                   .eta_width = args()->prm.eta_width};
            eta_v = rit_eta(x[0], x[1], x[2], prm);
        }
    }
    __device__ __forceinline__ void coords(double *x) const {
        auto b = block;
        asm volatile("" : "+s"(b));
        x[0] = coord(b->pmin[0], ox + local<0>(), b->h[0]);
        x[1] = coord(b->pmin[1], oy + local<1>(), b->h[1]);
        x[2] = coord(b->pmin[2], oz + local<2>(), b->h[2]);
    }

    // ---- the other builds' gauges --------------------------------------------
    __device__ __forceinline__ void after_chi(const double *g, double chi) {
        ConstIO *a = args();
        if (a->prm.eta_func)
            eta_v = eta_function<double>(g, d1, chi, a->prm.eta_r0, a->prm.eta_p0, a->prm.eta_p1);
    }
    __device__ __forceinline__ double slow_start(double alpha, double chi) const {
        ConstIO *a = args();
        if (!a->prm.ssl) return 0.0;
        return ssl_term<double>(alpha, chi, a->prm.ssl_dev ? a->prm.ssl_dev[1] : a->prm.ssl_e);
    }
    template <int N>
    __device__ __forceinline__ void put_beta(double adv, double standard, const double *be) {
        ConstIO *a = args();
        const bool r = a->prm.rochester;
        const double p = part<6 + N>((r ? a->prm.xi[1] : a->prm.lam[1]) * adv);
        put<6 + N>(p, r ? 0.75 * a->prm.xi[2] * fld<3 + N>() - eta_v * be[N] : standard, be[N]);
    }
    template <int N>
    __device__ __forceinline__ void put_B(double adv, double rest) {
        const bool r = args()->prm.rochester;
        const double p = part<9 + N>(r ? 0.0 : adv);
        put<9 + N>(p, r ? 0.0 : rest, centre);
    }
};

// One workgroup's tile, by its first C::FT threads, is the text of stream_tile.h,
// included in the kernels: as an inlined function the compiler duplicated more
// of the flagged kernel's tails (300 KB of code for 288) and it was 5% slower.
template <bool FACE, class C, bool HALO, bool GAUGE>
__global__ __launch_bounds__(C::FT, 2) void k_stream(const StreamIO io, const DBlock *__restrict__ blocks,
                                                     const dgr::AxisConsts *__restrict__ bconst,
                                                     const Tile *__restrict__ tiles,
                                                     const uint16_t *__restrict__ tabs) {
    __shared__ double s_tile[C::RB * C::NBUF];
    __shared__ double s_dx[C::DB * C::NSDX];
    __shared__ double s_dy[C::DB * C::NSDY];
    __shared__ double s_keep[dgr::kStreamKeep * C::FT];
#include "stream_tile.h"
}

// All tiles of a small plan in one launch: the regular ones first, from face0 on
// those of blocks with flagged faces, from full0 on the 7-deep ones. Its
// workgroups take a CU each (the 7-deep tile's LDS), which is what a list of at
// most SMALL_TILES tiles has anyway; launched kind by kind, each kind's single
// latency chain waited for the one before: 64 blocks of 13^3 of which 56 lie on
// the boundary (120 tiles), ten RK4 steps 5.04 -> 3.39 ms.
constexpr int SMALL_TILES = 256;  // the CUs
template <bool HALO, bool GAUGE>
__global__ __launch_bounds__(SFull::FT, 2) void k_stream_small(const StreamIO io, const DBlock *__restrict__ blocks,
                                                               const dgr::AxisConsts *__restrict__ bconst,
                                                               const Tile *__restrict__ tiles,
                                                               const uint16_t *__restrict__ tabs, int face0, int full0) {
    static_assert(SWide::LDS <= SFull::LDS && SWide::FT <= SFull::FT, "either fits");
    __shared__ double lds[SFull::LDS / sizeof(double)];
    auto run = [&](auto face, auto shape) {
        using C = decltype(shape);
        constexpr bool FACE = decltype(face)::value;
        double *const s_tile = lds, *const s_dx = s_tile + C::RB * C::NBUF, *const s_dy = s_dx + C::DB * C::NSDX,
                      *const s_keep = s_dy + C::DB * C::NSDY;
#include "stream_tile.h"
    };
    const int i = (int)blockIdx.x;
    if (i >= full0) {
        run(std::false_type(), SFull());
        return;
    }
    // whole waves end here; a barrier counts those that run
    if (threadIdx.x >= SWide::FT) return;
    if (i >= face0) run(std::true_type(), SWide());
    else run(std::false_type(), SWide());
}
