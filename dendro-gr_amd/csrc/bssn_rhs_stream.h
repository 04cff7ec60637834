// The BSSN right-hand side in streaming order, written for a small live set.
//
// The equations are those of gen_bssn_rhs.py (CodeGen/bssn.py:78-218 with the
// helpers of CodeGen/dendro.py:173-550); this form is written by hand so that
// every derivative is contracted in its variable's phase and only sums stay:
//   gt00..gt22   six second derivatives of gt_ij -> one sum in R_ij
//   (no phase)   Christoffel symbols, the quadratic part of R_ij, one first
//                index f of C1_fjk at a time
//   Gt0..2       R_ij += g_k(i d_j) Gt^k
//   chi, alpha   R_ij complete; X_ij = alpha R_ij - D_i D_j alpha replaces it,
//                its trace-free part times chi stays (6 values)
//   K            the Gt right-hand sides' terms without beta (3 values)
//   beta0..2     nine first derivatives; after them every Lie term: gt, Gt and
//                chi are done and At's rest is one value per component
//   At, B        advection only
// At most about 75 doubles are live (after the gt phases, without the fields
// of later phases), against 126 of the generated phase order: FP64 fits two
// waves per SIMD in 256 registers.
//
// Ctx provides, for the point the caller evaluates:
//   phase<V, K>(f)  makes variable V's derivatives current: d1[a] and, for the
//                   eleven variables that have them, d2[xx xy xz yy yz zz];
//                   K is V's position in kStreamVar. Every thread of a
//                   workgroup runs all of them. f() asks for what the next
//                   steps read from memory.
//   fld<V>(), flds<V, N>(x)  the field V; N fields from V on
//   part<V>(x)      x plus V's dissipation, in V's phase (on a flagged face
//                   the boundary value plus dissipation instead)
//   put<V>(p, x, f) the right-hand side p + x of the field f, p from part<V>()
//                   (on a flagged face p alone)
//   keep<S>(x), take<S>()  a value parked outside the registers, S < kStreamKeep
//   pin(x)          x is computed here, not sunk to a later use
//   lam(i), lamf(i)  BSSN_LAMBDA, BSSN_LAMBDA_F
//   here()          the current phase's field at the point
//   wants<V, N>()   put<V>() .. put<V + N - 1>() follow: what they read can be
//                   fetched now; destinations<V, N>() likewise where they write
//   metric_done(), curvature_done()  chi, alpha and gt (then At) have been put
//   eta()           B's damping
//   after_chi(g, chi), slow_start(alpha, chi), put_beta<N>(...), put_B<N>(...)
//                   the other builds' gauges (GAUGE only)
#pragma once

#ifndef DGR_HD
#define DGR_HD
#endif
#ifndef DGR_INLINE
#define DGR_INLINE inline
#endif
#ifdef __clang__
#define DGR_UNROLL _Pragma("unroll")
#else
#define DGR_UNROLL
#endif

namespace dgr {

constexpr int kStreamVar[24] = {12, 13, 14, 15, 16, 17, 3, 4, 5, 1, 0, 2, 6, 7, 8, 18, 19, 20, 21, 22, 23, 9, 10, 11};
constexpr int kStreamKeep = 11;  // gt's six partial sums, chi's, Gt's three, K

// index of the (i, j) component in 00 01 02 11 12 22
DGR_HD constexpr int sym6(int i, int j) { return i + j + (i && j ? 1 : 0); }

// sum_ij u^ij s_ij of two symmetric tensors
DGR_HD DGR_INLINE double trace6(const double *u, const double *s) {
    return (u[0] * s[0] + u[3] * s[3] + u[5] * s[5]) + 2.0 * (u[1] * s[1] + u[2] * s[2] + u[4] * s[4]);
}

// Phase C of the metric component C = 0..5 (variable 12 + C)
template <int C, typename Ctx>
DGR_HD DGR_INLINE void stream_gt(Ctx &c, const double *u, const double *be, double *R, double *dg) {
    c.template phase<12 + C, C>([] {});
    R[C] = -0.5 * trace6(u, c.d2);
    const double p = c.template part<12 + C>(be[0] * c.d1[0] + be[1] * c.d1[1] + be[2] * c.d1[2]);
    c.template keep<C>(p);
    DGR_UNROLL
    for (int a = 0; a < 3; a++) {
        dg[3 * C + a] = c.d1[a];
        c.pin(dg[3 * C + a]);
    }
    c.pin(R[C]);
}

// First index F of C1: its quadratic terms in the Ricci tensor
//   igt^lm (C2^k_li C1_jkm + C2^k_lj C1_ikm + C2^k_im C1_klj)
//   + 1/2 CalGt^k (C1_ijk + C1_jik)
// (dendro.py:495-541), with C1 raised on its last index one F at a time.
template <int F>
DGR_HD DGR_INLINE void stream_ricci(const double *u, const double (*C1)[6], const double (*C2)[6], const double *cal,
                                    double *R) {
    double D[3][3];  // D[k][l] = u^lm C1_Fkm
    DGR_UNROLL
    for (int k = 0; k < 3; k++)
        DGR_UNROLL
        for (int l = 0; l < 3; l++)
            D[k][l] = u[sym6(l, 0)] * C1[F][sym6(k, 0)] + u[sym6(l, 1)] * C1[F][sym6(k, 1)] +
                      u[sym6(l, 2)] * C1[F][sym6(k, 2)];
    DGR_UNROLL
    for (int i = 0; i < 3; i++) {
        double s = 0.5 * (cal[0] * C1[F][sym6(i, 0)] + cal[1] * C1[F][sym6(i, 1)] + cal[2] * C1[F][sym6(i, 2)]);
        DGR_UNROLL
        for (int k = 0; k < 3; k++)
            DGR_UNROLL
            for (int l = 0; l < 3; l++) s += C2[k][sym6(l, i)] * D[k][l];
        R[sym6(i, F)] += i == F ? 2.0 * s : s;
    }
    DGR_UNROLL
    for (int i = 0; i < 3; i++)
        DGR_UNROLL
        for (int j = i; j < 3; j++)
            R[sym6(i, j)] += C2[F][sym6(i, 0)] * D[j][0] + C2[F][sym6(i, 1)] * D[j][1] + C2[F][sym6(i, 2)] * D[j][2];
}

// Phase of Gt^N: its advection, and R_ij += 1/2 (g_ki d_j Gt^k + g_kj d_i Gt^k)
template <int N, typename Ctx>
DGR_HD DGR_INLINE void stream_Gt(Ctx &c, const double *be, const double *g, double *R, double *nB) {
    c.template phase<3 + N, 6 + N>([] {});
    const double adv = be[0] * c.d1[0] + be[1] * c.d1[1] + be[2] * c.d1[2];
    c.template keep<7 + N>(c.template part<3 + N>(adv));
    nB[N] = adv - c.lam(3) * adv;
    DGR_UNROLL
    for (int i = 0; i < 3; i++)
        DGR_UNROLL
        for (int j = i; j < 3; j++)
            R[sym6(i, j)] += 0.5 * (g[sym6(N, i)] * c.d1[j] + g[sym6(N, j)] * c.d1[i]);
    DGR_UNROLL
    for (int k = 0; k < 6; k++) c.pin(R[k]);
    c.pin(nB[N]);
}

// Phase of beta^N: G gets its second derivatives (trace) and Christoffel term,
// e the gradient of the divergence
template <int N, bool GAUGE, typename Ctx>
DGR_HD DGR_INLINE void stream_beta(Ctx &c, const double *be, const double *u, const double *cal, double alpha,
                                   double Bn, double *G, double *e, double (*db)[3],
                                   double *Gt) {
    // (the last beta completes chi, Gt and gt)
    c.template phase<6 + N, 12 + N>([&] {
        c.template destinations<6 + N, 1>();
        if constexpr (N < 2) {
            c.template wants<7 + N, 1>();
        } else {
            c.template wants<1, 1>();
            c.template flds<3, 3>(Gt);
            c.template wants<3, 3>();
            c.template wants<12, 6>();
        }
    });
    DGR_UNROLL
    for (int a = 0; a < 3; a++) {
        db[N][a] = c.d1[a];
        c.pin(db[N][a]);
    }
    G[N] += trace6(u, c.d2) - (cal[0] * c.d1[0] + cal[1] * c.d1[1] + cal[2] * c.d1[2]);
    c.pin(G[N]);
    DGR_UNROLL
    for (int a = 0; a < 3; a++) {
        e[a] += c.d2[sym6(a, N)];
        c.pin(e[a]);
    }
    const double adv = be[0] * c.d1[0] + be[1] * c.d1[1] + be[2] * c.d1[2];
    if constexpr (GAUGE) {
        c.template put_beta<N>(adv, 0.75 * (c.lamf(0) + c.lamf(1) * alpha) * Bn, be);
    } else {
        const double p = c.template part<6 + N>(c.lam(1) * adv);
        c.template put<6 + N>(p, 0.75 * (c.lamf(0) + c.lamf(1) * alpha) * Bn, be[N]);
    }
}

template <int C, typename Ctx>
DGR_HD DGR_INLINE void stream_At(Ctx &c, const double *be, const double *Z) {
    // (two right-hand sides ahead, on to B)
    c.template phase<18 + C, 15 + C>([&] { c.template wants<(C < 4 ? 20 + C : 5 + C), 1>(); });
    const double p = c.template part<18 + C>(be[0] * c.d1[0] + be[1] * c.d1[1] + be[2] * c.d1[2]);
    c.template put<18 + C>(p, Z[C], c.here());
}

template <int N, bool GAUGE, typename Ctx>
DGR_HD DGR_INLINE void stream_B(Ctx &c, const double *be, const double *nB) {
    c.template phase<9 + N, 21 + N>([&] {
        if constexpr (N == 0) c.template wants<11, 1>();
        c.template destinations<9 + N, 1>();
    });
    const double adv = be[0] * c.d1[0] + be[1] * c.d1[1] + be[2] * c.d1[2];
    if constexpr (GAUGE) {
        c.template put_B<N>(c.lam(2) * adv, nB[N] - c.eta() * c.here());
    } else {
        const double p = c.template part<9 + N>(c.lam(2) * adv);
        c.template put<9 + N>(p, nB[N] - c.eta() * c.here(), c.here());
    }
}

template <bool GAUGE, typename Ctx>
DGR_HD DGR_INLINE void bssn_rhs_stream(Ctx &c) {
    double be[3], g[6];
    c.template flds<12, 6>(g);
    c.template flds<6, 3>(be);
    // inverse conformal metric: adjugate over determinant (dendro.py:375-393)
    double u[6];
    {
        const double c00 = g[3] * g[5] - g[4] * g[4], c01 = g[2] * g[4] - g[1] * g[5], c02 = g[1] * g[4] - g[2] * g[3];
        const double id = 1.0 / (g[0] * c00 + g[1] * c01 + g[2] * c02);
        u[0] = id * c00;
        u[1] = id * c01;
        u[2] = id * c02;
        u[3] = id * (g[0] * g[5] - g[2] * g[2]);
        u[4] = id * (g[1] * g[2] - g[0] * g[4]);
        u[5] = id * (g[0] * g[3] - g[1] * g[1]);
        DGR_UNROLL
        for (int k = 0; k < 6; k++) c.pin(u[k]);
    }
    double R[6], cal[3], C2[3][6];
    {
        double dg[18];  // d_a gt_C at 3 C + a
        stream_gt<0>(c, u, be, R, dg);
        stream_gt<1>(c, u, be, R, dg);
        stream_gt<2>(c, u, be, R, dg);
        stream_gt<3>(c, u, be, R, dg);
        stream_gt<4>(c, u, be, R, dg);
        stream_gt<5>(c, u, be, R, dg);
        // C1_kij = 1/2 (d_j g_ki + d_i g_kj - d_k g_ij) (dendro.py:418-421)
        double C1[3][6];
        DGR_UNROLL
        for (int k = 0; k < 3; k++)
            DGR_UNROLL
            for (int i = 0; i < 3; i++)
                DGR_UNROLL
                for (int j = i; j < 3; j++)
                    C1[k][sym6(i, j)] =
                        0.5 * (dg[3 * sym6(k, i) + j] + dg[3 * sym6(k, j) + i] - dg[3 * sym6(i, j) + k]);
        DGR_UNROLL
        for (int k = 0; k < 3; k++)
            DGR_UNROLL
            for (int q = 0; q < 6; q++) c.pin(C1[k][q]);
        // C2^i_jk = igt^il C1_ljk (dendro.py:445-446), CalGt^i = igt^jk C2^i_jk (:512)
        DGR_UNROLL
        for (int i = 0; i < 3; i++) {
            DGR_UNROLL
            for (int q = 0; q < 6; q++) {
                C2[i][q] = u[sym6(i, 0)] * C1[0][q] + u[sym6(i, 1)] * C1[1][q] + u[sym6(i, 2)] * C1[2][q];
                c.pin(C2[i][q]);
            }
            cal[i] = trace6(u, C2[i]);
            c.pin(cal[i]);
        }
        stream_ricci<0>(u, C1, C2, cal, R);
        DGR_UNROLL
        for (int k = 0; k < 6; k++) c.pin(R[k]);
        stream_ricci<1>(u, C1, C2, cal, R);
        DGR_UNROLL
        for (int k = 0; k < 6; k++) c.pin(R[k]);
        stream_ricci<2>(u, C1, C2, cal, R);
        DGR_UNROLL
        for (int k = 0; k < 6; k++) c.pin(R[k]);
    }
    double nB[3];
    stream_Gt<0>(c, be, g, R, nB);
    stream_Gt<1>(c, be, g, R, nB);
    stream_Gt<2>(c, be, g, R, nB);

    // chi: R_ij += the conformal factor's part, with h = 1/(2 chi), v = h d chi:
    // h (d_ij chi - C2^k_ij d_k chi) - v_i v_j + g_ij (h igt^kl(...)_kl - 3 igt^kl v_k v_l)
    double alpha = 0.0, K = 0.0, A[6];
    c.template phase<1, 9>([&] {
        alpha = c.template fld<0>();
        K = c.template fld<2>();
        c.template flds<18, 6>(A);
        c.template wants<0, 1>();
    });
    const double chi = c.here();
    c.template keep<6>(c.template part<1>(be[0] * c.d1[0] + be[1] * c.d1[1] + be[2] * c.d1[2]));
    if constexpr (GAUGE) c.after_chi(g, chi);
    double v[3];
    {
        const double h = 0.5 / chi;
        double M[6];
        DGR_UNROLL
        for (int q = 0; q < 6; q++)
            M[q] = h * (c.d2[q] - (C2[0][q] * c.d1[0] + C2[1][q] * c.d1[1] + C2[2][q] * c.d1[2]));
        DGR_UNROLL
        for (int a = 0; a < 3; a++) v[a] = h * c.d1[a];
        const double vv[6] = {v[0] * v[0], v[0] * v[1], v[0] * v[2], v[1] * v[1], v[1] * v[2], v[2] * v[2]};
        const double lap = trace6(u, M) - 3.0 * trace6(u, vv);
        DGR_UNROLL
        for (int q = 0; q < 6; q++) {
            R[q] += (M[q] - vv[q]) + g[q] * lap;
            c.pin(R[q]);
        }
        DGR_UNROLL
        for (int a = 0; a < 3; a++) c.pin(v[a]);
    }

    // alpha: X_ij = alpha R_ij - D_i D_j alpha (dendro.py:181-183), trace-free part times chi
    double Y[6], G[3], lapse, asq;
    c.template phase<0, 10>([&] { c.template wants<2, 1>(); });
    {
        const double adv = be[0] * c.d1[0] + be[1] * c.d1[1] + be[2] * c.d1[2];
        const double p = c.template part<0>(c.lam(0) * adv);
        double rest = -2.0 * alpha * K;
        if constexpr (GAUGE) rest -= c.slow_start(alpha, chi);
        c.template put<0>(p, rest, alpha);
        const double w[3] = {c.d1[0], c.d1[1], c.d1[2]};
        double dot = 0.0;  // igt^lm v_m d_l alpha
        DGR_UNROLL
        for (int i = 0; i < 3; i++)
            dot += v[i] * (u[sym6(i, 0)] * w[0] + u[sym6(i, 1)] * w[1] + u[sym6(i, 2)] * w[2]);
        double DD[6];
        DGR_UNROLL
        for (int i = 0; i < 3; i++)
            DGR_UNROLL
            for (int j = i; j < 3; j++) {
                const int q = sym6(i, j);
                DD[q] = (c.d2[q] - (C2[0][q] * w[0] + C2[1][q] * w[1] + C2[2][q] * w[2])) +
                        ((v[i] * w[j] + v[j] * w[i]) - g[q] * dot);
            }
        lapse = trace6(u, DD);
        DGR_UNROLL
        for (int q = 0; q < 6; q++) Y[q] = alpha * R[q] - DD[q];
        const double tr = trace6(u, Y) * (1.0 / 3.0);
        DGR_UNROLL
        for (int q = 0; q < 6; q++) {
            Y[q] = chi * (Y[q] - g[q] * tr);
            c.pin(Y[q]);
        }
        // At raised (dendro.py:203-208): At_ij At^ij and the Gt terms it enters
        double AU[6];
        {
            double T[3][3];  // T[i][l] = u^ik A_kl
            DGR_UNROLL
            for (int i = 0; i < 3; i++)
                DGR_UNROLL
                for (int l = 0; l < 3; l++)
                    T[i][l] = u[sym6(i, 0)] * A[sym6(0, l)] + u[sym6(i, 1)] * A[sym6(1, l)] + u[sym6(i, 2)] * A[sym6(2, l)];
            DGR_UNROLL
            for (int i = 0; i < 3; i++)
                DGR_UNROLL
                for (int j = i; j < 3; j++)
                    AU[sym6(i, j)] = T[i][0] * u[sym6(0, j)] + T[i][1] * u[sym6(1, j)] + T[i][2] * u[sym6(2, j)];
        }
        asq = trace6(AU, A);
        double z[3];  // 2 d_j alpha + 3 alpha / chi d_j chi
        DGR_UNROLL
        for (int a = 0; a < 3; a++) z[a] = 2.0 * w[a] + 6.0 * alpha * v[a];
        DGR_UNROLL
        for (int i = 0; i < 3; i++) {
            G[i] = 2.0 * alpha * trace6(AU, C2[i]) -
                   (AU[sym6(i, 0)] * z[0] + AU[sym6(i, 1)] * z[1] + AU[sym6(i, 2)] * z[2]);
            c.pin(G[i]);
        }
        c.pin(lapse);
        c.pin(asq);
    }

    // K
    double Bf[3];
    c.template phase<2, 11>([&] {
        c.template flds<9, 3>(Bf);
        c.template destinations<2, 1>();
        c.template wants<6, 1>();
    });
    {
        const double p = c.template part<2>(be[0] * c.d1[0] + be[1] * c.d1[1] + be[2] * c.d1[2]);
        c.template put<2>(p, alpha * (K * K * (1.0 / 3.0) + asq) - chi * lapse, K);
        c.template keep<10>(K);
        const double s = (4.0 / 3.0) * alpha;
        DGR_UNROLL
        for (int i = 0; i < 3; i++) {
            G[i] -= s * (u[sym6(i, 0)] * c.d1[0] + u[sym6(i, 1)] * c.d1[1] + u[sym6(i, 2)] * c.d1[2]);
            c.pin(G[i]);
        }
    }

    // beta
    double Z[6];
    {
        double db[3][3];  // db[i][a] = d_a beta^i
        double e[3] = {0.0, 0.0, 0.0}, Gt[3];
        stream_beta<0, GAUGE>(c, be, u, cal, alpha, Bf[0], G, e, db, Gt);
        stream_beta<1, GAUGE>(c, be, u, cal, alpha, Bf[1], G, e, db, Gt);
        stream_beta<2, GAUGE>(c, be, u, cal, alpha, Bf[2], G, e, db, Gt);
        const double div = (2.0 / 3.0) * (db[0][0] + db[1][1] + db[2][2]);
        c.template destinations<3, 3>();
        K = c.template take<10>();
        c.template put<1>(c.template take<6>(), chi * ((2.0 / 3.0) * alpha * K - div), chi);
        DGR_UNROLL
        for (int i = 0; i < 3; i++) {
            G[i] += cal[i] * div + (1.0 / 3.0) * (u[sym6(i, 0)] * e[0] + u[sym6(i, 1)] * e[1] + u[sym6(i, 2)] * e[2]);
            nB[i] += G[i];
        }
        c.template put<3>(c.template take<7>(), G[0], Gt[0]);
        c.template put<4>(c.template take<8>(), G[1], Gt[1]);
        c.template put<5>(c.template take<9>(), G[2], Gt[2]);
        DGR_UNROLL
        for (int a = 0; a < 3; a++) c.pin(nB[a]);
        // At: Lie terms, alpha (K At_ij - 2 At_ik igt^kl At_lj) and Y
        {
            double T[3][3];  // T[k][j] = u^kl A_lj
            DGR_UNROLL
            for (int k = 0; k < 3; k++)
                DGR_UNROLL
                for (int j = 0; j < 3; j++)
                    T[k][j] = u[sym6(k, 0)] * A[sym6(0, j)] + u[sym6(k, 1)] * A[sym6(1, j)] + u[sym6(k, 2)] * A[sym6(2, j)];
            const double s = alpha * K - div;
            DGR_UNROLL
            for (int i = 0; i < 3; i++)
                DGR_UNROLL
                for (int j = i; j < 3; j++) {
                    const int q = sym6(i, j);
                    double lie = 0.0, sq = 0.0;
                    DGR_UNROLL
                    for (int k = 0; k < 3; k++) {
                        lie += A[sym6(i, k)] * db[k][j] + A[sym6(k, j)] * db[k][i];
                        sq += A[sym6(i, k)] * T[k][j];
                    }
                    Z[q] = Y[q] + (lie + (s * A[q] - 2.0 * alpha * sq));
                    c.pin(Z[q]);
                }
        }
        // gt
        double L[6];
        DGR_UNROLL
        for (int i = 0; i < 3; i++)
            DGR_UNROLL
            for (int j = i; j < 3; j++) {
                const int q = sym6(i, j);
                double lie = 0.0;
                DGR_UNROLL
                for (int k = 0; k < 3; k++) lie += g[sym6(i, k)] * db[k][j] + g[sym6(k, j)] * db[k][i];
                L[q] = lie - (div * g[q] + 2.0 * alpha * A[q]);
            }
        c.template put<12>(c.template take<0>(), L[0], g[0]);
        c.template put<13>(c.template take<1>(), L[1], g[1]);
        c.template put<14>(c.template take<2>(), L[2], g[2]);
        c.template put<15>(c.template take<3>(), L[3], g[3]);
        c.template put<16>(c.template take<4>(), L[4], g[4]);
        c.template put<17>(c.template take<5>(), L[5], g[5]);
    }
    c.template wants<18, 2>();
    c.metric_done();

    stream_At<0>(c, be, Z);
    stream_At<1>(c, be, Z);
    stream_At<2>(c, be, Z);
    stream_At<3>(c, be, Z);
    stream_At<4>(c, be, Z);
    stream_At<5>(c, be, Z);
    c.curvature_done();
    stream_B<0, GAUGE>(c, be, nB);
    stream_B<1, GAUGE>(c, be, nB);
    stream_B<2, GAUGE>(c, be, nB);
}

}  // namespace dgr
