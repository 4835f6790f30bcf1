// gam_emf.hip -- edge EMFs (CalcElecField, fields.F90:70-517).
#include "gam_launch.h"
#include <algorithm>

// ====================================================================
// Edge EMF: GetCornerV/GetCornerD/GetCornerB/EdgeLRs + VxB
// (fields.F90:187-224, 288-517).  One thread per active edge of ED.
// ====================================================================
template <int FD, int SD, int RM>
__device__ __forceinline__ void edge_lr(const Geo &g, const MParm &m, long c,
                                        const double *__restrict__ met,
                                        const double *__restrict__ mfH,
                                        const double *__restrict__ mfL,
                                        double &bL, double &bR)
{
    // EdgeLRs (fields.F90:288-362) for FD faces stacked along SD, area
    // weighted.  The weighted value A * (flux / max(A, TINY)) is the flux
    // itself on any face larger than TINY (and flux * A / TINY on a smaller
    // one), so the eight divisions and products are left out.
    const long N3 = g.N3;
    const long s = STRIDE<SD>(g);
    double A[8], q[8], nq[4];
#pragma unroll
    for (int n = 0; n < 8; n++) {
        A[n] = ldx<SD>(met + (M_FACE + FD) * N3, c, s, n - 4);
        q[n] = ldx<SD>(mfH + FD * N3, c, s, n - 4) * fmin(A[n] * (1.0 / GAM_TINY), 1.0);
    }
    // the limiter faces are the middle four of the stencil
#pragma unroll
    for (int n = 0; n < 4; n++) nq[n] = ldx<SD>(mfL + FD * N3, c, s, n - 2) * gam_rcp(dmax(A[n + 2], GAM_TINY));
    recon_lr_w<RM>(m.pdmb, gam_rcp(wsum8([&](int n) { return A[n]; })), nq, q, bL, bR);
}

// The EMF of one edge from its corner velocity vc, corner density Dc and the
// L/R normal fields of its two face pairs.
template <int ED, bool BG, bool BORIS>
__device__ __forceinline__ double edge_value(const MParm &m, const double *vc, double Dc, double b1L, double b1R,
                                             double b2L, double b2R, const double *Te, const double *Tb,
                                             const double *b0, double edge, double dt)
{
    const double v1 = vc[0] * Te[0] + vc[1] * Te[1] + vc[2] * Te[2];
    const double v2 = vc[0] * Te[3] + vc[1] * Te[4] + vc[2] * Te[5];
    double vDiff = gam_sqrt(v1 * v1 + v2 * v2);
    const double xni = Tb[0], yni = Tb[1], xnj = Tb[2], ynj = Tb[3];
    const double detT = gam_rcp(xni * ynj - xnj * yni);
    const double bT1 = 0.5 * (b1L + b1R);
    const double bT2 = 0.5 * (b2L + b2R);
    const double Jd = (b2R - b2L) - (b1R - b1L);
    double b1 = detT * (ynj * bT1 - yni * bT2);
    double b2 = detT * (-(xnj * bT1) + xni * bT2);
    if (BG) {
        b1 = b1 + b0[0];
        b2 = b2 + b0[1];
    }
    // vA = |b| / sqrt(D), with Boris Ca vA / sqrt(Ca^2 + vA^2)
    const double bb = b1 * b1 + b2 * b2, Ca2 = m.Ca * m.Ca;
    const double vA = gam_sqrt(BORIS ? Ca2 * bb * gam_rcp(Ca2 * Dc + bb) : bb * gam_rcp(Dc));
    vDiff = vDiff + vA;
    // no cap (infinite) where Model%dt is 0
    vDiff = dmin(vDiff, m.CFL * edge * (dt != 0.0 ? gam_rcp(dt) : HUGE_VAL));
    const double e = -(v1 * b2 - v2 * b1) + m.Vd0 * vDiff * Jd;
    return e * edge;
}

template <int ED, int RM, bool BG, bool BORIS, int NTH = BX * BY>
struct k_emf {
    static constexpr int NT = NTH;
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m,
                                               Tile b, const Clock *clk,
                                               const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ Vf,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ E) const
    {
        int i, j, k;
        if (!tile_point(b, (int)bi.x, i, j, k)) return;
        constexpr int T1 = (ED == 0) ? 1 : (ED == 1) ? 2 : 0;
        constexpr int T2 = (ED == 0) ? 2 : (ED == 1) ? 0 : 1;
        // getNormalPlane (metric.F90:151-167)
        constexpr int E1 = (ED == 0) ? 1 : 0;
        constexpr int E2 = (ED == 2) ? 1 : 2;
        const long N3 = g.N3;
        const long c = IX(g, i, j, k);
        const long s2 = STRIDE<T2>(g);

        // GetCornerV (fields.F90:457-517), doVdA
        double A[8];
#pragma unroll
        for (int n = 0; n < 8; n++) A[n] = ldx<T2>(met + (M_FACE + T1) * N3, c, s2, n - 4);
        const double rdA = gam_rcp(dmax(wsum8([&](int n) { return A[n]; }), GAM_TINY));
        double vc[3];
#pragma unroll
        for (int d = 0; d < 3; d++)
            vc[d] = wsum8([&](int n) { return A[n] * ldx<T2>(Vf + d * N3, c, s2, n - 4); }) * rdA;
        // GetCornerD (fields.F90:427-454)
        const long se1 = STRIDE<E1>(g), se2 = STRIDE<E2>(g);
        const double *Dh = H + (H_GAS + DEN) * N3;
        const double Dc = 0.25 * (Dh[c] + Dh[c - se1] + Dh[c - se2] + Dh[c - se1 - se2]);

        // GetCornerB (fields.F90:365-424)
        const double *mfH = H + H_MF * N3;
        const double *mfL = m.doLFM ? S + S_MF * N3 : mfH;
        double bT1L, bT1R, bT2L, bT2R;
        edge_lr<T1, T2, RM>(g, m, c, met, mfH, mfL, bT1L, bT1R);
        edge_lr<T2, T1, RM>(g, m, c, met, mfH, mfL, bT2L, bT2R);
        double Te[6], Tb[4], b0[2] = {0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 6; q++) Te[q] = met[(M_TE + 9 * ED + 3 + q) * N3 + c];
#pragma unroll
        for (int q = 0; q < 4; q++) Tb[q] = met[(M_TEB + 4 * ED + q) * N3 + c];
        if (BG) {
            b0[0] = bg[(B_EDGB0 + 0 + 2 * ED) * N3 + c];
            b0[1] = bg[(B_EDGB0 + 1 + 2 * ED) * N3 + c];
        }
        E[ED * N3 + c] = edge_value<ED, BG, BORIS>(m, vc, Dc, bT1L, bT1R, bT2L, bT2R, Te, Tb, b0,
                                                   met[(M_EDGE + ED) * N3 + c], clk->dt);
    }
};

// ====================================================================
// EMFs with the face stencils in LDS.  A workgroup of 256 threads owns a
// tile of edges, brings the areas, face velocities and fluxes of every face
// its stencils reach to LDS with all loads in flight at once, and each edge
// its own metrics meanwhile.  The T1 faces (areas, velocities, fluxes) are
// stacked along T2, the T2 faces (areas, fluxes) along T1:
//   ED = 1, 2: 32 (i) x 8 (the other axis of the stencil plane) edges; one
//              pair has 15 x 32 faces, the other (stacked along i) 8 x 39;
//   ED = 0:    16 (i) x 4 (j) x 4 (k) edges, 44 x 16 faces of each pair (the
//              stencil plane is across i: the 16 are one 128-byte line).
// The velocities are weighted and the limiter fluxes divided by their areas
// once per face staged instead of once per edge and stencil point.
// Bound by memory traffic: 256x256x384 shell 4.05 ms for the three directions
// with direct loads (76 to 80 registers, six waves per SIMD waiting on L1),
// 3.34 ms here (19.7 GB at 5.9 TB/s).  Numbering the tiles so that an XCD's
// run of 16 is a block of the stencil plane (4 x 4, or 2 x 8) fetches less
// but took 3.38 to 3.49 ms.
// ====================================================================
struct EdgeTile {
    int i0, i1, j0, j1, k0, k1;   // edges
    int ni, nb;                   // tiles along i; in all
    int bfirst;                   // ED = 1: numbered along i, j, k (else along i, the second axis, the third)
    FastDiv qi, q1;
    int xs;
};

template <int ED>
struct edge_geom {
    static constexpr int T1 = (ED == 0) ? 1 : (ED == 1) ? 2 : 0;
    static constexpr int T2 = (ED == 0) ? 2 : (ED == 1) ? 0 : 1;
    static constexpr int TX = ED == 0 ? 16 : 32;
    // faces of pair P (1: T1, 2: T2) staged; rows of pair P stacked along i
    static constexpr bool ALONG_I(int P) { return P == 1 ? T2 == 0 : T1 == 0; }
    static constexpr int NF(int P) { return ED == 0 ? 16 * 44 : ALONG_I(P) ? 39 * 8 : 15 * 32; }
    static constexpr int NQ(int P) { return ED == 0 ? 16 * 28 : ALONG_I(P) ? 39 * 8 : 11 * 32; }   // limiter entries
    // LDS step of the pair's stencil and of its limiter entries
    static constexpr int SF(int P) { return ED == 0 ? (P == 1 ? 64 : 16) : ALONG_I(P) ? 1 : 32; }
    static constexpr int LDS = 5 * NF(1) + NQ(1) + 2 * NF(2) + NQ(2);
};
#define EMF_LDS (edge_geom<0>::LDS)
static_assert(edge_geom<1>::LDS <= EMF_LDS && edge_geom<2>::LDS <= EMF_LDS, "LDS planes");

template <int ED, int RM, bool BG, bool BORIS, bool DIR>
struct edge_tile {
    using G = edge_geom<ED>;
    // face e of pair P: its place in the tile, as offsets from the tile's
    // first edge along i and the two other axes (j, k), and its limiter entry
    template <int P>
    __device__ __forceinline__ static int place(int e, int &di, int &dj, int &dk)
    {
        if (ED == 0) {
            const int r = e >> 4;
            di = e & 15;
            if (P == 1) {      // J faces along k
                dj = r & 3;
                dk = (r >> 2) - 4;
                return dk >= -2 && dk < 5 ? ((dk + 2) * 4 + dj) * 16 + di : -1;
            }
            dk = r / 11;       // K faces along j
            dj = r - 11 * dk - 4;
            return dj >= -2 && dj < 5 ? (dk * 7 + dj + 2) * 16 + di : -1;
        }
        int da, l;             // a: the tile's second axis, j (ED = 2) or k (ED = 1)
        if (G::ALONG_I(P)) {
            da = e / 39;
            di = e - 39 * da - 4;
            l = e;
        } else {
            di = e & 31;
            da = (e >> 5) - 4;
            l = da >= -2 && da < 9 ? e - 64 : -1;
        }
        dj = ED == 2 ? da : 0;
        dk = ED == 1 ? da : 0;
        return l;
    }
    __device__ __forceinline__ void operator()(double *lds, int w, const Geo &g, const MParm &m,
                                               const EdgeTile &t, const Clock *clk,
                                               const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ O,
                                               const double *__restrict__ Vf,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ E) const
    {
        const int L = xcd_tile(w, t.xs);
        if (L >= t.nb) return;                   // whole workgroup
        constexpr int T1 = G::T1, T2 = G::T2;
        constexpr int NF1 = G::NF(1), NF2 = G::NF(2);
        constexpr int Q1 = (NF1 + 255) / 256, Q2 = (NF2 + 255) / 256;
        double *sA1 = lds, *sV = lds + NF1, *sq1 = lds + 4 * NF1, *sn1 = lds + 5 * NF1;
        double *sA2 = sn1 + G::NQ(1), *sq2 = sA2 + NF2, *sn2 = sq2 + NF2;
        const int tid = (int)(threadIdx.x + BX * threadIdx.y);
        const long N3 = g.N3;
        const unsigned r = (unsigned)L / t.qi, r2 = r / t.q1;
        const int ti = L - (int)r * t.ni, rq = (int)r - (int)r2 * (int)t.q1.d;
        const int ta = t.bfirst ? (int)r2 : rq, tb = t.bfirst ? rq : (int)r2;
        const int i0 = t.i0 + ti * G::TX;
        const int j0 = t.j0 + (ED == 0 ? 4 * ta : ED == 2 ? 8 * ta : tb);
        const int k0 = t.k0 + (ED == 0 ? 4 * tb : ED == 1 ? 8 * ta : tb);
        // a face past those the box's edges reach reads the last of them
        // (only lanes of edges outside the box use it)
        constexpr int RI = ED == 0 ? 0 : 3, RJ = ED == 1 ? 0 : 3, RK = ED == 2 ? 0 : 3;
        auto at = [&](int di, int dj, int dk) -> unsigned {
            const int i = min(i0 + di, t.i1 + RI), j = min(j0 + dj, t.j1 + RJ), k = min(k0 + dk, t.k1 + RK);
            return (unsigned)(8 * IX(g, i, j, k));
        };
        int x, y, z;
        if (ED == 0) { x = tid & 15; y = (tid >> 4) & 3; z = tid >> 6; }
        else { x = tid & 31; y = ED == 2 ? tid >> 5 : 0; z = ED == 1 ? tid >> 5 : 0; }
        const bool act = i0 + x <= t.i1 && j0 + y <= t.j1 && k0 + z <= t.k1;
        const unsigned oc = at(min(x, t.i1 - i0), min(y, t.j1 - j0), min(z, t.k1 - k0));

        // the faces' loads
        double A1[Q1], V1[Q1][3], h1[Q1], l1[Q1], A2[Q2], h2[Q2], l2[Q2];
        // (half-state fluxes h and limiter fluxes l; DIR: of oState and State,
        // extrapolated below)
        const double *mfH = DIR ? O + S_MF * N3 : H + H_MF * N3;
        const double *mfL = DIR || m.doLFM ? S + S_MF * N3 : mfH;
        const double wt = DIR ? ab2_weight(clk) : 0.0;
        auto extrapolate = [&](double &h, double &l) {
            if (DIR) {
                h = ab2(l, h, wt);
                if (!m.doLFM) l = h;
            }
        };
#pragma unroll
        for (int q = 0; q < Q1; q++) {
            int di, dj, dk;
            place<1>(min(tid + 256 * q, NF1 - 1), di, dj, dk);
            const unsigned o = at(di, dj, dk);
            A1[q] = ldp(pln(met, (M_FACE + T1) * N3), o);
#pragma unroll
            for (int d = 0; d < 3; d++) V1[q][d] = ldp(pln(Vf, d * N3), o);
            h1[q] = ldp(pln(mfH, T1 * N3), o);
            l1[q] = ldp(pln(mfL, T1 * N3), o);
        }
#pragma unroll
        for (int q = 0; q < Q2; q++) {
            int di, dj, dk;
            place<2>(min(tid + 256 * q, NF2 - 1), di, dj, dk);
            const unsigned o = at(di, dj, dk);
            A2[q] = ldp(pln(met, (M_FACE + T2) * N3), o);
            h2[q] = ldp(pln(mfH, T2 * N3), o);
            l2[q] = ldp(pln(mfL, T2 * N3), o);
        }
        // the edge's own
        double Te[6], Tb[4], b0[2] = {0.0, 0.0}, D[4];
#pragma unroll
        for (int q = 0; q < 6; q++) Te[q] = ldp(pln(met, (M_TE + 9 * ED + 3 + q) * N3), oc);
#pragma unroll
        for (int q = 0; q < 4; q++) Tb[q] = ldp(pln(met, (M_TEB + 4 * ED + q) * N3), oc);
        if (BG) {
#pragma unroll
            for (int q = 0; q < 2; q++) b0[q] = ldp(pln(bg, (B_EDGB0 + q + 2 * ED) * N3), oc);
        }
        const double edge = ldp(pln(met, (M_EDGE + ED) * N3), oc);
        {
            constexpr int E1 = (ED == 0) ? 1 : 0, E2 = (ED == 2) ? 1 : 2;
            const unsigned s1 = (unsigned)(8 * STRIDE<E1>(g)), s2 = (unsigned)(8 * STRIDE<E2>(g));
            const unsigned od[4] = {oc, oc - s1, oc - s2, oc - s1 - s2};
            const double *Dh = DIR ? pln(S, (S_W + DEN) * N3) : pln(H, (H_GAS + DEN) * N3);
#pragma unroll
            for (int q = 0; q < 4; q++) D[q] = ldp(Dh, od[q]);
            if (DIR) {
                const double *Do = pln(O, (S_W + DEN) * N3);
#pragma unroll
                for (int q = 0; q < 4; q++) D[q] = half_prim(m, DEN, D[q], ldp(Do, od[q]), wt);
            }
        }
        // EdgeLRs' weighting (fields.F90:288-362), see edge_lr
#pragma unroll
        for (int q = 0; q < Q1; q++) {
            const int e = tid + 256 * q;
            if (e < NF1) {
                int di, dj, dk;
                const int l = place<1>(e, di, dj, dk);
                extrapolate(h1[q], l1[q]);
                sA1[e] = A1[q];
#pragma unroll
                for (int d = 0; d < 3; d++) sV[d * NF1 + e] = A1[q] * V1[q][d];
                sq1[e] = h1[q] * fmin(A1[q] * (1.0 / GAM_TINY), 1.0);
                if (l >= 0) sn1[l] = l1[q] * gam_rcp(dmax(A1[q], GAM_TINY));
            }
        }
#pragma unroll
        for (int q = 0; q < Q2; q++) {
            const int e = tid + 256 * q;
            if (e < NF2) {
                int di, dj, dk;
                const int l = place<2>(e, di, dj, dk);
                extrapolate(h2[q], l2[q]);
                sA2[e] = A2[q];
                sq2[e] = h2[q] * fmin(A2[q] * (1.0 / GAM_TINY), 1.0);
                if (l >= 0) sn2[l] = l2[q] * gam_rcp(dmax(A2[q], GAM_TINY));
            }
        }
        __syncthreads();
        // first stencil entry of this edge in each pair, and its limiter's
        auto first = [&](int P) {
            return ED == 0 ? (P == 1 ? (z * 4 + y) * 16 + x : (z * 11 + y) * 16 + x)
                           : G::ALONG_I(P) ? (y + z) * 39 + x : tid;
        };
        auto lim0 = [&](int P) {
            return ED == 0 ? (P == 1 ? (z * 4 + y) * 16 + x : (z * 7 + y) * 16 + x)
                           : G::ALONG_I(P) ? (y + z) * 39 + x + 2 : tid;
        };
        const int f1 = first(1), f2 = first(2), n1 = lim0(1), n2 = lim0(2);
        double b1L, b1R, b2L, b2R, vc[3];
        {
            const double Ai = wsum8([&](int n) { return sA1[f1 + n * G::SF(1)]; });
            // GetCornerV (fields.F90:457-517), doVdA
            const double rdA = gam_rcp(dmax(Ai, GAM_TINY));
#pragma unroll
            for (int d = 0; d < 3; d++)
                vc[d] = wsum8([&](int n) { return sV[d * NF1 + f1 + n * G::SF(1)]; }) * rdA;
            double q[8], nq[4];
#pragma unroll
            for (int n = 0; n < 8; n++) q[n] = sq1[f1 + n * G::SF(1)];
#pragma unroll
            for (int n = 0; n < 4; n++) nq[n] = sn1[n1 + n * G::SF(1)];
            recon_lr_w<RM>(m.pdmb, gam_rcp(Ai), nq, q, b1L, b1R);
        }
        {
            const double Ai = wsum8([&](int n) { return sA2[f2 + n * G::SF(2)]; });
            double q[8], nq[4];
#pragma unroll
            for (int n = 0; n < 8; n++) q[n] = sq2[f2 + n * G::SF(2)];
#pragma unroll
            for (int n = 0; n < 4; n++) nq[n] = sn2[n2 + n * G::SF(2)];
            recon_lr_w<RM>(m.pdmb, gam_rcp(Ai), nq, q, b2L, b2R);
        }
        // GetCornerD (fields.F90:427-454)
        const double Dc = 0.25 * (D[0] + D[1] + D[2] + D[3]);
        const double v = edge_value<ED, BG, BORIS>(m, vc, Dc, b1L, b1R, b2L, b2R, Te, Tb, b0, edge, clk->dt);
        if (act) stp(E + ED * N3, oc, v);
    }
};

// one edge direction, from the predictor's planes
template <int ED, int RM, bool BG, bool BORIS>
struct k_emf_t {
    static constexpr int NT = BX * BY;
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m, EdgeTile b, const Clock *clk,
                                               const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ Vf,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ E) const
    {
        __shared__ double lds[edge_geom<ED>::LDS];
        edge_tile<ED, RM, BG, BORIS, false>{}(lds, (int)bi.x, g, m, b, clk, H, S, nullptr, Vf, met, bg, E);
    }
};

static inline EdgeTile edge_tiles(int ED, const Box &b, bool slabs = false)
{
    EdgeTile t;
    t.i0 = b.i0; t.i1 = b.i1; t.j0 = b.j0; t.j1 = b.j1; t.k0 = b.k0; t.k1 = b.k1;
    const int nj = b.j1 - b.j0 + 1, nk = b.k1 - b.k0 + 1;
    t.ni = ED == 0 ? (b.i1 - b.i0 + 16) / 16 : (b.i1 - b.i0 + 32) / 32;
    const int n1 = ED == 0 ? (nj + 3) / 4 : ED == 2 ? (nj + 7) / 8 : (nk + 7) / 8;
    t.nb = t.ni * n1 * (ED == 0 ? (nk + 3) / 4 : ED == 2 ? nk : nj);
    t.qi = fast_div((unsigned)t.ni);
    t.bfirst = ED == 1 && slabs;
    t.q1 = fast_div((unsigned)(t.bfirst ? nj : n1));
    t.xs = xcd_shift(t.nb);
    return t;
}

// The three edge directions in one launch, in turn slab by slab along k (as
// k_flux3): they share face areas, fluxes and densities, which the second and
// third then find in the memory-side cache.  256x256x384 shell 3.49 -> 3.30
// ms, 192x192x256 1.33 -> 1.24, 96x96x128 0.182 -> 0.175; slabs of 16 the
// same, of 24 3.34.  Vf: the face velocities of all three directions; direction eD
// takes those of the faces along dT1.
struct Emf3 {
    EdgeTile t[3];
    int n[3];         // workgroups of each direction in a slab
    FastDiv slab;     // by the workgroups of a slab
};

template <int RM, bool BG, bool BORIS, bool DIR>
struct k_emf3 {
    static constexpr int NT = BX * BY;
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m, const Emf3 &f, const Clock *clk,
                                               const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ O,
                                               const double *__restrict__ Vf,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ E) const
    {
        __shared__ double lds[EMF_LDS];
        const int w = (int)bi.x;
        const int sl = (int)((unsigned)w / f.slab);
        int r = w - sl * (int)f.slab.d;
        if (r < f.n[0]) {
            edge_tile<0, RM, BG, BORIS, DIR>{}(lds, sl * f.n[0] + r, g, m, f.t[0], clk, H, S, O, Vf + 3 * g.N3, met, bg, E);
        } else if (r < f.n[0] + f.n[1]) {
            r -= f.n[0];
            edge_tile<1, RM, BG, BORIS, DIR>{}(lds, sl * f.n[1] + r, g, m, f.t[1], clk, H, S, O, Vf + 6 * g.N3, met, bg, E);
        } else {
            r -= f.n[0] + f.n[1];
            edge_tile<2, RM, BG, BORIS, DIR>{}(lds, sl * f.n[2] + r, g, m, f.t[2], clk, H, S, O, Vf, met, bg, E);
        }
    }
};

template <int RM, bool BG, bool BO>
static void emf3_t(hipStream_t s, const Geo &g, const MParm &m, const Box *b, const HalfSrc &h,
                   const double *Vf, const double *met, const double *bg, double *E)
{
    Emf3 f;
    int tot = 0;
    const EdgeTile t0 = edge_tiles(0, b[0]);
    const int ns = t0.nb < 2048 ? 1 : std::min((b[0].k1 - b[0].k0 + 8) / 8, t0.nb / (16 << t0.xs));
    for (int d = 0; d < 3; d++) {
        f.t[d] = edge_tiles(d, b[d], ns > 1);
        const int run = 8 << f.t[d].xs;
        f.n[d] = (f.t[d].nb + ns * run - 1) / (ns * run) * run;
        tot += f.n[d];
    }
    f.slab = fast_div((unsigned)tot);
    tot *= ns;
    const dim3 gr((unsigned)tot), bl(BX, BY);
    if (h.O) launch_f<k_emf3<RM, BG, BO, true>>(gr, bl, s, g, m, f, h.clk, h.H, h.S, h.O, Vf, met, bg, E);
    else launch_f<k_emf3<RM, BG, BO, false>>(gr, bl, s, g, m, f, h.clk, h.H, h.S, h.O, Vf, met, bg, E);
}

bool emf3_ok(const int *plan)
{
    for (int d = 0; d < 3; d++)
        if (!emf_lds(plan[d])) return false;
    return true;
}

void launch_emf3(hipStream_t s, const Geo &g, const MParm &m, const Box *b, const HalfSrc &h, const double *Vf,
                 const double *met, const double *bg, double *E)
{
    const int sel = (m.rmeth ? 4 : 0) + (m.doBG ? 2 : 0) + (m.doBoris ? 1 : 0);
    switch (sel) {
    case 0: emf3_t<0, false, false>(s, g, m, b, h, Vf, met, bg, E); break;
    case 1: emf3_t<0, false, true>(s, g, m, b, h, Vf, met, bg, E); break;
    case 2: emf3_t<0, true, false>(s, g, m, b, h, Vf, met, bg, E); break;
    case 3: emf3_t<0, true, true>(s, g, m, b, h, Vf, met, bg, E); break;
    case 4: emf3_t<1, false, false>(s, g, m, b, h, Vf, met, bg, E); break;
    case 5: emf3_t<1, false, true>(s, g, m, b, h, Vf, met, bg, E); break;
    case 6: emf3_t<1, true, false>(s, g, m, b, h, Vf, met, bg, E); break;
    default: emf3_t<1, true, true>(s, g, m, b, h, Vf, met, bg, E); break;
    }
}

template <int ED, int RM, bool BG, bool BO>
static void emf_t(hipStream_t s, int plan, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                  const double *Vf, const double *met, const double *bg, double *E)
{
    const double *H = h.H, *S = h.S;
    const Clock *clk = h.clk;
    if (emf_lds(plan)) {
        const EdgeTile t = edge_tiles(ED, b);
        const dim3 gr(xcd_grid(t.nb, t.xs)), bl(BX, BY);
        launch_f<k_emf_t<ED, RM, BG, BO>>(gr, bl, s, g, m, t, clk, H, S, Vf, met, bg, E);
        return;
    }
    const int ch = plan_chunk(plan);
    const Tile t = tile_of(b, plan_ax(plan), ch);
    if (ch == 512)
        launch_f<k_emf<ED, RM, BG, BO, 512>>(tgrid(t), dim3(BX, 8), s, g, m, t, clk, H, S, Vf, met, bg, E);
    else
        launch_f<k_emf<ED, RM, BG, BO, 128>>(tgrid(t), dim3(BX, 2), s, g, m, t, clk, H, S, Vf, met, bg, E);
}

template <int ED>
static void emf_d(hipStream_t s, int ax, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                  const double *Vf, const double *met, const double *bg, double *E)
{
    const int sel = (m.rmeth ? 4 : 0) + (m.doBG ? 2 : 0) + (m.doBoris ? 1 : 0);
    switch (sel) {
    case 0: emf_t<ED, 0, false, false>(s, ax, g, m, b, h, Vf, met, bg, E); break;
    case 1: emf_t<ED, 0, false, true>(s, ax, g, m, b, h, Vf, met, bg, E); break;
    case 2: emf_t<ED, 0, true, false>(s, ax, g, m, b, h, Vf, met, bg, E); break;
    case 3: emf_t<ED, 0, true, true>(s, ax, g, m, b, h, Vf, met, bg, E); break;
    case 4: emf_t<ED, 1, false, false>(s, ax, g, m, b, h, Vf, met, bg, E); break;
    case 5: emf_t<ED, 1, false, true>(s, ax, g, m, b, h, Vf, met, bg, E); break;
    case 6: emf_t<ED, 1, true, false>(s, ax, g, m, b, h, Vf, met, bg, E); break;
    default: emf_t<ED, 1, true, true>(s, ax, g, m, b, h, Vf, met, bg, E); break;
    }
}

void launch_emf(hipStream_t s, int eD, int ax, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                const double *Vf, const double *met, const double *bg, double *E)
{
    if (eD == 0) emf_d<0>(s, ax, g, m, b, h, Vf, met, bg, E);
    else if (eD == 1) emf_d<1>(s, ax, g, m, b, h, Vf, met, bg, E);
    else emf_d<2>(s, ax, g, m, b, h, Vf, met, bg, E);
}
