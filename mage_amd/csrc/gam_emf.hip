// gam_emf.hip -- edge EMFs (CalcElecField, fields.F90:70-517).
#include "gam_launch.h"

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

template <int ED, int RM, bool BG, bool BORIS>
struct edge_emf {
    __device__ __forceinline__ void operator()(int w, const Geo &g, const MParm &m,
                                               const Tile &b, const Clock *clk,
                                               const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ Vf,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ E) const
    {
        int i, j, k;
        if (!tile_point(b, w, i, j, k)) return;
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
        const double *Te = met + (long)(M_TE + 9 * ED) * N3 + c;
        const double v1 = vc[0] * Te[3 * N3] + vc[1] * Te[4 * N3] + vc[2] * Te[5 * N3];
        const double v2 = vc[0] * Te[6 * N3] + vc[1] * Te[7 * N3] + vc[2] * Te[8 * N3];
        double vDiff = gam_sqrt(v1 * v1 + v2 * v2);

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
        const double *Tb = met + (long)(M_TEB + 4 * ED) * N3 + c;
        const double xni = Tb[0], yni = Tb[N3], xnj = Tb[2 * N3], ynj = Tb[3 * N3];
        const double detT = gam_rcp(xni * ynj - xnj * yni);
        const double bT1 = 0.5 * (bT1L + bT1R);
        const double bT2 = 0.5 * (bT2L + bT2R);
        const double Jd = (bT2R - bT2L) - (bT1R - bT1L);
        double b1 = detT * (ynj * bT1 - yni * bT2);
        double b2 = detT * (-(xnj * bT1) + xni * bT2);
        if (BG) {
            b1 = b1 + bg[(B_EDGB0 + 0 + 2 * ED) * N3 + c];
            b2 = b2 + bg[(B_EDGB0 + 1 + 2 * ED) * N3 + c];
        }
        const double edge = met[(M_EDGE + ED) * N3 + c];
        // vA = |b| / sqrt(D), with Boris Ca vA / sqrt(Ca^2 + vA^2)
        const double bb = b1 * b1 + b2 * b2, Ca2 = m.Ca * m.Ca;
        const double vA = gam_sqrt(BORIS ? Ca2 * bb * gam_rcp(Ca2 * Dc + bb) : bb * gam_rcp(Dc));
        vDiff = vDiff + vA;
        vDiff = dmin(vDiff, m.CFL * edge * gam_rcp(clk->dt));
        const double e = -(v1 * b2 - v2 * b1) + m.Vd0 * vDiff * Jd;
        E[ED * N3 + c] = e * edge;
    }
};

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
        edge_emf<ED, RM, BG, BORIS>{}((int)bi.x, g, m, b, clk, H, S, Vf, met, bg, E);
    }
};

// The three edge directions in one launch, one range of workgroups after
// another.  Vf: the face velocities of all three directions; direction eD
// takes those of the faces along dT1.
struct Emf3 {
    Tile t[3];
    int start[2];     // first workgroup of edge direction 1, of direction 2
};

template <int RM, bool BG, bool BORIS>
struct k_emf3 {
    static constexpr int NT = BX * BY;
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m, const Emf3 &f, const Clock *clk,
                                               const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ Vf,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ E) const
    {
        const int w = (int)bi.x;
        if (w < f.start[0])
            edge_emf<0, RM, BG, BORIS>{}(w, g, m, f.t[0], clk, H, S, Vf + 3 * g.N3, met, bg, E);
        else if (w < f.start[1])
            edge_emf<1, RM, BG, BORIS>{}(w - f.start[0], g, m, f.t[1], clk, H, S, Vf + 6 * g.N3, met, bg, E);
        else
            edge_emf<2, RM, BG, BORIS>{}(w - f.start[1], g, m, f.t[2], clk, H, S, Vf, met, bg, E);
    }
};

template <int RM, bool BG, bool BO>
static void emf3_t(hipStream_t s, const int *plan, const Geo &g, const MParm &m, const Box *b, const Clock *clk,
                   const double *H, const double *S, const double *Vf, const double *met, const double *bg,
                   double *E)
{
    Emf3 f;
    int tot = 0;
    for (int d = 0; d < 3; d++) {
        f.t[d] = tile_of(b[d], plan_ax(plan[d]));
        tot += (int)tgrid(f.t[d]).x;
        if (d < 2) f.start[d] = tot;
    }
    launch_f<k_emf3<RM, BG, BO>>(dim3((unsigned)tot), dim3(BX, BY), s, g, m, f, clk, H, S, Vf, met, bg, E);
}

bool emf3_ok(const int *plan)
{
    for (int d = 0; d < 3; d++)
        if (plan_chunk(plan[d]) != BX * BY) return false;
    return true;
}

void launch_emf3(hipStream_t s, const int *plan, const Geo &g, const MParm &m, const Box *b, const Clock *clk,
                 const double *H, const double *S, const double *Vf, const double *met, const double *bg, double *E)
{
    const int sel = (m.rmeth ? 4 : 0) + (m.doBG ? 2 : 0) + (m.doBoris ? 1 : 0);
    switch (sel) {
    case 0: emf3_t<0, false, false>(s, plan, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 1: emf3_t<0, false, true>(s, plan, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 2: emf3_t<0, true, false>(s, plan, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 3: emf3_t<0, true, true>(s, plan, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 4: emf3_t<1, false, false>(s, plan, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 5: emf3_t<1, false, true>(s, plan, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 6: emf3_t<1, true, false>(s, plan, g, m, b, clk, H, S, Vf, met, bg, E); break;
    default: emf3_t<1, true, true>(s, plan, g, m, b, clk, H, S, Vf, met, bg, E); break;
    }
}

template <int ED, int RM, bool BG, bool BO>
static void emf_t(hipStream_t s, int plan, const Geo &g, const MParm &m, const Box &b, const Clock *clk,
                  const double *H, const double *S, const double *Vf, const double *met,
                  const double *bg, double *E)
{
    const int ch = plan_chunk(plan);
    const Tile t = tile_of(b, plan_ax(plan), ch);
    if (ch == 512)
        launch_f<k_emf<ED, RM, BG, BO, 512>>(tgrid(t), dim3(BX, 8), s, g, m, t, clk, H, S, Vf, met, bg, E);
    else if (ch == 128)
        launch_f<k_emf<ED, RM, BG, BO, 128>>(tgrid(t), dim3(BX, 2), s, g, m, t, clk, H, S, Vf, met, bg, E);
    else
        launch_f<k_emf<ED, RM, BG, BO>>(tgrid(t), dim3(BX, BY), s, g, m, t, clk, H, S, Vf, met, bg, E);
}

template <int ED>
static void emf_d(hipStream_t s, int ax, const Geo &g, const MParm &m, const Box &b, const Clock *clk,
                  const double *H, const double *S, const double *Vf, const double *met,
                  const double *bg, double *E)
{
    const int sel = (m.rmeth ? 4 : 0) + (m.doBG ? 2 : 0) + (m.doBoris ? 1 : 0);
    switch (sel) {
    case 0: emf_t<ED, 0, false, false>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 1: emf_t<ED, 0, false, true>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 2: emf_t<ED, 0, true, false>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 3: emf_t<ED, 0, true, true>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 4: emf_t<ED, 1, false, false>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 5: emf_t<ED, 1, false, true>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E); break;
    case 6: emf_t<ED, 1, true, false>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E); break;
    default: emf_t<ED, 1, true, true>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E); break;
    }
}

void launch_emf(hipStream_t s, int eD, int ax, const Geo &g, const MParm &m, const Box &b, const Clock *clk,
                const double *H, const double *S, const double *Vf, const double *met,
                const double *bg, double *E)
{
    if (eD == 0) emf_d<0>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E);
    else if (eD == 1) emf_d<1>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E);
    else emf_d<2>(s, ax, g, m, b, clk, H, S, Vf, met, bg, E);
}
