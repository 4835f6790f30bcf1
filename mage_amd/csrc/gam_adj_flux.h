// gam_adj_flux.h -- transpose of the MHD interface fluxes and of their
// reconstructions, and its gather into the cells.
#pragma once
#include "gam_adj.h"
#include "gam_launch.h"

// A workgroup of 256 threads owns 256 faces: a tile of 16 (i) x 16 (along
// D) for D = 1, 2, 256 consecutive faces of the rows along i for D = 0 (as
// the forward fluxes).  It stages the stencil cells of the half state in
// LDS with all loads in flight at once, forms the adjoint of every face
// flux, and then sums the transposed stencils of its faces over its cells
// in LDS, one variable at a time, so that what leaves are sums per cell (16
// values) and not stencil scalars per face (48).
//
// A cell within 4 of a tile's end receives from two tiles: the tile that
// holds the face of the cell's own index (the row's nearest face past the
// row's ends) writes planes 0 .. 15 of the direction's scratch, the other
// one planes 16 .. 31 (both: gas 5 and B 3 of the weighted values, then of
// the limiter values): FLUXADJ_NPL planes.  No cell is reached by three tiles, as only a
// row's last one holds fewer than 16 faces.
//
// 69 KB of LDS and 245-254 registers: two workgroups per CU either way.
// Bound by FP64 issue and by LDS reads (19 per variable and cell).  On a
// 96x96x128 shell, alone on the GPU: direct loads and 48 scalars per face
// took 259-340 us per direction and their gather 573 us; this takes 185-208
// and 259.
#define FA_I 16
#define FA_L 16

struct AdjTile {
    Tile t;                       // D = 0: the face rows; D = 1, 2: t.nb and t.xs
    int i0, i1, a0, a1, b0;       // D = 1, 2: faces along i and D, first along the third axis
    FastDiv q1, q2, q7;           // D = 1, 2: by the tiles along i and D; D = 0: by ni + 7
};

static inline AdjTile adj_tiles(int D, const Box &b)
{
    AdjTile t;
    t.t = tile_of(b, 1);
    t.q7 = t.q1 = t.q2 = fast_div((unsigned)t.t.ni + 7);
    t.i0 = b.i0;
    t.i1 = b.i1;
    t.a0 = t.a1 = t.b0 = 0;
    if (D != 0) {
        if (D == 1) { t.a0 = b.j0; t.a1 = b.j1; t.b0 = b.k0; }
        else { t.a0 = b.k0; t.a1 = b.k1; t.b0 = b.j0; }
        const int nti = (t.i1 - t.i0 + FA_I) / FA_I, nta = (t.a1 - t.a0 + FA_L) / FA_L;
        t.t.nb = nti * nta * (D == 1 ? b.k1 - b.k0 + 1 : b.j1 - b.j0 + 1);
        t.t.xs = xcd_shift(t.t.nb);
        t.q1 = fast_div((unsigned)nti);
        t.q2 = fast_div((unsigned)nta);
    }
    return t;
}

template <int D> struct adj_geom {
    static constexpr int NE = D == 0 ? 376 : (FA_L + 7) * FA_I;   // cells staged (D = 0: at most)
    static constexpr int NL = D == 0 ? 376 : (FA_L + 3) * FA_I;   // limiter cells staged
    static constexpr int SN = D == 0 ? 1 : FA_I;                  // LDS step of the stencil
    static constexpr int LO = D == 0 ? 0 : 2 * FA_I;              // first staged cell with a limiter entry
    static constexpr int G0 = 7 * SN;                             // zero slots before the first face's
    static constexpr int NS = G0 + NE;                            // face slots, zero where no face is
    static constexpr int LDS = 9 * NE + 8 * NL + 6 * NS;
};
#define FLUXADJ_LDS (adj_geom<0>::LDS)
static_assert(adj_geom<1>::LDS <= FLUXADJ_LDS, "LDS planes");

// workgroup w of the launch's range for direction D; lds: FLUXADJ_LDS doubles
template <int D, int RM, bool BG, bool BORIS>
__device__ __forceinline__ void flux_adj_tile(double *lds, int w, const Geo &g, const MParm &m, const AdjTile &t,
                                              const double *__restrict__ H,
                                              const double *__restrict__ S,
                                              const double *__restrict__ met,
                                              const double *__restrict__ bg,
                                              const double *__restrict__ ag,
                                              const double *__restrict__ amf,
                                              double *__restrict__ sc,
                                              double *__restrict__ aHMF,
                                              double *__restrict__ aHG)
{
    using A = adj_geom<D>;
    constexpr int NE = A::NE, NL = A::NL, SN = A::SN, LO = A::LO, G0 = A::G0, NS = A::NS;
    // volumes; weighted values and limiter values by variable; face slots
    double *const sv = lds, *const sq = lds + NE, *const sl = sq + 8 * NE, *const ss = sl + 8 * NL;
    const int L = xcd_tile(w, t.t.xs);
    if (L >= t.t.nb) return;                   // whole workgroup
    const int tid = (int)threadIdx.x;
    const long N3 = g.N3;
    const unsigned s8 = (unsigned)(8 * STRIDE<D>(g));

    // this thread's face (byte offset oc, stencil's first LDS entry f0) and
    // the two cells it stages, sums and writes (own: to the first 16 planes)
    unsigned oc, oe[2];
    bool act, put[2], own[2], wr[2];
    int f0;
    if (D == 0) {
        const unsigned ni = (unsigned)t.t.ni, tot = ni * (unsigned)(t.t.nj * t.t.nk);
        const unsigned p0 = (unsigned)L * 256u, R0 = p0 / t.t.qi, q0 = p0 - R0 * ni;
        const unsigned nf = tot - p0 < 256u ? tot - p0 : 256u;   // faces of this workgroup
        const unsigned n0 = (ni - q0 < nf ? ni - q0 : nf) + 7;   // cells of the first row
        const unsigned nr = (q0 + nf - 1) / t.t.qi;              // rows after the first
        const unsigned ne = nf + 7 * (nr + 1);                   // cells in all
        act = (unsigned)tid < nf;
        const unsigned p = act ? (unsigned)tid : 0u, r0 = (q0 + p) / t.t.qi;
        int j, k;
        tile_row(t.t, R0 + r0, j, k);
        oc = (unsigned)(8 * IX(g, t.t.b.i0 + (int)(q0 + p - r0 * ni), j, k));
        f0 = (int)(p + 7 * r0);
#pragma unroll
        for (int q = 0; q < 2; q++) {
            unsigned e = (unsigned)(tid + 256 * q);
            wr[q] = put[q] = e < ne;
            if (!put[q]) e = 0;
            // cells of the first row, then ni + 7 of each row after it
            const unsigned r = e < n0 ? 0u : 1u + (e - n0) / t.q7;
            const int x = (int)(e < n0 ? q0 + e : e - n0 - (r - 1u) * (ni + 7)) - 4;
            const unsigned xf = x < 0 ? 0u : (unsigned)x < ni ? (unsigned)x : ni - 1;
            own[q] = (((R0 + r) * ni + xf) >> 8) == (unsigned)L;
            tile_row(t.t, R0 + r, j, k);
            oe[q] = (unsigned)(8 * IX(g, t.t.b.i0 + x, j, k));
        }
    } else {
        const unsigned r = (unsigned)L / t.q1, ti = (unsigned)L - r * t.q1.d;
        const unsigned r2 = r / t.q2, ta = r - r2 * t.q2.d;
        const int b = t.b0 + (int)r2, i0 = t.i0 + (int)ti * FA_I, a0 = t.a0 + (int)ta * FA_L;
        // a cell past the box reads the last one inside (only lanes of
        // faces outside the box use it)
        auto at = [&](int i, int a) -> unsigned {
            i = i < t.i1 ? i : t.i1;
            a = a < t.a1 + 3 ? a : t.a1 + 3;
            return (unsigned)(8 * (D == 1 ? IX(g, i, a, b) : IX(g, i, b, a)));
        };
        const int tx = tid & (FA_I - 1), ty = tid / FA_I;
        act = i0 + tx <= t.i1 && a0 + ty <= t.a1;
        oc = at(i0 + tx, a0 + ty < t.a1 ? a0 + ty : t.a1);
        f0 = tid;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int a = a0 - 4 + ty + FA_L * q;
            put[q] = tid + 256 * q < NE;
            wr[q] = put[q] && i0 + tx <= t.i1 && a <= t.a1 + 3;
            const int af = a < t.a0 ? t.a0 : a < t.a1 ? a : t.a1;   // the cell's face
            own[q] = af >= a0 && af < a0 + FA_L;
            oe[q] = at(i0 + tx, put[q] ? a : a0);
        }
    }
    {
        const double *Wv = H + H_WH * N3, *Wl = H + H_WN * N3;
        const double *Bh = H + H_B * N3, *Bl = m.doLFM ? S + S_B * N3 : Bh;
        double v[2], wq[2][8], wl[2][8];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            v[q] = ldp(met + M_VOL * N3, oe[q]);
#pragma unroll
            for (int n = 0; n < 5; n++) {
                wq[q][n] = ldp(pln(Wv, n * N3), oe[q]);
                wl[q][n] = ldp(pln(Wl, n * N3), oe[q]);
            }
#pragma unroll
            for (int x = 0; x < 3; x++) {
                wq[q][5 + x] = ldp(pln(Bh, x * N3), oe[q]);
                wl[q][5 + x] = ldp(pln(Bl, x * N3), oe[q]);
            }
        }
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int e = tid + 256 * q;
            if (put[q]) {
                sv[e] = v[q];
#pragma unroll
                for (int n = 0; n < 8; n++) sq[n * NE + e] = n < 5 ? wq[q][n] : v[q] * wq[q][n];
                if (e >= LO && e - LO < NL)
#pragma unroll
                    for (int n = 0; n < 8; n++) sl[n * NL + e - LO] = wl[q][n];
            }
        }
        for (int e = tid; e < NS; e += 256)
#pragma unroll
            for (int n = 0; n < 6; n++) ss[n * NS + e] = 0.0;
    }
    __syncthreads();
    const double rVi = gam_rcp(wsum8([&](int n) { return sv[f0 + n * SN]; }));
    auto stencil = [&](int v, double *qv, double *nq) {
#pragma unroll
        for (int n = 0; n < 8; n++) qv[n] = sq[v * NE + f0 + n * SN];
#pragma unroll
        for (int n = 0; n < 4; n++) nq[n] = sl[v * NL + f0 + (D == 0 ? n + 2 : n * SN)];
    };
    // adjoints of the left and right states: gas 5, B 3
    double aL[8], aR[8];
#pragma unroll
    for (int v = 0; v < 8; v++) aL[v] = aR[v] = 0.0;
    if (act) {
        double WL[8], WR[8];
#pragma unroll
        for (int v = 0; v < 8; v++) {
            double qv[8], nq[4];
            stencil(v, qv, nq);
            recon_lr_w<RM>(m.pdmb, rVi, nq, qv, WL[v], WR[v]);
        }
        const double faB = ldp(met + (M_FACE + D) * N3, oc);
        double aF[5], aM[3];
        for (int v = 0; v < 5; v++) aF[v] = faB * ldp(ag + (v + 5 * D) * N3, oc);
        for (int x = 0; x < 3; x++) aM[x] = faB * ldp(amf + (x + 3 * D) * N3, oc);
        double T[9], vL[3], vR[3], aFt[3];
        for (int q = 0; q < 3; q++) T[q] = ldp(met + (M_TF + q + 9 * D) * N3, oc);
        if (m.ortho) {
            face_tangent_n(T, WL, vL);
            face_tangent_n(T, WR, vR);
            face_tangent_n(T, aF, aFt);
        } else {
            for (int q = 3; q < 9; q++) T[q] = ldp(met + (M_TF + q + 9 * D) * N3, oc);
            face_tangent(T, WL, vL);
            face_tangent(T, WR, vR);
            face_tangent(T, aF, aFt);
        }
        const double iFaB = gam_rcp(faB);
        const double Bn = ldp(H + (H_MF + D) * N3, oc) * iFaB;
        double B0[3] = {0, 0, 0}, B0n = 0.0;
        if (BG) {
            for (int x = 0; x < 3; x++) B0[x] = ldp(bg + (B_FCB0 + x + 3 * D) * N3, oc);
            B0n = ldp(bg + (B_BFLUX0 + D) * N3, oc) * iFaB;
        }
        // forward pieces the adjoint needs: VaD, bbD and the HOGS differences
        double mF[3] = {0, 0, 0}, bbD = 0.0, VaD = 0.0;
        mag_kin<BG, BORIS>(m, -1.0, WL, WL + 5, Bn, T, B0, B0n, mF, bbD, VaD);
        mag_kin<BG, BORIS>(m, +1.0, WR, WR + 5, Bn, T, B0, B0n, mF, bbD, VaD);
        double adW[5], aVaD = 0.0, abbD = 0.0, aBn = 0.0;
        {
            auto en = [&](const double *W) {
                return 0.5 * W[DEN] * (W[1] * W[1] + W[2] * W[2] + W[3] * W[3]) + W[PRS] * m.igm1;
            };
            const double dW[5] = {WR[DEN] - WL[DEN], WR[DEN] * WR[1] - WL[DEN] * WL[1],
                                  WR[DEN] * WR[2] - WL[DEN] * WL[2], WR[DEN] * WR[3] - WL[DEN] * WL[3],
                                  en(WR) - en(WL)};
            for (int v = 0; v < 5; v++) {
                adW[v] = -m.cHogH * VaD * aF[v];
                aVaD += -m.cHogH * dW[v] * aF[v];
            }
        }
        if (BORIS) {
            // mag-HOGS: mF -= cHogM VaD bbD (WR - WL)_v / Ca^2
            for (int x = 0; x < 3; x++) {
                const double dv = WR[1 + x] - WL[1 + x];
                const double deeP = bbD * dv * m.iCa2;
                aVaD += -m.cHogM * deeP * aM[x];
                const double adeeP = -m.cHogM * VaD * aM[x];
                abbD += dv * m.iCa2 * adeeP;
                aR[1 + x] += bbD * m.iCa2 * adeeP;
                aL[1 + x] -= bbD * m.iCa2 * adeeP;
            }
            // nuke: gF -= Ca (U(c) - U(c - s)) where the mean speed is large
            const double v2L = WL[1] * WL[1] + WL[2] * WL[2] + WL[3] * WL[3];
            const double v2R = WR[1] * WR[1] + WR[2] * WR[2] + WR[3] * WR[3];
            // (the forward's own test, made only near and past its line)
            bool nuke = v2L + v2R >= 4.49 * m.Ca * m.Ca;
            if (nuke) {
                const double sL = sqrt(v2L), sR = sqrt(v2R);
                nuke = sqrt(sL * sL + sR * sR) / GAM_SQRT2_SP >= 1.5 * m.Ca;
            }
            if (nuke)
                for (int v = 0; v < 5; v++) {
                    unsafeAtomicAdd((double *)((char *)(aHG + v * N3) + oc), -m.Ca * aF[v]);
                    unsafeAtomicAdd((double *)((char *)(aHG + v * N3) + (oc - s8)), m.Ca * aF[v]);
                }
        }
        gas_kin_adj_vt(m.igm1, -1.0, WL, T, vL, aF, aFt, aL, adW);
        gas_kin_adj_vt(m.igm1, +1.0, WR, T, vR, aF, aFt, aR, adW);
        mag_kin_adj<BG, BORIS>(m, -1.0, WL, WL + 5, Bn, T, B0, B0n, aM, aVaD, abbD, aL, aL + 5, aBn);
        mag_kin_adj<BG, BORIS>(m, +1.0, WR, WR + 5, Bn, T, B0, B0n, aM, aVaD, abbD, aR, aR + 5, aBn);
        // the only writer of this face since the EMF transpose's gather
        stp(aHMF + D * N3, oc, ldp(aHMF + D * N3, oc) + aBn * iFaB);
    }
    // the reconstructions' transposes, one variable at a time: per face the
    // stencil scalars and the four limiter adjoints, summed over the cells
    const int fs = G0 + f0;
    double *pc[2];   // the cells in the first of their 16 planes
#pragma unroll
    for (int q = 0; q < 2; q++) pc[q] = (double *)((char *)(own[q] ? sc : sc + 16 * N3) + oe[q]);
#pragma unroll
    for (int v = 0; v < 8; v++) {
        if (act) {
            double qv[8], nq[4], an[4] = {0, 0, 0, 0}, l, r;
            stencil(v, qv, nq);
            recon_lr_w_adj_s<RM>(m.pdmb, rVi, nq, qv, aL[v], aR[v], an, l, r);
            ss[fs] = l;
            ss[NS + fs] = r;
#pragma unroll
            for (int n = 0; n < 4; n++) ss[(2 + n) * NS + fs] = an[n];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (!wr[q]) continue;
            // staged cell e is stencil point n of the face in slot e - n
            const int e = G0 + tid + 256 * q;
            double gh = 0.0, gn = 0.0;
#pragma unroll
            for (int n = 0; n < 8; n++) {
                if (RM == 1) {
                    if (n <= 6) gh += UP7(n) * ss[e - n * SN];
                    if (n >= 1) gh += UP7(7 - n) * ss[NS + e - n * SN];
                } else {
                    gh += W8(n) * ss[e - n * SN];
                }
            }
#pragma unroll
            for (int n = 0; n < 4; n++) gn += ss[(2 + n) * NS + e - (n + 2) * SN];
            pc[q][v * N3] = gh;
            pc[q][(8 + v) * N3] = gn;
        }
        if (v < 7) __syncthreads();
    }
}

// The workgroups of the three directions one after another, as k_flux3
struct FluxAdj3 {
    AdjTile t[3];
    int start[2];     // first workgroup of direction 1, of direction 2
};

template <int RM, bool BG, bool BORIS>
__global__ __launch_bounds__(256, 2) void k_flux_adj_mhd(Geo g, MParm m, FluxAdj3 f,
                                                      const double *__restrict__ H,
                                                      const double *__restrict__ S,
                                                      const double *__restrict__ met,
                                                      const double *__restrict__ bg,
                                                      const double *__restrict__ ag,
                                                      const double *__restrict__ amf,
                                                      double *__restrict__ sc,
                                                      double *__restrict__ aHMF,
                                                      double *__restrict__ aHG)
{
    __shared__ double lds[FLUXADJ_LDS];
    const int w = (int)blockIdx.x;
    const long ns = FLUXADJ_NPL * g.N3;
    if (w < f.start[0])
        flux_adj_tile<0, RM, BG, BORIS>(lds, w, g, m, f.t[0], H, S, met, bg, ag, amf, sc, aHMF, aHG);
    else if (w < f.start[1])
        flux_adj_tile<1, RM, BG, BORIS>(lds, w - f.start[0], g, m, f.t[1], H, S, met, bg, ag, amf, sc + ns, aHMF, aHG);
    else
        flux_adj_tile<2, RM, BG, BORIS>(lds, w - f.start[1], g, m, f.t[2], H, S, met, bg, ag, amf, sc + 2 * ns, aHMF, aHG);
}
