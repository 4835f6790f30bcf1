// gam_flux.h -- interface-flux kernels (Fluxes, stress.F90:204-599) and
// their launches, one face direction per source file.
#pragma once
#include "gam_launch.h"

// ====================================================================
// The fluxes of one face from its reconstructed L/R states (the part of
// Fluxes, stress.F90:204-429, after BlockStateLRs): magnetic kinetic flux
// with the B0 terms, Boris mag-HOGS, gas kinetic flux, HOGS and the nuke
// term, times the face area, stored to gFlx/mFlx of direction D.  AT(p)
// reads plane p at the face point; HALF_MF() is the half-state face flux,
// HALF_DU the half-state gas less that of the cell below the face along D;
// RECON_B(BL, BR) fills the magnetic L/R states (called only with MHD on,
// after the metric loads, which keeps the register peak of the fused
// kernel at that of the gas part); oc is the face's byte offset for the
// stores.
// ====================================================================
template <int D, bool BG, bool BORIS, class AtF, class HalfF, class DuF, class ReconB>
__device__ __forceinline__ void face_flux_lr(const Geo &g, const MParm &m,
                                             const double *__restrict__ met,
                                             const double *__restrict__ bg, AtF AT, HalfF HALF_MF, DuF HALF_DU,
                                             ReconB RECON_B, const double *WL,
                                             const double *WR, double *BL, double *BR,
                                             unsigned oc,
                                             double *__restrict__ gflx,
                                             double *__restrict__ mflx)
{
    const long N3 = g.N3;
    // Of the triad only the normal is read where it is orthonormal (18 of the
    // step's ~310 words per point): the tangential velocity is what the
    // normal leaves.  256x256x384 shell: fluxes 5.67 -> 5.08 ms per step.
    double T[3], vtL[3], vtR[3];
#pragma unroll
    for (int q = 0; q < 3; q++) T[q] = AT(met + (M_TF + q + 9 * D) * N3);
    if (m.ortho) {
        face_tangent_n(T, WL, vtL);
        face_tangent_n(T, WR, vtR);
    } else {
        double Tt[9];
#pragma unroll
        for (int q = 3; q < 9; q++) Tt[q] = AT(met + (M_TF + q + 9 * D) * N3);
        face_tangent(Tt, WL, vtL);
        face_tangent(Tt, WR, vtR);
    }
    const double faB = AT(met + (M_FACE + D) * N3);

    double VaD = 0.0;
    if (m.doMHD) {
        RECON_B(BL, BR);
        const double iFaB = gam_rcp(faB);
        const double Bn = HALF_MF() * iFaB;
        double B0[3] = {0.0, 0.0, 0.0}, B0n = 0.0;
        if (BG) {
#pragma unroll
            for (int x = 0; x < 3; x++) B0[x] = AT(bg + (B_FCB0 + x + 3 * D) * N3);
            B0n = AT(bg + (B_BFLUX0 + D) * N3) * iFaB;
        }
        double mF[3] = {0.0, 0.0, 0.0}, bbD = 0.0;
        mag_kin<BG, BORIS>(m, -1.0, WL, BL, Bn, T, B0, B0n, mF, bbD, VaD);
        mag_kin<BG, BORIS>(m, +1.0, WR, BR, Bn, T, B0, B0n, mF, bbD, VaD);
        if (BORIS) {
#pragma unroll
            for (int x = 0; x < 3; x++) {
                double deeP = bbD * (WR[1 + x] - WL[1 + x]) * m.iCa2;
                mF[x] = mF[x] - m.cHogM * VaD * deeP;
            }
        }
#pragma unroll
        for (int x = 0; x < 3; x++) stp(mflx + (x + 3 * D) * N3, oc, faB * mF[x]);
    }

    double gF[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, dW[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    gas_kin_vt(m.igm1, -1.0, WL, T, vtL, gF, dW);
    gas_kin_vt(m.igm1, +1.0, WR, T, vtR, gF, dW);
#pragma unroll
    for (int v = 0; v < 5; v++) gF[v] = gF[v] - m.cHogH * VaD * dW[v];
    if (BORIS) {   // "nuclear option" (stress.F90:399-417)
        const double vL2 = WL[1] * WL[1] + WL[2] * WL[2] + WL[3] * WL[3];
        const double vR2 = WR[1] * WR[1] + WR[2] * WR[2] + WR[3] * WR[3];
        // the square roots of the test only where its square comes near
        bool nuke = vL2 + vR2 >= 4.4999 * m.Ca * m.Ca;
        if (nuke) {
            const double vL = sqrt(vL2), vR = sqrt(vR2);
            nuke = sqrt(vL * vL + vR * vR) / GAM_SQRT2_SP >= 1.5 * m.Ca;
        }
        if (nuke) {
            double dU[5];
            HALF_DU(dU);
#pragma unroll
            for (int v = 0; v < 5; v++) gF[v] = gF[v] - m.Ca * dU[v];
        }
    }
#pragma unroll
    for (int v = 0; v < 5; v++) stp(gflx + (v + 5 * D) * N3, oc, faB * gF[v]);
}

// ====================================================================
// Interface fluxes of one direction (Fluxes, stress.F90:204-429), every
// stencil point read from global memory (used along i, where the 8 points
// are contiguous and merge into wide loads)
// ====================================================================
template <int D, int RM, bool BG, bool BORIS, int NTH = BX * BY>
struct k_flux {
    static constexpr int NT = NTH;
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m,
                                               Tile b, const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ gflx,
                                               double *__restrict__ mflx,
                                               double *__restrict__ Vf) const
    {
        TILE_IJK(b);
        const long N3 = g.N3;
        const long c = IX(g, i, j, k);
        const long s = STRIDE<D>(g);
        // byte offsets of the 8 stencil points (cells c-4s .. c+3s), shared by
        // every plane; o[4] is the face point c itself.  Along i the points are
        // contiguous and the compiler merges them into wide loads from one
        // address, so that direction keeps plain indexing.
        unsigned o[8];
#pragma unroll
        for (int n = 0; n < 8; n++) o[n] = (unsigned)((c + (n - 4) * s) * 8);
        auto LD = [&](const double *__restrict__ plane, int n) -> double {
            if (D == 0) return plane[c + (n - 4)];
            return ldp(plane, o[n]);
        };

        double vol[8];
#pragma unroll
        for (int n = 0; n < 8; n++) vol[n] = LD(met + M_VOL * N3, n);
        const double Vi = wsum8([&](int n) { return vol[n]; });
        const double rVi = gam_rcp(Vi);

        // L/R primitives (BlockStateLRs, recon.F90:39-93); Wv holds V*W
        const double *Wv = H + H_WH * N3;
        const double *Wl = H + H_WN * N3;
        double WL[5], WR[5];
#pragma unroll
        for (int v = 0; v < 5; v++) {
            double qv[8], nq[4];
#pragma unroll
            for (int n = 0; n < 8; n++) qv[n] = LD(Wv + v * N3, n);
#pragma unroll
            for (int n = 0; n < 4; n++) nq[n] = LD(Wl + v * N3, n + 2);
            recon_lr_w<RM>(m.pdmb, rVi, nq, qv, WL[v], WR[v]);
            // Mom2Face of this face from the same velocity stencil
            // (written without a condition on Vf: a branch here keeps the
            // stencils alive and costs ~30 VGPRs)
            if (v >= 1 && v <= 3) stp(Vf + (v - 1) * N3, o[4], mom2face(qv, Vi, rVi));
        }
        auto recon_b = [&](double *BL, double *BR) {
            const double *Bh = H + H_B * N3;
            const double *Bl = m.doLFM ? S + S_B * N3 : Bh;
#pragma unroll
            for (int x = 0; x < 3; x++) {
                double q[8], nq[4];
#pragma unroll
                for (int n = 0; n < 8; n++) q[n] = LD(Bh + x * N3, n);
#pragma unroll
                for (int n = 0; n < 4; n++) nq[n] = LD(Bl + x * N3, n + 2);
                recon_lr<RM>(m.pdmb, vol, rVi, nq, q, BL[x], BR[x]);
            }
        };
        double BL[3], BR[3];
        face_flux_lr<D, BG, BORIS>(
            g, m, met, bg, [&](const double *p) { return LD(p, 4); }, [&]() { return LD(H + (H_MF + D) * N3, 4); },
            [&](double *dU) {
                for (int v = 0; v < 5; v++) dU[v] = LD(H + (H_GAS + v) * N3, 4) - LD(H + (H_GAS + v) * N3, 3);
            },
            recon_b, WL, WR, BL, BR, o[4], gflx, mflx);
    }
};

// ====================================================================
// Interface fluxes with the stencils in LDS.  A workgroup of 256 threads
// owns 256 faces and brings every stencil plane of their cells to LDS with
// ALL loads of the gas and field planes in flight at once: two waits on
// memory per workgroup (stencils, face data) instead of one per variable.
//   D = 1, 2: a tile of 32 (i) x 8 (along D) faces, 15 x 32 cells
//             (1.9 cells loaded per face);
//   D = 0:    256 consecutive faces of the rows along i (whole and partial
//             rows, no idle lane), their cells packed row by row with the 7
//             extra ones each row needs.
// Two phases share the LDS planes: the five gas variables, then the three
// field components, whose loads wait in registers meanwhile; 37 KB (33 for
// D = 0) and 128 registers leave room for four workgroups per CU.
// DIR (1; 2 without a magnetic field): the half state is formed as the cells are staged, from the primitives
// and cell B that the last two steps left (S_W, S_B of State and oState): as
// many words as the predictor's planes, which are then neither written nor
// read (HalfSrc says when).
// The tile's 32 points are two whole 128-byte lines of every row.
// Bound by memory traffic, close behind by FP64 issue (1075 vector
// instructions per face; at 1580 the clock fell to 1.8 GHz).  256x256x384
// shell, per launch: a 64 x 4 tile staged one variable at a time took 2.35
// ms for D = 1, 2 (9.15 GB), direct loads 2.02 ms for D = 0 (9.1 GB); this
// form 1.75-1.84 ms and 1.92 ms (9.0 GB at 5.0 TB/s; the streaming rate of
// 32 read and 11 written planes is 5.2-5.5).  With the normal alone of
// orthonormal triads and the directions in slabs (k_flux3) 1.68 ms a direction
// (9.6 GB at 5.7 TB/s).
// ====================================================================
struct FluxTile {
    Tile t;                       // D = 0: the face rows; D = 1, 2: t.nb and t.xs
    int i0, i1, a0, a1, b0;       // D = 1, 2: faces along i and D, first along the third axis
    int byD;                      // D = 1, 2: tiles numbered along i, D, the third axis (0),
                                  // along D, i, the third axis (1) or along i, the third, D (2)
    FastDiv q1, q2;               // D = 1, 2: by the tiles of the first and the second of those
    FastDiv q7;                   // D = 0: by ni + 7
};

#define FLUX_LDS ((8 + 3) * 376 > (8 + 7) * 32 * 6 + (8 + 3) * 32 * 5 ? (8 + 3) * 376 : (8 + 7) * 32 * 6 + (8 + 3) * 32 * 5)

template <int D, int RM, bool BG, bool BORIS, int DIR>
struct flux_tile {
    static constexpr int TI = 32, TA = 8;
    static constexpr int NE = D == 0 ? 376 : (TA + 7) * TI;   // cells staged (D = 0: at most)
    static constexpr int NL = D == 0 ? 376 : (TA + 3) * TI;   // limiter cells staged
    static constexpr int SN = D == 0 ? 1 : TI;                // LDS step of the stencil
    static constexpr int LO = D == 0 ? 0 : 2 * TI;            // first staged cell with a limiter entry
    static_assert(6 * NE + 5 * NL <= FLUX_LDS, "LDS planes");
    // workgroup w of the launch's range for this direction; lds: FLUX_LDS doubles
    __device__ __forceinline__ void operator()(double *lds, int w, const Geo &g, const MParm &m,
                                               const FluxTile &t, const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ O, const Clock *clk,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ gflx,
                                               double *__restrict__ mflx,
                                               double *__restrict__ Vf) const
    {
        double *sv = lds;                                     // volumes
        auto sq = [&](int n) { return lds + (1 + n) * NE; };  // weighted values
        auto sl = [&](int n) { return lds + 6 * NE + n * NL; };   // limiter values
        const int L = xcd_tile(w, t.t.xs);
        if (L >= t.t.nb) return;                   // whole workgroup
        const int tid = (int)(threadIdx.x + BX * threadIdx.y);
        const long N3 = g.N3;
        const unsigned s8 = (unsigned)(8 * STRIDE<D>(g));

        // this thread's face (byte offset oc, stencil's first LDS entry f0)
        // and the two cells it stages
        unsigned oc, oe[2];
        bool act, put[2];
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
                put[q] = e < ne;
                if (!put[q]) e = 0;
                // cells of the first row, then ni + 7 of each row after it
                const unsigned r = e < n0 ? 0u : 1u + (e - n0) / t.q7;
                const unsigned x = e < n0 ? q0 + e : e - n0 - (r - 1u) * (ni + 7);
                tile_row(t.t, R0 + r, j, k);
                oe[q] = (unsigned)(8 * IX(g, t.t.b.i0 - 4 + (int)x, j, k));
            }
        } else {
            // (byD says what x and y run along)
            const unsigned r = (unsigned)L / t.q1, x = (unsigned)L - r * t.q1.d;
            const unsigned r2 = r / t.q2, y = r - r2 * t.q2.d;
            const int ti = (int)(t.byD == 1 ? y : x), ta = (int)(t.byD == 1 ? x : t.byD ? r2 : y);
            const int b = t.b0 + (int)(t.byD == 2 ? y : r2);
            const int i0 = t.i0 + ti * TI, a0 = t.a0 + ta * TA;
            // a cell past the box reads the last one inside (only lanes of
            // faces outside the box use it)
            auto at = [&](int i, int a) -> unsigned {
                i = i < t.i1 ? i : t.i1;
                a = a < t.a1 + 3 ? a : t.a1 + 3;
                return (unsigned)(8 * (D == 1 ? IX(g, i, a, b) : IX(g, i, b, a)));
            };
            const int tx = tid & (TI - 1), ty = tid / TI;
            act = i0 + tx <= t.i1 && a0 + ty <= t.a1;
            oc = at(i0 + tx, a0 + ty < t.a1 ? a0 + ty : t.a1);
            f0 = tid;
            oe[0] = at(i0 + tx, a0 - 4 + ty);
            oe[1] = at(i0 + tx, a0 + 4 + (ty < TA - 1 ? ty : TA - 2));
            put[0] = true;
            put[1] = tid + 256 < NE;
        }
        // limiter entry of a staged cell
        auto lim = [&](int e) { return e >= LO && e - LO < NL; };

        // wq: volume-weighted half-state primitives, wl: limiter primitives,
        // bq: half-state cell B (weighted below), bl: limiter cell B
        const double *pv = met + M_VOL * N3;
        double v[2], wq[2][5], wl[2][5], bq[2][3], bl[2][3], wt = 0.0;
        if (DIR) {
            if (DIR == 2) __builtin_assume(!m.doMHD);
            wt = ab2_weight(clk);
#pragma unroll
            for (int q = 0; q < 2; q++) {
                v[q] = ldp(pv, oe[q]);
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    wl[q][n] = ldp(pln(S, (S_W + n) * N3), oe[q]);
                    wq[q][n] = ldp(pln(O, (S_W + n) * N3), oe[q]);
                }
            }
            if (DIR == 1) {
#pragma unroll
                for (int q = 0; q < 2; q++)
#pragma unroll
                    for (int x = 0; x < 3; x++) {
                        bl[q][x] = ldp(pln(S, (S_B + x) * N3), oe[q]);
                        bq[q][x] = ldp(pln(O, (S_B + x) * N3), oe[q]);
                    }
            }
#pragma unroll
            for (int q = 0; q < 2; q++) {
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    const double h = half_prim(m, n, wl[q][n], wq[q][n], wt);
                    if (!m.doLFM) wl[q][n] = h;
                    wq[q][n] = v[q] * h;
                }
                if (DIR == 2 && m.doLFM && wl[q][DEN] <= m.dFloor) {
                    // only a hydrodynamic update leaves densities below the
                    // floor, where the limiter's velocity and pressure
                    // (c2p_block) are not S_W's (c2p_cell)
                    double U[5];
#pragma unroll
                    for (int n = 0; n < 5; n++) U[n] = ldp(S + (S_GAS + n) * N3, oe[q]);
                    c2p_block(m, U, wl[q]);
                }
                if (DIR == 2) continue;
#pragma unroll
                for (int x = 0; x < 3; x++) {
                    const double h = ab2(bl[q][x], bq[q][x], wt);
                    if (!m.doLFM) bl[q][x] = h;
                    bq[q][x] = h;
                }
            }
        } else {
            const double *Wv = H + H_WH * N3, *Wl = H + H_WN * N3;
            const double *Bh = H + H_B * N3, *Bl = m.doLFM ? S + S_B * N3 : Bh;
#pragma unroll
            for (int q = 0; q < 2; q++) {
                v[q] = ldp(pv, oe[q]);
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    wq[q][n] = ldp(pln(Wv, n * N3), oe[q]);
                    wl[q][n] = ldp(pln(Wl, n * N3), oe[q]);
                }
            }
            if (m.doMHD) {
#pragma unroll
                for (int q = 0; q < 2; q++)
#pragma unroll
                    for (int x = 0; x < 3; x++) {
                        bq[q][x] = ldp(pln(Bh, x * N3), oe[q]);
                        bl[q][x] = ldp(pln(Bl, x * N3), oe[q]);
                    }
            }
        }
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int e = tid + 256 * q;
            if (put[q]) {
                sv[e] = v[q];
#pragma unroll
                for (int n = 0; n < 5; n++) sq(n)[e] = wq[q][n];
                if (lim(e))
#pragma unroll
                    for (int n = 0; n < 5; n++) sl(n)[e - LO] = wl[q][n];
            }
        }
        __syncthreads();
        const double Vi = wsum8([&](int n) { return sv[f0 + n * SN]; });
        const double rVi = gam_rcp(Vi);
        auto recon = [&](int n, double &l, double &r, double *vel) {
            double qv[8], nq[4];
#pragma unroll
            for (int x = 0; x < 8; x++) qv[x] = sq(n)[f0 + x * SN];
#pragma unroll
            for (int x = 0; x < 4; x++) nq[x] = sl(n)[f0 + (D == 0 ? x + 2 : x * SN)];
            recon_lr_w<RM>(m.pdmb, rVi, nq, qv, l, r);
            if (vel) *vel = mom2face(qv, Vi, rVi);
            // hold the two results here: their use lies inside the branch on
            // act, and the compiler would move this arithmetic there and carry
            // the twelve stencil values of every variable across the barriers
            asm volatile("" : "+v"(l), "+v"(r));
        };
        double WL[5], WR[5], BL[3] = {0.0, 0.0, 0.0}, BR[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int n = 0; n < 5; n++) {
            double vel;
            recon(n, WL[n], WR[n], DIR != 2 && n >= 1 && n <= 3 ? &vel : nullptr);
            // Mom2Face of this face from the same velocity stencil
            if (DIR != 2 && n >= 1 && n <= 3 && act) stp(Vf + (n - 1) * N3, oc, vel);
        }
        if (DIR == 1 || (DIR == 0 && m.doMHD)) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int e = tid + 256 * q;
                if (put[q]) {
#pragma unroll
                    for (int x = 0; x < 3; x++) sq(x)[e] = v[q] * bq[q][x];
                    if (lim(e))
#pragma unroll
                        for (int x = 0; x < 3; x++) sl(x)[e - LO] = bl[q][x];
                }
            }
            __syncthreads();
#pragma unroll
            for (int x = 0; x < 3; x++) recon(x, BL[x], BR[x], nullptr);
        }
        if (act)
            face_flux_lr<D, BG, BORIS>(
                g, m, met, bg, [&](const double *p) { return ldp(pln(p, 0), oc); },
                [&]() {
                    return DIR ? ab2(ldp(pln(S, (S_MF + D) * N3), oc), ldp(pln(O, (S_MF + D) * N3), oc), wt)
                               : ldp(pln(H, (H_MF + D) * N3), oc);
                },
                [&](double *dU) {
                    if (DIR) {
                        double W[5], U[5], Ul[5];
                        for (int n = 0; n < 5; n++)
                            W[n] = half_prim(m, n, ldp(S + (S_W + n) * N3, oc), ldp(O + (S_W + n) * N3, oc), wt);
                        p2c_cell(m, W, U);
                        for (int n = 0; n < 5; n++)
                            W[n] = half_prim(m, n, ldp(S + (S_W + n) * N3, oc - s8),
                                             ldp(O + (S_W + n) * N3, oc - s8), wt);
                        p2c_cell(m, W, Ul);
                        for (int n = 0; n < 5; n++) dU[n] = U[n] - Ul[n];
                    } else {
                        for (int n = 0; n < 5; n++)
                            dU[n] = ldp(H + (H_GAS + n) * N3, oc) - ldp(H + (H_GAS + n) * N3, oc - s8);
                    }
                },
                [](double *, double *) {}, WL, WR, BL, BR, oc, gflx, mflx);
    }
};

// one direction, from the predictor's planes
template <int D, int RM, bool BG, bool BORIS>
struct k_flux_t {
    static constexpr int NT = 256;
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m, FluxTile t,
                                               const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ gflx,
                                               double *__restrict__ mflx,
                                               double *__restrict__ Vf) const
    {
        __shared__ double lds[FLUX_LDS];
        flux_tile<D, RM, BG, BORIS, 0>{}(lds, (int)bi.x, g, m, t, H, S, nullptr, nullptr, met, bg, gflx, mflx, Vf);
    }
};

// The tiles of one direction's faces (box b); alt: their numbering (byD;
// 1: PLAN_LDS_D, for D = 0 the other row order)
static inline FluxTile flux_tiles(int D, const Box &b, int alt)
{
    FluxTile t;
    t.t = tile_of(b, D == 0 && alt ? 2 : 1);
    t.q7 = fast_div((unsigned)t.t.ni + 7);
    t.byD = alt;
    t.q1 = t.q2 = t.q7;
    t.i0 = b.i0;
    t.i1 = b.i1;
    t.a0 = t.a1 = t.b0 = 0;
    if (D != 0) {
        if (D == 1) { t.a0 = b.j0; t.a1 = b.j1; t.b0 = b.k0; }
        else { t.a0 = b.k0; t.a1 = b.k1; t.b0 = b.j0; }
        const int nti = (t.i1 - t.i0 + 32) / 32, nta = (t.a1 - t.a0 + 8) / 8;
        t.t.nb = nti * nta * (D == 1 ? b.k1 - b.k0 + 1 : b.j1 - b.j0 + 1);
        t.t.xs = xcd_shift(t.t.nb);
        t.q1 = fast_div((unsigned)(alt ? nta : nti));
        if (alt == 2) t.q1 = fast_div((unsigned)nti);
        t.q2 = fast_div((unsigned)(alt == 2 ? (D == 1 ? b.k1 - b.k0 + 1 : b.j1 - b.j0 + 1) : alt ? nti : nta));
    }
    return t;
}

template <int D, int RM, bool BG, bool BO>
static void flux_t(hipStream_t s, int form, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                   const double *met, const double *bg, double *gf, double *mf, double *vf)
{
    const double *H = h.H, *S = h.S;
    if (flux_lds(D, form)) {
        const FluxTile t = flux_tiles(D, b, flux_alt(D, form));
        launch_f<k_flux_t<D, RM, BG, BO>>(tgrid(t.t), dim3(BX, BY), s, g, m, t, H, S, met, bg, gf, mf, vf);
        return;
    }
    const int ch = plan_chunk(form);
    const Tile t = tile_of(b, plan_ax(form), ch);
    if (ch == 512)
        launch_f<k_flux<D, RM, BG, BO, 512>>(tgrid(t), dim3(BX, 8), s, g, m, t, H, S, met, bg, gf, mf, vf);
    else if (ch == 128)
        launch_f<k_flux<D, RM, BG, BO, 128>>(tgrid(t), dim3(BX, 2), s, g, m, t, H, S, met, bg, gf, mf, vf);
    else if (D != 0)
        launch_f<k_flux<D, RM, BG, BO, D == 0 ? 128 : BX * BY>>(tgrid(t), dim3(BX, BY), s, g, m, t, H, S, met, bg, gf,
                                                                mf, vf);
}

template <int D>
static void flux_d(hipStream_t s, int form, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                   const double *met, const double *bg, double *gf, double *mf, double *vf)
{
    const int sel = (m.rmeth ? 4 : 0) + (m.doBG ? 2 : 0) + (m.doBoris ? 1 : 0);
    switch (sel) {
    case 0: flux_t<D, 0, false, false>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 1: flux_t<D, 0, false, true>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 2: flux_t<D, 0, true, false>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 3: flux_t<D, 0, true, true>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 4: flux_t<D, 1, false, false>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 5: flux_t<D, 1, false, true>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 6: flux_t<D, 1, true, false>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    default: flux_t<D, 1, true, true>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    }
}
