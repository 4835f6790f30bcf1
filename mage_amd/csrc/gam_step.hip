// gam_step.hip -- gfx950 kernels of one GAMERA MHD step (FP64).
//
// Kernel sequence of one stepGamera (gamapp.F90:73-113):
//   k_predict    Predictor: AB2 face fluxes, half-step B and gas, plus the
//                primitives used by the flux sweeps.  Only where the fluxes
//                and EMFs cannot form the half state themselves (HalfSrc):
//                in the first two steps of a state that was put, in the
//                adjoint, with launch plans of direct loads and in contexts
//                without the primitives' planes (hydrodynamic ones with the
//                Boris or background option, full devices).  It moves 50
//                words per point, the step
//                without it 8 more; 256x256x384 shell 14.46 -> 12.80 ms per
//                step, 96x96x128 0.784 -> 0.691, 16^3 box 0.035 -> 0.032.
//   k_flux3      Lyon gas/magnetic fluxes of the three directions, the face
//                velocities (Mom2Face) of the same faces and of those the EMF
//                stencils read past them (gam_flux3.hip, gam_flux.h)
//   k_emf3       edge EMFs of the three directions (gam_emf.hip)
//                (k_flux_t or k_flux, k_vface_rim, k_emf_t or k_emf: the same
//                one direction at a time, after k_predict)
//   k_update     CT face-flux update, cell B of the new state, flux
//                divergence, Reynolds, Maxwell/Boris and the CFL
//                min-reduction of the new state
//   k_bc_i, k_bc_copy  boundary conditions, cell B of the ghost cells (the
//                active cells keep theirs: no BC writes a face of one),
//                time bookkeeping and CalcDT checks (gam_bc.hip)
// State and oState are two buffers that swap roles every step, which
// replaces CopyState (mhdgroup.F90:204-255): the update reads the current
// buffer and writes every point of the other.
#include "gam_launch.h"

static thread_local std::vector<EnsLaunch> *g_rec = nullptr;
void set_launch_recorder(std::vector<EnsLaunch> *r) { g_rec = r; }
std::vector<EnsLaunch> *launch_recorder() { return g_rec; }

static void order_mark(hipStream_t s, int mark, int ev)
{
    EnsLaunch e;
    e.launch = nullptr;
    e.grid = e.block = dim3(0, 0, 0);
    e.stream = s;
    e.mark = mark;
    e.ev = ev;
    g_rec->push_back(std::move(e));
}

void order_record(hipStream_t s, hipEvent_t e, int ev)
{
    if (g_rec) order_mark(s, 1, ev);
    else hipEventRecord(e, s);
}

void order_wait(hipStream_t s, hipEvent_t e, int ev)
{
    if (g_rec) order_mark(s, 2, ev);
    else hipStreamWaitEvent(s, e, 0);
}


// ====================================================================
// Predictor (mhdgroup.F90:444-561) fused with bFlux2Fld of the half state
// (gridutils.F90:281-301) and the primitive conversions of the flux
// stencils (BlockCon2Prim, recon.F90:75-90) for both the half state and
// the limiter state n.
// Domain: all face points isg..ieg+1 (x) jsg..jeg+1 (x) ksg..keg+1.
// ====================================================================
template <int NTH = BX * BY>
struct k_predict {
    static constexpr int NT = NTH;
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m,
                                               Tile fb, const Clock *clk,
                                               const double *__restrict__ S,
                                               const double *__restrict__ O,
                                               const double *__restrict__ met,
                                               double *__restrict__ H, int hfonly) const
    {
        TILE_IJK(fb);
        const long N3 = g.N3;
        const long c = IX(g, i, j, k);
        const unsigned oc = (unsigned)(c * 8);    // byte offset of the point
        // hfonly: the half state alone (H_GAS, H_MF, H_B) of the last step
        const double w = hfonly ? clk->whf : ab2_weight(clk);

        double f[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            f[d] = m.doMHD ? ab2(ldp(S + (S_MF + d) * N3, oc), ldp(O + (S_MF + d) * N3, oc), w)
                           : ldp(H + (H_MF + d) * N3, oc);
            stp(H + (H_MF + d) * N3, oc, f[d]);
        }
        if (i > g.ieg || j > g.jeg || k > g.keg) return;

        // half-state cell B from the six extrapolated face fluxes
        double fIp, fJp, fKp;
        const unsigned oI = oc + 8, oJ = oc + 8 * g.P, oK = oc + (unsigned)(8 * g.PP);
        if (m.doMHD) {
            fIp = ab2(ldp(S + (S_MF + 0) * N3, oI), ldp(O + (S_MF + 0) * N3, oI), w);
            fJp = ab2(ldp(S + (S_MF + 1) * N3, oJ), ldp(O + (S_MF + 1) * N3, oJ), w);
            fKp = ab2(ldp(S + (S_MF + 2) * N3, oK), ldp(O + (S_MF + 2) * N3, oK), w);
        } else {
            fIp = ldp(H + (H_MF + 0) * N3, oI);
            fJp = ldp(H + (H_MF + 1) * N3, oJ);
            fKp = ldp(H + (H_MF + 2) * N3, oK);
        }
        double B[3];
        cell_b(g, met, c, f[0], f[1], f[2], fIp, fJp, fKp, B);
#pragma unroll
        for (int x = 0; x < 3; x++) stp(H + (H_B + x) * N3, oc, B[x]);

        // PredictCell (mhdgroup.F90:528-561)
        double Q[5], oQ[5], W[5], oW[5], pW[5], pQ[5], Wb[5];
#pragma unroll
        for (int v = 0; v < 5; v++) { Q[v] = ldp(S + (S_GAS + v) * N3, oc); oQ[v] = ldp(O + (S_GAS + v) * N3, oc); }
        c2p_cell(m, oQ, oW);
        c2p_cell(m, Q, W);
#pragma unroll
        for (int v = 0; v < 5; v++) pW[v] = ab2(W[v], oW[v], w);
        pW[DEN] = dmax(pW[DEN], m.dFloor);
        pW[PRS] = dmax(pW[PRS], m.pFloor);
        p2c_cell(m, pW, pQ);
#pragma unroll
        for (int v = 0; v < 5; v++) stp(H + (H_GAS + v) * N3, oc, pQ[v]);
        if (hfonly) return;
        // primitives of the reconstruction stencils (half state), stored
        // multiplied by the cell volume: every use is the volume-weighted
        // interpolation <V q>/<V> (recon.F90:125-198, fields.F90:262-270), and
        // the product is the one those formulas would form.  The limiter
        // stencils take plain primitives: of state n (doLFMLim), else of the
        // half state.
        c2p_block(m, pQ, Wb);
        const double vol = ldp(met + M_VOL * N3, oc);
#pragma unroll
        for (int v = 0; v < 5; v++) stp(H + (H_WH + v) * N3, oc, vol * Wb[v]);
        if (m.doLFM) c2p_block(m, Q, Wb);
#pragma unroll
        for (int v = 0; v < 5; v++) stp(H + (H_WN + v) * N3, oc, Wb[v]);
    }
};

// ====================================================================
// CT update (E2Flux, fields.F90:18-51) + bFlux2Fld of the new state.
// Domain: all face points.  Faces outside is..ie+1 x js..je+1 x ks..ke+1
// keep their old flux; edges outside the active EMF boxes read as zero,
// as CalcElecField zeroes E before filling active edges (fields.F90:89).
// ====================================================================
__device__ __forceinline__ double e_at(const Geo &g, const EdgeBoxes &eb, const double *E, int d,
                                       int i, int j, int k, unsigned off)
{
    return in_box(eb.e[d], i, j, k) ? ldp(E + d * g.N3, off) : 0.0;
}

// New flux of face d at (i,j,k), whose byte offset is oc.
__device__ __forceinline__ double ct_face(const Geo &g, const EdgeBoxes &eb, const Box &ctb,
                                          const double *E, const double *mfOld, double dt,
                                          int d, int i, int j, int k, unsigned oc)
{
    const double old = ldp(mfOld + d * g.N3, oc);
    if (!in_box(ctb, i, j, k)) return old;
    const unsigned oI = oc + 8, oJ = oc + 8 * g.P, oK = oc + (unsigned)(8 * g.PP);
    double df;
    if (d == 0)
        df = e_at(g, eb, E, 2, i, j + 1, k, oJ) - e_at(g, eb, E, 2, i, j, k, oc)
           - e_at(g, eb, E, 1, i, j, k + 1, oK) + e_at(g, eb, E, 1, i, j, k, oc);
    else if (d == 1)
        df = e_at(g, eb, E, 0, i, j, k + 1, oK) - e_at(g, eb, E, 0, i, j, k, oc)
           - e_at(g, eb, E, 2, i + 1, j, k, oI) + e_at(g, eb, E, 2, i, j, k, oc);
    else
        df = e_at(g, eb, E, 1, i + 1, j, k, oI) - e_at(g, eb, E, 1, i, j, k, oc)
           - e_at(g, eb, E, 0, i, j + 1, k, oJ) + e_at(g, eb, E, 0, i, j, k, oc);
    return old - dt * df;
}

// ====================================================================
// Block min-reduction of positive doubles into clk->dtBits.
// ====================================================================
__device__ __forceinline__ void block_min_dt(double v, Clock *clk)
{
    __shared__ double red[512 / 64];   // up to 8 waves
    for (int off = 32; off > 0; off >>= 1) v = dmin(v, __shfl_xor(v, off, 64));
    const int tid = threadIdx.x + threadIdx.y * blockDim.x;
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    if (tid == 0) {
        double r = red[0];
        for (int w = 1; w < (int)(blockDim.x * blockDim.y) / 64; w++) r = dmin(r, red[w]);
        if (r > 0.0 && r < GAM_HUGE) atomicMin(&clk->dtBits, (unsigned long long)__double_as_longlong(r));
    }
}

// ====================================================================
// applyUpdate (mhdgroup.F90:79-258) in one pass over all face points:
//  * CT: E2Flux (fields.F90:18-51) on the point's three faces; faces
//    outside is..ie+1 x js..je+1 x ks..ke+1 keep the old flux, edges
//    outside the active EMF boxes read as zero (E is zeroed before the
//    active edges are filled, fields.F90:89);
//  * bFlux2Fld of the new state (the three upper faces are re-derived);
//  * Flux2Deltas (stress.F90:152-194), Reynolds with Model%dt (114-125)
//    and Maxwell/Boris (171-195, 299-441) on active cells; ghost cells copy
//    the old state (CopyState);
//  * CellDT of the new state on the CalcDT domain, min-reduced
//    (step.F90:91-101).
// Every thread reaches the block reduction.
// ====================================================================
template <bool BG, bool BORIS, int NTH = BX * BY>
struct k_update {
    static constexpr int NT = NTH;
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m,
                                               Tile ft, Box ctb, EdgeBoxes eb, Box ab, Box dtb,
                                               Clock *clk, const double *__restrict__ So,
                                               double *__restrict__ Sn, int writeW,
                                               const double *__restrict__ gflx,
                                               const double *__restrict__ mflx,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg) const
    {
        int i, j, k;
        const bool live = tile_point(ft, (int)bi.x, i, j, k);
        double dtc = GAM_HUGE;
        const long N3 = g.N3;
        const long c = IX(g, i, j, k);
        const unsigned oc = (unsigned)(c * 8);    // byte offset of the point
        const bool cell = live && i <= g.ieg && j <= g.jeg && k <= g.keg;
        double Bn[3] = {0.0, 0.0, 0.0};
        if (live) {
            const double dt = clk->dtA;
            const double *E = Sn + S_E * N3;
            const double *mfo = So + S_MF * N3;
            double f[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                f[d] = m.doMHD ? ct_face(g, eb, ctb, E, mfo, dt, d, i, j, k, oc) : ldp(mfo + d * N3, oc);
                stp(Sn + (S_MF + d) * N3, oc, f[d]);
            }
            if (cell) {
                double fIp, fJp, fKp;
                if (m.doMHD) {
                    fIp = ct_face(g, eb, ctb, E, mfo, dt, 0, i + 1, j, k, oc + 8);
                    fJp = ct_face(g, eb, ctb, E, mfo, dt, 1, i, j + 1, k, oc + 8 * g.P);
                    fKp = ct_face(g, eb, ctb, E, mfo, dt, 2, i, j, k + 1, oc + (unsigned)(8 * g.PP));
                } else {
                    fIp = mfo[0 * N3 + c + 1]; fJp = mfo[1 * N3 + c + g.P]; fKp = mfo[2 * N3 + c + g.PP];
                }
                cell_b(g, met, c, f[0], f[1], f[2], fIp, fJp, fKp, Bn);
#pragma unroll
                for (int x = 0; x < 3; x++) stp(Sn + (S_B + x) * N3, oc, Bn[x]);
            }
        }
        if (cell) {
            double U[5];
#pragma unroll
            for (int v = 0; v < 5; v++) U[v] = ldp(So + (S_GAS + v) * N3, oc);
            if (in_box(ab, i, j, k)) {
                const double idV = 1.0 / ldp(met + M_VOL * N3, oc);
                const unsigned oI = oc + 8, oJ = oc + 8 * g.P, oK = oc + (unsigned)(8 * g.PP);
                const double dtM = clk->dt, dt = clk->dtA;
                double dH[5], oU[5];
#pragma unroll
                for (int v = 0; v < 5; v++) {
                    const double *gv = gflx + (long)v * N3;
                    dH[v] = (ldp(gv, oc) - ldp(gv, oI) + ldp(gv + 5 * N3, oc) - ldp(gv + 5 * N3, oJ)
                             + ldp(gv + 10 * N3, oc) - ldp(gv + 10 * N3, oK)) * idV;
                    oU[v] = U[v];
                    U[v] = U[v] + dtM * dH[v];
                }
                if (m.doMHD) {
                    double dM[3], B[3], oB[3];
#pragma unroll
                    for (int x = 0; x < 3; x++) {
                        const double *mv = mflx + (long)x * N3;
                        double r = (ldp(mv, oc) - ldp(mv, oI) + ldp(mv + 3 * N3, oc) - ldp(mv + 3 * N3, oJ)
                                    + ldp(mv + 6 * N3, oc) - ldp(mv + 6 * N3, oK)) * idV;
                        if (BG) r = r + ldp(bg + (B_DPB0 + x) * N3, oc);
                        dM[x] = r;
                        B[x] = Bn[x];
                        oB[x] = ldp(So + (S_B + x) * N3, oc);
                        if (BG) {
                            const double b0 = ldp(bg + (B_B0 + x) * N3, oc);
                            B[x] = B[x] + b0;
                            oB[x] = oB[x] + b0;
                        }
                    }
                    if (BORIS) {
                        // CellBoris (mhdgroup.F90:336-441), single fluid
                        double W2[5];
                        c2p_cell(m, U, W2);
                        const double D2 = dmax(W2[DEN], m.dFloor);
                        const double P2 = dmax(W2[PRS], m.pFloor);
                        const double D0 = dmax(oU[DEN], m.dFloor);
                        const double iD0 = 1.0 / D0, iD2 = 1.0 / D2;
                        double V0[3] = {oU[MOMX] * iD0, oU[MOMY] * iD0, oU[MOMZ] * iD0};
                        double B1[3] = {0.5 * (B[0] + oB[0]), 0.5 * (B[1] + oB[1]), 0.5 * (B[2] + oB[2])};
                        const double alpha = (B1[0] * B1[0] + B1[1] * B1[1] + B1[2] * B1[2]) * (iD2 * m.iCa2);
                        const double dRho = dt * dH[DEN];
                        double dPG[3] = {dt * dH[MOMX], dt * dH[MOMY], dt * dH[MOMZ]};
                        double dPM[3] = {dt * dM[0], dt * dM[1], dt * dM[2]};
                        const double pCon = 1.0 / (1.0 + alpha);
                        double dMom[3];
                        if (alpha > GAM_TINY) {
                            const double nb = sqrt(B1[0] * B1[0] + B1[1] * B1[1] + B1[2] * B1[2]);
                            double bh[3];
                            if (nb <= GAM_TINY) { bh[0] = bh[1] = bh[2] = 0.0; }
                            else { const double inb = 1.0 / nb; bh[0] = B1[0] * inb; bh[1] = B1[1] * inb; bh[2] = B1[2] * inb; }
                            double sGM[3] = {dPG[0] + dPM[0], dPG[1] + dPM[1], dPG[2] + dPM[2]};
                            const double pG = dPG[0] * bh[0] + dPG[1] * bh[1] + dPG[2] * bh[2];
                            const double pS = sGM[0] * bh[0] + sGM[1] * bh[1] + sGM[2] * bh[2];
                            const double pV = V0[0] * bh[0] + V0[1] * bh[1] + V0[2] * bh[2];
#pragma unroll
                            for (int x = 0; x < 3; x++)
                                dMom[x] = pG * bh[x] + pCon * (sGM[x] - pS * bh[x]) + alpha * pCon * dRho * (V0[x] - pV * bh[x]);
                        } else {
#pragma unroll
                            for (int x = 0; x < 3; x++) dMom[x] = dPG[x] + dPM[x];
                        }
                        double Wn[5];
                        Wn[DEN] = D2;
#pragma unroll
                        for (int x = 0; x < 3; x++) Wn[1 + x] = (D0 * V0[x] + dMom[x]) * iD2;
                        Wn[PRS] = P2;
                        p2c_cell(m, Wn, U);
                    } else {
                        // CellMaxwell (mhdgroup.F90:299-329)
                        const double d = dmax(U[DEN], m.dFloor);
                        double mx = U[MOMX], my = U[MOMY], mz = U[MOMZ];
                        const double id = 1.0 / d;
                        double ke = 0.5 * (mx * mx + my * my + mz * mz) * id;
                        const double p = dmax((m.gamma - 1) * (U[ENER] - ke), m.pFloor);
                        mx = mx + dt * dM[0];
                        my = my + dt * dM[1];
                        mz = mz + dt * dM[2];
                        ke = 0.5 * (mx * mx + my * my + mz * mz) * id;
                        U[DEN] = d; U[MOMX] = mx; U[MOMY] = my; U[MOMZ] = mz;
                        U[ENER] = ke + p * m.igm1;
                    }
                }
            }
#pragma unroll
            for (int v = 0; v < 5; v++) stp(Sn + (S_GAS + v) * N3, oc, U[v]);
            // primitives of the active cells (the boundary launch adds the ghosts')
            if (writeW && in_box(ab, i, j, k)) {
                double W[5];
                c2p_cell(m, U, W);
#pragma unroll
                for (int v = 0; v < 5; v++) stp(Sn + (S_W + v) * N3, oc, W[v]);
            }
            if (in_box(dtb, i, j, k)) {
                double bx = Bn[0], by = Bn[1], bz = Bn[2];
                if (BG) {
                    bx = bx + ldp(bg + (B_B0 + 0) * N3, oc);
                    by = by + ldp(bg + (B_B0 + 1) * N3, oc);
                    bz = bz + ldp(bg + (B_B0 + 2) * N3, oc);
                }
                const double dl = ldp(met + M_DL * N3, oc);
                dtc = cell_dt<BORIS>(m, U, bx, by, bz, dl);
                if (!(dtc == dtc)) dtc = GAM_HUGE;
            }
        }
        block_min_dt(dtc, clk);
    }
};

// CalcDT over the DT box on a state (standalone CalcDT, step.F90:58-101)
template <bool BG, bool BORIS>
struct k_calc_dt {
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m,
                                               Tile dtb, Clock *clk, const double *__restrict__ S,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg) const
    {
        int i, j, k;
        const bool live = tile_point(dtb, (int)bi.x, i, j, k);
        double dtc = GAM_HUGE;
        if (live) {
            const long N3 = g.N3, c = IX(g, i, j, k);
            double U[5];
            for (int v = 0; v < 5; v++) U[v] = S[(S_GAS + v) * N3 + c];
            double bx = S[(S_B + 0) * N3 + c], by = S[(S_B + 1) * N3 + c], bz = S[(S_B + 2) * N3 + c];
            if (BG) { bx = bx + bg[(B_B0 + 0) * N3 + c]; by = by + bg[(B_B0 + 1) * N3 + c]; bz = bz + bg[(B_B0 + 2) * N3 + c]; }
            const double dl = met[M_DL * N3 + c];
            dtc = cell_dt<BORIS>(m, U, bx, by, bz, dl);
            if (!(dtc == dtc)) dtc = GAM_HUGE;
        }
        block_min_dt(dtc, clk);
    }
};

// DivB partial sums (gridutils.F90:717-770)
__global__ void k_divb(Geo g, Box ab, const double *__restrict__ mf, const double *__restrict__ bg,
                       int useBG, double *__restrict__ part)
{
    const int i = ab.i0 + blockIdx.x * BX + threadIdx.x;
    const int j = ab.j0 + blockIdx.y * BY + threadIdx.y;
    const int k = ab.k0 + blockIdx.z;
    double v = 0.0;
    if (i <= ab.i1 && j <= ab.j1) {
        const long N3 = g.N3, c = IX(g, i, j, k);
        double dFi = mf[c] - mf[c + 1], dFj = mf[N3 + c] - mf[N3 + c + g.P], dFk = mf[2 * N3 + c] - mf[2 * N3 + c + g.PP];
        double a0 = 0.0, a1 = 0.0, a2 = 0.0;
        if (useBG) {
            const double *b0 = bg + B_BFLUX0 * N3;
            a0 = b0[c] - b0[c + 1]; a1 = b0[N3 + c] - b0[N3 + c + g.P]; a2 = b0[2 * N3 + c] - b0[2 * N3 + c + g.PP];
        }
        v = fabs(dFi + dFj + dFk + a0 + a1 + a2);
    }
    __shared__ double red[BX * BY];
    const int tid = threadIdx.x + threadIdx.y * BX;
    red[tid] = v;
    __syncthreads();
    for (int s = BX * BY / 2; s > 0; s >>= 1) {
        if (tid < s) red[tid] += red[tid + s];
        __syncthreads();
    }
    if (tid == 0) part[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = red[0];
}

// Layout conversion between Fortran arrays and the padded device index
// space: planes of an (ni,nj,nk) Fortran array starting at isg, one plane per
// block y.  (Per plane and with a staging copy each, a 16^3 state took 38
// launches, 30 copies and 25 waits to put and get.)
template <bool IN>
__global__ __launch_bounds__(256) void k_repack(Geo g, int ni, int nj, int nk, FastDiv qi, FastDiv qj,
                                                const double *__restrict__ src, double *__restrict__ dst)
{
    const long tot = (long)ni * nj * nk;
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q >= tot) return;
    const unsigned r = (unsigned)q / qi, kk = r / qj;
    const int ii = (int)((unsigned)q - r * (unsigned)ni), jj = (int)(r - kk * (unsigned)nj);
    const long c = IX(g, g.isg + ii, g.jsg + jj, g.ksg + (int)kk);
    if (IN) dst[blockIdx.y * g.N3 + c] = src[blockIdx.y * tot + q];
    else dst[blockIdx.y * tot + q] = src[blockIdx.y * g.N3 + c];
}

__global__ void k_clock_state(Clock *clk, int st, double time)
{
    if (st) clk->st = time;
    else clk->ost = time;
}
__global__ void k_clock_time(Clock *clk, double t, double dt, int ts)
{
    clk->t = t;
    clk->dt = dt;
    clk->dtA = dt;
    clk->ts = ts;
}
__global__ void k_clock_dta(Clock *clk, double dt) { clk->dtA = dt; }
__global__ void k_clock_dt0(Clock *clk, double dt0) { clk->dt0 = dt0; }

// Zero the E entries outside the active EMF boxes (CalcElecField zeroes E
// before filling the active edges, fields.F90:89).
__global__ void k_mask_e(Geo g, Box all, EdgeBoxes eb, double *__restrict__ E)
{
    THREAD_IJK(all);
    const long c = IX(g, i, j, k);
    for (int d = 0; d < 3; d++)
        if (!in_box(eb.e[d], i, j, k)) E[d * g.N3 + c] = 0.0;
}

// ====================================================================
// Host-side launchers
// ====================================================================
#define LAUNCH(kern, grid, block, stream, ...) hipLaunchKernelGGL(kern, grid, block, 0, stream, __VA_ARGS__)

Plan default_plan()
{
    Plan p;
    // pointwise but for the next row and plane: row order 1 takes the
    // 256x256x384 step from 16.28 to 16.09 ms for either (slabs: 3)
    p.v[TS_PREDICT] = 1;
    p.v[TS_EMF_I] = 1;
    p.v[TS_EMF_J] = 1;
    p.v[TS_EMF_K] = 1;
    p.v[TS_FLUX_I] = 1;
    p.v[TS_FLUX_J] = PLAN_LDS;
    p.v[TS_FLUX_K] = PLAN_LDS;
    p.v[TS_UPDATE] = 1;
    return p;
}

int plan_candidates(int slot, int *vals)
{
    int n = 0;
    if (slot < 0 || slot >= TS_COUNT) return 0;
    const int maxax = (slot == TS_FLUX_I) ? 2 : 3;
    // row order x chunk size (256, 512, 128 points per workgroup)
    for (int c = 0; c < 3; c++)
        for (int a = 1; a <= maxax; a++) vals[n++] = a + 8 * c;
    if (slot == TS_FLUX_J || slot == TS_FLUX_K) {
        vals[n++] = PLAN_LDS;
        vals[n++] = PLAN_LDS_D;
        vals[n++] = PLAN_LDS + PLAN_ALIAS;
        vals[n++] = PLAN_LDS_D + PLAN_ALIAS;
    }
    return n;
}

void launch_predict(hipStream_t s, int plan, const Geo &g, const MParm &m, const Box &fb, const Clock *clk,
                    const double *S, const double *O, const double *met, double *H, int hfonly)
{
    const int ch = plan_chunk(plan);
    const Tile t = tile_of(fb, plan_ax(plan), ch);
    if (ch == 512) launch_f<k_predict<512>>(tgrid(t), dim3(BX, 8), s, g, m, t, clk, S, O, met, H, hfonly);
    else if (ch == 128) launch_f<k_predict<128>>(tgrid(t), dim3(BX, 2), s, g, m, t, clk, S, O, met, H, hfonly);
    else launch_f<k_predict<>>(tgrid(t), dim3(BX, BY), s, g, m, t, clk, S, O, met, H, hfonly);
}

void launch_flux(hipStream_t s, int d, int form, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                 const double *met, const double *bg, double *gf, double *mf, double *vf)
{
    (d == 0 ? launch_flux_i : d == 1 ? launch_flux_j : launch_flux_k)(s, form, g, m, b, h, met, bg, gf, mf, vf);
}

template <bool BG, bool BO>
static void update_t(hipStream_t s, int plan, const Geo &g, const MParm &m, const Box &fb, const Box &ctb,
                     const EdgeBoxes &eb, const Box &ab, const Box &dtb, Clock *clk, const double *So,
                     double *Sn, int writeW, const double *gf, const double *mf, const double *met,
                     const double *bg)
{
    const int ch = plan_chunk(plan);
    const Tile t = tile_of(fb, plan_ax(plan), ch);
    if (ch == 512)
        launch_f<k_update<BG, BO, 512>>(tgrid(t), dim3(BX, 8), s, g, m, t, ctb, eb, ab, dtb, clk, So, Sn, writeW, gf, mf,
                                        met, bg);
    else if (ch == 128)
        launch_f<k_update<BG, BO, 128>>(tgrid(t), dim3(BX, 2), s, g, m, t, ctb, eb, ab, dtb, clk, So, Sn, writeW, gf, mf,
                                        met, bg);
    else
        launch_f<k_update<BG, BO>>(tgrid(t), dim3(BX, BY), s, g, m, t, ctb, eb, ab, dtb, clk, So, Sn, writeW, gf, mf,
                                   met, bg);
}

void launch_update(hipStream_t s, int plan, const Geo &g, const MParm &m, const Box &fb, const Box &ctb,
                   const Box *eboxes, const Box &ab, const Box &dtb, Clock *clk, const double *So,
                   double *Sn, bool writeW, const double *gf, const double *mf, const double *met, const double *bg)
{
    EdgeBoxes eb;
    for (int d = 0; d < 3; d++) eb.e[d] = eboxes[d];
    const int sel = (m.doBG ? 2 : 0) + (m.doBoris ? 1 : 0);
    switch (sel) {
    case 0: update_t<false, false>(s, plan, g, m, fb, ctb, eb, ab, dtb, clk, So, Sn, writeW, gf, mf, met, bg); break;
    case 1: update_t<false, true>(s, plan, g, m, fb, ctb, eb, ab, dtb, clk, So, Sn, writeW, gf, mf, met, bg); break;
    case 2: update_t<true, false>(s, plan, g, m, fb, ctb, eb, ab, dtb, clk, So, Sn, writeW, gf, mf, met, bg); break;
    default: update_t<true, true>(s, plan, g, m, fb, ctb, eb, ab, dtb, clk, So, Sn, writeW, gf, mf, met, bg); break;
    }
}

void launch_calc_dt(hipStream_t s, const Geo &g, const MParm &m, const Box &dtb, Clock *clk,
                    const double *S, const double *met, const double *bg)
{
    const int sel = (m.doBG ? 2 : 0) + (m.doBoris ? 1 : 0);
    const Tile t = tile_of(dtb, 1);
    switch (sel) {
    case 0: launch_f<k_calc_dt<false, false>>(tgrid(t), dim3(BX, BY), s, g, m, t, clk, S, met, bg); break;
    case 1: launch_f<k_calc_dt<false, true>>(tgrid(t), dim3(BX, BY), s, g, m, t, clk, S, met, bg); break;
    case 2: launch_f<k_calc_dt<true, false>>(tgrid(t), dim3(BX, BY), s, g, m, t, clk, S, met, bg); break;
    default: launch_f<k_calc_dt<true, true>>(tgrid(t), dim3(BX, BY), s, g, m, t, clk, S, met, bg); break;
    }
}

void launch_divb(hipStream_t s, const Geo &g, const Box &ab, const double *mf, const double *bg,
                 int useBG, double *part, int *nparts)
{
    dim3 gr = grid_of(ab);
    *nparts = (int)(gr.x * gr.y * gr.z);
    LAUNCH(k_divb, gr, dim3(BX, BY), s, g, ab, mf, bg, useBG, part);
}

void launch_repack(hipStream_t s, int dir_in, const Geo &g, int ni, int nj, int nk, int ncomp,
                   const double *src, double *dst)
{
    const long tot = (long)ni * nj * nk;   // a plane: below 2^31 points, as everywhere
    const dim3 gr((unsigned)((tot + 255) / 256), (unsigned)ncomp);
    const FastDiv qi = fast_div((unsigned)ni), qj = fast_div((unsigned)nj);
    if (dir_in) LAUNCH(k_repack<true>, gr, dim3(256), s, g, ni, nj, nk, qi, qj, src, dst);
    else LAUNCH(k_repack<false>, gr, dim3(256), s, g, ni, nj, nk, qi, qj, src, dst);
}

void launch_clock_state(hipStream_t s, Clock *clk, bool st, double time)
{
    LAUNCH(k_clock_state, dim3(1), dim3(1), s, clk, st ? 1 : 0, time);
}
void launch_clock_time(hipStream_t s, Clock *clk, double t, double dt, int ts)
{
    LAUNCH(k_clock_time, dim3(1), dim3(1), s, clk, t, dt, ts);
}
void launch_clock_dta(hipStream_t s, Clock *clk, double dt)
{
    LAUNCH(k_clock_dta, dim3(1), dim3(1), s, clk, dt);
}
void launch_clock_dt0(hipStream_t s, Clock *clk, double dt0)
{
    LAUNCH(k_clock_dt0, dim3(1), dim3(1), s, clk, dt0);
}

void launch_mask_e(hipStream_t s, const Geo &g, const Box &all, const Box *eboxes, double *E)
{
    EdgeBoxes eb;
    for (int d = 0; d < 3; d++) eb.e[d] = eboxes[d];
    LAUNCH(k_mask_e, grid_of(all), dim3(BX, BY), s, g, all, eb, E);
}
