// gam_bc.hip -- time bookkeeping, boundary conditions and cell B of the
// ghost shell.
//
// EnforceBCs (step.F90:17-55) runs the sides in the order INI, OUTI, INJ,
// OUTJ, INK, OUTK, each reading what the sides before it wrote.  Here a
// ghost value looks up where the sides' copies would have brought it from,
// last side first (bc_source), and reads that place: one that no side of the
// launch writes, so the ghost values of several axes are independent and
// take one launch (k_bc_copy).  An axis joins the ones after it only where
// those are periodic: sides that are not leave the outermost faces of the
// earlier axes alone, which then hold what the earlier side made of the
// ghost data it found before them.  So: one launch when every side is
// periodic; the i sides on their own (k_bc_i, which also computes the
// inflow and the outer zero gradient) and the j and k sides together when k
// is periodic; else i, j and k.  Inside a step the last launch also forms
// cell B of every ghost cell from the faces it has looked up (bFlux2Fld,
// gridutils.F90:281-301; no side changes an active cell's faces) and does
// the time bookkeeping.
// Bound by latency on small grids: one wait on memory instead of one per
// layer and plane.  16^3 periodic box 35 -> 8 us per step (four launches to
// one), 96x96x128 shell 92 -> 56 us (six to two); 256x256x384 shell 0.39 ->
// 0.40 ms (the look-ups of 3 million ghost points); with the ghost cells'
// primitives, which replaced the predictor's pass over them, 62 us and 0.47 ms.
#include "gam_launch.h"
#include "gam_wind.h"

// ====================================================================
// Time bookkeeping and CalcDT checks (step.F90:103-166); one thread.
// ====================================================================
__device__ __forceinline__ void finalize_clock(const MParm &m, Clock *clk, int mode)
{
    Clock c = *clk;
    if (mode & FIN_ADVANCE) {          // applyUpdate: oState%time=State%time; State%time+=dt
        c.whf = ab2_weight(clk);
        c.ost = c.st;
        c.st = c.st + c.dtA;
    }
    if (mode & FIN_MODEL) {            // UpdateStateData (gamapp.F90:108-110)
        c.ts = c.ts + 1;
        c.t = c.t + c.dt;
    }
    if (mode & FIN_CALCDT) {
        const double dtMin = __longlong_as_double((long long)c.dtBits);
        int st = 0;
        if (dtMin == GAM_HUGE) st = 2;
        double dt = dtMin;
        if (c.ts > 0) {
            if (c.dt / dtMin >= 10) st = st > 1 ? st : 1;
            if ((c.dt0 > GAM_TINY) && (dtMin / c.dt0 <= m.limDT0)) st = st > 1 ? st : 1;
            if (dtMin <= GAM_TINY) st = 2;
        }
        if ((c.t + dt) > m.tFin) dt = dmax(m.tFin - c.t, GAM_TINY);
        if (c.dt0 > GAM_TINY && dt > (10.0 * c.dt0)) dt = 10.0 * c.dt0;
        c.dtRet = dt;
        c.lastStatus = st;
        c.status = c.status > st ? c.status : st;
        if (mode & FIN_SETDT) { c.dt = dt; c.dtA = dt; }
        if (mode & FIN_INIT) c.ost = c.st - c.dt;
    }
    c.dtBits = (unsigned long long)__double_as_longlong(GAM_HUGE);
    *clk = c;
}

struct k_finalize {
    __device__ __forceinline__ void operator()(const uint3 bi, MParm m, Clock *clk, int mode) const
    {
        if (threadIdx.x == 0 && bi.x == 0) finalize_clock(m, clk, mode);
    }
};

// ====================================================================
// bFlux2Fld (gridutils.F90:281-301) over all cells
// ====================================================================
struct k_bflux2fld {
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g,
                                               Tile cb, const double *__restrict__ mf,
                                               double *__restrict__ B,
                                               const double *__restrict__ met) const
    {
        TILE_IJK(cb);
        const long N3 = g.N3, c = IX(g, i, j, k);
        double b[3];
        cell_b(g, met, c, mf[c], mf[N3 + c], mf[2 * N3 + c], mf[c + 1], mf[N3 + c + g.P],
               mf[2 * N3 + c + g.PP], b);
        for (int x = 0; x < 3; x++) B[x * N3 + c] = b[x];
    }
};

// ====================================================================
// Where the copies of a launch's sides bring a ghost value from.
// ====================================================================
struct BcSet {
    int kind[6];
    int ax;       // axes of the look-up: 1 i (both periodic only), 2 j, 4 k
    int withB;    // EnforceBCs on its own: cell B as the sides copy it
};
enum { BC_GAS = 0, BC_FACE = 1, BC_B = 4 };   // BC_FACE + d: face flux of direction d

// One axis: index t of quantity q along axis A (ghosts below s and above e).
// in2: the two other indices lie in the range of cells, which bounds the
// sides that are not periodic.
template <int A>
__device__ __forceinline__ void bc_axis(int klo, int khi, int s, int e, bool in2, int &q, int &t)
{
    const bool nf = q == BC_FACE + A;           // faces normal to A: e + 1 is active
    const int n = e - s + 1;
    if (t < s) {
        if (klo == 0) t += n;                                       // periodic (bcs.F90:279-450)
        else if (in2 && (q != BC_B || klo == 2)) t = s;             // zero gradient (799-930), sphere in
    } else if (t > e + (nf ? 1 : 0) && (nf || t <= e + 4)) {
        if (khi == 0) t -= n;
        else if (in2 && (q != BC_B || khi == 3)) {
            if (nf && A == 2) { q = BC_FACE + 1; t = e; }           // takes the J flux (bcs.F90:925)
            else t = nf ? e + 1 : e;
        }
    }
}

__device__ __forceinline__ long bc_source(const Geo &g, const BcSet &b, int &q, int i, int j, int k)
{
    if (b.ax & 4) bc_axis<2>(b.kind[4], b.kind[5], g.ks, g.ke, i <= g.ieg && j <= g.jeg, q, k);
    if (b.ax & 2) bc_axis<1>(b.kind[2], b.kind[3], g.js, g.je, i <= g.ieg && k <= g.keg, q, j);
    if (b.ax & 1) bc_axis<0>(b.kind[0], b.kind[1], g.is, g.ie, j <= g.jeg && k <= g.keg, q, i);
    return IX(g, i, j, k);
}

// The ghost shell (cells and the faces past them): up to six boxes (the k,
// j and i slabs, disjoint), each cut into tiles of BX*BY threads that cover
// iw[q] points along i by BX*BY/iw[q] along j: 64 x 4 in the wide boxes, 4 x
// 64 or 8 x 32 in the i slabs (one point of a ghost row per lane).
struct GhostBoxes {
    Box b[6];
    int start[7];     // first tile of each box; start[6] = total
    int n0[6], n1[6], iw[6];
};

template <bool FIELD>
struct k_bc_copy {
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m, const BcSet &bc,
                                               const GhostBoxes &gb, Clock *clk, int finmode, int writeW,
                                               double *__restrict__ S, const double *__restrict__ met) const
    {
        const int w = (int)bi.x, tid = (int)(threadIdx.x + BX * threadIdx.y);
        if (finmode && w == 0 && tid == 0) finalize_clock(m, clk, finmode);
        int bq = 0;
#pragma unroll
        for (int p = 1; p < 6; p++) bq += (w >= gb.start[p]) ? 1 : 0;
        const int L = w - gb.start[bq];
        const Box &b = gb.b[bq];
        const int t0 = L % gb.n0[bq];
        const int r = L / gb.n0[bq];
        const int iw = gb.iw[bq];
        const int i = b.i0 + t0 * iw + tid % iw;
        const int j = b.j0 + (r % gb.n1[bq]) * (BX * BY / iw) + tid / iw;
        const int k = b.k0 + r / gb.n1[bq];
        if (i > b.i1 || j > b.j1 || k > b.k1) return;
        const long N3 = g.N3, c = IX(g, i, j, k);
        const bool cell = i <= g.ieg && j <= g.jeg && k <= g.keg;
        // every load before the first store: one wait
        int q = BC_GAS, qf[3];
        const long sg = cell ? bc_source(g, bc, q, i, j, k) : c;
        long sf[3];
        double U[5], f[3], B[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int d = 0; d < 3; d++) {
            qf[d] = BC_FACE + d;
            sf[d] = bc_source(g, bc, qf[d], i, j, k);
            f[d] = S[(S_MF + qf[d] - BC_FACE) * N3 + sf[d]];
        }
#pragma unroll
        for (int v = 0; v < 5; v++) U[v] = S[(S_GAS + v) * N3 + sg];
        long sb = c;
        if (FIELD) {
            if (cell) {
                int qI = BC_FACE, qJ = BC_FACE + 1, qK = BC_FACE + 2;
                const long sI = bc_source(g, bc, qI, i + 1, j, k), sJ = bc_source(g, bc, qJ, i, j + 1, k),
                           sK = bc_source(g, bc, qK, i, j, k + 1);
                cell_b(g, met, c, f[0], f[1], f[2], S[(S_MF + qI - BC_FACE) * N3 + sI],
                       S[(S_MF + qJ - BC_FACE) * N3 + sJ], S[(S_MF + qK - BC_FACE) * N3 + sK], B);
            }
        } else if (cell && bc.withB) {
            q = BC_B;
            sb = bc_source(g, bc, q, i, j, k);
#pragma unroll
            for (int x = 0; x < 3; x++) B[x] = S[(S_B + x) * N3 + sb];
        }
        if (sg != c) {
#pragma unroll
            for (int v = 0; v < 5; v++) S[(S_GAS + v) * N3 + c] = U[v];
        }
        if (FIELD && writeW && cell) {
            double W[5];
            c2p_cell(m, U, W);
#pragma unroll
            for (int v = 0; v < 5; v++) S[(S_W + v) * N3 + c] = W[v];
        }
#pragma unroll
        for (int d = 0; d < 3; d++)
            if (sf[d] != c || qf[d] != BC_FACE + d) S[(S_MF + d) * N3 + c] = f[d];
        if (FIELD ? cell : sb != c) {
#pragma unroll
            for (int x = 0; x < 3; x++) S[(S_B + x) * N3 + c] = B[x];
        }
    }
};

// ====================================================================
// The i sides.  The ghost slabs are 4 cells wide along the fastest index:
// one ghost layer per lane, the four layers of a (j, k) point in adjacent
// lanes (a 64-lane block covers 16 points along j), so that one load reads
// 32 contiguous bytes along i.
// ====================================================================
__device__ __forceinline__ bool is_cell(const Geo &g, int i, int j, int k)
{
    return i >= g.isg && i <= g.ieg && j >= g.jsg && j <= g.jeg && k >= g.ksg && k <= g.keg;
}

// Ghost layer n of INI and the copying kinds of OUTI (periodic, sphere out):
// gas, face fluxes and (withB, periodic and sphere only) cell B from cell
// s; the normal faces of OUTI lie one further out.
template <bool OUT>
__device__ __forceinline__ void bc_i_copy(const Geo &g, int kind, int withB, int n, int j, int k,
                                          double *__restrict__ S)
{
    if (kind != 0 && (j > g.jeg || k > g.keg)) return;
    const long N3 = g.N3;
    const int ig = OUT ? g.ie + n : g.is - n;
    const int is = kind == 0 ? (OUT ? g.is + n - 1 : g.ie - n + 1) : (OUT ? g.ie : g.is);
    const long d = IX(g, ig, j, k), s = IX(g, is, j, k);
    const long df = OUT ? d + 1 : d, sf = OUT && kind == 0 ? s + 1 : s;   // normal face
    const bool cell = is_cell(g, ig, j, k), cb = cell && withB && kind != 1;
    double U[5], f[3], B[3];
#pragma unroll
    for (int v = 0; v < 5; v++) U[v] = S[(S_GAS + v) * N3 + s];
    f[0] = S[S_MF * N3 + sf];
    f[1] = S[(S_MF + 1) * N3 + s];
    f[2] = S[(S_MF + 2) * N3 + s];
    if (cb)
#pragma unroll
        for (int x = 0; x < 3; x++) B[x] = S[(S_B + x) * N3 + s];
    if (cell)
#pragma unroll
        for (int v = 0; v < 5; v++) S[(S_GAS + v) * N3 + d] = U[v];
    S[S_MF * N3 + df] = f[0];
    S[(S_MF + 1) * N3 + d] = f[1];
    S[(S_MF + 2) * N3 + d] = f[2];
    if (cb)
#pragma unroll
        for (int x = 0; x < 3; x++) S[(S_B + x) * N3 + d] = B[x];
}

// Outer zero gradient: ghost faces take the last physical cell's B
__device__ __forceinline__ void bc_i_zerograd(const Geo &g, int n, int j, int k, double *__restrict__ S,
                                              const double *__restrict__ met)
{
    if (j > g.jeg || k > g.keg) return;
    const long N3 = g.N3;
    double *mf = S + S_MF * N3;
    const long s = IX(g, g.ie, j, k), d = IX(g, g.ie + n, j, k);
    double B[3], U[5];
    cell_b(g, met, s, mf[s], mf[N3 + s], mf[2 * N3 + s], mf[s + 1], mf[N3 + s + g.P], mf[2 * N3 + s + g.PP], B);
#pragma unroll
    for (int v = 0; v < 5; v++) U[v] = S[(S_GAS + v) * N3 + s];
    const long fi[3] = {d + 1, d, d};
    double f[3];
#pragma unroll
    for (int x = 0; x < 3; x++) {
        const double *nrm = met + (long)(M_TF + 9 * x) * N3 + fi[x];
        f[x] = met[(M_FACE + x) * N3 + fi[x]] * (B[0] * nrm[0] + B[1] * nrm[N3] + B[2] * nrm[2 * N3]);
    }
#pragma unroll
    for (int v = 0; v < 5; v++) S[(S_GAS + v) * N3 + d] = U[v];
#pragma unroll
    for (int x = 0; x < 3; x++) mf[x * N3 + fi[x]] = f[x];
}

// WindBC part 1 (wind.F90:226-335): ghost gas and blended face fluxes.
// Ghost layer n of the transverse point (j, k); tm = Model%t.
__device__ __forceinline__ void bc_i_wind(const Geo &g, const MParm &m, const WindDev &w, double tm, int n,
                                          int j, int k, double *__restrict__ S,
                                          const double *__restrict__ met)
{
    const long N3 = g.N3;
    double *mf = S + S_MF * N3;
    double vF[3];
    wind_front(w, tm, vF);
    const int ip = g.ie;
    {
        const int ig = g.ie + n;
        if (k <= g.keg && j <= g.jeg) {
            const long cg = IX(g, ig, j, k), cp = IX(g, ip, j, k);
            const double xc[3] = {met[(M_XYZCC + 0) * N3 + cg], met[(M_XYZCC + 1) * N3 + cg], met[(M_XYZCC + 2) * N3 + cg]};
            double r, p, V[3], B[3];
            wind_at(w, vF, xc, tm, &r, &p, V, B);
            const double wSW = wind_wgt_v(xc, V), wMHD = 1.0 - wSW;
            double gs[5] = {0, 0, 0, 0, 0}, gi[5] = {0, 0, 0, 0, 0};
            if (wSW > GAM_TINY) {
                gs[0] = r; gs[1] = V[0]; gs[2] = V[1]; gs[3] = V[2]; gs[4] = p;
            }
            if (wMHD > GAM_TINY) {
                double U[5], Bi[3];
                for (int v = 0; v < 5; v++) U[v] = S[(S_GAS + v) * N3 + cp];
                for (int x = 0; x < 3; x++) Bi[x] = S[(S_B + x) * N3 + cp];
                const long fp = IX(g, ip + 1, j, k);
                const double nH[3] = {met[(M_TF + 0) * N3 + fp], met[(M_TF + 1) * N3 + fp], met[(M_TF + 2) * N3 + fp]};
                wind_inner(m, U, Bi, nH, gi);
            }
            double gw[5], U[5];
            for (int v = 0; v < 5; v++) gw[v] = wSW * gs[v] + wMHD * gi[v];
            p2c_cell(m, gw, U);
            for (int v = 0; v < 5; v++) S[(S_GAS + v) * N3 + cg] = U[v];
        }
        const int fi[3] = {ig + 1, ig, ig};
        const int ii[3] = {ip + 1, ip, ip};
        for (int d = 0; d < 3; d++) {
            const long f = IX(g, fi[d], j, k);
            const double xf[3] = {met[(M_XFC + 0 + 3 * d) * N3 + f], met[(M_XFC + 1 + 3 * d) * N3 + f], met[(M_XFC + 2 + 3 * d) * N3 + f]};
            double r, p, V[3], B[3];
            wind_at(w, vF, xf, tm, &r, &p, V, B);
            const double wSW = wind_wgt_v(xf, V);
            const double *nrm = met + (long)(M_TF + 9 * d) * N3 + f;
            const double sw = met[(M_FACE + d) * N3 + f] * (nrm[0] * B[0] + nrm[N3] * B[1] + nrm[2 * N3] * B[2]);
            const double in = mf[d * N3 + IX(g, ii[d], j, k)];
            mf[d * N3 + f] = wSW * sw + (1 - wSW) * in;
        }
    }
}

// Both i sides, INI in the blocks with z = 0, OUTI in those with z = 1 (each
// reads active cells of its own side and writes its own ghosts).  With pend
// the clock has not taken this step's time yet (k_bc_copy does it after).
template <bool WIND>
struct k_bc_i {
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m, const BcSet &bc, const Clock *clk,
                                               int pend, const WindDev &w, double *__restrict__ S,
                                               const double *__restrict__ met) const
    {
        const int j = g.jsg + (int)(bi.x * 16 + (threadIdx.x >> 2)), k = g.ksg + (int)bi.y;
        const int n = 1 + (int)(threadIdx.x & 3);
        if (j > g.jeg + 1) return;
        if (bi.z == 0) bc_i_copy<false>(g, bc.kind[0], bc.withB, n, j, k, S);
        else if (WIND) bc_i_wind(g, m, w, pend ? clk->t + clk->dt : clk->t, n, j, k, S, met);
        else if (bc.kind[1] == 1) bc_i_zerograd(g, n, j, k, S, met);
        else bc_i_copy<true>(g, bc.kind[1], bc.withB, n, j, k, S);
    }
};

// WindBC part 2 (wind.F90:338-348): ghost Bxyz from the blended fluxes with
// the periodic k mapping of lfmIJKcc (ringutils.F90:482-518).
struct k_bc_wind_b {
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, Box t,
                                               double *__restrict__ S,
                                               const double *__restrict__ met) const
    {
        const int j = t.i0 + (int)(bi.x * 16 + (threadIdx.x >> 2));
        const int k = t.j0 + bi.y;
        if (j > t.i1 || k > t.j1) return;
        const long N3 = g.N3;
        const double *mf = S + S_MF * N3;
        int kp = k;
        if (k < g.ks) kp = k + g.Nkp;
        else if (k > g.ke) kp = k - g.Nkp;
        {
            const int n = 1 + (int)(threadIdx.x & 3);
            const int ig = g.ie + n;
            const long s = IX(g, ig, j, kp);
            double B[3];
            cell_b(g, met, s, mf[s], mf[N3 + s], mf[2 * N3 + s], mf[s + 1], mf[N3 + s + g.P], mf[2 * N3 + s + g.PP], B);
            const long d = IX(g, ig, j, k);
            for (int x = 0; x < 3; x++) S[(S_B + x) * N3 + d] = B[x];
        }
    }
};

void launch_finalize(hipStream_t s, const MParm &m, Clock *clk, int mode)
{
    launch_f<k_finalize>(dim3(1), dim3(64), s, m, clk, mode);
}

void launch_bflux2fld(hipStream_t s, const Geo &g, const Box &cb, const double *mf,
                      double *B, const double *met)
{
    const Tile t = tile_of(cb, 1);
    launch_f<k_bflux2fld>(tgrid(t), dim3(BX, BY), s, g, t, mf, B, met);
}

// EnforceBCs on S.  field = false: the sides alone, with cell B as they copy
// it (gam_enforce_bcs).  field = true: inside a step; cell B of every ghost
// cell from its faces instead (bFlux2Fld), and with finmode the time
// bookkeeping, whose Model%t the inflow then reads ahead of it.
void launch_bcs(hipStream_t s, const int *kind, bool field, bool writeW, int finmode, const Geo &g, const MParm &m, Clock *clk,
                const WindDev &w, double *S, const double *met)
{
    BcSet bc;
    for (int q = 0; q < 6; q++) bc.kind[q] = kind[q];
    bc.withB = !field;
    bool per[3];
    for (int a = 0; a < 3; a++) per[a] = kind[2 * a] == 0 && kind[2 * a + 1] == 0;
    const bool all = per[0] && per[1] && per[2];
    if (!all) {
        const dim3 gr((unsigned)((g.Nj + 1 + 15) / 16), (unsigned)(g.Nk + 1), 2);
        const int pend = finmode & FIN_MODEL;
        if (kind[1] == 4) launch_f<k_bc_i<true>>(gr, dim3(64), s, g, m, bc, clk, pend, w, S, met);
        else launch_f<k_bc_i<false>>(gr, dim3(64), s, g, m, bc, clk, pend, w, S, met);
        if (kind[1] == 4 && !field) {
            // ghost-cell B of the inflow side (wind.F90:338-348)
            const Box t = {g.jsg, g.jeg, g.ksg, g.keg, 0, 0};
            launch_f<k_bc_wind_b>(dim3((unsigned)((g.Nj + 15) / 16), (unsigned)g.Nk), dim3(64), s, g, t, S, met);
        }
    }
    const int I0 = g.isg, I1 = g.ieg + 1, J0 = g.jsg, J1 = g.jeg + 1, K0 = g.ksg, K1 = g.keg + 1;
    auto copy = [&](int ax, bool last) {
        const bool f = last && field;
        bc.ax = ax;
        // the ghost shell without overlap, or the j slabs over every k
        const bool jonly = ax == 2;
        const Box bx[6] = {
            {I0, I1, J0, J1, K0, g.ks - 1},                                       // k ghosts, all i, j
            {I0, I1, J0, J1, g.ke + 1, K1},
            {I0, I1, J0, g.js - 1, jonly ? K0 : g.ks, jonly ? K1 : g.ke},         // j ghosts
            {I0, I1, g.je + 1, J1, jonly ? K0 : g.ks, jonly ? K1 : g.ke},
            {I0, g.is - 1, g.js, g.je, g.ks, g.ke},                               // i ghosts, active j, k
            {g.ie + 1, I1, g.js, g.je, g.ks, g.ke}};
        const bool use[3] = {(ax & 4) != 0, (ax & 2) || f, (ax & 1) || f};        // k, j, i slabs
        GhostBoxes gb;
        int tot = 0;
        for (int q = 0; q < 6; q++) {
            gb.b[q] = bx[q];
            gb.start[q] = tot;
            gb.iw[q] = q == 4 ? 4 : q == 5 ? 8 : BX;
            const int jw = BX * BY / gb.iw[q];
            gb.n0[q] = (bx[q].i1 - bx[q].i0 + gb.iw[q]) / gb.iw[q];
            gb.n1[q] = (bx[q].j1 - bx[q].j0 + jw) / jw;
            if (use[q / 2]) tot += gb.n0[q] * gb.n1[q] * (bx[q].k1 - bx[q].k0 + 1);
        }
        gb.start[6] = tot;
        const int fm = last ? finmode : 0;
        if (f) launch_f<k_bc_copy<true>>(dim3((unsigned)tot), dim3(BX, BY), s, g, m, bc, gb, clk, fm, writeW ? 1 : 0, S, met);
        else launch_f<k_bc_copy<false>>(dim3((unsigned)tot), dim3(BX, BY), s, g, m, bc, gb, clk, fm, writeW ? 1 : 0, S, met);
    };
    if (all) copy(7, true);
    else if (per[2]) copy(6, true);
    else {
        copy(2, false);
        copy(4, true);
    }
}
