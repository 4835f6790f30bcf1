// gam_kernels.h -- host-side launchers of the gfx950 kernels.
#pragma once
#include "gam_common.h"
#include <string.h>
#include <vector>

// Argument record of one kernel launch: the arguments in order, as a
// nested aggregate (a0, then the record of the rest).  The host writes it
// to device memory for batched launches; layout is the same on both sides.
template <class... A>
struct Pack {};
template <class A0, class... A>
struct Pack<A0, A...> {
    A0 a0;
    Pack<A...> r;
};
__host__ __device__ inline Pack<> make_pack() { return Pack<>{}; }
template <class A0, class... A>
__host__ __device__ inline Pack<A0, A...> make_pack(A0 a0, A... a)
{
    return Pack<A0, A...>{a0, make_pack(a...)};
}

// Batched launch over the members of an ensemble: member m owns workgroups
// wg0[m] .. wg0[m+1]-1 (wg0[m] a multiple of 8) of which the first
// gx*gy*gz run its own grid.  In device memory the header is followed by
// an unsigned short per run of 8 workgroups: the member that owns it.
#define ENS_MAX 256
struct EnsHdr {
    unsigned n;
    unsigned wg0[ENS_MAX + 1];
    unsigned gx[ENS_MAX], gy[ENS_MAX], gz[ENS_MAX];
};

// One recorded launch of a step kernel: the function that issues the
// batched form for this kernel and argument types, the member's own grid
// and block, and the argument record bytes.
struct EnsLaunch {
    void (*launch)(hipStream_t s, const void *hdr, const void *rec, unsigned nwg, dim3 block);
    dim3 grid, block;
    std::vector<unsigned char> rec;
    hipStream_t stream;   // the stream the launch or marker was issued to
    int mark;             // 0 launch; 1 event ev recorded on stream; 2 stream waits for event ev
    int ev;
};
// While r is set, the step kernels that this thread would launch are
// appended to *r instead (nothing is issued); nullptr restores launching.
void set_launch_recorder(std::vector<EnsLaunch> *r);
std::vector<EnsLaunch> *launch_recorder();   // r, or nullptr
// Stream order of a branching step: hipEventRecord(e, s) and
// hipStreamWaitEvent(s, e) at once, or, while a recorder is set, appended
// to it as markers naming the event by its index ev.
void order_record(hipStream_t s, hipEvent_t e, int ev);
void order_wait(hipStream_t s, hipEvent_t e, int ev);

// Launch plan: the shape of every tunable launch of the step.  Values
// 1, 2, 3 are the Tile row orders (ax1: j fastest, k fastest, j-slabs), + 8
// or 16 for chunks of 512 or 128 points instead of 256.  The LDS-staged
// forms stand where direct loads in chunks of 256 were never faster: EMF 1,
// 2, 3 (one form), i flux 1 and 2 (its two row orders); j and k flux
// PLAN_LDS and PLAN_LDS_D (tiles numbered along i first, or along the flux
// direction first), which PLAN_ALIAS added to either also names.  So plans
// saved when these were other shapes stay valid and take the new ones.
enum { TS_PREDICT = 0, TS_EMF_I, TS_EMF_J, TS_EMF_K, TS_FLUX_I, TS_FLUX_J, TS_FLUX_K, TS_UPDATE,
       TS_COUNT };
#define PLAN_LDS 4
#define PLAN_LDS_D 5
#define PLAN_ALIAS 2
struct Plan {
    int v[TS_COUNT];
};
static inline bool emf_lds(int v) { return v <= 3; }
static inline bool flux_lds(int d, int v) { return d == 0 ? v <= 2 : (v & 7) >= PLAN_LDS; }
static inline int flux_alt(int d, int v) { return d == 0 ? v == 2 : v & 1; }   // the other numbering
// v names the same launch as a smaller value of the slot
static inline bool plan_alias(int slot, int v)
{
    if (slot >= TS_EMF_I && slot <= TS_EMF_K) return v == 2 || v == 3;
    return v >= PLAN_LDS + PLAN_ALIAS && v < 8;
}
Plan default_plan();
// candidate values of a slot; returns their number
int plan_candidates(int slot, int *vals);

// k_finalize modes
enum {
    FIN_ADVANCE = 1,   // State/oState times after applyUpdate
    FIN_MODEL = 2,     // Model%ts += 1, Model%t += Model%dt
    FIN_CALCDT = 4,    // evaluate CalcDT from the reduction
    FIN_SETDT = 8,     // Model%dt = CalcDT result
    FIN_INIT = 16      // oState%time = State%time - dt (init.F90:238-244)
};

// Sets the message gam_last_error() returns ("msg: detail") and returns code.
int gam_fail_(int code, const char *msg, const char *detail);

// Where the fluxes and EMFs take the half state from: H, the predictor's
// planes (O null); or, with O, State S and oState O themselves.  That needs
// both states as a step leaves them: the primitives of their gas in S_W and,
// with MHD, gas at or above the density floor and cell B that of the face
// fluxes in every cell (ghosts too), where extrapolating cell B and primitives
// is extrapolating face fluxes and gas; and launch plans of the LDS forms.
// (A hydrodynamic step applies no floor: its fluxes see to densities below it.)
struct HalfSrc {
    const double *H, *S, *O;
    const Clock *clk;
};

void launch_predict(hipStream_t s, int ax, const Geo &g, const MParm &m, const Box &fb, const Clock *clk,
                    const double *S, const double *O, const double *met, double *H, int hfonly = 0);
// Launches of one direction each take the half state from h.H (h.O null).
// Mom2Face on the faces the EMF stencils read past the interface-flux faces
// (the flux kernels write the rest): Vf planes [3*dT1 + comp]
void launch_vface_rim(hipStream_t s, const Geo &g, const HalfSrc &h, const double *met, double *Vf);
void launch_emf(hipStream_t s, int eD, int ax, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                const double *Vf, const double *met, const double *bg, double *E);
// Interface fluxes of direction d, and Mom2Face of the same faces into
// vf's three planes of direction d
void launch_flux(hipStream_t s, int d, int form, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                 const double *met, const double *bg, double *gf, double *mf, double *vf);
// All three directions (forms of the three slots, face boxes b[3]) and, with
// MHD, the Mom2Face rim in one launch; flux3_ok: the forms allow it
bool flux3_ok(const int *form);
void launch_flux3(hipStream_t s, const int *form, const Geo &g, const MParm &m, const Box *b, const HalfSrc &h,
                  const double *met, const double *bg, double *gf, double *mf, double *vf);
// the three edge directions (edge boxes b[3]) in one launch, if the plans of
// the three slots allow it
bool emf3_ok(const int *plan);
void launch_emf3(hipStream_t s, const Geo &g, const MParm &m, const Box *b, const HalfSrc &h, const double *Vf,
                 const double *met, const double *bg, double *E);
// one face direction each, one source file each
void launch_flux_i(hipStream_t s, int form, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                   const double *met, const double *bg, double *gf, double *mf, double *vf);
void launch_flux_j(hipStream_t s, int form, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                   const double *met, const double *bg, double *gf, double *mf, double *vf);
void launch_flux_k(hipStream_t s, int form, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                   const double *met, const double *bg, double *gf, double *mf, double *vf);
void launch_update(hipStream_t s, int ax, const Geo &g, const MParm &m, const Box &fb, const Box &ctb,
                   const Box *eboxes, const Box &ab, const Box &dtb, Clock *clk, const double *So,
                   double *Sn, bool writeW, const double *gf, const double *mf, const double *met,
                   const double *bg);
void launch_calc_dt(hipStream_t s, const Geo &g, const MParm &m, const Box &dtb, Clock *clk,
                    const double *S, const double *met, const double *bg);
// Clock fields set from the host: State%time (st) or oState%time; Model%t,
// dt, ts; AdvanceMHD's dt; Model%dt0
void launch_clock_state(hipStream_t s, Clock *clk, bool st, double time);
void launch_clock_time(hipStream_t s, Clock *clk, double t, double dt, int ts);
void launch_clock_dta(hipStream_t s, Clock *clk, double dt);
void launch_clock_dt0(hipStream_t s, Clock *clk, double dt0);
void launch_finalize(hipStream_t s, const MParm &m, Clock *clk, int mode);
void launch_bflux2fld(hipStream_t s, const Geo &g, const Box &cb, const double *mf,
                      double *B, const double *met);
// EnforceBCs of S: alone (field = false) or inside a step, with cell B of
// the ghost cells from their faces and, with finmode, launch_finalize's work
// writeW: also the primitives (S_W) of every ghost cell
void launch_bcs(hipStream_t s, const int *kind, bool field, bool writeW, int finmode, const Geo &g, const MParm &m, Clock *clk,
                const WindDev &w, double *S, const double *met);
void launch_divb(hipStream_t s, const Geo &g, const Box &ab, const double *mf, const double *bg,
                 int useBG, double *part, int *nparts);
// ncomp consecutive Fortran planes of (ni,nj,nk) to (dir_in) or from device planes
void launch_repack(hipStream_t s, int dir_in, const Geo &g, int ni, int nj, int nk, int ncomp,
                   const double *src, double *dst);
void launch_mask_e(hipStream_t s, const Geo &g, const Box &all, const Box *eboxes, double *E);

// Grid pre-compute (gam_grid.hip)
void launch_grid_from_corners(hipStream_t s, const Geo &g, double *met);
// the M_DL plane from di, dj, dk
void launch_min_length(hipStream_t s, const Geo &g, double *met);
// largest |T T^t - 1| of the active faces' triads into *err (set to 0 before)
void launch_triad_error(hipStream_t s, const Geo &g, const double *met, unsigned long long *err);
void launch_dipole_b0(hipStream_t s, const Geo &g, double M0, const double *met, double *bg,
                      double *scratch9);

// Adjoint of the hydrodynamic step (gam_adj.hip)
void launch_adj_objective(hipStream_t s, const Geo &g, const MParm &m, const double *S,
                          const double *wgt, double *aS, double *part, int *nparts);
void launch_bc_adj(hipStream_t s, int side, int kind, const Geo &g, double *aS);
// pdt (may be null): the dt-sensitivity plane (d/d(dt) shares, see
// launch_dt_fold); pw: the AB2-weight plane
void launch_update_adj(hipStream_t s, const Geo &g, const Box &ab, const Clock *clk, const double *aSn,
                       double *aSo, double *ag, const double *met, const double *gflx, double *pdt);
void launch_flux_adj(hipStream_t s, int d, const Geo &g, const MParm &m, const Box &fb, const double *H,
                     const double *met, const double *ag, double *aWH, double *aWN);
void launch_predict_adj(hipStream_t s, const Geo &g, const MParm &m, const Clock *clk, const double *S,
                        const double *O, const double *met, const double *aWH, const double *aWN,
                        double *aS, double *aO, double *pw);
void launch_set_dt(hipStream_t s, Clock *clk, const Clock *rec);
// dt = dtA = dts[n] on the device clock (replays with a given dt sequence)
void launch_set_dt_val(hipStream_t s, Clock *clk, const double *dts, int n);
// Reduce one adjoint step's dt planes (pdt, pw over the face box) into
// mu[n] (and mu[n-1] through the AB2 weight's odt); part holds 2 doubles
// per 64 x 4 block of the face box (dt_part_blocks).
long dt_part_blocks(const Geo &g);
void launch_dt_fold(hipStream_t s, const Geo &g, const double *pdt, const double *pw, double *part,
                    const Clock *clk, int n, double *mu);
// CalcDT's argmin over the DT box of S (the state the update has just
// written, before the boundary pass), recorded with its values as
// DT_REC doubles {cell, gas 5, total cell B 3, dl, valid} when its CellDT
// is the dt clk holds (valid = 0 where tFin or 10 dt0 capped it); part: 2
// doubles per 64 x 4 block of dtb (dt_record_blocks)
#define DT_REC 12
long dt_record_blocks(const Geo &g, const Box &dtb);
void launch_dt_record(hipStream_t s, const Geo &g, const MParm &m, const Box &dtb, const double *S,
                      const double *met, const double *bg, const Clock *clk, double *part, double *rec);
// CalcDT transpose: lam += mu * d(CellDT)/d(gas, cell B) at rec's cell
void launch_dt_inject(hipStream_t s, const Geo &g, const MParm &m, const double *rec, const double *mu,
                      double *lam);
void launch_cellb_adj(hipStream_t s, const Geo &g, int all, double *aS, const double *met);
// both: the two sides of its axis, which must have more than 8 cells
void launch_bc_periodic_adj(hipStream_t s, int side, const Geo &g, double *aS, bool both);
void launch_bc_mhd_adj(hipStream_t s, int side, int kind, const Geo &g, double *aS, const double *met);
// transpose of the inflow BC; adds the series adjoint into gQ (n,5), gB (n,3),
// each WIND_COPIES consecutive copies of those arrays (the caller sums them)
#define WIND_COPIES 32
void launch_bc_wind_adj(hipStream_t s, const Geo &g, const MParm &m, const Clock *clk, const WindDev &w,
                        const double *S, double *aS, const double *met, double *gQ, double *gB);
void launch_update_adj_mhd(hipStream_t s, const Geo &g, const MParm &m, const Box &ab, const Box &ctb,
                           const Box *eboxes, const Clock *clk, const double *So, const double *Sn1,
                           const double *gflx, const double *mflx, const double *met, const double *bg,
                           double *aSn, double *aSo, double *aUr, double *adM, double *ag, double *amf,
                           double *aE, double *pdt);
// pass 1 of the flux transpose: per tile of faces, the transposed
// reconstructions summed over the tile's cells into sc (FLUXADJ_NPL planes:
// weighted values and limiter values of the 8 variables, from the tile of
// the cell's own face and from the neighbouring one), aBn into aHMF, the
// Boris nuke term into aHG
#define FLUXADJ_NPL 32
void launch_flux_adj_mhd(hipStream_t s, const Geo &g, const MParm &m, const Box *fb, const double *H,
                         const double *S, const double *met, const double *bg, const double *ag,
                         const double *amf, double *sc, double *aHMF, double *aHG);
// pass 2 (all three directions' sc) fused with the Mom2Face transpose and the
// predictor's gas transpose: into aS, aO; writes aHB of every cell
void launch_recon_adj_gather(hipStream_t s, const Geo &g, const MParm &m, const Clock *clk, const double *sc,
                             const double *rv, const double *aVf, const double *met, const double *S,
                             const double *O, const double *aHG, double *aHB, double *aS, double *aO, double *pw);
// pass 1 of the edge EMF transpose: 16 planes per edge direction into sc
void launch_emf_adj(hipStream_t s, const Geo &g, const MParm &m, const Box *eb, const Clock *clk,
                    const double *H, const double *S, const double *Vf, const double *met, const double *bg,
                    const double *aE, double *sc, double *pdt);
// pass 2: writes aVf, aHMF and aHG at every point (adds the limiter parts
// to aSSMF with the LFM limiter)
void launch_emf_adj_gather(hipStream_t s, const Geo &g, const MParm &m, const Box *eboxes, const double *sc,
                           const double *met, double *aVf, double *aHMF, double *aHG, double *aSSMF);
void launch_vface_rv(hipStream_t s, const Geo &g, const double *met, double *rv);
void launch_predict_mf_adj(hipStream_t s, const Geo &g, const Clock *clk, const double *S, const double *O,
                           const double *met, double *aHB, double *aHMF, double *aS, double *aO, double *pw);
