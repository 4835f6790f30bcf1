// gam_flux3.hip -- the interface fluxes of all three directions and the
// Mom2Face rim in one launch.
#include "gam_flux.h"
#include "gam_rim.h"
#include <algorithm>

// The workgroups of the three directions in turn, slab by slab along k, and
// of the rim at the end (starts are multiples of 8, so each keeps its
// chunk-to-XCD mapping).  The directions read the same cells: in slabs the
// second and third find them in the memory-side cache (256 MB; a slab of
// the 256x256x384 shell is ~200 MB of cells and faces): flux 5.30 -> 5.15 ms,
// 192x192x256 1.97 -> 1.86, 96x96x128 0.263 -> 0.247; slabs of 16 5.24, of 32
// 5.35 ms.  One launch instead of four (or of three graph branches joined by events, whose
// waits cost more than the overlap gave).  Step with this and k_emf3: 16^3
// box 0.079 -> 0.037 ms, 64^3 box 0.225 -> 0.195, 48x48x64 shell 0.171 ->
// 0.142, 96x96x128 0.869 -> 0.850, 256x256x384 15.87 -> 15.88.
struct Flux3 {
    FluxTile t[3];
    RimSet rim;
    int n[3];         // workgroups of each direction in a slab
    FastDiv slab;     // by the workgroups of a slab
    int rim0;         // first workgroup of the rim
};

template <int RM, bool BG, bool BORIS, int DIR>
struct k_flux3 {
    static constexpr int NT = 256;
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, MParm m, const Flux3 &f,
                                               const double *__restrict__ H,
                                               const double *__restrict__ S,
                                               const double *__restrict__ O, const Clock *clk,
                                               const double *__restrict__ met,
                                               const double *__restrict__ bg,
                                               double *__restrict__ gflx,
                                               double *__restrict__ mflx,
                                               double *__restrict__ Vf) const
    {
        __shared__ double lds[FLUX_LDS];
        const int w = (int)bi.x;
        const long N3 = g.N3;
        if (w >= f.rim0) {
            vface_rim<DIR != 0>{}(w - f.rim0, g, f.rim, H, S, O, clk, met, Vf);
            return;
        }
        const int sl = (int)((unsigned)w / f.slab);
        int r = w - sl * (int)f.slab.d;
        if (r < f.n[0]) {
            flux_tile<0, RM, BG, BORIS, DIR>{}(lds, sl * f.n[0] + r, g, m, f.t[0], H, S, O, clk, met, bg, gflx, mflx, Vf);
        } else if (r < f.n[0] + f.n[1]) {
            r -= f.n[0];
            flux_tile<1, RM, BG, BORIS, DIR>{}(lds, sl * f.n[1] + r, g, m, f.t[1], H, S, O, clk, met, bg, gflx, mflx, Vf + 3 * N3);
        } else {
            r -= f.n[0] + f.n[1];
            flux_tile<2, RM, BG, BORIS, DIR>{}(lds, sl * f.n[2] + r, g, m, f.t[2], H, S, O, clk, met, bg, gflx, mflx, Vf + 6 * N3);
        }
    }
};

template <int RM, bool BG, bool BO>
static void flux3_t(hipStream_t s, const int *form, const Geo &g, const MParm &m, const Box *b, const HalfSrc &h,
                    const double *met, const double *bg, double *gf, double *mf, double *vf)
{
    Flux3 f;
    int tot = 0;
    // slabs of the 8 faces along k of a k tile, where a direction's faces and
    // cells (38 words a point) outgrow half the memory-side cache; no fewer than
    // two runs of every XCD per slab (whole runs are padded to the slab's end)
    const Tile t0 = tile_of(b[0], 1);
    const int ns = t0.nb < 2048 ? 1 : std::min((b[0].k1 - b[0].k0 + 8) / 8, t0.nb / (16 << t0.xs));
    for (int d = 0; d < 3; d++) {
        f.t[d] = flux_tiles(d, b[d], d == 2 && ns > 1 ? 2 : flux_alt(d, form[d]));
        const int run = 8 << f.t[d].t.xs;
        f.n[d] = (f.t[d].t.nb + ns * run - 1) / (ns * run) * run;
        tot += f.n[d];
    }
    f.slab = fast_div((unsigned)tot);
    tot *= ns;
    f.rim0 = tot;
    f.rim = rim_set(g);
    if (m.doMHD) tot += f.rim.start[6];
    const dim3 gr((unsigned)tot), bl(BX, BY);
    if (!h.O) launch_f<k_flux3<RM, BG, BO, 0>>(gr, bl, s, g, m, f, h.H, h.S, h.O, h.clk, met, bg, gf, mf, vf);
    else if (BG || BO || m.doMHD)
        launch_f<k_flux3<RM, BG, BO, 1>>(gr, bl, s, g, m, f, h.H, h.S, h.O, h.clk, met, bg, gf, mf, vf);
    else
        launch_f<k_flux3<RM, BG, BO, BG || BO ? 1 : 2>>(gr, bl, s, g, m, f, h.H, h.S, h.O, h.clk, met, bg, gf, mf, vf);
}

bool flux3_ok(const int *form)
{
    for (int d = 0; d < 3; d++)
        if (!flux_lds(d, form[d])) return false;
    return true;
}

void launch_flux3(hipStream_t s, const int *form, const Geo &g, const MParm &m, const Box *b, const HalfSrc &h,
                  const double *met, const double *bg, double *gf, double *mf, double *vf)
{
    const int sel = (m.rmeth ? 4 : 0) + (m.doBG ? 2 : 0) + (m.doBoris ? 1 : 0);
    switch (sel) {
    case 0: flux3_t<0, false, false>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 1: flux3_t<0, false, true>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 2: flux3_t<0, true, false>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 3: flux3_t<0, true, true>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 4: flux3_t<1, false, false>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 5: flux3_t<1, false, true>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    case 6: flux3_t<1, true, false>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    default: flux3_t<1, true, true>(s, form, g, m, b, h, met, bg, gf, mf, vf); break;
    }
}

void launch_vface_rim(hipStream_t s, const Geo &g, const HalfSrc &h, const double *met, double *Vf)
{
    const RimSet r = rim_set(g);
    launch_f<k_vface_rim>(dim3((unsigned)r.start[6]), dim3(BX, BY), s, g, r, h.H, met, Vf);
}
