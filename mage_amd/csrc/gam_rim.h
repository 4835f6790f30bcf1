// gam_rim.h -- Mom2Face past the interface-flux faces.
#pragma once
#include "gam_launch.h"

// ====================================================================
// The rest of Mom2Face.  The interface-flux kernels write the face
// velocities of their own faces; the EMF stencils (GetCornerV, 8 faces
// along dT2) also reach 4 faces past them on each side:
//   I faces at j in js-4..js-1 and je+1..je+4 (k-edges, dT2 = J),
//   J faces at k in ks-4..ks-1 and ke+1..ke+4 (i-edges, dT2 = K),
//   K faces at i in is-4..is-1 and ie+1..ie+4 (j-edges, dT2 = I).
// One launch covers the six slabs; slab q is face direction q / 2.
// ====================================================================
struct RimSet {
    Tile t[6];
    int start[7];    // first workgroup of each slab
};

template <bool DIR>
struct vface_rim {
    __device__ __forceinline__ void operator()(int w, const Geo &g, const RimSet &r,
                                               const double *__restrict__ H, const double *__restrict__ S,
                                               const double *__restrict__ O, const Clock *clk,
                                               const double *__restrict__ met,
                                               double *__restrict__ Vf) const
    {
        int q = 0;
#pragma unroll
        for (int p = 1; p < 6; p++) q += (w >= r.start[p]) ? 1 : 0;
        int i, j, k;
        if (!tile_point(r.t[q], w - r.start[q], i, j, k)) return;
        const int d = q >> 1;
        const long N3 = g.N3;
        const long c = IX(g, i, j, k);
        const long s = d == 0 ? 1L : (d == 1 ? (long)g.P : g.PP);
        const double *vol = met + (long)M_VOL * N3;
        const double *wv = H + (long)(H_WH + 1) * N3;   // V * velocity
        double v8[8];
#pragma unroll
        for (int n = 0; n < 8; n++) v8[n] = vol[c + (n - 4) * s];
        const double Vi = wsum8([&](int n) { return v8[n]; });
        const double rVi = gam_rcp(Vi), wt = DIR ? ab2_weight(clk) : 0.0;
#pragma unroll
        for (int x = 0; x < 3; x++) {
            double q8[8];
#pragma unroll
            for (int n = 0; n < 8; n++) {
                const long p = c + (n - 4) * s;
                q8[n] = DIR ? v8[n] * ab2(S[(S_W + 1 + x) * N3 + p], O[(S_W + 1 + x) * N3 + p], wt)
                            : wv[x * N3 + p];
            }
            Vf[(3 * d + x) * N3 + c] = mom2face(q8, Vi, rVi);
        }
    }
};

struct k_vface_rim {
    __device__ __forceinline__ void operator()(const uint3 bi, Geo g, RimSet r, const double *__restrict__ H,
                                               const double *__restrict__ met,
                                               double *__restrict__ Vf) const
    {
        vface_rim<false>{}((int)bi.x, g, r, H, nullptr, nullptr, nullptr, met, Vf);
    }
};

static inline RimSet rim_set(const Geo &g)
{
    const Box bx[6] = {
        {g.is, g.ie + 1, g.js - 4, g.js - 1, g.ks, g.ke},      // I faces, j rim
        {g.is, g.ie + 1, g.je + 1, g.je + 4, g.ks, g.ke},
        {g.is, g.ie, g.js, g.je + 1, g.ks - 4, g.ks - 1},      // J faces, k rim
        {g.is, g.ie, g.js, g.je + 1, g.ke + 1, g.ke + 4},
        {g.is - 4, g.is - 1, g.js, g.je, g.ks, g.ke + 1},      // K faces, i rim
        {g.ie + 1, g.ie + 4, g.js, g.je, g.ks, g.ke + 1}};
    RimSet r;
    int tot = 0;
    for (int q = 0; q < 6; q++) {
        r.t[q] = tile_of(bx[q], q < 4 ? 2 : 1);
        r.start[q] = tot;
        tot += (int)tgrid(r.t[q]).x;
    }
    r.start[6] = tot;
    return r;
}
