// gam_flux_k.hip -- interface fluxes of the k faces.
#include "gam_flux.h"

void launch_flux_k(hipStream_t s, int form, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                   const double *met, const double *bg, double *gf, double *mf, double *vf)
{
    flux_d<2>(s, form, g, m, b, h, met, bg, gf, mf, vf);
}
