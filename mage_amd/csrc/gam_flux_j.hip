// gam_flux_j.hip -- interface fluxes of the j faces.
#include "gam_flux.h"

void launch_flux_j(hipStream_t s, int form, const Geo &g, const MParm &m, const Box &b, const HalfSrc &h,
                   const double *met, const double *bg, double *gf, double *mf, double *vf)
{
    flux_d<1>(s, form, g, m, b, h, met, bg, gf, mf, vf);
}
