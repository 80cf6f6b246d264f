// Instantiations of the tiled flux_div (flux_tile.hpp): weno_t, fweno_t, weno_fds_t
#include "flux_tile.hpp"

namespace spd {

bool tile_weno(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f, int conv, int pdiss, bool inc,
               hipStream_t s, int cus)
{
    if (conv == CV_WENO && pdiss == 0) return tile_visc<CV_WENO, 0>(g, prims, rhs, f, inc, s, cus);
    if (conv == CV_FWENO && pdiss == 0) return tile_visc<CV_FWENO, 0>(g, prims, rhs, f, inc, s, cus);
    if (conv == CV_FDS && pdiss == 0) return tile_visc<CV_FDS, 0>(g, prims, rhs, f, inc, s, cus);
    return false;
}

} // namespace spd
