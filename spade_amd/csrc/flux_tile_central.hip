// Instantiations of the tiled flux_div (flux_tile.hpp): cent_keep<2>, pressure_diss_lr and visc_lr
#include "flux_tile.hpp"

namespace spd {

bool tile_central(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f, int conv, int pdiss, bool inc,
                  hipStream_t s, int cus)
{
    if (conv == CV_NONE && pdiss == 0) return tile_visc<CV_NONE, 0>(g, prims, rhs, f, inc, s, cus);
    if (conv == CV_KEEP2 && pdiss == 0) return tile_visc<CV_KEEP2, 0>(g, prims, rhs, f, inc, s, cus);
    return false;
}

} // namespace spd
