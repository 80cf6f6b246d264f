// Instantiations of the tiled flux_div (flux_tile.hpp): cent_keep<2> with pressure_diss_lr
#include "flux_tile.hpp"

namespace spd {

bool tile_pdiss(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f, int conv, int pdiss, bool inc,
                hipStream_t s, int cus)
{
    if (conv == CV_NONE && pdiss == 1) return tile_visc<CV_NONE, 1>(g, prims, rhs, f, inc, s, cus);
    if (conv == CV_NONE && pdiss == 2) return tile_visc<CV_NONE, 2>(g, prims, rhs, f, inc, s, cus);
    if (conv == CV_KEEP2 && pdiss == 1) return tile_visc<CV_KEEP2, 1>(g, prims, rhs, f, inc, s, cus);
    if (conv == CV_KEEP2 && pdiss == 2) return tile_visc<CV_KEEP2, 2>(g, prims, rhs, f, inc, s, cus);
    return false;
}

} // namespace spd
