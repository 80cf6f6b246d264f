// Instantiations of the tiled flux_div (flux_tile.hpp): cent_keep<4>, totani_lr, first_order_t
#include "flux_tile.hpp"

namespace spd {

bool tile_split(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f, int conv, int pdiss, bool inc,
                hipStream_t s, int cus)
{
    if (conv == CV_KEEP4 && pdiss == 0) return tile_visc<CV_KEEP4, 0>(g, prims, rhs, f, inc, s, cus);
    if (conv == CV_TOTANI && pdiss == 0) return tile_visc<CV_TOTANI, 0>(g, prims, rhs, f, inc, s, cus);
    if (conv == CV_FIRST && pdiss == 0) return tile_visc<CV_FIRST, 0>(g, prims, rhs, f, inc, s, cus);
    return false;
}

} // namespace spd
