// Host check of the tiled flux_div's launch: blocks of nx ny nz ng, one per
// line of the input; for each prints whether the kernel's 32-bit offsets fit
// the block and whether every stored cell's offset within a variable does.
#include <algorithm>
#include <climits>
#include <cstdio>
#include "../../spade_amd/csrc/flux_tile.hpp"

static spd::DevGeom block(const int nc[3], int ng)
{
    spd::DevGeom G{};
    G.ng = ng;
    for (int a = 0; a < 3; ++a) { G.nc[a] = nc[a]; G.N[a] = nc[a] + 2*ng; G.nb[a] = 1; }
    G.nblk = 1;
    G.sv = (long long)G.N[0]*G.N[1]*G.N[2];
    G.xh = (long long)G.N[1]*G.N[2]*G.nc[0];
    G.sb = ((5*G.sv + 31)/32)*32;
    G.identity = 1;
    return G;
}

int main()
{
    int nc[3], ng;
    while (std::scanf("%d %d %d %d", &nc[0], &nc[1], &nc[2], &ng) == 4)
    {
        const spd::DevGeom G = block(nc, ng);
        long long far = 0;
        for (int c = 0; c < 16; ++c)
        {
            // corners of the core and of the x-halo sections
            const int i = (c & 1) ? ((c & 8) ? nc[0] + ng - 1 : nc[0] - 1) : ((c & 8) ? -ng : 0);
            const int j = (c & 2) ? nc[1] + ng - 1 : -ng, k = (c & 4) ? nc[2] + ng - 1 : -ng;
            far = std::max(far, spd::stored_offset(G, i, j, k));
        }
        std::printf("%d %d\n", (int)spd::tile_offsets_fit(G), (int)(far <= INT_MAX));
    }
    return 0;
}
