// Host check of the tiled flux_div's launch and of rules on block shapes.  Commands on the input, one per
// line, with a block of nx ny nz cells and ng ghost layers each:
//   offsets nx ny nz ng          whether the kernel's 32-bit offsets fit the block, and
//                                whether every stored cell's offset within a variable does
//   plan nx ny nz ng blocks H SS map   the plan: wi wj tx ty zs threads bytes of LDS, and whether an
//                                exhaustive search of the same costs finds the same one
//   time nx ny nz ng             microseconds of one plan
//   pushes nx ny nz ng blocks    whether a Butcher-table stage writes the ghosts it feeds
#include <algorithm>
#include <chrono>
#include <climits>
#include <cstdio>
#include <cstring>
#include "../../spade_amd/csrc/flux_tile.hpp"

using namespace spd;

static DevGeom block(const int nc[3], int ng, int nblk)
{
    DevGeom G{};
    G.ng = ng;
    for (int a = 0; a < 3; ++a) { G.nc[a] = nc[a]; G.N[a] = nc[a] + 2*ng; G.nb[a] = 1; }
    G.nb[0] = G.nblk = nblk;
    G.sv = (long long)G.N[0]*G.N[1]*G.N[2];
    G.xh = (long long)G.N[1]*G.N[2]*G.nc[0];
    G.sb = ((5*G.sv + 31)/32)*32;
    G.identity = 1;
    return G;
}

constexpr int kCus = 256;

static TilePlan exhaustive(const DevGeom& G, int H, int SS, bool map)
{
    TilePlan best{};
    double best_cost = 1e299;
    for (int tx = ceil_div(G.nc[0], 64); tx <= ceil_div(G.nc[0], 4); ++tx)
        for (int ty = 1; ty <= G.nc[1]; ++ty)
        {
            const int wi = ceil_div(G.nc[0], tx), wj = ceil_div(G.nc[1], ty);
            if (wj > 64) continue;
            const double cost = tile_cost(G, H, wi, wj);
            if (cost < best_cost - 1e-9)
            {
                best_cost = cost;
                best = TilePlan{wi, wj, ceil_div(G.nc[0], wi), ceil_div(G.nc[1], wj), 1, tile_threads(H, wi, wj), 0};
            }
        }
    best_cost = 1e300;
    for (int zs = ceil_div(G.nc[2], 64); zs <= G.nc[2]; ++zs)
    {
        const size_t lds = sizeof(double)*(size_t)TileLds(best.wi, best.wj, ceil_div(G.nc[2], zs), H, SS, map).total;
        const double cost = share_cost(G, best, zs, lds, kCus);
        if (cost < best_cost - 1e-9) { best_cost = cost; best.zs = zs; best.lds = lds; }
    }
    return best;
}

int main()
{
    char cmd[16];
    int nc[3], ng;
    while (std::scanf("%15s %d %d %d %d", cmd, &nc[0], &nc[1], &nc[2], &ng) == 5)
    {
        if (!std::strcmp(cmd, "offsets"))
        {
            const DevGeom G = block(nc, ng, 1);
            long long far = 0;
            for (int c = 0; c < 16; ++c)
            {
                // corners of the core and of the x-halo sections
                const int i = (c & 1) ? ((c & 8) ? nc[0] + ng - 1 : nc[0] - 1) : ((c & 8) ? -ng : 0);
                const int j = (c & 2) ? nc[1] + ng - 1 : -ng, k = (c & 4) ? nc[2] + ng - 1 : -ng;
                far = std::max(far, stored_offset(G, i, j, k));
            }
            std::printf("%d %d\n", (int)tile_offsets_fit(G), (int)(far <= INT_MAX));
        }
        else if (!std::strcmp(cmd, "plan"))
        {
            int nblk, H, SS, map;
            if (std::scanf("%d %d %d %d", &nblk, &H, &SS, &map) != 4) return 1;
            const DevGeom G = block(nc, ng, nblk);
            const TilePlan p = plan_tile(G, H, SS, map, kCus), q = exhaustive(G, H, SS, map);
            const bool same = p.wi == q.wi && p.wj == q.wj && p.tx == q.tx && p.ty == q.ty && p.zs == q.zs
                && p.nt == q.nt && p.lds == q.lds;
            std::printf("%d %d %d %d %d %d %zu %d\n", p.wi, p.wj, p.tx, p.ty, p.zs, p.nt, p.lds, (int)same);
        }
        else if (!std::strcmp(cmd, "pushes"))
        {
            int nblk;
            if (std::scanf("%d", &nblk) != 1) return 1;
            std::printf("%d\n", (int)stage_pushes(block(nc, ng, nblk)));
        }
        else
        {
            const DevGeom G = block(nc, ng, 1);
            const int n = 20;
            long sum = 0;
            double us = 1e300;
            for (int batch = 0; batch < 20; ++batch)      // (the least: the machine may be busy)
            {
                const auto t0 = std::chrono::steady_clock::now();
                for (int r = 0; r < n; ++r) sum += plan_tile(G, 2, 7, false, kCus - (r & 1)).zs;
                const std::chrono::duration<double, std::micro> d = std::chrono::steady_clock::now() - t0;
                us = std::min(us, d.count()/n);
            }
            std::printf("%.3f %d\n", us, (int)(sum > 0));
        }
    }
    return 0;
}
