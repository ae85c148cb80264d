// The stencil kernels' tiling (csrc/c3d_tile.h) on the host: nx ny nz threads -> blocks launched, or a
// complaint if a cell is missed or taken twice, or a thread without one is given no valid cell, or the
// cells that stencils read are not those that they are said to read.
#include <cstdio>
#include <cstdlib>
#include <vector>

#define __host__
#define __device__
#include "c3d_tile.h"

int main(int argc, char **argv)
{
    if (argc != 5)
        return 3;
    const c3d::Grid G = c3d::make_grid(std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3]));
    const int tb = std::atoi(argv[4]);
    const unsigned blocks = c3d::tile_blocks(G, tb);
    std::vector<char> seen((size_t)G.NX * G.NY * G.NZ, 0);
    for (unsigned b = 0; b < blocks; ++b) {
        c3d::Tile T;
        if (!c3d::tile_of(G, b, blocks, tb, T))
            continue;
        size_t last = 0;
        bool ended = false;
        for (int t = 0; t < tb; ++t) {
            const c3d::TileCell c = c3d::tile_cell(G, T, t);
            const int i = T.i + c.di;
            if (c.di < 0 || i < 2 || i >= G.nx + 2 || c.j < 2 || c.j >= G.ny + 2 || c.k < 2 ||
                c.k >= G.nz + 2)
                return std::puts("outside the interior"), 1;
            // a block's offsets from its first plane are 32 bits of bytes
            if (8.0 * ((double)c.di * G.NY + c.j) * G.NZ >= 4.0e9)
                return std::puts("offset"), 1;
            const size_t x = G.idx(i, c.j, c.k);
            if (c.have && (ended || (t > 0 && x <= last) || seen[x]++))
                return std::puts("a cell twice or out of order"), 1;
            if (!c.have && t > 0 && x != last)
                return std::puts("not the run's last cell"), 1;
            ended = !c.have;
            last = x;
        }
    }
    for (int i = 2; i < G.nx + 2; ++i)
        for (int j = 2; j < G.ny + 2; ++j)
            for (int k = 2; k < G.nz + 2; ++k)
                if (!seen[G.idx(i, j, k)])
                    return std::puts("a cell is missed"), 1;
    // the cells that some interior cell's stencil reads
    std::vector<char> read(seen.size(), 0);
    for (int i = 2; i < G.nx + 2; ++i)
        for (int j = 2; j < G.ny + 2; ++j)
            for (int k = 2; k < G.nz + 2; ++k)
                for (int o = -2; o <= 2; ++o)
                    read[G.idx(i + o, j, k)] = read[G.idx(i, j + o, k)] =
                        read[G.idx(i, j, k + o)] = 1;
    for (size_t c = 0; c < read.size(); ++c)
        if (c3d::stencil_reads(G, (unsigned)c) != (read[c] != 0))
            return std::puts("a cell's use"), 1;
    std::printf("%u\n", blocks);
}
