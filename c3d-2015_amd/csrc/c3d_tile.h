// c3d_tile.h -- the grid with its ghosts, and how the stencil kernels tile its interior.  Plain
// index arithmetic that also compiles on the host, where its coverage is checked.
#pragma once
#include <cstddef>
#include <cstdint>

namespace c3d {

constexpr int kTB = 256;  // threads of a block (kTBSmall: below)

struct Grid {
    int nx, ny, nz;
    int NX, NY, NZ;  // with ghosts
    __host__ __device__ size_t idx(int i, int j, int k) const
    {
        return (size_t)k + (size_t)NZ * ((size_t)j + (size_t)NY * (size_t)i);
    }
};

inline Grid make_grid(int nx, int ny, int nz)
{
    return Grid{nx, ny, nz, nx + 4, ny + 4, nz + 4};
}

// A block of tb threads (a power of two) works on tb consecutive cells of a run of flattened interior cells (z
// fastest).  Block b goes to XCD b % kXcd, and XCD x takes the x-th eighth of an order of the
// blocks that keeps compact what it has in flight, so that a plane is fetched into that XCD's L2
// once and reused by the four planes after it; dealing consecutive blocks over the XCDs instead
// makes every L2 fetch its own copy of the y and x neighbours.
//   - Planes of at most kStripCells: the run is the whole interior, and the order is the cells'.
//     Only the last block is not full, however small the planes are.
//   - Larger planes: a run per x-plane, and the order walks strips of kStripCells of the plane
//     along x.  A plane's last block is not full: at most one block in kStripCells / tb + 1.
// Cutting small planes into runs of their own as well left most lanes idle: a 4096 x 4 x 4 grid took
// 2.4 (kinetic flux) to 6 (moment flux, nm = 9) times as long as with the whole interior
// flattened, a line of 100000 cells 10 to 50 times.
constexpr int kXcd = 8;
constexpr int kStripCells = 4096;
// Grids of at most a block of kTB per CU are cut into blocks of one wave, which spreads the waves
// over the CUs and their L1s.
constexpr int kTBSmall = 64;
__host__ __device__ inline int64_t plane_cells(const Grid &G) { return (int64_t)G.ny * G.nz; }
__host__ __device__ inline bool flat_tiles(const Grid &G) { return plane_cells(G) <= kStripCells; }
__host__ __device__ inline int64_t tile_count(const Grid &G, int tb)
{
    const int64_t run = flat_tiles(G) ? plane_cells(G) * G.nx : plane_cells(G);
    const int64_t n = (run + tb - 1) >> __builtin_ctz(tb);
    return flat_tiles(G) ? n : n * G.nx;
}
inline unsigned tile_blocks(const Grid &G, int tb)
{
    return (unsigned)((tile_count(G, tb) + kXcd - 1) / kXcd * kXcd);
}
inline int tile_threads(const Grid &G, int numCU)
{
    return tile_blocks(G, kTB) <= (unsigned)numCU ? kTBSmall : kTB;
}

struct Tile {
    int i;      // the first cell's plane, ghosts counted
    int64_t p;  // and its place in the plane's flattened interior
};
__host__ __device__ inline bool tile_of(const Grid &G, unsigned block, unsigned blocks, int tb,
                                        Tile &t)
{
    // a launch has fewer than 2^32 threads, so that blocks and cells are counted in 32 bits
    const unsigned b = block % kXcd * (blocks / kXcd) + block / kXcd;
    if (b >= tile_count(G, tb))
        return false;
    const unsigned P = (unsigned)plane_cells(G), sh = __builtin_ctz(tb);
    if (flat_tiles(G)) {
        const unsigned c = b << sh, i = c / P;
        t.i = 2 + (int)i;
        t.p = c - i * P;
        return true;
    }
    const unsigned nP = (P + tb - 1) >> sh, nS = kStripCells >> sh;
    const unsigned strip = b / (nS * G.nx), rem = b - strip * nS * G.nx;
    const unsigned width = nP - strip * nS < nS ? nP - strip * nS : nS;
    t.i = 2 + (int)(rem / width);
    t.p = (int64_t)(strip * nS + rem % width) << sh;
    return true;
}

// Thread `lane` of the tile's block.  Past the end of the run it has no cell of its own and is
// given the run's last one.
struct TileCell {
    int di;    // planes beyond the tile's (flat runs: at most (kTB - 1) / plane + 1)
    int j, k;  // ghosts counted
    bool have;
};
__host__ __device__ inline TileCell tile_cell(const Grid &G, const Tile &T, int lane)
{
    const unsigned P = (unsigned)plane_cells(G);
    unsigned r = (unsigned)T.p + (unsigned)lane, di = 0;
    bool have = r < P;
    if (flat_tiles(G)) {
        const unsigned left = (unsigned)(G.nx + 2 - T.i);  // planes from the tile's on
        di = r / P;
        r -= di * P;
        have = di < left;
        di = have ? di : left - 1;
    }
    r = have ? r : P - 1;
    const unsigned j = r / (unsigned)G.nz;
    return TileCell{(int)di, 2 + (int)j, 2 + (int)(r - j * (unsigned)G.nz), have};
}

// Whether a stencil (two cells each way along each axis, from an interior cell) reads the cell: not
// if two or three of its coordinates are ghosts'.  Those cells are never filled.
__host__ __device__ inline bool stencil_reads(const Grid &G, unsigned cell)
{
    const unsigned row = cell / (unsigned)G.NZ, plane = row / (unsigned)G.NY;
    const int k = (int)(cell - row * (unsigned)G.NZ), j = (int)(row - plane * (unsigned)G.NY),
              i = (int)plane;
    return (i < 2 || i >= G.nx + 2) + (j < 2 || j >= G.ny + 2) + (k < 2 || k >= G.nz + 2) <= 1;
}

}  // namespace c3d
