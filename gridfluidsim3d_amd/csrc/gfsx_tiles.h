// gfsx_tiles.h -- where the scatter P2G's tiles lie in memory; plain C++, for
// the host and the device.
#ifndef GFSX_TILES_H
#define GFSX_TILES_H

#include <cstddef>
#include <cstdint>

#ifdef __HIPCC__
#define GFSX_HD __host__ __device__ __forceinline__
#else
#define GFSX_HD inline
#endif

namespace gfsx {

// Tile entries of a scene in HBM: per component one array of
// (nbx*SX) x (nby*SY) x (nbz*SZ) entries (x fastest), brick (bx,by,bz)'s
// tile at (bx*SX, by*SY, bz*SZ), so that the tiles of neighbouring bricks
// along x sit side by side and a face row reads them in sequence.
struct TileGrid {
    size_t base;          // first entry of the component
    int tx, ty;           // entries along x and y
};

GFSX_HD size_t tile_at(const TileGrid &t, int ex, int ey, int ez) {
    return t.base + (size_t)ex + (size_t)t.tx * ((size_t)ey + (size_t)t.ty * (size_t)ez);
}

// Entry (x, y, z) of a tile from the tile's first entry.  Fewer than 2^26
// bricks keep a row's and a layer's entries below 2^32, but not some layers
// of a wide, thin grid (5501 x 5501 x 1 bricks: 1.1e9 entries a layer): the
// layers add up in 64 bits.
GFSX_HD size_t tile_entry(const TileGrid &t, uint32_t x, uint32_t y, uint32_t z) {
    const uint32_t ry = (uint32_t)t.tx, rz = (uint32_t)t.tx * (uint32_t)t.ty;
    return (size_t)(x + ry * y) + (size_t)rz * z;
}

}  // namespace gfsx

#endif
