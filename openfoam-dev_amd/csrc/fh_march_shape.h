// Which boxes the marching sweeps (fh_tile_march.hip) take, and the device
// memory they hold for one.  Plain host code.
#pragma once

#include <cstdint>

namespace fh
{

// cells of the packed coefficient order: whole pencils of 16 x 16 columns,
// and the skew of 21 steps rounded up to whole runs of blocks
inline int64_t march_padded(int32_t nx, int32_t ny, int32_t nz)
{
    return (int64_t)((nx + 15)/16)*((ny + 15)/16)*256*((int64_t)nz + 36);
}

// Boxes the marching sweeps take: below 16 planes along k the padding of
// the skewed coefficient order (21 steps per pencil) exceeds the cells
// themselves; a vector with 64 planes beyond each end, and a pencil's halo
// beyond the out-of-range mark, are within 32-bit byte offsets.  Boxes a few
// cells thick are mostly padding (2 x 2 columns: 64 times the cells), and a
// cell has up to 18 packed values: beyond 1 GiB of them the padding may be
// at most 4 times the cells (576 bytes a cell, beside about 400 of the
// matrix and its solver vectors), else the tiles keep the box.
constexpr int32_t kMarchMinNz = 16;
constexpr int64_t kMarchPaddedBytes = (int64_t)1 << 30;
inline bool march_fits(int32_t nx, int32_t ny, int32_t nz, int64_t valueBytes)
{
    const int64_t padded = march_padded(nx, ny, nz);
    return nz >= kMarchMinNz && nz <= (1 << 18)
           && valueBytes*nx*ny*((int64_t)nz + 128) <= 0xE0000000ll
           && (8*18*padded <= kMarchPaddedBytes || padded <= 4*((int64_t)nx*ny*nz));
}

// device bytes of all these buffers in FP64 (7 values per cell for DIC or
// DILU, 11 and one unpadded for Gauss-Seidel, the halos)
inline int64_t march_bytes(int32_t nx, int32_t ny, int32_t nz)
{
    if (!march_fits(nx, ny, nz, 8)) return 0;
    const int64_t col = (int64_t)((nx + 15)/16)*((ny + 15)/16)*16;
    return 8*(18*march_padded(nx, ny, nz) + (int64_t)nx*ny*nz + 2*col*(nz + 16));
}

} // namespace fh
