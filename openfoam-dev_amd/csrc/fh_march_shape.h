// Which boxes the marching sweeps (fh_tile_march.hip) take, and the device
// memory they hold for one.  Plain host code.
#pragma once

#include "foamhip.h"

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

// what a solve takes of them: the global DIC / DILU passes (FP64, FP32), the
// Gauss-Seidel rows ascending and descending (FP64)
enum : uint32_t { MARCH_DIC64 = 1, MARCH_DIC32 = 2, MARCH_GS_UP = 4, MARCH_GS_DOWN = 8 };

inline uint32_t march_use_smoother(int32_t smoother, bool f32)
{
    const uint32_t dic = f32 ? MARCH_DIC32 : MARCH_DIC64;
    // (the FP32 Gauss-Seidel sweeps run by colours)
    const uint32_t up = f32 ? 0u : MARCH_GS_UP, down = f32 ? 0u : MARCH_GS_DOWN;
    switch (smoother)
    {
        case FH_SMOOTH_GS: return up;
        case FH_SMOOTH_SYMGS: return up | down;
        case FH_SMOOTH_DIC:
        case FH_SMOOTH_FDIC:
        case FH_SMOOTH_DILU: return dic;
        case FH_SMOOTH_DICGS:
        case FH_SMOOTH_DILUGS: return dic | up;
        default: return 0;
    }
}

// the passes a solve with these controls runs on a box
inline uint32_t march_use(const fh_controls& c)
{
    const bool krylov = c.solver == FH_SOLVER_PCG || c.solver == FH_SOLVER_PBICGSTAB
                     || c.solver == FH_SOLVER_PBICG;
    const bool f32 = c.precision == FH_PRECISION_MIXED && c.solver != FH_SOLVER_SMOOTH
                  && c.solver != FH_SOLVER_PBICG;
    if (!krylov)
        return c.solver == FH_SOLVER_SMOOTH || c.solver == FH_SOLVER_GAMG
               ? march_use_smoother(c.smoother, f32) : 0u;
    int32_t p = c.preconditioner;
    if (f32 && c.solver == FH_SOLVER_PCG)
    {
        // the inner preconditioner: tile-local in place of the global DIC
        // unless one is asked for
        if (c.innerPreconditioner >= 0) p = c.innerPreconditioner;
        else if (p == FH_PRECON_DIC || p == FH_PRECON_FDIC) p = FH_PRECON_TILE_DIC;
    }
    if (p == FH_PRECON_DIC || p == FH_PRECON_FDIC || p == FH_PRECON_DILU)
        return f32 ? MARCH_DIC32 : MARCH_DIC64;
    if (p == FH_PRECON_GAMG)
        return march_use_smoother((c.preconditionerControls ? c.preconditionerControls
                                                            : &c)->smoother, f32);
    return 0;
}

// device bytes of the buffers of these uses: 7 packed values per padded cell
// for DIC or DILU, 7 and 4 for Gauss-Seidel and one vector, the halos
inline int64_t march_bytes(int32_t nx, int32_t ny, int32_t nz, uint32_t use)
{
    const int64_t padded = march_padded(nx, ny, nz);
    const int64_t halo = (int64_t)((nx + 15)/16)*((ny + 15)/16)*32*(nz + 16);
    int64_t bytes = 0;
    if ((use & ~MARCH_DIC32) && march_fits(nx, ny, nz, 8))
    {
        if (use & MARCH_DIC64) bytes += 8*7*padded;
        if (use & MARCH_GS_UP) bytes += 8*7*padded;
        if (use & MARCH_GS_DOWN) bytes += 8*4*padded + 8*(int64_t)nx*ny*nz;
        bytes += 8*halo;
    }
    if ((use & MARCH_DIC32) && march_fits(nx, ny, nz, 4)) bytes += 4*(7*padded + halo);
    return bytes;
}

} // namespace fh
