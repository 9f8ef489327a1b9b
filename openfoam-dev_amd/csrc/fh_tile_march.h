// Marching global DIC / DILU and Gauss-Seidel sweeps for hex boxes
// (fh_tile_march.hip).
#pragma once

#include "fh_march_shape.h"
#include "fh_tile_sweep.h"

namespace fh
{

// buffers of the marching sweeps of one matrix in one precision: the pass
// coefficients premultiplied by rD in the order the wavefronts read them,
// and the pencil halos (every value the sentinel between launches)
template<class T>
struct MarchBufs
{
    DBuf<T> fwd, bwd, halo;
    int kind = -1;             // factor the coefficients were packed with
    bool haloReady = false;
    // Gauss-Seidel: coefficients and diagonal of the two passes, products of
    // the old values (forward) and the source less the lower products
    // (backward) of the running sweep
    DBuf<T> gsFwd, gsBwd, gsOld, gsPrime;
    bool gsFwdReady = false, gsBwdReady = false;
};

// packs dir (k, j, i coefficients of the pass, read at the neighbour with
// dirShift) times rD for the forward or backward pass
template<class T>
void launch_march_pack(bool backward, const TileView& G, const T* rD, const T* const dir[3],
                       bool dirShift, MarchBufs<T>& b, hipStream_t s);
// the same for the Gauss-Seidel rows, with the diagonal
void launch_march_pack_gs(bool backward, const TileView& G, const double* diag,
                          const double* const dir[3], bool dirShift, MarchBufs<double>& b,
                          hipStream_t s);
template<class T>
void march_prepare_halo(const TileView& G, MarchBufs<T>& b, hipStream_t s);
// One global DIC / DILU pass; backward with d.dotR also sums w*dotR into
// one partial per pencil.  Returns the pencil count.
template<class T>
int32_t launch_sweep_march(bool backward, const TileView& G, const SweepData<T>& d,
                           const MarchBufs<T>& b, TileSync& sync, unsigned int* err,
                           DevState* st, hipStream_t s,
                           const FusedFinalize& F = FusedFinalize());

// One Gauss-Seidel sweep of d.w in place with source d.x; d.dir: the upper
// coefficients (k, j, i) forward, the lower ones backward (the other side of
// the sweep).  Forward reads d.w before, backward after the forward sweep.
void launch_sweep_march_gs(bool backward, const TileView& G, const SweepData<double>& d,
                           MarchBufs<double>& b, TileSync& sync, unsigned int* err,
                           DevState* st, hipStream_t s);

} // namespace fh
