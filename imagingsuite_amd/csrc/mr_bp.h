// Internal interface of the parallel-beam back-projection (mr_bp.hip) for
// the other translation units of the library: the plan's resident-table
// path and the kernel launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "muhrec_hip.h"

namespace mr {

// Arguments of the back-projection kernels (one stack).
struct BpArgs {
    const float *sino;
    float *vol;
    const float4 *tab;   // (fStartU, fCos, fSin, 0) per used projection
    const int2 *mask;    // [first, second) per y, 0-based x
    int nu, nv, vpad, nk, nz4, bstride, accumulate;
    int order;           // block -> tile mapping (tile_of_block)
    int ntx, nty, ntz;   // tiles along x, y and slice chunks
    int sw;              // stripe width (tiles) of the XCD-striped order
    // axis-tilt branch: 0 none, 1 MultiProjBPparallel, 2 MultiProjBP,
    // 3 NearestNeighborBP; centeroffset and centerinc of the block
    int tilt;
    float tilt_co, tilt_ci;
    const int *gate;     // LDS kernel without tilt: run only if *gate != 0 (NULL: always)
};

// Uploads the tables of n_proj projections (angles, weights) into the plan
// and sizes its buffers; synchronises s (the host tables are temporaries).
int bp_load_tables(mr_bp_plan *plan, size_t n_proj, const float *angles, const float *weights, hipStream_t s);
// Weighting/transposition and back-projection of d_proj [n_proj][slices][width]
// with the loaded tables into d_volume [width][width][slices]; no host sync.
int bp_enqueue(mr_bp_plan *plan, const float *d_proj, float *d_volume, int accumulate, hipStream_t s);
size_t bp_plan_slices(const mr_bp_plan *plan);
// First detector row of the next bp_enqueue's block (the tilt terms' roi[1]);
// no effect without tilt correction.
void bp_set_tilt_row0(mr_bp_plan *plan, size_t row0);
size_t bp_plan_width(const mr_bp_plan *plan);

// sino[k][u][v] = proj[idx[k]][v][u] * wts[idx[k]] for the nk used
// projections (v < nv; zero for nv <= v < vpad).  gate: only if *gate != 0.
int launch_bp_prep(const float *proj, float *sino, const int *idx, const float *wts, int nu, int nv,
                   int vpad, int nk, hipStream_t s, const int *gate = nullptr);
// Back-projection kernel for one stack.  impl 0: direct gathers (MultiProjBP
// with slices % 4 != 0, whose second column is read at a different offset);
// 1: LDS-staged tiles.  exact: the reference's float operation order.
int run_bp(const BpArgs &a, int interp, int impl, int exact, hipStream_t s);

// Matrix-core form of the fused mode (mr_bp_mfma.hip).
struct BpmArgs {
    const unsigned *split;   // split samples [k][pair][zt][plane][16] (launch_bp_split_prep)
    float *vol;
    const float4 *tab;       // as BpArgs
    const int2 *mask;
    const float2 *scale;     // per slice: factor on the samples, its inverse
    const int *flag;         // set: the samples do not fit the split, the kernel leaves at once
    int nu, nv, vp, npair, nk, nz4;   // vp: slices of whole groups of four, rounded up to 16; npair: column pairs
    int nvs;                 // slices of the projections and of the volume in memory (nv, or more for a slab of them)
    int chain;               // 1: the volume holds the sums of earlier projections, continue them
    int ntx, nty, ntz, zt0, sw;
};
// Voxel tile of the matrix-core kernel for a stack with nk used projections,
// or false where the VALU kernel serves it.
bool bpm_shape(int nu, int nv, int nk, int &tile);
inline int bpm_vp(int nv) { return ((nv & ~3) + 15) & ~15; }
inline int bpm_npair(int nu) { return (nu + 1) / 2; }
size_t bpm_part_words(size_t nv, size_t nk);   // words of launch_bp_scale's maxima and counts
int launch_bp_scale(const float *proj, const int *idx, const float *wts, int nu, int nv, int nk, unsigned *part,
                    float2 *scale, int *flag, hipStream_t s);
int launch_bp_split_prep(const BpmArgs &a, const float *proj, const int *idx, const float *wts, int vpad,
                         hipStream_t s);
int run_bpm(const BpmArgs &a, int tile, hipStream_t s);
// Persistent launch over a batch's items (bp_mfma_batch_kernel).
int bpm_batch_grid(int &grid);
int launch_bpm_batch(const BpmArgs *d_stacks, const int4 *d_items, const int *d_parts, int *d_counters, int grid,
                     hipStream_t s);

}  // namespace mr
