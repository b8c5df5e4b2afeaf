// ik_launch.hpp -- launch context shared by the engine's host code and the
// field-gather translation units (ik_gather_*.hip), which are compiled separately and in parallel.
#pragma once
#include <hip/hip_runtime.h>

#include "ik_device.hpp"
#include "ik_geom.hpp"
#include "ik_sweep.hpp"

namespace pgt {

// Everything a batch's bond-list and gather launches read.
struct LaunchCtx {
    Geom g;
    int n, G, nf;
    int cap;
    int block;
    int pl;     // grid points per gather lane
    bool pack;  // LDS list entries packed into one int (see k_gather)
    mutable int pl_launched;  // points per lane of the gather actually launched
    const double *grid;
    const int *perm;
    const TileRec *tiles;  // the tile gather's tiles
    const int *tperm;      // grid point of each slot, kTilePoints per tile, -1: none
    int ntiles;
    int tp;            // tile gather: grid points per workgroup (a divisor of kTilePoints)
    int unit;          // and of the window that orders its sums, at least tp
    GLRule R;
    const double *gld;
    double cgnorm;
    const int *cstart;
    const double *spos, *skin;
    const int *bcount;
    const float4 *rec;  // FP32 position and bond count per sorted particle
    const void *bonds;
    GatherOut out;
    int *flags;  // job flags: 1 an adaptive integral ran out of workspace, 2 a tile item had more than 255 bonds
    int tile;    // 1: item-balanced tile gather (tile_form), 0: lane gather
    int lane_terms;  // tile gather, FP32 entries: terms rounded as the lane gather's (see gather_tile_body)
    hipStream_t stream;
};

// Gather points per lane in use: the tuned value where the gather launchers
// pick the unrolled Octic 5-node rule, 1 elsewhere.
inline int gather_pl(int tuned, int cg, int nq, int D, int OD)
{
    return (cg == 0 && nq == 5 && !(D == 3 && OD == 2)) ? tuned : 1;
}

// Whether the tile gather serves this form: the Octic 5-node rule, and every
// fixed rule with FP64 entries.
inline bool tile_form(int cg, int nq, int D, int OD, bool fp32)
{
    return ((cg == 0 && nq == 5) || !fp32) && !(D == 3 && OD == 2);
}

// The tile gather's launch shape: a tile holds at most kTilePoints grid
// points; a workgroup of kTileThreads lanes (one wavefront) takes a tile or
// an equal part of it.
constexpr int kTilePoints = 64, kTileThreads = 64;
// Most particles per frame of a tile gather.
constexpr int64_t kTileMaxParticles = (int64_t)1 << 26;

// Field gather of one batch (fixed-order rule), one function per form and
// translation unit: 2D positions with FP64 or FP32 bond entries, 3D positions
// with 2 x 2 output tensors (a 2D system off the z = 0 plane), and 3D with
// FP64 or FP32 entries.  fields: PGT_FIELD_* bits; cg: kernel kind.
void launch_gather_2d64(const LaunchCtx &c, unsigned fields, int cg);  // ik_gather_2d64.hip
void launch_gather_2d32(const LaunchCtx &c, unsigned fields, int cg);  // ik_gather_2d32.hip
void launch_gather_3d2(const LaunchCtx &c, unsigned fields, int cg);   // ik_gather_3d2.hip
void launch_gather_3d64(const LaunchCtx &c, unsigned fields, int cg);  // ik_gather_3d64.hip
void launch_gather_3d32(const LaunchCtx &c, unsigned fields, int cg);  // ik_gather_3d32.hip
// The tile gather with rules other than the Octic 5-node one, FP64 entries.
void launch_tile_rules_2d(const LaunchCtx &c, unsigned fields, int cg);  // ik_gather_rules_2d.hip
void launch_tile_rules_3d(const LaunchCtx &c, unsigned fields, int cg);  // ik_gather_rules_3d.hip
// Lanes per grid point of the adaptive gather, a power of two from 1 to 32:
// about 64K lanes per frame, so that a small grid still fills the GPU.  Two
// points to a wavefront leave about 28 integrals to bisect in 2D, two lanes
// each (58 us a frame of 1,024 points; four points, a lane each, 106 us).
inline int adaptive_lanes(int64_t G)
{
    int l = 1;
    while (l < 32 && (int64_t)l * G < 65536) l <<= 1;
    return l;
}
inline int64_t adaptive_waves(int64_t G)
{
    const int64_t np = 64 / adaptive_lanes(G);
    return (G + np - 1) / np;
}

// Field gather with the adaptive (QAG) bond integral.  ws null: each
// integral's interval table in the lane's private memory (kQagMax
// intervals), and capped gets 1 when an integral needs more; else the global
// workspace ws of adaptive_workspace_doubles(c, wcap) doubles holds wcap
// intervals per lane.
void launch_gather_adaptive(const LaunchCtx &c, unsigned fields, int cg, int D, int OD, AdaptQ Q, int *capped,
                            double *ws, int wcap);
size_t adaptive_workspace_doubles(const LaunchCtx &c, int wcap);  // ik_gather_adaptive.hip

// The field gather of a sweep (ik_sweep.hpp): one launch over the gather
// ranges of every system, `blocks` workgroups of kTileThreads lanes.
struct SweepGatherCtx {
    const SweepSys *tab;  // device copy of the sweep's table
    int ns;
    int blocks;
    const TileRec *tiles;  // every system's tiles, and their points
    const int *tperm;
    GLRule R;
    const int *cstart;
    const double *spos, *skin;
    int cap;
    const int *bcount;
    const void *bonds;
    unsigned long long *wave_counts;
    int *flags;
    hipStream_t stream;
};
// D: 2 (2 x 2 fields) or 3 (3 x 3)
void launch_sweep_gather(const SweepGatherCtx &c, int D, bool fp32, unsigned fields);  // ik_sweep_gather.hip

}  // namespace pgt
