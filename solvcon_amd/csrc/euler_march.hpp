#pragma once
/*
 * What the march kernels of the multidimensional Euler solver share: the
 * kernel mode bits, the launch parameters (KP) and the view of one cell-type
 * group (GV).
 */

#include "euler_kernels.hpp"

namespace scamd
{

constexpr unsigned BLK = 256;

enum Mode : int
{
    M_SOLN = 1,
    M_BC = 2,
    M_CFL = 4,
    M_DSOLN = 8,
    M_STMEM = 16,
    M_BATCH = 32,
    M_W3 = 64,  // compiled for three wavefronts per SIMD (at most 168 registers)
    M_W2 = 128, // two wavefronts per SIMD (at most 256 registers)
    M_W4 = 256, // four wavefronts per SIMD (at most 128 registers)
    M_WAVES = M_W2 | M_W3 | M_W4,
    M_STAGE = 512, // stage the block's own rows in LDS for neighbour reads
    M_GDMA = 1024, // prefetch the sub-face geometry into LDS (LDS DMA)
    M_STNEXT = 4096, // also write so0t of the level being written (chained so0t)
    M_FAST = 8192, // skip the Jacobian's structural zeros, share reciprocals; report where inexact
    M_FUSED = M_SOLN | M_BC | M_CFL | M_DSOLN,
};

struct KP
{
    int64_t R;
    int64_t G;
    double hdt;
    double qdt;
    double sigma0;
    double taumin;
    double tauscale;
    double const * s0c;
    double const * s1c;
    double * s0n;
    double * s1n;
    double * st;
    double * stn; // so0t of the level being written (chained so0t)
    double const * gam;
    double * cflo;
    double * cflc;
    double const * cen;
    int32_t const * gkind;
    int32_t const * ginl;
    double const * gmat;
    double const * inlet;
    // Batched solves: the instance rank of every body cell (internal order)
    // and the half/quarter time increments of every rank.
    int32_t const * inst;
    double const * bhdt;
    double const * bqdt;
    // The fast/exact pair of every plain launch: the fast kernel stores seq
    // in *redo when one of its cells may differ from the exact arithmetic,
    // and the exact kernel launched after it with gate set returns at once
    // unless *redo holds that seq (then it rewrites the whole group).
    unsigned long long * redo = nullptr;
    unsigned long long seq = 0;
    int gate = 0;
};

struct GV
{
    int64_t off;
    int64_t n;   // cells of the group: the stride of its SoA tables
    int32_t const * nbr;
    double const * geo;
    int64_t cnt; // cells to process, a prefix of the group
};

// The face-lane kernels (euler_lane.hip): one launch for every type group of
// a mesh, several lanes per cell.
constexpr int LANE_GROUPS = 4;

struct LaneGroups
{
    int ng = 0;
    int32_t type[LANE_GROUPS] = {};
    unsigned blk0[LANE_GROUPS + 1] = {}; // first block of each group
    GV g[LANE_GROUPS] = {};
};

// Adds a type group to a launch.
void lane_add(LaneGroups & lg, int32_t type, GV const & g);
// One fused substep over the groups; mode: 0, or M_STNEXT for a single one.
void lane_launch(int ndim, int mode, KP const & p, LaneGroups const & lg, hipStream_t stream);

} /* end namespace scamd */
