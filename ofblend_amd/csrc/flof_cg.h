// flof_cg.h -- solver state and geometry of one pyramid level's PCG, shared by
// the launch-per-kernel form (flof_solve.hip) and the resident form
// (flof_resident.hip).
#pragma once

#include <vector>

#include "flof_internal.h"

namespace flof {

struct CgState {
    double sigma;
    double alpha;
    double alpha_prev;  // alpha of the previous iteration (deferred x update)
    double beta;
    double acc;      // stopping threshold cgAccuracy * resIni
    double resIni;   // signed max of the initial residual
    double resRel;   // (float)(residual / resIni), as ret_residual
    double r2, b2;   // warm-start residual check
    double bb, rr;   // ||b||^2 of the rhs and ||r||^2 of the final residual
    double gamma;    // warm-start scale
    int iters;
    int done;
    int status;  // 0 converged, 1 not converged, 2 sigma 0/NaN, 3 tiny rhs
    int maxIter;
    int warm;    // warm start kept
    int zero;    // result must be zeroed (failed solve)
    int dir_mode;  // k_cg_dir: 0 skip, 1 x and p update, 2 x update only
    int fast_rcp;  // set-up: every interior g_d^2 + diag in rcp_newton's range
};

struct LevelGeom {
    Dims4 D;
    Coord4 C;
    float offd;   // -wSmooth (times mDx2Inv = 1)
    float diag;   // 8*wSmooth + wEnergy, formed as the reference does
    int use_offd; // offd != 0
    float eps;    // VECTOR_EPSILON of FP32 builds
    int fast_rcp; // every interior diagonal entry g_d^2 + diag of the level
                  // lies in the range of rcp_newton (set after the set-up)
};

__device__ __forceinline__ void dd_add4(DD &a, const float4 &u, const float4 &v)
{
    dd_add(a, (double)(u.x * v.x));
    dd_add(a, (double)(u.y * v.y));
    dd_add(a, (double)(u.z * v.z));
    dd_add(a, (double)(u.w * v.w));
}

// x + a p, FP64 product and sum rounded once per component
__device__ __forceinline__ float4 x_plus(const float4 &x, double a, const float4 &p)
{
    return make_float4((float)((double)x.x + a * (double)p.x),
                       (float)((double)x.y + a * (double)p.y),
                       (float)((double)x.z + a * (double)p.z),
                       (float)((double)x.w + a * (double)p.w));
}

// ---------------------------------------------------------------------------
// The resident form: one launch runs every iteration of a level (or of several
// levels of independent problems side by side).

// how a level's interior is dealt to workgroups: py x pz x pt boxes
struct ResPlan {
    int py = 0, pz = 0, pt = 0;
    int nwg = 0;      // py * pz * pt, 0: the level does not fit
    int cells = 0;    // of the largest box
    double cost = 0;  // estimated microseconds per iteration
};
// one level to iterate: its set-up state and vectors (interior cells are used)
struct ResLevel {
    Dims4 D;
    float offd, diag;
    int use_offd;
    const float4 *g, *prec;  // gradients and Jacobi preconditioner
    float4 *x, *r;           // start values in, results out
    const float4 *p;         // first search direction
    float4 *z;               // scratch of the grid's size (exchange)
    CgState *st;
};
// the cheapest plan of at most `budget` workgroups, or the one of the fewest
// (fewest = true); nwg 0 if the level does not fit
ResPlan resident_plan(const Dims4 &D, int budget, bool fewest = false);
// Runs the iterations of all levels (plans[j] for levels[j], at most the
// chip's CUs in total) until each has converged or reached its cap; x, r and
// the solver states hold the results.  false: not run to the end (the launch
// was refused or a workgroup waited too long for another one): the vectors
// are then invalid and the levels must be set up again.
bool resident_iterate(flof_ctx *ctx, const std::vector<ResLevel> &levels,
                      const std::vector<ResPlan> &plans);

}  // namespace flof
