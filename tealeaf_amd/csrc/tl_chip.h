// Whole solver loops in one launch, the fields resident in registers and LDS
// (tl_chip.hip): grids that fit the chip, 2D and 3D, any row length.
//
// A launch-per-pass loop spends its time on such grids in launches, drains
// and the serial march of each wave, not on data: at 512^2 an iteration's
// four kernels took 58 us for 2 MB fields.  Here one block per CU holds a
// tile, and blocks meet once per iteration.
#pragma once

#include "tl_loop.h"

namespace tl {
namespace chip {

// How a grid is cut into tiles, one block of kThreads threads each.  A
// thread owns `k` adjacent cells along y (2D) or z (3D); 2^lxs threads lie
// along x, the others along y.
struct Plan {
    bool ok = false;
    bool refuse = false;        // take every launch for refused (tests)
    int dims = 0, x = 0, y = 0, z = 0, hd = 0;
    int k = 0, lxs = 0;
    int tx = 0, ty = 0, tz = 0;
    int blocks() const { return tx * ty * tz; }
};

// The plan for a grid (halo included), ok = false where it does not fit.
Plan plan(int dims, int x, int y, int z, int hd);

// Returned by the loops when not all of their blocks can be resident at once
// (CUs masked from the stream, or a launch the runtime refuses for it):
// nothing has run and no field has changed.
constexpr int kRefused = -1;

// What a run of iterations ended with.
struct Outcome {
    loop::Report rep;      // of the last iteration
    int last;              // that iteration
    double alpha, beta;    // its alpha and rrn / rro
};

// CG iterations it0, it0 + 1, ... of r, p and u (in place, r and p of the
// state before it0): at most `count`, fewer when `rule` fires.  p has the
// last iteration's calc_p applied; halos are not touched.  alpha and beta of
// every iteration go to the loop's logs (loop::reserve_logs has been called).
int cg(const Plan& pl, double* u, double* p, double* r, const double* kx, const double* ky,
       const double* kz, int it0, int count, const loop::StopRule& rule, Outcome* out);

// Chebyshev iterations it0, it0 + 1, ... with coefficients k0, k0 + 1, ...
// (alphas[0], betas[0], ... on the host): at most `count`, fewer when the squared norm of r (its root with sqrt_err),
// formed every tenth iteration from coefficient `est` on, falls below eps.
// u, p and r in place (r is only written).  out->alpha: the last iteration
// that formed the norm (rep), or -1.
int cheby(const Plan& pl, double* u, double* p, double* r, const double* u0, const double* kx,
          const double* ky, const double* kz, int it0, int count, int k0, int est,
          const double* alphas, const double* betas, double eps, bool sqrt_err, Outcome* out);

// Jacobi iterations it0, it0 + 1, ... of u in place; last_u: the interior
// that the last one read.  rep: the last one's error.
int jacobi(const Plan& pl, double* u, double* last_u, const double* u0, const double* kx,
           const double* ky, const double* kz, int it0, int count, const loop::StopRule& rule,
           Outcome* out);

// Free the device and pinned memory (tlhip_finalise).
void release();

}  // namespace chip
}  // namespace tl
