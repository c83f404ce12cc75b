// One CG iteration in one pass over memory (tl_cg_pass.hip), for grids that
// do not fit the chip.
//
// The pass of an iteration applies the last one's alpha and beta and forms
// all the sums of the next (the predict-and-recompute form of CG that
// tl_chip.hip describes): r' = r - alpha A p, u += alpha p, p' = beta p + r',
// and with q = A p' the sums p'.q, q.q, r'.q and r'.r'.  CG with two sums
// a pass apart reads p, r and cond twice.
#pragma once

#include "tl_loop.h"

namespace tl {
namespace pass {

// The sums of a pass, in this order.
enum : int { kPQ, kQQ, kRQ, kRR };

// Whether the r.r after an iteration can be predicted: not where it falls
// below 1% of the one before, as the terms of the prediction then cancel (the
// prediction's error above that line is in tl_chip.hip).
__host__ __device__ inline bool predictable(double next, double rr)
{
    return !(next < 0.01 * rr);
}

// alpha = r.r / p.q; beta from the predicted r.r of the next iteration.
// False where the prediction cancels: that iteration has to sum the new r.r,
// two sums a pass apart.
__host__ __device__ inline bool scalars(const double s[4], double* alpha, double* beta)
{
    const double a = s[kRR] / s[kPQ];
    const double next = (s[kRR] - 2.0 * a * s[kRQ]) + a * a * s[kQQ];
    *alpha = a;
    *beta = next / s[kRR];
    return predictable(next, s[kRR]);
}

// Whether a 2D grid can take the pass (the cond pair's conditions, and room
// for the partial sums of every strip).
bool fits2d(int x, int y, int hd);

// The host's form: with update, one iteration's pass (r_in, p_in -> r_out,
// p_out, u in place); without, only the sums of the r_in and p_in in hand.
int step2d(int x, int y, int hd, bool update, double alpha, double beta, double* u,
           const double* r_in, double* r_out, const double* p_in, double* p_out,
           const double* cond, double rx, double ry, double sums[4]);

}  // namespace pass

namespace loop {
// The sums of a pass finished on the device: the iteration's rrn, beta log,
// stop rule and report, and the next iteration's alpha, beta and alpha log.
// Where those cancel, the report carries kTurn and the loop ends.
int finish_pass(unsigned nblocks, const StopRule& rule, const char* what);
// After begin(), before the first pass: the sums of the state it starts from.
int start_pass(int j0, const double sums[4]);
}  // namespace loop

namespace loop2d {
// step2d's update with alpha and beta from the loop and the sums finished
// there.
int cg_pass(int x, int y, int hd, double* u, const double* r_in, double* r_out,
            const double* p_in, double* p_out, const double* cond, double rx, double ry,
            const loop::StopRule& rule);
}  // namespace loop2d
}  // namespace tl
