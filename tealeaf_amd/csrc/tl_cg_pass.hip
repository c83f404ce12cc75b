// One CG iteration in one pass over memory (tl_cg_pass.h).
//
// Bound by HBM: 56 B/cell (read u, r, p, cond; write u, r, p) against the
// 80 of the pair of passes this replaces.  Each wave marches up a tile of
// rows of its own 128-column window (two cells per lane), two levels deep:
// level 1 forms A p, r', u and p' of row m while row m + 1 is being loaded,
// level 2 forms A p' of row m - 1 for the sums.  The window reaches two
// columns beyond the columns it writes on each side and level 1 runs one row
// beyond the tile, so no level needs another wave's results; r and p are
// written to other buffers because the neighbours still read the old ones.
#include "tl_cg_pass.h"
#include "tl_fused.h"
#include "tl_lanes.h"
#include "tl_ops.h"
#include "tealeaf_hip.h"

#include <algorithm>

namespace tl {
namespace pass {
namespace {

// A lane's cells to memory; NT: not kept in the caches.
template <bool NT>
__device__ __forceinline__ void put(double* p, long i, const Cells<double>& c)
{
    if constexpr (NT)
        __builtin_nontemporal_store(__builtin_bit_cast(dvec2, c), reinterpret_cast<dvec2*>(p + i));
    else
        stc(p, i, c);
}

template <bool UPDATE, bool NT>
__global__ void __launch_bounds__(TL_WAVE)
k_cg_pass2d(PitchGrid g, StripTile t, double alpha_arg, double beta_arg,
            const double* __restrict__ alpha_dev, const double* __restrict__ beta_dev,
            double* __restrict__ u, const double* __restrict__ r_in, double* __restrict__ r_out,
            const double* __restrict__ p_in, double* __restrict__ p_out,
            const double* __restrict__ cond, double rx, double ry, TlReduce rd, TlGate gate)
{
    if (gate.closed()) return;
    constexpr int N = 2;
    using C = Cells<double>;
    const double alpha = alpha_dev ? *alpha_dev : alpha_arg;
    const double beta = beta_dev ? *beta_dev : beta_arg;
    const int lane = threadIdx.x;
    const int tile = xcd_tile_of(blockIdx.x, t.nbx * t.nby);
    const int sx = tile % t.nbx, by = tile / t.nbx;
    const int xin0 = g.hd, xin1 = g.hd + g.nx, yin0 = g.hd, yin1 = g.hd + g.ny;
    const int c = t.cw0 + sx * t.w + N * lane;
    const int o0 = g.hd + sx * t.w, o1 = min(o0 + t.w, xin1);    // columns written
    const bool ld_ok = c >= 0 && c + N <= g.X;
    const long X = g.X;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    const int j0 = yin0 + by * t.ty, j1 = min(j0 + t.ty, yin1);
    if (j0 < j1) {                  // uniform per wave
        auto ld = [&](const double* __restrict__ f, long i) -> C {
            return ld_ok ? ldc(f, i) : zeros<double>();
        };
        bool out[N];
#pragma unroll
        for (int k = 0; k < N; ++k) out[k] = c + k >= o0 && c + k < o1;
        const bool all_out = out[0] && out[N - 1];
        // rows yin0-2 .. yin1+1 exist (halo depth >= 2)
        const int ma = max(j0 - 1, yin0), mb = min(j1, yin1 - 1);
        long i0 = (long)ma * X + c;              // cell of row m
        C pd = ld(p_in, i0 - X), pc = ld(p_in, i0), pu = ld(p_in, i0 + X);
        C wc = ld(cond, i0), wu = ld(cond, i0 + X);
        C kyc = ky_of_rows(ry, ld(cond, i0 - X), wc);
        C rc = ld(r_in, i0);
        C uc = UPDATE ? ld(u, i0) : zeros<double>();
        // level 2: p' of rows m-2 and m-1, and row m-1's r', kx and ky below it
        C q2 = zeros<double>(), q1 = zeros<double>(), r1 = zeros<double>();
        C kx1 = zeros<double>(), ky1 = zeros<double>();
        auto level2 = [&](int j, const C& up, const C& kyu) {
            const C dn = j == yin0 ? q1 : q2;
            const C a = apply_a_lane(q1, j == yin1 - 1 ? q1 : up, dn, kx1, kyu, ky1, c, xin0, xin1);
#pragma unroll
            for (int k = 0; k < N; ++k)
                if (out[k]) {
                    acc[kPQ] += a.v[k] * q1.v[k];
                    acc[kQQ] += a.v[k] * a.v[k];
                    acc[kRQ] += r1.v[k] * a.v[k];
                    acc[kRR] += r1.v[k] * r1.v[k];
                }
        };
        for (int m = ma; m <= mb; ++m, i0 += X) {
            // the next row's loads, in flight during this row's arithmetic
            // (beyond the last row: unused, and inside the arrays)
            const C pn = ld(p_in, i0 + 2 * X), wn = ld(cond, i0 + 2 * X), rn = ld(r_in, i0 + X);
            const C un = UPDATE ? ld(u, i0 + X) : zeros<double>();
            const C kyu = ky_of_rows(ry, wc, wu);
            const C kxc = kx_of_row(rx, wc, wc.v[0]);
            C q0 = pc, r0 = rc;
            if constexpr (UPDATE) {
                const C a = apply_a_lane(pc, m == yin1 - 1 ? pc : pu, m == yin0 ? pc : pd, kxc, kyu,
                                         kyc, c, xin0, xin1);
                C u0;
#pragma unroll
                for (int k = 0; k < N; ++k) {
                    r0.v[k] = rc.v[k] - alpha * a.v[k];
                    u0.v[k] = uc.v[k] + alpha * pc.v[k];
                    q0.v[k] = beta * pc.v[k] + r0.v[k];
                }
                if (m >= j0 && m < j1) {
                    if (all_out) {
                        put<NT>(r_out, i0, r0);
                        put<NT>(p_out, i0, q0);
                        put<NT>(u, i0, u0);
                    } else {
#pragma unroll
                        for (int k = 0; k < N; ++k)
                            if (out[k]) {
                                r_out[i0 + k] = r0.v[k];
                                p_out[i0 + k] = q0.v[k];
                                u[i0 + k] = u0.v[k];
                            }
                    }
                }
            }
            if (m > j0) level2(m - 1, q0, kyc);
            q2 = q1;
            q1 = q0;
            r1 = r0;
            kx1 = kxc;
            ky1 = kyc;
            kyc = kyu;
            pd = pc;
            pc = pu;
            pu = pn;
            wc = wu;
            wu = wn;
            rc = rn;
            uc = un;
        }
        // the last interior row has no row above it to wait for; kyc is now
        // the coefficient of its upper face
        if (j1 == yin1) level2(yin1 - 1, q1, kyc);
    }
    tl_reduce_partial<4, TL_WAVE>(acc, rd);
}

// One wave per block, and two per SIMD: the waves then run side by side from
// start to end, and the rows that a tile shares with its neighbours are a
// small part of it.  At 4096^2 (56 B/cell) tiles of 69 rows took 217 us an
// iteration, 8 to 56 rows 229 to 240; at 3072^2 38 rows 105, 17 rows 117, 77
// rows 116; blocks of four waves 234 at their best size at 4096^2.
StripTile geometry(int x, int y, int hd, PitchGrid* g)
{
    *g = PitchGrid{x, hd, x - 2 * hd, y - 2 * hd};
    StripTile t = strip_tile<double>(*g, 2, 1, 1);
    int ty = tl_tile_rows_override();
    if (ty <= 0) {
        const int tiles = std::max(1, 2 * 4 * fused::device_cus() / t.ns);
        ty = (int)tl_cdiv(g->ny, tiles);
    }
    for (;; ty *= 2) {
        t = strip_tile<double>(*g, 2, ty, 1);
        if ((long)t.nbx * t.nby <= TL_MAX_RED_BLOCKS) return t;
    }
}

// Whether the six fields of a pass exceed the 256 MB memory-side cache: what
// a pass writes is then gone before the next reads it, and storing past the
// caches leaves them to the rows that tiles share (4096^2 220 -> 217 us,
// 3072^2 124 -> 105 us; at 2000^2, where the fields stay, 44 -> 52 us).
bool beyond_cache(int x, int y) { return 6.0 * sizeof(double) * x * y > 256e6; }

// The launch under the current gate; *nb: its partials.
int launch2d(const char* what, int x, int y, int hd, bool update, double alpha, double beta,
             const double* alpha_dev, const double* beta_dev, double* u, const double* r_in,
             double* r_out, const double* p_in, double* p_out, const double* cond, double rx,
             double ry, unsigned* nb)
{
    TL_TRY(tl_ensure_init());
    if (!fits2d(x, y, hd))
        return tl_fail(TLHIP_ERR_ARG, "%s: needs halo depth >= 2, an even x and at most %d strips "
                       "of columns (x=%d y=%d hd=%d)", what, TL_MAX_RED_BLOCKS, x, y, hd);
    TL_REQUIRE(r_in && p_in && cond && (!update || (u && r_out && p_out)), what, "null field");
    TL_REQUIRE(!update || (r_out != r_in && p_out != p_in && r_out != p_out && u != r_in &&
                           u != p_in && u != r_out && u != p_out),
               what, "the fields must be distinct buffers");
    TL_REQUIRE(all_aligned(u, r_in, r_out, p_in, p_out, cond), what,
               "fields must be 16-byte aligned");
    PitchGrid g;
    const StripTile t = geometry(x, y, hd, &g);
    *nb = (unsigned)(t.nbx * t.nby);
    const int slot = tl_timer_begin(what);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(*nb), dim3(TL_WAVE), 0, tl_stream(), g, t, alpha, beta,
                           alpha_dev, beta_dev, u, r_in, r_out, p_in, p_out, cond, rx, ry,
                           tl_reduce_slots(), tl_gate());
    };
    if (!update) go(k_cg_pass2d<false, false>);
    else if (beyond_cache(x, y)) go(k_cg_pass2d<true, true>);
    else go(k_cg_pass2d<true, false>);
    tl_timer_end(slot);
    return tl_check_launch(what);
}

const char* const kName2 = "tl_cg_pass2d";

}  // namespace

bool fits2d(int x, int y, int hd)
{
    if (hd < 2 || x % 2 || x <= 2 * hd || y <= 2 * hd || (long)x * y > (1L << 31) - 1) return false;
    // one block, with its partial sums, per strip at the least (8.1 million columns)
    const PitchGrid g{x, hd, x - 2 * hd, y - 2 * hd};
    return strip_tile<double>(g, 2, g.ny, 1).nbx <= TL_MAX_RED_BLOCKS;
}

int step2d(int x, int y, int hd, bool update, double alpha, double beta, double* u,
           const double* r_in, double* r_out, const double* p_in, double* p_out,
           const double* cond, double rx, double ry, double sums[4])
{
    unsigned nb;
    TL_TRY(launch2d(kName2, x, y, hd, update, alpha, beta, nullptr, nullptr, u, r_in, r_out, p_in,
                    p_out, cond, rx, ry, &nb));
    TL_TRY(tl_finish_reduce(4, nb, kName2));
    return tl_fetch(4, sums, kName2);
}

}  // namespace pass

namespace loop2d {
int cg_pass(int x, int y, int hd, double* u, const double* r_in, double* r_out,
            const double* p_in, double* p_out, const double* cond, double rx, double ry,
            const loop::StopRule& rule)
{
    unsigned nb;
    TL_TRY(pass::launch2d(pass::kName2, x, y, hd, true, 0.0, 0.0, loop::alpha(), loop::beta(), u,
                          r_in, r_out, p_in, p_out, cond, rx, ry, &nb));
    return loop::finish_pass(nb, rule, pass::kName2);
}
}  // namespace loop2d
}  // namespace tl
