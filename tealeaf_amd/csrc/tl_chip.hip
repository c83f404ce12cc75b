// Whole solver loops in one launch with the fields in registers and LDS
// (tl_chip.h).
//
// A block of 1024 threads owns a tile of up to 8192 cells and at most one
// block runs per CU, so up to 2.1 million cells stay on the chip for the
// whole loop: r, A p and all but one of the coefficients of a thread's cells
// in registers, p (with a ring of the neighbours' cells) and the coefficient
// left (kx, in 3D ky) in LDS.  CG's u stays in memory, read and written by its
// own thread only; so does Chebyshev's and Jacobi's u0 with 8 cells a thread.
//
// Blocks meet once per iteration.  CG has two dot products with a data
// dependence (alpha = r.r / p.Ap, then beta from the new r.r); here all of
// an iteration's sums are formed in one meeting, as the predict-and-
// recompute form of CG does (Chen and Carson, "Predict-and-recompute
// conjugate gradient variants", SIAM J. Sci. Comput. 42 (2020); the
// prediction is Meurant's): with q = A p,
//     r'.r' is predicted as r.r - 2 alpha r.q + alpha^2 q.q   (for beta),
//     r.r is summed from the r in hand                        (for alpha,
//                                        the stop test and the logs).
// alpha and every vector update are the reference's expressions; beta carries
// more rounding error than the ratio of two sums, as its terms cancel: against
// the sum of the same r in extended precision (medians) 2e-16 where an
// iteration leaves half of r.r, 2e-15 where it leaves a tenth, 1e-14 at a
// fiftieth (largest seen 3e-14), where the sum itself is off by 1e-16.  alpha
// comes from the real r.r, so nothing of it accumulates, and solutions are as
// far from an exact solve as with two sums.  Where the residual falls further
// in one iteration (below 1% of r.r, from where the error could pass 1e-13),
// the blocks meet again and sum the new r.r, as the two-sum form does.
//
// The same meeting hands the tile's outer cells of q to the neighbours: each
// block also keeps r and p of its ring and updates them with that q, so the
// ring's p equals the owner's bit for bit and no second meeting is needed.
//
// What bounds an iteration is the meeting: a block's sums reach the others in
// about 1 us and are read back in another, beside 0.3 to 3 us of arithmetic
// (1 to 4 cells per thread).  512^2 (K = 1) 4.6 us, 1024^2 (K = 4) 6.7; 128^3
// (K = 8) 19, most of which the meeting and the arithmetic do not account for.
// Launch by launch they took 57, 76 and 63 us.  Chebyshev and Jacobi, 1001 x
// 777: 4.9 us an iteration, 512^2: 4.3 us a sweep (25 and 13).
//
// Coherence: everything blocks exchange (q of outer cells, the sums) goes
// through agent-scope atomic loads and stores, which the XCDs' L2s do not
// hold back; a wave waits for its stores (vmcnt) before the block publishes
// its sums.  Nothing else is shared while the kernel runs, so no L2
// write-back or invalidate is needed.  Every block must be resident at once:
// the launch is cooperative, and a wait gives up after kWaitS seconds.
#include "tl_chip.h"
#include "tl_lanes.h"
#include "tealeaf_hip.h"

#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <type_traits>

namespace tl {
namespace chip {
namespace {

constexpr int kThreads = 1024;
constexpr int kWavesB = kThreads / TL_WAVE;
constexpr int kMaxBlocks = 256;        // one per CU, and 4 sums of each poll in one go
constexpr int kSums = 4;
constexpr int kPhases = 3;             // meetings whose slots rotate
constexpr double kWaitS = 10.0;
constexpr long kChunk = 4096;          // iterations per launch

// ------------------------------------------------------------ geometry

struct Geo {
    int x, y, hd, nx, ny, nz;
    long xy;
    int tx, ty, tz;
};

// Cells of the faces a block hands over: x low, x high, y low, y high (, z
// low, z high), in this order.
struct Faces {
    int nx, ny, nz;        // cells of an x, y and z face
    __host__ __device__ constexpr int total() const { return 2 * (nx + ny + nz); }
};

template <int DIMS, int K>
__host__ __device__ constexpr Faces faces_of(int lxs)
{
    const int lx = 1 << lxs, ry = kThreads >> lxs;
    return DIMS == 2 ? Faces{ry * K, lx, 0} : Faces{ry * K, lx * K, lx * ry};
}

// Ring cells of the x and y faces that a thread looks after.  A z face has
// one cell per thread.
template <int DIMS, int K, int LXS>
constexpr int ring_per_thread()
{
    const Faces f = faces_of<DIMS, K>(LXS);
    return (2 * (f.nx + f.ny) + kThreads - 1) / kThreads;
}

template <int DIMS, int K>
__host__ __device__ constexpr int lds_p(int lxs)
{
    const int lx = 1 << lxs, ry = kThreads >> lxs;
    return DIMS == 2 ? (lx + 2) * (ry * K + 2) : (lx + 2) * (ry + 2) * (K + 2);
}
// Coefficients in LDS: kx with the column right of the tile (2D); ky with
// the row above it, and kx of that column (3D).
template <int DIMS, int K>
__host__ __device__ constexpr int lds_k(int lxs)
{
    const int lx = 1 << lxs, ry = kThreads >> lxs;
    return DIMS == 2 ? (lx + 1) * ry * K : lx * (ry + 1) * K + ry * K;
}

// ------------------------------------------------------------ exchange

__device__ __forceinline__ double ld_agent(const double* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(double* p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// This wave's stores have reached the point they are coherent at.
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ double lane_value(double v, int lane)
{
    const int2 a = __builtin_bit_cast(int2, v);
    int2 r;
    r.x = __builtin_amdgcn_readlane(a.x, lane);
    r.y = __builtin_amdgcn_readlane(a.y, lane);
    return __builtin_bit_cast(double, r);
}

// The four sums of a wave in lanes 0, 16, 32, 48 (value 0, 1, 2, 3): two
// halving exchanges spread the values over the lanes, then one butterfly.
__device__ __forceinline__ double wave_sum4(const double v[kSums], int lane)
{
    const bool h32 = lane & 32, h16 = lane & 16;
    const double s0 = h32 ? v[0] : v[2], s1 = h32 ? v[1] : v[3];
    const double k0 = h32 ? v[2] : v[0], k1 = h32 ? v[3] : v[1];
    const double a = k0 + __shfl_xor(s0, 32, TL_WAVE), b = k1 + __shfl_xor(s1, 32, TL_WAVE);
    double c = (h16 ? b : a) + __shfl_xor(h16 ? a : b, 16, TL_WAVE);
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) c += __shfl_xor(c, off, TL_WAVE);
    return c;
}

// Sums over 16 groups of four: value i of the total in lane i.
__device__ __forceinline__ double sum_groups(double v)
{
#pragma unroll
    for (int off = 4; off <= 32; off <<= 1) v += __shfl_xor(v, off, TL_WAVE);
    return v;
}

struct Mail {           // pinned, host-mapped; armed with TL_MAIL_EMPTY
    double rrn, err, flags, last, alpha, beta;
};

// part alternates between two buffers by meeting: with one block a wave may
// start the next meeting while another still reads the last one's parts, and
// it passes that meeting's barrier only after everybody has.
struct Shared {
    double part[2][kWavesB][kSums];
    double tot[kWavesB][kSums];
    int expired;
};

// All blocks' sums of meeting n: every block publishes its own four and reads
// everybody's.  A value is its own ready flag (TL_MAIL_EMPTY is a signalling
// NaN that no sum can be); the slots of the next meeting are emptied
// by their owner while nobody can be reading them: the last meeting that used
// them is two back, and a block publishes one only after it has read the one
// before.  Returns false when a wait expired.
__device__ __forceinline__ bool all_sums(const double v[kSums], Shared& sh, double* slots, int n,
                                         int nb, double out[kSums])
{
    const int tid = threadIdx.x, lane = tid & (TL_WAVE - 1), wave = tid / TL_WAVE;
    const double c = wave_sum4(v, lane);
    double (*part)[kSums] = sh.part[n & 1];
    if ((lane & 15) == 0) part[wave][lane >> 4] = c;
    double* next = slots + (size_t)((n + 1) % kPhases) * kMaxBlocks * kSums;
    double* mine = slots + (size_t)(n % kPhases) * kMaxBlocks * kSums;
    if (nb > 1 && tid < kSums)
        st_agent(&next[blockIdx.x * kSums + tid],
                 __builtin_bit_cast(double, (unsigned long long)TL_MAIL_EMPTY));
    wait_stores();
    __syncthreads();
    double t;
    if (nb == 1) {
        t = sum_groups(part[lane >> 2][lane & 3]);
    } else {
        if (wave == 0) {
            const double s = sum_groups(part[lane >> 2][lane & 3]);
            if (lane < kSums) st_agent(&mine[blockIdx.x * kSums + lane], s);
        }
        double got = 0.0;
        if (tid < nb * kSums) {
            got = ld_agent(&mine[tid]);
            unsigned spin = 0;
            unsigned long long t0 = 0;
            while (__builtin_bit_cast(unsigned long long, got) == TL_MAIL_EMPTY) {
                if ((++spin & 255u) == 0) {
                    const unsigned long long now = __builtin_amdgcn_s_memrealtime();   // 100 MHz
                    if (!t0) t0 = now;
                    if (now - t0 > (unsigned long long)(kWaitS * 1e8)) {
                        sh.expired = 1;
                        break;
                    }
                }
                got = ld_agent(&mine[tid]);
            }
        }
        got = sum_groups(got);
        if (lane < kSums) sh.tot[wave][lane] = got;
        __syncthreads();
        if (sh.expired) return false;
        t = sum_groups(sh.tot[lane >> 2][lane & 3]);
    }
#pragma unroll
    for (int i = 0; i < kSums; ++i) out[i] = lane_value(t, i);
    return true;
}

__global__ void __launch_bounds__(256) k_empty(double* slots, int n, unsigned* rounds)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < kMaxBlocks) rounds[i] = 0;
    if (i < n) slots[i] = __builtin_bit_cast(double, (unsigned long long)TL_MAIL_EMPTY);
}

// ------------------------------------------------------------ tile

// An address part formed anew where it is used, so that the addresses of all
// of a thread's cells are not kept in registers from iteration to iteration.
__device__ __forceinline__ unsigned opaque(unsigned v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// A thread's place in its tile, its cells' offsets in the fields and in LDS,
// and its ring cells.
template <int DIMS, int K, int LXS>
struct Tile {
    static constexpr int NE = ring_per_thread<DIMS, K, LXS>();
    static constexpr int LX = 1 << LXS, RY = kThreads >> LXS;
    // LDS pitches of p: row, plane (3D), in-thread step
    static constexpr int PX = LX + 2, PP = PX * (RY + 2), KP = DIMS == 2 ? PX : PP;
    // of the coefficients there: in-thread step, step to a cell's other face,
    // and 3D's column right of the tile
    static constexpr int k_step = DIMS == 2 ? LX + 1 : (RY + 1) * LX;
    static constexpr int k_next = DIMS == 2 ? 1 : LX;
    static constexpr int e_step = RY;
    static constexpr Faces f = faces_of<DIMS, K>(LXS);
    int lx, t;                  // thread column and row
    unsigned first, kstep;      // offset of cell 0 in a field and step to the next
    int kn;                     // cells inside the domain (0..K)
    int at;                     // LDS index of cell 0 of p
    int k_at, e_at;             // of its coefficients, and of kx right of the tile
    bool edge_x;                // 3D: the tile's last column
    int lo, hi;                 // LDS offset of the left and right neighbour (0: mirror)
    int ylo, yhi;               // 3D: of the row neighbours
    bool first_k, last_k;       // the domain starts at cell 0 / ends at cell kn - 1 here
    unsigned xmine;             // this block's faces in the exchange buffer
    size_t xall;                // doubles of one parity of it
    bool face_xl, face_xh, face_yl, face_yh, face_zl, face_zh;   // neighbours there

    __device__ __forceinline__ Tile(const Geo& g)
    {
        const int tid = threadIdx.x, b = blockIdx.x;
        lx = tid & (LX - 1);
        t = tid >> LXS;
        const int bx = b % g.tx, by = (b / g.tx) % g.ty, bz = b / (g.tx * g.ty);
        const int X = bx * LX + lx;
        int Y, Z = 0, n;
        if constexpr (DIMS == 2) {
            Y = by * (RY * K) + t * K;
            n = X < g.nx ? g.ny - Y : 0;
            kstep = g.x;
            at = (t * K + 1) * PX + lx + 1;
            k_at = t * K * (LX + 1) + lx;
            e_at = 0;
            first_k = Y == 0;
            last_k = Y + K >= g.ny;
            ylo = yhi = 0;
        } else {
            Y = by * RY + t;
            Z = bz * K;
            n = X < g.nx && Y < g.ny ? g.nz - Z : 0;
            kstep = (unsigned)g.xy;
            at = PP + (t + 1) * PX + lx + 1;
            k_at = tid;
            e_at = K * (RY + 1) * LX + t;
            first_k = Z == 0;
            last_k = Z + K >= g.nz;
            ylo = Y == 0 ? 0 : -PX;
            yhi = Y == g.ny - 1 ? 0 : PX;
        }
        kn = n < 0 ? 0 : (n > K ? K : n);
        first = (unsigned)((g.hd + X) + (long)(g.hd + Y) * g.x +
                           (DIMS == 3 ? (long)(g.hd + Z) * g.xy : 0));
        edge_x = lx == LX - 1;
        lo = X == 0 ? 0 : -1;
        hi = X == g.nx - 1 ? 0 : 1;
        xmine = (unsigned)(b * f.total());
        xall = (size_t)gridDim.x * f.total();
        face_xl = bx > 0;
        face_xh = bx < g.tx - 1;
        face_yl = by > 0;
        face_yh = by < g.ty - 1;
        face_zl = DIMS == 3 && bz > 0;
        face_zh = DIMS == 3 && bz < g.tz - 1;
    }

    // Entry e of the ring's x and y faces: its LDS index in p, where its owner
    // hands the value over, and its cell; false where there is none.
    __device__ __forceinline__ bool ring(const Geo& g, int e, int* dst, unsigned* src, long* cell,
                                         bool* inside) const
    {
        const int b = blockIdx.x;
        const int bx = b % g.tx, by = (b / g.tx) % g.ty, bz = b / (g.tx * g.ty);
        const int X0 = bx * LX, Y0 = by * (DIMS == 2 ? RY * K : RY), Z0 = DIMS == 3 ? bz * K : 0;
        const int h = DIMS == 2 ? RY * K : RY;      // tile rows
        int face, m = e;
        if (m < 2 * f.nx) {
            face = m >= f.nx;
            m -= face * f.nx;
        } else if ((m -= 2 * f.nx) < 2 * f.ny) {
            face = m >= f.ny;
            m -= face * f.ny;
            face += 2;
        } else {
            return false;
        }
        int cx, cy, cz, nbk;      // the cell within the tile (-1 or the size: the ring)
        bool have;
        if (face < 2) {
            cx = face == 0 ? -1 : LX;
            cy = DIMS == 2 ? m : m % RY;
            cz = DIMS == 2 ? 0 : m / RY;
            have = face == 0 ? face_xl : face_xh;
            nbk = face == 0 ? b - 1 : b + 1;
        } else {
            cy = face == 2 ? -1 : h;
            cx = m & (LX - 1);
            cz = m >> LXS;
            have = face == 2 ? face_yl : face_yh;
            nbk = face == 2 ? b - g.tx : b + g.tx;
        }
        if (!have) return false;
        const int opposite = face ^ 1;
        const int off = opposite < 2 ? opposite * f.nx : 2 * f.nx + (opposite - 2) * f.ny;
        *src = (unsigned)(nbk * f.total() + off + m);
        *dst = DIMS == 2 ? (cy + 1) * PX + cx + 1 : (cz + 1) * PP + (cy + 1) * PX + cx + 1;
        const int X = X0 + cx, Y = Y0 + cy, Z = Z0 + cz;
        *inside = X < g.nx && Y < g.ny && (DIMS == 2 || Z < g.nz);
        *cell = (long)(g.hd + X) + (long)(g.hd + Y) * g.x + (DIMS == 3 ? (long)(g.hd + Z) * g.xy : 0);
        return true;
    }

    // 3D: where the blocks below and above hand over their z faces (this
    // thread's cell of them; the ring cells are LDS at - PP and at + K PP).
    __device__ __forceinline__ unsigned zlow(const Geo& g) const
    {
        return xmine - g.tx * g.ty * f.total() + 2 * (f.nx + f.ny) + f.nz + threadIdx.x;
    }
    __device__ __forceinline__ unsigned zhigh(const Geo& g) const
    {
        return xmine + g.tx * g.ty * f.total() + 2 * (f.nx + f.ny) + threadIdx.x;
    }

    // Hand the tile's outer cells of v to the neighbours.
    __device__ __forceinline__ void hand_over(const double* v, double* xb) const
    {
        double* my = xb + opaque(xmine);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int m = DIMS == 2 ? t * K + k : k * RY + t;
            if (lx == 0 && face_xl) st_agent(&my[m], v[k]);
            if (lx == LX - 1 && face_xh) st_agent(&my[f.nx + m], v[k]);
            if constexpr (DIMS == 3) {
                if (t == 0 && face_yl) st_agent(&my[2 * f.nx + k * LX + lx], v[k]);
                if (t == RY - 1 && face_yh) st_agent(&my[2 * f.nx + f.ny + k * LX + lx], v[k]);
            }
        }
        if constexpr (DIMS == 2) {
            if (t == 0 && face_yl) st_agent(&my[2 * f.nx + lx], v[0]);
            if (t == RY - 1 && face_yh) st_agent(&my[2 * f.nx + f.ny + lx], v[K - 1]);
        } else {
            const int m = t * LX + lx;
            if (face_zl) st_agent(&my[2 * (f.nx + f.ny) + m], v[0]);
            if (face_zh) st_agent(&my[2 * (f.nx + f.ny) + f.nz + m], v[K - 1]);
        }
    }
};

// Coefficients of a thread's cells.  2D: kx in LDS, ky in registers.  3D: ky
// in LDS, kx and kz in registers (kx of the right face comes from the next
// lane).  What each leaves in registers is what keeps 8 cells per thread
// inside 128 of them.
template <int DIMS, int K, int LXS>
struct Coefs {
    using T = Tile<DIMS, K, LXS>;
    double kk[K + 1];                      // ky (2D) or kz (3D) of cells 0..K
    double kx[DIMS == 3 ? K : 1];

    __device__ __forceinline__ void load(const Geo& g, const T& tl, double* s_k,
                                         const double* __restrict__ kx_,
                                         const double* __restrict__ ky_,
                                         const double* __restrict__ kz_)
    {
        const double* along = DIMS == 2 ? ky_ : kz_;
        const double* lds = DIMS == 2 ? kx_ : ky_;
        const long other = DIMS == 2 ? 1 : g.x;
#pragma unroll
        for (int k = 0; k <= K; ++k)
            kk[k] = tl.kn > 0 && k <= tl.kn ? along[tl.first + k * tl.kstep] : 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const bool in = k < tl.kn;
            const long c = tl.first + k * tl.kstep;
            if constexpr (DIMS == 3) kx[k] = in ? kx_[c] : 0.0;
            // both faces of the cell; two threads write a shared one the same
            if (in) {
                double* sk = s_k + tl.k_at + k * tl.k_step;
                sk[0] = lds[c];
                sk[tl.k_next] = lds[c + other];
                if constexpr (DIMS == 3) {
                    if (tl.edge_x || tl.hi == 0) s_k[tl.e_at + k * tl.e_step] = kx_[c + 1];
                }
            }
        }
    }

    // f(k, c, x, y, z) for each of the thread's cells: the cell's value of s
    // (in LDS with its ring) and per axis the two faces' coefficients and the
    // values beyond them.  Cells beyond a domain edge mirror the cell (a
    // depth-1 reflective halo).
    struct Axis {
        double kc, ku, lo, hi;        // lower and upper face, lower and upper neighbour
    };
    template <class F>
    __device__ __forceinline__ void visit(const T& tl, const double* s, const double* s_k,
                                          F&& f) const
    {
        const double* p = s + tl.at;
        double below = p[-tl.KP], c = p[0];
        if (tl.first_k) below = c;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double above = p[(k + 1) * tl.KP];
            const double next = above;
            if (tl.last_k && k == tl.kn - 1) above = c;
            const double* sk = s_k + tl.k_at + k * tl.k_step;
            const Axis along{kk[k], kk[k + 1], below, above};
            Axis x{0.0, 0.0, p[k * tl.KP + tl.lo], p[k * tl.KP + tl.hi]};
            if constexpr (DIMS == 2) {
                x.kc = sk[0];
                x.ku = sk[1];
                f(k, c, x, along, Axis{});
            } else {
                const double e = s_k[tl.e_at + k * tl.e_step];
                x.kc = kx[k];
                x.ku = tl_lane_next(x.kc, e);
                if (tl.edge_x || tl.hi == 0) x.ku = e;
                const Axis y{sk[0], sk[tl.k_next], p[k * tl.KP + tl.ylo], p[k * tl.KP + tl.yhi]};
                f(k, c, x, y, along);
            }
            below = c;
            c = next;
        }
    }

    // A s at a cell; the association is 2d/shared.h:50-54 / 3d/shared.h:52-58.
    static __device__ __forceinline__ double product(double c, const Axis& x, const Axis& y,
                                                     const Axis& z)
    {
        const double d = (1.0 + (x.ku + x.kc)) + (y.ku + y.kc);
        const double a = (DIMS == 2 ? d : d + (z.ku + z.kc)) * c - (x.ku * x.hi + x.kc * x.lo)
                         - (y.ku * y.hi + y.kc * y.lo);
        return DIMS == 2 ? a : a - (z.ku * z.hi + z.kc * z.lo);
    }

    // q = A s of the thread's cells (0 outside the domain), and s.q added to
    // *dot.
    __device__ __forceinline__ void apply(const T& tl, const double* s, const double* s_k,
                                          double* dot, double q[K]) const
    {
        visit(tl, s, s_k, [&](int k, double c, const Axis& x, const Axis& y, const Axis& z) {
            q[k] = k < tl.kn ? product(c, x, y, z) : 0.0;
            *dot += q[k] * c;
        });
    }
};

// The ring of a field in LDS: where each of the block's ring cells is and
// where its owner hands it over.
template <int DIMS, int K, int LXS>
struct Ring {
    using T = Tile<DIMS, K, LXS>;
    static constexpr int NE = T::NE;
    int dst[NE];            // < 0: none
    unsigned src[NE];
    bool zl, zh;            // 3D: the cells below and above this thread's

    // load(slot, LDS index, cell) for every ring cell there is; slots NE and
    // NE + 1 are the z cells (a tile with a neighbour above is full along z)
    template <class F>
    __device__ __forceinline__ void init(const Geo& g, const T& tl, F&& load)
    {
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            unsigned from = 0;
            long cell = 0;
            bool in = false;
            int to = 0;
            dst[i] = -1;
            src[i] = 0;
            if (tl.ring(g, (int)threadIdx.x + i * kThreads, &to, &from, &cell, &in) && in) {
                dst[i] = to;
                src[i] = from;
                load(i, to, cell);
            }
        }
        zl = DIMS == 3 && tl.face_zl && tl.kn > 0;
        zh = DIMS == 3 && tl.face_zh && tl.kn > 0;
        if (zl) load(NE, tl.at - tl.KP, (long)tl.first - tl.kstep);
        if (zh) load(NE + 1, tl.at + K * tl.KP, (long)tl.first + (long)K * tl.kstep);
    }

    // What the owners handed over, on its way; use() gives it to
    // put(slot, LDS index, value).  Between the two there is time for work
    // that does not need it.
    struct Handed {
        double v[NE], w[2];
    };
    __device__ __forceinline__ Handed fetch(const Geo& g, const T& tl, const double* xb) const
    {
        Handed h;
#pragma unroll
        for (int i = 0; i < NE; ++i) h.v[i] = dst[i] >= 0 ? ld_agent(&xb[src[i]]) : 0.0;
        h.w[0] = zl ? ld_agent(&xb[tl.zlow(g)]) : 0.0;
        h.w[1] = zh ? ld_agent(&xb[tl.zhigh(g)]) : 0.0;
        return h;
    }
    template <class F>
    __device__ __forceinline__ void use(const T& tl, const Handed& h, F&& put) const
    {
#pragma unroll
        for (int i = 0; i < NE; ++i)
            if (dst[i] >= 0) put(i, dst[i], h.v[i]);
        if (zl) put(NE, tl.at - tl.KP, h.w[0]);
        if (zh) put(NE + 1, tl.at + K * tl.KP, h.w[1]);
    }
};

// Wait until the blocks this one shares a face with have handed over their
// cells of round n (1, 2, ...).  What is handed over alternates between two
// buffers: a block writes a buffer again two rounds later, after its
// neighbours have published the round between, which they do after they read
// it.
template <class T>
__device__ __forceinline__ bool meet_neighbours(const Geo& g, const T& tl, unsigned* rounds,
                                                unsigned n, Shared& sh)
{
    const int tid = threadIdx.x, b = blockIdx.x;
    wait_stores();
    __syncthreads();
    if (tid == 0) __hip_atomic_store(&rounds[b], n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid < 6) {
        const int step[3] = {1, g.tx, g.tx * g.ty};
        const bool have[6] = {tl.face_xl, tl.face_xh, tl.face_yl, tl.face_yh, tl.face_zl, tl.face_zh};
        bool mine = false;
        int at = b;
#pragma unroll
        for (int i = 0; i < 6; ++i)
            if (tid == i) {
                mine = have[i];
                at = b + (i & 1 ? step[i >> 1] : -step[i >> 1]);
            }
        if (mine) {
            unsigned spin = 0;
            unsigned long long t0 = 0;
            while (__hip_atomic_load(&rounds[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < n) {
                if ((++spin & 255u) == 0) {
                    const unsigned long long now = __builtin_amdgcn_s_memrealtime();   // 100 MHz
                    if (!t0) t0 = now;
                    if (now - t0 > (unsigned long long)(kWaitS * 1e8)) {
                        sh.expired = 1;
                        break;
                    }
                }
            }
        }
    }
    __syncthreads();
    return !sh.expired;
}

// A kernel's start: p's place in LDS zeroed (outside the domain and in a
// ring without neighbours, where the mirror is read instead, it stays zero),
// the coefficients loaded.
template <int DIMS, int K, int LXS>
__device__ __forceinline__ void begin_tile(const Geo& g, const Tile<DIMS, K, LXS>& tl,
                                           Coefs<DIMS, K, LXS>& co, double* s, double* s_k,
                                           Shared& sh, const double* kx, const double* ky,
                                           const double* kz)
{
    if (threadIdx.x == 0) sh.expired = 0;
    for (int i = threadIdx.x; i < lds_p<DIMS, K>(LXS); i += kThreads) s[i] = 0.0;
    for (int i = threadIdx.x; i < lds_k<DIMS, K>(LXS); i += kThreads) s_k[i] = 0.0;
    __syncthreads();
    co.load(g, tl, s_k, kx, ky, kz);
}

// The run's outcome to the host, by one thread of the grid.
__device__ __forceinline__ void report(Mail* mail, double rrn, double err, int flags, int last,
                                       double a, double b)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const double m[6] = {rrn, err, (double)flags, (double)last, a, b};
    double* to = &mail->rrn;
#pragma unroll
    for (int i = 0; i < 6; ++i)
        __hip_atomic_store(to + i, m[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ------------------------------------------------------------ CG

struct CgArgs {
    Geo g;
    double *u, *p, *r;
    const double *kx, *ky, *kz;
    double *xbuf, *slots, *alog, *blog;
    Mail* mail;
    int it0, count;
    loop::StopRule rule;
};

__device__ __forceinline__ int stop_flags(const loop::StopRule& rule, int j, double rrn, double err)
{
    int flags = 0;
    if (rule.rel ? rrn <= rule.rel_target : fabs(err) < rule.eps) flags |= loop::kConverged;
    if (rule.sw == 1 && err < rule.eps_lim && j + 1 > 20) flags |= loop::kSwitch;
    if (rule.sw == 2 && j + 1 > rule.presteps && err < 1.0) flags |= loop::kSwitch;
    return flags;
}

template <int DIMS, int K, int LXS>
__global__ void __launch_bounds__(kThreads) k_chip_cg(CgArgs A)
{
    extern __shared__ double lds[];
    __shared__ Shared sh;
    const Geo& g = A.g;
    const Tile<DIMS, K, LXS> tl(g);
    double* s_p = lds;
    double* s_k = lds + lds_p<DIMS, K>(LXS);
    const int nb = (int)gridDim.x;
    constexpr int NE = decltype(tl)::NE;
    Coefs<DIMS, K, LXS> co;
    begin_tile(g, tl, co, s_p, s_k, sh, A.kx, A.ky, A.kz);
    double r[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const bool in = k < tl.kn;
        const long c = tl.first + k * tl.kstep;
        r[k] = in ? A.r[c] : 0.0;
        if (in) s_p[tl.at + k * tl.KP] = A.p[c];
    }
    // the ring: r in registers, p in LDS
    double rr[NE + 2] = {};
    Ring<DIMS, K, LXS> ring;
    ring.init(g, tl, [&](int i, int to, long cell) {
        rr[i] = A.r[cell];
        s_p[to] = A.p[cell];
    });
    __syncthreads();

    const unsigned any_cell = (unsigned)(g.hd + (long)g.hd * g.x + (DIMS == 3 ? g.hd * g.xy : 0));
    double prev = 0.0, alpha = 0.0, beta_true = 0.0;
    double rrn = 0.0, err = 0.0;
    int flags = 0, n = 0, meeting = 0;
    for (;; ++n) {
        double q[K], v[kSums] = {0.0, 0.0, 0.0, 0.0}, tot[kSums];
        co.apply(tl, s_p, s_k, &v[0], q);          // p.Ap
#pragma unroll
        for (int k = 0; k < K; ++k) {
            v[1] += q[k] * q[k];
            v[2] += r[k] * q[k];
            v[3] += r[k] * r[k];
        }
        double* xb = A.xbuf + (size_t)(n & 1) * tl.xall;
        if (nb > 1) tl.hand_over(q, xb);
        const bool go_on = n < A.count;
        // with few cells per thread, u is loaded ahead of the meeting (whose
        // drain it shares: the loads are back before the sums are published)
        constexpr bool kEarlyU = K <= 2;
        double u[kEarlyU ? K : 1];
        if constexpr (kEarlyU) {
            // (every lane loads something: a load that only some paths wait
            // for makes the next iteration wait for this one's stores)
#pragma unroll
            for (int k = 0; k < K; ++k) u[k] = A.u[k < tl.kn ? tl.first + k * tl.kstep : any_cell];
        }
        if (!all_sums(v, sh, A.slots, meeting++, nb, tot)) {
            flags = -1;
            break;
        }
        const double rro = tot[3];
        if (n > 0) {                    // iteration it0 + n - 1 ends with this r.r
            const int j = A.it0 + n - 1;
            rrn = rro;
            beta_true = rro / prev;
            err = A.rule.sqrt_err ? sqrt(rrn) : rrn;
            flags = stop_flags(A.rule, j, rrn, err);
            if (blockIdx.x == 0 && threadIdx.x == 0) A.blog[j] = beta_true;
            if (flags || !go_on) break;
        }
        prev = rro;
        alpha = rro / tot[0];
        const double predicted = (rro - 2.0 * alpha * tot[2]) + alpha * alpha * tot[1];
        double beta = predicted / rro;
        if (blockIdx.x == 0 && threadIdx.x == 0) A.alog[A.it0 + n] = alpha;
        typename decltype(ring)::Handed handed{};
        if (nb > 1) handed = ring.fetch(g, tl, xb);
        const unsigned cell0 = opaque(tl.first);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            // outside the domain p, q and r are zero, and stay so
            const double step = alpha * s_p[tl.at + k * tl.KP];
            double* ug = A.u + cell0 + k * tl.kstep;
            if constexpr (kEarlyU) {
                u[k] += step;
                if (k < tl.kn) *ug = u[k];
            } else if (k < tl.kn) {
                *ug += step;
            }
            r[k] -= alpha * q[k];
            if (K == 8 && k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        if (!(predicted >= 0.01 * rro)) {          // the same decision in every block
            double w[kSums] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < K; ++k) w[3] += r[k] * r[k];
            if (!all_sums(w, sh, A.slots, meeting++, nb, tot)) {
                flags = -1;
                break;
            }
            beta = tot[3] / rro;
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (k < tl.kn) s_p[tl.at + k * tl.KP] = beta * s_p[tl.at + k * tl.KP] + r[k];
        if (nb > 1) {
            ring.use(tl, handed, [&](int i, int at, double q_ring) {
                rr[i] -= alpha * q_ring;
                s_p[at] = beta * s_p[at] + rr[i];
            });
        }
        __syncthreads();
    }
    // the state after the last iteration, back to the fields
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (k < tl.kn) {
            const long c = tl.first + k * tl.kstep;
            A.r[c] = r[k];
            A.p[c] = s_p[tl.at + k * tl.KP];
        }
    }
    report(A.mail, rrn, err, flags, A.it0 + n - 1, alpha, beta_true);
}

// ------------------------------------------------------------ Chebyshev

// A field that the loop only reads at a thread's own cells: in registers, or
// with 8 cells per thread, which leave none, from the L2 each time.
template <int DIMS, int K, int LXS>
struct Steady {
    static constexpr bool kHeld = K < 8;
    double v[kHeld ? K : 1];
    const double* f;
    unsigned step;
    int kn;
    __device__ __forceinline__ Steady(const Tile<DIMS, K, LXS>& tl, const double* field)
        : f(field), step(tl.kstep), kn(tl.kn)
    {
        if constexpr (kHeld)
#pragma unroll
            for (int k = 0; k < K; ++k)
                v[k] = k < kn ? f[tl.first + k * step] : 0.0;
    }
    __device__ __forceinline__ double operator()(int k, unsigned cell0) const
    {
        if constexpr (kHeld) return v[k];
        else return k < kn ? f[cell0 + k * step] : 0.0;
    }
};

struct ChebyArgs {
    Geo g;
    double *u, *p, *r;
    const double *u0, *kx, *ky, *kz;
    double *xbuf, *slots;
    unsigned* rounds;
    Mail* mail;
    const double *alphas, *betas;     // of the run's iterations
    int it0, count, k0, est;
    double eps;
    int sqrt_err;
};

// Iterations of the Chebyshev loop (2d/drivers/cheby_driver.c with
// cheby.c:57-85): w = A u, r = u0 - w, p = alpha p + beta r, u += p.  Blocks
// meet their neighbours only, except where the norm of r is due (every tenth
// iteration from the estimate on) and in the launch's last iteration: a block
// whose wait expired far from block 0, which reports, would otherwise leave
// its tile behind and go unnoticed.
template <int DIMS, int K, int LXS>
__global__ void __launch_bounds__(kThreads) k_chip_cheby(ChebyArgs A)
{
    extern __shared__ double lds[];
    __shared__ Shared sh;
    const Geo& g = A.g;
    const Tile<DIMS, K, LXS> tl(g);
    double* s_u = lds;
    double* s_k = lds + lds_p<DIMS, K>(LXS);
    const int nb = (int)gridDim.x;
    Coefs<DIMS, K, LXS> co;
    begin_tile(g, tl, co, s_u, s_k, sh, A.kx, A.ky, A.kz);
    double p[K];
    const Steady<DIMS, K, LXS> u0(tl, A.u0);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const bool in = k < tl.kn;
        const long c = tl.first + k * tl.kstep;
        p[k] = in ? A.p[c] : 0.0;
        if (in) s_u[tl.at + k * tl.KP] = A.u[c];
    }
    Ring<DIMS, K, LXS> ring;
    ring.init(g, tl, [&](int, int to, long cell) { s_u[to] = A.u[cell]; });
    __syncthreads();

    double rrn = 0.0, err = 0.0, normed = -1.0;
    int flags = 0, n = 0, meeting = 0;
    for (;; ++n) {
        const double alpha = A.alphas[n], beta = A.betas[n];
        double un[K], v[kSums] = {0.0, 0.0, 0.0, 0.0};
        const int t = A.it0 + n;
        const bool norm = A.k0 + n >= A.est && (t + 1) % 10 == 0;
        const bool may_end = norm || n + 1 >= A.count;
        const unsigned cell0 = opaque(tl.first);
        co.visit(tl, s_u, s_k, [&](int k, double c, const auto& x, const auto& y, const auto& z) {
            const double r = u0(k, cell0) - co.product(c, x, y, z);
            p[k] = alpha * p[k] + beta * r;
            un[k] = c + p[k];
            if (k < tl.kn) {
                v[0] += r * r;
                if (may_end) A.r[cell0 + k * tl.kstep] = r;
            }
        });
        __syncthreads();          // everybody has read the old u
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (k < tl.kn) s_u[tl.at + k * tl.KP] = un[k];
        double* xb = A.xbuf + (size_t)(n & 1) * tl.xall;
        if (nb > 1) tl.hand_over(un, xb);
        bool fine = true;
        if (may_end) {
            double tot[kSums];
            fine = all_sums(v, sh, A.slots, meeting++, nb, tot);
            if (norm) {
                rrn = tot[0];
                err = A.sqrt_err ? sqrt(rrn) : rrn;
                normed = t;
                if (fabs(err) < A.eps) flags = loop::kConverged;
            }
        } else if (nb > 1) {
            fine = meet_neighbours(g, tl, A.rounds, n + 1, sh);
        }
        if (!fine) {
            flags = -1;
            break;
        }
        if (flags || n + 1 >= A.count) break;
        if (nb > 1) {
            ring.use(tl, ring.fetch(g, tl, xb), [&](int, int to, double v) { s_u[to] = v; });
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (k < tl.kn) {
            const long c = tl.first + k * tl.kstep;
            A.u[c] = s_u[tl.at + k * tl.KP];
            A.p[c] = p[k];
        }
    }
    report(A.mail, rrn, err, flags, A.it0 + n, normed, 0.0);
}

// ------------------------------------------------------------ Jacobi

struct JacobiArgs {
    Geo g;
    double *u, *last_u;
    const double *u0, *kx, *ky, *kz;
    double *xbuf, *slots;
    Mail* mail;
    int it0, count;
    loop::StopRule rule;
};

// Jacobi sweeps (jacobi.c:61-100): the error, the sum of |change|, is due
// every iteration, so the blocks all meet; every 50th iteration the squared
// norm of the residual is added to it (jacobi_driver.c:22-40).
template <int DIMS, int K, int LXS>
__global__ void __launch_bounds__(kThreads) k_chip_jacobi(JacobiArgs A)
{
    extern __shared__ double lds[];
    __shared__ Shared sh;
    const Geo& g = A.g;
    const Tile<DIMS, K, LXS> tl(g);
    double* s_u = lds;
    double* s_k = lds + lds_p<DIMS, K>(LXS);
    const int nb = (int)gridDim.x;
    Coefs<DIMS, K, LXS> co;
    begin_tile(g, tl, co, s_u, s_k, sh, A.kx, A.ky, A.kz);
    double old[K];
    const Steady<DIMS, K, LXS> u0(tl, A.u0);
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (k < tl.kn) s_u[tl.at + k * tl.KP] = A.u[tl.first + k * tl.kstep];
    Ring<DIMS, K, LXS> ring;
    ring.init(g, tl, [&](int, int to, long cell) { s_u[to] = A.u[cell]; });
    __syncthreads();

    double e = 0.0, err = 0.0;
    int flags = 0, n = 0, meeting = 0;
    for (;; ++n) {
        double un[K], v[kSums] = {0.0, 0.0, 0.0, 0.0}, tot[kSums];
        const unsigned cell0 = opaque(tl.first);
        co.visit(tl, s_u, s_k, [&](int k, double c, const auto& x, const auto& y, const auto& z) {
            double num = (u0(k, cell0) + (x.ku * x.hi + x.kc * x.lo)) + (y.ku * y.hi + y.kc * y.lo);
            double den = (1.0 + (x.kc + x.ku)) + (y.kc + y.ku);
            if constexpr (DIMS == 3) {
                num = num + (z.ku * z.hi + z.kc * z.lo);
                den = den + (z.kc + z.ku);
            }
            un[k] = num / den;
            old[k] = c;
            if (k < tl.kn) v[0] += fabs(un[k] - c);
        });
        __syncthreads();          // everybody has read the old u
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (k < tl.kn) s_u[tl.at + k * tl.KP] = un[k];
        double* xb = A.xbuf + (size_t)(n & 1) * tl.xall;
        if (nb > 1) tl.hand_over(un, xb);
        if (!all_sums(v, sh, A.slots, meeting++, nb, tot)) {
            flags = -1;
            break;
        }
        if (nb > 1) {
            ring.use(tl, ring.fetch(g, tl, xb), [&](int, int to, double w) { s_u[to] = w; });
        }
        __syncthreads();
        e = tot[0];
        const int t = A.it0 + n;
        if (t % 50 == 0) {
            double w[kSums] = {0.0, 0.0, 0.0, 0.0};
            co.visit(tl, s_u, s_k,
                     [&](int k, double c, const auto& x, const auto& y, const auto& z) {
                         const double d = u0(k, cell0) - co.product(c, x, y, z);
                         if (k < tl.kn) w[0] += d * d;
                     });
            if (!all_sums(w, sh, A.slots, meeting++, nb, tot)) {
                flags = -1;
                break;
            }
            e = e + tot[0];
        }
        err = A.rule.sqrt_err ? sqrt(e) : e;
        flags = stop_flags(A.rule, t, e, err);
        if (flags || n + 1 >= A.count) break;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (k < tl.kn) {
            const long c = tl.first + k * tl.kstep;
            A.u[c] = s_u[tl.at + k * tl.KP];
            A.last_u[c] = old[k];
        }
    }
    report(A.mail, e, err, flags, A.it0 + n, 0.0, 0.0);
}

// ------------------------------------------------------------ host

struct Host {
    double* xbuf = nullptr;
    size_t xlen = 0;
    double* slots = nullptr;
    unsigned* rounds = nullptr;
    double* coefs = nullptr;      // [2 * kChunk]
    Mail* mail = nullptr;
    bool late = false;            // a launch whose report was given up on may still run
    int cus = 0;
};
Host g_chip;

int hip_fail(hipError_t e, const char* what)
{
    return tl_fail(TLHIP_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}
#define CHIP_HIP(call, what)                                  \
    do {                                                      \
        hipError_t _e = (call);                               \
        if (_e != hipSuccess) return hip_fail(_e, what);      \
    } while (0)

int compute_units()
{
    if (g_chip.cus) return g_chip.cus;
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    return g_chip.cus = n;
}

template <int DIMS, int K>
size_t lds_bytes(int lxs)
{
    return sizeof(double) * (lds_p<DIMS, K>(lxs) + lds_k<DIMS, K>(lxs));
}

template <int N>
using Int = std::integral_constant<int, N>;

// f(dims, cells per thread, log2 of the row's threads) as constants
template <class F>
int with_plan(const Plan& pl, F&& f)
{
    auto row = [&](auto d, auto k) -> int {
        switch (pl.lxs) {
        case 4: return f(d, k, Int<4>{});
        case 5: return f(d, k, Int<5>{});
        case 6: return f(d, k, Int<6>{});
        }
        return tl_fail(TLHIP_ERR_ARG, "tl::chip: no kernel for rows of 2^%d", pl.lxs);
    };
    auto cells = [&](auto d) -> int {
        switch (pl.k) {
        case 1: return row(d, Int<1>{});
        case 2: return row(d, Int<2>{});
        case 4: return row(d, Int<4>{});
        case 8: return row(d, Int<8>{});
        }
        return tl_fail(TLHIP_ERR_ARG, "tl::chip: no kernel for %d cells per thread", pl.k);
    };
    return pl.dims == 2 ? cells(Int<2>{}) : cells(Int<3>{});
}

int prepare(int nb, size_t xdoubles, const char* what)
{
    Host& h = g_chip;
    TL_TRY(tl_ensure_init());
    if (h.late) {       // its report must not be taken for the next launch's
        CHIP_HIP(hipStreamSynchronize(tl_stream()), what);
        h.late = false;
    }
    if (!h.slots) {
        CHIP_HIP(hipMalloc(&h.slots, sizeof(double) * kPhases * kMaxBlocks * kSums), what);
        CHIP_HIP(hipMalloc(&h.rounds, sizeof(unsigned) * kMaxBlocks), what);
        CHIP_HIP(hipHostMalloc(&h.mail, sizeof(Mail), hipHostMallocMapped | hipHostMallocCoherent),
                 what);
    }
    if (xdoubles > h.xlen) {
        CHIP_HIP(hipStreamSynchronize(tl_stream()), what);
        if (h.xbuf) CHIP_HIP(hipFree(h.xbuf), what);
        h.xbuf = nullptr;
        h.xlen = 0;
        CHIP_HIP(hipMalloc(&h.xbuf, sizeof(double) * xdoubles), what);
        h.xlen = xdoubles;
    }
    if (nb == 1) return 0;        // a single block has nobody to meet
    const int n = kPhases * kMaxBlocks * kSums;
    hipLaunchKernelGGL(k_empty, dim3((n + 255) / 256), dim3(256), 0, tl_stream(), h.slots, n, h.rounds);
    return tl_check_launch(what);
}

constexpr int kMailWords = sizeof(Mail) / sizeof(double);

void arm_mail()
{
    volatile unsigned long long* b = (volatile unsigned long long*)g_chip.mail;
    for (int i = 0; i < kMailWords; ++i) b[i] = TL_MAIL_EMPTY;
    std::atomic_thread_fence(std::memory_order_seq_cst);
}

bool mail_ready()
{
    volatile unsigned long long* b = (volatile unsigned long long*)g_chip.mail;
    for (int i = 0; i < kMailWords; ++i)
        if (b[i] == TL_MAIL_EMPTY) return false;
    return true;
}

int wait_mail(Mail* out, const char* what)
{
    const auto start = std::chrono::steady_clock::now();
    auto t0 = start;
    for (unsigned spin = 1; !mail_ready(); ++spin) {
        if ((spin & 1023u) != 0) continue;
        const auto now = std::chrono::steady_clock::now();
        if (now - t0 < std::chrono::milliseconds(1)) continue;
        t0 = now;
        const hipError_t e = hipStreamQuery(tl_stream());
        if (e == hipErrorNotReady) {
            const double waited = std::chrono::duration<double>(now - start).count();
            if (waited > tl_wait_limit_s())
                return tl_fail(TLHIP_ERR_HIP, "%s: no report after %.0f s (wait limit)", what,
                               waited);
            continue;
        }
        if (e != hipSuccess) return hip_fail(e, what);
        if (!mail_ready()) return tl_fail(TLHIP_ERR_HIP, "%s: the loop did not report", what);
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    memcpy(out, g_chip.mail, sizeof(Mail));
    return 0;
}

Geo geo_of(const Plan& pl)
{
    Geo g{};
    g.x = pl.x, g.y = pl.y, g.hd = pl.hd;
    g.xy = (long)pl.x * pl.y;
    g.nx = pl.x - 2 * pl.hd, g.ny = pl.y - 2 * pl.hd, g.nz = pl.dims == 3 ? pl.z - 2 * pl.hd : 1;
    g.tx = pl.tx, g.ty = pl.ty, g.tz = pl.tz;
    return g;
}

}  // namespace

namespace {
size_t plan_lds(const Plan& pl)
{
    size_t n = 0;
    (void)with_plan(pl, [&](auto dims, auto kc, auto) -> int {
        n = lds_bytes<decltype(dims)::value, decltype(kc)::value>(pl.lxs);
        return 0;
    });
    return n;
}
// 160 KB of LDS per CU, less the kernel's own
constexpr size_t kMaxLds = 160 * 1024 - sizeof(Shared) - 64;
}  // namespace

Plan plan(int dims, int x, int y, int z, int hd)
{
    Plan best;
    const int nx = x - 2 * hd, ny = y - 2 * hd, nz = dims == 3 ? z - 2 * hd : 1;
    if (nx < 1 || ny < 1 || nz < 1) return best;
    // (an environment that masks CUs does not show in the device's count)
    if (getenv("HSA_CU_MASK") || getenv("ROC_GLOBAL_CU_MASK")) return best;
    const int most = std::min(kMaxBlocks, compute_units());
    // A block per CU at most: blocks wait for each other.  The fewest cells
    // per thread that fit are fastest or nearly so (us per CG iteration with 1,
    // 2, 4, 8 cells: 300 x 260 4.2 4.6 5.5 7.8; 512^2 4.7 4.7 5.6 8.1; 1024^2
    // - - 6.9 9.2; 32^3 4.3 4.7 5.7 10.2; 64^3 6.6 5.6 6.4 11.2), except that
    // a grid which fits one block needs no meeting across the chip.  That is
    // worth up to 4 cells, not 8 (CG, Chebyshev, Jacobi: 64^2, 4 cells in one
    // block 3.7 1.3 2.6, 1 cell in four 3.4 1.7 3.0; 64 x 128, 8 cells in one
    // 5.8 2.6 5.0, 1 cell in eight 3.6 2.1 3.2).
    double cost = 1e30;
    for (int k = 1; k <= 8; k *= 2) {
        for (int lxs = 6; lxs >= 4; --lxs) {
            const int lx = 1 << lxs, ry = kThreads >> lxs;
            Plan p;
            p.ok = true;
            p.dims = dims, p.x = x, p.y = y, p.z = z, p.hd = hd, p.k = k, p.lxs = lxs;
            p.tx = (int)tl_cdiv(nx, lx);
            p.ty = (int)tl_cdiv(ny, dims == 2 ? ry * k : ry);
            p.tz = dims == 3 ? (int)tl_cdiv(nz, k) : 1;
            if ((long)p.tx * p.ty * p.tz > most || plan_lds(p) > kMaxLds) continue;
            const double c = k + (p.blocks() > 1 ? 5.0 : 0.0) + p.blocks() * 1e-3;
            if (c < cost) {
                cost = c;
                best = p;
            }
        }
    }
    return best;
}

namespace {
// Whether the stream's CUs hold all blocks at once.
bool room_for(int blocks)
{
    uint32_t mask[32] = {};
    if (hipExtStreamGetCUMask(tl_stream(), 32, mask) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    int cus = 0;
    for (uint32_t m : mask) cus += __builtin_popcount(m);
    return cus >= blocks;
}

// Launch one of the loops, args(g) giving its arguments, and wait for its
// report.
template <template <int, int, int> class Kernel, class Args>
int run(const Plan& pl, int count, const char* what, Args&& args, Mail* m)
{
    if (!pl.ok) return tl_fail(TLHIP_ERR_ARG, "%s: the grid does not fit", what);
    if (count < 1) return tl_fail(TLHIP_ERR_ARG, "%s: no iteration to run", what);
    return with_plan(pl, [&](auto dims, auto kc, auto row) -> int {
        constexpr int D = decltype(dims)::value, K = decltype(kc)::value;
        constexpr int LXS = decltype(row)::value;
        const int nb = pl.blocks();
        if (pl.refuse || !room_for(nb)) return kRefused;
        TL_TRY(prepare(nb, 2 * (size_t)nb * faces_of<D, K>(LXS).total(), what));
        const size_t lds = lds_bytes<D, K>(LXS);
        const void* fn = Kernel<D, K, LXS>::fn();
        CHIP_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), what);
        auto a = args(geo_of(pl));
        arm_mail();
        void* ptrs[] = {&a};
        const int slot = tl_timer_begin(what);
        const hipError_t e = hipLaunchCooperativeKernel(fn, dim3(nb), dim3(kThreads), ptrs,
                                                        (unsigned)lds, tl_stream());
        if (e == hipErrorCooperativeLaunchTooLarge || e == hipErrorNotSupported ||
            e == hipErrorInvalidConfiguration || e == hipErrorLaunchOutOfResources) {
            (void)hipGetLastError();
            return kRefused;
        }
        CHIP_HIP(e, what);
        tl_timer_end(slot);
        g_chip.late = true;
        TL_TRY(wait_mail(m, what));
        g_chip.late = false;
        if (m->flags < 0.0)
            return tl_fail(TLHIP_ERR_HIP, "%s: a block waited over %.0f s for another", what, kWaitS);
        return 0;
    });
}

template <int D, int K, int L> struct Cg {
    static const void* fn() { return (const void*)k_chip_cg<D, K, L>; }
};
template <int D, int K, int L> struct Cheby {
    static const void* fn() { return (const void*)k_chip_cheby<D, K, L>; }
};
template <int D, int K, int L> struct Jacobi {
    static const void* fn() { return (const void*)k_chip_jacobi<D, K, L>; }
};

void outcome(const Mail& m, Outcome* out)
{
    out->rep.rrn = m.rrn;
    out->rep.err = m.err;
    out->rep.flags = (int)m.flags;
    out->last = (int)m.last;
    out->alpha = m.alpha;
    out->beta = m.beta;
}
}  // namespace

int cg(const Plan& pl, double* u, double* p, double* r, const double* kx, const double* ky,
       const double* kz, int it0, int count, const loop::StopRule& rule, Outcome* out)
{
    Mail m;
    double *alog, *blog;
    loop::log_ptrs(&alog, &blog);
    const int cnt = (int)std::min<long>(count, kChunk);
    TL_TRY((run<Cg>(pl, cnt, "tl_chip_cg", [&](const Geo& g) {
        return CgArgs{g, u, p, r, kx, ky, kz, g_chip.xbuf, g_chip.slots, alog, blog, g_chip.mail,
                      it0, cnt, rule};
    }, &m)));
    outcome(m, out);
    return 0;
}

int cheby(const Plan& pl, double* u, double* p, double* r, const double* u0, const double* kx,
          const double* ky, const double* kz, int it0, int count, int k0, int est,
          const double* alphas, const double* betas, double eps, bool sqrt_err, Outcome* out)
{
    const char* what = "tl_chip_cheby";
    Mail m;
    const int cnt = (int)std::min<long>(count, kChunk);
    TL_TRY(tl_ensure_init());
    Host& h = g_chip;
    if (!h.coefs) CHIP_HIP(hipMalloc(&h.coefs, sizeof(double) * 2 * kChunk), what);
    if (cnt > 0) {
        const size_t bytes = sizeof(double) * cnt;
        CHIP_HIP(hipMemcpyAsync(h.coefs, alphas, bytes, hipMemcpyHostToDevice, tl_stream()), what);
        CHIP_HIP(hipMemcpyAsync(h.coefs + kChunk, betas, bytes, hipMemcpyHostToDevice, tl_stream()),
                 what);
    }
    TL_TRY((run<Cheby>(pl, cnt, what, [&](const Geo& g) {
        return ChebyArgs{g, u, p, r, u0, kx, ky, kz, g_chip.xbuf, g_chip.slots, g_chip.rounds,
                         g_chip.mail, g_chip.coefs, g_chip.coefs + kChunk, it0, cnt, k0, est, eps,
                         (int)sqrt_err};
    }, &m)));
    outcome(m, out);
    return 0;
}

int jacobi(const Plan& pl, double* u, double* last_u, const double* u0, const double* kx,
           const double* ky, const double* kz, int it0, int count, const loop::StopRule& rule,
           Outcome* out)
{
    Mail m;
    const int cnt = (int)std::min<long>(count, kChunk);
    TL_TRY((run<Jacobi>(pl, cnt, "tl_chip_jacobi", [&](const Geo& g) {
        return JacobiArgs{g, u, last_u, u0, kx, ky, kz, g_chip.xbuf, g_chip.slots, g_chip.mail, it0,
                          cnt, rule};
    }, &m)));
    outcome(m, out);
    return 0;
}

void release()
{
    Host& h = g_chip;
    if (h.xbuf) (void)hipFree(h.xbuf);
    if (h.slots) (void)hipFree(h.slots);
    if (h.rounds) (void)hipFree(h.rounds);
    if (h.coefs) (void)hipFree(h.coefs);
    if (h.mail) (void)hipHostFree(h.mail);
    h = Host{};
}

}  // namespace chip
}  // namespace tl
