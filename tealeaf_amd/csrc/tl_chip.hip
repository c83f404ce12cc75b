// Whole solver loops in one launch with the fields in registers and LDS
// (tl_chip.h).
//
// A block of 1024 threads owns a tile of up to 8192 cells and at most one
// block runs per CU, so up to 2.1 million cells stay on the chip for the
// whole loop: r, A p and the coefficients of a thread's cells in registers,
// p (with a ring of the neighbours' cells) and kx in LDS.  u is read and
// written by its own thread only and stays in the CU's cache path.
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
// beta differs from the two-sum form by a few rounding errors; alpha and
// every vector update are the reference's expressions.  Where the residual
// falls so far in one iteration that the prediction cancels (below 1% of
// r.r: its error could pass 1e-13), the blocks meet again and sum the new
// r.r, as the two-sum form does.
//
// The same meeting hands the tile's outer cells of q to the neighbours: each
// block also keeps r and p of its ring and updates them with that q, so the
// ring's p equals the owner's bit for bit and no second meeting is needed.
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

struct Shared {
    double part[kWavesB][kSums];
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
    if ((lane & 15) == 0) sh.part[wave][lane >> 4] = c;
    double* next = slots + (size_t)((n + 1) % kPhases) * kMaxBlocks * kSums;
    double* mine = slots + (size_t)(n % kPhases) * kMaxBlocks * kSums;
    if (nb > 1 && tid < kSums)
        st_agent(&next[blockIdx.x * kSums + tid],
                 __builtin_bit_cast(double, (unsigned long long)TL_MAIL_EMPTY));
    wait_stores();
    __syncthreads();
    double t;
    if (nb == 1) {
        t = sum_groups(sh.part[lane >> 2][lane & 3]);
    } else {
        if (wave == 0) {
            const double s = sum_groups(sh.part[lane >> 2][lane & 3]);
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

__global__ void __launch_bounds__(256) k_empty(double* slots, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) slots[i] = __builtin_bit_cast(double, (unsigned long long)TL_MAIL_EMPTY);
}

// ------------------------------------------------------------ tile

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
        // (an address is formed when it is used, not once for all iterations:
        // 8 cells' addresses would take the registers of their fields)
        unsigned at0 = xmine;
        asm volatile("" : "+v"(at0));
        double* my = xb + at0;
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

    // q = A s of the thread's cells, s in LDS with its ring, and s.q added to
    // *dot; cells beyond a domain edge mirror the cell (a depth-1 reflective
    // halo).  The association is 2d/shared.h:50-54 / 3d/shared.h:52-58.
    // Cells outside the domain get 0.
    __device__ __forceinline__ void apply(const T& tl, const double* s,
                                          const double* s_k, double* dot, double q[K]) const
    {
        const double* p = s + tl.at;
        double below = p[-tl.KP], c = p[0];
        if (tl.first_k) below = c;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double above = p[(k + 1) * tl.KP];
            const double next = above;
            if (tl.last_k && k == tl.kn - 1) above = c;
            const double l = p[k * tl.KP + tl.lo], r = p[k * tl.KP + tl.hi];
            const double* sk = s_k + tl.k_at + k * tl.k_step;
            double a;
            if constexpr (DIMS == 2) {
                const double kxc = sk[0], kxr = sk[1];
                const double d = (1.0 + (kxr + kxc)) + (kk[k + 1] + kk[k]);
                a = d * c - (kxr * r + kxc * l) - (kk[k + 1] * above + kk[k] * below);
            } else {
                const double kyc = sk[0], kyu = sk[tl.k_next], kxc = kx[k];
                const double e = s_k[tl.e_at + k * tl.e_step];
                double kxr = tl_lane_next(kxc, e);
                if (tl.edge_x || tl.hi == 0) kxr = e;
                const double so = p[k * tl.KP + tl.ylo], no = p[k * tl.KP + tl.yhi];
                const double d = ((1.0 + (kxr + kxc)) + (kyu + kyc)) + (kk[k + 1] + kk[k]);
                a = d * c - (kxr * r + kxc * l) - (kyu * no + kyc * so)
                    - (kk[k + 1] * above + kk[k] * below);
            }
            q[k] = k < tl.kn ? a : 0.0;
            *dot += q[k] * c;
            below = c;
            c = next;
        }
    }
};

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
    if (threadIdx.x == 0) sh.expired = 0;
    constexpr int NE = decltype(tl)::NE;

    // p is zero outside the domain and in a ring without neighbours, where
    // the mirror is read instead
    for (int i = threadIdx.x; i < lds_p<DIMS, K>(LXS); i += kThreads) s_p[i] = 0.0;
    for (int i = threadIdx.x; i < lds_k<DIMS, K>(LXS); i += kThreads) s_k[i] = 0.0;
    __syncthreads();
    Coefs<DIMS, K, LXS> co;
    co.load(g, tl, s_k, A.kx, A.ky, A.kz);
    double r[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const bool in = k < tl.kn;
        const long c = tl.first + k * tl.kstep;
        r[k] = in ? A.r[c] : 0.0;
        if (in) s_p[tl.at + k * tl.KP] = A.p[c];
    }
    // the ring: r in registers, p in LDS
    double rr[NE], rz[2] = {0.0, 0.0};
    int rdst[NE];
    unsigned rsrc[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        unsigned src = 0;
        long cell = 0;
        bool in = false;
        int dst = 0;
        rr[i] = 0.0;
        rdst[i] = -1;
        rsrc[i] = 0;
        if (tl.ring(g, (int)threadIdx.x + i * kThreads, &dst, &src, &cell, &in) && in) {
            rr[i] = A.r[cell];
            s_p[dst] = A.p[cell];
            rdst[i] = dst;
            rsrc[i] = src;
        }
    }
    // the cells below and above this thread's (a tile with a neighbour above
    // is full along z)
    const bool zl = DIMS == 3 && tl.face_zl && tl.kn > 0, zh = DIMS == 3 && tl.face_zh && tl.kn > 0;
    if (zl) {
        rz[0] = A.r[tl.first - tl.kstep];
        s_p[tl.at - tl.KP] = A.p[tl.first - tl.kstep];
    }
    if (zh) {
        rz[1] = A.r[tl.first + K * tl.kstep];
        s_p[tl.at + K * tl.KP] = A.p[tl.first + K * tl.kstep];
    }
    __syncthreads();

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
        // with few cells per thread, u is on its way while the blocks meet
        constexpr bool kEarlyU = K <= 2;
        double u[kEarlyU ? K : 1];
        if constexpr (kEarlyU) {
#pragma unroll
            for (int k = 0; k < K; ++k)
                u[k] = go_on && k < tl.kn ? A.u[tl.first + k * tl.kstep] : 0.0;
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
        double qr[NE], qz[2] = {0.0, 0.0};
        if (nb > 1) {
#pragma unroll
            for (int i = 0; i < NE; ++i) qr[i] = rdst[i] >= 0 ? ld_agent(&xb[rsrc[i]]) : 0.0;
            if (zl) qz[0] = ld_agent(&xb[tl.zlow(g)]);
            if (zh) qz[1] = ld_agent(&xb[tl.zhigh(g)]);
        }
        unsigned cell0 = tl.first;
        asm volatile("" : "+v"(cell0));
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (k < tl.kn) {
                double* ug = A.u + cell0 + k * tl.kstep;
                double uk;
                if constexpr (kEarlyU) uk = u[k];
                else uk = *ug;
                uk += alpha * s_p[tl.at + k * tl.KP];
                r[k] -= alpha * q[k];
                *ug = uk;
            }
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
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                if (rdst[i] >= 0) {
                    rr[i] -= alpha * qr[i];
                    s_p[rdst[i]] = beta * s_p[rdst[i]] + rr[i];
                }
            }
            if (zl) {
                rz[0] -= alpha * qz[0];
                s_p[tl.at - tl.KP] = beta * s_p[tl.at - tl.KP] + rz[0];
            }
            if (zh) {
                rz[1] -= alpha * qz[1];
                s_p[tl.at + K * tl.KP] = beta * s_p[tl.at + K * tl.KP] + rz[1];
            }
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
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const double m[6] = {rrn, err, (double)flags, (double)(A.it0 + n - 1), alpha, beta_true};
        double* to = &A.mail->rrn;
#pragma unroll
        for (int i = 0; i < 6; ++i)
            __hip_atomic_store(to + i, m[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ------------------------------------------------------------ host

struct Host {
    double* xbuf = nullptr;
    size_t xlen = 0;
    double* slots = nullptr;
    Mail* mail = nullptr;
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
    if (!h.slots) {
        CHIP_HIP(hipMalloc(&h.slots, sizeof(double) * kPhases * kMaxBlocks * kSums), what);
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
    hipLaunchKernelGGL(k_empty, dim3((n + 255) / 256), dim3(256), 0, tl_stream(), h.slots, n);
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
    const int most = std::min(kMaxBlocks, compute_units());
    // One meeting costs what about eight more cells per thread do, so a grid
    // that fits one block runs in one; otherwise the fewest cells per thread.
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
            const double c = k + (p.blocks() > 1 ? 8.0 : 0.0) + p.blocks() * 1e-3;
            if (c < cost) {
                cost = c;
                best = p;
            }
        }
    }
    return best;
}

int cg(const Plan& pl, double* u, double* p, double* r, const double* kx, const double* ky,
       const double* kz, int it0, int count, const loop::StopRule& rule, Outcome* out)
{
    const char* what = "tl::chip::cg";
    if (!pl.ok) return tl_fail(TLHIP_ERR_ARG, "%s: the grid does not fit", what);
    if (count < 1) return tl_fail(TLHIP_ERR_ARG, "%s: no iteration to run", what);
    return with_plan(pl, [&](auto dims, auto kc, auto row) -> int {
        constexpr int D = decltype(dims)::value, K = decltype(kc)::value;
        constexpr int LXS = decltype(row)::value;
        const Geo g = geo_of(pl);
        const int nb = pl.blocks();
        TL_TRY(prepare(nb, 2 * (size_t)nb * faces_of<D, K>(pl.lxs).total(), what));
        const size_t lds = lds_bytes<D, K>(pl.lxs);
        const void* fn = (const void*)k_chip_cg<D, K, LXS>;
        CHIP_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), what);
        CgArgs a{g, u, p, r, kx, ky, kz, g_chip.xbuf, g_chip.slots, nullptr, nullptr, g_chip.mail,
                 it0, (int)std::min<long>(count, kChunk), rule};
        loop::log_ptrs(&a.alog, &a.blog);
        arm_mail();
        void* args[] = {&a};
        CHIP_HIP(hipLaunchCooperativeKernel(fn, dim3(nb), dim3(kThreads), args, (unsigned)lds,
                                            tl_stream()), what);
        Mail m;
        TL_TRY(wait_mail(&m, what));
        if (m.flags < 0.0)
            return tl_fail(TLHIP_ERR_HIP, "%s: a block waited over %.0f s for another", what, kWaitS);
        out->rep.rrn = m.rrn;
        out->rep.err = m.err;
        out->rep.flags = (int)m.flags;
        out->last = (int)m.last;
        out->alpha = m.alpha;
        out->beta = m.beta;
        return 0;
    });
}

void release()
{
    Host& h = g_chip;
    if (h.xbuf) (void)hipFree(h.xbuf);
    if (h.slots) (void)hipFree(h.slots);
    if (h.mail) (void)hipHostFree(h.mail);
    h = Host{};
}

}  // namespace chip
}  // namespace tl
