// Adjoint (reverse-time) kernels of the constant-density forward operator.
//
// The forward step n maps (u^{n-1}, u^n) to u^{n+1} (cd-3d wave.c:142-480):
//   interior p:  u^{n+1}_p = a_p u^n_p - b_p u^{n-1}_p + c_p (L u^n)_p
//   sources:     u^{n+1}_p += c_p kws_{s,p} w_s^{n-1}
//   boundaries:  per face line, Dirichlet zeroes and Neumann copies
// with den = 1 + e, a = 2/den, b = (1 - e)/den, c = q/den, q = dt^2 v^2,
// e = damp dt v^2 / 2, and receivers d^n = K u^n (wave.c:499-566).  These
// kernels apply the transpose of that linear map, step by step backwards,
// and accumulate the derivative of the data with respect to the velocity:
//   da/dv = db/dv = -4 e / (v den^2),  dc/dv = 2 q / (v den^2).
// L is the stencil sum over the axes of c2-weighted pairs divided by h^2;
// it is symmetric, so its transpose is the same stencil evaluated on a
// field that is zero outside the interior.
#pragma once
#include "sw_kernels.hpp"
#include "sw_step3d.hpp"

namespace sw {

// Point of this thread in a whole-grid launch (adj_grid): 64 threads along
// the contiguous axis, 4 lines per block.
constexpr int kAdjLines = 4;

__device__ __forceinline__ bool thread_point(const Params &P, int &i, int &j, int &k)
{
#if SW_DIM == 3
    i = blockIdx.z;
    j = blockIdx.y * kAdjLines + threadIdx.y;
    k = blockIdx.x * 64 + threadIdx.x;
    return j < P.nx && k < P.ny;
#else
    i = blockIdx.y * kAdjLines + threadIdx.y;
    j = blockIdx.x * 64 + threadIdx.x;
    k = 0;
    return i < P.nz && j < P.nx;
#endif
}

inline dim3 adj_grid(const Params &P)
{
#if SW_DIM == 3
    return dim3((unsigned)((P.ny + 63) / 64), (unsigned)((P.nx + kAdjLines - 1) / kAdjLines),
                (unsigned)P.nz);
#else
    return dim3((unsigned)((P.nx + 63) / 64), (unsigned)((P.nz + kAdjLines - 1) / kAdjLines), 1u);
#endif
}

inline dim3 adj_block() { return dim3(64u, (unsigned)kAdjLines, 1u); }

__device__ __forceinline__ bool interior(const Params &P, int i, int j, int k)
{
    const int r = P.r;
    bool in = i >= r && i < P.nz - r && j >= r && j < P.nx - r;
#if SW_DIM == 3
    in = in && k >= r && k < P.ny - r;
#else
    (void)k;
#endif
    return in;
}

// Whether interior point (i, j, k) lies on a Dirichlet plane of an axis
// (0 z, 1 x, 2 y; 2D: 0 z, 2 x) after `axis`.
__device__ __forceinline__ bool dirichlet_after(const Params &P, int i, int j, int k, int axis)
{
    const int r = P.r;
    bool d = axis < 0 && ((P.bc[0] == 1 && i == r) || (P.bc[1] == 1 && i == P.nz - r - 1));
#if SW_DIM == 3
    d = d || (axis < 1 && ((P.bc[2] == 1 && j == r) || (P.bc[3] == 1 && j == P.nx - r - 1)));
    d = d || (axis < 2 && ((P.bc[4] == 1 && k == r) || (P.bc[5] == 1 && k == P.ny - r - 1)));
#else
    (void)k;
    d = d || (axis < 2 && ((P.bc[2] == 1 && j == r) || (P.bc[3] == 1 && j == P.nx - r - 1)));
#endif
    return d;
}

// ubar += K^T res: each receiver spreads its residual over its box.
__global__ void __launch_bounds__(256)
k_adj_receivers(Params P, const Box *__restrict__ rbox, const real_t *__restrict__ rw,
                int nrec, const real_t *__restrict__ res, real_t *ubar)
{
    const int q = blockIdx.x;
    if (q >= nrec)
        return;
    const Box b = rbox[q];
    const real_t rv = res[q];
    if (rv == (real_t)0)
        return;
    const int cz = b.hi[0] - b.lo[0] + 1, cx = b.hi[1] - b.lo[1] + 1;
#if SW_DIM == 3
    const int cy = b.hi[2] - b.lo[2] + 1;
#else
    const int cy = 1;
#endif
    for (int t = threadIdx.x; t < cz * cx * cy; t += blockDim.x) {
        const int ii = t / (cx * cy), rem = t - ii * cx * cy;
        const int jj = rem / cy, kk = rem - jj * cy;
        const int i = b.lo[0] + ii, j = b.lo[1] + jj;
#if SW_DIM == 3
        const int k = b.lo[2] + kk;
#else
        const int k = 0;
        (void)kk;
#endif
        const long long p = (long long)i * P.sz + (long long)j * P.sx + k;
        atomicAdd(&ubar[p], box_weight(b, rw, i, j, k) * rv);
    }
}

// grad += gacc and gacc = 0 where gacc holds anything: the float64
// gradient takes the working-precision sums of the last few reverse steps
// (the update kernels add each step's term to gacc, which halves their
// gradient traffic in float32).
__global__ void __launch_bounds__(256)
k_grad_flush(real_t *__restrict__ gacc, double *__restrict__ grad, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const real_t g = gacc[i];
        if (g != (real_t)0) {
            grad[i] += (double)g;
            gacc[i] = (real_t)0;
        }
    }
}

// The same spread as a gather, with no atomics and a fixed order.  Built
// once per gradient: every (point, receiver) pair of the receiver boxes as
// an entry, sorted by point (a stable sort of entries made in receiver
// order), so each touched point sums its receivers' terms in ascending
// receiver order, as the receiver loop of the transposed step does.

// Entry off[q] + t is point t of receiver q's box: its linear point index
// (sort key) and its own position (sort value).
__global__ void __launch_bounds__(256)
k_adj_rec_entries(Params P, const Box *__restrict__ rbox, int nrec,
                  const unsigned *__restrict__ off, unsigned *__restrict__ key,
                  unsigned *__restrict__ idx)
{
    const int q = blockIdx.x;
    if (q >= nrec)
        return;
    const Box b = rbox[q];
    const int cz = b.hi[0] - b.lo[0] + 1, cx = b.hi[1] - b.lo[1] + 1;
#if SW_DIM == 3
    const int cy = b.hi[2] - b.lo[2] + 1;
#else
    const int cy = 1;
#endif
    const unsigned base = off[q];
    for (int t = threadIdx.x; t < cz * cx * cy; t += blockDim.x) {
        const int ii = t / (cx * cy), rem = t - ii * cx * cy;
        const int jj = rem / cy, kk = rem - jj * cy;
#if SW_DIM == 3
        const long long p = (long long)(b.lo[0] + ii) * P.sz +
                            (long long)(b.lo[1] + jj) * P.sx + (b.lo[2] + kk);
#else
        (void)kk;
        const long long p = (long long)(b.lo[0] + ii) * P.sz + (b.lo[1] + jj);
#endif
        key[base + t] = (unsigned)p;
        idx[base + t] = base + t;
    }
}

// Sorted entry s (point key[s], original entry idx[s]): its receiver (the q
// with off[q] <= idx[s] < off[q+1]) and weight.
__global__ void __launch_bounds__(256)
k_adj_rec_permute(Params P, const Box *__restrict__ rbox, const real_t *__restrict__ rw,
                  int nrec, const unsigned *__restrict__ off,
                  const unsigned *__restrict__ key, const unsigned *__restrict__ idx,
                  unsigned n, unsigned *__restrict__ qs, real_t *__restrict__ ws)
{
    const unsigned s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n)
        return;
    const unsigned e = idx[s];
    int lo = 0, hi = nrec;                 // off[lo] <= e < off[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (off[mid] <= e)
            lo = mid;
        else
            hi = mid;
    }
    const long long p = key[s];
#if SW_DIM == 3
    const int i = (int)(p / P.sz);
    const long long rem = p - (long long)i * P.sz;
    const int j = (int)(rem / P.sx), k = (int)(rem - (long long)j * P.sx);
#else
    const int i = (int)(p / P.sz), j = (int)(p - (long long)i * P.sz), k = 0;
#endif
    qs[s] = (unsigned)lo;
    ws[s] = box_weight(rbox[lo], rw, i, j, k);
}

// Per reverse step: each touched point adds its receivers' terms in
// receiver order (receivers whose residual is zero add nothing, as in
// k_adj_receivers), is zeroed on a Dirichlet plane, and W follows it.
__global__ void __launch_bounds__(256)
k_adj_rec_gather(Params P, const real_t *__restrict__ C, const unsigned *__restrict__ pts,
                 const unsigned *__restrict__ start, const unsigned *__restrict__ cnt, int nu,
                 const unsigned *__restrict__ qs, const real_t *__restrict__ ws,
                 const real_t *__restrict__ res, real_t *__restrict__ ubar,
                 real_t *__restrict__ W)
{
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= nu)
        return;
    const unsigned p = pts[u];
    real_t acc = ubar[p];
    unsigned s = start[u];
    const unsigned s1 = s + cnt[u];
    // four entries' loads in flight, then their terms in order
    for (; s + 4 <= s1; s += 4) {
        real_t w[4], rv[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            w[t] = ws[s + t];
            rv[t] = res[qs[s + t]];
        }
#pragma unroll
        for (int t = 0; t < 4; t++)
            if (rv[t] != (real_t)0)
                acc += w[t] * rv[t];
    }
    for (; s < s1; s++) {
        const real_t rv = res[qs[s]];
        if (rv != (real_t)0)
            acc += ws[s] * rv;
    }
    const unsigned sz = (unsigned)P.sz, i = p / sz, rem = p - i * sz;
#if SW_DIM == 3
    const unsigned sx = (unsigned)P.sx, j = rem / sx, k = rem - j * sx;
#else
    const unsigned j = rem, k = 0;
#endif
    if (interior(P, i, j, k)) {
        if (dirichlet_after(P, i, j, k, -1))
            acc = 0;
        W[p] = C[p] * acc;
    }
    ubar[p] = acc;
}

// Transpose of one boundary phase (k_bc_phase) on an axis with a Neumann
// face: per face line, the after face's Neumann copies, then its Dirichlet
// zero, then the same for the before face.  Axes without a Neumann face need
// no launch: whatever writes an interior point zeroes it on a Dirichlet
// plane, and a point this phase adds to is zeroed again where a later axis'
// phase does.  The halo values it adds (k_adj_update's) are left as they are:
// the step that next uses their buffer writes them before they are read.
// W = C ub follows the points that change.
__global__ void k_adj_bc_phase(Params P, const real_t *__restrict__ C, real_t *ub,
                               real_t *__restrict__ W, int axis)
{
    const int r = P.r;
    const long long li = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    long long base, st;
    int n, before, after, i = 0, j = 0, k = 0;
#if SW_DIM == 3
    const long long Iy = P.ny - 2 * r, Ix = P.nx - 2 * r, Iz = P.nz - 2 * r;
    if (axis == 2) {
        if (li >= Iz * Ix) return;
        j = r + (int)(li % Ix), i = r + (int)(li / Ix);
        base = (long long)i * P.sz + (long long)j * P.sx; st = 1; n = P.ny;
        before = P.bc[4]; after = P.bc[5];
    } else if (axis == 1) {
        if (li >= Iz * Iy) return;
        k = r + (int)(li % Iy), i = r + (int)(li / Iy);
        base = (long long)i * P.sz + k; st = P.sx; n = P.nx;
        before = P.bc[2]; after = P.bc[3];
    } else {
        if (li >= Ix * Iy) return;
        k = r + (int)(li % Iy), j = r + (int)(li / Iy);
        base = (long long)j * P.sx + k; st = P.sz; n = P.nz;
        before = P.bc[0]; after = P.bc[1];
    }
#else
    const long long Ix = P.nx - 2 * r, Iz = P.nz - 2 * r;
    if (axis == 2) {
        if (li >= Iz) return;
        i = r + (int)li;
        base = (long long)i * P.sz; st = 1; n = P.nx;
        before = P.bc[2]; after = P.bc[3];
    } else {
        if (li >= Ix) return;
        j = r + (int)li;
        base = j; st = P.sz; n = P.nz;
        before = P.bc[0]; after = P.bc[1];
    }
#endif
    const long long lo = base + (long long)r * st;
    const long long hi = base + (long long)(n - r - 1) * st;
    auto put = [&](long long p, real_t v) {
        ub[p] = v;
        W[p] = C[p] * v;
    };
    // the line's transverse position decides the later axes' zeros
    const bool zero = dirichlet_after(P, i, j, k, axis);
    if (after == 2)
        for (int m = 1; m <= r; m++)
            put(hi - m * st, zero ? (real_t)0 : ub[hi - m * st] + ub[hi + m * st]);
    if (after == 1)
        put(hi, 0);
    if (before == 2)
        for (int m = 1; m <= r; m++)
            put(lo + m * st, zero ? (real_t)0 : ub[lo + m * st] + ub[lo - m * st]);
    if (before == 1)
        put(lo, 0);
}

// Dirichlet zeros and W = c * ubar on the interior, after the atomic spread
// (k_adj_receivers).
__global__ void __launch_bounds__(64 * kAdjLines)
k_adj_cw(Params P, const real_t *__restrict__ C, real_t *__restrict__ ub, real_t *__restrict__ W)
{
    int i, j, k;
    if (!thread_point(P, i, j, k) || !interior(P, i, j, k))
        return;
    const long long p = (long long)i * P.sz + (long long)j * P.sx + k;
    real_t v = ub[p];
    if (dirichlet_after(P, i, j, k, -1))
        ub[p] = v = 0;
    W[p] = C[p] * v;
}

// The transpose of the interior update of step n and the velocity derivative,
// as a two-level recurrence of the adjoint levels l^k (k = n+1, W = c l^k):
//   l^{k-1} = a l^k - b l^{k+1} + L^T W,  W' = c l^{k-1},
//   grad += l^k (da (u^n - u^{n-1}) + dc (L u^n + s))
// where s is the source term of the step.  c (L u^n + s) is what the step
// added to a u^n - b u^{n-1}, so (L u^n + s) = (u^{n+1} - a u^n + b u^{n-1}) / c
// and dc / c = 2 / (v den): no second stencil is needed.  In image mode grad
// collects the zero-lag cross-correlation l^k u^{n+1} instead.
//
// l^{k-1} takes the buffer of l^{k+1} and forms -b l^{k+1} when it needs it,
// and W' is written here (the receiver and boundary kernels keep it in step),
// so a point's step moves l^k, l^{k+1}, W, c in and l^{k-1}, W' out; writing
// -b l^k ahead and forming W in a pass of its own moved nine values.  The
// gradient of two steps is added at once, when both l^k and l^{k+1} are here:
// four forward levels, v and the sums for two steps instead of for one each
// (mode 2; mode 0 leaves its step's term to the next launch, mode 1 adds its
// own alone).  The sums keep their order.
//
// Outside the interior W is zero.  The adjoint of the halo is non-zero on
// the Neumann faces' mirror points only (k_adj_bc_phase reads no others):
// blocks behind the interior's compute them from W's line (adj_halo_lines).
struct AdjArgs {
    const real_t *vel, *C;
    const real_t *l, *W;        // l^k, c l^k
    real_t *lp, *Wn;            // in l^{k+1}, out l^{k-1}; out c l^{k-1}
    const real_t *u[4];         // u^{n+2} (mode 2), u^{n+1}, u^n, u^{n-1}
    real_t *gacc;
    int image;
};

__device__ __forceinline__ real_t adj_level(double a, double b, real_t l, real_t lp, real_t lt)
{
    const real_t b1 = (real_t)(-b * (double)lp);
    return (real_t)((double)b1 + a * (double)l + (double)lt);
}

// One step's gradient term; tr = 2 / (v den).
__device__ __forceinline__ real_t adj_grad(double a, double b, double da, double tr, real_t g,
                                           real_t l, real_t u0, real_t u1, real_t u2)
{
    const double x0 = (double)u0, x1 = (double)u1, x2 = (double)u2;
    const double step = x0 - a * x1 + b * x2;     // c (L u^n + s)
    const real_t t = (real_t)((double)l * (da * (x1 - x2) + tr * step));
    return l != (real_t)0 ? g + t : g;
}

__device__ __forceinline__ real_t adj_image(real_t g, real_t l, real_t u0)
{
    return l != (real_t)0 ? g + (real_t)((double)l * (double)u0) : g;
}

// a, b, da of a point with damping e, and tr from rv = 1 / v.
struct AdjCoef {
    double a, b, da, tr;
};

__device__ __forceinline__ AdjCoef adj_coef(double e, double rv)
{
    const double rden = 1.0 / (1.0 + e);
    return {2.0 * rden, (1.0 - e) * rden, -4.0 * e * rden * rden * rv, 2.0 * rden * rv};
}

// The update of one point from its operands; returns l^{k-1}.
template <int GM>
__device__ __forceinline__ real_t adj_point(const AdjArgs &A, double e, double rv, real_t l,
                                            real_t lp, real_t lt, const real_t (&u)[4], real_t &g)
{
    const AdjCoef c = adj_coef(e, rv);
    if constexpr (GM != 0) {
        if (A.image) {
            if (GM == 2)
                g = adj_image(g, lp, u[0]);
            g = adj_image(g, l, u[1]);
        } else {
            if (GM == 2)
                g = adj_grad(c.a, c.b, c.da, c.tr, g, lp, u[0], u[1], u[2]);
            g = adj_grad(c.a, c.b, c.da, c.tr, g, l, u[1], u[2], u[3]);
        }
    }
    return adj_level(c.a, c.b, l, lp, lt);
}

// Adjoint of the mirror points of Neumann-face line `li` (lines of all
// Neumann faces in face order): the stencil of W there has the face's axis
// alone, W being zero beside the line.
template <int R>
__device__ __forceinline__ void adj_halo_line(const Params &P, const AdjArgs &A, long long li)
{
    const long long Ix = P.nx - 2 * R, Iz = P.nz - 2 * R;
#if SW_DIM == 3
    const long long Iy = P.ny - 2 * R;
    const long long lines[3] = {Ix * Iy, Iz * Iy, Iz * Ix};
#else
    const long long lines[2] = {Ix, Iz};
#endif
#pragma unroll
    for (int f = 0; f < 2 * SW_DIM; f++) {
        if (P.bc[f] != 2)
            continue;
        if (li >= lines[f / 2]) {
            li -= lines[f / 2];
            continue;
        }
        long long p, st;        // the face's interior plane, the step inwards
        real_t h2;
#if SW_DIM == 3
        if (f / 2 == 0) {
            p = (long long)(f == 0 ? R : P.nz - R - 1) * P.sz + (R + li / Iy) * P.sx + R + li % Iy;
            st = P.sz;
            h2 = P.dz2;
        } else if (f / 2 == 1) {
            p = (R + li / Iy) * P.sz + (long long)(f == 2 ? R : P.nx - R - 1) * P.sx + R + li % Iy;
            st = P.sx;
            h2 = P.dx2;
        } else {
            p = (R + li / Ix) * P.sz + (R + li % Ix) * P.sx + (f == 4 ? R : P.ny - R - 1);
            st = 1;
            h2 = P.dy2;
        }
#else
        if (f / 2 == 0) {
            p = (long long)(f == 0 ? R : P.nz - R - 1) * P.sz + R + li;
            st = P.sz;
            h2 = P.dz2;
        } else {
            p = (R + li) * P.sz + (f == 2 ? R : P.nx - R - 1);
            st = 1;
            h2 = P.dx2;
        }
#endif
        if (f & 1)
            st = -st;
        real_t w[R];
#pragma unroll
        for (int m = 0; m < R; m++)
            w[m] = A.W[p + m * st];
#pragma unroll
        for (int m = 1; m <= R; m++) {
            real_t s = 0;
#pragma unroll
            for (int d = m; d <= R; d++)
                s += P.c2[d] * w[d - m];
            A.lp[p - m * st] = s / h2;
        }
        return;
    }
}

#if SW_DIM == 3
// The update marching z with 16-byte lanes: k_step3d_vec's tile (one row per
// lane, 2R+1 z planes of W in registers, the plane's x and y neighbours in
// LDS, operands of the next plane loaded behind the stores), over the
// interior.  One point per thread with neighbours through the caches issued
// 27 loads per point and was bound by the load path: 288 us at 220 x 316 x
// 316 so8, besides 71 us for W's own pass.  Here 4 points share a load: 220 us
// for both, 0.87 GB at 4.0 TB/s (a large copy reaches 4.6).  One wavefront per
// block: 4 rows by 64 (float64 32) points; two or four wavefronts per tile take
// as long on large grids and longer on small ones (120 x 180 x 200 so2 81 / 84
// / 83 us, 50 x 70 x 70 so8 14.5 / 16.7 / 18.1).
constexpr int kAdjRows = 4;

template <int R, int GM>
__global__ void __launch_bounds__(64)
k_adj_update_tiled(Params P, LapDiv D, AdjArgs A, Tiling T, int tiled_blocks)
{
    constexpr int WR = kAdjRows, NW = 1;
    using S = TileShape<R, WR, 1, NW, kVec16>;
    typedef typename LaneVec<kVec16>::type vreal;
    constexpr int V = S::V, LW = S::LW, TY = S::TY, TXR = S::TXR, PADL = S::PADL;
    constexpr int HV = S::HV, LS = S::LS, H = S::H, SLOTS = S::SLOTS, HX = S::HX;
    constexpr int NYV = S::NYV, HY = S::HY, NT = 64 * NW;
    constexpr int NU = GM == 2 ? 4 : 3;      // forward levels read (image: fewer)
    constexpr unsigned esz = sizeof(real_t);
    constexpr int DUMP = H * LS, PLANE = H * LS + NT * V;
    __shared__ __align__(16) real_t lds[2 * PLANE];

    const int lane = threadIdx.x, tid = lane;
    const int bid = blockIdx.x;
    if (bid >= tiled_blocks) {
        adj_halo_line<R>(P, A, (long long)(bid - tiled_blocks) * NT + tid);
        return;
    }
    const int slot = lane / LW, lc = lane % LW;
    const int nx = P.nx, ny = P.ny, nz = P.nz;
    const unsigned PB = (unsigned)P.sz * esz;
    // columns in 8 contiguous chunks, one per XCD
    const int xcd = bid & 7, s = bid >> 3;
    const int zc = s / T.chunk, col = xcd * T.chunk + s % T.chunk;
    if (col >= T.ncols)
        return;
    const int k0 = R + col % T.gk * TY, j0 = R + col / T.gk * TXR;
    const int z0 = R + zc * T.zlen, z1 = min(z0 + T.zlen, nz - R);
    const int zb = z0 - R;

    // descriptors over the planes zb .. z1+R-1 (below 2^31 bytes, checked by
    // the host); kOOB is out of range for all of them
    const unsigned long long off0 = (unsigned long long)zb * (unsigned long long)P.sz;
    const unsigned rem = (unsigned)(z1 + R - zb) * PB;
    const rsrc_t r_W = make_rsrc(A.W + off0, rem), r_Wn = make_rsrc(A.Wn + off0, rem);
    const rsrc_t r_l = make_rsrc(A.l + off0, rem), r_lp = make_rsrc(A.lp + off0, rem);
    const rsrc_t r_C = make_rsrc(A.C + off0, rem), r_e = make_rsrc(P.e + off0, rem);
    const rsrc_t r_v = make_rsrc(A.vel + off0, rem), r_g = make_rsrc(A.gacc + off0, rem);
    rsrc_t r_u[4];
#pragma unroll
    for (int t = 0; t < 4; t++)
        r_u[t] = make_rsrc((t >= 4 - NU ? A.u[t] : A.u[3]) + off0, rem);

    const int j = j0 + slot, k = k0 + lc * V;
    const int kl = k < ny ? k : 0;
    const bool act = j < nx - R && k < ny - R;
    const bool full = act && k + V <= ny - R;
    const unsigned cb = ((unsigned)min(j, nx - 1) * (unsigned)ny + (unsigned)kl) * esz;
    const unsigned ob = act ? cb : kOOB;          // operands
    const unsigned sb = full ? cb : kOOB;         // whole-vector stores
    const bool ragged = (ny - 2 * R) % V != 0 && k0 + TY > ny - R;   // tile-uniform
    unsigned xh_off[HX];
    int xh_lds[HX];
#pragma unroll
    for (int h = 0; h < HX; h++) {
        const int hr = slot + SLOTS * h;
        const int jr = hr < R ? j0 - R + hr : j0 + TXR + (hr - R);
        xh_off[h] = ((unsigned)min(jr, nx - 1) * (unsigned)ny + (unsigned)kl) * esz;
        const int xr = hr < 2 * R ? (hr < R ? hr : hr + TXR) : -1;
        xh_lds[h] = xr >= 0 ? xr * LS + PADL + lc * V : DUMP + tid * V;
    }
    unsigned yh_off[HY];
    int yh_lds[HY];
#pragma unroll
    for (int h = 0; h < HY; h++) {
        const int idx = tid + NT * h;
        const int row = idx / (2 * HV), c = idx % (2 * HV);
        const int jl = min(j0 + row, nx - 1);
        int kr = c < HV ? k0 - PADL + V * c : k0 + TY + V * (c - HV);
        kr = kr < ny ? kr : 0;
        // kr > -V and jl >= R >= 1 with ny >= V, so the offset is not negative
        yh_off[h] = (unsigned)((int)((unsigned)jl * (unsigned)ny) + kr) * esz;
        yh_lds[h] = idx < NYV ? (R + row) * LS + (c < HV ? V * c : PADL + TY + V * (c - HV))
                              : DUMP + tid * V;
    }
    // Dirichlet planes: z tile-uniform, x by the lane's row, y by the element
    const int zpb = P.bc[0] == 1 ? R : -1, zpa = P.bc[1] == 1 ? nz - R - 1 : -1;
    const bool drow = (P.bc[2] == 1 && j == R) || (P.bc[3] == 1 && j == nx - R - 1);
    const int yb = P.bc[4] == 1 ? R - k : -1, ya = P.bc[5] == 1 ? ny - R - 1 - k : -1;
    const bool dxy = (P.bc[2] == 1 && j0 == R) || (P.bc[3] == 1 && j0 + TXR > nx - R - 1) ||
                     (P.bc[4] == 1 && k0 == R) || (P.bc[5] == 1 && k0 + TY > ny - R - 1);
    const unsigned long long dbits = damp_bits(T, col, z0);

    vreal qz[2 * R + 1];
#pragma unroll
    for (int m = 0; m < 2 * R; m++)
        qz[m + 1] = vload<V>(r_W, cb + (unsigned)m * PB, 0u);
    vreal nc, nhx[HX], nhy[HY];
    vreal nl, np, nC, ne, nv, ng, nu[4];
    auto load_centre = [&](int I) {
        const bool live = I < z1;
        const unsigned sp = live ? (unsigned)(I - zb) * PB : 0u;
        const unsigned vc = (unsigned)(I + R - zb) * PB;
        nc = vload<V>(r_W, live ? cb + vc : kOOB, 0u);
#pragma unroll
        for (int h = 0; h < HX; h++)
            nhx[h] = vload<V>(r_W, live ? xh_off[h] : kOOB, sp);
#pragma unroll
        for (int h = 0; h < HY; h++)
            nhy[h] = vload<V>(r_W, live ? yh_off[h] : kOOB, sp);
    };
    auto load_update = [&](int I) {
        const bool live = I < z1;
        const unsigned sp = live ? (unsigned)(I - zb) * PB : 0u, o = live ? ob : kOOB;
        nl = vload<V>(r_l, o, sp);
        np = vload<V>(r_lp, o, sp);
        nC = vload<V>(r_C, o, sp);
        ne = vload<V>(r_e, live && ((dbits >> (I - z0)) & 1) ? o : kOOB, sp);
        if constexpr (GM != 0) {
            nv = vload<V>(r_v, o, sp);
            ng = vload<V>(r_g, o, sp);
#pragma unroll
            for (int t = 4 - NU; t < 4; t++)
                nu[t] = vload<V>(r_u[t], o, sp);
        }
    };
    load_centre(z0);
    __builtin_amdgcn_sched_barrier(0);
    load_update(z0);
    __builtin_amdgcn_sched_barrier(0);

    for (int i = z0; i < z1; i++) {
        real_t *lb = lds + ((i - z0) & 1) * PLANE;
#pragma unroll
        for (int m = 0; m < 2 * R; m++)
            qz[m] = qz[m + 1];
        qz[2 * R] = nc;
        *(vreal *)&lb[(R + slot) * LS + PADL + lc * V] = qz[R];
#pragma unroll
        for (int h = 0; h < HX; h++)
            *(vreal *)&lb[xh_lds[h]] = nhx[h];
#pragma unroll
        for (int h = 0; h < HY; h++)
            *(vreal *)&lb[yh_lds[h]] = nhy[h];
        load_centre(i + 1);
        __syncthreads();

        const real_t *lrow0 = lb + (R + slot) * LS + lc * V + PADL;
        real_t win[V + 2 * PADL];
#pragma unroll
        for (int h = 0; h < HV; h++) {
            const vreal a = *(const vreal *)&lrow0[V * h - PADL];
            const vreal b = *(const vreal *)&lrow0[V + V * h];
#pragma unroll
            for (int x = 0; x < V; x++) {
                win[V * h + x] = a[x];
                win[PADL + V + V * h + x] = b[x];
            }
        }
        real_t ay[V], ax[V], az[V], lap[V];
#pragma unroll
        for (int x = 0; x < V; x++) {
            win[PADL + x] = qz[R][x];
            ay[x] = ax[x] = az[x] = P.c2[0] * qz[R][x];
        }
#pragma unroll
        for (int m = 1; m <= R; m++) {
            const vreal xp = *(const vreal *)&lrow0[m * LS];
            const vreal xm = *(const vreal *)&lrow0[-m * LS];
#pragma unroll
            for (int x = 0; x < V; x++) {
                ay[x] += P.c2[m] * (win[PADL + x + m] + win[PADL + x - m]);
                ax[x] += P.c2[m] * (xp[x] + xm[x]);
                az[x] += P.c2[m] * (qz[R + m][x] + qz[R - m][x]);
            }
        }
#pragma unroll
        for (int x = 0; x < V; x++)
            lap[x] = lap_quotients(P, D, ay[x], ax[x], az[x]);
        // the operands are first touched here, behind the stencil
        __builtin_amdgcn_sched_barrier(0);
        double rv[V];
        if constexpr (GM != 0) {
#if defined(SW_DOUBLE)
#pragma unroll
            for (int x = 0; x < V; x++)
                rv[x] = 1.0 / nv[x];
#else
            bool in_range = true;
#pragma unroll
            for (int x = 0; x < V; x++)
                in_range &= fabsf(nv[x]) >= 0x1p-60f && fabsf(nv[x]) <= 0x1p60f;
            if (__all(in_range)) {
#pragma unroll
                for (int x = 0; x < V; x++)
                    rv[x] = recip_f64(nv[x]);
            } else {
#pragma unroll
                for (int x = 0; x < V; x++)
                    rv[x] = 1.0 / (double)nv[x];
            }
#endif
        }
        vreal out;
        // e = 0 folds to a = 2, b = 1
        auto update = [&](auto damped) {
#pragma unroll
            for (int x = 0; x < V; x++) {
                const real_t u[4] = {GM == 2 ? nu[0][x] : (real_t)0, nu[1][x], nu[2][x], nu[3][x]};
                real_t g = GM != 0 ? ng[x] : (real_t)0;
                out[x] = adj_point<GM>(A, decltype(damped)::value ? (double)ne[x] : 0.0,
                                       GM != 0 ? rv[x] : 0.0, nl[x], np[x], lap[x], u, g);
                if (GM != 0)
                    ng[x] = g;
            }
        };
        if ((dbits >> (i - z0)) & 1)
            update(std::true_type{});
        else
            update(std::false_type{});
        if (dxy || i == zpb || i == zpa) {
#pragma unroll
            for (int x = 0; x < V; x++)
                if (i == zpb || i == zpa || drow || x == yb || x == ya)
                    out[x] = 0;
        }
        const unsigned so = (unsigned)(i - zb) * PB;
        const vreal wn = nC * out;
        vstore(out, r_lp, sb, so);
        vstore(wn, r_Wn, sb, so);
        if constexpr (GM != 0)
            vstore(ng, r_g, sb, so);
        if (ragged && act && !full) {
#pragma unroll
            for (int x = 0; x < V; x++) {
                if (k + x < ny - R) {
                    sstore(out[x], r_lp, cb + x * esz, so);
                    sstore(wn[x], r_Wn, cb + x * esz, so);
                    if constexpr (GM != 0)
                        sstore(ng[x], r_g, cb + x * esz, so);
                }
            }
        }
        load_update(i + 1);
    }
}
#endif

// One point per thread, 64-bit addresses.  3D: grids whose planes exceed the
// tiled kernel's 32-bit offsets, whole grid in one launch.  2D: each thread
// owns an x column of a chunk of `zlen` rows; W's z neighbours sit in a
// register queue and the next row's operands are loaded while the current one
// is computed.
#if SW_DIM == 3
template <int R>
__global__ void __launch_bounds__(256)
k_adj_halo(Params P, AdjArgs A)
{
    adj_halo_line<R>(P, A, (long long)blockIdx.x * 256 + threadIdx.x);
}

template <int R, int GM>
__global__ void __launch_bounds__(64 * kAdjLines)
k_adj_update(Params P, AdjArgs A)
{
    int i, j, k;
    if (!thread_point(P, i, j, k) || !interior(P, i, j, k))
        return;
    const long long p = (long long)i * P.sz + (long long)j * P.sx + k;
    const real_t c0 = A.W[p] * P.c2[0];
    real_t sz = c0, sx = c0, sy = c0;
#pragma unroll
    for (int m = 1; m <= R; m++) {
        sz += P.c2[m] * (A.W[p + m * P.sz] + A.W[p - m * P.sz]);
        sx += P.c2[m] * (A.W[p + m * P.sx] + A.W[p - m * P.sx]);
        sy += P.c2[m] * (A.W[p + m] + A.W[p - m]);
    }
    const real_t lt = sy / P.dy2 + sx / P.dx2 + sz / P.dz2;
    real_t u[4] = {0, 0, 0, 0}, g = 0;
    double rv = 0;
    if constexpr (GM != 0) {
        rv = 1.0 / (double)A.vel[p];
        g = A.gacc[p];
        for (int t = GM == 2 ? 0 : 1; t < 4; t++)
            u[t] = A.u[t][p];
    }
    real_t v = adj_point<GM>(A, (double)P.e[p], rv, A.l[p], A.lp[p], lt, u, g);
    if (dirichlet_after(P, i, j, k, -1))
        v = 0;
    A.lp[p] = v;
    A.Wn[p] = A.C[p] * v;
    if (GM != 0)
        A.gacc[p] = g;
}
#else
template <int R, int GM>
__global__ void __launch_bounds__(256)
k_adj_update_z2d(Params P, AdjArgs A, int zlen, int gx, int step_blocks)
{
    if ((int)blockIdx.x >= step_blocks) {
        adj_halo_line<R>(P, A, (long long)(blockIdx.x - step_blocks) * 256 + threadIdx.x);
        return;
    }
    const int j = R + (int)blockIdx.x % gx * 256 + (int)threadIdx.x;
    if (j >= P.nx - R)
        return;
    const int z0 = R + (int)blockIdx.x / gx * zlen;
    const int z1 = min(z0 + zlen, P.nz - R);
    const real_t *__restrict__ W = A.W;
    real_t wq[2 * R + 1];
#pragma unroll
    for (int d = 0; d < 2 * R; d++)
        wq[d + 1] = W[(long long)(z0 + d - R) * P.sz + j];
    struct Ops {
        real_t head, l, lp, c, e, v, g, u[4], xn[2 * R];
    };
    auto load = [&](int i, Ops &o) {
        const long long p = (long long)i * P.sz + j;
        o.head = W[p + R * P.sz];
#pragma unroll
        for (int m = 1; m <= R; m++) {
            o.xn[2 * m - 2] = W[p + m];
            o.xn[2 * m - 1] = W[p - m];
        }
        o.l = A.l[p];
        o.lp = A.lp[p];
        o.c = A.C[p];
        o.e = P.e[p];
        if constexpr (GM != 0) {
            o.v = A.vel[p];
            o.g = A.gacc[p];
#pragma unroll
            for (int t = GM == 2 ? 0 : 1; t < 4; t++)
                o.u[t] = A.u[t][p];
        }
    };
    const bool drow = (P.bc[2] == 1 && j == R) || (P.bc[3] == 1 && j == P.nx - R - 1);
    Ops cur, nxt;
    load(z0, cur);
    for (int i = z0; i < z1; i++) {
        if (i + 1 < z1)
            load(i + 1, nxt);
#pragma unroll
        for (int d = 0; d < 2 * R; d++)
            wq[d] = wq[d + 1];
        wq[2 * R] = cur.head;
        const real_t c0 = wq[R] * P.c2[0];
        real_t sz = c0, sx = c0;
#pragma unroll
        for (int m = 1; m <= R; m++) {
            sz += P.c2[m] * (wq[R + m] + wq[R - m]);
            sx += P.c2[m] * (cur.xn[2 * m - 2] + cur.xn[2 * m - 1]);
        }
        const real_t lt = sx / P.dx2 + sz / P.dz2;
        const real_t u[4] = {GM == 2 ? cur.u[0] : (real_t)0, GM ? cur.u[1] : (real_t)0,
                             GM ? cur.u[2] : (real_t)0, GM ? cur.u[3] : (real_t)0};
        real_t g = GM != 0 ? cur.g : (real_t)0;
        real_t v = adj_point<GM>(A, (double)cur.e, GM != 0 ? 1.0 / (double)cur.v : 0.0, cur.l,
                                 cur.lp, lt, u, g);
        if (drow || (P.bc[0] == 1 && i == R) || (P.bc[1] == 1 && i == P.nz - R - 1))
            v = 0;
        const long long p = (long long)i * P.sz + j;
        A.lp[p] = v;
        A.Wn[p] = cur.c * v;
        if (GM != 0)
            A.gacc[p] = g;
        cur = nxt;
    }
}
#endif

// Velocity derivative of step n on a Dirichlet plane (`face`) whose points have
// an adjoint: an earlier boundary phase mirrors the plane before its own zeroes
// it, and a receiver box holds the mirrored values.  The levels are zero there,
// so the update's step difference adds nothing; what the step added before the
// zero is formed here, l^k dc (L u^n + s).  Rare and small (one plane, few
// points with l != 0): a launch of its own, one thread per point.  planes: all
// faces so treated; a point on several is the first one's.
__global__ void __launch_bounds__(256)
k_adj_zeroed_plane(Params P, const real_t *__restrict__ vel, const real_t *__restrict__ l,
                   const real_t *__restrict__ u, real_t *__restrict__ gacc, int face,
                   unsigned planes, int n)
{
    const int r = P.r, axis = face >> 1;
    const int N[3] = {P.nz, P.nx, SW_DIM == 3 ? P.ny : 1};
    int x[3] = {0, 0, 0};
    long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
    for (int a = SW_DIM - 1; a >= 0; a--) {
        if (a == axis)
            continue;
        const int len = N[a] - 2 * r;
        x[a] = r + (int)(t % len);
        t /= len;
    }
    if (t != 0)
        return;
    x[axis] = face & 1 ? N[axis] - r - 1 : r;
    for (int f = 0; f < face; f++)
        if ((planes >> f & 1) && x[f >> 1] == (f & 1 ? N[f >> 1] - r - 1 : r))
            return;
    const long long p = (long long)x[0] * P.sz + (long long)x[1] * P.sx + x[2];
    const real_t lv = l[p];
    if (lv == (real_t)0)
        return;
    const long long st[3] = {P.sz, P.sx, 1};
    const double h2[3] = {(double)P.dz2, (double)P.dx2, (double)P.dy2};
    double term = 0;
#pragma unroll
    for (int a = 0; a < SW_DIM; a++) {
        double acc = (double)P.c2[0] * (double)u[p];
        for (int m = 1; m <= r; m++)
            acc += (double)P.c2[m] * ((double)u[p + m * st[a]] + (double)u[p - m * st[a]]);
        term += acc / h2[a];
    }
    for (int s = 0; s < P.nsrc; s++) {
        const Box b = P.sbox[s];
        bool in = true;
#pragma unroll
        for (int a = 0; a < SW_DIM; a++)
            in = in && x[a] >= b.lo[a] && x[a] <= b.hi[a];
        if (in)
            term += (double)box_weight(b, P.sw, x[0], x[1], x[2]) * (double)wavelet_amp(P, n, s);
    }
    const double den = 1.0 + (double)P.e[p];
    const double dc = 2.0 * (double)P.q[p] / ((double)vel[p] * den * den);
    gacc[p] += (real_t)((double)lv * dc * term);
}

// Wavelet gradient of step n (k = n+1): gw[s] = sum_p kws_{s,p} c_p ub_p
// (c = q / den) over the source box's interior points, in float64, one
// block per source.  (The velocity derivative of the source term is part
// of the update's step difference.)
__global__ void __launch_bounds__(256)
k_adj_sources(Params P, const real_t *__restrict__ ub, real_t *__restrict__ gw)
{
    __shared__ double part[256];
    const int s = blockIdx.x;
    if (s >= P.nsrc)
        return;
    const Box b = P.sbox[s];
    const int cz = b.hi[0] - b.lo[0] + 1, cx = b.hi[1] - b.lo[1] + 1;
#if SW_DIM == 3
    const int cy = b.hi[2] - b.lo[2] + 1;
#else
    const int cy = 1;
#endif
    double acc = 0;
    for (int t = threadIdx.x; t < cz * cx * cy; t += blockDim.x) {
        const int ii = t / (cx * cy), rem = t - ii * cx * cy;
        const int jj = rem / cy, kk = rem - jj * cy;
        const int i = b.lo[0] + ii, j = b.lo[1] + jj;
#if SW_DIM == 3
        const int k = b.lo[2] + kk;
#else
        const int k = 0;
        (void)kk;
#endif
        if (!interior(P, i, j, k))
            continue;
        const long long p = (long long)i * P.sz + (long long)j * P.sx + k;
        const double kws = (double)box_weight(b, P.sw, i, j, k);
        const double q = (double)P.q[p], den = 1.0 + (double)P.e[p];
        acc += kws * (q / den) * (double)ub[p];
    }
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
            part[threadIdx.x] += part[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        gw[s] = (real_t)part[0];
}

__global__ void k_fill(real_t *p, long long n, real_t v)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

// r = d - o (the L2 misfit's adjoint source from the shot record d and the
// observed data o)
__global__ void k_residual(const real_t *__restrict__ d, const real_t *__restrict__ o,
                           real_t *__restrict__ r, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        r[i] = d[i] - o[i];
}

__global__ void k_fill_f64(double *p, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = 0.0;
}

}  // namespace sw
