// CDNA4 kernels of the implicit Euler family: FP64 element derivatives, force gather, block-sparse
// Hessian assembly, BSR SpMV and the conjugate gradient, all with fixed summation orders (the results
// do not depend on scheduling).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>

#include "implicit_device.h"
#include "implicit_element.h"

namespace spgvbd {

namespace {

inline int blocksFor(int64_t n, int bs) { return static_cast<int>((n + bs - 1) / bs); }

// One element per thread: gradient (tangent-free values of the first pass) and the Hessian one column
// per forward-mode pass, written straight to the element's column-major slot. One instantiation per
// energy type keeps each kernel's registers to that energy's closed form.
template <int TYPE>
__global__ void __launch_bounds__(128) elementDerivKernel(ImplicitElems e, const double *__restrict__ x)
{
    constexpr int NS = fullStencilSize(TYPE);
    constexpr int N = 3 * NS;
    constexpr int NP = fullParams(TYPE);
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= e.n) return;
    double p[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) p[k] = e.prm[i * NP + k];
    double xs[N];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int64_t v = e.idx[i * NS + s];
        xs[3 * s] = x[3 * v];
        xs[3 * s + 1] = x[3 * v + 1];
        xs[3 * s + 2] = x[3 * v + 2];
    }
    double *H = e.hess + i * N * N;
    double *g = e.grad + i * N;
#pragma unroll 1
    for (int j = 0; j < N; ++j) {
        V3<Dual1> xd[NS], gd[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s)
            xd[s] = {Dual1(xs[3 * s], 3 * s == j ? 1.0 : 0.0), Dual1(xs[3 * s + 1], 3 * s + 1 == j ? 1.0 : 0.0),
                     Dual1(xs[3 * s + 2], 3 * s + 2 == j ? 1.0 : 0.0)};
        fullGrad<NS, Dual1>(TYPE, xd, p, gd);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            H[j * N + 3 * s] = gd[s].x.d;
            H[j * N + 3 * s + 1] = gd[s].y.d;
            H[j * N + 3 * s + 2] = gd[s].z.d;
        }
        if (j == 0)
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                g[3 * s] = gd[s].x.v;
                g[3 * s + 1] = gd[s].y.v;
                g[3 * s + 2] = gd[s].z.v;
            }
    }
}

// Gradient only (no Hessian), in plain FP64: the force of the line-search trials.
template <int TYPE>
__global__ void __launch_bounds__(256) elementGradKernel(ImplicitElems e, const double *__restrict__ x)
{
    constexpr int NS = fullStencilSize(TYPE);
    constexpr int NP = fullParams(TYPE);
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= e.n) return;
    double p[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) p[k] = e.prm[i * NP + k];
    V3<double> xd[NS], gd[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int64_t v = e.idx[i * NS + s];
        xd[s] = {x[3 * v], x[3 * v + 1], x[3 * v + 2]};
    }
    fullGrad<NS, double>(TYPE, xd, p, gd);
    double *g = e.grad + i * 3 * NS;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        g[3 * s] = gd[s].x;
        g[3 * s + 1] = gd[s].y;
        g[3 * s + 2] = gd[s].z;
    }
}

// Workgroups are dealt round-robin over the 8 XCDs; this renumbering gives each XCD a contiguous band of
// the logical range, so neighbouring particles (which share elements and blocks) share that XCD's L2.
__device__ __forceinline__ int32_t xcdContiguous(int32_t b, int32_t nb)
{
    const int32_t xcd = b & 7, i = b >> 3, q = nb >> 3, r = nb & 7;
    return xcd < r ? xcd * (q + 1) + i : r * (q + 1) + (xcd - r) * q + i;
}

__global__ void __launch_bounds__(256) gatherForceKernel(int64_t n, const double *__restrict__ mass, double gx,
                                                         double gy, double gz, const int64_t *__restrict__ incPtr,
                                                         const int64_t *__restrict__ incOff,
                                                         const double *__restrict__ grad, double *__restrict__ f)
{
    const int64_t i = xcdContiguous(blockIdx.x, gridDim.x) * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    const double m = mass[i];
    double fx = gx * m, fy = gy * m, fz = gz * m;
    for (int64_t k = incPtr[i]; k < incPtr[i + 1]; ++k) {
        const double *g = grad + 3 * incOff[k];
        fx -= g[0];
        fy -= g[1];
        fz -= g[2];
    }
    f[3 * i] = fx;
    f[3 * i + 1] = fy;
    f[3 * i + 2] = fz;
}

__global__ void __launch_bounds__(256) assembleHessianKernel(int64_t nUpper, const int32_t *__restrict__ upRow,
                                                             const int32_t *__restrict__ upCol,
                                                             const int64_t *__restrict__ contribPtr,
                                                             const int64_t *__restrict__ contrib,
                                                             const double *__restrict__ hess, double *__restrict__ H)
{
    const int64_t u = xcdContiguous(blockIdx.x, gridDim.x) * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (u >= nUpper) return;
    double b[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t k = contribPtr[u]; k < contribPtr[u + 1]; ++k) {
        const int64_t c = contrib[k];
        const double *h = hess + (c >> 4);
        const int N3 = static_cast<int>(c & 15);
        for (int cc = 0; cc < 3; ++cc)
            for (int r = 0; r < 3; ++r) b[r * 3 + cc] += h[cc * N3 + r];
    }
    double *out = H + 9 * u;
    if (upRow[u] == upCol[u]) {  // diagonal block: symmetric part
        for (int r = 0; r < 3; ++r)
            for (int cc = 0; cc < 3; ++cc) out[r * 3 + cc] = 0.5 * (b[r * 3 + cc] + b[cc * 3 + r]);
        return;
    }
    for (int k = 0; k < 9; ++k) out[k] = b[k];
}

__global__ void __launch_bounds__(256) combineKernel(int64_t nBlocks, const double *__restrict__ H, double c,
                                                     double *__restrict__ A)
{
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k >= 9 * nBlocks) return;
    A[k] = c * H[k];
}

__global__ void __launch_bounds__(256) addMassKernel(int64_t n, const int64_t *__restrict__ diagBlock,
                                                     const double *__restrict__ mass, double a, double *__restrict__ A)
{
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    double *d = A + 9 * diagBlock[i];
    const double am = a * mass[i];
    d[0] += am;
    d[4] += am;
    d[8] += am;
}

__device__ __forceinline__ double blockSumFixed(double v, double *sh)
{
    // wave-level fixed butterfly, then the waves' sums in order
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < static_cast<int>(blockDim.x >> 6); ++w) s += sh[w];
    __syncthreads();
    return s;
}

// Symmetric block-row SpMV: kSpmvG lanes per block row; lane l takes the row's upper blocks l, l + G, ...
// whole (9 values, the column, the 3 x entries), then its lower blocks l, l + G, ... as transposes of the
// upper blocks that hold them, then a fixed butterfly over the G lanes. Workgroups are renumbered so
// each XCD streams a contiguous band of rows: the upper blocks a row reads transposed belong to rows a
// band streamed just before. Eight lanes per row (more than a cloth row's four upper blocks) keep fewer rows
// in flight per XCD, so those blocks are more often still in its L2 when they are read again: 40.5 us per
// product at 512x512 against 46.3 us with four lanes (two: 61.2, sixteen: 54.8).
constexpr int kSpmvG = 8;
constexpr int kSpmvBlock = 1024;

__device__ __forceinline__ V3<double> at3(const double *__restrict__ v, int64_t j)
{
    return {v[3 * j], v[3 * j + 1], v[3 * j + 2]};
}
// This lane's part of row `row` of A x
__device__ __forceinline__ V3<double> symRowPart(const SymBsr &A, int64_t row, int lig, const double *__restrict__ x)
{
    V3<double> y = {0.0, 0.0, 0.0};
    const int64_t u1 = A.upPtr[row + 1];
    for (int64_t k = A.upPtr[row] + lig; k < u1; k += kSpmvG) {
        const double *v = A.val + 9 * k;
        const V3<double> xc = at3(x, A.upCol[k]);
        y.x += v[0] * xc.x + v[1] * xc.y + v[2] * xc.z;
        y.y += v[3] * xc.x + v[4] * xc.y + v[5] * xc.z;
        y.z += v[6] * xc.x + v[7] * xc.y + v[8] * xc.z;
    }
    const int64_t l1 = A.loPtr[row + 1];
    for (int64_t k = A.loPtr[row] + lig; k < l1; k += kSpmvG) {
        const double *v = A.val + 9 * static_cast<int64_t>(A.loIdx[k]);
        const V3<double> xc = at3(x, A.loCol[k]);
        y.x += v[0] * xc.x + v[3] * xc.y + v[6] * xc.z;
        y.y += v[1] * xc.x + v[4] * xc.y + v[7] * xc.z;
        y.z += v[2] * xc.x + v[5] * xc.y + v[8] * xc.z;
    }
    return y;
}

// v + the v of the lane that CTRL pairs this lane with: a permutation of the lanes of a row by the moving instruction
// (DPP), without the hundred cycles of the LDS crossbar that a shuffle takes.
template <int CTRL>
__device__ __forceinline__ double addPartner(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
// the sum over the 4, 8 or 16 lanes of each aligned group, in every lane of it: quads by exchange of neighbours and of
// pairs, then mirrored halves and rows, whose quads hold equal sums by then
template <int G>
__device__ __forceinline__ double laneSum(double v)
{
    static_assert(G == 4 || G == 8 || G == 16, "lanes of a row");
    v = addPartner<0xB1>(v);                         // quad_perm 1 0 3 2
    v = addPartner<0x4E>(v);                         // quad_perm 2 3 0 1
    if constexpr (G >= 8) v = addPartner<0x141>(v);  // row_half_mirror
    if constexpr (G >= 16) v = addPartner<0x140>(v);  // row_mirror
    return v;
}
__device__ __forceinline__ double lane(double v, int l)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l), __builtin_amdgcn_readlane(__double2loint(v), l));
}
// the sum over the wavefront, in every lane (all of them active)
__device__ __forceinline__ double waveSum(double v)
{
    v = laneSum<16>(v);
    return (lane(v, 0) + lane(v, 16)) + (lane(v, 32) + lane(v, 48));
}

__device__ __forceinline__ V3<double> rowSum(V3<double> y)
{
    static_assert(kSpmvG == 8, "lanes of a block row");
    return {laneSum<8>(y.x), laneSum<8>(y.y), laneSum<8>(y.z)};
}

__device__ __forceinline__ void store3(double *__restrict__ v, int64_t j, V3<double> a)
{
    v[3 * j] = a.x;
    v[3 * j + 1] = a.y;
    v[3 * j + 2] = a.z;
}

// cg (may be null): the solve whose iteration `iteration` the product belongs to; nothing is done once it has ended.
__global__ void __launch_bounds__(kSpmvBlock) symSpmvKernel(SymBsr A, const double *__restrict__ x, double s,
                                                           double *__restrict__ y, double *__restrict__ partial,
                                                           const CgScalars *cg, int32_t iteration)
{
    __shared__ double sh[kSpmvBlock / 64];
    if (cg && cg->last < iteration) return;
    const int32_t blk = xcdContiguous(static_cast<int32_t>(blockIdx.x), static_cast<int32_t>(gridDim.x));
    const int64_t t = blk * static_cast<int64_t>(kSpmvBlock) + threadIdx.x;
    const int64_t row = t / kSpmvG;
    const int lig = static_cast<int>(t % kSpmvG);
    V3<double> r = {0.0, 0.0, 0.0};
    if (row < A.rows) r = symRowPart(A, row, lig, x);
    r = rowSum(r);
    double dot = 0.0;
    if (row < A.rows && lig == 0) {
        const V3<double> z = {s * r.x, s * r.y, s * r.z}, xr = at3(x, row);
        store3(y, row, z);
        dot = xr.x * z.x + xr.y * z.y + xr.z * z.z;
    }
    if (partial) {  // per-workgroup partial sums, in row order
        const double b = blockSumFixed(dot, sh);
        if (threadIdx.x == 0) partial[blk] = b;
    }
}

// Full block rows of s * A from the upper storage: one thread per block row.
__global__ void __launch_bounds__(256) expandSymKernel(SymBsr A, double s, const int64_t *__restrict__ rowPtr,
                                                       const int32_t *__restrict__ col,
                                                       const int64_t *__restrict__ diagBlock, double *__restrict__ out)
{
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= A.rows) return;
    for (int64_t k = rowPtr[i]; k < rowPtr[i + 1]; ++k) {
        const int32_t j = col[k];
        double *o = out + 9 * k;
        if (j >= i) {
            const double *v = A.val + 9 * (A.upPtr[i] + (k - diagBlock[i]));
            for (int e = 0; e < 9; ++e) o[e] = s * v[e];
            continue;
        }
        // upper block (j, i): binary search of column i in row j's upper blocks
        int64_t lo = A.upPtr[j], hi = A.upPtr[j + 1];
        while (hi - lo > 1) {
            const int64_t mid = (lo + hi) / 2;
            if (A.upCol[mid] <= i) lo = mid;
            else hi = mid;
        }
        const double *v = A.val + 9 * lo;
        for (int r = 0; r < 3; ++r)
            for (int c = 0; c < 3; ++c) o[r * 3 + c] = s * v[c * 3 + r];
    }
}

// Fixed-order partial sums: block b owns a contiguous chunk; its threads sum strided, then a fixed
// block reduction.
template <class F>
__device__ __forceinline__ double chunkSum(int64_t n, F term, double *sh)
{
    const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
    const int64_t b = blockIdx.x * chunk, e = b + chunk < n ? b + chunk : n;
    double acc = 0.0;
    for (int64_t i = b + threadIdx.x; i < e; i += blockDim.x) acc += term(i);
    return blockSumFixed(acc, sh);
}

__device__ __forceinline__ double finalSum(const double *__restrict__ partial, int n, double *sh)
{
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) acc += partial[i];
    return blockSumFixed(acc, sh);
}

__global__ void __launch_bounds__(256) cgInitKernel(int64_t n, const double *__restrict__ b,
                                                    const double *__restrict__ invdiag, double *__restrict__ x,
                                                    double *__restrict__ r, double *__restrict__ z,
                                                    double *__restrict__ p, double *__restrict__ q,
                                                    double *__restrict__ partial)
{
    // z null: an iteration in three kernels, whose first direction this is
    __shared__ double sh[4];
    const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
    const int64_t b0 = blockIdx.x * chunk, e0 = b0 + chunk < n ? b0 + chunk : n;
    for (int64_t i = b0 + threadIdx.x; i < e0; i += blockDim.x) {
        const double bi = b[i];
        x[i] = 0.0;
        r[i] = bi;
        const double zi = invdiag[i] * bi;
        p[i] = z ? 0.0 : zi;
        if (!z) continue;
        z[i] = zi;
        q[i] = 0.0;
    }
    const double bb = chunkSum(n, [&](int64_t i) { return b[i] * b[i]; }, sh);
    const double rp = chunkSum(n, [&](int64_t i) { return b[i] * (invdiag[i] * b[i]); }, sh);
    if (threadIdx.x == 0) {
        partial[blockIdx.x] = bb;
        partial[gridDim.x + blockIdx.x] = rp;
    }
}

__global__ void __launch_bounds__(1024) cgInitFinalKernel(const double *__restrict__ partial, int nb, CgScalars *s,
                                                          double tol)
{
    __shared__ double sh[16];
    const double bb = finalSum(partial, nb, sh);
    const double rp = finalSum(partial + nb, nb, sh);
    if (threadIdx.x == 0) {
        s->rhsNorm2 = bb;
        s->absNew[0] = rp;
        s->absNew[1] = 0.0;
        s->iters = 0;
        s->residualNorm2 = bb;  // r = b - A 0
        const double th = tol * tol * bb;
        s->threshold = th > DBL_MIN ? th : DBL_MIN;
        s->done = (bb == 0.0 || bb < s->threshold) ? 1 : 0;
        s->last = s->done ? -2 : INT32_MAX;
    }
}

// The sums of a[0, n) and b[0, n) (b may be null) in a fixed order, the same values in every thread and every
// workgroup. In two parts, so that other work can go between the loads and the sum: thread t's entries t, t + B, t + 2B,
// ... in that order, eight of its loads issued together; then one barrier. WAVES: wavefronts of the workgroup (B = 64
// WAVES); sh: 2 WAVES values.
template <int WAVES>
__device__ __forceinline__ void threadTotals(const double *__restrict__ a, const double *__restrict__ b, int n, double &u,
                                             double &v)
{
    constexpr int B = 64 * WAVES;
    u = v = 0.0;
    int i = threadIdx.x;
    for (; i + 7 * B < n; i += 8 * B) {
        double x[8], y[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            x[k] = a[i + k * B];
            y[k] = b ? b[i + k * B] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            u += x[k];
            v += y[k];
        }
    }
    for (; i < n; i += B) {
        u += a[i];
        if (b) v += b[i];
    }
}
// The totals of the wavefronts' sums in sh, in every lane.
template <int WAVES>
__device__ __forceinline__ void wavesTotal(const double *sh, int lane, double &ta, double &tb)
{
    ta = laneSum<WAVES>(sh[lane % WAVES]);
    tb = laneSum<WAVES>(sh[WAVES + lane % WAVES]);
}
template <int WAVES>
__device__ __forceinline__ void blockTotals(double u, double v, double *sh, double &ta, double &tb)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u = waveSum(u);
    v = waveSum(v);
    if (lane == 0) {
        sh[wave] = u;
        sh[WAVES + wave] = v;
    }
    __syncthreads();
    wavesTotal<WAVES>(sh, lane, ta, tb);
}

// Per-workgroup sums of u and v into a and b, fixed order.
template <int WAVES>
__device__ __forceinline__ void storeBlockSums(double u, double v, double *sh, double *a, double *b)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u = waveSum(u);
    v = waveSum(v);
    __syncthreads();  // sh may still be read
    if (lane == 0) {
        sh[wave] = u;
        sh[WAVES + wave] = v;
    }
    __syncthreads();
    if (wave > 0) return;
    wavesTotal<WAVES>(sh, lane, u, v);
    if (lane == 0) {
        *a = u;
        if (b) *b = v;
    }
}

// The end of CG iteration `iteration` - 1 from its sums rr = r.r and rz = r.D^-1 r: the convergence test, and beta. False:
// the solve is over. The first thread of the first workgroup (`lead`) stores the scalars while other workgroups read
// them, so what they read is the same before and after: absNew is double-buffered by iteration parity, and `last` is
// compared so that it ends later kernels only.
__device__ __forceinline__ bool cgNext(CgScalars *s, double rr, double rz, double before, double threshold,
                                       int32_t iteration, bool lead, double &beta)
{
    beta = rz / before;
    if (lead) s->residualNorm2 = rr;
    if (rr < threshold) {
        if (lead) {
            s->last = iteration - 1;
            s->done = 1;
        }
        return false;
    }
    if (lead) {
        s->absNew[iteration & 1] = rz;
        s->iters = iteration;
    }
    return true;
}

// An iteration in two kernels, for systems that the caches hold (cgInTwoKernels). The first closes the iteration before
// (convergence, beta) and forms p = z + beta p and q = A p = A z + beta q, z = D^-1 r: the product is taken of z, which the
// kernel before left whole, so no kernel in between has to form p for the gather, and its loads do not wait for beta. The
// second (cgUpdateKernel) takes alpha and updates x, r and z. Every workgroup adds up the partial sums itself, in the same
// order, and loads its first entries before that.
//
// What bounds an iteration: at 200x200 particles the latency of two dependent launches with a reduction each (the matrix,
// 20 MB, comes from the L2s; the product takes 12.5 us of the 17.4, 8.2 by itself), from 500x500 on the memory. Cloths of
// n x n particles, us an iteration, in two kernels and in three (product, update, direction p = D^-1 r + beta p):
//    48: 12.9  17.8    200: 17.4  20.5    330: 30.8  32.6    420: 41.9  43.5    480: 52.4  53.5    512: 55.4  54.0
//   570: 67.0  64.5    700:  123   115    850:  185   175   1000:  253   235   1200:  362   333
// Beyond the caches p and q, read and written by one lane of eight at the end of a product, cost more than the passes over
// the vectors that they save. Of what two kernels gain where they do, the sums by lane permutations are 2 to 3 us,
// workgroups of 512 instead of 1024 threads 1.5 (the barrier waits for fewer). With sums through shuffles that waited for each
// other three kernels took 20.8 us at 48x48, 23.5 at 200x200, 57.2 at 512x512 and 239 at 1000x1000. Forming p in the gather
// (z + beta p of every neighbour) took 4 to 11 us more than q's recurrence, which costs little accuracy: after 1517 iterations
// at 200x200 particles b - A x is 9.7347e-11 |b| and the r that was carried along 9.7350e-11 |b| (9.7229e-11 and 9.7228e-11
// with q = A p).
constexpr int kCgProductBlock = 512;
__global__ void __launch_bounds__(kCgProductBlock) cgProductKernel(SymBsr A, const double *__restrict__ z,
                                                              double *__restrict__ p, double *__restrict__ q,
                                                              const double *__restrict__ uPartial,
                                                              double *__restrict__ partial, CgScalars *s,
                                                              int32_t iteration)
{
    constexpr int WAVES = kCgProductBlock / 64;
    __shared__ double sh[2 * WAVES];
    const int32_t last = s->last;
    const double before = s->absNew[(iteration & 1) ^ 1], threshold = s->threshold;
    const int32_t blk = xcdContiguous(static_cast<int32_t>(blockIdx.x), static_cast<int32_t>(gridDim.x));
    const int64_t t = blk * static_cast<int64_t>(kCgProductBlock) + threadIdx.x;
    const int64_t row = t / kSpmvG;
    const int lig = static_cast<int>(t % kSpmvG);
    const bool store = row < A.rows && lig == 0;
    double u = 0.0, v = 0.0;
    static_assert(kCgBlocks <= kCgProductBlock, "a partial sum to a thread");
    if (iteration > 0 && threadIdx.x < kCgBlocks) {
        u = uPartial[threadIdx.x];
        v = uPartial[kCgBlocks + threadIdx.x];
    }
    // `last` is iteration - 1 at the most while this kernel may store it (cgNext): every thread takes the same branch
    if (last < iteration - 1) return;
    V3<double> zr = {0.0, 0.0, 0.0}, pr = zr, qr = zr, w = zr;
    if (row < A.rows) w = symRowPart(A, row, lig, z);
    __builtin_amdgcn_sched_barrier(0);  // the row's own entries after its product's: together they exceed 64 registers
    if (store) {
        zr = at3(z, row);
        pr = at3(p, row);
        qr = at3(q, row);
    }
    w = rowSum(w);
    double beta = 0.0;
    if (iteration > 0) {
        double rr, rz;
        blockTotals<WAVES>(u, v, sh, rr, rz);
        if (!cgNext(s, rr, rz, before, threshold, iteration, blockIdx.x == 0 && threadIdx.x == 0, beta)) return;
    }
    double dot = 0.0;
    if (store) {
        pr = {zr.x + beta * pr.x, zr.y + beta * pr.y, zr.z + beta * pr.z};
        qr = {w.x + beta * qr.x, w.y + beta * qr.y, w.z + beta * qr.z};
        store3(p, row, pr);
        store3(q, row, qr);
        dot = pr.x * qr.x + pr.y * qr.y + pr.z * qr.z;
    }
    storeBlockSums<WAVES>(dot, 0.0, sh, partial + blk, nullptr);
}

// alpha = r.z / p.q, x += alpha p, r -= alpha q, z = D^-1 r; partial sums of r.r and r.z. Workgroups take contiguous
// chunks of the vectors, renumbered so that each XCD's chunks are the rows whose products it forms: what one kernel
// writes the next finds in the same L2. TWO: of an iteration in two kernels, which reads z again.
constexpr int kCgAhead = 4;  // entries of a thread loaded together
template <bool TWO>
__global__ void __launch_bounds__(256) cgUpdateKernel(int64_t n, const double *__restrict__ invdiag,
                                                      double *__restrict__ x, double *__restrict__ r,
                                                      double *__restrict__ z, const double *__restrict__ p,
                                                      const double *__restrict__ q,
                                                      const double *__restrict__ pPartial, int nbP,
                                                      double *__restrict__ partial, const CgScalars *s,
                                                      int32_t iteration)
{
    __shared__ double sh[8];
    const int32_t last = s->last;
    const double absNew = s->absNew[iteration & 1];
    const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
    const int64_t b0 = xcdContiguous(blockIdx.x, gridDim.x) * chunk, e0 = b0 + chunk < n ? b0 + chunk : n;
    double xv[kCgAhead], pv[kCgAhead], rv[kCgAhead], qv[kCgAhead], dv[kCgAhead];
    const auto load = [&](int64_t i0) {
#pragma unroll
        for (int k = 0; k < kCgAhead; ++k) {
            const int64_t i = i0 + k * 256;
            if (i < e0) {
                xv[k] = x[i];
                pv[k] = p[i];
                rv[k] = r[i];
                qv[k] = q[i];
                dv[k] = invdiag[i];
            }
        }
    };
    int64_t i0 = b0 + threadIdx.x;
    load(i0);
    double u, v, pq, unused;
    threadTotals<4>(pPartial, nullptr, nbP, u, v);
    if (last < iteration) return;
    blockTotals<4>(u, v, sh, pq, unused);
    const double alpha = absNew / pq;
    double rr = 0.0, rz = 0.0;
    while (i0 < e0) {
#pragma unroll
        for (int k = 0; k < kCgAhead; ++k) {
            const int64_t i = i0 + k * 256;
            if (i < e0) {
                const double ri = rv[k] - alpha * qv[k], zi = dv[k] * ri;
                x[i] = xv[k] + alpha * pv[k];
                r[i] = ri;
                if constexpr (TWO) z[i] = zi;
                rr += ri * ri;
                rz += ri * zi;
            }
        }
        i0 += kCgAhead * 256;
        load(i0);
    }
    storeBlockSums<4>(rr, rz, sh, partial + blockIdx.x, partial + gridDim.x + blockIdx.x);
}

// The third kernel of an iteration in three: its end (convergence, beta) and p = D^-1 r + beta p.
__global__ void __launch_bounds__(256) cgDirectionKernel(int64_t n, const double *__restrict__ invdiag,
                                                         const double *__restrict__ r, double *__restrict__ p,
                                                         const double *__restrict__ uPartial, int nbU, CgScalars *s,
                                                         int32_t iteration)
{
    __shared__ double sh[8];
    const int32_t last = s->last;
    const double before = s->absNew[iteration & 1], threshold = s->threshold;
    const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
    const int64_t b0 = xcdContiguous(blockIdx.x, gridDim.x) * chunk, e0 = b0 + chunk < n ? b0 + chunk : n;
    double pv[kCgAhead], rv[kCgAhead], dv[kCgAhead];
    const auto load = [&](int64_t i0) {
#pragma unroll
        for (int k = 0; k < kCgAhead; ++k) {
            const int64_t i = i0 + k * 256;
            if (i < e0) {
                pv[k] = p[i];
                rv[k] = r[i];
                dv[k] = invdiag[i];
            }
        }
    };
    int64_t i0 = b0 + threadIdx.x;
    load(i0);
    double u, v, rr, rz, beta;
    threadTotals<4>(uPartial, uPartial + nbU, nbU, u, v);
    if (last < iteration) return;  // `iteration` at the least while this kernel may store it
    blockTotals<4>(u, v, sh, rr, rz);
    if (!cgNext(s, rr, rz, before, threshold, iteration + 1, blockIdx.x == 0 && threadIdx.x == 0, beta)) return;
    while (i0 < e0) {
#pragma unroll
        for (int k = 0; k < kCgAhead; ++k) {
            const int64_t i = i0 + k * 256;
            if (i < e0) p[i] = dv[k] * rv[k] + beta * pv[k];
        }
        i0 += kCgAhead * 256;
        load(i0);
    }
}

// After the last iteration of the budget: its convergence test (x is the last iterate either way).
__global__ void __launch_bounds__(256) cgFinishKernel(const double *__restrict__ uPartial, int nbU, CgScalars *s,
                                                      int32_t iterations)
{
    __shared__ double sh[8];
    double u, v, rr, rz, beta;
    const int32_t last = s->last;
    const double before = s->absNew[(iterations & 1) ^ 1], threshold = s->threshold;
    threadTotals<4>(uPartial, uPartial + nbU, nbU, u, v);
    if (last < iterations) return;
    blockTotals<4>(u, v, sh, rr, rz);
    if (cgNext(s, rr, rz, before, threshold, iterations, threadIdx.x == 0, beta) && threadIdx.x == 0) {
        s->last = iterations - 1;
        s->done = 2;
    }
}

__global__ void __launch_bounds__(256) invDiagKernel(int64_t n, const int64_t *__restrict__ diagBlock,
                                                     const double *__restrict__ A, double *__restrict__ invdiag)
{
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    const double *d = A + 9 * diagBlock[i];
    for (int k = 0; k < 3; ++k) {
        const double a = d[4 * k];
        invdiag[3 * i + k] = a != 0.0 ? 1.0 / a : 1.0;
    }
}

__global__ void __launch_bounds__(256) linCombKernel(int64_t n, double *__restrict__ out, double a,
                                                     const double *__restrict__ x, double b,
                                                     const double *__restrict__ y, double c,
                                                     const double *__restrict__ z)
{
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    double v = a * x[i];
    if (y) v += b * y[i];
    if (z) v += c * z[i];
    out[i] = v;
}

__global__ void __launch_bounds__(256) massLinCombKernel(int64_t n, double *__restrict__ out, double a,
                                                         const double *__restrict__ mass,
                                                         const double *__restrict__ x, double b,
                                                         const double *__restrict__ y)
{
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    double v = a * mass[i / 3] * x[i];
    if (y) v += b * y[i];
    out[i] = v;
}

__global__ void __launch_bounds__(256) norm2PartialKernel(int64_t n, const double *__restrict__ x,
                                                          double *__restrict__ partial)
{
    __shared__ double sh[4];
    const double t = chunkSum(n, [&](int64_t i) { return x[i] * x[i]; }, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

__global__ void __launch_bounds__(1024) sumFinalKernel(const double *__restrict__ partial, int nb, double *out)
{
    __shared__ double sh[16];
    const double t = finalSum(partial, nb, sh);
    if (threadIdx.x == 0) *out = t;
}

}  // namespace

#define SPG_ELEMENT_CASES(KERNEL, BS)                                                                              \
    switch (e.type) {                                                                                          \
    case 1: KERNEL<1><<<grid, BS, 0, stream>>>(e, x); break;                                                   \
    case 2: KERNEL<2><<<grid, BS, 0, stream>>>(e, x); break;                                                   \
    case 3: KERNEL<3><<<grid, BS, 0, stream>>>(e, x); break;                                                   \
    case 4: KERNEL<4><<<grid, BS, 0, stream>>>(e, x); break;                                                   \
    case 5: KERNEL<5><<<grid, BS, 0, stream>>>(e, x); break;                                                   \
    case 6: KERNEL<6><<<grid, BS, 0, stream>>>(e, x); break;                                                   \
    case 7: KERNEL<7><<<grid, BS, 0, stream>>>(e, x); break;                                                   \
    case 8: KERNEL<8><<<grid, BS, 0, stream>>>(e, x); break;                                                   \
    case 9: KERNEL<9><<<grid, BS, 0, stream>>>(e, x); break;                                                   \
    case 10: KERNEL<10><<<grid, BS, 0, stream>>>(e, x); break;                                                 \
    case 11: KERNEL<11><<<grid, BS, 0, stream>>>(e, x); break;                                                 \
    case 12: KERNEL<12><<<grid, BS, 0, stream>>>(e, x); break;                                                 \
    case 13: KERNEL<13><<<grid, BS, 0, stream>>>(e, x); break;                                                 \
    default: return hipErrorInvalidValue;                                                                      \
    }

hipError_t launchElementDerivatives(const ImplicitElems &e, const double *x, hipStream_t stream)
{
    if (e.n <= 0) return hipSuccess;
    const int grid = blocksFor(e.n, 128);
    SPG_ELEMENT_CASES(elementDerivKernel, 128)
    return hipGetLastError();
}

hipError_t launchElementGradients(const ImplicitElems &e, const double *x, hipStream_t stream)
{
    if (e.n <= 0) return hipSuccess;
    const int grid = blocksFor(e.n, 256);
    SPG_ELEMENT_CASES(elementGradKernel, 256)
    return hipGetLastError();
}

#undef SPG_ELEMENT_CASES

hipError_t launchGatherForce(int64_t nParticles, const double *mass, double gx, double gy, double gz,
                             const int64_t *incPtr, const int64_t *incOff, const double *gradBase, double *f,
                             hipStream_t stream)
{
    if (nParticles <= 0) return hipSuccess;
    gatherForceKernel<<<blocksFor(nParticles, 256), 256, 0, stream>>>(nParticles, mass, gx, gy, gz, incPtr, incOff,
                                                                       gradBase, f);
    return hipGetLastError();
}

hipError_t launchAssembleHessian(int64_t nUpper, const int32_t *upRow, const int32_t *upCol, const int64_t *contribPtr,
                                 const int64_t *contrib, const double *hessBase, double *H, hipStream_t stream)
{
    if (nUpper <= 0) return hipSuccess;
    assembleHessianKernel<<<blocksFor(nUpper, 256), 256, 0, stream>>>(nUpper, upRow, upCol, contribPtr, contrib,
                                                                       hessBase, H);
    return hipGetLastError();
}

hipError_t launchCombine(int64_t nBlocks, const double *H, double c, int64_t nParticles, const int64_t *diagBlock,
                         const double *mass, double a, double *A, hipStream_t stream)
{
    if (nBlocks <= 0) return hipSuccess;
    combineKernel<<<blocksFor(9 * nBlocks, 256), 256, 0, stream>>>(nBlocks, H, c, A);
    if (nParticles > 0 && a != 0.0)
        addMassKernel<<<blocksFor(nParticles, 256), 256, 0, stream>>>(nParticles, diagBlock, mass, a, A);
    return hipGetLastError();
}

namespace {
int spmvGrid(int64_t rows) { return blocksFor(rows * kSpmvG, kSpmvBlock); }
}  // namespace

int cgProductGrid(int64_t rows) { return blocksFor(rows * kSpmvG, kCgProductBlock); }
int spmvPartials(int64_t rows) { return std::max(spmvGrid(rows), cgProductGrid(rows)); }

hipError_t launchSymSpmv(const SymBsr &A, const double *x, double s, double *y, hipStream_t stream)
{
    if (A.rows <= 0) return hipSuccess;
    symSpmvKernel<<<spmvGrid(A.rows), kSpmvBlock, 0, stream>>>(A, x, s, y, nullptr, nullptr, 0);
    return hipGetLastError();
}

hipError_t launchExpandSym(const SymBsr &A, double s, const int64_t *rowPtr, const int32_t *col,
                           const int64_t *diagBlock, double *out, hipStream_t stream)
{
    if (A.rows <= 0) return hipSuccess;
    expandSymKernel<<<blocksFor(A.rows, 256), 256, 0, stream>>>(A, s, rowPtr, col, diagBlock, out);
    return hipGetLastError();
}

hipError_t launchCgInit(int64_t n, const double *b, const double *invdiag, double *x, double *r, double *z, double *p,
                        double *q, double *partial, CgScalars *s, double tol, hipStream_t stream)
{
    cgInitKernel<<<kCgBlocks, 256, 0, stream>>>(n, b, invdiag, x, r, z, p, q, partial);
    cgInitFinalKernel<<<1, 1024, 0, stream>>>(partial, kCgBlocks, s, tol);
    return hipGetLastError();
}

hipError_t launchCgIteration(const SymBsr &A, int64_t n, const double *invdiag, double *x, double *r, double *z,
                             double *p, double *q, double *pPartial, double *uPartial, CgScalars *s, int32_t maxIters,
                             int32_t iteration, hipStream_t stream, hipEvent_t spmvStart, hipEvent_t spmvEnd)
{
    if (spmvStart) {
        const hipError_t e = hipEventRecord(spmvStart, stream);
        if (e != hipSuccess) return e;
    }
    const int grid = z ? cgProductGrid(A.rows) : spmvGrid(A.rows);
    if (z)
        cgProductKernel<<<grid, kCgProductBlock, 0, stream>>>(A, z, p, q, uPartial, pPartial, s, iteration);
    else
        symSpmvKernel<<<grid, kSpmvBlock, 0, stream>>>(A, p, 1.0, q, pPartial, s, iteration);
    if (spmvEnd) {
        const hipError_t e = hipEventRecord(spmvEnd, stream);
        if (e != hipSuccess) return e;
    }
    const auto update = z ? cgUpdateKernel<true> : cgUpdateKernel<false>;
    update<<<kCgBlocks, 256, 0, stream>>>(n, invdiag, x, r, z, p, q, pPartial, grid, uPartial, s, iteration);
    if (iteration + 1 == maxIters)
        cgFinishKernel<<<1, 256, 0, stream>>>(uPartial, kCgBlocks, s, maxIters);
    else if (!z)
        cgDirectionKernel<<<kCgBlocks, 256, 0, stream>>>(n, invdiag, r, p, uPartial, kCgBlocks, s, iteration);
    return hipGetLastError();
}

hipError_t launchInvDiag(int64_t nParticles, const int64_t *diagBlock, const double *A, double *invdiag,
                         hipStream_t stream)
{
    if (nParticles <= 0) return hipSuccess;
    invDiagKernel<<<blocksFor(nParticles, 256), 256, 0, stream>>>(nParticles, diagBlock, A, invdiag);
    return hipGetLastError();
}

hipError_t launchLinComb(int64_t n, double *out, double a, const double *x, double b, const double *y, double c,
                         const double *z, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    linCombKernel<<<blocksFor(n, 256), 256, 0, stream>>>(n, out, a, x, b, y, c, z);
    return hipGetLastError();
}

hipError_t launchMassLinComb(int64_t n, double *out, double a, const double *mass, const double *x, double b,
                             const double *y, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    massLinCombKernel<<<blocksFor(n, 256), 256, 0, stream>>>(n, out, a, mass, x, b, y);
    return hipGetLastError();
}

hipError_t launchNorm2(int64_t n, const double *x, double *partial, double *out, hipStream_t stream)
{
    norm2PartialKernel<<<kCgBlocks, 256, 0, stream>>>(n, x, partial);
    sumFinalKernel<<<1, 1024, 0, stream>>>(partial, kCgBlocks, out);
    return hipGetLastError();
}

}  // namespace spgvbd
