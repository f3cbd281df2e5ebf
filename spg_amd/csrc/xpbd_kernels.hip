// CDNA4 kernels of the XPBD step (spg/source/sim/solver/xpbd.cpp:16-132): substep boundaries and one
// projection kernel per energy type. A projection launch runs one stencil group (a colour, or a level of
// the serial order) of one energy: a thread per stencil gathers its particles, solves the stencil's
// nC x nC system and writes the displaced particles back. No two stencils of a launch share a
// particle, so the writes need no atomics and the result does not depend on the thread order.
#include <hip/hip_ext.h>

#include <type_traits>

#include "element.h"
#include "vbd_device.h"
#include "xpbd_device.h"
#include "xpbd_element.h"

namespace spgvbd {

namespace {

using V3f = V3<float>;

__device__ __forceinline__ V3f xyz(float4 p) { return {p.x, p.y, p.z}; }
__device__ __forceinline__ float4 moved(float4 p, V3f d) { return make_float4(p.x + d.x, p.y + d.y, p.z + d.z, p.w); }

__device__ __forceinline__ void countFp64(bool fell, unsigned long long *counters)
{
    if (fell && counters) atomicAdd(counters, 1ull);
}

// The projection of one stencil of each type (xpbd.cpp:84-95) on the positions `pos` of the particles i0 .. i3: global
// memory, or a tile's LDS. s: 1 / dt^2. `counters` receives whether it was solved in FP64, if it `counts` (the address is the
// same in every lane: a wavefront adds once), ahead of the stores: the records are then written whole, where the compiler
// would otherwise leave out their unchanged fourth value, and scattered 12-byte stores cost more than 16-byte ones (a
// substep with a launch per group, the count after and ahead of the stores, us: 1024x1024 cloth 196 and 192, 80^3-cell
// solid 206 and 201, 700x700 cloth with continuum springs 256 and 251).
template <class P>
__device__ __forceinline__ void projectSpring(P pos, int32_t i0, int32_t i1, float L0, float c, float s)
{
    const float4 X0 = pos[i0], X1 = pos[i1];
    V3f d0, d1;
    xpbdSpring<float>(xyz(X0), xyz(X1), X0.w, X1.w, L0, c * s, d0, d1);
    pos[i0] = moved(X0, d0);
    pos[i1] = moved(X1, d1);
}

template <class P>
__device__ __forceinline__ void projectAnchor(P pos, int32_t i0, float4 p, float s)
{
    const float4 X = pos[i0];
    pos[i0] = moved(X, xpbdAnchor<float>(xyz(X), X.w, V3f{p.x, p.y, p.z}, p.w * s));
}

template <class P>
__device__ __forceinline__ void projectStvk(P pos, int32_t i0, int32_t i1, int32_t i2, float4 D, float4 c, float2 c2,
                                            float s, unsigned long long *counters, bool counts)
{
    const float4 X0 = pos[i0], X1 = pos[i1], X2 = pos[i2];
    V3f o0, o1, o2;
    const bool fell = xpbdStvkF(xyz(X0), xyz(X1), xyz(X2), X0.w, X1.w, X2.w, D.x, D.y, D.z, D.w, c.x * s, c.y * s,
                                c.z * s, c.w * s, c2.x * s, c2.y * s, o0, o1, o2);
    countFp64(fell && counts, counters);
    pos[i0] = moved(X0, o0);
    pos[i1] = moved(X1, o1);
    pos[i2] = moved(X2, o2);
}

template <class P>
__device__ __forceinline__ void projectBending(P pos, int32_t i0, int32_t i1, int32_t i2, int32_t i3, float theta0,
                                               float c, float s)
{
    const float4 X0 = pos[i0], X1 = pos[i1], X2 = pos[i2], X3 = pos[i3];
    V3f o0, o1, o2, o3;
    xpbdBending<float>(xyz(X0), xyz(X1), xyz(X2), xyz(X3), X0.w, X1.w, X2.w, X3.w, theta0, c * s, o0, o1, o2, o3);
    pos[i0] = moved(X0, o0);
    pos[i1] = moved(X1, o1);
    pos[i2] = moved(X2, o2);
    pos[i3] = moved(X3, o3);
}

// d2: D22 and the compliances c00, c01, c11
template <class P>
__device__ __forceinline__ void projectSnh(P pos, int32_t i0, int32_t i1, int32_t i2, int32_t i3, float4 d0, float4 d1,
                                           float4 d2, float hyd, float s, unsigned long long *counters, bool counts)
{
    const float D[9] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w, d2.x};
    const float4 X0 = pos[i0], X1 = pos[i1], X2 = pos[i2], X3 = pos[i3];
    V3f o0, o1, o2, o3;
    const bool fell = xpbdSnhF(xyz(X0), xyz(X1), xyz(X2), xyz(X3), X0.w, X1.w, X2.w, X3.w, D, d2.y * s, d2.z * s,
                               d2.w * s, hyd, o0, o1, o2, o3);
    countFp64(fell && counts, counters);
    pos[i0] = moved(X0, o0);
    pos[i1] = moved(X1, o1);
    pos[i2] = moved(X2, o2);
    pos[i3] = moved(X3, o3);
}

template <int T, class P>
__device__ __forceinline__ void projectFurther(P pos, const int32_t (&vv)[4], const float4 (&c)[3], float s,
                                               unsigned long long *counters, bool counts)
{
    constexpr int NS = xpbdFurtherStencil(T);
    float4 X[4];
    double xs[12], ws[4], ps[12], dx[12];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        X[k] = pos[vv[k]];
        xs[3 * k] = X[k].x;
        xs[3 * k + 1] = X[k].y;
        xs[3 * k + 2] = X[k].z;
        ws[k] = X[k].w;
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        ps[4 * q] = c[q].x;
        ps[4 * q + 1] = c[q].y;
        ps[4 * q + 2] = c[q].z;
        ps[4 * q + 3] = c[q].w;
    }
    const bool fell = xpbdFurtherRecord<true>(T, xs, ws, ps, s, dx);
    countFp64(fell && counts, counters);
#pragma unroll
    for (int k = 0; k < NS; ++k)
        pos[vv[k]] = moved(X[k], V3f{float(dx[3 * k]), float(dx[3 * k + 1]), float(dx[3 * k + 2])});
}

// The projection of stencil record i of type T on the positions in global memory.
template <int T>
__device__ __forceinline__ void projectStencil(const XpbdArgs &a, int32_t i)
{
    if constexpr (T == kSpring) {
        const int2 id = a.sprI[i];
        const float2 p = a.sprP[i];
        projectSpring(a.pos, id.x, id.y, p.x, p.y, a.invdt2);
    } else if constexpr (T == kAnchor) {
        const int32_t id = a.ancI[i];
        projectAnchor(a.pos, id, a.ancP[i], a.invdt2);
    } else if constexpr (T == kStvk) {
        const int4 id = a.triI[i];
        projectStvk(a.pos, id.x, id.y, id.z, a.triD[i], a.triC0[i], a.triC1[i], a.invdt2, a.counters, true);
    } else if constexpr (T == kBending) {
        const int4 id = a.hinI[i];
        const float2 p = a.hinP[i];
        projectBending(a.pos, id.x, id.y, id.z, id.w, p.x, p.y, a.invdt2);
    } else if constexpr (T == kSnh) {
        const int4 id = a.tetI[i];
        projectSnh(a.pos, id.x, id.y, id.z, id.w, a.tetD0[i], a.tetD1[i], a.tetD2[i], a.tetH[i], a.invdt2, a.counters, true);
    } else if constexpr (T >= 6) {
        const int4 id = a.extI[i];
        const int64_t q = 3 * static_cast<int64_t>(i);
        const int32_t vv[4] = {id.x, id.y, id.z, id.w};
        const float4 c[3] = {a.extP[q], a.extP[q + 1], a.extP[q + 2]};
        projectFurther<T>(a.pos, vv, c, a.invdt2, a.counters, true);
    }
}

// One stencil group (a colour of one energy) over the whole chip: a thread per record. The grid size and
// threads per block come with the arguments, so the prologue waits for one round of scalar loads.
template <int T>
__global__ void __launch_bounds__(256) xpbdProjectKernel(XpbdArgs a, int32_t begin, int32_t end)
{
    asm volatile("" ::"s"(a.pos), "s"(a.hinI), "s"(a.hinP), "s"(a.triI), "s"(a.triD), "s"(a.triC0), "s"(a.triC1));
    const int32_t blk = xcdContiguousBlock(blockIdx.x, a.gridBlocks);
    const int32_t i = begin + blk * a.blockThreads + static_cast<int32_t>(threadIdx.x);
    if (i >= end) return;
    projectStencil<T>(a, i);
}

// A run of consecutive small stencil groups in one workgroup: the groups in order, each spread over the
// workgroup's threads, a workgroup barrier between two groups (the writes of one group are visible to the
// next: the whole run stays on one CU). Stencils of one group share no particle, so the result equals one
// launch per group.
__global__ void __launch_bounds__(256) xpbdProjectRunKernel(XpbdArgs a, XpbdRun run)
{
    for (int32_t r = 0; r < run.count; ++r) {
        const int32_t t = run.type[r];
        for (int32_t i = run.begin[r] + static_cast<int32_t>(threadIdx.x); i < run.end[r];
             i += static_cast<int32_t>(blockDim.x)) {
            switch (t) {
            case kSpring: projectStencil<kSpring>(a, i); break;
            case kStvk: projectStencil<kStvk>(a, i); break;
            case kBending: projectStencil<kBending>(a, i); break;
            case kSnh: projectStencil<kSnh>(a, i); break;
            case kAnchor: projectStencil<kAnchor>(a, i); break;
            case 6: projectStencil<6>(a, i); break;
            case 7: projectStencil<7>(a, i); break;
            case 8: projectStencil<8>(a, i); break;
            case 9: projectStencil<9>(a, i); break;
            case 10: projectStencil<10>(a, i); break;
            case 11: projectStencil<11>(a, i); break;
            case 12: projectStencil<12>(a, i); break;
            default: projectStencil<13>(a, i);
            }
        }
        __syncthreads();
    }
}

// ---- tiles (the plan: xpbd_tiles.h) ----

// The start of a substep for one particle (xpbd.cpp:47-70 with particleGroup.cpp:57-63). START 1: the first substep, v
// from memory; 2: v = (x - x_prev) / h_prev from the positions one substep before; other: x as it is.
template <int START>
__device__ __forceinline__ float4 substepStart(const XpbdTileArgs &a, int32_t id)
{
    float4 x = a.in[id];
    if constexpr (START == 1 || START == 2) {
        const float4 o = a.prev[id];
        float3 v;
        if constexpr (START == 1)
            v = make_float3(o.x, o.y, o.z);
        else
            v = make_float3((x.x - o.x) * a.invhPrev, (x.y - o.y) * a.invhPrev, (x.z - o.z) * a.invhPrev);
        v.x += a.hgx;
        v.y += a.hgy;
        v.z += a.hgz;
        x.x += v.x * a.h;
        x.y += v.y * a.h;
        x.z += v.z * a.h;
    }
    return x;
}

// A stencil's tile record: r[0] holds its particles' places (16 bits each) and two coefficients, r[1 ...] the rest
// (written by tileRecordsKernel).
template <int T>
__device__ __forceinline__ void projectTileRecord(float4 *pos, const float4 (&r)[4], float s,
                                                  unsigned long long *counters)
{
    const uint32_t lo = __float_as_uint(r[0].x), hi = __float_as_uint(r[0].y);
    const int32_t i0 = lo & 0x7fff, i1 = lo >> 16, i2 = hi & 0xffff, i3 = hi >> 16;
    const bool counts = lo & kTileCounts;  // else another tile counts it
    if constexpr (T == kSpring)
        projectSpring(pos, i0, i1, r[0].z, r[0].w, s);
    else if constexpr (T == kAnchor)
        projectAnchor(pos, i0, r[1], s);
    else if constexpr (T == kStvk)
        projectStvk(pos, i0, i1, i2, r[1], r[2], make_float2(r[0].z, r[0].w), s, counters, counts);
    else if constexpr (T == kBending)
        projectBending(pos, i0, i1, i2, i3, r[0].z, r[0].w, s);
    else if constexpr (T == kSnh)
        projectSnh(pos, i0, i1, i2, i3, r[1], r[2], r[3], r[0].z, s, counters, counts);
    else {
        const int32_t vv[4] = {i0, i1, i2, i3};
        const float4 c[3] = {r[1], r[2], r[3]};
        projectFurther<T>(pos, vv, c, s, counters, counts);
    }
}

// A batch of stencil groups over tiles of particles: one workgroup per tile loads the tile's particles into LDS (with
// START, advanced to the start of the substep), runs the groups in order with a workgroup barrier between two, and
// writes its own particles. A thread's record of the next group is loaded before it projects the present one, so the
// loads' latency falls into the projection and the barrier.
//
// What bounds it: the chain of groups, about 1 us each (LDS reads, 300 to 400 dependent instructions, barrier), in which
// a thread has one stencil. Hence as many threads as the registers allow on tiles of 256 to 1024 particles: the halo's
// stencils fill threads that would be idle. A 512x512 cloth's 256 tiles issue vector instructions in 73% of a SIMD's cycles
// (16 wavefronts a tile, 2,700 each), of which half are for the halo (2.4 million projections for 1.3 million stencils). A
// solid of 17^3 cells has 24 tiles for 256 compute units, which project 155,000 times for 29,800 stencils; its SIMDs issue
// in 41% of the cycles, the rest is the latency of two wavefronts' chains, and no projection takes FP64. One launch a substep
// instead of 20 on the cloth: 89 us a substep with a launch per group (small ones in runs), 31 us in tiles; the solid
// (three launches) 125 us and 60 us; 32x32 cloth 80 and 19 us.
//
// SET: the energy types compiled in (tileSet), so that a cloth's kernel holds no registers for the FP64 solve of a
// tetrahedron.
template <int START, int SET>
__global__ void __launch_bounds__(tileThreads(SET)) xpbdTileKernel(XpbdTileArgs a)
{
    constexpr int kThreads = tileThreads(SET);
    extern __shared__ float4 tilePos[];
    __shared__ TileSegment seg[kTileMaxGroups];
    const int32_t tile = xcdContiguousBlock(blockIdx.x, a.tiles);
    const TileHeader hd = a.headers[tile];
    const int32_t t = threadIdx.x, n = hd.particleEnd - hd.particleBegin;
    const int32_t *ids = a.particles + hd.particleBegin;
    if (t < a.groups) seg[t] = a.segments[hd.segBegin + t];
    for (int32_t i = t; i < n; i += kThreads) tilePos[i] = substepStart<START>(a, ids[i]);
    __syncthreads();
    auto planesOf = [](int32_t type) { return tilePlanes(type); };
    auto load = [&](const TileSegment &s, int32_t i, float4 (&r)[4]) {
        const float4 *p = a.records + s.base + i;
        const int32_t planes = planesOf(s.type);
        r[0] = p[0];
        if (planes > 1) r[1] = p[s.count];
        if (planes > 2) r[2] = p[2 * static_cast<int64_t>(s.count)];
        if (planes > 3) r[3] = p[3 * static_cast<int64_t>(s.count)];
    };
    auto uniform = [&](int32_t g) {  // the segment in scalar registers: its type is a uniform branch
        const TileSegment s = seg[g];
        return TileSegment{__builtin_amdgcn_readfirstlane(s.type), __builtin_amdgcn_readfirstlane(s.count),
                           __builtin_amdgcn_readfirstlane(s.base)};
    };
    auto project = [&](int32_t type, const float4 (&r)[4]) {
        switch (type) {
        case kSpring: projectTileRecord<kSpring>(tilePos, r, a.invdt2, a.counters); break;
        case kStvk: projectTileRecord<kStvk>(tilePos, r, a.invdt2, a.counters); break;
        case kBending: projectTileRecord<kBending>(tilePos, r, a.invdt2, a.counters); break;
        case kAnchor: projectTileRecord<kAnchor>(tilePos, r, a.invdt2, a.counters); break;
        case kSnh:
            if constexpr (SET != kTileSurface) projectTileRecord<kSnh>(tilePos, r, a.invdt2, a.counters);
            break;
        default:
            if constexpr (SET == kTileFurther) {
                switch (type) {
                case 6: projectTileRecord<6>(tilePos, r, a.invdt2, a.counters); break;
                case 7: projectTileRecord<7>(tilePos, r, a.invdt2, a.counters); break;
                case 8: projectTileRecord<8>(tilePos, r, a.invdt2, a.counters); break;
                case 9: projectTileRecord<9>(tilePos, r, a.invdt2, a.counters); break;
                case 10: projectTileRecord<10>(tilePos, r, a.invdt2, a.counters); break;
                case 11: projectTileRecord<11>(tilePos, r, a.invdt2, a.counters); break;
                case 12: projectTileRecord<12>(tilePos, r, a.invdt2, a.counters); break;
                default: projectTileRecord<13>(tilePos, r, a.invdt2, a.counters);
                }
            }
        }
    };
    float4 next[4] = {};
    TileSegment s = uniform(0);
    if (t < s.count) load(s, t, next);
    for (int32_t g = 0; g < a.groups; ++g) {
        const TileSegment now = s;
        float4 r[4] = {next[0], next[1], next[2], next[3]};
        if (g + 1 < a.groups) {
            s = uniform(g + 1);
            if (t < s.count) load(s, t, next);
        }
        if (t < now.count) project(now.type, r);
        for (int32_t i = t + kThreads; i < now.count; i += kThreads) {
            load(now, i, r);
            project(now.type, r);
        }
        __syncthreads();
    }
    for (int32_t i = t; i < hd.owned; i += kThreads) a.out[ids[i]] = tilePos[i];
}

// A substep whose first group runs alone: the particles at its start.
template <int START>
__global__ void __launch_bounds__(256) xpbdStartKernel(XpbdTileArgs a, int32_t n)
{
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a.out[i] = substepStart<START>(a, i);
}

// The tile records of one segment per workgroup, from the stencils' records and their places in the tile.
__global__ void __launch_bounds__(256) tileRecordsKernel(XpbdArgs a, const TileSegment *__restrict__ segments,
                                                         const int64_t *__restrict__ segmentEntry,
                                                         const TileEntry *__restrict__ entries,
                                                         float4 *__restrict__ records)
{
    const TileSegment s = segments[blockIdx.x];
    const TileEntry *e = entries + segmentEntry[blockIdx.x];
    for (int32_t i = threadIdx.x; i < s.count; i += blockDim.x) {
        const int32_t k = e[i].record;
        float4 r[4] = {};
        r[0].x = __uint_as_float(static_cast<uint32_t>(e[i].place[0]) | static_cast<uint32_t>(e[i].place[1]) << 16);
        r[0].y = __uint_as_float(static_cast<uint32_t>(e[i].place[2]) | static_cast<uint32_t>(e[i].place[3]) << 16);
        switch (s.type) {
        case kSpring:
            r[0].z = a.sprP[k].x;
            r[0].w = a.sprP[k].y;
            break;
        case kAnchor: r[1] = a.ancP[k]; break;
        case kStvk:
            r[0].z = a.triC1[k].x;
            r[0].w = a.triC1[k].y;
            r[1] = a.triD[k];
            r[2] = a.triC0[k];
            break;
        case kBending:
            r[0].z = a.hinP[k].x;
            r[0].w = a.hinP[k].y;
            break;
        case kSnh:
            r[0].z = a.tetH[k];
            r[1] = a.tetD0[k];
            r[2] = a.tetD1[k];
            r[3] = a.tetD2[k];
            break;
        default:
            for (int q = 0; q < 3; ++q) r[1 + q] = a.extP[3 * static_cast<int64_t>(k) + q];
        }
        const int32_t planes = tilePlanes(s.type);
        for (int q = 0; q < planes; ++q) records[s.base + static_cast<int64_t>(q) * s.count + i] = r[q];
    }
}

// xpbd.cpp:47-70 with particleGroup.cpp:57-63: x_old = x; v += h g; x += h v (every particle).
__global__ void __launch_bounds__(256) xpbdBeginKernel(float4 *__restrict__ pos, float4 *__restrict__ vel,
                                                       float4 *__restrict__ xold, int32_t n, float h, float hgx,
                                                       float hgy, float hgz)
{
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 x = pos[i], v = vel[i];
    xold[i] = x;
    v.x += hgx;
    v.y += hgy;
    v.z += hgz;
    x.x += v.x * h;
    x.y += v.y * h;
    x.z += v.z * h;
    vel[i] = v;
    pos[i] = x;
}

// End of one substep (particleGroup.cpp:65-72, v = (x - x_old) / h) fused with the start of the next.
// The velocity lives in registers only: inside a step nothing reads vel between two substeps, and the
// end kernel writes the last substep's velocity.
__global__ void __launch_bounds__(256) xpbdBoundaryKernel(float4 *__restrict__ pos, float4 *__restrict__ xold,
                                                          int32_t n, float invhPrev, float h, float hgx, float hgy,
                                                          float hgz)
{
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 x = pos[i];
    const float4 o = xold[i];
    float3 v = make_float3((x.x - o.x) * invhPrev, (x.y - o.y) * invhPrev, (x.z - o.z) * invhPrev);
    xold[i] = x;
    v.x += hgx;
    v.y += hgy;
    v.z += hgz;
    x.x += v.x * h;
    x.y += v.y * h;
    x.z += v.z * h;
    pos[i] = x;
}

// `copy` (where not null) may be xold itself, the start of a step of one substep: each thread reads its entry before it
// writes it, so neither is __restrict__.
__global__ void __launch_bounds__(256) xpbdEndKernel(const float4 *pos, const float4 *xold, float4 *__restrict__ vel,
                                                     int32_t n, float invh, float4 *copy)
{
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 x = pos[i], o = xold[i];
    vel[i] = make_float4((x.x - o.x) * invh, (x.y - o.y) * invh, (x.z - o.z) * invh, 0.f);
    if (copy) copy[i] = x;
}

// Check hook: one projection per thread from FP64 inputs in the C-ABI parameter layout, by the device
// functions of the projection kernels (precision 0, with their FP64 fallback) or in double (1).
__global__ void xpbdCheckKernel(int type, int64_t n, const double *__restrict__ xs, const double *__restrict__ w,
                                const double *__restrict__ params, double invdt2, int precision,
                                double *__restrict__ dx)
{
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    const int ns = type == kAnchor ? 1 : type == kSpring ? 2 : type == kStvk ? 3 : 4;
    const int np = type == kStvk ? 13 : type == kSnh ? 14 : type == kAnchor ? 4 : 2;
    if (precision == 0)
        xpbdProjectRecord<true>(type, xs + i * ns * 3, w + i * ns, params + i * np, invdt2, dx + i * ns * 3);
    else
        xpbdProjectRecord<false>(type, xs + i * ns * 3, w + i * ns, params + i * np, invdt2, dx + i * ns * 3);
}

inline int blocksFor(int64_t n, int bs) { return static_cast<int>((n + bs - 1) / bs); }

template <int T>
void projectLaunch(const XpbdArgs &args, int32_t begin, int32_t end, int bs, hipStream_t stream, hipEvent_t start,
                   hipEvent_t stop)
{
    const int grid = blocksFor(end - begin, bs);
    XpbdArgs a = args;
    a.gridBlocks = grid;
    a.blockThreads = bs;
    if (start)
        hipExtLaunchKernelGGL(xpbdProjectKernel<T>, dim3(grid), dim3(bs), 0, stream, start, stop, 0, a, begin, end);
    else
        xpbdProjectKernel<T><<<grid, bs, 0, stream>>>(a, begin, end);
}

}  // namespace

hipError_t launchXpbdProject(int type, const XpbdArgs &a, int32_t begin, int32_t end, int blockSize,
                             hipStream_t stream, hipEvent_t start, hipEvent_t stop)
{
    if (end <= begin) return hipSuccess;
    if (blockSize < 64 || blockSize > 256 || blockSize % 64) return hipErrorInvalidValue;
    switch (type) {
    case kSpring: projectLaunch<kSpring>(a, begin, end, blockSize, stream, start, stop); break;
    case kStvk: projectLaunch<kStvk>(a, begin, end, blockSize, stream, start, stop); break;
    case kBending: projectLaunch<kBending>(a, begin, end, blockSize, stream, start, stop); break;
    case kSnh: projectLaunch<kSnh>(a, begin, end, blockSize, stream, start, stop); break;
    case kAnchor: projectLaunch<kAnchor>(a, begin, end, blockSize, stream, start, stop); break;
    case 6: projectLaunch<6>(a, begin, end, blockSize, stream, start, stop); break;
    case 7: projectLaunch<7>(a, begin, end, blockSize, stream, start, stop); break;
    case 8: projectLaunch<8>(a, begin, end, blockSize, stream, start, stop); break;
    case 9: projectLaunch<9>(a, begin, end, blockSize, stream, start, stop); break;
    case 10: projectLaunch<10>(a, begin, end, blockSize, stream, start, stop); break;
    case 11: projectLaunch<11>(a, begin, end, blockSize, stream, start, stop); break;
    case 12: projectLaunch<12>(a, begin, end, blockSize, stream, start, stop); break;
    case 13: projectLaunch<13>(a, begin, end, blockSize, stream, start, stop); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launchXpbdProjectRun(const XpbdArgs &a, const XpbdRun &run, hipStream_t stream, hipEvent_t start,
                                hipEvent_t stop)
{
    if (run.count < 1 || run.count > kXpbdRunMax) return hipErrorInvalidValue;
    for (int32_t r = 0; r < run.count; ++r)
        if (run.type[r] < 1 || run.type[r] > 13 || run.end[r] < run.begin[r]) return hipErrorInvalidValue;
    if (start)
        hipExtLaunchKernelGGL(xpbdProjectRunKernel, dim3(1), dim3(kXpbdRunThreads), 0, stream, start, stop, 0, a, run);
    else
        xpbdProjectRunKernel<<<1, kXpbdRunThreads, 0, stream>>>(a, run);
    return hipGetLastError();
}

hipError_t launchXpbdBegin(float4 *pos, float4 *vel, float4 *xold, int32_t n, float h, float gx, float gy, float gz,
                           hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    xpbdBeginKernel<<<blocksFor(n, 256), 256, 0, stream>>>(pos, vel, xold, n, h, gx, gy, gz);
    return hipGetLastError();
}

hipError_t launchXpbdBoundary(float4 *pos, float4 *xold, int32_t n, float invhPrev, float h, float gx, float gy,
                              float gz, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    xpbdBoundaryKernel<<<blocksFor(n, 256), 256, 0, stream>>>(pos, xold, n, invhPrev, h, gx, gy, gz);
    return hipGetLastError();
}

hipError_t launchXpbdEnd(const float4 *pos, const float4 *xold, float4 *vel, int32_t n, float invh,
                         hipStream_t stream, float4 *copy)
{
    if (n <= 0) return hipSuccess;
    xpbdEndKernel<<<blocksFor(n, 256), 256, 0, stream>>>(pos, xold, vel, n, invh, copy);
    return hipGetLastError();
}

hipError_t launchXpbdTiles(const XpbdTileArgs &a, int start, int set, int32_t maxParticles, hipStream_t stream)
{
    if (a.tiles < 1 || a.groups < 1 || a.groups > kTileMaxGroups || maxParticles > kTileMaxParticles || start < 0 ||
        start > 2 || set < kTileSurface || set > kTileFurther)
        return hipErrorInvalidValue;
    const size_t lds = sizeof(float4) * maxParticles;
    auto launch = [&](auto kernel) { kernel<<<a.tiles, tileThreads(set), lds, stream>>>(a); };
    auto withStart = [&](auto set) {
        constexpr int S = decltype(set)::value;
        if (start == 0)
            launch(xpbdTileKernel<0, S>);
        else if (start == 1)
            launch(xpbdTileKernel<1, S>);
        else
            launch(xpbdTileKernel<2, S>);
    };
    if (set == kTileSurface)
        withStart(std::integral_constant<int, kTileSurface>{});
    else if (set == kTileFive)
        withStart(std::integral_constant<int, kTileFive>{});
    else
        withStart(std::integral_constant<int, kTileFurther>{});
    return hipGetLastError();
}

hipError_t launchXpbdStart(const XpbdTileArgs &a, int start, int32_t n, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    if (start == 1)
        xpbdStartKernel<1><<<blocksFor(n, 256), 256, 0, stream>>>(a, n);
    else if (start == 2)
        xpbdStartKernel<2><<<blocksFor(n, 256), 256, 0, stream>>>(a, n);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launchTileRecords(const XpbdArgs &a, const TileSegment *segments, int32_t nSegments,
                             const int64_t *segmentEntry, const TileEntry *entries, float4 *records, hipStream_t stream)
{
    if (nSegments <= 0) return hipSuccess;
    tileRecordsKernel<<<nSegments, 256, 0, stream>>>(a, segments, segmentEntry, entries, records);
    return hipGetLastError();
}

hipError_t launchXpbdProjectCheck(int type, int64_t n, const double *xs, const double *w, const double *params,
                                  double invdt2, int precision, double *dx, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    xpbdCheckKernel<<<blocksFor(n, 64), 64, 0, stream>>>(type, n, xs, w, params, invdt2, precision, dx);
    return hipGetLastError();
}

}  // namespace spgvbd
