// Kernels of the learned warm start: a per-vertex MLP (24 -> 128 -> 128 -> 128 -> 3, SiLU) with BF16
// weights and activations on CDNA4 matrix cores (v_mfma_f32_16x16x32_bf16), FP32 accumulation: inference, the
// gradient of a batch (forward and backward in one kernel), and the update of the weights.
//
// MFMA operand layout (16x16x32): lane l holds row (l % 16) of A and row (l % 16) of B at K offsets 8 (l / 16) .. +7
// (the same K split for both operands, so the products pair up); the accumulator holds C[4 (l / 16) + r][l % 16],
// r = 0 .. 3.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "mlp_device.h"

namespace spgvbd {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ float sigmoidf(float z) { return 1.0f / (1.0f + __expf(-z)); }
__device__ __forceinline__ float silu(float z) { return z * sigmoidf(z); }

__device__ __forceinline__ bf16x8 zeroFrag()
{
    bf16x8 z;
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i] = static_cast<__bf16>(0.0f);
    return z;
}

// ------------------------------------------------------------------------------------------------
// Fused inference: all four layers in registers, one wavefront per kNT x 16 rows.
//
// Each layer is computed transposed, H^T = W X^T: the weights are the MFMA A operand (M = output
// features) and the rows are the B operand (N = 16 rows per tile), so the accumulator of tile i holds,
// in lane l, output features 16 i + 4 (l / 16) + r (r = 0..3) of row l % 16. The B fragment a layer
// needs for K step kk is, in lane l, 8 features of row l % 16; the lane already holds features
// 32 kk + 4 q + r (tile 2 kk) and 32 kk + 16 + 4 q + r (tile 2 kk + 1), q = l / 16. Using exactly those 8
// (a fixed permutation of K inside the step) needs no data exchange between lanes; the weight
// fragments are stored with the same permutation (mlpFragKernel), so the products pair up. The input
// layer uses the plain order: lane l holds features 8 q .. 8 q + 7.
// Weight fragments (76 KB) and biases are staged in LDS once per persistent workgroup.
constexpr int kFragL1 = 0, kFragL2 = 512, kFragL3 = 2560, kFragL4 = 4608, kFragTotal = 4864;
constexpr int kNT = 4;  // 16-row tiles per wavefront task (each weight fragment read from LDS feeds kNT MFMAs)
constexpr int kTaskRows = 16 * kNT;
constexpr int kBiasTotal = 3 * kMlpHidden + kMlpOutPad;

// The backward pass multiplies by the transposed weights: A holds W^T (M = input features of the layer), K the layer's
// outputs in the permuted order of the hidden layers (the last layer's 32 padded outputs in the plain order).
constexpr int kFragT2 = kFragTotal, kFragT3 = kFragT2 + 2048, kFragT4 = kFragT3 + 2048, kFragAll = kFragT4 + 512;

// Place of (row, k) of an operand in its fragments (in bf16 values): tiles of 16 rows, K steps of 32. In the permuted
// order value p of lane quarter q holds k = 32 kk + (p < 4 ? 4 q + p : 16 + 4 q + p - 4), in the plain one 8 q + p.
__device__ __forceinline__ int fragPlace(int row, int k, int ksteps, bool permuted)
{
    const int w = k & 31;
    const int q = permuted ? (w & 15) >> 2 : w >> 3, p = permuted ? (w & 3) + (w & 16) / 4 : w & 7;
    return (((row >> 4) * ksteps + (k >> 5)) * 64 + q * 16 + (row & 15)) * 8 + p;
}

// The padded master layout: per layer W (out x in, row-major), then its biases.
constexpr int kW1 = 0, kB1 = kW1 + kMlpHidden * kMlpIn, kW2 = kB1 + kMlpHidden, kB2 = kW2 + kMlpHidden * kMlpHidden,
              kW3 = kB2 + kMlpHidden, kB3 = kW3 + kMlpHidden * kMlpHidden, kW4 = kB3 + kMlpHidden,
              kB4 = kW4 + kMlpOutPad * kMlpHidden;
static_assert(kB4 + kMlpOutPad == kMlpPadded, "padded parameter count");

// Writes parameter k of the padded layout, if it is a weight, to its places in the fragments.
__device__ __forceinline__ void storeFrags(int k, float value, __bf16 *frag)
{
    const __bf16 v = static_cast<__bf16>(value);
    if (k < kB1) {
        frag[8 * kFragL1 + fragPlace(k / kMlpIn, k % kMlpIn, 1, false)] = v;
    } else if ((k >= kW2 && k < kB2) || (k >= kW3 && k < kB3)) {
        const bool second = k < kB2;
        const int e = k - (second ? kW2 : kW3), o = e / kMlpHidden, i = e % kMlpHidden;
        frag[8 * (second ? kFragL2 : kFragL3) + fragPlace(o, i, 4, true)] = v;
        frag[8 * (second ? kFragT2 : kFragT3) + fragPlace(i, o, 4, true)] = v;
    } else if (k >= kW4 && k < kB4) {
        const int e = k - kW4, o = e / kMlpHidden, i = e % kMlpHidden;
        if (o < 16) frag[8 * kFragL4 + fragPlace(o, i, 4, true)] = v;
        frag[8 * kFragT4 + fragPlace(i, o, 1, false)] = v;
    }
}

__global__ void __launch_bounds__(256) mlpFragKernel(const float *__restrict__ p, __bf16 *__restrict__ frag)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < kMlpPadded) storeFrags(k, p[k], frag);
}

__device__ __forceinline__ void hiddenEpilogue(const f32x4 (&acc)[8][kNT], const float *bias, int q,
                                               bf16x8 (&hb)[4][kNT])
{
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                hb[kk][nt][r] = static_cast<__bf16>(silu(acc[2 * kk][nt][r] + bias[32 * kk + 4 * q + r]));
                hb[kk][nt][4 + r] = static_cast<__bf16>(silu(acc[2 * kk + 1][nt][r] + bias[32 * kk + 16 + 4 * q + r]));
            }
}

__device__ __forceinline__ void hiddenLayer(const bf16x8 *wl, const bf16x8 (&hb)[4][kNT], int lane,
                                            f32x4 (&acc)[8][kNT])
{
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) acc[i][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const bf16x8 a = wl[(i * 4 + kk) * 64 + lane];
#pragma unroll
            for (int nt = 0; nt < kNT; ++nt) acc[i][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, hb[kk][nt], acc[i][nt], 0, 0, 0);
        }
    }
}

__global__ void __launch_bounds__(256) mlpInferKernel(const float *__restrict__ f, int n, const float *__restrict__ mean,
                                                      const float *__restrict__ invStd, const bf16x8 *__restrict__ frag,
                                                      const float *__restrict__ b1, const float *__restrict__ b2,
                                                      const float *__restrict__ b3, const float *__restrict__ b4,
                                                      float *__restrict__ y, int ldy)
{
    __shared__ bf16x8 wl[kFragTotal];
    __shared__ float bl[kBiasTotal];
    __shared__ float nl[2 * kMlpIn];
    for (int i = threadIdx.x; i < kFragTotal; i += blockDim.x) wl[i] = frag[i];
    for (int i = threadIdx.x; i < kMlpHidden; i += blockDim.x) {
        bl[i] = b1[i];
        bl[kMlpHidden + i] = b2[i];
        bl[2 * kMlpHidden + i] = b3[i];
    }
    if (threadIdx.x < kMlpOutPad) bl[3 * kMlpHidden + threadIdx.x] = b4[threadIdx.x];
    if (threadIdx.x < kMlpIn) {
        const bool real = threadIdx.x < kMlpFeatures;
        nl[threadIdx.x] = real ? mean[threadIdx.x] : 0.f;
        nl[kMlpIn + threadIdx.x] = real ? invStd[threadIdx.x] : 0.f;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, q = lane >> 4, r16 = lane & 15;
    const int ntask = (n + kTaskRows - 1) / kTaskRows;
    const int waves = gridDim.x * (blockDim.x >> 6);
    for (int task = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); task < ntask; task += waves) {
        // compiler-level memory barrier: keeps the weight fragments in LDS (re-read per task) instead of
        // hoisting all 76 of them out of the loop into registers
        asm volatile("" ::: "memory");
        const int row0 = task * kTaskRows;
        bf16x8 hb[4][kNT];
        // standardised inputs, plain K order; features 24..31 and rows past n are zero
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) {
            const int row = row0 + 16 * nt + r16;
            bf16x8 x = zeroFrag();
            if (row < n && q < 3) {
                const float4 *src = reinterpret_cast<const float4 *>(f + static_cast<int64_t>(row) * kMlpFeatures + 8 * q);
                const float4 u0 = src[0], u1 = src[1];
                const float u[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
                for (int p = 0; p < 8; ++p) x[p] = static_cast<__bf16>((u[p] - nl[8 * q + p]) * nl[kMlpIn + 8 * q + p]);
            }
            hb[0][nt] = x;
            hb[1][nt] = zeroFrag();
            hb[2][nt] = zeroFrag();
            hb[3][nt] = zeroFrag();
        }
        f32x4 acc[8][kNT];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const bf16x8 a = wl[kFragL1 + i * 64 + lane];
#pragma unroll
            for (int nt = 0; nt < kNT; ++nt)
                acc[i][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, hb[0][nt], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        }
        hiddenEpilogue(acc, bl, q, hb);
        hiddenLayer(wl + kFragL2, hb, lane, acc);
        hiddenEpilogue(acc, bl + kMlpHidden, q, hb);
        hiddenLayer(wl + kFragL3, hb, lane, acc);
        hiddenEpilogue(acc, bl + 2 * kMlpHidden, q, hb);
        f32x4 o[kNT];
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) o[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const bf16x8 a = wl[kFragL4 + kk * 64 + lane];
#pragma unroll
            for (int nt = 0; nt < kNT; ++nt) o[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, hb[kk][nt], o[nt], 0, 0, 0);
        }
        if (q == 0) {
#pragma unroll
            for (int nt = 0; nt < kNT; ++nt) {
                const int row = row0 + 16 * nt + r16;
                if (row < n)
#pragma unroll
                    for (int r = 0; r < kMlpOut; ++r) y[static_cast<int64_t>(row) * ldy + r] = o[nt][r] + bl[3 * kMlpHidden + r];
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// The gradient of a batch: forward and backward of 64 rows per workgroup, 16 per wavefront, in one kernel.
//
// The layers run as in inference, rows as the B operand, activations and their gradients from layer to layer in
// registers (SiLU' of the pre-activations stays there for the way back). A weight gradient sums over rows, dW = dZ^T H, so every
// wavefront also stores its activations and dZ to LDS, features by rows, and the workgroup multiplies them with the 64
// rows as K. Its sums over the row blocks it takes go to its own part of `partial`; mlpUpdateKernel adds the parts up in
// a fixed order.
//
// What bounds it: latency. A minibatch of 4096 rows is 64 workgroups of one wavefront a SIMD, each with 224 MFMAs a row block
// (148 forward and back, 76 for its part of the weight gradients) and 2,800 vector instructions in a chain: a quarter of its
// cycles issue one. As separate products (eleven of them, and 12 further launches) a minibatch took 420 us, most of it the
// weight gradients' serial K loop over the batch in four workgroups. Now it is this kernel, 24 us, and mlpUpdateKernel, 7 us.
constexpr int kTrainRows = 64;
constexpr int kRowStride = kTrainRows + 8;  // bf16 per LDS feature row: 16-byte aligned, no bank conflicts
constexpr int kSplit = 4;                   // threads that share a parameter's partial sums in mlpUpdateKernel

// out[feature][row] of the tiles of v: this lane's features 16 i + 4 q + r of its row
template <int TILES>
__device__ __forceinline__ void storeRows(const f32x4 (&v)[TILES], __bf16 *out, int q, int row)
{
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(16 * i + 4 * q + r) * kRowStride + row] = static_cast<__bf16>(v[i][r]);
}

// the tiles as B fragments of the next product (permuted K order)
__device__ __forceinline__ void toFrags(const f32x4 (&v)[8], bf16x8 (&b)[4])
{
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            b[kk][r] = static_cast<__bf16>(v[2 * kk][r]);
            b[kk][4 + r] = static_cast<__bf16>(v[2 * kk + 1][r]);
        }
}

// The fragments as a buffer: a load is a scalar offset and the lane's, so the 148 loads of a row block need one address
// register (as pointers each kept two of its own, and they spilled).
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
__device__ __forceinline__ bf16x8 fragAt(__amdgpu_buffer_rsrc_t w, int f, int lane)
{
    return __builtin_bit_cast(bf16x8, static_cast<u32x4>(__builtin_amdgcn_raw_buffer_load_b128(w, lane * 16, f * 1024, 0)));
}

// acc = W b over 128 K: 8 tiles of 16 features, fragments in global memory, half of them loaded at once. The
// compiler-level barrier keeps one product's loads from being issued with another's.
__device__ __forceinline__ void product128(__amdgpu_buffer_rsrc_t w, int first, const bf16x8 (&b)[4], int lane, f32x4 (&acc)[8])
{
    asm volatile("" ::: "memory");
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        bf16x8 f[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) f[k] = fragAt(w, first + 16 * half + k, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f32x4 &c = acc[4 * half + i];
            c = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[4 * i + kk], b[kk], c, 0, 0, 0);
        }
    }
}

// v plus its value N lanes further round the 16 lanes of a row of the wavefront
template <int N>
__device__ __forceinline__ float addRotated(float v)
{
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x120 + N, 0xf, 0xf, true));
}

// Sums over the 16 rows of this wavefront (its lanes of one q), added to its own bias sums of the layer.
template <int TILES>
__device__ __forceinline__ void addBias(const f32x4 (&v)[TILES], float *sums, int q, int row16)
{
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
        f32x4 t;
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] = addRotated<8>(addRotated<4>(addRotated<2>(addRotated<1>(v[i][r]))));
        if (row16 == 0) {
            f32x4 *s = reinterpret_cast<f32x4 *>(sums + 16 * i + 4 * q);
            *s += t;
        }
    }
}

// D H^T over the workgroup's rows, output features 16 tile0 .. and input features 16 ntile0 .., to (add: onto) out.
template <int MT, int NT>
__device__ __forceinline__ void weightGrad(const __bf16 *D, int tile0, const __bf16 *H, int ntile0, int q, int r16, int in,
                                           float *out, bool add)
{
    f32x4 acc[MT][NT] = {};
#pragma unroll
    for (int ks = 0; ks < kTrainRows / 32; ++ks) {
        bf16x8 d[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
            d[m] = *reinterpret_cast<const bf16x8 *>(D + (16 * (tile0 + m) + r16) * kRowStride + 32 * ks + 8 * q);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const bf16x8 h = *reinterpret_cast<const bf16x8 *>(H + (16 * (ntile0 + n) + r16) * kRowStride + 32 * ks + 8 * q);
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d[m], h, acc[m][n], 0, 0, 0);
        }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float *o = out + (16 * (tile0 + m) + 4 * q + r) * in + 16 * (ntile0 + n) + r16;
                *o = add ? *o + acc[m][n][r] : acc[m][n][r];
            }
}

__global__ void __launch_bounds__(256, 1) mlpTrainKernel(MlpTrainArgs a)
{
    __shared__ __align__(16) __bf16 ht[3][kMlpHidden * kRowStride];
    __shared__ __align__(16) __bf16 dt[3][kMlpHidden * kRowStride];
    __shared__ __align__(16) __bf16 xt[kMlpIn * kRowStride];
    __shared__ __align__(16) __bf16 yt[16 * kRowStride];
    __shared__ __align__(16) float bias[4][3 * kMlpHidden + 16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, q = lane >> 4, r16 = lane & 15;
    for (int i = lane; i < 3 * kMlpHidden + 16; i += 64) bias[wave][i] = 0.f;  // a wavefront's own sums
    // raw buffer of 32-bit elements
    const __amdgpu_buffer_rsrc_t frag =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(a.frag), 0, kFragAll * sizeof(bf16x8), 0x00027000);
    const float *b1 = a.params + kB1, *b2 = a.params + kB2, *b3 = a.params + kB3, *b4 = a.params + kB4;
    float *out = a.partial + static_cast<int64_t>(blockIdx.x) * kMlpPadded;
    double se = 0.0;
    for (int block = blockIdx.x; block < a.rowBlocks; block += gridDim.x) {
        // compiler-level memory barrier: the weight fragments are read again for every row block, not kept in registers
        asm volatile("" ::: "memory");
        const int lrow = wave * 16 + r16, row = block * kTrainRows + lrow;
        const int src = row < a.n ? (a.index ? a.index[row] : row) : -1;
        bf16x8 x = zeroFrag();
        if (src >= 0 && q < 3) {
            const float4 *f = reinterpret_cast<const float4 *>(a.features + static_cast<int64_t>(src) * kMlpFeatures + 8 * q);
            const float4 u0 = f[0], u1 = f[1];
            const float u[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
            for (int p = 0; p < 8; ++p) x[p] = static_cast<__bf16>((u[p] - a.mean[8 * q + p]) * a.invStd[8 * q + p]);
        }
#pragma unroll
        for (int p = 0; p < 8; ++p) xt[(8 * q + p) * kRowStride + lrow] = x[p];
        // forward: z the pre-activations (then SiLU' of them, for the way back), h the activations
        auto activate = [&](f32x4 (&z)[8], const float *b, __bf16 *out, bf16x8 (&next)[4]) {
            f32x4 h[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const f32x4 bi = *reinterpret_cast<const f32x4 *>(b + 16 * i + 4 * q);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float v = z[i][r] + bi[r], sg = sigmoidf(v);
                    h[i][r] = v * sg;
                    z[i][r] = sg * (1.0f + v * (1.0f - sg));
                }
            }
            storeRows(h, out, q, lrow);
            toFrags(h, next);
        };
        f32x4 z1[8], z2[8], z3[8];
        bf16x8 hb[4];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            z1[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fragAt(frag, kFragL1 / 64 + i, lane), x, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        activate(z1, b1, ht[0], hb);
        product128(frag, kFragL2 / 64, hb, lane, z2);
        activate(z2, b2, ht[1], hb);
        product128(frag, kFragL3 / 64, hb, lane, z3);
        activate(z3, b3, ht[2], hb);
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
            y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fragAt(frag, kFragL4 / 64 + kk, lane), hb[kk], y, 0, 0, 0);
        // dY = 2 (y - t) / n on the real rows and outputs (features 0 .. 2: lanes of q 0), zero elsewhere
        f32x4 dy[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
        bf16x8 dyb = zeroFrag();
        if (src >= 0 && q == 0) {
            float e = 0.f;
#pragma unroll
            for (int r = 0; r < kMlpOut; ++r) {
                const float d = y[r] + b4[r] - a.targets[static_cast<int64_t>(src) * kMlpOut + r];
                e += d * d;
                dy[0][r] = 2.0f * d / static_cast<float>(a.n);
                dyb[r] = static_cast<__bf16>(dy[0][r]);
            }
            se += static_cast<double>(e);
        }
        storeRows(dy, yt, q, lrow);
        addBias(dy, bias[wave] + 3 * kMlpHidden, q, r16);
        // backward: dZ = (W^T dZ of the layer above) SiLU'
        auto back = [&](f32x4 (&d)[8], const f32x4 (&z)[8], __bf16 *out, float *sums, bf16x8 (&next)[4]) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) d[i][r] *= z[i][r];
            storeRows(d, out, q, lrow);
            toFrags(d, next);
            addBias(d, sums, q, r16);
        };
        f32x4 d[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            d[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fragAt(frag, kFragT4 / 64 + i, lane), dyb, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        back(d, z3, dt[2], bias[wave] + 2 * kMlpHidden, hb);
        product128(frag, kFragT3 / 64, hb, lane, d);
        back(d, z2, dt[1], bias[wave] + kMlpHidden, hb);
        product128(frag, kFragT2 / 64, hb, lane, d);
        back(d, z1, dt[0], bias[wave], hb);
        __syncthreads();
        // wavefront w: output features 32 w .. of the hidden layers, input features 32 w .. of the last
        const bool add = block != static_cast<int>(blockIdx.x);
        weightGrad<1, 2>(yt, 0, ht[2], 2 * wave, q, r16, kMlpHidden, out + kW4, add);
        weightGrad<2, 8>(dt[2], 2 * wave, ht[1], 0, q, r16, kMlpHidden, out + kW3, add);
        weightGrad<2, 8>(dt[1], 2 * wave, ht[0], 0, q, r16, kMlpHidden, out + kW2, add);
        weightGrad<2, 2>(dt[0], 2 * wave, xt, 0, q, r16, kMlpIn, out + kW1, add);
        __syncthreads();
    }
    for (int i = t; i < 3 * kMlpHidden + 16; i += blockDim.x) {
        const float v = ((bias[0][i] + bias[1][i]) + bias[2][i]) + bias[3][i];
        const int layer = i / kMlpHidden, o = i % kMlpHidden;
        out[(layer == 0 ? kB1 : layer == 1 ? kB2 : layer == 2 ? kB3 : kB4) + o] = v;
    }
    for (int o = 32; o > 0; o >>= 1) se += __shfl_down(se, o, 64);
    __shared__ double waveSe[4];
    if (lane == 0) waveSe[wave] = se;
    __syncthreads();
    if (t == 0) a.lossPartial[blockIdx.x] = ((waveSe[0] + waveSe[1]) + waveSe[2]) + waveSe[3];
}

// Whether parameter k of the padded layout has partial sums: outputs past the 16 that are computed have none.
__device__ __forceinline__ bool trained(int k)
{
    return k < kW4 + 16 * kMlpHidden || (k >= kB4 && k < kB4 + 16);
}

// The gradient from the workgroups' partial sums (kSplit threads a parameter, each over a contiguous range of
// workgroups, then in order), then, with ADAM (Kingma & Ba 2015), the new FP32 parameter and its places in the
// operand fragments. The first workgroup also adds the batch's squared error to *loss.
//
// What bounds it: 10.6 MB of partial sums for 4096 rows, from the Infinity Cache.
template <bool ADAM>
__global__ void __launch_bounds__(256) mlpUpdateKernel(MlpUpdateArgs a)
{
    __shared__ float part[kSplit][64];
    const int t = threadIdx.x & 63, seg = threadIdx.x >> 6, k = blockIdx.x * 64 + t;
    float v = 0.f;
    if (k < kMlpPadded && trained(k)) {
        const int each = (a.parts + kSplit - 1) / kSplit, b = seg * each, e = min(b + each, a.parts);
        const float *p = a.partial + static_cast<int64_t>(b) * kMlpPadded + k;
        int i = b;
        for (; i + 8 <= e; i += 8, p += 8 * kMlpPadded) {
            float u[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) u[j] = p[j * kMlpPadded];
#pragma unroll
            for (int j = 0; j < 8; ++j) v += u[j];
        }
        for (; i < e; ++i, p += kMlpPadded) v += *p;
    }
    part[seg][t] = v;
    __syncthreads();
    if (seg == 0 && k < kMlpPadded) {
        float g = part[0][t];
#pragma unroll
        for (int j = 1; j < kSplit; ++j) g += part[j][t];
        if constexpr (ADAM) {
            const float mi = a.b1 * a.m[k] + (1.f - a.b1) * g;
            const float vi = a.b2 * a.v[k] + (1.f - a.b2) * g * g;
            a.m[k] = mi;
            a.v[k] = vi;
            const float w = a.params[k] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
            a.params[k] = w;
            storeFrags(k, w, static_cast<__bf16 *>(a.frag));
        } else {
            a.grad[k] = g;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        double s = 0.0;
        for (int i = 0; i < a.parts; ++i) s += a.lossPartial[i];
        *a.loss += s;
    }
}

inline int blocksFor(int64_t n, int bs) { return static_cast<int>((n + bs - 1) / bs); }

}  // namespace

hipError_t launchMlpTrain(const MlpTrainArgs &a, int parts, hipStream_t stream)
{
    if (a.n <= 0 || parts <= 0 || a.rowBlocks <= 0) return hipErrorInvalidValue;
    mlpTrainKernel<<<parts, 256, 0, stream>>>(a);
    return hipGetLastError();
}

int mlpTrainBlocks(int64_t rows) { return static_cast<int>((rows + kTrainRows - 1) / kTrainRows); }

hipError_t launchMlpUpdate(const MlpUpdateArgs &a, bool adam, hipStream_t stream)
{
    const int grid = blocksFor(kMlpPadded, 64);
    if (adam)
        mlpUpdateKernel<true><<<grid, 256, 0, stream>>>(a);
    else
        mlpUpdateKernel<false><<<grid, 256, 0, stream>>>(a);
    return hipGetLastError();
}

hipError_t launchMlpFrag(const float *params, void *frag, hipStream_t stream)
{
    mlpFragKernel<<<blocksFor(kMlpPadded, 256), 256, 0, stream>>>(params, static_cast<__bf16 *>(frag));
    return hipGetLastError();
}

size_t mlpFragBytes() { return sizeof(bf16x8) * kFragAll; }

hipError_t launchMlpInfer(const float *f, int n, const float *mean, const float *invStd, const void *frag,
                          const float *b1, const float *b2, const float *b3, const float *b4, float *y, int ldy,
                          int maxBlocks, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    if (ldy < kMlpOut) return hipErrorInvalidValue;
    const int tasks = (n + kTaskRows - 1) / kTaskRows;
    const int grid = std::max(1, std::min((tasks + 3) / 4, maxBlocks));
    mlpInferKernel<<<grid, 256, 0, stream>>>(f, n, mean, invStd, static_cast<const bf16x8 *>(frag), b1, b2, b3, b4, y,
                                             ldy);
    return hipGetLastError();
}

}  // namespace spgvbd
