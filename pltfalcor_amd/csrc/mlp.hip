// Learned BSDF surrogate (no counterpart in the reference): a 22-128-128-128-16 ReLU MLP whose
// forward pass, backward pass and Adam update run on CDNA4 matrix cores.
//
// Every MFMA operand is bf16 and contiguous along the contracted dimension, so that a fragment (8
// consecutive k of one row) is one 16 B load. Accumulation is FP32 (v_mfma_f32_16x16x32_bf16); master
// weights and Adam moments are FP32; weight gradients are partial sums per workgroup reduced in a
// fixed order (the result does not depend on scheduling).
//
// Layers (parameter order of plt_surrogate_params): W1 [128 x 22], b1 [128], W2 [128 x 128], b2,
// W3 [128 x 128], b3, W4 [16 x 128], b4 [16] = 38,032 FP32 values. Inputs are padded to 32
// features with zeros (W1's padding columns stay zero).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <type_traits>
#include <vector>
#include "plt_internal.hpp"
#include "surrogate.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace plt {
namespace mlp {

constexpr int kIn = 22, kInPad = 32, kHid = 128, kOut = 16, kOutPad = 32;
constexpr int kParams = kHid * kIn + kHid + 2 * (kHid * kHid + kHid) + kOut * kHid + kOut;  // 38,032
static_assert(kParams == 38032, "parameter count");

// ---------------------------------------------------------------------------------------
// Plain NT GEMM, C[M x N] = A[M x K] * Bt[N x K]^T (plt_mlp_gemm_nt).
// ---------------------------------------------------------------------------------------
struct GemmArgs {
    const __bf16* A;   // [M x K]
    const __bf16* Bt;  // [N x K]
    int M, N, K;
    float* C;
};

constexpr int kTile = 64, kKStep = 32, kLdsRow = kKStep + 8;  // +8 bf16 per row breaks bank conflicts
constexpr int kGemmThreads = 256;

__global__ void __launch_bounds__(kGemmThreads) gemm_nt_kernel(GemmArgs g) {
    __shared__ __bf16 As[kTile * kLdsRow];
    __shared__ __bf16 Bs[kTile * kLdsRow];
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int m0 = blockIdx.y * kTile, n0 = blockIdx.x * kTile;
    // staging: thread t copies 8 bf16 of row t/4, k offset 8*(t%4), of both tiles
    const int sr = t >> 2, sk = (t & 3) * 8;
    // wave w computes rows 32*(w/2)..+31 and columns 32*(w%2)..+31 of the tile: 2 x 2 MFMA blocks
    const int wr = 32 * (wave >> 1), wc = 32 * (wave & 1);
    const int fr = lane & 15, fk = 8 * (lane >> 4);
    f32x4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < g.K; k0 += kKStep) {
        bf16x8 va = {}, vb = {};
        if (m0 + sr < g.M) va = *reinterpret_cast<const bf16x8*>(g.A + size_t(m0 + sr) * g.K + k0 + sk);
        if (n0 + sr < g.N) vb = *reinterpret_cast<const bf16x8*>(g.Bt + size_t(n0 + sr) * g.K + k0 + sk);
        *reinterpret_cast<bf16x8*>(As + sr * kLdsRow + sk) = va;
        *reinterpret_cast<bf16x8*>(Bs + sr * kLdsRow + sk) = vb;
        __syncthreads();
        bf16x8 fa[2], fb[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) fa[a] = *reinterpret_cast<const bf16x8*>(As + (wr + 16 * a + fr) * kLdsRow + fk);
#pragma unroll
        for (int b = 0; b < 2; ++b) fb[b] = *reinterpret_cast<const bf16x8*>(Bs + (wc + 16 * b + fr) * kLdsRow + fk);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[a], fb[b], acc[a][b], 0, 0, 0);
        __syncthreads();
    }
    // D layout of a 16 x 16 block: lane holds rows 4*(lane/16) + r (r = 0..3) of column lane%16
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = m0 + wr + 16 * a + 4 * (lane >> 4) + r;
                const int j = n0 + wc + 16 * b + (lane & 15);
                if (i < g.M && j < g.N) g.C[size_t(i) * g.N + j] = acc[a][b][r];
            }
}

int gemm(const GemmArgs& g, hipStream_t st) {
    if (g.M <= 0 || g.N <= 0 || g.K <= 0 || g.K % kKStep)
        return set_error(PLT_EINVAL, "mlp gemm: shapes must be multiples of 32 (K) and 8 (leading dimensions)");
    const dim3 grid((g.N + kTile - 1) / kTile, (g.M + kTile - 1) / kTile);
    hipLaunchKernelGGL(gemm_nt_kernel, grid, dim3(kGemmThreads), 0, st, g);
    return check_launch("gemm_nt_kernel");
}

// ---------------------------------------------------------------------------------------
// Fused inference: all four layers in one persistent kernel. A workgroup of four waves loads
// the bf16 weights once into registers -- wave w holds the fragments of output features
// 32w..32w+31 of layers 1-3 and all of layer 4 -- and then walks 64-sample tiles. Each product
// is computed transposed, out[feature x sample] = W x in^T: the weights are the MFMA's A operand
// (registers), the tile's activations the B operand (LDS rows of 8 consecutive features), and the
// bias is the accumulator's initial value. The D layout then gives each lane four consecutive
// features of one sample, written to the next layer's LDS rows as one 8-byte store, and the
// output layer's four consecutive outputs of a sample are one Mueller row.
// ---------------------------------------------------------------------------------------
constexpr int kFTile = 64, kFThreads = 256;
constexpr int kXRow = kInPad + 8, kHRow = kHid + 8;  // padded LDS rows (bank spread, 16 B aligned)

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// ReLU of an MFMA result as one integer max on its bits: negative floats (sign bit set, -0
// included) read as negative integers and become +0; fmaxf would add a NaN canonicalisation.
__device__ __forceinline__ float relu_bits(float x) { return __int_as_float(max(__float_as_int(x), 0)); }

// sinh for the decode: (e^y - e^-y) / 2 from one hardware exponential where |y| > 1/2, the Taylor
// series through y^9 below (relative error under 1e-8 there, so no cancellation).
__device__ __forceinline__ float sinh_fast(float y) {
    const float a = fabsf(y);
    if (a > 0.5f) {
        const float e = __expf(a);
        return copysignf(0.5f * (e - 1.f / e), y);
    }
    const float y2 = y * y;
    return y * (1.f + y2 * (1.f / 6.f + y2 * (1.f / 120.f + y2 * (1.f / 5040.f + y2 * (1.f / 362880.f)))));
}

// With Sout: instead of writing the raw outputs, each sample inside the training box
// (stats[32..54) / [54..76)) has its Mueller matrix decoded (M00 = exp(y0), Mk = M00 sinh(yk)
// after de-standardising with stats[0..16) / [16..32)) and applied to Sin; samples outside the box
// are left for the exact pass.
// With n_dev, the row count is min(*n_dev, n), read from device memory (a count a previous kernel
// on the stream produced), so the launch needs no host synchronisation.
__global__ void __launch_bounds__(kFThreads) mlp_infer_kernel(int n, const float* __restrict__ X, const __bf16* __restrict__ W1,
                                                              const __bf16* __restrict__ W2, const __bf16* __restrict__ W3,
                                                              const __bf16* __restrict__ W4, const float* __restrict__ params,
                                                              float* __restrict__ Y, const float* __restrict__ stats,
                                                              const float* __restrict__ Sin, float* __restrict__ Sout,
                                                              const uint32_t* __restrict__ n_dev) {
    if (n_dev) n = int(min(uint32_t(n), *n_dev));
    __shared__ __bf16 xs[kFTile * kXRow];
    __shared__ __bf16 ha[kFTile * kHRow];
    __shared__ __bf16 hb[kFTile * kHRow];
    __shared__ int outside[kFTile];  // sample outside the training box (apply mode)
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int fr = lane & 15, fg = lane >> 4, fk = 8 * fg;
    // register-resident A fragments: (feature block cb, k block kb) = W[feature][32 kb + fk .. +7]
    bf16x8 w1[2], w2[2][4], w3[2][4], w4[4];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        const int col = 32 * w + 16 * cb + fr;
        w1[cb] = *reinterpret_cast<const bf16x8*>(W1 + size_t(col) * kInPad + fk);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            w2[cb][kb] = *reinterpret_cast<const bf16x8*>(W2 + size_t(col) * kHid + 32 * kb + fk);
            w3[cb][kb] = *reinterpret_cast<const bf16x8*>(W3 + size_t(col) * kHid + 32 * kb + fk);
        }
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) w4[kb] = *reinterpret_cast<const bf16x8*>(W4 + size_t(fr) * kHid + 32 * kb + fk);
    // the biases of the lane's D rows: features 32w + 16cb + 4fg + r, outputs 4fg + r
    const float* b1 = params + kHid * kIn;
    const float* b2 = b1 + kHid + kHid * kHid;
    const float* b3 = b2 + kHid + kHid * kHid;
    const float* b4 = b3 + kHid + kOut * kHid;
    f32x4 c1[2], c2[2], c3[2], c4;
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int f = 32 * w + 16 * cb + 4 * fg + r;
            c1[cb][r] = b1[f];
            c2[cb][r] = b2[f];
            c3[cb][r] = b3[f];
        }
#pragma unroll
    for (int r = 0; r < 4; ++r) c4[r] = b4[4 * fg + r];
    // staging: thread t always loads input features 2p, 2p + 1 (p = t % 16) of rows t / 16 + 16 j
    // (j < 4) as one 8-byte load, so its box bounds are loaded once; the pair is one 4-byte LDS store
    const int sp = t & 15, sr = t >> 4;
    const bool inPair = 2 * sp < kIn;  // kIn is even: a pair is all in or all padding
    float blo[2] = {0.f, 0.f}, bhi[2] = {0.f, 0.f};
    if (Sout && inPair)
        for (int c = 0; c < 2; ++c) {
            blo[c] = stats[2 * kOut + 2 * sp + c];
            bhi[c] = stats[2 * kOut + kIn + 2 * sp + c];
        }
    const int ntiles = (n + kFTile - 1) / kFTile;
    // the thread's four input pairs of a tile, loaded back to back (the row index is clamped so every
    // load is in bounds; rows past n and padding features are zeroed when staged); the next
    // tile's are fetched while this one is computed
    const int lp = inPair ? sp : 0;
    float2 xv[kFTile / 16];
    auto fetch = [&](int tile) {
        const int r0 = tile * kFTile;
#pragma unroll
        for (int j = 0; j < kFTile / 16; ++j)
            xv[j] = *reinterpret_cast<const float2*>(X + size_t(min(r0 + sr + 16 * j, n - 1)) * kIn + 2 * lp);
    };
    if (int(blockIdx.x) < ntiles) fetch(blockIdx.x);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int r0 = tile * kFTile;
#pragma unroll
        for (int j = 0; j < kFTile / 16; ++j) {
            const int r = sr + 16 * j;
            const bool live = r0 + r < n && inPair;
            const float v0 = live ? xv[j].x : 0.f, v1 = live ? xv[j].y : 0.f;
            bf16x2 pv;
            pv[0] = static_cast<__bf16>(v0);
            pv[1] = static_cast<__bf16>(v1);
            *reinterpret_cast<bf16x2*>(xs + r * kXRow + 2 * sp) = pv;
            if (Sout) {
                // a wave stages four rows (16 lanes each): a row is outside when any lane's pair is
                const bool out = live && !(v0 >= blo[0] && v0 <= bhi[0] && v1 >= blo[1] && v1 <= bhi[1]);
                const uint64_t m = __ballot(out);
                if ((lane & 15) == 0) outside[r] = ((m >> (lane & 48)) & 0xFFFFull) != 0 ? 1 : 0;
            }
        }
        __syncthreads();
        if (tile + int(gridDim.x) < ntiles) fetch(tile + gridDim.x);
        // hidden layers: wave w computes features 32w..32w+31 of all 64 samples
        auto hidden = [&](const __bf16* in, int in_row, int kblocks, const bf16x8 (*wf)[4], const bf16x8* wf1, const f32x4* bias,
                          __bf16* out) {
            f32x4 acc[2][4];
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                for (int sb = 0; sb < 4; ++sb) acc[cb][sb] = bias[cb];
#pragma unroll
            for (int sb = 0; sb < 4; ++sb)
#pragma unroll
                for (int kb = 0; kb < 4; ++kb) {
                    if (kb >= kblocks) break;
                    const bf16x8 bfrag = *reinterpret_cast<const bf16x8*>(in + (16 * sb + fr) * in_row + 32 * kb + fk);
#pragma unroll
                    for (int cb = 0; cb < 2; ++cb) acc[cb][sb] = mfma(wf ? wf[cb][kb] : wf1[cb], bfrag, acc[cb][sb]);
                }
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                for (int sb = 0; sb < 4; ++sb) {
                    bf16x4 h;
#pragma unroll
                    for (int r = 0; r < 4; ++r) h[r] = static_cast<__bf16>(relu_bits(acc[cb][sb][r]));
                    *reinterpret_cast<bf16x4*>(out + (16 * sb + fr) * kHRow + 32 * w + 16 * cb + 4 * fg) = h;
                }
        };
        hidden(xs, kXRow, 1, nullptr, w1, c1, ha);
        __syncthreads();
        hidden(ha, kHRow, 4, w2, nullptr, c2, hb);
        __syncthreads();
        hidden(hb, kHRow, 4, w3, nullptr, c3, ha);
        __syncthreads();
        // output layer: wave w computes samples 16w..16w+15, all 16 outputs; lane (fr, fg) holds
        // outputs 4fg..4fg+3 of sample 16w + fr: row fg of its Mueller matrix
        f32x4 acc = c4;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) acc = mfma(w4[kb], *reinterpret_cast<const bf16x8*>(ha + (16 * w + fr) * kHRow + 32 * kb + fk), acc);
        const int srow = 16 * w + fr, row = r0 + srow;
        if (!Sout) {
            if (row < n) *reinterpret_cast<f32x4*>(Y + size_t(row) * kOut + 4 * fg) = acc;
        } else {
            // M00 = exp(y0) from the lane holding output 0 of the same sample (fg = 0)
            const float m00 = __shfl(__expf(acc[0] * stats[kOut] + stats[0]), fr);
            if (row < n && !outside[srow]) {
                const float* S = Sin + size_t(row) * 4;
                float acc4 = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int k = 4 * fg + c;
                    const float v = k == 0 ? 1.f : sinh_fast(acc[c] * stats[kOut + k] + stats[k]);
                    acc4 += v * S[c];
                }
                Sout[size_t(row) * 4 + fg] = m00 * acc4;
            }
        }
        __syncthreads();  // the next tile overwrites xs, ha and outside
    }
}

// ---------------------------------------------------------------------------------------
// Element-wise kernels.
// ---------------------------------------------------------------------------------------
constexpr int kEw = 256;

// bf16 operand copies of one layer: W [out x in_pad] and Wt [in x out_pad] from the master
// weights [out x in] (padding zero).
__global__ void cast_weights_kernel(int out, int in, int in_pad, int out_pad, const float* __restrict__ Wm, __bf16* __restrict__ W,
                                    __bf16* __restrict__ Wt) {
    const int e = blockIdx.x * kEw + threadIdx.x;
    if (e >= out_pad * in_pad) return;
    const int o = e / in_pad, i = e % in_pad;
    const __bf16 v = static_cast<__bf16>(o < out && i < in ? Wm[size_t(o) * in + i] : 0.f);
    if (o < out) W[size_t(o) * in_pad + i] = v;
    if (i < in) Wt[size_t(i) * out_pad + o] = v;
}

}  // namespace mlp
}  // namespace plt

using namespace plt;
using namespace plt::mlp;



namespace {

// Offsets of each tensor in the public parameter order.
constexpr size_t kOffW1 = 0, kOffB1 = kOffW1 + size_t(kHid) * kIn, kOffW2 = kOffB1 + kHid, kOffB2 = kOffW2 + size_t(kHid) * kHid,
                 kOffW3 = kOffB2 + kHid, kOffB3 = kOffW3 + size_t(kHid) * kHid, kOffW4 = kOffB3 + kHid,
                 kOffB4 = kOffW4 + size_t(kOut) * kHid;
constexpr size_t kTrainStateWords = 16;

template <class T>
int dev_alloc(plt_surrogate* s, T** p, size_t count) {
    void* q = nullptr;
    if (hipMalloc(&q, count * sizeof(T)) != hipSuccess) return set_error(PLT_ENOMEM, "plt_surrogate: device allocation failed");
    s->owned.push_back(q);
    *p = static_cast<T*>(q);
    return PLT_OK;
}

int cast_all(plt_surrogate* s, hipStream_t st) {
    struct L { size_t off; int out, in, in_pad, out_pad; __bf16 *W, *Wt; };
    const L layers[4] = {{kOffW1, kHid, kIn, kInPad, kHid, s->W1, s->W1t},
                         {kOffW2, kHid, kHid, kHid, kHid, s->W2, s->W2t},
                         {kOffW3, kHid, kHid, kHid, kHid, s->W3, s->W3t},
                         {kOffW4, kOut, kHid, kHid, kOutPad, s->W4, s->W4t}};
    for (const L& l : layers) {
        const int count = l.out_pad * l.in_pad;
        hipLaunchKernelGGL(cast_weights_kernel, dim3((count + kEw - 1) / kEw), dim3(kEw), 0, st, l.out, l.in, l.in_pad, l.out_pad,
                           s->params + l.off, l.W, l.Wt);
    }
    return check_launch("cast_weights_kernel");
}

// ---------------------------------------------------------------------------------------
// Training data pipeline and device-driven training (plt_surrogate_prepare / plt_surrogate_train).
// ---------------------------------------------------------------------------------------
// Loss weights per output, applied through the standardisation (an output scaled by 1/s weighs
// s^2 in the mean-squared error): the radiance row (ln M00, then M01..M03) first.
__constant__ float kOutputScale[kOut] = {4.f, 2.f, 2.f, 2.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};

// The training targets of one exact Mueller matrix: ln M00 and asinh(Mk / M00), in double; a row
// is valid when every entry is finite and M00 > 1e-12.
__device__ bool targets_of(const float* __restrict__ Mrow, double* y) {
    bool ok = Mrow[0] > 1e-12f;
#pragma unroll
    for (int k = 0; k < kOut; ++k) ok = ok && isfinite(Mrow[k]);
    const double m00 = ok ? double(Mrow[0]) : 1.0;
    y[0] = log(m00);
#pragma unroll
    for (int k = 1; k < kOut; ++k) y[k] = asinh(double(Mrow[k]) / m00);
    return ok;
}

// The column sums of a block's rows, each as sixteen sums of every sixteenth row added in order.
__device__ void column_sums(double (&ys)[kEw][kOut], int rows, double* __restrict__ out) {
    __shared__ double part[kEw / kOut][kOut];
    const int c = threadIdx.x % kOut, q = threadIdx.x / kOut;
    double acc = 0.0;
    for (int r = q; r < rows; r += kEw / kOut) acc += ys[r][c];
    part[q][c] = acc;
    __syncthreads();
    if (threadIdx.x < kOut) {
        double sum = 0.0;
        for (int k = 0; k < kEw / kOut; ++k) sum += part[k][threadIdx.x];
        out[threadIdx.x] = sum;
    }
}

// Pass 1, per block of kEw rows: valid count, column sums of the targets (double), and the box of
// the valid rows' inputs, in a fixed order. Every thread takes a sixteenth of a column and an eighth of a
// feature (one thread per column and feature walked the block's 256 rows one after the other, with a
// dependent load each: 264,000 rows 152 us).
__global__ void __launch_bounds__(kEw) prep_sums_kernel(int n, const float* __restrict__ X, const float* __restrict__ M,
                                                        double* __restrict__ psum, float* __restrict__ plo, float* __restrict__ phi,
                                                        uint32_t* __restrict__ pcount) {
    __shared__ double ys[kEw][kOut];
    __shared__ uint8_t valid[kEw];
    __shared__ float lo_s[kEw / 32][32], hi_s[kEw / 32][32];
    const int t = threadIdx.x, i = blockIdx.x * kEw + t;
    double y[kOut];
    bool ok = false;
    if (i < n) ok = targets_of(M + size_t(i) * kOut, y);
#pragma unroll
    for (int k = 0; k < kOut; ++k) ys[t][k] = ok ? y[k] : 0.0;
    valid[t] = ok ? 1 : 0;
    __syncthreads();
    const int rows = min(kEw, n - int(blockIdx.x) * kEw);
    column_sums(ys, rows, psum + size_t(blockIdx.x) * kOut);
    // the box: feature t % 32 (< 22) over rows t / 32 + 8 k, then the eight partial boxes
    {
        const int f = t & 31, q = t >> 5;
        float lo = __builtin_inff(), hi = -__builtin_inff();
        if (f < kIn)
            for (int r = q; r < rows; r += kEw / 32)
                if (valid[r]) {
                    const float v = X[(size_t(blockIdx.x) * kEw + r) * kIn + f];
                    lo = fminf(lo, v);
                    hi = fmaxf(hi, v);
                }
        lo_s[q][f] = lo;
        hi_s[q][f] = hi;
    }
    const int c = __syncthreads_count(valid[t] != 0);
    if (t < kIn) {
        float lo = lo_s[0][t], hi = hi_s[0][t];
#pragma unroll
        for (int q = 1; q < kEw / 32; ++q) {
            lo = fminf(lo, lo_s[q][t]);
            hi = fmaxf(hi, hi_s[q][t]);
        }
        plo[size_t(blockIdx.x) * kIn + t] = lo;
        phi[size_t(blockIdx.x) * kIn + t] = hi;
    } else if (t == 64) {
        pcount[blockIdx.x] = uint32_t(c);
    }
}

// One block of 1024 threads: the means, the box (into stats), the total valid count, and each
// block's first slot in the compacted index list. Every sum splits the blocks into contiguous
// chunks, one per thread, and combines the chunk results in chunk order (deterministic).
constexpr int kPrepThreads = 1024;
__global__ void __launch_bounds__(kPrepThreads) prep_mean_kernel(int blocks, const double* __restrict__ psum, const float* __restrict__ plo,
                                                                 const float* __restrict__ phi, uint32_t* __restrict__ pcount,
                                                                 double* __restrict__ dstat, float* __restrict__ stats,
                                                                 uint32_t* __restrict__ n_valid) {
    __shared__ uint32_t chunk_count[kPrepThreads];
    __shared__ double col[kPrepThreads / kOut][kOut];
    __shared__ float lo_s[kPrepThreads / 32][kIn], hi_s[kPrepThreads / 32][kIn];
    const int t = threadIdx.x;
    // counts: chunk t of the blocks, then an exclusive scan over the chunks
    const int per = (blocks + kPrepThreads - 1) / kPrepThreads;
    const int b0 = min(blocks, t * per), b1 = min(blocks, b0 + per);
    uint32_t c = 0;
    for (int b = b0; b < b1; ++b) c += pcount[b];
    chunk_count[t] = c;
    // column sums: column t % 16 over chunk t / 16
    {
        const int cc = t % kOut, q = t / kOut, nq = kPrepThreads / kOut, pq = (blocks + nq - 1) / nq;
        double acc = 0.0;
        for (int b = q * pq; b < min(blocks, (q + 1) * pq); ++b) acc += psum[size_t(b) * kOut + cc];
        col[q][cc] = acc;
    }
    // box: feature t % 32 (< 22) over chunk t / 32
    {
        const int f = t % 32, q = t / 32, nq = kPrepThreads / 32, pq = (blocks + nq - 1) / nq;
        if (f < kIn) {
            float lo = __builtin_inff(), hi = -__builtin_inff();
            for (int b = q * pq; b < min(blocks, (q + 1) * pq); ++b) {
                lo = fminf(lo, plo[size_t(b) * kIn + f]);
                hi = fmaxf(hi, phi[size_t(b) * kIn + f]);
            }
            lo_s[q][f] = lo;
            hi_s[q][f] = hi;
        }
    }
    __syncthreads();
    __shared__ uint32_t total;
    if (t == 0) {
        uint32_t run = 0;
        for (int q = 0; q < kPrepThreads; ++q) {
            const uint32_t x = chunk_count[q];
            chunk_count[q] = run;
            run += x;
        }
        total = run;
        *n_valid = run;
    }
    __syncthreads();
    {
        uint32_t run = chunk_count[t];
        for (int b = b0; b < b1; ++b) {
            const uint32_t x = pcount[b];
            pcount[b] = run;
            run += x;
        }
    }
    if (t < kOut) {
        double acc = 0.0;
        for (int q = 0; q < kPrepThreads / kOut; ++q) acc += col[q][t];
        const double mean = total ? acc / double(total) : 0.0;
        dstat[t] = mean;
        stats[t] = float(mean);
    } else if (t >= 32 && t < 32 + kIn) {
        const int f = t - 32;
        float lo = __builtin_inff(), hi = -__builtin_inff();
        for (int q = 0; q < kPrepThreads / 32; ++q) {
            lo = fminf(lo, lo_s[q][f]);
            hi = fmaxf(hi, hi_s[q][f]);
        }
        stats[2 * kOut + f] = lo;
        stats[2 * kOut + kIn + f] = hi;
    }
}

// Pass 2: per block, the column sums of squared deviations from the mean (double) and the valid
// rows' indices, compacted in row order.
__global__ void __launch_bounds__(kEw) prep_dev_kernel(int n, const float* __restrict__ M, const double* __restrict__ dstat,
                                                       const uint32_t* __restrict__ boffset, double* __restrict__ psum,
                                                       uint32_t* __restrict__ idx) {
    __shared__ double ys[kEw][kOut];
    __shared__ uint32_t wcount[kEw / 64];
    const int t = threadIdx.x, i = blockIdx.x * kEw + t;
    double y[kOut];
    bool ok = false;
    if (i < n) ok = targets_of(M + size_t(i) * kOut, y);
#pragma unroll
    for (int k = 0; k < kOut; ++k) {
        const double d = ok ? y[k] - dstat[k] : 0.0;
        ys[t][k] = d * d;
    }
    const uint64_t m = __ballot(ok);
    const int lane = t & 63, wave = t >> 6;
    if (lane == 0) wcount[wave] = uint32_t(__popcll(m));
    __syncthreads();
    if (ok) {
        uint32_t before = uint32_t(__popcll(m & ((uint64_t(1) << lane) - 1u)));
        for (int w = 0; w < wave; ++w) before += wcount[w];
        idx[boffset[blockIdx.x] + before] = uint32_t(i);
    }
    column_sums(ys, min(kEw, n - int(blockIdx.x) * kEw), psum + size_t(blockIdx.x) * kOut);
}

// One block of 1024 threads: the standard deviations (population), scaled by the output weights,
// into stats (chunked sums combined in chunk order).
__global__ void __launch_bounds__(kPrepThreads) prep_std_kernel(int blocks, const double* __restrict__ psum, const uint32_t* __restrict__ n_valid,
                                                                double* __restrict__ dstat, float* __restrict__ stats) {
    __shared__ double col[kPrepThreads / kOut][kOut];
    const int t = threadIdx.x;
    const int cc = t % kOut, q = t / kOut, nq = kPrepThreads / kOut, pq = (blocks + nq - 1) / nq;
    double acc = 0.0;
    for (int b = q * pq; b < min(blocks, (q + 1) * pq); ++b) acc += psum[size_t(b) * kOut + cc];
    col[q][cc] = acc;
    __syncthreads();
    if (t >= kOut) return;
    double sum = 0.0;
    for (int k = 0; k < nq; ++k) sum += col[k][t];
    const uint32_t c = *n_valid;
    double sd = c ? sqrt(sum / double(c)) : 1.0;
    sd = (sd > 1e-6 ? sd : 1.0) / double(kOutputScale[t]);
    dstat[kOut + t] = sd;
    stats[kOut + t] = float(sd);
}

// Pass 3: the standardised targets T = (y - mean) / std of every row (rows that are not valid are
// never drawn).
__global__ void __launch_bounds__(kEw) prep_targets_kernel(int n, const float* __restrict__ M, const double* __restrict__ dstat,
                                                           float* __restrict__ T) {
    const int i = blockIdx.x * kEw + threadIdx.x;
    if (i >= n) return;
    double y[kOut];
    (void)targets_of(M + size_t(i) * kOut, y);
#pragma unroll
    for (int k = 0; k < kOut; ++k) T[size_t(i) * kOut + k] = float((y[k] - dstat[k]) / dstat[kOut + k]);
}

__host__ __device__ inline uint32_t mix32(uint32_t h) {
    h ^= h >> 16;
    h *= 0x7FEB352Du;
    h ^= h >> 15;
    h *= 0x846CA68Bu;
    h ^= h >> 16;
    return h;
}
// A bijection of [0, 2^(2 half)): a four-round balanced Feistel network keyed by `key`.
__device__ uint32_t feistel(uint32_t x, int half, uint32_t key) {
    const uint32_t mask = (1u << half) - 1u;
    uint32_t l = x >> half, r = x & mask;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t t = l ^ (mix32(r ^ mix32(key + k)) & mask);
        l = r;
        r = t;
    }
    return (l << half) | r;
}
// The epoch's shuffle of [0, n), n > 2^(2 half - 2): cycle-walking the Feistel bijection (the walk
// from x < n ends: the bijection's cycle through x returns to x; it takes under four steps on
// average).
__device__ uint32_t shuffle_index(uint32_t x, uint32_t n, int half, uint32_t key) {
    uint32_t y = feistel(x, half, key);
    while (y >= n) y = feistel(y, half, key);
    return y;
}

__host__ __device__ inline uint32_t epoch_key(uint32_t seed, uint32_t epoch) { return mix32(seed * 0x9E3779B9u + epoch); }
int shuffle_half(uint32_t n) {
    int bits = 2;
    while (bits < 32 && (uint64_t(1) << bits) < n) ++bits;
    return (bits + (bits & 1)) / 2;
}

// The epoch's order itself (plt_surrogate_shuffle).
__global__ void shuffle_kernel(uint32_t n, int half, uint32_t key, uint32_t* __restrict__ out) {
    const uint32_t x = blockIdx.x * kEw + threadIdx.x;
    if (x < n) out[x] = shuffle_index(x, n, half, key);
}

// ---------------------------------------------------------------------------------------
// Fused training step: forward pass, loss, backward pass and the weight gradients of one batch in
// one kernel. A workgroup of four waves takes every gridDim.x-th tile of 64 samples; a tile's
// activations never leave LDS, and the gradients of all 38,032 parameters are summed over the
// group's tiles in its waves' accumulators (176 registers a lane) and written once, as one partial
// per group. grad_reduce_kernel sums the partials in group order (and, in training, applies Adam), so
// a step is two launches.
//
// Products are computed transposed as in mlp_infer_kernel (weights the A operand, out[feature x
// sample]); wave w holds features 32w..32w+31. Each activation and each back-propagated gradient is
// stored twice: sample-major rows (the next product's B operand: 8 consecutive features) and
// feature-major rows (the weight gradients contract over samples, so both their operands are 8
// consecutive samples of one feature). A hidden unit's ReLU mask is one bit in the lane that
// computed it, which is the lane that computes its gradient.
//
// It is bound by the chain of ten barriers per tile, about 2 us each, with one group per CU (125 KB of
// LDS) and one wave per SIMD. A batch of 16,384 rows is one tile for each of 256 groups: 30 us and 9 us
// for the reduction, with 128 groups 43 and 6 us. Loading the next product's weights a phase ahead,
// across barriers that order LDS only, spilled registers and took 46 us. Before, a step was eighteen
// dependent launches (a GEMM per product and gradient, 9 us each, every activation through memory in
// two layouts): 141 us.
// ---------------------------------------------------------------------------------------
constexpr int kGroupsMax = 256;  // partials to sum (40 MB at 256): one group per CU
constexpr int kTRow = kFTile + 8;  // feature-major LDS rows

// The layout of one group's partial: W4, W3, W2, W1 (its 32 padded inputs), then the biases b4, b3, b2, b1.
constexpr int kPartW4 = 0, kPartW3 = kPartW4 + kOut * kHid, kPartW2 = kPartW3 + kHid * kHid, kPartW1 = kPartW2 + kHid * kHid,
              kGradTotal = kPartW1 + kHid * kInPad;  // 38,912
constexpr int kBiasCols = kOut + 3 * kHid;
constexpr int kPartTotal = kGradTotal + kBiasCols;

// Device-side state of plt_surrogate_train: every launch of a training step reads what it needs
// from here, so one captured step replays as every step. The train kernel reads `step` and publishes
// the step it runs, its learning rate and Adam's corrections (group 0); the reduction reads those and
// advances `step`.
struct TrainState {
    uint32_t step, steps_per_epoch, steps_total, batch, n_valid, seed, adam_t0;
    float lr0;
    uint32_t now;
    float lr, c1, c2;
};

struct TrainArgs {
    int n;                 // rows of the batch
    const float *X, *T;    // inputs [. x 22] and targets [. x 16]
    const uint32_t* idx;   // with st: row i of the batch is idx[shuffle(step's i-th position)]
    int half;
    TrainState* st;
    const __bf16 *W1, *W2, *W3, *W4, *W2t, *W3t, *W4t;
    const float *b1, *b2, *b3, *b4;
    float* part;           // [gridDim.x x kPartTotal]
    float* loss_part;      // [gridDim.x]
};

__global__ void __launch_bounds__(kFThreads, 1) mlp_train_kernel(TrainArgs g) {
    __shared__ __bf16 xs[kFTile * kXRow], xt[kInPad * kTRow];
    __shared__ __bf16 sa[kFTile * kHRow], sb[kFTile * kHRow];          // sample-major, ping-pong
    __shared__ __bf16 h1t[kHid * kTRow], h2t[kHid * kTRow], h3t[kHid * kTRow], gt[kHid * kTRow];
    __shared__ __bf16 dy[kFTile * kXRow], dyt[kOut * kTRow];
    __shared__ uint32_t rows[kFTile];
    __shared__ float red[kFThreads / 64][1 + kOut];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int fr = lane & 15, fg = lane >> 4, fk = 8 * fg;
    uint32_t step = 0, epoch_pos = 0, key = 0, n_valid = 0;
    if (g.st) {
        const TrainState s = *g.st;
        step = s.step;
        n_valid = s.n_valid;
        epoch_pos = (step % s.steps_per_epoch) * s.batch;
        key = epoch_key(s.seed, step / s.steps_per_epoch);
        if (blockIdx.x == 0 && t == 0) {
            // the cosine-decayed rate (at least 1e-6) and the corrections of Adam step adam_t0 + step + 1
            const double tt = double(s.adam_t0) + double(step) + 1.0;
            g.st->now = step;
            g.st->c1 = float(1.0 - pow(double(0.9f), tt));
            g.st->c2 = float(1.0 - pow(double(0.999f), tt));
            const double cs = cos(3.14159265358979323846 * double(step) / double(max(1u, s.steps_total)));
            g.st->lr = float(fmax(double(s.lr0) * 0.5 * (1.0 + cs), 1e-6));
        }
    }
    // outputs 16..31 of dY pad its K dimension with zeros
    for (int i = t; i < kFTile * kXRow; i += kFThreads) dy[i] = static_cast<__bf16>(0.f);
    f32x4 c1[2], c2[2], c3[2], c4;
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int f = 32 * w + 16 * cb + 4 * fg + r;
            c1[cb][r] = g.b1[f];
            c2[cb][r] = g.b2[f];
            c3[cb][r] = g.b3[f];
        }
#pragma unroll
    for (int r = 0; r < 4; ++r) c4[r] = g.b4[4 * fg + r];
    const f32x4 zero{0.f, 0.f, 0.f, 0.f};
    f32x4 dw1[2][2], dw2[2][8], dw3[2][8], dw4[2], db1[2], db2[2], db3[2], db4 = zero;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int b = 0; b < 8; ++b) dw2[a][b] = dw3[a][b] = zero;
        dw1[a][0] = dw1[a][1] = dw4[a] = db1[a] = db2[a] = db3[a] = zero;
    }
    float loss = 0.f;
    const float scale = 2.f / (float(g.n) * float(kOut));

    // out[32w..32w+31 x 64 samples] from kb blocks of 32 sample-major inputs and the weight rows Wm
    auto product = [&](auto kblocks, const __bf16* in, int in_row, const __bf16* Wm, int ldw, const f32x4* init, f32x4 (&acc)[2][4]) {
        constexpr int kK = decltype(kblocks)::value;
        bf16x8 wf[2][kK];
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int kb = 0; kb < kK; ++kb)
                wf[cb][kb] = *reinterpret_cast<const bf16x8*>(Wm + size_t(32 * w + 16 * cb + fr) * ldw + 32 * kb + fk);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int s = 0; s < 4; ++s) acc[cb][s] = init ? init[cb] : zero;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int kb = 0; kb < kK; ++kb) {
                const bf16x8 b = *reinterpret_cast<const bf16x8*>(in + (16 * s + fr) * in_row + 32 * kb + fk);
#pragma unroll
                for (int cb = 0; cb < 2; ++cb) acc[cb][s] = mfma(wf[cb][kb], b, acc[cb][s]);
            }
    };
    // stores a lane's four features of sample 16 s + fr in both layouts (sm may be null)
    auto store = [&](bf16x4 h, int cb, int s, __bf16* sm, __bf16* fm) {
        const int f = 32 * w + 16 * cb + 4 * fg, row = 16 * s + fr;
        if (sm) *reinterpret_cast<bf16x4*>(sm + row * kHRow + f) = h;
#pragma unroll
        for (int r = 0; r < 4; ++r) fm[(f + r) * kTRow + row] = h[r];
    };
    auto forward = [&](auto kblocks, const __bf16* in, int in_row, const __bf16* Wm, int ldw, const f32x4* bias, __bf16* sm, __bf16* fm) {
        f32x4 acc[2][4];
        product(kblocks, in, in_row, Wm, ldw, bias, acc);
        uint32_t mask = 0;
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    h[r] = static_cast<__bf16>(relu_bits(acc[cb][s][r]));
                    mask |= static_cast<float>(h[r]) > 0.f ? 1u << (16 * cb + 4 * s + r) : 0u;
                }
                store(h, cb, s, sm, fm);
            }
        return mask;
    };
    auto backward = [&](auto kblocks, const __bf16* in, int in_row, const __bf16* Wt, int ldw, uint32_t mask, __bf16* sm, __bf16* fm, f32x4 (&db)[2]) {
        f32x4 acc[2][4];
        product(kblocks, in, in_row, Wt, ldw, nullptr, acc);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    h[r] = static_cast<__bf16>((mask >> (16 * cb + 4 * s + r)) & 1u ? acc[cb][s][r] : 0.f);
                    db[cb][r] += static_cast<float>(h[r]);
                }
                store(h, cb, s, sm, fm);
            }
    };
    // dW[32w..32w+31 x 16 B..] += G H^T over the tile's 64 samples (feature-major operands)
    auto weight_grad = [&](auto nb, const __bf16* gm, const __bf16* hm, auto& dw) {
        constexpr int kB = decltype(nb)::value;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            bf16x8 a[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf16x8*>(gm + (32 * w + 16 * i + fr) * kTRow + 32 * kb + fk);
#pragma unroll
            for (int b = 0; b < kB; ++b) {
                const bf16x8 h = *reinterpret_cast<const bf16x8*>(hm + (16 * b + fr) * kTRow + 32 * kb + fk);
#pragma unroll
                for (int i = 0; i < 2; ++i) dw[i][b] = mfma(a[i], h, dw[i][b]);
            }
        }
    };
    using K1 = std::integral_constant<int, 1>;
    using K2 = std::integral_constant<int, 2>;
    using K4 = std::integral_constant<int, 4>;
    using K8 = std::integral_constant<int, 8>;

    const int ntiles = (g.n + kFTile - 1) / kFTile;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int r0 = tile * kFTile;
        __syncthreads();  // the previous tile's last reads of xt, gt and rows
        if (t < kFTile) {
            uint32_t row = uint32_t(min(r0 + t, g.n - 1));
            if (g.st) row = g.idx[shuffle_index(epoch_pos + row, n_valid, g.half, key)];
            rows[t] = row;
        }
        __syncthreads();
        {
            // thread t stages input features 2p, 2p + 1 (p = t % 16) of rows t / 16 + 16 j; rows past n
            // and padding features are zero
            const int p = t & 15, sr = t >> 4;
            const bool in = 2 * p < kIn;
            float2 v[kFTile / 16];
#pragma unroll
            for (int j = 0; j < kFTile / 16; ++j)
                v[j] = *reinterpret_cast<const float2*>(g.X + size_t(rows[sr + 16 * j]) * kIn + (in ? 2 * p : 0));
#pragma unroll
            for (int j = 0; j < kFTile / 16; ++j) {
                const int r = sr + 16 * j;
                const bool live = in && r0 + r < g.n;
                bf16x2 pv;
                pv[0] = static_cast<__bf16>(live ? v[j].x : 0.f);
                pv[1] = static_cast<__bf16>(live ? v[j].y : 0.f);
                *reinterpret_cast<bf16x2*>(xs + r * kXRow + 2 * p) = pv;
                xt[(2 * p) * kTRow + r] = pv[0];
                xt[(2 * p + 1) * kTRow + r] = pv[1];
            }
        }
        // the lane's four targets: outputs 4 fg.. of sample 16 w + fr
        const int srow = 16 * w + fr;
        const f32x4 target = *reinterpret_cast<const f32x4*>(g.T + size_t(rows[srow]) * kOut + 4 * fg);
        __syncthreads();
        const uint32_t m1 = forward(K1{}, xs, kXRow, g.W1, kInPad, c1, sa, h1t);
        __syncthreads();
        const uint32_t m2 = forward(K4{}, sa, kHRow, g.W2, kHid, c2, sb, h2t);
        __syncthreads();
        const uint32_t m3 = forward(K4{}, sb, kHRow, g.W3, kHid, c3, sa, h3t);
        __syncthreads();
        {
            f32x4 y = c4;
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
                y = mfma(*reinterpret_cast<const bf16x8*>(g.W4 + size_t(fr) * kHid + 32 * kb + fk),
                         *reinterpret_cast<const bf16x8*>(sa + srow * kHRow + 32 * kb + fk), y);
            const bool live = r0 + srow < g.n;
            bf16x4 d;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float e = live ? y[r] - target[r] : 0.f;
                loss += e * e;
                d[r] = static_cast<__bf16>(scale * e);
                db4[r] += static_cast<float>(d[r]);
                dyt[(4 * fg + r) * kTRow + srow] = d[r];
            }
            *reinterpret_cast<bf16x4*>(dy + srow * kXRow + 4 * fg) = d;
        }
        __syncthreads();
        backward(K1{}, dy, kXRow, g.W4t, kOutPad, m3, sb, gt, db3);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {  // dW4[16 x 32w..32w+31]
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(dyt + fr * kTRow + 32 * kb + fk);
#pragma unroll
            for (int b = 0; b < 2; ++b)
                dw4[b] = mfma(a, *reinterpret_cast<const bf16x8*>(h3t + (32 * w + 16 * b + fr) * kTRow + 32 * kb + fk), dw4[b]);
        }
        __syncthreads();
        weight_grad(K8{}, gt, h2t, dw3);
        backward(K4{}, sb, kHRow, g.W3t, kHid, m2, sa, h3t, db2);  // h3t now holds the second layer's gradient
        __syncthreads();
        weight_grad(K8{}, h3t, h1t, dw2);
        backward(K4{}, sa, kHRow, g.W2t, kHid, m1, static_cast<__bf16*>(nullptr), gt, db1);
        __syncthreads();
        weight_grad(K2{}, gt, xt, dw1);
    }
    // the group's partial. D layout: the lane holds rows 4 fg + r of column fr of each 16 x 16 block
    float* part = g.part + size_t(blockIdx.x) * kPartTotal;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = 32 * w + 16 * i + 4 * fg + r;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                part[kPartW3 + o * kHid + 16 * b + fr] = dw3[i][b][r];
                part[kPartW2 + o * kHid + 16 * b + fr] = dw2[i][b][r];
            }
#pragma unroll
            for (int b = 0; b < 2; ++b) part[kPartW1 + o * kInPad + 16 * b + fr] = dw1[i][b][r];
            part[kPartW4 + (4 * fg + r) * kHid + 32 * w + 16 * i + fr] = dw4[i][r];
        }
    // bias sums over the 16 lanes of a feature (xor steps 1..8), in a fixed order
    auto lanes16 = [](float v) {
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o);
        return v;
    };
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int f = 32 * w + 16 * i + 4 * fg + r;
            const float s3 = lanes16(db3[i][r]), s2 = lanes16(db2[i][r]), s1 = lanes16(db1[i][r]);
            if (fr == 0) {
                part[kGradTotal + kOut + f] = s3;
                part[kGradTotal + kOut + kHid + f] = s2;
                part[kGradTotal + kOut + 2 * kHid + f] = s1;
            }
        }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float s = lanes16(db4[r]);
        if (fr == 0) red[w][1 + 4 * fg + r] = s;
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) loss += __shfl_xor(loss, o);
    if (lane == 0) red[w][0] = loss;
    __syncthreads();
    if (t <= kOut) {
        const float s = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
        if (t == 0) g.loss_part[blockIdx.x] = s;
        else part[kGradTotal + t - 1] = s;
    }
}
static_assert(sizeof(TrainState) <= kTrainStateWords * 4, "train state size");

// Every gradient from the groups' partials, in one launch. A block takes 64 elements of a partial
// with four threads each: thread group q sums the partials of groups q, q + 4, ... (16 loads issued
// before their adds), and the four sums are combined in order. The sum goes to `grads`, or (grads
// null) through Adam to the FP32 master parameters and their bf16 copies, whose padding stays zero;
// the learning rate and the corrections come from the arguments, or with `st` from the device state
// that the train kernel published. Block 0 then also records the step's mean loss and advances the
// state's step, which no thread of this kernel reads.
struct WeightCopies {
    __bf16 *W1, *W1t, *W2, *W2t, *W3, *W3t, *W4, *W4t;
};
struct ReduceArgs {
    int groups;
    const float *part, *loss_part;
    float* grads;
    float *p, *m, *v;
    TrainState* st;
    float lr, c1, c2;
    WeightCopies w;
    float* loss_hist;
};
constexpr int kReduceLanes = 64, kReduceBatch = 16;  // elements per block; loads in flight per thread
__global__ void __launch_bounds__(256) grad_reduce_kernel(ReduceArgs a) {
    __shared__ float sums[4][kReduceLanes];
    const int el = threadIdx.x & (kReduceLanes - 1), q = threadIdx.x >> 6;
    const int e = blockIdx.x * kReduceLanes + el;
    const bool live = e < kPartTotal;
    float acc = 0.f;
    if (live) {
        for (int z0 = q; z0 < a.groups; z0 += 4 * kReduceBatch) {
            float v[kReduceBatch];
#pragma unroll
            for (int j = 0; j < kReduceBatch; ++j) {
                const int z = z0 + 4 * j;
                v[j] = z < a.groups ? a.part[size_t(z) * kPartTotal + e] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < kReduceBatch; ++j) acc += v[j];
        }
    }
    sums[q][el] = acc;
    __syncthreads();
    if (a.st && blockIdx.x == 0 && q == 1) {
        double l = 0.0;
        for (int z = el; z < a.groups; z += kReduceLanes) l += double(a.loss_part[z]);
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) l += __shfl_xor(l, o);
        if (el == 0) {
            const uint32_t now = a.st->now;
            a.loss_hist[now] = float(l / (double(a.st->batch) * kOut));
            a.st->step = now + 1u;
        }
    }
    if (q != 0 || !live) return;
    const float ge = (sums[0][el] + sums[1][el]) + (sums[2][el] + sums[3][el]);
    // the element's parameter and, for a weight, its places in the two bf16 copies
    size_t dst;
    __bf16 *W = nullptr, *Wt = nullptr;
    if (e < kPartW3) {
        const int o = e / kHid, i = e % kHid;
        dst = kOffW4 + e;
        W = a.w.W4 + e;
        Wt = a.w.W4t + i * kOutPad + o;
    } else if (e < kPartW1) {
        const bool third = e < kPartW2;
        const int l = e - (third ? kPartW3 : kPartW2), o = l / kHid, i = l % kHid;
        dst = (third ? kOffW3 : kOffW2) + l;
        W = (third ? a.w.W3 : a.w.W2) + l;
        Wt = (third ? a.w.W3t : a.w.W2t) + i * kHid + o;
    } else if (e < kGradTotal) {
        const int l = e - kPartW1, o = l / kInPad, i = l % kInPad;
        if (i >= kIn) return;  // padding
        dst = kOffW1 + size_t(o) * kIn + i;
        W = a.w.W1 + l;
        Wt = a.w.W1t + i * kHid + o;
    } else {
        const int c = e - kGradTotal;
        dst = c < kOut ? kOffB4 + c : c < kOut + kHid ? kOffB3 + (c - kOut) : c < kOut + 2 * kHid ? kOffB2 + (c - kOut - kHid)
                                                                                      : kOffB1 + (c - kOut - 2 * kHid);
    }
    if (a.grads) {
        a.grads[dst] = ge;
        return;
    }
    constexpr float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float lr = a.st ? a.st->lr : a.lr, c1 = a.st ? a.st->c1 : a.c1, c2 = a.st ? a.st->c2 : a.c2;
    const float me = b1 * a.m[dst] + (1.f - b1) * ge;
    const float ve = b2 * a.v[dst] + (1.f - b2) * ge * ge;
    a.m[dst] = me;
    a.v[dst] = ve;
    const float pe = a.p[dst] - lr * (me / c1) / (sqrtf(ve / c2) + eps);
    a.p[dst] = pe;
    if (W) {
        const __bf16 h = static_cast<__bf16>(pe);
        *W = h;
        *Wt = h;
    }
}
WeightCopies weight_copies(const plt_surrogate* s) { return WeightCopies{s->W1, s->W1t, s->W2, s->W2t, s->W3, s->W3t, s->W4, s->W4t}; }

int train_groups(uint32_t n) { return int(std::min<uint32_t>(kGroupsMax, (n + kFTile - 1) / kFTile)); }

// The two launches of a step over n rows of X and T (with `st`, rows idx[shuffle]): the partials, then
// their sums into `grads` or through Adam.
int train_launch(plt_surrogate* s, int n, const float* X, const float* T, const uint32_t* idx, int half, TrainState* st, float* grads, float lr,
                 float c1, float c2, float* loss_hist, hipStream_t qs) {
    const int groups = train_groups(uint32_t(n));
    const TrainArgs ta{n, X, T, idx, half, st, s->W1, s->W2, s->W3, s->W4, s->W2t, s->W3t, s->W4t,
                       s->params + kOffB1, s->params + kOffB2, s->params + kOffB3, s->params + kOffB4, s->part, s->loss_part};
    hipLaunchKernelGGL(mlp_train_kernel, dim3(groups), dim3(kFThreads), 0, qs, ta);
    int rc = check_launch("mlp_train_kernel");
    if (rc < 0) return rc;
    const ReduceArgs ra{groups, s->part, s->loss_part, grads, s->params, s->adam_m, s->adam_v, st, lr, c1, c2, weight_copies(s), loss_hist};
    hipLaunchKernelGGL(grad_reduce_kernel, dim3((kPartTotal + kReduceLanes - 1) / kReduceLanes), dim3(256), 0, qs, ra);
    return check_launch("grad_reduce_kernel");
}

// The mean loss of the last train_launch over n rows.
int read_loss(plt_surrogate* s, uint32_t n, float* loss, hipStream_t st) {
    std::vector<float> lp(static_cast<size_t>(train_groups(n)));
    if (hipMemcpyAsync(lp.data(), s->loss_part, lp.size() * sizeof(float), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return set_error(PLT_EHIP, "plt_surrogate: loss read-back failed");
    double sum = 0.0;
    for (float v : lp) sum += v;
    *loss = float(sum / (double(n) * kOut));
    return PLT_OK;
}

}  // namespace

int plt::surrogate_infer(plt_surrogate* s, int n, const float* X, float* Y, const float* Sin, float* Sout, hipStream_t st) {
    if (n <= 0) return PLT_OK;
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    const int tiles = (n + kFTile - 1) / kFTile;
    const int grid = std::max(1, std::min(tiles, 2 * cus));
    hipLaunchKernelGGL(mlp_infer_kernel, dim3(grid), dim3(kFThreads), 0, st, n, X, s->W1, s->W2, s->W3, s->W4, s->params, Y, s->stats,
                       Sin, Sout, nullptr);
    return check_launch("mlp_infer_kernel");
}

int plt::surrogate_infer_counted(plt_surrogate* s, const uint32_t* n_dev, uint32_t cap, const float* X, float* Y, hipStream_t st) {
    if (cap == 0) return PLT_OK;
    if (cap > (1u << 30)) return set_error(PLT_EINVAL, "surrogate inference: too many rows");
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    const int tiles = int((cap + kFTile - 1) / kFTile);
    const int grid = std::max(1, std::min(tiles, 2 * cus));
    hipLaunchKernelGGL(mlp_infer_kernel, dim3(grid), dim3(kFThreads), 0, st, int(cap), X, s->W1, s->W2, s->W3, s->W4, s->params, Y,
                       s->stats, nullptr, nullptr, n_dev);
    return check_launch("mlp_infer_kernel");
}

extern "C" {

int plt_surrogate_create(plt_context* ctx, uint32_t max_batch, uint32_t seed, plt_surrogate** out) {
    if (!ctx || !out || max_batch == 0 || max_batch % 32 || max_batch > (1u << 24))
        return set_error(PLT_EINVAL, "plt_surrogate_create: bad arguments (max_batch a multiple of 32, at most 2^24)");
    *out = nullptr;
    auto* s = new plt_surrogate;
    s->ctx = ctx;
    s->max_batch = max_batch;
    int rc = PLT_OK;
    auto A = [&](auto** p, size_t count) { if (rc == PLT_OK) rc = dev_alloc(s, p, count); };
    A(&s->params, kParams); A(&s->grads, kParams); A(&s->adam_m, kParams); A(&s->adam_v, kParams);
    A(&s->W1, size_t(kHid) * kInPad); A(&s->W1t, size_t(kInPad) * kHid);
    A(&s->W2, size_t(kHid) * kHid); A(&s->W2t, size_t(kHid) * kHid);
    A(&s->W3, size_t(kHid) * kHid); A(&s->W3t, size_t(kHid) * kHid);
    A(&s->W4, size_t(kOut) * kHid); A(&s->W4t, size_t(kHid) * kOutPad);
    A(&s->part, size_t(train_groups(max_batch)) * kPartTotal);
    A(&s->loss_part, size_t(train_groups(max_batch)));
    A(&s->train_state, kTrainStateWords);
    A(&s->stats, 2 * kOut + 2 * kIn);
    A(&s->counter, 1);
    if (rc != PLT_OK) { plt_surrogate_destroy(s); return rc; }
    // He-uniform initialisation of the weights (bound sqrt(6 / fan_in)), zero biases
    std::vector<float> p(kParams, 0.f);
    std::mt19937 gen(seed);
    std::uniform_real_distribution<float> u(-1.f, 1.f);
    auto init = [&](size_t off, int out_, int in_) {
        const float b = std::sqrt(6.f / float(in_));
        for (size_t e = 0; e < size_t(out_) * in_; ++e) p[off + e] = b * u(gen);
    };
    init(kOffW1, kHid, kIn); init(kOffW2, kHid, kHid); init(kOffW3, kHid, kHid); init(kOffW4, kOut, kHid);
    if (rc == PLT_OK && (hipMemcpy(s->params, p.data(), kParams * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
                         hipMemset(s->adam_m, 0, kParams * sizeof(float)) != hipSuccess ||
                         hipMemset(s->adam_v, 0, kParams * sizeof(float)) != hipSuccess))
        rc = set_error(PLT_EHIP, "plt_surrogate_create: upload failed");
    if (rc == PLT_OK) rc = cast_all(s, nullptr);
    if (rc == PLT_OK && hipDeviceSynchronize() != hipSuccess) rc = set_error(PLT_EHIP, "plt_surrogate_create: synchronize failed");
    if (rc != PLT_OK) { plt_surrogate_destroy(s); return rc; }
    *out = s;
    return PLT_OK;
}

void plt_surrogate_destroy(plt_surrogate* s) {
    if (!s) return;
    for (void* p : s->owned) (void)hipFree(p);
    delete s;
}

uint32_t plt_surrogate_param_count(void) { return uint32_t(kParams); }

int plt_surrogate_params(plt_surrogate* s, float* host, int set) {
    if (!s || !host) return set_error(PLT_EINVAL, "plt_surrogate_params: bad arguments");
    if (set) {
        if (hipMemcpy(s->params, host, kParams * sizeof(float), hipMemcpyHostToDevice) != hipSuccess)
            return set_error(PLT_EHIP, "plt_surrogate_params: upload failed");
        s->step = 0;
        if (hipMemset(s->adam_m, 0, kParams * sizeof(float)) != hipSuccess || hipMemset(s->adam_v, 0, kParams * sizeof(float)) != hipSuccess)
            return set_error(PLT_EHIP, "plt_surrogate_params: reset failed");
        const int rc = cast_all(s, nullptr);
        if (rc < 0) return rc;
        return hipDeviceSynchronize() == hipSuccess ? PLT_OK : set_error(PLT_EHIP, "plt_surrogate_params: synchronize failed");
    }
    return hipMemcpy(host, s->params, kParams * sizeof(float), hipMemcpyDeviceToHost) == hipSuccess
               ? PLT_OK
               : set_error(PLT_EHIP, "plt_surrogate_params: download failed");
}

int plt_surrogate_forward(plt_surrogate* s, uint32_t n, const float* X, float* Y, plt_stream stream) {
    if (!s || (n && (!X || !Y))) return set_error(PLT_EINVAL, "plt_surrogate_forward: bad arguments");
    if (n > (1u << 30)) return set_error(PLT_EINVAL, "plt_surrogate_forward: n too large");
    return surrogate_infer(s, int(n), X, Y, nullptr, nullptr, static_cast<hipStream_t>(stream));
}

int plt_surrogate_gradients(plt_surrogate* s, uint32_t n, const float* X, const float* T, float* grads_host, float* loss,
                            plt_stream stream) {
    if (!s || n == 0 || n % 32 || n > s->max_batch || !X || !T)
        return set_error(PLT_EINVAL, "plt_surrogate_gradients: bad arguments (n a multiple of 32, at most max_batch)");
    const hipStream_t st = static_cast<hipStream_t>(stream);
    int rc;
    if ((rc = train_launch(s, int(n), X, T, nullptr, 0, nullptr, s->grads, 0.f, 1.f, 1.f, nullptr, st)) < 0) return rc;
    if (loss && (rc = read_loss(s, n, loss, st)) < 0) return rc;
    if (grads_host) {
        if (hipMemcpyAsync(grads_host, s->grads, kParams * sizeof(float), hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            return set_error(PLT_EHIP, "plt_surrogate_gradients: download failed");
    }
    return PLT_OK;
}

int plt_surrogate_train_step(plt_surrogate* s, uint32_t n, const float* X, const float* T, float lr, float* loss, plt_stream stream) {
    if (!s || n == 0 || n % 32 || n > s->max_batch || !X || !T || !(lr > 0.f))
        return set_error(PLT_EINVAL, "plt_surrogate_train_step: bad arguments (n a multiple of 32, at most max_batch)");
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const float b1 = 0.9f, b2 = 0.999f;
    const float k = float(s->step + 1), c1 = 1.f - std::pow(b1, k), c2 = 1.f - std::pow(b2, k);
    int rc;
    if ((rc = train_launch(s, int(n), X, T, nullptr, 0, nullptr, nullptr, lr, c1, c2, nullptr, st)) < 0) return rc;
    ++s->step;
    return loss ? read_loss(s, n, loss, st) : PLT_OK;
}

int plt_surrogate_prepare(plt_surrogate* s, uint32_t n, const float* X, const float* M, float* T, uint32_t* idx, uint32_t* n_valid,
                          plt_stream stream) {
    if (!s || n == 0 || !X || !M || !T || !idx || !n_valid || n > (1u << 30))
        return set_error(PLT_EINVAL, "plt_surrogate_prepare: bad arguments");
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const int blocks = int((n + kEw - 1) / kEw);
    // scratch of the reductions: per-block sums, boxes and counts, the double statistics, the count
    const size_t bytes = size_t(blocks) * (kOut * 8 + 2 * kIn * 4 + 4) + 2 * kOut * 8 + 64;
    void* q = nullptr;
    if (hipMalloc(&q, bytes) != hipSuccess) return set_error(PLT_ENOMEM, "plt_surrogate_prepare: scratch allocation failed");
    char* b = static_cast<char*>(q);
    double* psum = reinterpret_cast<double*>(b);
    double* dstat = psum + size_t(blocks) * kOut;
    float* plo = reinterpret_cast<float*>(dstat + 2 * kOut);
    float* phi = plo + size_t(blocks) * kIn;
    uint32_t* pcount = reinterpret_cast<uint32_t*>(phi + size_t(blocks) * kIn);
    uint32_t* nv = pcount + blocks;
    int rc = PLT_OK;
    hipLaunchKernelGGL(prep_sums_kernel, dim3(blocks), dim3(kEw), 0, st, int(n), X, M, psum, plo, phi, pcount);
    hipLaunchKernelGGL(prep_mean_kernel, dim3(1), dim3(kPrepThreads), 0, st, blocks, psum, plo, phi, pcount, dstat, s->stats, nv);
    hipLaunchKernelGGL(prep_dev_kernel, dim3(blocks), dim3(kEw), 0, st, int(n), M, dstat, pcount, psum, idx);
    hipLaunchKernelGGL(prep_std_kernel, dim3(1), dim3(kPrepThreads), 0, st, blocks, psum, nv, dstat, s->stats);
    hipLaunchKernelGGL(prep_targets_kernel, dim3(blocks), dim3(kEw), 0, st, int(n), M, dstat, T);
    rc = check_launch("plt_surrogate_prepare kernels");
    if (rc == PLT_OK && (hipMemcpyAsync(n_valid, nv, sizeof(uint32_t), hipMemcpyDeviceToHost, st) != hipSuccess ||
                         hipStreamSynchronize(st) != hipSuccess))
        rc = set_error(PLT_EHIP, "plt_surrogate_prepare: read-back failed");
    (void)hipFree(q);
    if (rc == PLT_OK) s->has_stats = *n_valid > 0;
    return rc;
}

int plt_surrogate_shuffle(uint32_t n, uint32_t seed, uint32_t epoch, uint32_t* out, plt_stream stream) {
    if (n == 0 || !out) return set_error(PLT_EINVAL, "plt_surrogate_shuffle: bad arguments");
    hipLaunchKernelGGL(shuffle_kernel, dim3((n + kEw - 1) / kEw), dim3(kEw), 0, static_cast<hipStream_t>(stream), n, shuffle_half(n),
                       epoch_key(seed, epoch), out);
    return check_launch("shuffle_kernel");
}

int plt_surrogate_get_stats(const plt_surrogate* s, float* y_mean, float* y_std, float* x_lo, float* x_hi) {
    if (!s || !y_mean || !y_std || !x_lo || !x_hi) return set_error(PLT_EINVAL, "plt_surrogate_get_stats: bad arguments");
    if (!s->has_stats) return set_error(PLT_ESTATE, "plt_surrogate_get_stats: no statistics set");
    float h[2 * kOut + 2 * kIn];
    if (hipMemcpy(h, s->stats, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess)
        return set_error(PLT_EHIP, "plt_surrogate_get_stats: read-back failed");
    std::memcpy(y_mean, h, kOut * sizeof(float));
    std::memcpy(y_std, h + kOut, kOut * sizeof(float));
    std::memcpy(x_lo, h + 2 * kOut, kIn * sizeof(float));
    std::memcpy(x_hi, h + 2 * kOut + kIn, kIn * sizeof(float));
    return PLT_OK;
}

int plt_surrogate_train(plt_surrogate* s, uint32_t n_valid, const uint32_t* idx, const float* X, const float* T, uint32_t batch,
                        uint32_t epochs, float lr, uint32_t seed, int graph, float* epoch_loss, plt_stream stream) {
    if (!s || !idx || !X || !T || !epoch_loss || batch == 0 || batch % 32 || batch > s->max_batch || epochs == 0 || n_valid < batch ||
        !(lr > 0.f))
        return set_error(PLT_EINVAL, "plt_surrogate_train: bad arguments (batch a multiple of 32, at most max_batch and n_valid)");
    const uint32_t spe = n_valid / batch;
    const uint64_t total = uint64_t(epochs) * spe;
    if (total >= (uint64_t(1) << 31)) return set_error(PLT_EINVAL, "plt_surrogate_train: too many steps");
    const int half = shuffle_half(n_valid);
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const TrainState ts{0u, spe, uint32_t(total), batch, n_valid, seed, s->step, lr, 0u, lr, 1.f, 1.f};
    void* q = nullptr;  // the per-step losses
    if (hipMalloc(&q, size_t(total) * 4) != hipSuccess) return set_error(PLT_ENOMEM, "plt_surrogate_train: buffer allocation failed");
    float* loss_hist = static_cast<float*>(q);
    auto* state = reinterpret_cast<TrainState*>(s->train_state);
    int rc = PLT_OK;
    if (hipMemcpyAsync(state, &ts, sizeof(ts), hipMemcpyHostToDevice, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
        rc = set_error(PLT_EHIP, "plt_surrogate_train: state upload failed");
    auto step = [&](hipStream_t qs) -> int {
        return train_launch(s, int(batch), X, T, idx, half, state, nullptr, 0.f, 1.f, 1.f, loss_hist, qs);
    };
    if (rc == PLT_OK && graph) {
        // one step captured and replayed: every step-dependent value is in the device state
        hipStream_t cs = nullptr;
        hipGraph_t g = nullptr;
        hipGraphExec_t exec = nullptr;
        if (hipStreamCreateWithFlags(&cs, hipStreamNonBlocking) != hipSuccess ||
            hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) != hipSuccess) {
            rc = set_error(PLT_EHIP, "plt_surrogate_train: capture failed to start");
        } else {
            rc = step(cs);
            if (hipStreamEndCapture(cs, &g) != hipSuccess || !g) rc = rc < 0 ? rc : set_error(PLT_EHIP, "plt_surrogate_train: capture failed");
            if (rc == PLT_OK && hipGraphInstantiate(&exec, g, nullptr, nullptr, 0) != hipSuccess)
                rc = set_error(PLT_EHIP, "plt_surrogate_train: graph instantiation failed");
            for (uint64_t k = 0; rc == PLT_OK && k < total; ++k)
                if (hipGraphLaunch(exec, st) != hipSuccess) rc = set_error(PLT_EHIP, "plt_surrogate_train: graph launch failed");
        }
        if (hipStreamSynchronize(st) != hipSuccess && rc == PLT_OK) rc = set_error(PLT_EHIP, "plt_surrogate_train: synchronize failed");
        if (exec) (void)hipGraphExecDestroy(exec);
        if (g) (void)hipGraphDestroy(g);
        if (cs) (void)hipStreamDestroy(cs);
    } else {
        for (uint64_t k = 0; rc == PLT_OK && k < total; ++k) rc = step(st);
    }
    std::vector<float> lh(total);
    if (rc == PLT_OK && (hipMemcpyAsync(lh.data(), loss_hist, total * 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
                         hipStreamSynchronize(st) != hipSuccess))
        rc = set_error(PLT_EHIP, "plt_surrogate_train: loss read-back failed");
    (void)hipStreamSynchronize(st);
    (void)hipFree(q);
    if (rc < 0) return rc;
    for (uint32_t e = 0; e < epochs; ++e) {
        double acc = 0.0;
        for (uint32_t k = 0; k < spe; ++k) acc += lh[size_t(e) * spe + k];
        epoch_loss[e] = float(acc / spe);
    }
    s->step += uint32_t(total);
    return PLT_OK;
}

// Raw GEMM (C = A * Bt^T, bf16 operands, FP32 output) for tests of the matrix-core kernel.
int plt_mlp_gemm_nt(uint32_t M, uint32_t N, uint32_t K, const void* A, const void* Bt, float* C, plt_stream stream) {
    if (!A || !Bt || !C) return set_error(PLT_EINVAL, "plt_mlp_gemm_nt: bad arguments");
    return gemm(GemmArgs{static_cast<const __bf16*>(A), static_cast<const __bf16*>(Bt), int(M), int(N), int(K), C}, static_cast<hipStream_t>(stream));
}

}  // extern "C"
