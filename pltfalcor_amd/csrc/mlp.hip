// Learned BSDF surrogate (no counterpart in the reference): a 22-128-128-128-16 ReLU MLP whose
// forward pass, backward pass and Adam update run on CDNA4 matrix cores.
//
// Every MFMA operand is bf16 and contiguous along the contracted dimension, so that a fragment (8
// consecutive k of one row) is one 16 B load. Accumulation is FP32 (v_mfma_f32_16x16x32_bf16); master
// weights and Adam moments are FP32; weight gradients are split sums over the batch reduced in a
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
// Plain NT GEMM, C[M x N] = A[M x K] * Bt[N x K]^T, the entry point plt_mlp_gemm_nt; neither training nor
// inference uses it.
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
        return set_error(PLT_EINVAL, "mlp gemm: shapes must be positive, K a multiple of 32");
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

// bf16 operand copies of one layer: W [out x in_pad] and, if Wt, Wt [in x out_pad] from the master
// weights [out x in] (padding zero).
__global__ void cast_weights_kernel(int out, int in, int in_pad, int out_pad, const float* __restrict__ Wm, __bf16* __restrict__ W,
                                    __bf16* __restrict__ Wt) {
    const int e = blockIdx.x * kEw + threadIdx.x;
    if (e >= out_pad * in_pad) return;
    const int o = e / in_pad, i = e % in_pad;
    const __bf16 v = static_cast<__bf16>(o < out && i < in ? Wm[size_t(o) * in + i] : 0.f);
    if (o < out) W[size_t(o) * in_pad + i] = v;
    if (Wt && i < in) Wt[size_t(i) * out_pad + o] = v;
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
    const L layers[4] = {{kOffW1, kHid, kIn, kInPad, kHid, s->W1, nullptr},
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

// The column sums of a block's rows, in row order; sixteen rows are read before their adds (an FP64 add
// per row is the chain, about a microsecond a block).
__device__ void column_sums(const double (&ys)[kEw][kOut], int rows, double* __restrict__ out) {
    if (threadIdx.x >= kOut) return;
    double acc = 0.0;
    for (int r0 = 0; r0 < rows; r0 += 16) {
        double v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = ys[r0 + j][threadIdx.x];  // kEw rows are there
#pragma unroll
        for (int j = 0; j < 16; ++j) acc = r0 + j < rows ? acc + v[j] : acc;
    }
    out[threadIdx.x] = acc;
}

// Pass 1, per block of kEw rows: valid count, column sums of the targets (double), and the box of
// the valid rows' inputs. Every thread takes an eighth of a feature's box (one thread per feature walked
// the block's 256 rows one after the other, with a dependent load each: 264,000 rows 152 us).
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
// Training step: three launches. mlp_train_kernel runs the forward pass, the loss and the backward
// pass, a workgroup of four waves per tile of 64 samples, whose activations and back-propagated
// gradients go from layer to layer in LDS and to memory once; mlp_weight_grad_kernel contracts them
// over the batch into split sums of the weights' gradients; grad_reduce_kernel adds the splits in
// order (and, in training, applies Adam).
//
// Products are computed transposed as in mlp_infer_kernel (weights the A operand, out[feature x
// sample]); wave w holds features 32w..32w+31. Each activation and each back-propagated gradient is
// stored twice: sample-major rows (the next product's B operand: 8 consecutive features) and
// feature-major rows (the weight gradients contract over samples, so both their operands are 8
// consecutive samples of one feature), which are also what goes to memory. A hidden unit's ReLU mask
// is one bit in the lane that computed it, which is the lane that computes its gradient.
//
// Every sum has an order that does not depend on the grid: a product adds its blocks of 32 k in order
// and its bias last, a split is a chain over at most 1/64 of the batch (rounded up to 32 rows), and the
// splits, the tiles' bias sums and the losses are added as grad_reduce_kernel says. Groups that kept their
// tiles' weight gradients in accumulators (two launches, 30 and 9 us for 16,384 rows) rounded otherwise for
// another number of groups, and summed their losses in one FP32 chain.
//
// A batch of 16,384 rows: 19.9, 7.4 and 5.9 us. The first is bound by the chain of its nine LDS barriers
// (256 tiles, one per CU; 14 us for a single tile), so a product's weights are loaded a phase ahead, and the
// barriers leave the stores of what is kept in flight. The second reads 26 MB and writes 10, 3.3 TB/s
// after the latency of its two rounds of loads. (Eighteen launches, a GEMM per product and gradient with
// every activation through memory in two layouts: 141 us.)
// ---------------------------------------------------------------------------------------
constexpr int kTRow = kFTile + 8;  // feature-major LDS rows

// What a tile leaves in memory for the weight gradients: its 64 samples of every feature, as the MFMA
// fragments that contract over samples, each 1 KB in lane order: [16 features][32 samples][lane][8 samples].
constexpr int kActX = 0, kActH1 = kActX + kInPad * kFTile, kActH2 = kActH1 + kHid * kFTile, kActH3 = kActH2 + kHid * kFTile,
              kActDY = kActH3 + kHid * kFTile, kActG3 = kActDY + kOut * kFTile, kActG2 = kActG3 + kHid * kFTile,
              kActG1 = kActG2 + kHid * kFTile, kActTile = kActG1 + kHid * kFTile;  // 104,448 B

// One split's weight gradients: W4, W3, W2, W1 (its 32 padded inputs). The biases' sums, a row per tile
// (b4, b3, b2, b1), follow them in grad_reduce_kernel's list of elements.
constexpr int kPartW4 = 0, kPartW3 = kPartW4 + kOut * kHid, kPartW2 = kPartW3 + kHid * kHid, kPartW1 = kPartW2 + kHid * kHid,
              kGradTotal = kPartW1 + kHid * kInPad;  // 38,912
constexpr int kBiasCols = kOut + 3 * kHid;
constexpr int kSplitTarget = 64;  // splits of the batch at most
// Rows of one split (a multiple of 32).
int split_len(uint32_t n) { return int((n / kKStep + kSplitTarget - 1) / kSplitTarget * kKStep); }
int tiles_of(uint32_t n) { return int((n + kFTile - 1) / kFTile); }
constexpr int kLossRows = 256;  // rows whose losses are summed in FP32; those sums are added in double
int loss_blocks(uint32_t n) { return int((n + kLossRows - 1) / kLossRows); }

// Device-side state of plt_surrogate_train: every launch of a training step reads what it needs
// from here, so one captured step replays as every step. The train kernel reads `step` and publishes
// the step it runs, its learning rate and Adam's corrections (tile 0); the reduction reads those and
// advances `step`.
struct TrainState {
    uint32_t step, steps_per_epoch, steps_total, batch, n_valid, seed, adam_t0;
    float lr0;
    uint32_t now;
    float lr, c1, c2;
};
static_assert(sizeof(TrainState) <= kTrainStateWords * 4, "train state size");

struct TrainArgs {
    int n;                 // rows of the batch
    const float *X, *T;    // inputs [. x 22] and targets [. x 16], at any address that floats may have
    const uint32_t* idx;   // with st: row i of the batch is idx[shuffle(step's i-th position)]
    int half;
    TrainState* st;
    const __bf16 *W1, *W2, *W3, *W4, *W2t, *W3t, *W4t;
    const float *b1, *b2, *b3, *b4;
    __bf16* act;           // [tiles x kActTile]
    float* bias_part;      // [tiles x kBiasCols]
    float* row_loss;       // [n]
};
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// A barrier that orders the workgroup's LDS accesses only: loads from and stores to memory stay in
// flight across it. (Within mlp_train_kernel no thread reads what another wrote to memory.)
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__global__ void __launch_bounds__(kFThreads, 2) mlp_train_kernel(TrainArgs g) {
    __shared__ __bf16 xs[kFTile * kXRow];                              // the inputs; after the first layer dY, K padded to 32
    __shared__ __bf16 sa[kFTile * kHRow], sb[kFTile * kHRow];          // sample-major, ping-pong
    __shared__ __bf16 f0[kHid * kTRow], f1[kHid * kTRow];              // feature-major, ping-pong
    __shared__ __bf16 dyt[kOut * kTRow];
    __shared__ uint32_t rows[kFTile];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int fr = lane & 15, fg = lane >> 4, fk = 8 * fg;
    const int r0 = int(blockIdx.x) * kFTile;
    __bf16* act = g.act + size_t(blockIdx.x) * kActTile;
    float* bias_part = g.bias_part + size_t(blockIdx.x) * kBiasCols;
    // rows past n repeat the last one; what they give is zeroed
    if (t < kFTile) {
        uint32_t row = uint32_t(min(r0 + t, g.n - 1));
        if (g.st) {
            const TrainState s = *g.st;
            row = g.idx[shuffle_index((s.step % s.steps_per_epoch) * s.batch + row, s.n_valid, g.half, epoch_key(s.seed, s.step / s.steps_per_epoch))];
        }
        rows[t] = row;
    } else if (t == kFTile && blockIdx.x == 0 && g.st) {
        // the cosine-decayed rate (at least 1e-6) and the corrections of Adam step adam_t0 + step + 1
        const TrainState s = *g.st;
        const double tt = double(s.adam_t0) + double(s.step) + 1.0;
        g.st->now = s.step;
        g.st->c1 = float(1.0 - pow(double(0.9f), tt));
        g.st->c2 = float(1.0 - pow(double(0.999f), tt));
        const double cs = cos(3.14159265358979323846 * double(s.step) / double(max(1u, s.steps_total)));
        g.st->lr = float(fmax(double(s.lr0) * 0.5 * (1.0 + cs), 1e-6));
    }
    using K1 = std::integral_constant<int, 1>;
    using K4 = std::integral_constant<int, 4>;
    const f32x4 zero{0.f, 0.f, 0.f, 0.f};
    // a product's weight fragments, rows 32w..32w+31 of Wm: loaded a phase ahead
    bf16x8 wf[2][4];
    auto weights = [&](auto kblocks, const __bf16* Wm, int ldw) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int kb = 0; kb < decltype(kblocks)::value; ++kb)
                wf[cb][kb] = *reinterpret_cast<const bf16x8*>(Wm + size_t(32 * w + 16 * cb + fr) * ldw + 32 * kb + fk);
    };
    // out[32w..32w+31 x 64 samples] from blocks of 32 sample-major inputs and the fragments
    auto product = [&](auto kblocks, const __bf16* in, int in_row, f32x4 (&acc)[2][4]) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int s = 0; s < 4; ++s) acc[cb][s] = zero;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int kb = 0; kb < decltype(kblocks)::value; ++kb) {
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
    auto relu = [&](const f32x4 (&acc)[2][4], const float* bias, __bf16* sm, __bf16* fm) {
        uint32_t mask = 0;
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float v = acc[cb][s][r] + bias[32 * w + 16 * cb + 4 * fg + r];
                    h[r] = static_cast<__bf16>(fmaxf(v, 0.f));
                    mask |= static_cast<float>(h[r]) > 0.f ? 1u << (16 * cb + 4 * s + r) : 0u;
                }
                store(h, cb, s, sm, fm);
            }
        return mask;
    };
    auto masked = [&](const f32x4 (&acc)[2][4], uint32_t mask, __bf16* sm, __bf16* fm) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) h[r] = static_cast<__bf16>((mask >> (16 * cb + 4 * s + r)) & 1u ? acc[cb][s][r] : 0.f);
                store(h, cb, s, sm, fm);
            }
    };
    // `count` feature-major rows to memory as fragments, 16 B per thread and round
    auto keep = [&](const __bf16* fm, int count, __bf16* dst) {
        for (int c = t; c < count * (kFTile / 8); c += kFThreads)
            *reinterpret_cast<bf16x8*>(dst + 8 * c) =
                *reinterpret_cast<const bf16x8*>(fm + (16 * (c >> 7) + fr) * kTRow + 32 * ((c >> 6) & 1) + fk);
    };
    // a bias gradient's sums over the tile: thread t adds half t % 2 of feature t / 2, as the four sums of
    // rows 4 q .. 4 q + 3 and 16 + 4 q .. of the half, those in pairs, then the halves
    auto bias_sums = [&](const __bf16* fm, float* dst) {
        const __bf16* row = fm + (t >> 1) * kTRow + 32 * (t & 1);
        float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(row + 8 * c);
#pragma unroll
            for (int j = 0; j < 8; ++j) s[(2 * c + j / 4) & 3] += static_cast<float>(v[j]);
        }
        const float h = (s[0] + s[1]) + (s[2] + s[3]);
        const float both = h + __shfl_xor(h, 1);
        if ((t & 1) == 0) dst[t >> 1] = both;
    };
    f32x4 acc[2][4];
    weights(K1{}, g.W1, kInPad);
    lds_barrier();
    {
        // thread t stages input features 2p, 2p + 1 (p = t % 16) of rows t / 16 + 16 j; rows past n
        // and padding features are zero
        const int p = t & 15, sr = t >> 4;
        const bool in = 2 * p < kIn;
        f32x2u v[kFTile / 16];
#pragma unroll
        for (int j = 0; j < kFTile / 16; ++j)
            v[j] = *reinterpret_cast<const f32x2u*>(g.X + size_t(rows[sr + 16 * j]) * kIn + (in ? 2 * p : 0));
#pragma unroll
        for (int j = 0; j < kFTile / 16; ++j) {
            const int r = sr + 16 * j;
            const bool live = in && r0 + r < g.n;
            bf16x2 pv;
            pv[0] = static_cast<__bf16>(live ? v[j].x : 0.f);
            pv[1] = static_cast<__bf16>(live ? v[j].y : 0.f);
            *reinterpret_cast<bf16x2*>(xs + r * kXRow + 2 * p) = pv;
            f1[(2 * p) * kTRow + r] = pv[0];
            f1[(2 * p + 1) * kTRow + r] = pv[1];
        }
    }
    // the lane's four targets: outputs 4 fg.. of sample 16 w + fr
    const int srow = 16 * w + fr;
    const f32x4u target = *reinterpret_cast<const f32x4u*>(g.T + size_t(rows[srow]) * kOut + 4 * fg);
    lds_barrier();
    product(K1{}, xs, kXRow, acc);
    weights(K4{}, g.W2, kHid);
    const uint32_t m1 = relu(acc, g.b1, sa, f0);
    keep(f1, kInPad, act + kActX);
    lds_barrier();
    product(K4{}, sa, kHRow, acc);
    weights(K4{}, g.W3, kHid);
    const uint32_t m2 = relu(acc, g.b2, sb, f1);
    keep(f0, kHid, act + kActH1);
    lds_barrier();
    product(K4{}, sb, kHRow, acc);
    bf16x8 w4[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) w4[kb] = *reinterpret_cast<const bf16x8*>(g.W4 + size_t(fr) * kHid + 32 * kb + fk);
    const uint32_t m3 = relu(acc, g.b3, sa, f0);
    keep(f1, kHid, act + kActH2);
    lds_barrier();
    {
        f32x4 y = zero;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) y = mfma(w4[kb], *reinterpret_cast<const bf16x8*>(sa + srow * kHRow + 32 * kb + fk), y);
        weights(K1{}, g.W4t, kOutPad);
        const bool live = r0 + srow < g.n;
        const float scale = 2.f / (float(g.n) * float(kOut));
        bf16x4 d;
        float e[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float out = y[r] + g.b4[4 * fg + r];
            e[r] = live ? out - target[r] : 0.f;
            d[r] = static_cast<__bf16>(scale * e[r]);
            dyt[(4 * fg + r) * kTRow + srow] = d[r];
        }
        *reinterpret_cast<bf16x4*>(xs + srow * kXRow + 4 * fg) = d;
        *reinterpret_cast<bf16x4*>(xs + srow * kXRow + kOut + 4 * fg) = bf16x4{};
        // the row's loss: its sixteen outputs in order, across the four lanes that hold them
        float l = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int r = 0; r < 4; ++r) l += e[r] * e[r];
            l = __shfl(l, 16 * q + fr);
        }
        if (live && fg == 0) g.row_loss[r0 + srow] = l;
    }
    keep(f0, kHid, act + kActH3);
    lds_barrier();
    {
        // b4: output t / 16 over the tile's 64 rows, by halves (32 apart, 16 apart, ... 1 apart)
        const __bf16* row = dyt + (t >> 4) * kTRow + (t & 15);
        float s = (static_cast<float>(row[0]) + static_cast<float>(row[32])) + (static_cast<float>(row[16]) + static_cast<float>(row[48]));
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if ((t & 15) == 0) bias_part[t >> 4] = s;
    }
    product(K1{}, xs, kXRow, acc);
    weights(K4{}, g.W3t, kHid);
    masked(acc, m3, sb, f1);
    keep(dyt, kOut, act + kActDY);
    lds_barrier();
    product(K4{}, sb, kHRow, acc);
    weights(K4{}, g.W2t, kHid);
    masked(acc, m2, sa, f0);
    keep(f1, kHid, act + kActG3);
    bias_sums(f1, bias_part + kOut);
    lds_barrier();
    product(K4{}, sa, kHRow, acc);
    masked(acc, m1, static_cast<__bf16*>(nullptr), f1);
    keep(f0, kHid, act + kActG2);
    bias_sums(f0, bias_part + kOut + kHid);
    lds_barrier();
    keep(f1, kHid, act + kActG1);
    bias_sums(f1, bias_part + kOut + 2 * kHid);
}

// The weights' gradients of each split of the batch, dW[out x in] = sum of G[out, row] H[in, row], a
// chain over the split's rows. Jobs 0, 1: halves of W3; 2, 3: of W2; 4: W1; 5: W4; a workgroup per job and
// split, and the jobs of a split `splits` groups apart: with a multiple of eight of them on one XCD, whose
// L2 then holds the split's rows. The groups after those sum 256 rows' losses per wave, and the rows'
// b4 sums of their four tiles.
struct WeightGradArgs {
    int n, splits, per;  // rows, splits, rows per split
    const __bf16* act;
    const float *bias_part, *row_loss;
    float* part;         // [splits x kGradTotal]
    float* loss_part;    // [loss blocks]
    float* b4_part;      // [loss blocks x kOut]
};
__global__ void __launch_bounds__(kFThreads, 2) mlp_weight_grad_kernel(WeightGradArgs g) {
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int fr = lane & 15, fg = lane >> 4;
    const int job = int(blockIdx.x) / g.splits, z = int(blockIdx.x) % g.splits;
    if (job >= 6) {
        const int b = 4 * (int(blockIdx.x) - 6 * g.splits) + w, first = b * kLossRows;
        if (first >= g.n) return;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = first + 64 * j + lane < g.n ? g.row_loss[first + 64 * j + lane] : 0.f;
        float l = (v[0] + v[2]) + (v[1] + v[3]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o);
        if (lane == 0) g.loss_part[b] = l;
        if (lane < kOut) {
            const int tiles = (g.n + kFTile - 1) / kFTile;
            float s = 0.f;
            for (int k = 4 * b; k < min(4 * b + 4, tiles); ++k) s += g.bias_part[size_t(k) * kBiasCols + lane];
            g.b4_part[size_t(b) * kOut + lane] = s;
        }
        return;
    }
    const int kbeg = z * (g.per / kKStep), kend = min(g.n / kKStep, kbeg + g.per / kKStep);
    float* part = g.part + size_t(z) * kGradTotal;
    using N1 = std::integral_constant<int, 1>;
    using N2 = std::integral_constant<int, 2>;
    using N4 = std::integral_constant<int, 4>;
    using N8 = std::integral_constant<int, 8>;
    // dW[a .. a + 16 kA x b .. b + 16 kB] from the arrays at offA and offB
    auto chain = [&](auto na, auto nb, int offA, int a, int offB, int b, float* dst, int ld) {
        constexpr int kA = decltype(na)::value, kB = decltype(nb)::value;
        f32x4 acc[kA][kB];
#pragma unroll
        for (int i = 0; i < kA; ++i)
#pragma unroll
            for (int c = 0; c < kB; ++c) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto blocks = [&](auto nu, int k0) {  // all loads in flight, then the products in order
            constexpr int kU = decltype(nu)::value;
            bf16x8 ga[kU][kA], hb[kU][kB];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const __bf16* base = g.act + size_t((k0 + u) >> 1) * kActTile + 512 * ((k0 + u) & 1) + 8 * lane;
#pragma unroll
                for (int i = 0; i < kA; ++i) ga[u][i] = *reinterpret_cast<const bf16x8*>(base + offA + (a + 16 * i) * kFTile);
#pragma unroll
                for (int c = 0; c < kB; ++c) hb[u][c] = *reinterpret_cast<const bf16x8*>(base + offB + (b + 16 * c) * kFTile);
            }
            __builtin_amdgcn_sched_barrier(0);  // the compiler would move each load to its product
#pragma unroll
            for (int u = 0; u < kU; ++u)
#pragma unroll
                for (int i = 0; i < kA; ++i)
#pragma unroll
                    for (int c = 0; c < kB; ++c) acc[i][c] = mfma(ga[u][i], hb[u][c], acc[i][c]);
        };
        int k = kbeg;
        for (; k + 4 <= kend; k += 4) blocks(N4{}, k);
        for (; k < kend; ++k) blocks(N1{}, k);
        // D layout: the lane holds rows 4 fg + r of column fr of each 16 x 16 block
#pragma unroll
        for (int i = 0; i < kA; ++i)
#pragma unroll
            for (int c = 0; c < kB; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) dst[(a + 16 * i + 4 * fg + r) * ld + b + 16 * c + fr] = acc[i][c][r];
    };
    if (job < 4) {
        const bool third = job < 2;
        chain(N1{}, N8{}, third ? kActG3 : kActG2, 64 * (job & 1) + 16 * w, third ? kActH2 : kActH1, 0, part + (third ? kPartW3 : kPartW2), kHid);
    } else if (job == 4) {
        chain(N2{}, N2{}, kActG1, 32 * w, kActX, 0, part + kPartW1, kInPad);
    } else {
        chain(N1{}, N2{}, kActDY, 0, kActH3, 32 * w, part + kPartW4, kHid);
    }
}

// Every gradient from its partial sums, in one launch. A weight has a partial per split, a hidden bias one
// per tile, an output's bias one per 256 rows; four threads per element each add partials q, q + 4, ... in
// order, and the four sums are combined in order. A block takes 64 weights, whose (at most 16) partials a
// thread loads by itself, or 16 biases, whose many partials the block's threads stage 256 at a time.
// The sum goes to `grads`, or (grads null) through Adam to the FP32 master parameters and their bf16
// copies, whose padding stays zero; the learning rate and the corrections come from the arguments, or with
// `st` from the device state that the train kernel published. Block 0 then also records the step's mean
// loss, the losses' sums added in double in order, and advances the state's step, which no thread of this
// kernel reads.
struct WeightCopies {
    __bf16 *W1, *W2, *W2t, *W3, *W3t, *W4, *W4t;
};
struct ReduceArgs {
    int splits, tiles, lblocks;
    const float *part, *bias_part, *b4_part, *loss_part;
    float* grads;
    float *p, *m, *v;
    TrainState* st;
    float lr, c1, c2;
    WeightCopies w;
    float* loss_hist;
};
constexpr int kReduceLanes = 64, kReduceBias = 16;  // weights and biases per block
constexpr int kWeightBlocks = kGradTotal / kReduceLanes, kReduceBlocks = kWeightBlocks + kBiasCols / kReduceBias;
static_assert(kGradTotal % kReduceLanes == 0 && kBiasCols % kReduceBias == 0 && kOut == kReduceBias, "whole blocks");
__global__ void __launch_bounds__(256) grad_reduce_kernel(ReduceArgs a) {
    __shared__ float sums[4][kReduceLanes];
    __shared__ float stage[256][kReduceBias];
    const int t = threadIdx.x, block = int(blockIdx.x);
    const bool bias = block >= kWeightBlocks;
    if (!bias) {
        const int el = t & (kReduceLanes - 1), q = t >> 6;
        float v[kSplitTarget / 4], acc = 0.f;
#pragma unroll
        for (int j = 0; j < kSplitTarget / 4; ++j) {
            const int z = q + 4 * j;
            v[j] = z < a.splits ? a.part[size_t(z) * kGradTotal + block * kReduceLanes + el] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < kSplitTarget / 4; ++j) acc += v[j];
        sums[q][el] = acc;
    } else {
        const int first = (block - kWeightBlocks) * kReduceBias, el = t & (kReduceBias - 1), row = t / kReduceBias;
        const float* src = (first == 0 ? a.b4_part : a.bias_part + first) + el;
        const size_t stride = first == 0 ? kOut : kBiasCols;
        const int count = first == 0 ? a.lblocks : a.tiles;
        float acc = 0.f;
        for (int z0 = 0; z0 < count; z0 += 256) {
            float v[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int z = z0 + row + 16 * j;
                v[j] = z < count ? src[size_t(z) * stride] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) stage[row + 16 * j][el] = v[j];
            __syncthreads();
            if (row < 4) {
#pragma unroll 16
                for (int j = 0; j < 64; ++j) acc += stage[row + 4 * j][el];
            }
            __syncthreads();
        }
        if (row < 4) sums[row][el] = acc;
    }
    __syncthreads();
    if (a.st && block == 0 && t >= 64 && t < 128) {
        const int el = t & 63;
        double l = 0.0;
        for (int z0 = 0; z0 < a.lblocks; z0 += 64) {
            const float v = z0 + el < a.lblocks ? a.loss_part[z0 + el] : 0.f;
            const int m = min(64, a.lblocks - z0);
            for (int k = 0; k < m; ++k) l += double(__shfl(v, k));
        }
        if (el == 0) {
            const uint32_t now = a.st->now;
            a.loss_hist[now] = float(l / (double(a.st->batch) * kOut));
            a.st->step = now + 1u;
        }
    }
    if (t >= (bias ? kReduceBias : kReduceLanes)) return;
    const int el = t, e = bias ? kGradTotal + (block - kWeightBlocks) * kReduceBias + el : block * kReduceLanes + el;
    const float ge = (sums[0][el] + sums[1][el]) + (sums[2][el] + sums[3][el]);
    // the element's parameter and, for a weight, its places in the bf16 copies
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
        if (Wt) *Wt = h;
    }
}
WeightCopies weight_copies(const plt_surrogate* s) { return WeightCopies{s->W1, s->W2, s->W2t, s->W3, s->W3t, s->W4, s->W4t}; }

// The launches of a step over n rows of X and T (with `st`, rows idx[shuffle]): the activations and
// gradients, the splits' sums, then their sums into `grads` or through Adam.
int train_launch(plt_surrogate* s, int n, const float* X, const float* T, const uint32_t* idx, int half, TrainState* st, float* grads, float lr,
                 float c1, float c2, float* loss_hist, hipStream_t qs) {
    const int tiles = tiles_of(uint32_t(n)), lblocks = loss_blocks(uint32_t(n));
    const int per = split_len(uint32_t(n)), splits = (n + per - 1) / per;
    const TrainArgs ta{n, X, T, idx, half, st, s->W1, s->W2, s->W3, s->W4, s->W2t, s->W3t, s->W4t,
                       s->params + kOffB1, s->params + kOffB2, s->params + kOffB3, s->params + kOffB4, s->act, s->bias_part, s->row_loss};
    hipLaunchKernelGGL(mlp_train_kernel, dim3(tiles), dim3(kFThreads), 0, qs, ta);
    int rc = check_launch("mlp_train_kernel");
    if (rc < 0) return rc;
    const WeightGradArgs wa{n, splits, per, s->act, s->bias_part, s->row_loss, s->part, s->loss_part, s->b4_part};
    hipLaunchKernelGGL(mlp_weight_grad_kernel, dim3(6 * splits + (lblocks + 3) / 4), dim3(kFThreads), 0, qs, wa);
    if ((rc = check_launch("mlp_weight_grad_kernel")) < 0) return rc;
    const ReduceArgs ra{splits, tiles, lblocks, s->part, s->bias_part, s->b4_part, s->loss_part, grads, s->params, s->adam_m, s->adam_v, st, lr, c1,
                        c2, weight_copies(s), loss_hist};
    hipLaunchKernelGGL(grad_reduce_kernel, dim3(kReduceBlocks), dim3(256), 0, qs, ra);
    return check_launch("grad_reduce_kernel");
}

// The mean loss of the last train_launch over n rows.
int read_loss(plt_surrogate* s, uint32_t n, float* loss, hipStream_t st) {
    std::vector<float> lp(static_cast<size_t>(loss_blocks(n)));
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
    A(&s->W1, size_t(kHid) * kInPad);
    A(&s->W2, size_t(kHid) * kHid); A(&s->W2t, size_t(kHid) * kHid);
    A(&s->W3, size_t(kHid) * kHid); A(&s->W3t, size_t(kHid) * kHid);
    A(&s->W4, size_t(kOut) * kHid); A(&s->W4t, size_t(kHid) * kOutPad);
    A(&s->act, size_t(tiles_of(max_batch)) * kActTile);
    A(&s->bias_part, size_t(tiles_of(max_batch)) * kBiasCols);
    A(&s->row_loss, max_batch);
    A(&s->part, size_t(std::min(kSplitTarget, int(max_batch / kKStep))) * kGradTotal);
    A(&s->loss_part, size_t(loss_blocks(max_batch)));
    A(&s->b4_part, size_t(loss_blocks(max_batch)) * kOut);
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
