// Learned chemistry surrogate: a small MLP (T, p, Y_k, dt) -> (dT, dY_k)
// trained and evaluated on the GPU with BF16 matrix-core (MFMA) GEMMs and
// FP32 accumulation, Adam on FP32 master weights.
//
// Layers: 16 (NIN = NS + 3 features, zero-padded) -> 128 -> 128 -> 128 -> 16
// (NOUT = NS + 1 outputs, zero-padded), GELU (tanh form) on the hidden layers.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "surrogate.h"

#include <utility>
#include "surrogate_device.h"

namespace lbm {
namespace sur {

// ------------------------------------------------------- gradient kernel
// Forward pass, loss and all gradients of the batch in one pass over its rows:
// a block takes GROWS rows at a time through the four layers and back and keeps
// its weight gradients in registers.  One wavefront per 16 neurons of the
// 128-wide layers: with Z^T = W H^T (A operand the weights, i = neuron; B
// operand the batch rows) the pre-activations a wavefront makes going forward
// are in its own registers, in place, when the backward pass wants gelu' of
// them.  Activations and dZ pass between wavefronts as BF16 in LDS, by row for
// the next layer's product and transposed for the weight gradients, whose
// reduction index is the row; both strides spread 16 rows of 16 bytes over all
// banks.  Weights are read where they are used (72 KiB from L2).
// Bound by the chain of eight phases between barriers.  With a pass per layer
// and operand (forward, transposes, partial products, their sums, bias sums:
// 33 launches) a caller's gradient of 4096 rows took 395 us, host copies
// included, and takes 127.
constexpr int GWAVES = 8, GROWS = 64, GTILES = GROWS / 16, GSTEPS = GROWS / 32;
constexpr int GRAD_BLOCKS = 256;       // one per CU: more rows go round
constexpr int HSTRIDE = 128 + 8, TSTRIDE = GROWS + 8, DSTRIDE = 16 + 8;
static_assert(GWAVES * 16 == 128, "one wavefront per 16 neurons");

// Offsets of W[L] and b[L] in the flat gradient.
constexpr int grad_w(int L) { return frag_offset(L) + bias_offset(L); }
constexpr int grad_b(int L) { return grad_w(L) + DIMS[L] * DIMS[L + 1]; }
static_assert(grad_b(NL - 1) + DIMS[NL] == NPARAM, "flat gradient");

// Four neurons n0 + 0..3 of row r, by row and transposed.
__device__ __forceinline__ void put_rows(uint16_t* h, int r, int n0, const v4s x)
{
    uint2 u;
    __builtin_memcpy(&u, &x, 8);
    *reinterpret_cast<uint2*>(h + r * HSTRIDE + n0) = u;
}
__device__ __forceinline__ void put_cols(uint16_t* hT, int r, int n0, const v4s x)
{
#pragma unroll
    for (int q = 0; q < 4; ++q) hT[(n0 + q) * TSTRIDE + r] = (uint16_t)x[q];
}
// acc += A[16 a0 + ..][rows] B[16 b0 + ..][rows]^T over the block's rows
__device__ __forceinline__ v4f row_products(const v8bf a[GSTEPS], const uint16_t* bT, int b0, v4f acc)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int s = 0; s < GSTEPS; ++s)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a[s], load_frag8(bT + (16 * b0 + (lane & 15)) * TSTRIDE + 32 * s + 8 * (lane >> 4)), acc, 0, 0, 0);
    return acc;
}
__device__ __forceinline__ void row_operand(const uint16_t* aT, int a0, v8bf a[GSTEPS])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int s = 0; s < GSTEPS; ++s)
        a[s] = load_frag8(aT + (16 * a0 + (lane & 15)) * TSTRIDE + 32 * s + 8 * (lane >> 4));
}
// sum over the block's rows of A: the product with ones
__device__ __forceinline__ v4f row_sums(const v8bf a[GSTEPS], v4f acc)
{
    v8bf one;
#pragma unroll
    for (int e = 0; e < 8; ++e) one[e] = (__bf16)1.0f;
#pragma unroll
    for (int s = 0; s < GSTEPS; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s], one, acc, 0, 0, 0);
    return acc;
}
// out[bt] = W[16 w0 + ..][0..128) h[row][0..128)^T for the block's row tiles
__device__ __forceinline__ void product128(const uint16_t* W, int w0, const uint16_t* h, v4f out[GTILES])
{
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    v8bf a[KSTEPS];
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) a[s] = load_frag8(W + (16 * w0 + j) * 128 + 32 * s + 8 * g);
#pragma unroll
    for (int bt = 0; bt < GTILES; ++bt) {
        out[bt] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
            out[bt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a[s], load_frag8(h + (16 * bt + j) * HSTRIDE + 32 * s + 8 * g), out[bt], 0, 0, 0);
    }
}
__device__ __forceinline__ v4s bf_frag(const v4f z)
{
    v4s r;
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] = (short)f2bf(z[q]);
    return r;
}

// grid: at most GRAD_BLOCKS blocks of 64 GWAVES threads, M a multiple of 16;
// part [gridDim.x][NPARAM] receives each block's share of the flat gradient,
// loss_rows [M] the rows' squared errors.  dZ of the output layer is that of
// the mean-squared loss over NOUT outputs, 2 (z - t) / (M NOUT), and 0 for
// padded outputs and for rows past M.
__global__ __launch_bounds__(64 * GWAVES) void k_grad(Mlp net, const uint16_t* X, const float* T, int M, float* part,
                                                      float* loss_rows)
{
    __shared__ __align__(16) uint16_t h[2][GROWS * HSTRIDE];   // by row: activations, then dZ
    __shared__ __align__(16) uint16_t hT[3][128 * TSTRIDE];    // transposed activations
    __shared__ __align__(16) uint16_t dT[2][128 * TSTRIDE];    // transposed dZ
    __shared__ __align__(16) uint16_t xT[16 * TSTRIDE], d3T[16 * TSTRIDE], d3[GROWS * DSTRIDE];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, j = lane & 15, g = lane >> 4;
    const int n0 = 16 * w + 4 * g;  // the neurons of this lane's D fragments
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    v4f g0 = zero, g1[8], g2[8], g3 = zero, s0 = zero, s1 = zero, s2 = zero, s3 = zero;
#pragma unroll
    for (int t = 0; t < 8; ++t) g1[t] = g2[t] = zero;
    for (int r0 = blockIdx.x * GROWS; r0 < M; r0 += gridDim.x * GROWS) {
        v4f z0[GTILES], z1[GTILES], z2[GTILES], acc[GTILES];
        v8bf a[GSTEPS];
        {  // ---- layer 0, K = 16
            const v4s wf = load_frag(net.Wb[0] + (16 * w + j) * 16 + 4 * g);
            const v4f b = bias_frag(net.b[0], 16 * w, lane);
#pragma unroll
            for (int bt = 0; bt < GTILES; ++bt) {
                const int r = 16 * bt + j;
                v4s x = {0, 0, 0, 0};
                if (r0 + r < M) x = load_frag(X + (size_t)(r0 + r) * 16 + 4 * g);
                if (w == bt) put_cols(xT, r, 4 * g, x);
                z0[bt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wf, x, zero, 0, 0, 0) + b;
                const v4s hf = act_frag(z0[bt]);
                put_rows(h[0], r, n0, hf);
                put_cols(hT[0], r, n0, hf);
            }
        }
        __syncthreads();
        // ---- layers 1 and 2
        auto hidden = [&](int L, const uint16_t* from, uint16_t* to, uint16_t* toT, v4f z[GTILES]) {
            product128(net.Wb[L], w, from, z);
            const v4f b = bias_frag(net.b[L], 16 * w, lane);
#pragma unroll
            for (int bt = 0; bt < GTILES; ++bt) {
                z[bt] += b;
                const v4s hf = act_frag(z[bt]);
                put_rows(to, 16 * bt + j, n0, hf);
                put_cols(toT, 16 * bt + j, n0, hf);
            }
        };
        hidden(1, h[0], h[1], hT[1], z1);
        __syncthreads();
        hidden(2, h[1], h[0], hT[2], z2);
        __syncthreads();
        // ---- output layer and loss: row tile w
        if (w < GTILES) {
            const int r = 16 * w + j, row = r0 + r;
            v4f z = zero;
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s)
                z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_frag8(net.Wb[3] + j * 128 + 32 * s + 8 * g),
                                                           load_frag8(h[0] + r * HSTRIDE + 32 * s + 8 * g), z, 0, 0, 0);
            z += bias_frag(net.b[3], 0, lane);
            v4f dz = zero;
            float sum = 0.f;
            if (row < M) {
                const v4f t = *reinterpret_cast<const v4f*>(T + (size_t)row * 16 + 4 * g);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (4 * g + q < NOUT) {
                        const float d = z[q] - t[q];
                        sum += d * d;
                        dz[q] = 2.f * d / (float)(M * NOUT);
                    }
            }
            sum += __shfl_xor(sum, 16);
            sum += __shfl_xor(sum, 32);
            if (g == 0 && row < M) loss_rows[row] = sum;
            const v4s df = bf_frag(dz);
            uint2 u;
            __builtin_memcpy(&u, &df, 8);
            *reinterpret_cast<uint2*>(d3 + r * DSTRIDE + 4 * g) = u;
            put_cols(d3T, r, 4 * g, df);
        }
        __syncthreads();
        // ---- back through the output layer; its weight gradient
        {
            const v4s wf = load_frag(net.WbT[3] + (16 * w + j) * 16 + 4 * g);
#pragma unroll
            for (int bt = 0; bt < GTILES; ++bt) {
                const int r = 16 * bt + j;
                v4f d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wf, load_frag(d3 + r * DSTRIDE + 4 * g), zero, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 4; ++q) d[q] *= gelu_grad(z2[bt][q]);
                const v4s df = bf_frag(d);
                put_rows(h[1], r, n0, df);
                put_cols(dT[0], r, n0, df);
            }
            row_operand(d3T, 0, a);
            g3 = row_products(a, hT[2], w, g3);
            s3 = row_sums(a, s3);
        }
        __syncthreads();
        // ---- layer 2
        product128(net.WbT[2], w, h[1], acc);
#pragma unroll
        for (int bt = 0; bt < GTILES; ++bt) {
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[bt][q] *= gelu_grad(z1[bt][q]);
            const v4s df = bf_frag(acc[bt]);
            put_rows(h[0], 16 * bt + j, n0, df);
            put_cols(dT[1], 16 * bt + j, n0, df);
        }
        row_operand(dT[0], w, a);
#pragma unroll
        for (int t = 0; t < 8; ++t) g2[t] = row_products(a, hT[1], t, g2[t]);
        s2 = row_sums(a, s2);
        __syncthreads();
        // ---- layer 1
        product128(net.WbT[1], w, h[0], acc);
#pragma unroll
        for (int bt = 0; bt < GTILES; ++bt) {
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[bt][q] *= gelu_grad(z0[bt][q]);
            put_cols(dT[0], 16 * bt + j, n0, bf_frag(acc[bt]));
        }
        row_operand(dT[1], w, a);
#pragma unroll
        for (int t = 0; t < 8; ++t) g1[t] = row_products(a, hT[0], t, g1[t]);
        s1 = row_sums(a, s1);
        __syncthreads();
        // ---- layer 0
        row_operand(dT[0], w, a);
        g0 = row_products(a, xT, 0, g0);
        s0 = row_sums(a, s0);
        __syncthreads();
    }
    // ---- the block's share, in the flat order
    float* out = part + (size_t)blockIdx.x * NPARAM;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        out[grad_w(0) + (n0 + q) * 16 + j] = g0[q];
        out[grad_w(3) + (4 * g + q) * 128 + 16 * w + j] = g3[q];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            out[grad_w(1) + (n0 + q) * 128 + 16 * t + j] = g1[t][q];
            out[grad_w(2) + (n0 + q) * 128 + 16 * t + j] = g2[t][q];
        }
        if (j == 0) {
            out[grad_b(0) + n0 + q] = s0[q];
            out[grad_b(1) + n0 + q] = s1[q];
            out[grad_b(2) + n0 + q] = s2[q];
            if (w == 0) out[grad_b(3) + 4 * g + q] = s3[q];
        }
    }
}

// Sums the blocks' shares in a fixed order: 64 parameters per block of 256, a
// quarter of the shares per wavefront.
__global__ __launch_bounds__(256) void k_grad_sum(const float* part, int nblk, float* grad)
{
    __shared__ float red[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    float s = 0.f;
    if (i < NPARAM) {
#pragma unroll 8
        for (int b = w; b < nblk; b += 4) s += part[(size_t)b * NPARAM + i];
    }
    red[w][lane] = s;
    __syncthreads();
    if (w == 0 && i < NPARAM) grad[i] = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

// Adam on FP32 master weights; refreshes the BF16 copies W and W^T.  The
// bias corrections of iteration *it are c12[2 it] and c12[2 it + 1].
__global__ void k_adam(float* w, const float* g, float* m, float* v, int n, float lr, float b1, float b2, float eps,
                       const float* c12, const int* it, uint16_t* wb, uint16_t* wbT, int rows, int cols)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float c1 = c12[2 * *it], c2 = c12[2 * *it + 1];
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    if (wb) {
        wb[i] = f2bf(wi);
        const int r = i / cols, c = i % cols;
        wbT[(size_t)c * rows + r] = f2bf(wi);
    }
}

__global__ void k_to_bf(const float* in, uint16_t* out, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = f2bf(in[i]);
}

// W[L] (FP32, [N][K]) into the fragment-ordered BF16 block of layer L: the
// 16-deep K-steps of layer 0, the 32-deep ones (k32_neuron order) of the others.
__global__ void k_to_frag(const float* W, int N, int K, uint16_t* Wf)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N * K) return;
    if (K == 16) {
        const int q = i & 3, lane = (i >> 2) & 63, t = i >> 8;
        const int n = 16 * t + (lane & 15), k = 4 * (lane >> 4) + q;
        Wf[i] = f2bf(W[n * K + k]);
        return;
    }
    const int KS = K / 32;
    const int e = i & 7, lane = (i >> 3) & 63, ts = i >> 9;
    const int t = ts / KS, s = ts % KS;
    const int n = 16 * t + (lane & 15), k = k32_neuron(s, lane >> 4, e);
    Wf[i] = f2bf(W[n * K + k]);
}

__global__ void k_to_bf_T(const float* in, int rows, int cols, uint16_t* out, uint16_t* outT)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * cols) return;
    const uint16_t h = f2bf(in[i]);
    out[i] = h;
    outT[(size_t)(i % cols) * rows + i / cols] = h;
}

// ------------------------------------------------------------------ host
static inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// ------------------------------------------------------ inference kernel
// 512 threads (8 wavefronts x 32 rows), weights and biases staged in LDS
// once per block, grid-stride over groups of 256 rows.
constexpr int IWAVES = 8, IROWS = IWAVES * 32;

__global__ __launch_bounds__(512) void k_mlp_infer(Mlp net, const float* X, int M, float* Y)
{
    __shared__ __align__(16) uint16_t Wf[FRAG_TOTAL];
    __shared__ float bias[BIAS_TOTAL];
    __shared__ __align__(16) uint16_t xin[IWAVES][32 * 16];
    __shared__ __align__(16) float yout[IWAVES][32 * 16];
    stage_net(net, Wf, bias);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int base = blockIdx.x * IROWS; base < M; base += gridDim.x * IROWS) {
        __syncthreads();
        for (int i = lane; i < 32 * 16; i += 64) {
            const int row = base + wave * 32 + i / 16;
            xin[wave][i] = f2bf(row < M ? X[(size_t)row * 16 + (i % 16)] : 0.f);
        }
        __syncthreads();
        const v4s x[2] = {input_frag(xin[wave], 0), input_frag(xin[wave], 1)};
        v4f y[2];
        mlp_rows32(Wf, bias, x, y);
        output_frag(yout[wave], 0, y[0]);
        output_frag(yout[wave], 1, y[1]);
        __syncthreads();
        for (int i = lane; i < 32 * 16; i += 64) {
            const int row = base + wave * 32 + i / 16;
            if (row < M) Y[(size_t)row * 16 + (i % 16)] = yout[wave][i];
        }
    }
}

int infer_grid(int M)
{
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    const int groups = cdiv(M, IROWS);
    return groups < cus ? (groups > 0 ? groups : 1) : cus;
}

void mlp_infer(const Mlp& net, const float* X, int M, float* Y, hipStream_t s)
{
    hipLaunchKernelGGL(k_mlp_infer, dim3(infer_grid(M)), dim3(512), 0, s, net, X, M, Y);
}

// ---------------------------------------------------- training data
// Per-block partial sum, sum of squares, min and max of the 32 capture
// columns: thread t owns column t % 32 of rows (t / 32) + 8 (block + k grid).
__global__ __launch_bounds__(256) void k_cap_stats(const float* cap, int64_t rows, double* part)
{
    __shared__ double red[256][4];
    const int q = threadIdx.x & 31, g = threadIdx.x >> 5;
    double s = 0, s2 = 0, lo = INFINITY, hi = -INFINITY;
    for (int64_t r = (int64_t)blockIdx.x * 8 + g; r < rows; r += (int64_t)gridDim.x * 8) {
        const double x = cap[r * CAP_STRIDE + q];
        s += x;
        s2 += x * x;
        lo = x < lo ? x : lo;
        hi = x > hi ? x : hi;
    }
    red[threadIdx.x][0] = s;
    red[threadIdx.x][1] = s2;
    red[threadIdx.x][2] = lo;
    red[threadIdx.x][3] = hi;
    __syncthreads();
    if (g == 0) {
        for (int k = 1; k < 8; ++k) {
            const double* o = red[k * 32 + q];
            s += o[0];
            s2 += o[1];
            lo = o[2] < lo ? o[2] : lo;
            hi = o[3] > hi ? o[3] : hi;
        }
        double* p = part + ((size_t)blockIdx.x * 32 + q) * 4;
        p[0] = s;
        p[1] = s2;
        p[2] = lo;
        p[3] = hi;
    }
}

// Final reduction (fixed order) into the normalisation record.  Feature
// scales are at least 1e-3 of the feature's mean, so that rounding-level
// spread (a composition that barely varies) maps to small network inputs;
// the envelope is the captured [min, max] widened by 10 % of its width plus
// 1e-3 of the mean.  A target column with no spread (an inert species) gets
// scale 0: it is not learned and decodes to its mean.
// envelope_only: keep the normalisation (the network's input and output
// scaling) and reset only the training envelope (SS_LO, SS_HI).
__global__ void k_cap_stats_final(const double* part, int nblk, int64_t rows, float* st, int envelope_only)
{
    const int q = threadIdx.x;
    if (q >= 32) return;
    double s = 0, s2 = 0, lo = INFINITY, hi = -INFINITY;
    for (int b = 0; b < nblk; ++b) {
        const double* p = part + ((size_t)b * 32 + q) * 4;
        s += p[0];
        s2 += p[1];
        lo = p[2] < lo ? p[2] : lo;
        hi = p[3] > hi ? p[3] : hi;
    }
    const double mean = s / (double)rows;
    const double var = s2 / (double)rows - mean * mean;
    double sd = var > 0 ? sqrt(var) : 0.0;
    if (q < 16) {
        const bool used = q < NIN;
        sd = fmax(sd, 1e-3 * fabs(mean));
        if (!(sd > 1e-30)) sd = 1.0;
        const double margin = 0.1 * (hi - lo) + 1e-3 * fabs(mean);
        if (!envelope_only) {
            st[SS_FMEAN + q] = used ? (float)mean : 0.f;
            st[SS_FSTD + q] = used ? (float)sd : 1.f;
        }
        st[SS_LO + q] = used ? (float)(lo - margin) : 0.f;
        st[SS_HI + q] = used ? (float)(hi + margin) : 0.f;
    } else if (!envelope_only) {
        if (!(sd > 1e-6 * fabs(mean)) || !(sd > 1e-30)) sd = 0.0;
        const int t = q - 16;
        const bool used = t < NOUT;
        st[SS_TMEAN + t] = used ? (float)mean : 0.f;
        st[SS_TSTD + t] = used ? (float)sd : 0.f;
    }
}

void capture_stats(const float* cap, int64_t rows, double* part, float* stats, hipStream_t s, bool envelope_only)
{
    hipLaunchKernelGGL(k_cap_stats, dim3(STATS_BLOCKS), dim3(256), 0, s, cap, rows, part);
    hipLaunchKernelGGL(k_cap_stats_final, dim3(1), dim3(64), 0, s, part, STATS_BLOCKS, rows, stats,
                       envelope_only ? 1 : 0);
}

__device__ inline uint64_t splitmix(uint64_t z)
{
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void k_gather(const float* cap, int64_t rows, const float* st, uint64_t seed, const int* itp, int B,
                         uint16_t* X, float* T)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    const int it = *itp;
    const uint64_t h = splitmix(seed ^ splitmix(((uint64_t)it << 32) | (uint64_t)b));
    const int64_t r = (int64_t)(h % (uint64_t)rows);
    const float* row = cap + r * CAP_STRIDE;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        X[(size_t)b * 16 + q] = f2bf(q < NIN ? (row[q] - st[SS_FMEAN + q]) / st[SS_FSTD + q] : 0.f);
        T[(size_t)b * 16 + q] =
            (q < NOUT && st[SS_TSTD + q] > 0.f) ? (row[16 + q] - st[SS_TMEAN + q]) / st[SS_TSTD + q] : 0.f;
    }
}

void gather_batch(const float* cap, int64_t rows, const float* stats, uint64_t seed, const int* it, int B,
                  uint16_t* X, float* T, hipStream_t s)
{
    hipLaunchKernelGGL(k_gather, dim3(cdiv(B, 256)), dim3(256), 0, s, cap, rows, stats, seed, it, B, X, T);
}

__global__ void k_next_iteration(int* it) { *it += 1; }

void next_iteration(int* it, hipStream_t s) { hipLaunchKernelGGL(k_next_iteration, dim3(1), dim3(1), 0, s, it); }

// out[*idx] (out[0] without idx) = sum(lr[0..B)) * scale
__global__ __launch_bounds__(256) void k_loss_sum(const float* lr, int B, float scale, float* out, const int* idx)
{
    __shared__ float red[256];
    float s = 0.f;
    for (int i = threadIdx.x; i < B; i += 256) s += lr[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[idx ? *idx : 0] = red[0] * scale;
}

void loss_sum(const float* loss_rows, int B, float scale, float* out, hipStream_t s, const int* idx)
{
    hipLaunchKernelGGL(k_loss_sum, dim3(1), dim3(256), 0, s, loss_rows, B, scale, out, idx);
}

static int grad_blocks(int M) { return cdiv(M, GROWS) < GRAD_BLOCKS ? cdiv(M, GROWS) : GRAD_BLOCKS; }

void mlp_grad(const Mlp& net, const uint16_t* X, const float* T, int M, Work& w, hipStream_t s)
{
    const int nblk = grad_blocks(M);
    hipLaunchKernelGGL(k_grad, dim3(nblk), dim3(64 * GWAVES), 0, s, net, X, T, M, w.part, w.loss_rows);
    hipLaunchKernelGGL(k_grad_sum, dim3(cdiv(NPARAM, 64)), dim3(256), 0, s, w.part, nblk, w.grad);
}

void adam_corrections(int first_step, int iters, float* c12)
{
    for (int k = 0; k < iters; ++k) {
        const float step = (float)(first_step + k);
        c12[2 * k] = 1.f - powf(ADAM_B1, step);
        c12[2 * k + 1] = 1.f - powf(ADAM_B2, step);
    }
}

void mlp_adam(Mlp& net, Work& w, float lr, const float* c12, const int* it, hipStream_t s)
{
    const float b1 = ADAM_B1, b2 = ADAM_B2, eps = ADAM_EPS;
    for (int L = 0; L < NL; ++L) {
        const int n = DIMS[L] * DIMS[L + 1];
        hipLaunchKernelGGL(k_adam, dim3(cdiv(n, 256)), dim3(256), 0, s, net.W[L], w.gW[L], net.mW[L], net.vW[L], n, lr,
                           b1, b2, eps, c12, it, net.Wb[L], net.WbT[L], DIMS[L + 1], DIMS[L]);
        hipLaunchKernelGGL(k_adam, dim3(cdiv(DIMS[L + 1], 256)), dim3(256), 0, s, net.b[L], w.gb[L], net.mb[L],
                           net.vb[L], DIMS[L + 1], lr, b1, b2, eps, c12, it, (uint16_t*)nullptr, (uint16_t*)nullptr, 0,
                           1);
        hipLaunchKernelGGL(k_to_frag, dim3(cdiv(n, 256)), dim3(256), 0, s, net.W[L], DIMS[L + 1], DIMS[L],
                           net.Wf + frag_offset(L));
    }
}

void to_bf16(const float* in, uint16_t* out, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL(k_to_bf, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, in, out, n);
}

void refresh_bf16(Mlp& net, hipStream_t s)
{
    for (int L = 0; L < NL; ++L) {
        const int n = DIMS[L] * DIMS[L + 1];
        hipLaunchKernelGGL(k_to_bf_T, dim3(cdiv(n, 256)), dim3(256), 0, s, net.W[L], DIMS[L + 1], DIMS[L], net.Wb[L],
                           net.WbT[L]);
        hipLaunchKernelGGL(k_to_frag, dim3(cdiv(n, 256)), dim3(256), 0, s, net.W[L], DIMS[L + 1], DIMS[L],
                           net.Wf + frag_offset(L));
    }
}

}  // namespace sur
}  // namespace lbm

namespace lbm {
namespace sur {

// Glorot-uniform initial weights from a SplitMix64 stream, zero biases.
hipError_t mlp_alloc(Mlp& net, uint64_t seed, hipStream_t s)
{
    uint64_t st = seed;
    auto rnd = [&]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (double)(z >> 11) * (1.0 / 9007199254740992.0);
    };
    hipError_t e;
    if ((e = hipMalloc((void**)&net.Wf, 2 * FRAG_TOTAL)) != hipSuccess) return e;
    for (int L = 0; L < NL; ++L) {
        const int rows = DIMS[L + 1], cols = DIMS[L], n = rows * cols;
        float** f32s[] = {&net.W[L], &net.mW[L], &net.vW[L]};
        for (float** p : f32s)
            if ((e = hipMalloc((void**)p, sizeof(float) * n)) != hipSuccess) return e;
        float** bs[] = {&net.b[L], &net.mb[L], &net.vb[L]};
        for (float** p : bs)
            if ((e = hipMalloc((void**)p, sizeof(float) * rows)) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&net.Wb[L], 2 * n)) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&net.WbT[L], 2 * n)) != hipSuccess) return e;
        // real fan-in / fan-out (padding excluded)
        const int fin = L == 0 ? NIN : cols, fout = L == NL - 1 ? NOUT : rows;
        const double lim = sqrt(6.0 / (fin + fout));
        float* h = new float[n];
        for (int r = 0; r < rows; ++r)
            for (int c = 0; c < cols; ++c) {
                const bool pad = (L == 0 && c >= NIN) || (L == NL - 1 && r >= NOUT);
                h[r * cols + c] = pad ? 0.f : (float)((2.0 * rnd() - 1.0) * lim);
            }
        (void)hipMemcpyAsync(net.W[L], h, sizeof(float) * n, hipMemcpyHostToDevice, s);
        (void)hipStreamSynchronize(s);
        delete[] h;
        (void)hipMemsetAsync(net.mW[L], 0, sizeof(float) * n, s);
        (void)hipMemsetAsync(net.vW[L], 0, sizeof(float) * n, s);
        (void)hipMemsetAsync(net.b[L], 0, sizeof(float) * rows, s);
        (void)hipMemsetAsync(net.mb[L], 0, sizeof(float) * rows, s);
        (void)hipMemsetAsync(net.vb[L], 0, sizeof(float) * rows, s);
    }
    refresh_bf16(net, s);
    return hipStreamSynchronize(s);
}

hipError_t mlp_alloc_empty(Mlp& net)
{
    hipError_t e;
    if ((e = hipMalloc((void**)&net.Wf, 2 * FRAG_TOTAL)) != hipSuccess) return e;
    for (int L = 0; L < NL; ++L) {
        const int rows = DIMS[L + 1], n = rows * DIMS[L];
        float** f32s[] = {&net.W[L], &net.mW[L], &net.vW[L]};
        for (float** p : f32s)
            if ((e = hipMalloc((void**)p, sizeof(float) * n)) != hipSuccess) return e;
        float** bs[] = {&net.b[L], &net.mb[L], &net.vb[L]};
        for (float** p : bs)
            if ((e = hipMalloc((void**)p, sizeof(float) * rows)) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&net.Wb[L], 2 * n)) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&net.WbT[L], 2 * n)) != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t mlp_copy(Mlp& dst, const Mlp& src, hipStream_t s)
{
    hipError_t e = hipMemcpyAsync(dst.Wf, src.Wf, 2 * FRAG_TOTAL, hipMemcpyDeviceToDevice, s);
    for (int L = 0; L < NL && e == hipSuccess; ++L) {
        const size_t rows = DIMS[L + 1], n = rows * DIMS[L];
        const std::pair<void*, const void*> f[] = {{dst.W[L], src.W[L]}, {dst.mW[L], src.mW[L]}, {dst.vW[L], src.vW[L]}};
        for (const auto& pr : f)
            if (e == hipSuccess) e = hipMemcpyAsync(pr.first, pr.second, sizeof(float) * n, hipMemcpyDeviceToDevice, s);
        const std::pair<void*, const void*> b[] = {{dst.b[L], src.b[L]}, {dst.mb[L], src.mb[L]}, {dst.vb[L], src.vb[L]}};
        for (const auto& pr : b)
            if (e == hipSuccess)
                e = hipMemcpyAsync(pr.first, pr.second, sizeof(float) * rows, hipMemcpyDeviceToDevice, s);
        if (e == hipSuccess) e = hipMemcpyAsync(dst.Wb[L], src.Wb[L], 2 * n, hipMemcpyDeviceToDevice, s);
        if (e == hipSuccess) e = hipMemcpyAsync(dst.WbT[L], src.WbT[L], 2 * n, hipMemcpyDeviceToDevice, s);
    }
    return e;
}

void mlp_free(Mlp& net)
{
    for (int L = 0; L < NL; ++L) {
        void* ps[] = {net.W[L], net.b[L], net.mW[L], net.vW[L], net.mb[L], net.vb[L], net.Wb[L], net.WbT[L]};
        for (void* p : ps)
            if (p) (void)hipFree(p);
    }
    if (net.Wf) (void)hipFree(net.Wf);
    net = Mlp{};
}

// (cap is set once everything is there: a caller asks it whether to allocate)
hipError_t work_alloc(Work& w, int cap)
{
    hipError_t e = hipMalloc((void**)&w.part, sizeof(float) * NPARAM * (size_t)grad_blocks(cap));
    if (e == hipSuccess) e = hipMalloc((void**)&w.grad, sizeof(float) * NPARAM);
    if (e == hipSuccess) e = hipMalloc((void**)&w.loss_rows, sizeof(float) * (size_t)cap);
    if (e == hipSuccess) e = hipMalloc((void**)&w.xf, sizeof(float) * 16 * (size_t)cap);
    if (e != hipSuccess) {
        work_free(w);
        return e;
    }
    for (int L = 0; L < NL; ++L) {
        w.gW[L] = w.grad + grad_w(L);
        w.gb[L] = w.grad + grad_b(L);
    }
    w.cap = cap;
    return hipSuccess;
}

void work_free(Work& w)
{
    void* ps[] = {w.part, w.grad, w.loss_rows, w.xf};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    w = Work{};
}

}  // namespace sur
}  // namespace lbm
