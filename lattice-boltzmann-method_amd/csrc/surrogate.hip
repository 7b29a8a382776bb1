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

// ------------------------------------------------------ gradient kernels
// Forward pass, loss and all gradients of a batch in three launches of small
// blocks with few registers and little LDS:
//   k_grad_rows     16 rows a block through the four layers and back, with the
//                   transposed products Z^T = W H^T of the in-step network;
//                   activations and dZ leave transposed, as the operands of
//   k_grad_weights  the weight and bias gradients of a part of the rows, and
//   k_grad_sum      their sum.
// Training also runs beside the steps, whose kernels fill the CUs: a block
// starts only where its registers, wavefronts and LDS fall free at once.  One
// kernel of 64 rows a block (eight wavefronts of 236 registers, 132 KB of LDS: a
// whole CU) took 21 us for 4096 rows by itself, but beside the steps it waited
// for the end of nearly every step kernel: 100 iterations beside 256x128x128
// FP32 steps took 150 ms or 21 steps.  A block of k_grad_rows takes the place of
// one block of a collide kernel (124 registers, a wavefront per SIMD, 12 KB): 25
// ms or 3 steps.  By themselves: k_grad_rows 13 us, bound by its chain of six
// exchanges between the wavefronts and, from 16384 rows (28 us), by reading the
// weights per 16 rows; k_grad_weights 10 us, bound by its loads; the sum 3.  A
// caller's gradient of 4096 rows takes 125 us, host copies included (130 as one
// kernel), of 16384 rows 198 (206), of 262144 rows 1900 (1500).
constexpr int GT_H = 0, GT_D = 24, GT_X = 48, GT_D3 = 49, GTILES = 50;  // tiles of a group of 16 rows
constexpr int GCHUNK = 32768;       // rows whose tiles are held at once (52 MB)
constexpr int GPART = 8;            // groups (128 rows) whose operands a wavefront holds at once
constexpr int GPARTS = 64;          // parts of a chunk at most: more groups go round
// strips of up to four tiles: 16 of each 128x128 layer, 8 of the first, 2 of the last
constexpr int GSTRIPS = 42;

// Offsets of W[L] and b[L] in the flat gradient.
constexpr int grad_w(int L) { return frag_offset(L) + bias_offset(L); }
constexpr int grad_b(int L) { return grad_w(L) + DIMS[L] * DIMS[L + 1]; }
static_assert(grad_b(NL - 1) + DIMS[NL] == NPARAM, "flat gradient");

// BF16 of a D fragment: the B operand of the next product.
__device__ __forceinline__ v4s bf_frag(const v4f z)
{
    v4s r;
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] = (short)f2bf(z[q]);
    return r;
}
// N tiles from D order (lane: row lane % 16, neurons 4 (lane / 16) + 0..3) to
// operand order with the row as the reduction index (lane: neuron lane % 16,
// rows 4 (lane / 16) + 0..3), through the wavefront's own LDS, to `to`.  A
// wavefront's LDS operations complete in order; the fences keep the compiler to
// it.
template <int N>
__device__ __forceinline__ void put_transposed(uint16_t* lds, const v4s x[N], uint16_t* to)
{
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < N; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) lds[t * 256 + (4 * g + q) * 16 + j] = (uint16_t)x[t][q];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int t = 0; t < N; ++t)
        *reinterpret_cast<uint2*>(to + t * 256 + lane * 4) =
            *reinterpret_cast<const uint2*>(lds + t * 256 + j * 16 + 4 * g);
}
// The A operands of the two output tiles t0, t0 + 1 of a 128-deep product,
// forward from the weights in fragment order, backward from W^T by row, and
// the product with the activations (or dZ) of a layer.
struct Weights2 {
    v8bf a[2][KSTEPS];
};
__device__ __forceinline__ Weights2 forward_weights(const uint16_t* Wl, int t0)
{
    const int lane = threadIdx.x & 63;
    Weights2 w;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) w.a[t][s] = load_frag8(Wl + (((t0 + t) * KSTEPS + s) * 64 + lane) * 8);
    return w;
}
__device__ __forceinline__ Weights2 backward_weights(const uint16_t* WT, int t0)
{
    const int lane = threadIdx.x & 63;
    Weights2 w;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint16_t* row = WT + (16 * (t0 + t) + (lane & 15)) * 128 + 4 * (lane >> 4);
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) w.a[t][s] = pair_frag(load_frag(row + 32 * s), load_frag(row + 32 * s + 16));
    }
    return w;
}
__device__ __forceinline__ v4f product128(const v8bf w[KSTEPS], const v4s h[8])
{
    v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s], pair_frag(h[2 * s], h[2 * s + 1]), acc, 0, 0, 0);
    return acc;
}

// Block b: rows row0 + 16 b + 0..15 (M a multiple of 16, so every row is one of
// the batch), wavefront w neurons 32 w + 0..31 of each 128-wide layer; the
// output layer is evaluated by every wavefront.  X holds BF16 features, or binary32
// ones that are rounded here.  loss_rows [M] receives the rows' squared errors.
// dZ of the output layer is that of the mean-squared loss over NOUT outputs,
// 2 (z - t) / (M NOUT), and 0 for padded outputs.  Each layer's weights are on
// their way while the layer before it is evaluated and shared.
template <typename XT>
__global__ __launch_bounds__(256) void k_grad_rows(Mlp net, const XT* X, const float* T, int M, int row0, uint16_t* tiles,
                                                   float* loss_rows)
{
    __shared__ __align__(16) uint16_t turn[4][2 * 256];
    __shared__ __align__(16) uint16_t frags[2][8 * 256];  // a layer's activations or dZ, from all wavefronts
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, j = lane & 15, g = lane >> 4;
    const int row = row0 + blockIdx.x * 16 + j;
    uint16_t* const out = tiles + (size_t)blockIdx.x * (GTILES * 256);
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    v4f z0[2], z1[2], z2[2];
    v4s mine[2], all[8];
    // the wavefront's two tiles to the others (buffer p) and, transposed, to memory
    auto share = [&](int p, int tile) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            uint2 u;
            __builtin_memcpy(&u, &mine[t], 8);
            *reinterpret_cast<uint2*>(frags[p] + (2 * w + t) * 256 + lane * 4) = u;
        }
        put_transposed<2>(turn[w], mine, out + (tile + 2 * w) * 256);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 8; ++t) all[t] = load_frag(frags[p] + t * 256 + lane * 4);
    };
    // ---- forward
    const int n0 = 32 * w;
    Weights2 wt = forward_weights(net.Wf + frag_offset(1), 2 * w);
    v4s x[1];
    if constexpr (sizeof(XT) == 2) x[0] = load_frag(X + (size_t)row * 16 + 4 * g);
    else x[0] = bf_frag(*reinterpret_cast<const v4f*>(X + (size_t)row * 16 + 4 * g));
    if (w == 0) put_transposed<1>(turn[0], x, out + GT_X * 256);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        z0[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(load_frag(net.Wb[0] + (n0 + 16 * t + j) * 16 + 4 * g), x[0],
                                                         zero, 0, 0, 0) +
                bias_frag(net.b[0], n0 + 16 * t, lane);
        mine[t] = act_frag(z0[t]);
    }
    share(0, GT_H);
    Weights2 nx = forward_weights(net.Wf + frag_offset(2), 2 * w);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        z1[t] = product128(wt.a[t], all) + bias_frag(net.b[1], n0 + 16 * t, lane);
        mine[t] = act_frag(z1[t]);
    }
    share(1, GT_H + 8);
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) wt.a[0][s] = load_frag8(net.Wf + frag_offset(3) + (s * 64 + lane) * 8);
    const v4f target = *reinterpret_cast<const v4f*>(T + (size_t)row * 16 + 4 * g);
    const v4s w3[2] = {load_frag(net.WbT[3] + (n0 + j) * 16 + 4 * g), load_frag(net.WbT[3] + (n0 + 16 + j) * 16 + 4 * g)};
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        z2[t] = product128(nx.a[t], all) + bias_frag(net.b[2], n0 + 16 * t, lane);
        mine[t] = act_frag(z2[t]);
    }
    share(0, GT_H + 16);
    nx = backward_weights(net.WbT[2], 2 * w);
    const v4f z3 = product128(wt.a[0], all) + bias_frag(net.b[3], 0, lane);
    // ---- loss and its gradient
    v4f dz = zero;
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (4 * g + q < NOUT) {
            const float d = z3[q] - target[q];
            sum += d * d;
            dz[q] = 2.f * d / (float)(M * NOUT);
        }
    const v4s d3[1] = {bf_frag(dz)};
    if (w == 0) {
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        if (g == 0) loss_rows[row] = sum;
        put_transposed<1>(turn[0], d3, out + GT_D3 * 256);
    }
    // ---- backward
    auto through_gelu = [&](v4f d, const v4f z) {
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] *= gelu_grad(z[q]);
        return bf_frag(d);
    };
#pragma unroll
    for (int t = 0; t < 2; ++t)
        mine[t] = through_gelu(__builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w3[t], d3[0], zero, 0, 0, 0), z2[t]);
    share(1, GT_D + 16);
    wt = backward_weights(net.WbT[1], 2 * w);
#pragma unroll
    for (int t = 0; t < 2; ++t) mine[t] = through_gelu(product128(nx.a[t], all), z1[t]);
    share(0, GT_D + 8);
#pragma unroll
    for (int t = 0; t < 2; ++t) mine[t] = through_gelu(product128(wt.a[t], all), z0[t]);
    put_transposed<2>(turn[w], mine, out + (GT_D + 2 * w) * 256);
}

// NB 16x16 tiles of a weight gradient over groups [first, last), two groups (32
// rows) to an instruction, operand tile ta against tb + 0..NB-1, and the sums
// over the rows of ta (its product with ones).
template <int NB>
__device__ __forceinline__ void weight_strip(const uint16_t* tiles, int ta, int tb, int first, int last, v4f acc[NB],
                                             v4f& sums)
{
    const int lane = threadIdx.x & 63;
    v8bf one;
#pragma unroll
    for (int e = 0; e < 8; ++e) one[e] = (__bf16)1.0f;
    // every load ahead of its use: groups past the last one read the part's
    // first and count as zero
    uint2 x[GPART][NB + 1];
#pragma unroll
    for (int r = 0; r < GPART; ++r) {
        const uint16_t* p = tiles + (size_t)(first + r < last ? first + r : first) * (GTILES * 256) + lane * 4;
        x[r][0] = *reinterpret_cast<const uint2*>(p + ta * 256);
#pragma unroll
        for (int t = 0; t < NB; ++t) x[r][1 + t] = *reinterpret_cast<const uint2*>(p + (tb + t) * 256);
    }
#pragma unroll
    for (int r = 0; r < GPART; ++r)
#pragma unroll
        for (int t = 0; t <= NB; ++t)
            if (first + r >= last) x[r][t] = make_uint2(0, 0);
    auto operand = [](const uint2 lo, const uint2 hi) {
        const uint2 u[2] = {lo, hi};
        v8bf o;
        __builtin_memcpy(&o, u, 16);
        return o;
    };
#pragma unroll
    for (int r = 0; r < GPART; r += 2) {
        const v8bf a = operand(x[r][0], x[r + 1][0]);
#pragma unroll
        for (int t = 0; t < NB; ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, operand(x[r][1 + t], x[r + 1][1 + t]), acc[t], 0, 0, 0);
        sums = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, one, sums, 0, 0, 0);
    }
}

// grid (GSTRIPS, parts): one wavefront forms a strip of one layer's weight gradient
// over its part of the groups and, with a neuron tile's first strip, its
// bias gradient.  part [blockIdx.y][NPARAM] is written, or added to when `more`.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 4))) void
k_grad_weights(const uint16_t* tiles, int groups, int more, float* part)
{
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    float* const out = part + (size_t)blockIdx.y * NPARAM;
    auto put = [&](int i, float v) { out[i] = more ? out[i] + v : v; };
    // tiles na (neurons) x nb.. (inputs) of layer L
    auto strip = [&](auto count, int L, int na, int nb, int ta, int tb) {
        constexpr int NB = decltype(count)::value;
        v4f acc[NB], sums = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < NB; ++t) acc[t] = sums;
        for (int first = blockIdx.y * GPART; first < groups; first += gridDim.y * GPART)
            weight_strip<NB>(tiles, ta, tb, first, min(first + GPART, groups), acc, sums);
#pragma unroll
        for (int t = 0; t < NB; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                put(grad_w(L) + (16 * na + 4 * g + q) * DIMS[L] + 16 * (nb + t) + j, acc[t][q]);
        if (j == 0 && nb == 0) {
#pragma unroll
            for (int q = 0; q < 4; ++q) put(grad_b(L) + 16 * na + 4 * g + q, sums[q]);
        }
    };
    using One = std::integral_constant<int, 1>;
    using Four = std::integral_constant<int, 4>;
    const int id = blockIdx.x;
    if (id < 32) {
        const int L = 1 + (id >> 4), na = (id & 15) >> 1, nb = 4 * (id & 1);
        strip(Four{}, L, na, nb, GT_D + 8 * L + na, GT_H + 8 * (L - 1) + nb);
    } else if (id < 40) {
        strip(One{}, 0, id - 32, 0, GT_D + id - 32, GT_X);
    } else {
        strip(Four{}, 3, 0, 4 * (id - 40), GT_D3, GT_H + 16 + 4 * (id - 40));
    }
}

// Sums the parts in a fixed order: 64 parameters per block of 256, a quarter of
// the parts per wavefront.
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
    int i = threadIdx.x;
    for (; i + 7 * 256 < B; i += 8 * 256) {  // eight loads on their way, added in order
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = lr[i + k * 256];
#pragma unroll
        for (int k = 0; k < 8; ++k) s += x[k];
    }
    for (; i < B; i += 256) s += lr[i];
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

// parts of the (first) chunk of M rows
static int grad_parts(int M)
{
    const int n = cdiv((M < GCHUNK ? M : GCHUNK) / 16, GPART);
    return n < GPARTS ? n : GPARTS;
}

template <typename XT>
void mlp_grad(const Mlp& net, const XT* X, const float* T, int M, Work& w, hipStream_t s)
{
    for (int row0 = 0; row0 < M; row0 += GCHUNK) {
        const int groups = (M - row0 < GCHUNK ? M - row0 : GCHUNK) / 16;
        hipLaunchKernelGGL(k_grad_rows<XT>, dim3(groups), dim3(256), 0, s, net, X, T, M, row0, w.tiles, w.loss_rows);
        hipLaunchKernelGGL(k_grad_weights, dim3(GSTRIPS, grad_parts(M - row0)), dim3(64), 0, s, w.tiles, groups,
                           row0 > 0 ? 1 : 0, w.part);
    }
    hipLaunchKernelGGL(k_grad_sum, dim3(cdiv(NPARAM, 64)), dim3(256), 0, s, w.part, grad_parts(M), w.grad);
}
template void mlp_grad<uint16_t>(const Mlp&, const uint16_t*, const float*, int, Work&, hipStream_t);
template void mlp_grad<float>(const Mlp&, const float*, const float*, int, Work&, hipStream_t);

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
    const size_t rows = (size_t)(cap < GCHUNK ? cap : GCHUNK);
    hipError_t e = hipMalloc((void**)&w.tiles, sizeof(uint16_t) * 16 * GTILES * rows);
    if (e == hipSuccess) e = hipMalloc((void**)&w.part, sizeof(float) * NPARAM * (size_t)grad_parts(cap));
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
    void* ps[] = {w.tiles, w.part, w.grad, w.loss_rows, w.xf};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    w = Work{};
}

}  // namespace sur
}  // namespace lbm
