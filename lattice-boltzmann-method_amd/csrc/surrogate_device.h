// Device building blocks of the chemistry surrogate MLP shared by the
// training kernels (surrogate.hip) and the fused in-step inference kernel
// (lbm_multi.hip).
//
// v_mfma_f32_16x16x16_bf16 operand layout (64 lanes, 4 BF16 per operand and
// lane, 4 FP32 accumulators per lane):
//   A[i][k]: i = lane % 16, k = 4 (lane / 16) + 0..3
//   B[k][j]: j = lane % 16, k = 4 (lane / 16) + 0..3
//   D[i][j]: j = lane % 16, i = 4 (lane / 16) + 0..3
// v_mfma_f32_16x16x32_bf16 (gfx950, twice the K per instruction at the same
// issue cost): 8 BF16 per operand and lane, k = 8 (lane / 16) + 0..7, the same
// D layout.
//
// In-step inference computes every layer transposed, Z^T = W H^T: the weights
// are the A operand (i = neuron) and the activations the B operand (j = batch
// row).  The D fragment of output tile t then holds neurons 16 t + 4 (lane / 16)
// + 0..3 of row lane % 16.  Layer 0 (K = 16) runs 16x16x16; the 128-wide
// layers run 16x16x32 with K-step s made of the D fragments of tiles 2s and
// 2s + 1 side by side: its element e of lane group g is neuron k32_neuron(s, g,
// e).  The weight fragments are stored in that K order, so activations stay
// in registers from layer to layer and no lane exchanges data.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "surrogate.h"

namespace lbm {
namespace sur {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// Neuron held by element e (0..7) of lane group g in 32-deep K-step s.
__host__ __device__ constexpr int k32_neuron(int s, int g, int e)
{
    return 32 * s + (e < 4 ? 4 * g + e : 16 + 4 * g + (e - 4));
}

// FP32 -> BF16, round to nearest even (v_cvt_pk_bf16_f32 on gfx950).
__device__ __forceinline__ uint16_t f2bf(float x)
{
    const __bf16 h = (__bf16)x;
    uint16_t u;
    __builtin_memcpy(&u, &h, 2);
    return u;
}

// GELU in its tanh form, x (1 + tanh(v)) / 2 with v = sqrt(2/pi) (x + 0.044715
// x^3), written as x / (1 + exp(-2 v)); and its derivative s + x s (1 - s) 2 v'
// with s = 1 / (1 + exp(-2 v)).
constexpr float GELU_C = 1.5957691216057308f;  // 2 sqrt(2 / pi)
constexpr float GELU_A = 0.044715f;
// (v_exp_f32 and v_rcp_f32: ~1 ulp, far below the BF16 rounding that follows;
// exp(-u) = 2^(x (K1 + K2 x^2)))
constexpr float GELU_K1 = -GELU_C * 1.4426950408889634f, GELU_K2 = -GELU_C * GELU_A * 1.4426950408889634f;
__device__ __forceinline__ float gelu(float x)
{
    const float e = __builtin_amdgcn_exp2f(x * __builtin_fmaf(GELU_K2, x * x, GELU_K1));
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float gelu_grad(float x)
{
    const float u = GELU_C * x * (1.0f + GELU_A * x * x);
    const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-u));
    return s + x * s * (1.0f - s) * (GELU_C * (1.0f + 3.0f * GELU_A * x * x));
}

// Fragment-ordered BF16 weights.  Layer 0 (K = 16): element (t 64 + lane) 4 + q
// holds W[16 t + lane % 16][4 (lane / 16) + q].  Layers with K = 32 KS:
// element ((t KS + s) 64 + lane) 8 + e holds W[16 t + lane % 16][k32_neuron(s,
// lane / 16, e)].  A wavefront reads one A fragment as 64 consecutive 8- or
// 16-byte words.
constexpr int frag_offset(int L)
{
    int off = 0;
    for (int i = 0; i < L; ++i) off += DIMS[i] * DIMS[i + 1];
    return off;
}
constexpr int FRAG_TOTAL = frag_offset(NL);      // 36864 BF16 = 72 KiB
constexpr int BIAS_TOTAL = 128 + 128 + 128 + 16;  // FP32
constexpr int bias_offset(int L)
{
    int off = 0;
    for (int i = 0; i < L; ++i) off += DIMS[i + 1];
    return off;
}

__device__ __forceinline__ v8bf load_frag8(const uint16_t* p)
{
    const uint4 w = *reinterpret_cast<const uint4*>(p);
    v8bf r;
    __builtin_memcpy(&r, &w, 16);
    return r;
}
// The B operand of a 32-deep K-step from the activations of two output tiles.
__device__ __forceinline__ v8bf pair_frag(const v4s lo, const v4s hi)
{
    short t[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    v8bf r;
    __builtin_memcpy(&r, t, 16);
    return r;
}

__device__ __forceinline__ v4s load_frag(const uint16_t* p)
{
    const uint2 w = *reinterpret_cast<const uint2*>(p);
    v4s r;
    r[0] = (short)(w.x & 0xffffu);
    r[1] = (short)(w.x >> 16);
    r[2] = (short)(w.y & 0xffffu);
    r[3] = (short)(w.y >> 16);
    return r;
}

// The bias of the 4 neurons of one D fragment (the accumulator's start).
__device__ __forceinline__ v4f bias_frag(const float* bias, int n0, int lane)
{
    const float* b = bias + n0 + 4 * (lane >> 4);
    return v4f{b[0], b[1], b[2], b[3]};
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// BF16(GELU(z)) for the 4 neurons of one D fragment, converted in pairs.
__device__ __forceinline__ v4s act_frag(const v4f z)
{
    const bf16x2 lo = __builtin_convertvector((f32x2){gelu(z[0]), gelu(z[1])}, bf16x2);
    const bf16x2 hi = __builtin_convertvector((f32x2){gelu(z[2]), gelu(z[3])}, bf16x2);
    uint32_t w[2];
    __builtin_memcpy(&w[0], &lo, 4);
    __builtin_memcpy(&w[1], &hi, 4);
    v4s h;
    __builtin_memcpy(&h, w, 8);
    return h;
}

// Evaluates the network for 32 rows (two batch tiles) held by one wavefront.
// `Wf` and `bias` are the fragment-ordered weights and the biases (LDS), x[bt]
// the BF16 inputs of batch tile bt (row lane % 16, features 4 (lane / 16) +
// 0..3), out[bt] its FP32 outputs in the same places.  Each accumulator
// starts from the layer's bias.
//
// Bound by the activations (5 vector operations, an exp2 and a reciprocal each:
// two thirds of the pass).  Output tile t + 1 is multiplied while tile t goes
// through its activation: the two are independent, so the matrix
// instructions and the LDS reads of their weights run under the activations
// instead of ahead of them.
constexpr int HTILES = 128 / 16, KSTEPS = 128 / 32;
struct Acc2 {
    v4f c[2];
};
template <int L>
__device__ __forceinline__ Acc2 hidden_tile(const uint16_t* Wf, const float* bias, const v4s act[2][HTILES], int t,
                                            int lane)
{
    const uint16_t* W = Wf + frag_offset(L);
    Acc2 a;
    a.c[0] = a.c[1] = bias_frag(bias + bias_offset(L), 16 * t, lane);
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
        const v8bf w = load_frag8(W + ((t * KSTEPS + s) * 64 + lane) * 8);
#pragma unroll
        for (int bt = 0; bt < 2; ++bt)
            a.c[bt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, pair_frag(act[bt][2 * s], act[bt][2 * s + 1]), a.c[bt],
                                                             0, 0, 0);
    }
    return a;
}
__device__ __forceinline__ Acc2 input_tile(const uint16_t* Wf, const float* bias, const v4s x[2], int t, int lane)
{
    const v4s w = load_frag(Wf + frag_offset(0) + (t * 64 + lane) * 4);
    const v4f b = bias_frag(bias + bias_offset(0), 16 * t, lane);
    Acc2 a;
#pragma unroll
    for (int bt = 0; bt < 2; ++bt) a.c[bt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w, x[bt], b, 0, 0, 0);
    return a;
}
// `next(t)` multiplies tile t of a layer; to[bt][t] receives its activations.
template <typename Next>
__device__ __forceinline__ void layer_tiles(Next next, v4s to[2][HTILES])
{
    Acc2 a = next(0);
#pragma unroll
    for (int t = 0; t < HTILES; ++t) {
        Acc2 b = a;
        if (t + 1 < HTILES) b = next(t + 1);
        to[0][t] = act_frag(a.c[0]);
        to[1][t] = act_frag(a.c[1]);
        a = b;
    }
}
__device__ __forceinline__ void mlp_rows32(const uint16_t* Wf, const float* bias, const v4s x[2], v4f out[2])
{
    const int lane = threadIdx.x & 63;
    v4s h0[2][HTILES], h1[2][HTILES];
    layer_tiles([&](int t) { return input_tile(Wf, bias, x, t, lane); }, h0);
    layer_tiles([&](int t) { return hidden_tile<1>(Wf, bias, h0, t, lane); }, h1);
    layer_tiles([&](int t) { return hidden_tile<2>(Wf, bias, h1, t, lane); }, h0);
    const Acc2 a = hidden_tile<3>(Wf, bias, h0, 0, lane);  // 128 -> 16, no activation
    out[0] = a.c[0];
    out[1] = a.c[1];
}
// The inputs of batch tile bt from BF16 rows [..][16] in LDS.
__device__ __forceinline__ v4s input_frag(const uint16_t* xin, int bt)
{
    const int lane = threadIdx.x & 63;
    return load_frag(xin + (bt * 16 + (lane & 15)) * 16 + (lane >> 4) * 4);
}
// The outputs of batch tile bt into FP32 rows [..][16] in LDS.
__device__ __forceinline__ void output_frag(float* yout, int bt, const v4f o)
{
    const int lane = threadIdx.x & 63;
    *reinterpret_cast<v4f*>(yout + (bt * 16 + (lane & 15)) * 16 + (lane >> 4) * 4) = o;
}

// Stages the fragment-ordered weights and biases of `net` into LDS.
__device__ __forceinline__ void stage_net(const Mlp& net, uint16_t* Wf, float* bias)
{
    const uint4* src = reinterpret_cast<const uint4*>(net.Wf);
    uint4* dst = reinterpret_cast<uint4*>(Wf);
    for (int i = threadIdx.x; i < FRAG_TOTAL / 8; i += blockDim.x) dst[i] = src[i];
    for (int i = threadIdx.x; i < BIAS_TOTAL; i += blockDim.x) {
        int L = 0;
        while (L < NL - 1 && i >= bias_offset(L + 1)) ++L;
        bias[i] = net.b[L][i - bias_offset(L)];
    }
}

}  // namespace sur
}  // namespace lbm
