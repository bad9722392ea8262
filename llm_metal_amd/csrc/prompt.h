// Many tokens of one sequence in one step, for the models whose decoding runs a token at a time (prompt.hip; the host side is
// in inference.hip).  Every product reads its weight once for all of them on the matrix cores, with 22 bits of every fp32
// activation kept (rows_to_f16_split), in sums of short parts (plan_short_sums); everything else is fp32.  No further from 64 bits
// than the tokens one by one (tests/test_gpu_prompt.py).
#pragma once
#include "gemm.h"

namespace lmhip {

// A product as the GEMM leaves it: S planes of [lo + M, N], rows m and lo + m the value and residual images of row m, inv their
// factors.  whole: planes of the product itself, [M, N], S or as many as the pair kernel's walk left.  P2 not null: S2 more planes of [M, N] of the value rows with what
// rounding the weights to fp16 lost, times 2^11.
struct SplitPlanes {
    const float *P, *inv;
    size_t plane;
    int S, N, lo;
    bool whole;
    PairWalk walk;                       // whole and walk.steps: so many of the S planes hold a column
    const float *P2;
    size_t plane2;
    int S2;
    __device__ __forceinline__ int planes(int n) const { return walk.steps ? walk.count(n) : S; }
};
constexpr float Q8_RESIDUAL_SCALE = 2048.f;
__device__ __forceinline__ float planes_at(const SplitPlanes &p, int m, int n)
{
    float v = 0.f;
    if (p.whole) {
        const float *P = p.P + (size_t)m * p.N + n;
        const int S = p.planes(n);
        for (int s0 = 0; s0 < S; s0 += 4) {                // (requested four at a time and added in their order)
            float h[4];
#pragma unroll
            for (int q = 0; q < 4; q++) h[q] = P[(size_t)min(s0 + q, S - 1) * p.plane];
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (s0 + q < S) v += h[q];
        }
    } else v = split_planes_value(p.P, p.S, p.plane, p.N, p.inv, p.lo, m, n);
    if (p.P2) {
        float r = 0.f;
        for (int s = 0; s < p.S2; s++) r += p.P2[s * p.plane2 + (size_t)m * p.N + n];
        v = fmaf(r, p.inv[m] * (1.0f / Q8_RESIDUAL_SCALE), v);
    }
    return v;
}

// Four neighbouring elements (n, N and the plane strides multiples of four, P and P2 16-byte aligned); the planes are requested
// four at a time and added in their order.
__device__ __forceinline__ float4v planes4_at(const SplitPlanes &p, int m, int n)
{
    const float *ph = p.P + (size_t)m * p.N + n, *pl = ph + (size_t)p.lo * p.N;
    float4v r;
    if (p.whole) {
        const int S = p.planes(n);
        r = *reinterpret_cast<const float4v *>(ph);
        if (S == 2) r += *reinterpret_cast<const float4v *>(ph + p.plane);
        else for (int s0 = 1; s0 < S; s0 += 4) {
            float4v h[4];
#pragma unroll
            for (int q = 0; q < 4; q++) h[q] = *reinterpret_cast<const float4v *>(ph + (size_t)min(s0 + q, S - 1) * p.plane);
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (s0 + q < S) r += h[q];
        }
    } else {
        float4v hi = *reinterpret_cast<const float4v *>(ph), lo = *reinterpret_cast<const float4v *>(pl);
        for (int s0 = 1; s0 < p.S; s0 += 4) {
            float4v h[4], l[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const size_t o = (size_t)min(s0 + q, p.S - 1) * p.plane;
                h[q] = *reinterpret_cast<const float4v *>(ph + o);
                l[q] = *reinterpret_cast<const float4v *>(pl + o);
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (s0 + q < p.S) { hi += h[q]; lo += l[q]; }
        }
        const float ih = p.inv[m], il = p.inv[p.lo + m];
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = fmaf(lo[e], il, hi[e] * ih);
    }
    if (p.P2) {
        const float ih = p.inv[m];
        float4v z = {};
        for (int s = 0; s < p.S2; s++) z += *reinterpret_cast<const float4v *>(p.P2 + s * p.plane2 + (size_t)m * p.N + n);
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = fmaf(z[e], ih * (1.0f / Q8_RESIDUAL_SCALE), r[e]);
    }
    return r;
}

// What follows the Q|K|V product for M tokens at positions pos .. pos + M - 1: adapter terms, per-head RMSNorm and RoPE; q to
// [M][Hq * hd], k and v into the rows of the caches [Hkv, max_seq, hd].
struct PromptHeads {
    SplitPlanes qkv;                     // columns q | k | v, and the adapters' A_q x | A_v x behind them when t is null and R > 0
    const float *g_q, *g_k;              // per-head norm gammas or null
    const float *t, *Bq, *Bv;            // t [M][2R]
    const float2 *rope;                  // (cos, sin) of position pos, hd / 2 pairs per position
    float *q, *kc, *vc;
    int M, Hq, Hkv, hd, R, pos, max_seq;
    float eps, sc;
};
void launch_prompt_heads(const PromptHeads &a);

// out [M][Hq * hd] = causal attention of the M queries at positions pos .. pos + M - 1 over the cache rows 0 .. pos + M - 1
bool prompt_attention_supported(int hd);
void launch_prompt_attention(const float *q, const float *kc, const float *vc, float *out, int M, int pos, int Hq, int Hkv, int hd, int max_seq);

// rows m and lo + m of the tiled operand a16 and their factors from act(gate) * up of the [gate | up] product
bool prompt_glu_supported(int IS);
// out [M, N] (row stride ldc) = the product
void launch_planes_to_rows(const SplitPlanes &p, float *out, int M, int N, int ldc);
void launch_prompt_glu(const SplitPlanes &gu, half_t *a16, float *inv, int M, int lo, int IS, int gelu);

// x[m] = emb[ids[m]] * scale
void launch_embed_ids(const float *emb, const int *ids, float scale, float *x, int M, int D);
// positions 0 .. len - 1 of sequence 0's caches to sequences 1 .. B - 1; k, v: [B][Hkv, max_seq, hd]
void launch_copy_caches(float *k, float *v, int B, int Hkv, int max_seq, int hd, int len);

// infer_kernels.hip: a Q8_0 matrix as two tiled F16 images, half(d q) and 2^11 times what that rounding lost; 22 bits of d q
void q8_to_tiled_pair(struct ::MetalBuf *W, int rows, int cols, half_t *hi, half_t *lo);
// raises *out on the device, the bits of a float, to the largest |d| over the scales of a Q8_0 matrix (a NaN is above all)
void q8_max_scale(struct ::MetalBuf *W, int rows, int cols, unsigned *out);

}  // namespace lmhip
