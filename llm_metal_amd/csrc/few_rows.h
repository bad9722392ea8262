// Products of a batch's step and of a short prompt: a few fp32 rows (up to 32) with F16 or Q8_0 weights, kept to 22 bits of every
// activation as everywhere in generation (few_rows.hip).
#pragma once
#include "gemm.h"

namespace lmhip {

constexpr int FEW_ROWS = 32;

// K-split planes of such a product: S planes of [B, N], their sum is the product
struct FewPlanes {
    const float *P;
    size_t plane;
    int S, N;
};
// out[b][n] (row stride ldo) = x[b] . W[n] for n < N; rows b and B + b of the tiled operand a16 are the value and residual images
// of x[b], inv their factors.  W: F16 tiles.
void launch_few_full(const half_t *a16, const float *inv, const half_t *W, float *out, int ldo, int B, int N, int K);
// act[b][i] = silu | gelu (gate) * up with the rows gate | up of W [2 IS, K] (IS a multiple of 32)
void launch_few_glu(const half_t *a16, const float *inv, const half_t *W, float *act, int B, int IS, int K, int gelu);
// the same over Q8_0 rows: codes [rows][K] and a scale per 32 of them (few_q8_of, infer_kernels.hip: kept with the matrix); K a multiple of 32
struct FewQ8 {
    const int8_t *q;
    const half_t *d;
};
FewQ8 few_q8_of(struct ::MetalBuf *W, int rows, int cols);
// (`chunks` planes of [B, ldo] whose sum is the product; few_chunks: as many as pay where the consumer adds planes)
int few_chunks(int N, int K);
FewPlanes launch_few_full_q8(const half_t *a16, const float *inv, const FewQ8 &W, float *out, int ldo, int B, int N, int K, int chunks = 1);
void launch_few_glu_q8(const half_t *a16, const float *inv, const FewQ8 &W, float *act, int B, int IS, int K, int gelu);
// x [B, D] += br's sum, or RMSNorm(it; g_branch) (br.S 0: nothing); the operand a16 and factors inv of RMSNorm(x; g), and that in fp32 where
// ln is not null.  D a multiple of four up to 8192, pointers 16-byte aligned.
void launch_few_norm(float *x, const FewPlanes &br, const float *g_branch, const float *g, float *ln, half_t *a16, float *inv, int B, int D, float eps);
// planes of x [B, K] fp32 (K a multiple of four, x 16-byte aligned) times W [N, K]^T, N a multiple of four; P: few_planes(N, K)
// planes of B * N floats
int few_planes(int N, int K);
FewPlanes launch_few_split(const float *x, const half_t *W, float *P, int B, int N, int K);

}  // namespace lmhip
