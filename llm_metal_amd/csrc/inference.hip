// Token-by-token generation on top of the inference enqueues: the host pipeline of the reference's
// src/nn/fast_inference.c (state, forward_token, generate, sharing with the SFT state) for the HIP backend.
// Every step is enqueued on the library's one stream; the host waits once per token, for the logits or for
// the argmax computed on the GPU.
//
// One decode step computes what src/nn/fast_inference.c:376-467 computes: where the host waits for the step, in one launch (token.hip),
// otherwise, and for shapes, adapters and contexts that it does not take, in 5 launches per layer instead of 17: Q|K|V and
// gate|up are one matrix each (row concatenation, built when the state is created), the products that follow a norm form it
// themselves (matvec_norm, matvec_norms_around), and the attention launch does LoRA up-projection, per-head RMSNorm, RoPE and
// the KV-cache store for the new token.  Prompts of five tokens and more run many tokens per step (PromptRun).
#include "backend.h"
#include "devutil.h"
#include "fused.h"
#include "prompt.h"
#include "few_rows.h"
#include "token.h"
#include "stack.h"
#include "../../include/inference_hip.h"
#include "../../include/loader_hip.h"

#include <fstream>
#include <functional>
#include <math.h>
#include <sstream>
#include <string.h>
#include <string>
#include <sys/stat.h>
#include <unistd.h>
#include <vector>

using namespace lmhip;

extern "C" MetalBuf *sft_get_token_emb_buf(SFTState *s);

namespace {
struct BatchRun;
struct PromptRun;
struct TokenRun;
void batch_release(BatchRun *r);
void prompt_release(PromptRun *r);
void token_release(TokenRun *r);
// a state on a training state's tiles, or of a layer-by-layer model: one token through the lock-step path with a run of
// one sequence
void step_on_run(InferenceState *s, int token, int pos);
const float *step_logits_on_run(InferenceState *s, int token, int pos);
const float *logits_on_run(InferenceState *s);
int argmax_on_run(InferenceState *s);
void prefill_on_run(InferenceState *s, const uint32_t *tokens, int n, int pos);
int forward_rows(InferenceState *s, const int *tokens, int n, const int *want, int n_want, float *logits);
// the other models: n tokens of one sequence in steps of many rows, where the shape and memory allow that
bool prompt_takes(InferenceState *s, int n);
int prompt_forward(InferenceState *s, const int *tokens, int n, const int *want, int n_want, float *logits);
void prompt_fill(InferenceState *s, const uint32_t *tokens, int n);
}

struct InferenceState {
    int D, Hq, Hkv, hd, IS, V, NL, max_seq, cur_len, use_fp16;
    ModelType model_type;
    float emb_scale, eps;
    int eos[4], n_eos;
    std::vector<float> thetas;
    MetalBuf *rope_tabs;                 // (cos, sin) [distinct thetas][max_seq][hd/2], as rope forms them
    std::vector<int> theta_slot;         // table of each layer
    MetalBuf *x, *x2, *branch, *ln, *qkv, *att, *gu, *gate_v, *up_v, *logits, *best;   // gate_v / up_v: the halves of gu
    float *logits_host;
    int *best_host;
    std::vector<MetalBuf *> kc, vc;
    // per layer: fused [Wq; Wk; Wv] and [Wgate; Wup] (owned), Wo and Wdown and the norm gammas (owned, or the SFT state's)
    struct Layer { WMat qkv, gu; WMat *o, *down; MetalBuf *g_in, *g_post_attn, *g_pre_ff, *g_post_ff, *g_q, *g_k; };
    // A state made from a training state owns no weights at all: `borrowed` holds the training state's tiled images
    // (F16 or Q8_0 tiles, the operands of its own forward), read in place, so whatever training writes there is what the
    // next token sees.  Such a state has no row-major matrices for the matrix-vector kernels; every step, also of a
    // single sequence, goes through the matrix-core products of the lock-step batch path (`single`: its run of one).
    int borrows_tiles;
    std::vector<BorrowedLayer> borrowed;
    WeightOp borrowed_lm;
    BatchRun *single;
    // A model that is described layer by layer (stack.h): its configuration and weights; every step goes through a run
    // here as well.  NULL for the other models.
    LayerStack *stack;
    std::vector<Layer> layers;
    WMat *lm_head;
    MetalBuf *g_final, *emb;
    int owns_weights;
    SFTState *sft;                       // source of borrowed weights, or NULL
    struct Lora { MetalBuf *Aq, *Bq, *Av, *Bv; };
    std::vector<Lora> lora;
    int R;
    float scaling;
    MetalBuf *lora_t;                    // [2R]: A_q ln | A_v ln
    PromptRun *prompt;                   // scratch of prompts taken many tokens at a time (NULL until used)
    bool prompt_refused;                 // no room for it
    uint64_t q8_fit_version;             // versions of the weights that q8_fit was found for (0: none)
    bool q8_fit;
    TokenRun *one_launch;                // what a step in one launch needs (NULL until used)
    bool steps_in_launches;              // it cannot be had
    uint64_t step_ticks;                 // of the 100 MHz clock that a wait in it may last
    size_t step_bytes;                   // of device memory that it may take
    BatchRun *batch;                     // scratch and caches of the lock-step batch path, kept from call to call (NULL until used)
};

namespace {

constexpr int TB = 256;
constexpr uint64_t STEP_TICKS = 2000000;                     // 20 ms: a step takes up to six, longer only on a device that is not ours alone
// Steps in launches after a wait that ran out, twice as many after each further one up to PAUSE_MOST, half as many once as many have gone well: two
// processes that decode on one device may hold a part of its CUs each whenever their steps meet, and lose a hundredth of their time so
constexpr int PAUSE = 64, PAUSE_MOST = 4096;

// x = emb[token] * scale: the embedding row, scaled by sqrt(D) for Gemma3 (src/nn/fast_inference.c:385-391)
__global__ __launch_bounds__(TB) void k_embed_row(const float *__restrict__ emb, int token, float scale, float *__restrict__ x, int D)
{
    const int i = blockIdx.x * TB + threadIdx.x;
    if (i < D) x[i] = emb[(size_t)token * D + i] * scale;
}

// index of the first maximum of v[0..n) (src/nn/fast_inference.c:469-476) in two launches: AM_WGS workgroups leave
// (value, index) of their slice, one workgroup picks among them
constexpr int AM_WGS = 128;

__device__ __forceinline__ void am_pick(float &best, int &idx, float ob, int oi)
{
    if (ob > best || (ob == best && oi < idx)) { best = ob; idx = oi; }
}

__device__ __forceinline__ void am_block(float &best, int &idx, float *bv, int *bi)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) am_pick(best, idx, __shfl_xor(best, o, 64), __shfl_xor(idx, o, 64));
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) { bv[w] = best; bi[w] = idx; }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int i = 1; i < (int)(blockDim.x >> 6); i++) am_pick(best, idx, bv[i], bi[i]);
}

__global__ __launch_bounds__(TB) void k_argmax_part(const float *__restrict__ v, int n, float *__restrict__ pv, int *__restrict__ pi)
{
    __shared__ float bv[4];
    __shared__ int bi[4];
    float best = -INFINITY;
    int idx = 0x7fffffff;
    for (int i = blockIdx.x * TB + threadIdx.x; i < n; i += AM_WGS * TB) am_pick(best, idx, v[i], i);
    am_block(best, idx, bv, bi);
    if (threadIdx.x == 0) { pv[blockIdx.x] = best; pi[blockIdx.x] = idx; }
}

// out: pinned host memory (with a copy of the four bytes behind the kernel a token took 2 us more: 172.4 -> 170.6 on the 2048 wide Paposun)
__global__ __launch_bounds__(AM_WGS) void k_argmax_final(const float *__restrict__ pv, const int *__restrict__ pi, int *__restrict__ out)
{
    __shared__ float bv[AM_WGS / 64];
    __shared__ int bi[AM_WGS / 64];
    float best = pv[threadIdx.x];
    int idx = pi[threadIdx.x];
    am_block(best, idx, bv, bi);
    if (threadIdx.x == 0) *out = idx == 0x7fffffff ? 0 : idx;
}

// x += b (b = branch, or RMSNorm(branch; g_branch) where Gemma3 norms the branch output first); ln = RMSNorm(x; g).
// branch == NULL: only the norm.  One workgroup of 1024 threads: the vector is a few thousand floats.
__global__ __launch_bounds__(1024) void k_add_norm(float *__restrict__ x, const float *__restrict__ branch,
                                                   const float *__restrict__ g_branch, const float *__restrict__ g,
                                                   float *__restrict__ ln, int D, float eps)
{
    __shared__ float sm[16];
    x += (size_t)blockIdx.x * D; ln += (size_t)blockIdx.x * D;           // one workgroup per vector of a batch
    if (branch) branch += (size_t)blockIdx.x * D;
    float inv_b = 1.f;
    if (branch && g_branch) {
        float ss = 0.f;
        for (int i = threadIdx.x; i < D; i += 1024) { const float v = branch[i]; ss += v * v; }
        inv_b = rsqrtf(block_sum(ss, sm) / (float)D + eps);
    }
    float ss = 0.f;
    for (int i = threadIdx.x; i < D; i += 1024) {
        float v = x[i];
        if (branch) { v += g_branch ? branch[i] * inv_b * g_branch[i] : branch[i]; x[i] = v; }
        ss += v * v;
    }
    const float inv = rsqrtf(block_sum(ss, sm) / (float)D + eps);
    for (int i = threadIdx.x; i < D; i += 1024) ln[i] = x[i] * inv * g[i];       // own elements only: no barrier needed
}

// t[r] = A_q[r] . ln for r < R, t[R + r] = A_v[r] . ln: one wave per adapter row
__global__ __launch_bounds__(64) void k_lora_down(const float *__restrict__ ln, const float *__restrict__ Aq,
                                                  const float *__restrict__ Av, float *__restrict__ t, int R, int D)
{
    const int r = blockIdx.x;
    ln += (size_t)blockIdx.y * D; t += (size_t)blockIdx.y * 2 * R;       // one vector of a batch per blockIdx.y
    const float *a = r < R ? Aq + (size_t)r * D : Av + (size_t)(r - R) * D;
    float s = 0.f;
    if ((D & 3) == 0) {                                                   // 16-byte loads, eight pairs of them in flight per lane
        const float4 *a4 = reinterpret_cast<const float4 *>(a), *l4 = reinterpret_cast<const float4 *>(ln);
        const int n4 = D >> 2;
        for (int i0 = threadIdx.x; i0 < n4; i0 += 64 * 8) {
            float4 av[8], lv[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int i = i0 + 64 * u;
                av[u] = lv[u] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (i < n4) { av[u] = a4[i]; lv[u] = l4[i]; }
            }
#pragma unroll
            for (int u = 0; u < 8; u++) s += av[u].x * lv[u].x + av[u].y * lv[u].y + av[u].z * lv[u].z + av[u].w * lv[u].w;
        }
    } else {
        for (int i = threadIdx.x; i < D; i += 64) s = fmaf(a[i], ln[i], s);
    }
    s = wave_sum(s);
    if (threadIdx.x == 0) t[r] = s;
}

// act[b][i] = silu | gelu (gate) * up from the planes of the [gate | up] product of a batch
__global__ __launch_bounds__(TB) void k_glu_planes(SplitPlanes gu, float *__restrict__ act, int IS, int gelu)
{
    const int b = blockIdx.y, i = blockIdx.x * TB + threadIdx.x;
    if (i >= IS) return;
    const float g = planes_at(gu, b, i), u = planes_at(gu, b, IS + i);
    float a;
    if (gelu) {                                                           // shaders/q8_kernels.metal:349-362
        float t = 0.7978845608f * (g + 0.044715f * g * g * g);
        t = fminf(fmaxf(t, -15.f), 15.f);
        a = 0.5f * g * (1.0f + tanhf(t));
    } else a = g / (1.0f + expf(-g));                                     // :337-347
    act[(size_t)b * IS + i] = a * u;
}

// k_add_norm for row blockIdx.x of a batch, with the branch taken from a product's planes (br.P) or absent, and with
// ln also written as the next product's operand: rows b and lo + b of the tiled fp16 image a16 [lo + B, D] and their factors
// (what rows_to_f16_split makes of ln, element for element).  A thread holds elements tid + 1024 u, u < EPT, so
// 1024 EPT >= the padded row; the sums run in k_add_norm's order.
template <int EPT>
__global__ __launch_bounds__(1024) void k_add_norm_split(float *__restrict__ x, SplitPlanes br, const float *__restrict__ g_branch,
                                                         const float *__restrict__ g, float *__restrict__ ln,
                                                         half_t *__restrict__ a16, float *__restrict__ inv_out, int lo, int D, float eps)
{
    __shared__ float sm[32];
    const int b = blockIdx.x, Kb = tiled_kb(D);
    x += (size_t)b * D;
    float bv[EPT], v[EPT], xv[EPT], gv[EPT], gbv[EPT];
    float inv_b = 1.f;
    // the row, the norm weights and the branch norm's weights are requested with the planes, not after the reductions
    // (a round trip each)
#pragma unroll
    for (int u = 0; u < EPT; u++) {
        const int i = threadIdx.x + 1024 * u;
        xv[u] = gv[u] = gbv[u] = 0.f;
        if (i < D) { xv[u] = x[i]; gv[u] = g[i]; if (br.P && g_branch) gbv[u] = g_branch[i]; }
    }
    if (br.P) {
#pragma unroll
        for (int u = 0; u < EPT; u++) { const int i = threadIdx.x + 1024 * u; bv[u] = i < D ? planes_at(br, b, i) : 0.f; }
        if (g_branch) {
            float ss = 0.f;
#pragma unroll
            for (int u = 0; u < EPT; u++) ss += bv[u] * bv[u];
            inv_b = rsqrtf(block_sum(ss, sm) / (float)D + eps);
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < EPT; u++) {
        const int i = threadIdx.x + 1024 * u;
        v[u] = 0.f;
        if (i < D) {
            v[u] = xv[u];
            if (br.P) { v[u] += g_branch ? bv[u] * inv_b * gbv[u] : bv[u]; x[i] = v[u]; }
        }
        ss += v[u] * v[u];
    }
    // the row maximum of v g, which the factor 1 / rms scales like every entry, goes through the same pair of barriers
    // as the sum of squares
    float mxg = 0.f;
#pragma unroll
    for (int u = 0; u < EPT; u++) mxg = fmaxf(mxg, fabsf(v[u] * gv[u]));
    block_sum_max(ss, mxg, sm);
    const float inv = rsqrtf(ss / (float)D + eps);
#pragma unroll
    for (int u = 0; u < EPT; u++) {
        const int i = threadIdx.x + 1024 * u;
        v[u] = i < D ? v[u] * inv * gv[u] : 0.f;
        if (ln && i < D) ln[(size_t)b * D + i] = v[u];
    }
    const float s = row_scale_for(mxg * inv), is = 1.0f / s;
#pragma unroll
    for (int u = 0; u < EPT; u++) {
        const int i = threadIdx.x + 1024 * u;
        const half_t h = f2h(v[u] * s);
        if (i < Kb * 64) {
            a16[tiled_a_index(b, i, Kb)] = h;
            a16[tiled_a_index(lo + b, i, Kb)] = f2h((v[u] * s - h2f(h)) * PAIR_RESIDUAL_SCALE);
        }
    }
    if (threadIdx.x == 0) { inv_out[b] = is; inv_out[lo + b] = is / PAIR_RESIDUAL_SCALE; }
}

// The same with four neighbouring columns per piece, C pieces per thread (D and the product's strides multiples of four): the
// planes of a row -- 390 KB at eight sequences of the 4B shape, which one CU has to pull -- come in 16-byte loads, nine in
// flight where k_add_norm_split waits for every pair of planes: 6.1 us there against 10.2, 500 rows of a prompt 11.8 against 13.0.
template <int NT, int C>
__global__ __launch_bounds__(NT) void k_add_norm_split4(float *__restrict__ x, SplitPlanes br, const float *__restrict__ g_branch,
                                                        const float *__restrict__ g, float *__restrict__ ln,
                                                        half_t *__restrict__ a16, float *__restrict__ inv_out, int lo, int D, float eps)
{
    __shared__ float sm[32];
    const int b = blockIdx.x, Kb = tiled_kb(D);
    x += (size_t)b * D;
    float4v v[C], bv[C], gv[C], gb[C];
    float inv_b = 1.f, ss = 0.f;
#pragma unroll
    for (int u = 0; u < C; u++) {
        const int i = 4 * (threadIdx.x + NT * u);
        v[u] = gv[u] = gb[u] = bv[u] = float4v{};
        if (i >= D) continue;
        v[u] = *reinterpret_cast<const float4v *>(x + i);
        gv[u] = *reinterpret_cast<const float4v *>(g + i);
        if (br.P && g_branch) gb[u] = *reinterpret_cast<const float4v *>(g_branch + i);
    }
    if (br.P) {
#pragma unroll
        for (int u = 0; u < C; u++) {
            const int i = 4 * (threadIdx.x + NT * u);
            if (i < D) bv[u] = planes4_at(br, b, i);
        }
        if (g_branch) {
#pragma unroll
            for (int u = 0; u < C; u++)
#pragma unroll
                for (int e = 0; e < 4; e++) ss += bv[u][e] * bv[u][e];
            inv_b = rsqrtf(block_sum(ss, sm) / (float)D + eps);
        }
    }
    ss = 0.f;
    float mxg = 0.f;
#pragma unroll
    for (int u = 0; u < C; u++) {
        const int i = 4 * (threadIdx.x + NT * u);
        if (br.P) {
            v[u] += g_branch ? bv[u] * inv_b * gb[u] : bv[u];
            if (i < D) *reinterpret_cast<float4v *>(x + i) = v[u];
        }
#pragma unroll
        for (int e = 0; e < 4; e++) { ss += v[u][e] * v[u][e]; mxg = fmaxf(mxg, fabsf(v[u][e] * gv[u][e])); }
    }
    block_sum_max(ss, mxg, sm);
    const float inv = rsqrtf(ss / (float)D + eps), s = row_scale_for(mxg * inv), is = 1.0f / s;
#pragma unroll
    for (int u = 0; u < C; u++) {
        const int i = 4 * (threadIdx.x + NT * u);
        v[u] = v[u] * inv * gv[u];
        if (ln && i < D) *reinterpret_cast<float4v *>(ln + (size_t)b * D + i) = v[u];
        half4 h, l;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            h[e] = f2h(v[u][e] * s);
            l[e] = f2h((v[u][e] * s - h2f(h[e])) * PAIR_RESIDUAL_SCALE);
        }
        if (i < Kb * 64) {
            *reinterpret_cast<half4 *>(a16 + tiled_a_index(b, i, Kb)) = h;
            *reinterpret_cast<half4 *>(a16 + tiled_a_index(lo + b, i, Kb)) = l;
        }
    }
    if (threadIdx.x == 0) { inv_out[b] = is; inv_out[lo + b] = is / PAIR_RESIDUAL_SCALE; }
}

// rows x[0 .. M) of a step: one workgroup each, of 1024 threads while there are fewer rows than CUs and latency is what counts,
// of 256 beyond
void launch_add_norm_split(float *x, const SplitPlanes &br, const float *g_branch, const float *g, float *ln, half_t *a16, float *inv, int M, int lo, int D, float eps)
{
    const int pad = tiled_kb(D) * 64;
    const bool four = D % 4 == 0 && br.N % 4 == 0 && (br.plane | br.plane2) % 4 == 0 &&
                      !(((uintptr_t)x | (uintptr_t)br.P | (uintptr_t)br.P2 | (uintptr_t)g_branch | (uintptr_t)g | (uintptr_t)ln) & 15);
#define NORM_SPLIT(KERNEL, NT_) hipLaunchKernelGGL((KERNEL), dim3(M), dim3(NT_), 0, stream(), x, br, g_branch, g, ln, a16, inv, lo, D, eps)
    if (four && M < 192) { if (pad <= 4096) NORM_SPLIT((k_add_norm_split4<1024, 1>), 1024); else NORM_SPLIT((k_add_norm_split4<1024, 2>), 1024); }
    else if (four) {
        if (pad <= 2048) NORM_SPLIT((k_add_norm_split4<256, 2>), 256);
        else if (pad <= 3072) NORM_SPLIT((k_add_norm_split4<256, 3>), 256);
        else if (pad <= 4096) NORM_SPLIT((k_add_norm_split4<256, 4>), 256);
        else NORM_SPLIT((k_add_norm_split4<1024, 2>), 1024);
    }
    else if (pad <= 4096) NORM_SPLIT(k_add_norm_split<4>, 1024);
    else NORM_SPLIT(k_add_norm_split<8>, 1024);
#undef NORM_SPLIT
}

MetalBuf *fbuf(size_t n) { return metal_buf_create(n * sizeof(float)); }

void matvec(InferenceState *s, const WMat *w, MetalBuf *x, MetalBuf *y)
{
    if (s->use_fp16) metal_enqueue_f16_matvec(w->mbuf, x, y, w->rows, w->cols);
    else metal_enqueue_q8_matvec(w->mbuf, x, y, w->rows, w->nb);
}

void add_norm(InferenceState *s, MetalBuf *x, MetalBuf *branch, MetalBuf *g_branch, MetalBuf *g)
{
    hipLaunchKernelGGL(k_add_norm, dim3(1), dim3(1024), 0, stream(), dptr_as<float>(x), branch ? dptr_as<float>(branch) : nullptr,
                       g_branch ? dptr_as<float>(g_branch) : nullptr, dptr_as<float>(g), dptr_as<float>(s->ln), s->D, s->eps);
}

// src/nn/fast_inference.c:376-467
// host: pinned memory for the logits besides, or null; true: they go there as they are formed
bool forward_token(InferenceState *s, int token, int pos, float *host = nullptr)
{
    const int D = s->D, Hq = s->Hq, Hkv = s->Hkv, hd = s->hd;
    const bool gemma = s->model_type == MODEL_GEMMA3;
    hipLaunchKernelGGL(k_embed_row, dim3((D + TB - 1) / TB), dim3(TB), 0, stream(), dptr_as<float>(s->emb), token, s->emb_scale,
                       dptr_as<float>(s->x), D);
    MetalBuf *pending = nullptr, *pending_g = nullptr;           // FFN branch of the previous layer, added by the next norm kernel
    // Where the branch enters the sum as it is (Qwen3), the product after a norm forms sum and norm itself
    // (matvec_norm) and the sum goes to the other of two residual buffers; the Q|K|V product only without adapters,
    // whose down-projection reads the normed vector too.
    MetalBuf *x = s->x, *x_other = s->x2;
    // (Gemma3's branch is normed on its way into the sum: matvec_norms_around does that too; a model may come without the norm of
    // its feed-forward branch)
    const bool fuse_ffn = D <= 12288, fuse_qkv = fuse_ffn && s->lora.empty();
    const int q8 = s->use_fp16 ? 0 : 1;
    auto normed_product = [&](MetalBuf *W, MetalBuf *branch, MetalBuf *g_branch, MetalBuf *g, MetalBuf *y, int rows, int glu, float *y_host = nullptr) {
        NormIn n{dptr_as<float>(x), branch ? dptr_as<float>(branch) : nullptr, dptr_as<float>(g), branch ? dptr_as<float>(x_other) : nullptr,
                 s->eps, D, g_branch ? dptr_as<float>(g_branch) : nullptr, nullptr, y_host};
        if (gemma && (g_branch || !branch)) { matvec_norms_around(W, n, dptr_as<float>(y), rows, D, q8, glu); mark_written(y); }
        else matvec_norm(W, n, y, rows, D, q8, glu);
        if (branch) std::swap(x, x_other);
    };
    for (int L = 0; L < s->NL; L++) {
        const InferenceState::Layer &lw = s->layers[L];
        if (fuse_qkv) normed_product(lw.qkv.mbuf, pending, pending_g, lw.g_in, s->qkv, lw.qkv.rows, 0);
        else {
            add_norm(s, x, pending, pending_g, lw.g_in);
            matvec(s, &lw.qkv, s->ln, s->qkv);
        }
        // LoRA on q and v, per-head RMSNorm and RoPE on q and k, k and v into the caches, and the attention over the
        // cache: one launch (infer_kernels.hip: k_attn_decode<.., FUSED>)
        HeadPost a{};
        a.qkv = dptr_as<float>(s->qkv);
        a.g_q = lw.g_q ? dptr_as<float>(lw.g_q) : nullptr; a.g_k = lw.g_k ? dptr_as<float>(lw.g_k) : nullptr;
        a.kc = dptr_as<float>(s->kc[L]); a.vc = dptr_as<float>(s->vc[L]);
        a.Hq = Hq; a.Hkv = Hkv; a.pos = pos;
        a.rope = dptr_as<float2>(s->rope_tabs) + ((size_t)s->theta_slot[L] * s->max_seq + pos) * (hd / 2); a.eps = s->eps;
        if (!s->lora.empty()) {
            const InferenceState::Lora &lr = s->lora[L];
            hipLaunchKernelGGL(k_lora_down, dim3(2 * s->R), dim3(64), 0, stream(), dptr_as<float>(s->ln), dptr_as<float>(lr.Aq),
                               dptr_as<float>(lr.Av), dptr_as<float>(s->lora_t), s->R, D);
            a.t = dptr_as<float>(s->lora_t); a.Bq = dptr_as<float>(lr.Bq); a.Bv = dptr_as<float>(lr.Bv);
            a.R = s->R; a.sc = s->scaling;
        }
        // the O weights (F16 rows; up to 24 MB) travel while the attention's few workgroups run: 128 more workgroups ask
        // for them, 2.324 -> 2.290 ms per token (64: 2.305, 192: 2.305; 48 MB, i.e. part of the gate|up rows as well: no change)
        if (!q8) { a.pf_base = (const char *)dptr(lw.o->mbuf); a.pf_bytes = std::min<size_t>(lw.o->mbuf->size, (size_t)24 << 20) & ~(size_t)15; a.pf_wgs = 128; }
        attention_decode_fused(a, s->kc[L], s->vc[L], dptr_as<float>(s->att), hd, s->max_seq);
        mark_written(s->att);
        matvec(s, lw.o, s->att, s->branch);
        // x += o (Gemma3: RMSNorm(o; g_post_attn)); ln = RMSNorm(x; g_pre_ff | g_post_attn);
        // act = silu | gelu (gate) * up, formed in the epilogue of the [gate; up] product
        if (fuse_ffn) normed_product(lw.gu.mbuf, s->branch, gemma ? lw.g_post_attn : nullptr, gemma ? lw.g_pre_ff : lw.g_post_attn, s->gate_v, s->IS, gemma ? 2 : 1);
        else {
            add_norm(s, x, s->branch, gemma ? lw.g_post_attn : nullptr, gemma ? lw.g_pre_ff : lw.g_post_attn);
            matvec_glu(lw.gu.mbuf, s->ln, s->gate_v, s->IS, D, q8, gemma ? 1 : 0);
        }
        matvec(s, lw.down, s->gate_v, s->branch);
        pending = s->branch;
        pending_g = gemma ? lw.g_post_ff : nullptr;
    }
    // (matvec_norm, which a branch without a norm of its own takes, wants whole blocks of 32 columns)
    const bool normed = D <= NORMED_COLS && (D % 32 == 0 || pending_g);
    if (normed) normed_product(s->lm_head->mbuf, pending, pending_g, s->g_final, s->logits, s->V, 0, host);
    else {
        add_norm(s, x, pending, pending_g, s->g_final);
        matvec(s, s->lm_head, s->ln, s->logits);
    }
    HIP_CHECK(hipGetLastError());
    return normed && host;
}

const float *logits_to_host(InferenceState *s)
{
    HIP_CHECK(hipMemcpyAsync(s->logits_host, dptr(s->logits), (size_t)s->V * 4, hipMemcpyDeviceToHost, stream()));
    HIP_CHECK(hipStreamSynchronize(stream()));
    return s->logits_host;
}

int argmax_to_host(InferenceState *s)
{
    float *pv = dptr_as<float>(s->best);
    int *pi = dptr_as<int>(s->best) + AM_WGS;
    hipLaunchKernelGGL(k_argmax_part, dim3(AM_WGS), dim3(TB), 0, stream(), dptr_as<float>(s->logits), s->V, pv, pi);
    hipLaunchKernelGGL(k_argmax_final, dim3(1), dim3(AM_WGS), 0, stream(), pv, pi, s->best_host);
    HIP_CHECK(hipStreamSynchronize(stream()));
    return *s->best_host;
}

// every step of the state is one of a run (BatchRun), also with a single sequence
bool steps_on_run(const InferenceState *s) { return s->borrows_tiles || s->stack; }

// ---- a step in one launch (token.hip)

struct TokenRun {
    TokenShape shape;
    TokenArgs args;                      // what stays from step to step
    unsigned long long *words;           // hand-overs, and behind them
    uint64_t *table;                     // the layers' addresses
    std::vector<TokenLayer> layers;      // as the table holds them
    int *fail;                           // pinned: a wait ran out
    size_t n_words;
    uint64_t tag;                        // the next step's first; a step's NL + 1 fit 32 bits (next_tags)
    long steps;
    int rest, pause, good;               // steps that go in launches yet; as many after the next wait that runs out; taken since the last one
};

void token_release(TokenRun *r)
{
    if (!r) return;
    hipStreamSynchronize(stream());
    if (r->words) hipFree(r->words);
    if (r->fail) hipHostFree(r->fail);
    delete r;
}

__global__ __launch_bounds__(TB) void k_clear_words(unsigned long long *w, size_t n)
{
    const size_t i = (size_t)blockIdx.x * TB + threadIdx.x;
    if (i < n) w[i] = 0;
}

void clear_words(TokenRun &r)
{
    hipLaunchKernelGGL(k_clear_words, dim3((unsigned)((r.n_words + TB - 1) / TB)), dim3(TB), 0, stream(), r.words, r.n_words);
    HIP_CHECK(hipGetLastError());
}

// Tags of a step: one per layer and one behind them, for all kinds of words alike, none of which a word may hold.  Every step writes all words but those
// of the argmax, so only these could keep a tag until it is given out again: before that the words are cleared.
uint32_t next_tags(TokenRun &r)
{
    if (r.tag + r.args.NL > UINT32_MAX) { clear_words(r); r.tag = 1; }
    const uint32_t first = (uint32_t)r.tag;
    r.tag += r.args.NL + 1;
    return first;
}

// addresses of a weight's rows; false where they do not stay with the buffer or are not aligned
bool token_rows(InferenceState *s, const WMat *w, int rows, int cols, uint64_t *data, uint64_t *scales)
{
    const void *p = nullptr, *d = nullptr;
    if (s->use_fp16) {
        if (w->mbuf->size < (size_t)rows * cols * 2) return false;
        p = dptr(w->mbuf);
    } else if (!q8_rows_of(w->mbuf, rows, cols, &p, &d)) return false;
    *data = (uint64_t)p; *scales = (uint64_t)d;
    return !((uintptr_t)p & 15);
}

// The run, with the layers' addresses as they are now; NULL: the step goes in launches.  Those it is for: the matrix-vector pipeline's own
// weights without adapters, contexts of up to TOKEN_KEYS keys, shapes that the kernel holds (token_fits) and for which it is the faster way (token_pays).
// A profile of the products wants launches to count.
// TOKEN_KEYS is where k_attn_short ends, up to which launches and one launch were compared, and not where the one launch falls behind.  Microseconds of
// a greedy token at 200 / 300 / 1000 / 2000 keys, launches -> its attention's loop carried on: eight Gemma3-1B layers F16 273 -> 245 / 573 -> 271 /
// 579 -> 428 / 588 -> 657, Q8_0 261 -> 211 / 557 -> 227 / 576 -> 351 / 577 -> 534; six 4B layers F16 340 -> 319 / 518 -> 328 / 531 -> 390 / 537 -> 479, Q8_0 267 ->
// 250 / 448 -> 259 / 459 -> 321 / 462 -> 411; twelve of width 1024 F16 288 -> 272 / 541 -> 293 / 556 -> 448 / 570 -> 669.
TokenRun *token_acquire(InferenceState *s, int pos)
{
    if (s->steps_in_launches || steps_on_run(s) || !s->lora.empty() || pos >= TOKEN_KEYS || gemm_profiling()) return nullptr;
    const bool gemma = s->model_type == MODEL_GEMMA3;
    const TokenShape shape{s->D, s->IS, s->Hq, s->Hkv, s->hd, s->NL, s->V};
    const int qd = s->Hq * s->hd, kd = s->Hkv * s->hd;
    bool ok = s->one_launch || (token_fits(shape) && token_pays(shape, s->use_fp16 ? 0 : 1));
    std::vector<TokenLayer> now(ok ? s->NL : 0);
    for (int L = 0; ok && L < s->NL; L++) {
        const InferenceState::Layer &lw = s->layers[L];
        TokenLayer &t = now[L];
        ok = token_rows(s, &lw.qkv, qd + 2 * kd, s->D, &t.qkv, &t.qkv_d) && token_rows(s, lw.o, s->D, qd, &t.o, &t.o_d) &&
             token_rows(s, &lw.gu, 2 * s->IS, s->D, &t.gu, &t.gu_d) && token_rows(s, lw.down, s->D, s->IS, &t.down, &t.down_d);
        auto norm = [](MetalBuf *b) { return b ? (uint64_t)dptr(b) : 0; };
        t.g_in = norm(lw.g_in); t.g_post_attn = gemma ? norm(lw.g_post_attn) : 0; t.g_ff = norm(gemma ? lw.g_pre_ff : lw.g_post_attn);
        t.g_post_ff = gemma ? norm(lw.g_post_ff) : 0; t.g_q = norm(lw.g_q); t.g_k = norm(lw.g_k);
        t.kc = (uint64_t)dptr(s->kc[L]); t.vc = (uint64_t)dptr(s->vc[L]);
        t.rope = (uint64_t)(dptr_as<float2>(s->rope_tabs) + (size_t)s->theta_slot[L] * s->max_seq * (s->hd / 2));
        ok = ok && t.g_in && t.g_ff && (!gemma || (t.g_post_attn && t.g_post_ff));
        for (uint64_t p : {t.g_in, t.g_post_attn, t.g_ff, t.g_post_ff, t.g_q, t.g_k, t.kc, t.vc, t.rope}) ok = ok && !(p & 15);
    }
    uint64_t head = 0, head_d = 0;
    ok = ok && token_rows(s, s->lm_head, s->V, s->D, &head, &head_d) && s->emb && s->g_final && !(((uintptr_t)dptr(s->emb) | (uintptr_t)dptr(s->g_final)) & 15);
    if (!ok) { s->steps_in_launches = true; return nullptr; }
    if (!s->one_launch) {
        TokenRun *r = new TokenRun();
        const size_t n = token_words(shape, nullptr, nullptr), bytes = n * 8 + s->NL * sizeof(TokenLayer);
        // (a state that fills the device goes on in launches, which need none of this)
        bool there = bytes <= s->step_bytes;
        if (there && hipMalloc((void **)&r->words, bytes) != hipSuccess) { r->words = nullptr; there = false; }
        if (there && hipHostMalloc((void **)&r->fail, sizeof(int), hipHostMallocDefault) != hipSuccess) { r->fail = nullptr; there = false; }
        if (!there) {
            (void)hipGetLastError();
            token_release(r);
            s->steps_in_launches = true;
            return nullptr;
        }
        *r->fail = 0;
        r->shape = shape; r->tag = 1; r->pause = PAUSE;
        r->n_words = n;
        r->table = (uint64_t *)(r->words + n);
        clear_words(*r);
        TokenArgs &a = r->args;
        token_words(shape, &a, r->words);
        a.layers = r->table;
        a.fail = r->fail;
        a.NL = s->NL; a.D = s->D; a.IS = s->IS; a.Hq = s->Hq; a.Hkv = s->Hkv; a.hd = s->hd; a.max_seq = s->max_seq; a.V = s->V;
        a.gemma = gemma; a.emb_scale = s->emb_scale; a.eps = s->eps; a.scale = 1.0f / sqrtf((float)s->hd);
        s->one_launch = r;
    }
    TokenRun &r = *s->one_launch;
    if (r.layers.size() != now.size() || memcmp(r.layers.data(), now.data(), now.size() * sizeof(TokenLayer)) != 0) {
        r.layers = now;
        HIP_CHECK(hipMemcpyAsync(r.table, r.layers.data(), now.size() * sizeof(TokenLayer), hipMemcpyHostToDevice, stream()));
        HIP_CHECK(hipStreamSynchronize(stream()));
    }
    r.args.head = (const void *)head; r.args.head_d = (const void *)head_d;
    r.args.g_final = dptr_as<float>(s->g_final);
    r.args.logits = dptr_as<float>(s->logits);
    return &r;
}

// One step and the wait for it: the logits in logits_host, or the argmax in best_host.  false: not taken, or a wait ran out (the step is
// to be taken again, and the state's next ones go in launches).
bool token_in_one_launch(InferenceState *s, int token, int pos, bool logits)
{
    TokenRun *r = token_acquire(s, pos);
    if (!r) return false;
    if (r->rest > 0) { r->rest--; return false; }
    TokenArgs &a = r->args;
    a.emb_row = dptr_as<float>(s->emb) + (size_t)token * s->D;
    a.logits_host = logits ? s->logits_host : nullptr;
    a.best_host = logits ? nullptr : s->best_host;
    a.ticks = s->step_ticks; a.tag = next_tags(*r); a.pos = pos;
    launch_token(a, r->shape, s->use_fp16 ? 0 : 1);
    for (int L = 0; L < s->NL; L++) { mark_written(s->kc[L]); mark_written(s->vc[L]); }
    mark_written(s->logits);
    HIP_CHECK(hipStreamSynchronize(stream()));
    if (*(volatile int *)r->fail) {
        *r->fail = 0;
        r->rest = r->pause; r->pause = std::min(2 * r->pause, PAUSE_MOST); r->good = 0;
        return false;
    }
    r->steps++;
    if (++r->good >= r->pause) { r->pause = std::max(r->pause / 2, PAUSE); r->good = 0; }
    return true;
}

void default_eos(InferenceState *s)
{
    if (s->stack) { s->n_eos = 0; return; }                           // a design without end tokens of its own
    if (s->model_type == MODEL_GEMMA3) { s->eos[0] = 1; s->eos[1] = 106; }            // <eos>, <end_of_turn>
    else { s->eos[0] = 151645; s->eos[1] = 151643; }
    s->n_eos = 2;
}

// what every state has: sizes, end tokens, the host copies of logits and argmax
InferenceState *base_state(ModelType mt, int D, int V, int NL, int max_seq, LayerStack *stack = nullptr)
{
    InferenceState *s = new InferenceState();
    s->D = D; s->V = V; s->NL = NL;
    s->max_seq = max_seq; s->cur_len = 0; s->model_type = mt;
    s->stack = stack;
    s->step_ticks = STEP_TICKS; s->step_bytes = SIZE_MAX;
    default_eos(s);
    HIP_CHECK(hipHostMalloc((void **)&s->logits_host, (size_t)V * 4, hipHostMallocDefault));
    HIP_CHECK(hipHostMalloc((void **)&s->best_host, sizeof(int), hipHostMallocDefault));
    return s;
}

InferenceState *new_state(ModelType mt, int D, int Hq, int Hkv, int hd, int IS, int V, int NL, int max_seq, int use_fp16,
                          const float *thetas, bool matvec_path = true)
{
    if (fast_metal_init() != 0) { fprintf(stderr, "[FastGen] no GPU: fast_metal_init failed\n"); return nullptr; }
    if (Hkv <= 0 || Hq % Hkv || hd > 256 || (hd & 1) || Hq / Hkv > 16 || max_seq <= 0 || (IS & 3)) {
        fprintf(stderr, "[FastGen] unsupported shape: %d / %d heads of %d (head_dim even and <= 256, group ratio <= 16, FFN width a multiple of 4)\n", Hq, Hkv, hd);
        fast_metal_shutdown();
        return nullptr;
    }
    InferenceState *s = base_state(mt, D, V, NL, max_seq);
    s->Hq = Hq; s->Hkv = Hkv; s->hd = hd; s->IS = IS; s->use_fp16 = use_fp16;
    s->emb_scale = mt == MODEL_GEMMA3 ? sqrtf((float)D) : 1.0f;
    s->eps = 1e-6f;                                                       // src/nn/fast_inference.c:383
    s->thetas.assign(thetas, thetas + NL);
    {                                                                     // one table per distinct RoPE base
        std::vector<float> distinct;
        for (int L = 0; L < NL; L++) {
            size_t k = 0;
            while (k < distinct.size() && distinct[k] != thetas[L]) k++;
            if (k == distinct.size()) distinct.push_back(thetas[L]);
            s->theta_slot.push_back((int)k);
        }
        const size_t per = (size_t)max_seq * (hd / 2);
        s->rope_tabs = metal_buf_create(distinct.size() * per * sizeof(float2));
        for (size_t k = 0; k < distinct.size(); k++) launch_rope_table(dptr_as<float2>(s->rope_tabs) + k * per, max_seq, hd, distinct[k]);
    }
    const int qd = Hq * hd, kd = Hkv * hd;
    if (matvec_path) {                                                    // scratch and caches of the matrix-vector pipeline
        s->x = fbuf(D); s->x2 = fbuf(D); s->branch = fbuf(D); s->ln = fbuf(D);
        s->qkv = fbuf(qd + 2 * kd); s->att = fbuf(qd);
        s->gu = fbuf(2 * (size_t)IS);
        s->gate_v = metal_buf_view(s->gu, 0, (size_t)IS * 4); s->up_v = metal_buf_view(s->gu, (size_t)IS * 4, (size_t)IS * 4);
        s->logits = fbuf(V); s->best = metal_buf_create(2 * AM_WGS * sizeof(int));   // the per-workgroup values, then indices
        const size_t cache_bytes = (size_t)Hkv * max_seq * hd * sizeof(float);
        for (int L = 0; L < NL; L++) { s->kc.push_back(metal_buf_create(cache_bytes)); s->vc.push_back(metal_buf_create(cache_bytes)); }
    }
    s->R = 0; s->scaling = 0.f; s->lora_t = nullptr;
    s->sft = nullptr; s->owns_weights = 0;
    s->layers.resize(NL);
    s->lm_head = nullptr; s->g_final = s->emb = nullptr;
    return s;
}

// "eos_token_id": 7  or  "eos_token_id": [1, 106]  in the text of a config.json
int eos_ids_in(const std::string &text, int *out, int max_out)
{
    const std::string key = "\"eos_token_id\"";
    size_t p = text.find(key);
    if (p == std::string::npos) return 0;
    p = text.find(':', p + key.size());
    if (p == std::string::npos) return 0;
    p = text.find_first_not_of(" \t\r\n", p + 1);
    if (p == std::string::npos) return 0;
    int n = 0;
    const bool list = text[p] == '[';
    if (list) p++;
    while (p < text.size() && n < max_out) {
        p = text.find_first_not_of(" \t\r\n,", p);
        if (p == std::string::npos || text[p] == ']') break;
        char *end = nullptr;
        const long id = strtol(text.c_str() + p, &end, 10);
        if (end == text.c_str() + p) break;
        out[n++] = (int)id;
        p = (size_t)(end - text.c_str());
        if (!list) break;
    }
    return n;
}

}  // namespace

extern "C" {

InferenceState *inference_state_create_from_ref(const SFTModelRef *m, int max_seq_len, int use_fp16)
{
    if (model_type_layered(m->model_type)) { fprintf(stderr, "[FastGen] %s models are created by inference_state_create_from_file\n", model_type_name(m->model_type)); return nullptr; }
    InferenceState *s = new_state(m->model_type, m->d_model, m->n_q_heads, m->n_kv_heads, m->head_dim, m->intermediate_size,
                                  m->vocab_size, m->n_layers, max_seq_len, use_fp16, m->rope_thetas);
    if (!s) return nullptr;
    // [Wq; Wk; Wv] and [Wgate; Wup] are converted as one matrix each: F16 rounding and Q8_0 blocks are per row, so
    // the rows of the fused matrix are bit for bit those of wmat_create_f16 / wmat_create_q8 on the parts
    std::vector<float> cat;
    auto fused = [&](std::initializer_list<const WeightRef *> parts) {
        int rows = 0;
        const int cols = (*parts.begin())->cols;
        for (const WeightRef *w : parts) rows += w->rows;
        cat.resize((size_t)rows * cols);
        size_t o = 0;
        for (const WeightRef *w : parts) { memcpy(cat.data() + o, w->data, (size_t)w->rows * cols * sizeof(float)); o += (size_t)w->rows * cols; }
        WMat *t = wmat_convert(cat.data(), rows, cols, use_fp16);
        WMat out = *t;
        free(t);                                                          // the handle only; the buffer lives on in `out`
        return out;
    };
    for (int L = 0; L < m->n_layers; L++) {
        const LayerWeightRef *r = &m->layers[L];
        InferenceState::Layer &lw = s->layers[L];
        lw.qkv = fused({&r->q_proj, &r->k_proj, &r->v_proj});
        lw.gu = fused({&r->gate_proj, &r->up_proj});
        lw.o = wmat_convert(r->o_proj.data, r->o_proj.rows, r->o_proj.cols, use_fp16);
        lw.down = wmat_convert(r->down_proj.data, r->down_proj.rows, r->down_proj.cols, use_fp16);
        lw.g_in = norm_upload(r->input_norm_g, r->d_model);
        lw.g_post_attn = norm_upload(r->post_attn_norm_g, r->d_model);
        lw.g_pre_ff = r->pre_ff_norm_g ? norm_upload(r->pre_ff_norm_g, r->d_model) : nullptr;
        lw.g_post_ff = r->post_ff_norm_g ? norm_upload(r->post_ff_norm_g, r->d_model) : nullptr;
        lw.g_q = r->q_norm_g ? norm_upload(r->q_norm_g, r->head_dim) : nullptr;
        lw.g_k = r->k_norm_g ? norm_upload(r->k_norm_g, r->head_dim) : nullptr;
    }
    s->lm_head = wmat_convert(m->lm_head, m->vocab_size, m->d_model, use_fp16);
    s->g_final = norm_upload(m->final_norm_g, m->d_model);
    s->emb = metal_buf_from_data(m->token_emb, (size_t)m->vocab_size * m->d_model * sizeof(float));
    s->owns_weights = 1;
    return s;
}

// Straight from the file to HBM: every matrix is uploaded as stored and converted on the GPU (F16 and Q8_0 tensors that
// already have the wanted format are used bit for bit); Q|K|V and gate|up are joined by device copies of whole rows.
static InferenceState *stack_state_from_file(const char *path, ModelType model_type, int max_seq_len, int weight_format);

InferenceState *inference_state_create_from_file(const char *path, ModelType model_type, int max_seq_len, int use_fp16)
{
    if (model_type_layered(model_type)) return stack_state_from_file(path, model_type, max_seq_len, use_fp16);
    if (use_fp16 == 2) { fprintf(stderr, "[FastGen] %s weights are F16 or Q8_0\n", model_type_name(model_type)); return nullptr; }
    ModelFile *f = model_file_open(path);
    if (!f) return nullptr;
    const bool gg = model_file_is_gguf(f);
    if (gg && model_type == MODEL_GEMMA3) { fprintf(stderr, "[FastGen] Gemma3 is read from safetensors only\n"); model_file_close(f); return nullptr; }
    auto lname = [&](int L, const char *hf, const char *g) {
        char buf[256];
        if (gg) snprintf(buf, sizeof buf, "blk.%d.%s.weight", L, g); else snprintf(buf, sizeof buf, "model.layers.%d.%s.weight", L, hf);
        return std::string(buf);
    };
    const char *emb_name = gg ? "token_embd.weight" : "model.embed_tokens.weight";
    int V = 0, D = 0, NL = 0, qd = 0, kd = 0, IS = 0, hd = 0, one = 0, c = 0;
    bool ok = model_file_matrix_shape(f, emb_name, &V, &D) != 0;
    while (ok && model_file_find(f, lname(NL, "self_attn.q_proj", "attn_q").c_str(), nullptr, nullptr, nullptr)) NL++;
    ok = ok && NL > 0 && model_file_matrix_shape(f, lname(0, "self_attn.q_proj", "attn_q").c_str(), &qd, &c) && c == D &&
         model_file_matrix_shape(f, lname(0, "self_attn.k_proj", "attn_k").c_str(), &kd, &c) && c == D &&
         model_file_matrix_shape(f, lname(0, "mlp.gate_proj", "ffn_gate").c_str(), &IS, &c) && c == D &&
         model_file_matrix_shape(f, lname(0, "self_attn.q_norm", "attn_q_norm").c_str(), &one, &hd) && hd > 0 && qd % hd == 0 && kd % hd == 0;
    if (!ok) { fprintf(stderr, "[FastGen] %s: embedding or layer 0 tensors missing or inconsistent\n", path); model_file_close(f); return nullptr; }
    const bool gemma = model_type == MODEL_GEMMA3;
    std::vector<float> thetas(NL);
    for (int L = 0; L < NL; L++) thetas[L] = gemma ? ((L % 6) != 0 ? 1e4f : 1e6f) : 1e6f;   // src/nn/fast_sft.c:308-313
    InferenceState *s = new_state(model_type, D, qd / hd, kd / hd, hd, IS, V, NL, max_seq_len, use_fp16, thetas.data());
    if (!s) { model_file_close(f); return nullptr; }
    s->owns_weights = 1;
    auto gamma = [&](const std::string &name, int dim) -> MetalBuf * {
        size_t n = 0;
        float *g = model_file_load_f32(f, name.c_str(), &n);
        if (!g || (int)n != dim) { free(g); ok = false; return nullptr; }
        if (gemma) for (size_t i = 0; i < n; i++) g[i] += 1.0f;                            // src/nn/gemma3.c:259-278
        MetalBuf *b = norm_upload(g, dim);
        free(g);
        return b;
    };
    auto matrix = [&](const std::string &name, int rows, int cols) -> WMat * {
        WMat *w = model_file_load_wmat(f, name.c_str(), use_fp16);
        if (!w || w->rows != rows || w->cols != cols) { fprintf(stderr, "[FastGen] %s: expected %d x %d\n", name.c_str(), rows, cols); wmat_free(w); ok = false; return nullptr; }
        return w;
    };
    auto fuse = [&](std::initializer_list<WMat *> parts, int cols) {
        int rows = 0;
        for (WMat *w : parts) { if (!w) return WMat{nullptr, 0, 0, 0}; rows += w->rows; }
        const size_t row_bytes = use_fp16 ? (size_t)cols * 2 : (size_t)(cols / 32) * 34;
        WMat out{metal_buf_create((size_t)rows * row_bytes), rows, cols, use_fp16 ? 0 : cols / 32};
        size_t o = 0;
        for (WMat *w : parts) {
            HIP_CHECK(hipMemcpyAsync((char *)dptr(out.mbuf) + o, dptr(w->mbuf), (size_t)w->rows * row_bytes, hipMemcpyDeviceToDevice, stream()));
            o += (size_t)w->rows * row_bytes;
        }
        mark_written(out.mbuf);
        for (WMat *w : parts) wmat_free(w);                                                // synchronises the stream first
        return out;
    };
    for (int L = 0; L < NL && ok; L++) {
        InferenceState::Layer &lw = s->layers[L];
        lw.g_in = gamma(lname(L, "input_layernorm", "attn_norm"), D);
        lw.qkv = fuse({matrix(lname(L, "self_attn.q_proj", "attn_q"), qd, D), matrix(lname(L, "self_attn.k_proj", "attn_k"), kd, D),
                       matrix(lname(L, "self_attn.v_proj", "attn_v"), kd, D)}, D);
        lw.g_q = gamma(lname(L, "self_attn.q_norm", "attn_q_norm"), hd);
        lw.g_k = gamma(lname(L, "self_attn.k_norm", "attn_k_norm"), hd);
        lw.o = matrix(lname(L, "self_attn.o_proj", "attn_output"), D, qd);
        lw.g_post_attn = gamma(lname(L, "post_attention_layernorm", "ffn_norm"), D);
        if (gemma) lw.g_pre_ff = gamma(lname(L, "pre_feedforward_layernorm", ""), D);
        lw.gu = fuse({matrix(lname(L, "mlp.gate_proj", "ffn_gate"), IS, D), matrix(lname(L, "mlp.up_proj", "ffn_up"), IS, D)}, D);
        lw.down = matrix(lname(L, "mlp.down_proj", "ffn_down"), D, IS);
        if (gemma) lw.g_post_ff = gamma(lname(L, "post_feedforward_layernorm", ""), D);
    }
    if (ok) {
        s->g_final = gamma(gg ? "output_norm.weight" : "model.norm.weight", D);
        const char *head = gg ? "output.weight" : "lm_head.weight";
        const bool tied = gemma || !model_file_find(f, head, nullptr, nullptr, nullptr);   // src/nn/qwen3.c:264-270, 363-367
        s->lm_head = matrix(tied ? emb_name : head, V, D);
        size_t n = 0;
        float *emb = model_file_load_f32(f, emb_name, &n);
        if (emb && n == (size_t)V * D) s->emb = metal_buf_from_data(emb, n * sizeof(float)); else ok = false;
        free(emb);
    }
    model_file_close(f);
    if (!ok) { fprintf(stderr, "[FastGen] %s: a tensor is missing or mis-shaped\n", path); inference_state_free(s); return nullptr; }
    return s;
}

// A model described layer by layer: config.json beside the weights says what the layers are.
static InferenceState *stack_state_from_file(const char *path, ModelType model_type, int max_seq_len, int weight_format)
{
    if (weight_format != 1 && weight_format != 2) { fprintf(stderr, "[FastGen] %s weights are F16 or 32-bit\n", model_type_name(model_type)); return nullptr; }
    if (max_seq_len <= 0) return nullptr;
    const std::string cfg_path = config_path_of(path);
    std::ifstream in(cfg_path);
    std::stringstream text;
    if (in) text << in.rdbuf();
    StackConfig cfg;
    std::string why;
    if (!in || !read_stack_config(text.str(), model_type, cfg, why)) {
        fprintf(stderr, "[FastGen] %s: %s\n", cfg_path.c_str(), in ? why.c_str() : "cannot be read");
        return nullptr;
    }
    if (fast_metal_init() != 0) { fprintf(stderr, "[FastGen] no GPU: fast_metal_init failed\n"); return nullptr; }
    ModelFile *f = model_file_open(path);
    LayerStack *st = f ? stack_load(f, cfg, weight_format == 2, max_seq_len) : nullptr;
    model_file_close(f);
    if (!st) { fast_metal_shutdown(); return nullptr; }
    InferenceState *s = base_state(model_type, cfg.width, cfg.vocab, (int)cfg.layers.size(), max_seq_len, st);
    s->use_fp16 = weight_format;
    return s;
}

InferenceState *inference_state_create_from_sft(SFTState *sft, int max_seq_len)
{
    InferenceState *s = new_state(sft_get_model_type(sft), sft_get_d_model(sft), sft_get_n_q_heads(sft), sft_get_n_kv_heads(sft),
                                  sft_get_head_dim(sft), sft_get_intermediate_size(sft), sft_get_vocab_size(sft),
                                  sft_get_n_layers(sft), max_seq_len, 1, sft_get_rope_thetas(sft), false);
    if (!s) return nullptr;
    if (s->D > 8192) { fprintf(stderr, "[FastGen] hidden size %d not supported for a state on a training state's weights (<= 8192)\n", s->D); inference_state_free(s); return nullptr; }
    s->sft = sft;
    s->g_final = sft_get_final_norm_g(sft);
    s->emb = sft_get_token_emb_buf(sft);
    s->borrows_tiles = 1;
    s->borrowed.resize(s->NL);
    for (int L = 0; L < s->NL; L++) {
        sft_borrow_layer(sft, L, &s->borrowed[L]);
        const BorrowedLayer &b = s->borrowed[L];
        InferenceState::Layer &lw = s->layers[L];
        lw.g_in = b.g_in; lw.g_post_attn = b.g_post_attn; lw.g_pre_ff = b.g_pre_ff; lw.g_post_ff = b.g_post_ff; lw.g_q = b.g_q; lw.g_k = b.g_k;
    }
    s->borrowed_lm = sft_borrow_lm_head(sft);
    s->use_fp16 = s->borrowed_lm.fmt == 0;
    inference_state_set_lora(s, sft);
    return s;
}

// Kept for callers written against copies: a state made from a training state reads that state's weights in place, so
// there is nothing to refresh after a full-parameter update.
void inference_state_refresh_from_sft(InferenceState *s) { (void)s; }

void inference_state_set_lora(InferenceState *s, SFTState *sft)
{
    if (s->stack) { fprintf(stderr, "[FastGen] %s takes no adapters\n", model_type_name(s->model_type)); return; }
    const int R = sft_get_lora_rank(sft);
    if (R == 0) return;                                                   // full-parameter state: no adapters
    if (!s->lora_t && !s->borrows_tiles) s->lora_t = fbuf(2 * (size_t)R);
    s->lora.resize(s->NL);
    for (int L = 0; L < s->NL; L++)
        s->lora[L] = InferenceState::Lora{sft_get_lora_weight_buf(sft, L, 0), sft_get_lora_weight_buf(sft, L, 1),
                                          sft_get_lora_weight_buf(sft, L, 2), sft_get_lora_weight_buf(sft, L, 3)};
    s->R = R;
    s->scaling = sft_get_lora_scaling(sft);
}

void inference_state_free(InferenceState *s)
{
    if (!s) return;
    metal_flush();
    batch_release(s->batch);
    batch_release(s->single);
    prompt_release(s->prompt);
    token_release(s->one_launch);
    stack_free(s->stack);
    for (MetalBuf *b : {s->gate_v, s->up_v, s->x, s->x2, s->branch, s->ln, s->qkv, s->att, s->gu, s->logits, s->best, s->lora_t, s->rope_tabs})
        metal_buf_free(b);
    for (MetalBuf *b : s->kc) metal_buf_free(b);
    for (MetalBuf *b : s->vc) metal_buf_free(b);
    hipHostFree(s->logits_host);
    hipHostFree(s->best_host);
    for (InferenceState::Layer &lw : s->layers) {
        metal_buf_free(lw.qkv.mbuf);
        metal_buf_free(lw.gu.mbuf);
        if (s->owns_weights) {
            wmat_free(lw.o); wmat_free(lw.down);
            for (MetalBuf *b : {lw.g_in, lw.g_post_attn, lw.g_pre_ff, lw.g_post_ff, lw.g_q, lw.g_k}) metal_buf_free(b);
        }
    }
    if (s->owns_weights) {
        wmat_free(s->lm_head);
        metal_buf_free(s->g_final);
        metal_buf_free(s->emb);
    }
    delete s;
    fast_metal_shutdown();
}

ModelType inference_state_model_type(InferenceState *s) { return s->model_type; }
int inference_state_vocab_size(InferenceState *s) { return s->V; }
void inference_state_reset(InferenceState *s) { s->cur_len = 0; }
long hip_inference_steps_in_one_launch(InferenceState *s) { return s && s->one_launch ? s->one_launch->steps : 0; }
void hip_inference_step_wait(InferenceState *s, long long ticks) { if (s && ticks >= 0) s->step_ticks = (uint64_t)ticks; }
void hip_inference_step_memory(InferenceState *s, size_t bytes) { if (s) s->step_bytes = bytes; }
long long hip_inference_step_tag(InferenceState *s, long long set)
{
    if (!s || !s->one_launch) return 0;
    if (set > 0) { clear_words(*s->one_launch); s->one_launch->tag = (uint64_t)set; }
    return (long long)s->one_launch->tag;
}
int inference_state_position(InferenceState *s) { return s->cur_len; }

static bool token_ok(InferenceState *s, int token)
{
    if (token < 0 || token >= s->V) { fprintf(stderr, "[FastGen] token %d outside the vocabulary (%d)\n", token, s->V); return false; }
    if (s->cur_len >= s->max_seq) { fprintf(stderr, "[FastGen] KV cache full (%d positions)\n", s->max_seq); return false; }
    return true;
}

static void step_token(InferenceState *s, int token, int pos)
{
    if (steps_on_run(s)) step_on_run(s, token, pos);
    else forward_token(s, token, pos);
}
static int argmax_host(InferenceState *s) { return steps_on_run(s) ? argmax_on_run(s) : argmax_to_host(s); }
// a step whose result the host waits for
static const float *step_logits(InferenceState *s, int token, int pos)
{
    if (token_in_one_launch(s, token, pos, true)) return s->logits_host;
    if (steps_on_run(s)) return step_logits_on_run(s, token, pos);
    if (!forward_token(s, token, pos, s->logits_host)) return logits_to_host(s);
    HIP_CHECK(hipStreamSynchronize(stream()));
    return s->logits_host;
}
static int step_argmax(InferenceState *s, int token, int pos)
{
    if (token_in_one_launch(s, token, pos, false)) return *s->best_host;
    step_token(s, token, pos);
    return argmax_host(s);
}

const float *inference_forward_token(InferenceState *s, int token)
{
    if (!token_ok(s, token)) return nullptr;
    return step_logits(s, token, s->cur_len++);
}

int inference_forward_token_argmax(InferenceState *s, int token)
{
    if (!token_ok(s, token)) return -1;
    return step_argmax(s, token, s->cur_len++);
}

// The next n tokens of the sequence from the current position on, and the logits at the places want[0 .. n_want)
// (ascending) among them.
int inference_forward_tokens(InferenceState *s, const int *tokens, int n, const int *want, int n_want, float *logits)
{
    if (!s || !tokens || n <= 0 || n_want < 0 || (n_want && (!want || !logits))) return -1;
    if (n > s->max_seq - s->cur_len) { fprintf(stderr, "[FastGen] %d more tokens do not fit %d positions\n", n, s->max_seq); return -1; }
    for (int i = 0; i < n; i++) if (!token_ok(s, tokens[i])) return -1;
    for (int i = 0; i < n_want; i++)
        if (want[i] < 0 || want[i] >= n || (i && want[i] <= want[i - 1])) { fprintf(stderr, "[FastGen] wanted places must ascend inside the portion\n"); return -1; }
    if (s->stack) return forward_rows(s, tokens, n, want, n_want, logits);
    if (prompt_takes(s, n)) return prompt_forward(s, tokens, n, want, n_want, logits);
    for (int i = 0, w = 0; i < n; i++) {                                  // the other models take one token per step
        if (w < n_want && want[w] == i) memcpy(logits + (size_t)w++ * s->V, step_logits(s, tokens[i], s->cur_len), (size_t)s->V * sizeof(float));
        else step_token(s, tokens[i], s->cur_len);
        s->cur_len++;
    }
    metal_flush();
    return 0;
}

int inference_generate(InferenceState *s, const uint32_t *prompt_tokens, int prompt_len, uint32_t *output_tokens, int max_gen_len)
{
    s->cur_len = 0;
    if (prompt_len <= 0 || max_gen_len <= 0 || prompt_len > s->max_seq) return 0;
    int good = 0;                                                     // tokens ahead of one outside the vocabulary, if there is one
    while (good < prompt_len && token_ok(s, (int)prompt_tokens[good])) good++;
    // prefill: only the last logits are looked at
    if (s->stack) {
        if (good < prompt_len) return 0;
        prefill_on_run(s, prompt_tokens, prompt_len, 0);
    }
    else if (good == prompt_len && prompt_takes(s, prompt_len)) prompt_fill(s, prompt_tokens, prompt_len);
    else for (int i = 0; i < good; i++) step_token(s, (int)prompt_tokens[i], i);
    s->cur_len = good;
    if (good < prompt_len) return 0;
    int next = argmax_host(s);
    output_tokens[0] = (uint32_t)next;
    int n_gen = 1;
    for (int gen = 1; gen < max_gen_len && s->cur_len < s->max_seq; gen++) {
        bool is_eos = false;
        for (int e = 0; e < s->n_eos; e++) is_eos |= next == s->eos[e];
        if (is_eos) break;
        next = step_argmax(s, next, s->cur_len++);
        output_tokens[n_gen++] = (uint32_t)next;
    }
    return n_gen;
}

namespace {

// the embedding rows of a batch of tokens, scaled: x[b] = emb[tokens.id[b]] * scale
struct TokenIds { int id[32]; };
__global__ __launch_bounds__(TB) void k_embed_rows(const float *__restrict__ emb, TokenIds tokens, float scale, float *__restrict__ x, int D)
{
    const int i = blockIdx.x * TB + threadIdx.x, b = blockIdx.y;
    if (i < D) x[(size_t)b * D + i] = emb[(size_t)tokens.id[b] * D + i] * scale;
}

// k_argmax_part and k_argmax_final for every vector of a batch at once (blockIdx.y: the vector)
__global__ __launch_bounds__(TB) void k_argmax_part_batch(const float *__restrict__ v, int n, float *__restrict__ pv, int *__restrict__ pi)
{
    __shared__ float bv[4];
    __shared__ int bi[4];
    v += (size_t)blockIdx.y * n; pv += (size_t)blockIdx.y * AM_WGS; pi += (size_t)blockIdx.y * AM_WGS;
    float best = -INFINITY;
    int idx = 0x7fffffff;
    for (int i = blockIdx.x * TB + threadIdx.x; i < n; i += AM_WGS * TB) am_pick(best, idx, v[i], i);
    am_block(best, idx, bv, bi);
    if (threadIdx.x == 0) { pv[blockIdx.x] = best; pi[blockIdx.x] = idx; }
}

__global__ __launch_bounds__(AM_WGS) void k_argmax_final_batch(const float *__restrict__ pv, const int *__restrict__ pi, int *__restrict__ out)
{
    __shared__ float bv[AM_WGS / 64];
    __shared__ int bi[AM_WGS / 64];
    float best = pv[(size_t)blockIdx.x * AM_WGS + threadIdx.x];
    int idx = pi[(size_t)blockIdx.x * AM_WGS + threadIdx.x];
    am_block(best, idx, bv, bi);
    if (threadIdx.x == 0) out[blockIdx.x] = idx == 0x7fffffff ? 0 : idx;
}

// Scratch and KV caches of a batch of B sequences decoded in lock step (BatchState of src/nn/fast_inference.c:699-776).
struct BatchRun {
    StackRun *stk;                                                       // a layer-by-layer model's caches, states and scratch (then only logits and best besides)
    int B, R, len;                                                       // sequences; adapter rank the scratch was sized for; positions held by the caches
    bool few;                                                            // its products take the kernels for a few rows (few_rows_fit)
    MetalBuf *x, *ln, *qkv, *att, *act, *logits, *best, *lora_t;
    MetalBuf *a16, *inv_ln, *inv_br, *planes;                            // a product's operand, its factors (of ln | of att and act), its planes
    std::vector<MetalBuf *> kc, vc;                                      // per layer: [B][Hkv, max_seq, hd]
    int *best_host;
    float *logits_host;                                                  // pinned [B][V], made by the first step that hands logits out (batch_logits_to)
    hipEvent_t part_there[4];                                            // a part of it has arrived; those that are needed, made with it
};

void batch_release(BatchRun *r)
{
    if (!r) return;
    stack_run_free(r->stk);
    for (MetalBuf *b : {r->x, r->ln, r->qkv, r->att, r->act, r->logits, r->best, r->lora_t, r->a16, r->inv_ln, r->inv_br, r->planes}) metal_buf_free(b);
    for (MetalBuf *b : r->kc) metal_buf_free(b);
    for (MetalBuf *b : r->vc) metal_buf_free(b);
    if (r->best_host) hipHostFree(r->best_host);
    if (r->logits_host) hipHostFree(r->logits_host);
    for (hipEvent_t e : r->part_there) if (e) hipEventDestroy(e);
    delete r;
}

// A state whose batches take the kernels of few_rows.h: F16 weights, widths that fill their loads.  GPU time per step of 8 sequences,
// nine layers of the 4B shape: 662 us against 788 for the ring kernel's products with their planes summed, gated and split
// between them, which Q8_0 tiles and other widths keep.  It holds for any batch: four layers and logits, 2 / 8 / 32 sequences, ms
// per step 0.32 / 0.36 / 0.45 (before 0.36 / 0.38 / 0.51), of the Gemma3-1B shape 0.22 / 0.24 / 0.28 (0.27 / 0.28 / 0.36).
bool few_rows_fit(const InferenceState *s)
{
    const int qd = s->Hq * s->hd;
    if (s->D % 4 || s->D > 8192 || qd % 4 || s->IS % 32) return false;
    auto aligned = [](const MetalBuf *g) { return !g || ((uintptr_t)dptr(g) & 15) == 0; };
    if (!aligned(s->g_final) || (s->borrows_tiles && s->borrowed_lm.fmt)) return false;
    for (int L = 0; L < s->NL; L++) {
        const InferenceState::Layer &w = s->layers[L];
        if (!aligned(w.g_in) || !aligned(w.g_post_attn) || !aligned(w.g_pre_ff) || !aligned(w.g_post_ff)) return false;
        if (s->borrows_tiles) {
            const BorrowedLayer &b = s->borrowed[L];
            if (b.qkv.fmt || b.o.fmt || b.gu.fmt || b.down.fmt) return false;
        }
    }
    return true;
}

// Logits that the head's kernel stores into pinned memory leave it in parts of the vocabulary (whole row blocks of the weight, enough of them to fill the
// chip), so that the caller's copy of one part is made while the next one is formed.
int batch_parts(const InferenceState *s, const BatchRun &r)
{
    const size_t bytes = (size_t)r.B * s->V * sizeof(float);
    return bytes < ((size_t)512 << 10) || s->V < 16384 ? 1 : bytes < ((size_t)4 << 20) || s->V < 32768 ? 2 : 4;
}
int batch_part(const InferenceState *s, int i, int parts) { return i < parts ? (int)((long)s->V * i / parts / 32 * 32) : s->V; }   // its first column

// One step for B tokens at the same position: forward_token_batch, src/nn/fast_inference.c:808-893.  Every product
// reads its weight once for all B vectors (matrix cores over the tiled image, 22 bits of every activation); what
// is per sequence -- adapter terms, per-head RMSNorm, RoPE, cache store, attention -- has the sequence as a grid
// dimension, so a layer is the same 7 launches (one more with adapters) for any B, or 11 where few_rows_fit does not hold.  A
// product's planes are summed by the kernel that consumes them and the norm kernel writes the next product's operand itself,
// where a row is one workgroup's.
// host: pinned memory for the logits of a single sequence besides, or null; true: they go there as they are formed.
// to_host (r.few, r.logits_host there): the logits go to r.logits_host instead of r.logits, an event behind each part of batch_parts.
bool forward_token_batch(InferenceState *s, BatchRun &r, const int *tokens, int pos, float *host = nullptr, bool to_host = false)
{
    if (s->stack) {
        stack_forward(s->stack, r.stk, tokens, 1, pos);
        return stack_logits(s->stack, r.stk, nullptr, r.B, dptr_as<float>(r.logits), host);
    }
    const int D = s->D, Hq = s->Hq, Hkv = s->Hkv, hd = s->hd, IS = s->IS, B = r.B;
    const int qd = Hq * hd, kd = Hkv * hd, nqkv = qd + 2 * kd;
    const bool gemma = s->model_type == MODEL_GEMMA3;
    TokenIds ids{};
    for (int b = 0; b < B; b++) ids.id[b] = tokens[b];
    hipLaunchKernelGGL(k_embed_rows, dim3((D + TB - 1) / TB, B), dim3(TB), 0, stream(), dptr_as<float>(s->emb), ids, s->emb_scale,
                       dptr_as<float>(r.x), D);
    half_t *a16 = dptr_as<half_t>(r.a16);
    float *inv_ln = dptr_as<float>(r.inv_ln), *inv_br = dptr_as<float>(r.inv_br), *P = dptr_as<float>(r.planes);
    // x += branch (the planes `br` of the product before, none at the start); ln = RMSNorm(x) as fp32 (only the adapters
    // read it) and as the operand of the next product
    auto add_norm_b = [&](const auto &br, MetalBuf *g_branch, MetalBuf *g) {
        float *ln = (s->lora.empty() || s->borrows_tiles) ? nullptr : dptr_as<float>(r.ln);      // fp32 copy: only k_lora_down reads it
        const float *gb = g_branch ? dptr_as<float>(g_branch) : nullptr;
        if constexpr (std::is_same_v<std::decay_t<decltype(br)>, FewPlanes>) launch_few_norm(dptr_as<float>(r.x), br, gb, dptr_as<float>(g), ln, a16, inv_ln, B, D, s->eps);
        else launch_add_norm_split(dptr_as<float>(r.x), br, gb, dptr_as<float>(g), ln, a16, inv_ln, B, B, D, s->eps);
    };
    // planes of (the operand in a16) x w^T; `inv`: the factors that operand's rows were split with.  The weight: the
    // tiled image of the state's own row-major matrix (made on first use), or the training state's tiles
    auto weight = [&](const WMat *w, const WeightOp *tiles, int rows, int cols) { return tiles ? *tiles : weight_f16(tiled_weight_of(w->mbuf, rows, cols)); };
    auto product = [&](const WMat *w, const WeightOp *tiles, int rows, int cols, const float *inv) {
        const WeightOp op = weight(w, tiles, rows, cols);
        const GemmPlan p = plan_gemm(2 * B, rows, cols, op.fmt ? op.nbq : 0, op.fmt);
        const size_t plane = (size_t)2 * B * rows;
        launch_gemm(a16, nullptr, op, P, rows, plane, 2 * B, rows, cols, p);
        return SplitPlanes{P, inv, plane, p.S, rows, B};
    };
    const bool bt = s->borrows_tiles;
    auto split = [&](MetalBuf *in, int K) { launch_rows_to_f16_split(dptr_as<float>(in), a16, inv_br, B, K); };
    SplitPlanes pending{};                                               // FFN branch of the layer before, added by the next norm kernel
    FewPlanes pending_few{};
    MetalBuf *pending_g = nullptr;
    for (int L = 0; L < s->NL; L++) {
        const InferenceState::Layer &lw = s->layers[L];
        const BorrowedLayer *bl = bt ? &s->borrowed[L] : nullptr;
        if (r.few) add_norm_b(pending_few, pending_g, lw.g_in);
        else add_norm_b(pending, pending_g, lw.g_in);
        // a training state's fused matrix continues with the rows of A_q and A_v (their fp16 images, as its own forward
        // reads them): the product then yields the adapters' down-projections as well, and no launch forms them
        const bool t_in_product = bt && !s->lora.empty();
        const int nq_rows = nqkv + (t_in_product ? 2 * s->R : 0);
        if (r.few) launch_few_full(a16, inv_ln, weight(&lw.qkv, bt ? &bl->qkv : nullptr, nq_rows, D).w16, dptr_as<float>(r.qkv), nq_rows, B, nq_rows, D);
        else {
            const SplitPlanes qkv = product(&lw.qkv, bt ? &bl->qkv : nullptr, nq_rows, D, inv_ln);
            launch_reduce_planes_split(qkv.P, qkv.S, qkv.plane, qkv.N, qkv.inv, dptr_as<float>(r.qkv), B, qkv.N);
        }
        HeadPost a{};
        a.qkv = dptr_as<float>(r.qkv); a.qkv_step = (size_t)nq_rows;
        a.g_q = lw.g_q ? dptr_as<float>(lw.g_q) : nullptr; a.g_k = lw.g_k ? dptr_as<float>(lw.g_k) : nullptr;
        a.kc = dptr_as<float>(r.kc[L]); a.vc = dptr_as<float>(r.vc[L]); a.cache_step = (size_t)Hkv * s->max_seq * hd;
        a.Hq = Hq; a.Hkv = Hkv; a.pos = pos;
        a.rope = dptr_as<float2>(s->rope_tabs) + ((size_t)s->theta_slot[L] * s->max_seq + pos) * (hd / 2); a.eps = s->eps;
        if (!s->lora.empty()) {
            const InferenceState::Lora &lr = s->lora[L];
            if (t_in_product) { a.t = dptr_as<float>(r.qkv) + nqkv; a.t_step = (size_t)nq_rows; }
            else {
                hipLaunchKernelGGL(k_lora_down, dim3(2 * s->R, B), dim3(64), 0, stream(), dptr_as<float>(r.ln), dptr_as<float>(lr.Aq),
                                   dptr_as<float>(lr.Av), dptr_as<float>(r.lora_t), s->R, D);
                a.t = dptr_as<float>(r.lora_t); a.t_step = (size_t)2 * s->R;
            }
            a.Bq = dptr_as<float>(lr.Bq); a.Bv = dptr_as<float>(lr.Bv); a.R = s->R; a.sc = s->scaling;
        }
        attention_decode_fused(a, r.kc[L], r.vc[L], dptr_as<float>(r.att), hd, s->max_seq, B);
        MetalBuf *g_post = gemma ? lw.g_post_attn : nullptr, *g_ff = gemma ? lw.g_pre_ff : lw.g_post_attn;
        if (r.few) {
            add_norm_b(launch_few_split(dptr_as<float>(r.att), weight(lw.o, bt ? &bl->o : nullptr, D, qd).w16, P, B, D, qd), g_post, g_ff);
            launch_few_glu(a16, inv_ln, weight(&lw.gu, bt ? &bl->gu : nullptr, 2 * IS, D).w16, dptr_as<float>(r.act), B, IS, D, gemma ? 1 : 0);
            pending_few = launch_few_split(dptr_as<float>(r.act), weight(lw.down, bt ? &bl->down : nullptr, D, IS).w16, P, B, D, IS);
        }
        else {
            split(r.att, qd);
            const SplitPlanes o = product(lw.o, bt ? &bl->o : nullptr, D, qd, inv_br);
            add_norm_b(o, g_post, g_ff);
            const SplitPlanes gu = product(&lw.gu, bt ? &bl->gu : nullptr, 2 * IS, D, inv_ln);
            hipLaunchKernelGGL(k_glu_planes, dim3((IS + TB - 1) / TB, B), dim3(TB), 0, stream(), gu, dptr_as<float>(r.act), IS, gemma ? 1 : 0);
            split(r.act, IS);
            pending = product(lw.down, bt ? &bl->down : nullptr, D, IS, inv_br);
        }
        pending_g = gemma ? lw.g_post_ff : nullptr;
    }
    if (r.few) {
        add_norm_b(pending_few, pending_g, s->g_final);
        const half_t *W = weight(s->lm_head, bt ? &s->borrowed_lm : nullptr, s->V, D).w16;
        if (!to_host) launch_few_full(a16, inv_ln, W, dptr_as<float>(r.logits), s->V, B, s->V, D);
        for (int i = 0, n = to_host ? batch_parts(s, r) : 0; i < n; i++) {
            const int c0 = batch_part(s, i, n), cols = batch_part(s, i + 1, n) - c0;
            launch_few_full(a16, inv_ln, W + (size_t)c0 * tiled_kb(D) * 64, r.logits_host + c0, s->V, B, cols, D);
            HIP_CHECK(hipEventRecord(r.part_there[i], stream()));
        }
    }
    else {
        add_norm_b(pending, pending_g, s->g_final);
        const SplitPlanes lg = product(s->lm_head, bt ? &s->borrowed_lm : nullptr, s->V, D, inv_ln);
        launch_reduce_planes_split(lg.P, lg.S, lg.plane, lg.N, lg.inv, dptr_as<float>(r.logits), B, lg.N);
    }
    HIP_CHECK(hipGetLastError());
    return false;
}

// argmax of every sequence's logits, computed on the GPU; one wait for all of them
void argmax_batch(InferenceState *s, BatchRun &r, int *out)
{
    float *pv = dptr_as<float>(r.best);                                  // [B][AM_WGS] values, then as many indices
    int *pi = reinterpret_cast<int *>(pv) + (size_t)r.B * AM_WGS;
    hipLaunchKernelGGL(k_argmax_part_batch, dim3(AM_WGS, r.B), dim3(TB), 0, stream(), dptr_as<float>(r.logits), s->V, pv, pi);
    hipLaunchKernelGGL(k_argmax_final_batch, dim3(r.B), dim3(AM_WGS), 0, stream(), pv, pi, r.best_host);
    HIP_CHECK(hipStreamSynchronize(stream()));
    for (int b = 0; b < r.B; b++) out[b] = r.best_host[b];
}

// The state's batch run for B sequences: the one kept from the call before when that had the same B and rank (its buffers
// are strided by B), else a new one in its place.  Caches are not cleared: a step at position pos reads what steps
// 0..pos-1 of the same run wrote.
BatchRun &batch_acquire(InferenceState *s, BatchRun *&slot, int B)
{
    const int R = s->lora.empty() ? 0 : s->R;
    if (slot && slot->B == B && slot->R == R) return *slot;
    metal_flush();
    batch_release(slot);
    slot = new BatchRun{};
    BatchRun &r = *slot;
    if (s->stack) {
        r.B = B;
        r.stk = stack_run_create(s->stack, B);
        r.logits = fbuf((size_t)std::max(B, STACK_WANT) * s->V);
        r.best = metal_buf_create((size_t)B * 2 * AM_WGS * sizeof(int));
        HIP_CHECK(hipHostMalloc((void **)&r.best_host, (size_t)B * sizeof(int), hipHostMallocDefault));
        return r;
    }
    const int D = s->D, qd = s->Hq * s->hd, kd = s->Hkv * s->hd, IS = s->IS, V = s->V;
    r.B = B; r.R = R; r.len = 0;
    r.x = fbuf((size_t)B * D); r.ln = fbuf((size_t)B * D);
    r.qkv = fbuf((size_t)B * (qd + 2 * kd + 2 * R)); r.att = fbuf((size_t)B * qd);
    r.act = fbuf((size_t)B * IS); r.logits = fbuf((size_t)B * V);
    size_t a16_elems = 0, plane_floats = 0;                              // the largest operand and planes of the step's products
    const int shapes[5][2] = {{qd + 2 * kd + (s->borrows_tiles ? 2 * R : 0), D}, {D, qd}, {2 * IS, D}, {D, IS}, {V, D}};
    const int fmt = s->borrows_tiles ? s->borrowed_lm.fmt : 0;
    for (const auto &nk : shapes) {
        a16_elems = std::max(a16_elems, tiled_elems(2 * B, nk[1]));
        for (int ring = 0; ring < 2; ring++)                             // either kernel policy may be switched in later
            for (int wide = 0; wide <= ring; wide++) {                   // (the wide workgroups of the ring kernel may take twice the K chunks)
                const int was = gemm_ring_enabled(), wide_was = gemm_ring_wide_mode();
                set_gemm_ring(ring);
                set_gemm_ring_wide(wide);
                const int nbq = !fmt ? 0 : &nk == &shapes[0] ? tiled_rb(qd + 2 * kd) : tiled_rb(nk[0]);   // the adapter rows are F16 tiles
                plane_floats = std::max(plane_floats, (size_t)plan_gemm(2 * B, nk[0], nk[1], nbq, fmt).S * 2 * B * nk[0]);
                set_gemm_ring(was);
                set_gemm_ring_wide(wide_was);
            }
    }
    r.few = few_rows_fit(s);
    if (r.few) plane_floats = std::max(plane_floats, (size_t)std::max(few_planes(D, qd), few_planes(D, IS)) * B * D);
    r.a16 = metal_buf_create(a16_elems * sizeof(half_t)); r.planes = fbuf(plane_floats);
    r.inv_ln = fbuf((size_t)2 * B); r.inv_br = fbuf((size_t)2 * B);
    r.best = metal_buf_create((size_t)B * 2 * AM_WGS * sizeof(int));
    r.lora_t = R ? fbuf((size_t)B * 2 * R) : nullptr;
    HIP_CHECK(hipHostMalloc((void **)&r.best_host, (size_t)B * sizeof(int), hipHostMallocDefault));
    const size_t cache_bytes = (size_t)s->Hkv * s->max_seq * s->hd * sizeof(float);
    for (int L = 0; L < s->NL; L++) { r.kc.push_back(metal_buf_create(cache_bytes * B)); r.vc.push_back(metal_buf_create(cache_bytes * B)); }
    return r;
}

// pinned memory and events for the run's logits; false: none left
bool batch_logits_room(InferenceState *s, BatchRun &r)
{
    if (!r.logits_host && hipHostMalloc((void **)&r.logits_host, (size_t)r.B * s->V * sizeof(float), hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        r.logits_host = nullptr;
        return false;
    }
    for (hipEvent_t &e : r.part_there) if (!e) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    return true;
}

// The run's logits to the caller's memory, through pinned memory of the run's own.  While the step runs, the pages of `out` are made
// present (new ones cost a fault each, half of what the runtime's copy takes); then a part is copied while the next one arrives.
// formed: the head's kernel has stored them there (forward_token_batch, to_host); else they are copied there first.
// us a step, of which the kernels / with the runtime's copy / in one / two / four parts: 8 sequences of a vocabulary of 32 768 (1 MB,
// nine layers of the 4B shape) 662 / 910 / 750 / 718 / 738, 32 of 16 384 (2 MB) 278 / 405 / 395 / 364 / 368, 20 of 70 000 (5.6 MB,
// nine layers of Gemma3-1B's) 1130 with the runtime's, 850 / 800 / 770; 2 of 9 000 (72 KB) 28 more in four parts than in one.
// Stored by the head's kernel, a copy in pinned memory ahead of that -> so: 8 sequences of 32 768 722 -> 701 us in two parts (716 / 705 / 699 in one / three /
// four), 2 of 9 000 with three layers 239 -> 222 in one (225 in two), 4 of 30 000 402 -> 387, 32 of 16 384 463 -> 457, 20 of 70 000 833 -> 815 in four (853 in one).
void batch_logits_to(InferenceState *s, BatchRun &r, float *out, bool formed)
{
    const size_t V = s->V, bytes = (size_t)r.B * V * sizeof(float);
    auto pages = [&] { for (size_t at = 0; at < bytes; at += 4096) ((volatile char *)out)[at] = 0; };
    if (formed) {
        pages();
        for (int i = 0, n = batch_parts(s, r); i < n; i++) {
            const size_t c0 = batch_part(s, i, n), cols = batch_part(s, i + 1, n) - c0;
            HIP_CHECK(hipEventSynchronize(r.part_there[i]));
            if (cols == V) memcpy(out, r.logits_host, bytes);
            else for (int b = 0; b < r.B; b++) memcpy(out + b * V + c0, r.logits_host + b * V + c0, cols * sizeof(float));
        }
        return;
    }
    if (!batch_logits_room(s, r)) {
        HIP_CHECK(hipMemcpyAsync(out, dptr(r.logits), bytes, hipMemcpyDeviceToHost, stream()));
        HIP_CHECK(hipStreamSynchronize(stream()));
        return;
    }
    const size_t parts = bytes < ((size_t)512 << 10) ? 1 : bytes < ((size_t)4 << 20) ? 2 : 4;
    auto from = [&](size_t i) { return i < parts ? bytes / 64 * i / parts * 64 : bytes; };
    for (size_t i = 0; i < parts; i++) {
        HIP_CHECK(hipMemcpyAsync((char *)r.logits_host + from(i), (const char *)dptr(r.logits) + from(i), from(i + 1) - from(i), hipMemcpyDeviceToHost, stream()));
        HIP_CHECK(hipEventRecord(r.part_there[i], stream()));
    }
    pages();
    for (size_t i = 0; i < parts; i++) {
        HIP_CHECK(hipEventSynchronize(r.part_there[i]));
        memcpy((char *)out + from(i), (const char *)r.logits_host + from(i), from(i + 1) - from(i));
    }
}

void step_on_run(InferenceState *s, int token, int pos)
{
    BatchRun &r = batch_acquire(s, s->single, 1);
    forward_token_batch(s, r, &token, pos);
    r.len = pos + 1;
}
const float *step_logits_on_run(InferenceState *s, int token, int pos)
{
    BatchRun &r = batch_acquire(s, s->single, 1);
    const bool there = forward_token_batch(s, r, &token, pos, s->logits_host);
    r.len = pos + 1;
    if (!there) return logits_on_run(s);
    HIP_CHECK(hipStreamSynchronize(stream()));
    return s->logits_host;
}
// ---- prompts of the models that decode a token at a time, many tokens per step

constexpr int PROMPT_ROWS = 1024;        // tokens of one step
constexpr int PROMPT_WANT = 32;          // rows of logits formed together
constexpr int PROMPT_HEAD_ROWS = 65536;  // rows of the head multiplied at a time

struct PromptRun {
    int cap;                             // rows the buffers are sized for
    MetalBuf *x, *ln, *q, *att, *act, *t, *a16, *inv_ln, *inv_br, *planes, *planes2, *ids, *sel, *sel_logits;
    int *ids_host;                       // [max_seq], a token at its position: portions of one prompt do not overwrite each other
};

void prompt_release(PromptRun *r)
{
    if (!r) return;
    for (MetalBuf *b : {r->x, r->ln, r->q, r->att, r->act, r->t, r->a16, r->inv_ln, r->inv_br, r->planes, r->planes2, r->ids, r->sel, r->sel_logits}) metal_buf_free(b);
    if (r->ids_host) hipHostFree(r->ids_host);
    delete r;
}

size_t free_memory()
{
    size_t f = 0, t = 0;
    HIP_CHECK(hipMemGetInfo(&f, &t));
    return f;
}

// Whether `bytes` are free besides 2 GB for everything allocated later.  The driver clears freed memory before it counts as free
// again, some milliseconds after the call that freed it; settled: a figure that is too low is read until it stands still for 20 ms.
bool memory_for(size_t bytes, bool settled)
{
    bytes += (size_t)2 << 30;
    size_t before = free_memory();
    for (int same = 0, i = 0; settled && before < bytes && same < 4 && i < 100; i++) {
        usleep(5000);
        const size_t now = free_memory();
        same = now == before ? same + 1 : 0;
        before = now;
    }
    return before >= bytes;
}

// What the products of a step of up to `cap` tokens need: planes, and the F16 images of the largest matrix where none is kept
size_t prompt_product_bytes(const InferenceState *s, int cap)
{
    const bool q8 = !s->use_fp16 && !s->borrows_tiles;
    const int qd = s->Hq * s->hd, kd = s->Hkv * s->hd;
    const int shapes[4][2] = {{qd + 2 * kd + (s->borrows_tiles ? 2 * s->R : 0), s->D}, {s->D, qd}, {2 * s->IS, s->D}, {s->D, s->IS}};
    const int head = s->borrows_tiles ? s->V : std::min(PROMPT_HEAD_ROWS, s->V), want = std::min(PROMPT_WANT, cap);
    auto pair_bytes = [](int M, int N, int K) { return pair_plane_floats(plan_short_pair(M, N, K, 0, 0), M, N) * sizeof(float); };
    size_t planes = pair_bytes(want, head, s->D), planes2 = 0, image = tiled_elems(head, s->D) * sizeof(half_t);
    for (const auto &sh : shapes) {
        image = std::max(image, tiled_elems(sh[0], sh[1]) * sizeof(half_t));
        for (int m = 32; m - 32 < cap; m += 32) {
            const int M = std::min(m, cap);
            planes = std::max(planes, pair_bytes(M, sh[0], sh[1]));
            planes2 = std::max(planes2, (size_t)plan_short_sums(M, sh[0], sh[1], 0, 0).planes() * M * sh[0] * sizeof(float));
        }
    }
    return planes + (q8 ? planes2 + 2 * image : image);
}

// The weights' Q8_0 scales are small enough that two F16 images hold d q.  Asked once for what the weights hold (their versions).
bool q8_scales_fit(InferenceState *s)
{
    uint64_t version = 1;                                             // (0: not asked yet)
    for (int L = 0; L < s->NL; L++) {
        const InferenceState::Layer &lw = s->layers[L];
        for (const WMat *w : {&lw.qkv, (const WMat *)lw.o, &lw.gu, (const WMat *)lw.down}) version += w->mbuf->version;
    }
    if (s->q8_fit_version == version) return s->q8_fit;
    MetalBuf *top = metal_buf_create(sizeof(unsigned));
    unsigned bits = 0;
    metal_buf_write(top, 0, &bits, sizeof bits);
    for (int L = 0; L < s->NL; L++) {
        const InferenceState::Layer &lw = s->layers[L];
        for (const WMat *w : {&lw.qkv, (const WMat *)lw.o, &lw.gu, (const WMat *)lw.down}) q8_max_scale(w->mbuf, w->rows, w->cols, dptr_as<unsigned>(top));
    }
    metal_buf_read(top, 0, &bits, sizeof bits);
    metal_buf_free(top);
    float d;
    memcpy(&d, &bits, sizeof d);
    s->q8_fit_version = version;
    return s->q8_fit = d * 128.f < 65504.f;                           // (false for a NaN)
}

// Whether n tokens go many to a step: from five on.  Nine layers of the 4B shape, ms at 5 / 8 / 16 / 32 / 64 tokens: F16 weights
// 0.75 / 0.79 / 0.85 / 1.02 / 1.27, Q8_0 0.78 / 0.81 / 0.86 / 1.03 / 1.98 (1.8 and 2.4 four tokens one by one); 500 tokens take 3.7 instead of
// 460 ms; portions of up to four stay bit for bit what single tokens give.  A state's first prompt
// pays for the buffers and the tiles that are kept besides: at five tokens up to 2 ms more than one by one, once, at sixteen none.
// A state takes its tokens one by one where a Q8_0 weight is beyond what a half holds and, decided once with its first prompt,
// where there is no room for a step's buffers.
bool prompt_takes(InferenceState *s, int n)
{
    if (s->stack || n < 5 || !prompt_attention_supported(s->hd) || s->D > 8192 || s->R > 64 || s->prompt_refused) return false;
    if (!s->use_fp16 && !s->borrows_tiles && !q8_scales_fit(s)) return false;
    if (s->prompt) return true;
    const int qd = s->Hq * s->hd, cap = std::min(PROMPT_ROWS, s->max_seq);
    size_t a16 = 0;
    for (int K : {s->D, qd, s->IS}) a16 = std::max(a16, tiled_elems(2 * pair_row(cap), K));
    const size_t rows = (size_t)cap * (2 * (size_t)s->D + 2 * (size_t)qd + (prompt_glu_supported(s->IS) ? 0 : s->IS) + 4 + 2 * s->R) + s->max_seq + (size_t)PROMPT_WANT * s->D;
    if (!memory_for(rows * sizeof(float) + a16 * sizeof(half_t) + prompt_product_bytes(s, cap), true)) { s->prompt_refused = true; return false; }
    s->prompt = new PromptRun{};
    PromptRun &r = *s->prompt;
    r.cap = cap;
    r.x = fbuf((size_t)cap * s->D); r.ln = fbuf((size_t)cap * s->D);
    r.q = fbuf((size_t)cap * qd); r.att = fbuf((size_t)cap * qd);
    if (!prompt_glu_supported(s->IS)) r.act = fbuf((size_t)cap * s->IS);
    r.a16 = metal_buf_create(a16 * sizeof(half_t));
    r.inv_ln = fbuf((size_t)2 * pair_row(cap)); r.inv_br = fbuf((size_t)2 * pair_row(cap));
    r.ids = metal_buf_create((size_t)s->max_seq * sizeof(int));
    r.sel = fbuf((size_t)PROMPT_WANT * s->D);
    HIP_CHECK(hipHostMalloc((void **)&r.ids_host, (size_t)s->max_seq * sizeof(int), hipHostMallocDefault));
    return true;
}

// Rows row0 .. row0 + rows of a row-major F16 matrix as GEMM tiles (row0 a multiple of 32): a part of its image, which is kept with
// the matrix when there is room for it, or else formed in scratch for this product -- the same tiles, so the same results.
const half_t *prompt_tiles(const WMat *w, int row0, int rows)
{
    const size_t Kb = tiled_kb(w->cols);
    if (w->mbuf->tiled[0].dev || (image_budget() && memory_for(tiled_elems(w->rows, w->cols) * sizeof(half_t), false)))
        return tiled_weight_of(w->mbuf, w->rows, w->cols) + (size_t)(row0 / 32) * Kb * 2048;
    const size_t n = tiled_elems(rows, w->cols);
    half_t *img = (half_t *)scratch(SCR_WF16, n * sizeof(half_t));
    if (rows % 32 || w->cols % 64) launch_fill_f32((float *)img, 0.f, n / 2);         // (the tiling writes no padding)
    launch_tile_f16(dptr_as<half_t>(w->mbuf) + (size_t)row0 * w->cols, rows, w->cols, img, (int)Kb, 0, 0, 0);
    return img;
}

// a buffer of at least n floats (what it held is gone when it grows)
float *at_least(MetalBuf *&b, size_t n)
{
    if (!b || b->size < n * sizeof(float)) { metal_buf_free(b); b = fbuf(n); }       // (the free waits for the stream)
    return dptr_as<float>(b);
}

// the plan of a prompt's product with a matrix [rows, cols]: the state's own (F16 images in any case) or a training state's tiles
ShortPlan prompt_plan(const WeightOp *tiles, int rows, int cols, int M)
{
    return tiles ? plan_short_pair(M, rows, cols, (tiles->fmt == 1 && tiles->nbq < tiled_rb(rows)) ? tiles->nbq : 0, tiles->fmt) : plan_short_pair(M, rows, cols, 0, 0);
}

// planes of (the operand in r.a16, rows split by `inv`, residuals from row p.lo on) x w^T: w the state's own matrix (its tiled F16 image, or for Q8_0 the
// two images of d q and of what rounding that to F16 lost) or a training state's tiles
SplitPlanes prompt_product(InferenceState *s, PromptRun &r, const WMat *w, const WeightOp *tiles, int rows, int cols, const float *inv, int M, const ShortPlan &p, int row0 = 0)
{
    const half_t *a16 = dptr_as<half_t>(r.a16);
    SplitPlanes out{};
    out.inv = inv; out.N = rows; out.lo = p.lo;
    auto pairs = [&](const WeightOp &op) {
        float *P = at_least(r.planes, pair_plane_floats(p, M, rows));
        const PairPlanes q = launch_short_pair(a16, inv, p.big ? f16_image_of(op, rows, cols) : op, P, M, rows, cols, p);
        out.S = q.S; out.plane = q.plane; out.whole = q.whole; out.walk = q.walk;
    };
    if (tiles) pairs(*tiles);
    else if (s->use_fp16) pairs(weight_f16(prompt_tiles(w, row0, rows)));
    else {
        const size_t n = tiled_elems(rows, cols);
        half_t *hi = (half_t *)scratch(SCR_WF16, 2 * n * sizeof(half_t)), *lo = hi + n;
        q8_to_tiled_pair(w->mbuf, rows, cols, hi, lo);
        pairs(weight_f16(hi));
        out.plane2 = (size_t)M * rows;
        const ShortPlan p2 = plan_short_sums(M, rows, cols, 0, 0);
        out.S2 = launch_short_sums(a16, weight_f16(lo), at_least(r.planes2, out.plane2 * p2.planes()), out.plane2, M, rows, cols, p2);
        out.P2 = dptr_as<float>(r.planes2);
    }
    out.P = dptr_as<float>(r.planes);
    return out;
}

// A step of up to FEW_ROWS tokens takes the batch's products (few_rows.h) where the state's widths fit them: at 8 / 32 tokens of nine 4B
// layers 0.79 / 1.02 ms against 0.94 / 1.07 of the short sums (F16), 0.81 / 1.03 against 2.40 / 2.45 with F16 images formed for each product (Q8_0)
bool prompt_few(const InferenceState *s, int M) { return M <= FEW_ROWS && few_rows_fit(s); }

// One step: the M tokens at positions pos .. pos + M - 1, their keys and values into kc and vc (the first sequence's part),
// the final norm's rows into r.ln.  Per layer the launches of forward_token_batch, with the tokens as rows: ten, for a few rows of
// F16 weights eight (of Q8_0 ten: the rows ahead of O and of down are split by launches of their own).
void prompt_step(InferenceState *s, PromptRun &r, std::vector<MetalBuf *> &kc, std::vector<MetalBuf *> &vc, int M, int pos)
{
    const int D = s->D, Hq = s->Hq, Hkv = s->Hkv, hd = s->hd, IS = s->IS, qd = Hq * hd, nqkv = qd + 2 * Hkv * hd;
    const bool gemma = s->model_type == MODEL_GEMMA3, bt = s->borrows_tiles, adapters = !s->lora.empty();
    const int *ids = dptr_as<int>(r.ids) + pos;
    HIP_CHECK(hipMemcpyAsync((void *)ids, r.ids_host + pos, (size_t)M * sizeof(int), hipMemcpyHostToDevice, stream()));
    launch_embed_ids(dptr_as<float>(s->emb), ids, s->emb_scale, dptr_as<float>(r.x), M, D);
    half_t *a16 = dptr_as<half_t>(r.a16);
    float *inv_ln = dptr_as<float>(r.inv_ln), *inv_br = dptr_as<float>(r.inv_br);
    auto norm = [&](const SplitPlanes &br, MetalBuf *g_branch, MetalBuf *g, bool keep, int lo) {
        float *ln = keep ? dptr_as<float>(r.ln) : nullptr;
        const float *gb = g_branch ? dptr_as<float>(g_branch) : nullptr;
        launch_add_norm_split(dptr_as<float>(r.x), br, gb, dptr_as<float>(g), ln, a16, inv_ln, M, lo, D, s->eps);
    };
    const bool few = prompt_few(s, M), q8 = !s->use_fp16 && !bt;
    const int nq_rows = nqkv + (bt && adapters ? 2 * s->R : 0);               // (a training state's fused matrix continues with the rows of A_q and A_v)
    float *P = nullptr, *act = nullptr;
    if (few) {
        P = at_least(r.planes, (size_t)M * std::max(nq_rows, D * (q8 ? std::max(few_chunks(D, qd), few_chunks(D, IS)) : std::max(few_planes(D, qd), few_planes(D, IS)))));
        act = at_least(r.act, (size_t)std::min(FEW_ROWS, r.cap) * IS);
    }
    auto few_norm = [&](const FewPlanes &br, MetalBuf *g_branch, MetalBuf *g, bool keep) {
        launch_few_norm(dptr_as<float>(r.x), br, g_branch ? dptr_as<float>(g_branch) : nullptr, dptr_as<float>(g), keep ? dptr_as<float>(r.ln) : nullptr, a16, inv_ln, M, D, s->eps);
    };
    auto tiles = [&](const WMat *w, const WeightOp *op, int rows) { return op ? op->w16 : prompt_tiles(w, 0, rows); };
    auto few_branch = [&](const WMat *w, const WeightOp *op, const float *in, int K) {       // [M, D] of the rows `in`
        if (!q8) return launch_few_split(in, tiles(w, op, D), P, M, D, K);
        launch_rows_to_f16_split(in, a16, inv_br, M, K);
        return launch_few_full_q8(a16, inv_br, few_q8_of(w->mbuf, D, K), P, D, M, D, K, few_chunks(D, K));
    };
    SplitPlanes pending{};
    FewPlanes pending_few{};
    MetalBuf *pending_g = nullptr;
    for (int L = 0; L < s->NL; L++) {
        const InferenceState::Layer &lw = s->layers[L];
        const BorrowedLayer *bl = bt ? &s->borrowed[L] : nullptr;
        PromptHeads h{};
        if (few) {
            few_norm(pending_few, pending_g, lw.g_in, adapters && !bt);
            if (q8) launch_few_full_q8(a16, inv_ln, few_q8_of(lw.qkv.mbuf, nq_rows, D), P, nq_rows, M, nq_rows, D);
            else launch_few_full(a16, inv_ln, tiles(&lw.qkv, bt ? &bl->qkv : nullptr, nq_rows), P, nq_rows, M, nq_rows, D);
            h.qkv.P = P; h.qkv.S = 1; h.qkv.N = nq_rows; h.qkv.whole = true;
        } else {
            const ShortPlan p = prompt_plan(bt ? &bl->qkv : nullptr, nq_rows, D, M);
            norm(pending, pending_g, lw.g_in, adapters && !bt, p.lo);
            h.qkv = prompt_product(s, r, &lw.qkv, bt ? &bl->qkv : nullptr, nq_rows, D, inv_ln, M, p);
        }
        h.g_q = lw.g_q ? dptr_as<float>(lw.g_q) : nullptr; h.g_k = lw.g_k ? dptr_as<float>(lw.g_k) : nullptr;
        h.rope = dptr_as<float2>(s->rope_tabs) + ((size_t)s->theta_slot[L] * s->max_seq + pos) * (hd / 2);
        h.q = dptr_as<float>(r.q); h.kc = dptr_as<float>(kc[L]); h.vc = dptr_as<float>(vc[L]);
        h.M = M; h.Hq = Hq; h.Hkv = Hkv; h.hd = hd; h.pos = pos; h.max_seq = s->max_seq; h.eps = s->eps;
        if (adapters) {
            const InferenceState::Lora &lr = s->lora[L];
            h.R = s->R; h.sc = s->scaling; h.Bq = dptr_as<float>(lr.Bq); h.Bv = dptr_as<float>(lr.Bv);
            if (!bt) {
                float *t = at_least(r.t, (size_t)r.cap * 2 * s->R);
                hipLaunchKernelGGL(k_lora_down, dim3(2 * s->R, M), dim3(64), 0, stream(), dptr_as<float>(r.ln), dptr_as<float>(lr.Aq), dptr_as<float>(lr.Av), t, s->R, D);
                h.t = t;
            }
        }
        launch_prompt_heads(h);
        launch_prompt_attention(h.q, h.kc, h.vc, dptr_as<float>(r.att), M, pos, Hq, Hkv, hd, s->max_seq);
        mark_written(kc[L]); mark_written(vc[L]);
        if (few) {
            few_norm(few_branch(lw.o, bt ? &bl->o : nullptr, dptr_as<float>(r.att), qd), gemma ? lw.g_post_attn : nullptr, gemma ? lw.g_pre_ff : lw.g_post_attn, false);
            if (q8) launch_few_glu_q8(a16, inv_ln, few_q8_of(lw.gu.mbuf, 2 * IS, D), act, M, IS, D, gemma ? 1 : 0);
            else launch_few_glu(a16, inv_ln, tiles(&lw.gu, bt ? &bl->gu : nullptr, 2 * IS), act, M, IS, D, gemma ? 1 : 0);
            pending_few = few_branch(lw.down, bt ? &bl->down : nullptr, act, IS);
            pending_g = gemma ? lw.g_post_ff : nullptr;
            continue;
        }
        const ShortPlan po = prompt_plan(bt ? &bl->o : nullptr, D, qd, M), pgu = prompt_plan(bt ? &bl->gu : nullptr, 2 * IS, D, M),
                        pd = prompt_plan(bt ? &bl->down : nullptr, D, IS, M);
        launch_rows_to_f16_split(dptr_as<float>(r.att), a16, inv_br, M, qd, po.lo);
        const SplitPlanes o = prompt_product(s, r, lw.o, bt ? &bl->o : nullptr, D, qd, inv_br, M, po);
        norm(o, gemma ? lw.g_post_attn : nullptr, gemma ? lw.g_pre_ff : lw.g_post_attn, false, pgu.lo);
        const SplitPlanes gu = prompt_product(s, r, &lw.gu, bt ? &bl->gu : nullptr, 2 * IS, D, inv_ln, M, pgu);
        if (prompt_glu_supported(IS)) launch_prompt_glu(gu, a16, inv_br, M, pd.lo, IS, gemma ? 1 : 0);
        else {
            hipLaunchKernelGGL(k_glu_planes, dim3((IS + TB - 1) / TB, M), dim3(TB), 0, stream(), gu, dptr_as<float>(r.act), IS, gemma ? 1 : 0);
            launch_rows_to_f16_split(dptr_as<float>(r.act), a16, inv_br, M, IS, pd.lo);
        }
        pending = prompt_product(s, r, lw.down, bt ? &bl->down : nullptr, D, IS, inv_br, M, pd);
        pending_g = gemma ? lw.g_post_ff : nullptr;
    }
    if (few) few_norm(pending_few, pending_g, s->g_final, true);
    else norm(pending, pending_g, s->g_final, true, M);
    HIP_CHECK(hipGetLastError());
}

// logits of rows m[0 .. count) of the step, count <= PROMPT_WANT, to out [count][V]: one by one through the matrix-vector
// kernel while that reads the head a few times at most, else (and always on a training state's tiles) as one product
void prompt_logits(InferenceState *s, PromptRun &r, const int *m, int count, float *out)
{
    const int D = s->D;
    auto row = [&](int i, float *dst) {
        HIP_CHECK(hipMemcpyAsync(dst, dptr_as<float>(r.ln) + (size_t)m[i] * D, (size_t)D * 4, hipMemcpyDeviceToDevice, stream()));
    };
    const bool one_by_one = !s->borrows_tiles && (!s->use_fp16 || count < 4);
    if (one_by_one) {
        for (int i = 0; i < count; i++) {
            row(i, dptr_as<float>(s->ln));
            mark_written(s->ln);
            matvec(s, s->lm_head, s->ln, s->logits);
            if (out != dptr_as<float>(s->logits))
                HIP_CHECK(hipMemcpyAsync(out + (size_t)i * s->V, dptr(s->logits), (size_t)s->V * 4, hipMemcpyDeviceToDevice, stream()));
        }
        return;
    }
    for (int i = 0; i < count; i++) row(i, dptr_as<float>(r.sel) + (size_t)i * D);
    const WeightOp *tiles = s->borrows_tiles ? &s->borrowed_lm : nullptr;
    for (int n0 = 0, n, lo = 0; n0 < s->V; n0 += n) {      // (own weights: in parts, for which there is room in scratch if not for the whole head's image)
        n = s->borrows_tiles ? s->V : std::min(PROMPT_HEAD_ROWS, s->V - n0);
        const ShortPlan p = prompt_plan(tiles, n, D, count);
        if (p.lo != lo) launch_rows_to_f16_split(dptr_as<float>(r.sel), dptr_as<half_t>(r.a16), dptr_as<float>(r.inv_br), count, D, lo = p.lo);
        const SplitPlanes lg = prompt_product(s, r, s->lm_head, tiles, n, D, dptr_as<float>(r.inv_br), count, p, n0);
        launch_planes_to_rows(lg, out + n0, count, n, s->V);
    }
}

// n tokens from position pos on, in portions of equal size; after each, f(first token of the portion, its length)
void prompt_portions(InferenceState *s, const int *tokens, int n, int pos, std::vector<MetalBuf *> &kc, std::vector<MetalBuf *> &vc,
                     const std::function<void(int, int)> &f)
{
    PromptRun &r = *s->prompt;
    // (Q8_0: two short steps take less time than one whose products form F16 images of their weights -- 1.98 against 2.71 ms for 64 tokens
    // of nine 4B layers -- three do not)
    const bool q8 = !s->use_fp16 && !s->borrows_tiles;
    const int cap = q8 && n <= 2 * FEW_ROWS && few_rows_fit(s) ? std::min(FEW_ROWS, r.cap) : r.cap;
    const int portions = (n + cap - 1) / cap, each = (n + portions - 1) / portions;
    for (int i = 0; i < n; i++) r.ids_host[pos + i] = tokens[i];
    for (int at = 0; at < n; at += each) {
        const int M = std::min(each, n - at);
        prompt_step(s, r, kc, vc, M, pos + at);
        f(at, M);
    }
}

// a whole prompt from position 0 on; the last token's logits to `logits`
void prompt_rows_all(InferenceState *s, const uint32_t *tokens, int n, std::vector<MetalBuf *> &kc, std::vector<MetalBuf *> &vc, MetalBuf *logits)
{
    prompt_portions(s, (const int *)tokens, n, 0, kc, vc, [&](int at, int M) {
        const int last = M - 1;
        if (at + M == n) prompt_logits(s, *s->prompt, &last, 1, dptr_as<float>(logits));
    });
}

// the same on the sequence that the state itself holds
void prompt_fill(InferenceState *s, const uint32_t *tokens, int n)
{
    if (!s->borrows_tiles) { prompt_rows_all(s, tokens, n, s->kc, s->vc, s->logits); return; }
    BatchRun &r = batch_acquire(s, s->single, 1);
    prompt_rows_all(s, tokens, n, r.kc, r.vc, r.logits);
    r.len = n;
}

// k rows of logits to the caller's memory.  A single one comes through the state's pinned memory (there: the step writes it there itself); while
// the step runs, the pages of `out` are made present.  Against the runtime's copy to the caller's memory: prompts of 5 to 100 tokens of four 4B
// layers 340 -> 331 to 664 -> 654 us (32 KB), of Gemma3-1B with its vocabulary of 262 144 385 -> 367 to 624 -> 617; a further token of Paposun 1k 155 -> 126.
void rows_to_caller(InferenceState *s, const float *rows, int k, bool there, float *out)
{
    const size_t bytes = (size_t)k * s->V * sizeof(float);
    if (k > 1) {
        HIP_CHECK(hipMemcpyAsync(out, rows, bytes, hipMemcpyDeviceToHost, stream()));
        HIP_CHECK(hipStreamSynchronize(stream()));
        return;
    }
    if (!there) HIP_CHECK(hipMemcpyAsync(s->logits_host, rows, bytes, hipMemcpyDeviceToHost, stream()));
    for (size_t at = 0; at < bytes; at += 4096) ((volatile char *)out)[at] = 0;
    HIP_CHECK(hipStreamSynchronize(stream()));
    memcpy(out, s->logits_host, bytes);
}

int prompt_forward(InferenceState *s, const int *tokens, int n, const int *want, int n_want, float *logits)
{
    BatchRun *run = s->borrows_tiles ? &batch_acquire(s, s->single, 1) : nullptr;
    std::vector<MetalBuf *> &kc = run ? run->kc : s->kc, &vc = run ? run->vc : s->vc;
    MetalBuf *row = run ? run->logits : s->logits;
    int w = 0;
    prompt_portions(s, tokens, n, s->cur_len, kc, vc, [&](int at, int M) {
        while (w < n_want && want[w] < at + M) {
            int m[PROMPT_WANT], k = 0;
            while (w + k < n_want && k < PROMPT_WANT && want[w + k] < at + M) { m[k] = want[w + k] - at; k++; }
            float *out = k == 1 ? dptr_as<float>(row) : at_least(s->prompt->sel_logits, (size_t)PROMPT_WANT * s->V);
            prompt_logits(s, *s->prompt, m, k, out);
            rows_to_caller(s, out, k, false, logits + (size_t)w * s->V);
            w += k;
        }
    });
    s->cur_len += n;
    if (run) run->len = s->cur_len;
    HIP_CHECK(hipStreamSynchronize(stream()));
    return 0;
}

// A prompt, or a portion of one, for every sequence of the run, in as few steps as its scratch allows; the logits of the
// last token stay in the run.
void prefill_rows(InferenceState *s, BatchRun &r, const uint32_t *tokens, int n, int pos)
{
    const int portion = stack_portion(r.stk);
    std::vector<int> ids;
    for (int at = 0; at < n; at += portion) {
        const int T = std::min(portion, n - at);
        ids.resize((size_t)r.B * T);
        for (int b = 0; b < r.B; b++) for (int t = 0; t < T; t++) ids[(size_t)b * T + t] = (int)tokens[at + t];
        stack_forward(s->stack, r.stk, ids.data(), T, pos + at);
    }
    stack_logits(s->stack, r.stk, nullptr, r.B, dptr_as<float>(r.logits));
    r.len = pos + n;
}
void prefill_on_run(InferenceState *s, const uint32_t *tokens, int n, int pos) { prefill_rows(s, batch_acquire(s, s->single, 1), tokens, n, pos); }
int forward_rows(InferenceState *s, const int *tokens, int n, const int *want, int n_want, float *logits)
{
    BatchRun &r = batch_acquire(s, s->single, 1);
    const int portion = stack_portion(r.stk);
    int w = 0;
    for (int at = 0; at < n; at += portion) {
        const int T = std::min(portion, n - at);
        stack_forward(s->stack, r.stk, tokens + at, T, s->cur_len);
        s->cur_len += T;
        r.len = s->cur_len;
        while (w < n_want && want[w] < at + T) {                          // the wanted rows of this step, STACK_WANT at a time
            int rows[STACK_WANT], k = 0;
            while (w + k < n_want && k < STACK_WANT && want[w + k] < at + T) { rows[k] = want[w + k] - at; k++; }
            const bool there = stack_logits(s->stack, r.stk, rows, k, dptr_as<float>(r.logits), s->logits_host);
            rows_to_caller(s, dptr_as<float>(r.logits), k, there, logits + (size_t)w * s->V);
            w += k;
        }
    }
    HIP_CHECK(hipStreamSynchronize(stream()));
    return 0;
}
const float *logits_on_run(InferenceState *s)
{
    HIP_CHECK(hipMemcpyAsync(s->logits_host, dptr(s->single->logits), (size_t)s->V * 4, hipMemcpyDeviceToHost, stream()));
    HIP_CHECK(hipStreamSynchronize(stream()));
    return s->logits_host;
}
int argmax_on_run(InferenceState *s)
{
    int best = 0;
    argmax_batch(s, *s->single, &best);
    return best;
}

bool batch_args_ok(InferenceState *s, int B)
{
    if (s->stack) return B >= 1 && B <= 32;
    if (!s->use_fp16 && !s->borrows_tiles) { fprintf(stderr, "[BatchGen] F16 weights only\n"); return false; }
    if (B < 1 || B > 32) return false;
    if (s->D > 8192) { fprintf(stderr, "[BatchGen] hidden size %d not supported (<= 8192)\n", s->D); return false; }
    return true;
}

}  // namespace

// qwen3_generate_fast_batch, src/nn/fast_inference.c:895-1000, on a state's weights: batch_size copies of one prompt are
// prefilled and then decoded greedily in lock step, so that a step reads every weight once for all of them.  The loop
// ends when every sequence has emitted an end token (the state's EOS ids, or token 0 as in the reference, :944-947),
// after max_gen_len tokens or when the cache is full; sequences that have ended keep being stepped and written, as in
// the reference.  output_tokens: [batch_size][max_gen_len].  Returns the tokens written per sequence, 0 when the
// arguments do not fit (F16 weights only, 1 <= batch_size <= 32, prompt within the cache).
int inference_generate_batch(InferenceState *s, const uint32_t *prompt_tokens, int prompt_len, uint32_t *output_tokens,
                             int max_gen_len, int batch_size)
{
    const int B = batch_size;
    if (!batch_args_ok(s, B) || prompt_len <= 0 || max_gen_len <= 0 || prompt_len > s->max_seq) return 0;
    for (int i = 0; i < prompt_len; i++)
        if (prompt_tokens[i] >= (uint32_t)s->V) { fprintf(stderr, "[BatchGen] token %u outside the vocabulary (%d)\n", prompt_tokens[i], s->V); return 0; }
    BatchRun &r = batch_acquire(s, s->batch, B);
    int tokens[32], next[32], active[32];
    if (s->stack) prefill_rows(s, r, prompt_tokens, prompt_len, 0);
    else if (prompt_takes(s, prompt_len)) {                                   // once, into the first sequence's caches, and copied to the others
        prompt_rows_all(s, prompt_tokens, prompt_len, r.kc, r.vc, r.logits);
        for (int L = 0; L < s->NL; L++)
            launch_copy_caches(dptr_as<float>(r.kc[L]), dptr_as<float>(r.vc[L]), B, s->Hkv, s->max_seq, s->hd, prompt_len);
        for (int b = 1; b < B; b++)
            HIP_CHECK(hipMemcpyAsync(dptr_as<float>(r.logits) + (size_t)b * s->V, dptr(r.logits), (size_t)s->V * 4, hipMemcpyDeviceToDevice, stream()));
    }
    else for (int i = 0; i < prompt_len; i++) {                               // prefill: the same token for every sequence (:910-916)
        for (int b = 0; b < B; b++) tokens[b] = (int)prompt_tokens[i];
        forward_token_batch(s, r, tokens, i);
    }
    int cur_len = prompt_len;
    argmax_batch(s, r, next);
    for (int b = 0; b < B; b++) { output_tokens[(size_t)b * max_gen_len] = (uint32_t)next[b]; active[b] = 1; }
    int n_gen = 1;
    for (int gen = 1; gen < max_gen_len && cur_len < s->max_seq; gen++) {
        int any_active = 0;
        for (int b = 0; b < B; b++) {
            bool ended = next[b] == 0 && !s->stack;                      // (token 0 is the reference's rule for its models)
            for (int e = 0; e < s->n_eos; e++) ended |= next[b] == s->eos[e];
            if (active[b] && ended) active[b] = 0;
            any_active |= active[b];
        }
        if (!any_active) break;
        forward_token_batch(s, r, next, cur_len);
        cur_len++;
        argmax_batch(s, r, next);
        for (int b = 0; b < B; b++) output_tokens[(size_t)b * max_gen_len + n_gen] = (uint32_t)next[b];
        n_gen++;
    }
    r.len = cur_len;
    return n_gen;
}

// One lock-step step with a token of its own for every sequence (what forward_token_batch, src/nn/fast_inference.c:808-893,
// is given by a sampling caller): tokens[b] enters sequence b at position pos, logits [batch_size][vocab] come back when
// `logits` is not NULL.  Positions run 0, 1, 2, ... on the state's kept batch caches; pos = 0 starts new sequences, any
// other pos must be the one after the step before (of this call or of inference_generate_batch with the same batch_size).
// Returns 0, or -1 when the arguments do not fit.
int inference_step_batch(InferenceState *s, const int *tokens, int batch_size, int pos, float *logits)
{
    const int B = batch_size;
    if (!s || !tokens || !batch_args_ok(s, B) || pos < 0 || pos >= s->max_seq) return -1;
    for (int b = 0; b < B; b++)
        if (tokens[b] < 0 || tokens[b] >= s->V) { fprintf(stderr, "[BatchGen] token %d outside the vocabulary (%d)\n", tokens[b], s->V); return -1; }
    BatchRun &r = batch_acquire(s, s->batch, B);
    if (pos != 0 && pos != r.len) { fprintf(stderr, "[BatchGen] step at position %d, but the batch's caches hold %d\n", pos, r.len); return -1; }
    const bool formed = logits && r.few && batch_logits_room(s, r);
    forward_token_batch(s, r, tokens, pos, nullptr, formed);
    r.len = pos + 1;
    if (logits) batch_logits_to(s, r, logits, formed);
    return 0;
}

void inference_state_set_eos(InferenceState *s, const int *eos_tokens, int n_eos)
{
    if (n_eos <= 0 || !eos_tokens) { default_eos(s); return; }
    s->n_eos = n_eos > 4 ? 4 : n_eos;
    for (int i = 0; i < s->n_eos; i++) s->eos[i] = eos_tokens[i];
}

// src/nn/fast_inference.c:13-49, 324-342: config.json inside model_path when that is a directory, else next to it
void inference_state_load_eos(InferenceState *s, const char *model_path)
{
    const std::string path = config_path_of(model_path);
    int ids[4], n = 0;
    std::ifstream f(path);
    if (f) {
        std::stringstream ss;
        ss << f.rdbuf();
        n = eos_ids_in(ss.str(), ids, 4);
    }
    inference_state_set_eos(s, ids, n);
    fprintf(stderr, "[FastGen] EOS tokens (%d):", s->n_eos);
    for (int i = 0; i < s->n_eos; i++) fprintf(stderr, " %d", s->eos[i]);
    fprintf(stderr, "\n");
}

}  // extern "C"
