// Kernels of a prompt's step: many tokens of one sequence at once (prompt.h).  Measured for 500 tokens, 32 / 8 heads of 128, width
// 2560, FFN 9728, F16: nine layers 3.3 to 3.5 ms by box; in a trace of 3.56 the products 2.66 and attention 0.26; one token at a time, as these prompts ran before,
// 460 ms.
#include "backend.h"
#include "bf16pair.h"
#include "lds_copy.h"
#include "prompt.h"
#include <algorithm>
#include <stdio.h>

using namespace lmhip;

namespace {

constexpr int TB = 256;

__global__ __launch_bounds__(TB) void k_embed_ids(const float *__restrict__ emb, const int *__restrict__ ids, float scale, float *__restrict__ x, int D)
{
    const int i = blockIdx.x * TB + threadIdx.x, m = blockIdx.y;
    if (i < D) x[(size_t)m * D + i] = emb[(size_t)ids[m] * D + i] * scale;
}

__global__ __launch_bounds__(TB) void k_copy_caches(float *__restrict__ k, float *__restrict__ v, size_t seq_step, size_t head_step, int n)
{
    const int i = blockIdx.x * TB + threadIdx.x;
    if (i >= n) return;
    float *c = blockIdx.z & 1 ? v : k;
    const size_t at = (size_t)blockIdx.y * head_step + i;
    c[(size_t)(1 + (blockIdx.z >> 1)) * seq_step + at] = c[at];
}

// One wave per (token, head); lane i owns the rotary pairs i and i + 64 of up to 256 values, as finish_head of the decoding
// kernel does, with the same expressions.  Reads the product's planes (2 S loads per value) and writes each value once:
// bound by those bytes, 25 MB at 500 tokens of the 4B shape: 12.8 us.
__global__ __launch_bounds__(TB) void k_prompt_heads(PromptHeads a)
{
    const int lane = threadIdx.x & 63, slot = blockIdx.x * 4 + (threadIdx.x >> 6), m = blockIdx.y;
    if (slot >= a.Hq + 2 * a.Hkv) return;
    const int kind = slot < a.Hq ? 0 : slot < a.Hq + a.Hkv ? 1 : 2;         // q, k, v
    const int h = kind == 0 ? slot : kind == 1 ? slot - a.Hq : slot - a.Hq - a.Hkv;
    const int hd = a.hd, half = hd / 2, nqkv = (a.Hq + 2 * a.Hkv) * hd;
    float t = 0.f;                                                          // lane r < R: this token's A x, row r
    const bool adapters = a.R > 0 && kind != 1;
    if (adapters && lane < a.R) {
        const int r = (kind == 0 ? 0 : a.R) + lane;
        t = a.t ? a.t[(size_t)m * 2 * a.R + r] : planes_at(a.qkv, m, nqkv + r);
    }
    float x0[2] = {0.f, 0.f}, x1[2] = {0.f, 0.f};
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int i = lane + 64 * u;
        if (i < half) { x0[u] = planes_at(a.qkv, m, slot * hd + i); x1[u] = planes_at(a.qkv, m, slot * hd + i + half); }
        if (adapters) {
            const float *B = (kind == 0 ? a.Bq : a.Bv) + (size_t)h * hd * a.R;
            float d0 = 0.f, d1 = 0.f;
            for (int r = 0; r < a.R; r++) {
                const float tr = __shfl(t, r, 64);
                if (i < half) { d0 = fmaf(B[(size_t)i * a.R + r], tr, d0); d1 = fmaf(B[(size_t)(i + half) * a.R + r], tr, d1); }
            }
            if (i < half) { x0[u] = fmaf(a.sc, d0, x0[u]); x1[u] = fmaf(a.sc, d1, x1[u]); }
        }
        ss += x0[u] * x0[u] + x1[u] * x1[u];
    }
    if (kind != 2) {
        const float *g = kind == 0 ? a.g_q : a.g_k;
        const float inv = g ? rsqrtf(wave_sum(ss) / (float)hd + a.eps) : 1.f;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int i = lane + 64 * u;
            if (i >= half) continue;
            if (g) { x0[u] *= inv * g[i]; x1[u] *= inv * g[i + half]; }
            const float2 c = a.rope[(size_t)m * half + i];
            const float r0 = x0[u] * c.x - x1[u] * c.y, r1 = x0[u] * c.y + x1[u] * c.x;
            x0[u] = r0; x1[u] = r1;
        }
    }
    float *dst = kind == 0 ? a.q + ((size_t)m * a.Hq + h) * hd : (kind == 1 ? a.kc : a.vc) + ((size_t)h * a.max_seq + a.pos + m) * hd;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int i = lane + 64 * u;
        if (i < half) { dst[i] = x0[u]; dst[i + half] = x1[u]; }
    }
}

// One (token, query head) by one wave, key by key, reading only what it sees: for rows beside which a later key's value is not
// finite (below), where the tiles' zero probabilities would turn into NaN.
template <int HD>
__device__ __attribute__((noinline)) void attend_plain(const float *Q, const float *Kh, const float *Vh, float *out, int m, int head, int qpos, int Hq, float scale)
{
    constexpr int U = (HD + 63) / 64;
    const int lane = threadIdx.x & 63;
    const float *q = Q + ((size_t)m * Hq + head) * HD;
    float o[U] = {}, mx = -3.0e38f, l = 0.f;
    for (int j = 0; j <= qpos; j++) {
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < U; u++) if (lane + 64 * u < HD) s = fmaf(q[lane + 64 * u], Kh[(size_t)j * HD + lane + 64 * u], s);
        s = wave_sum(s) * scale;
        const float now = fmaxf(mx, s), keep = expf(mx - now), p = expf(s - now);
        mx = now;
        l = fmaf(l, keep, p);
#pragma unroll
        for (int u = 0; u < U; u++) if (lane + 64 * u < HD) o[u] = fmaf(o[u], keep, p * Vh[(size_t)j * HD + lane + 64 * u]);
    }
#pragma unroll
    for (int u = 0; u < U; u++) if (lane + 64 * u < HD) out[((size_t)m * Hq + head) * HD + lane + 64 * u] = o[u] / l;
}

// The four waves' shares of 32 rows become one: lane's row, output columns by register (BY4: 4 i + c of 128 for accumulator c, its row i)
template <int HD, bool BY4>
__device__ __forceinline__ void finish_rows(float16v (&O)[HD / 32], float mx, float l, float (*part)[HD / 32 * 16][64], float (*st)[2][64], float *op, bool write)
{
    constexpr int CB = HD / 32;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5;
    l = xor_add<32>(l);
    st[wave][0][lane] = mx; st[wave][1][lane] = l;
    __syncthreads();
    float all = st[0][0][lane];
#pragma unroll
    for (int w = 1; w < 4; w++) all = fmaxf(all, st[w][0][lane]);
    float den = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) den = fmaf(st[w][1][lane], expf(st[w][0][lane] - all), den);
    const float f = expf(mx - all);
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
        for (int j = 0; j < 16; j++) O[c][j] *= f;
    auto put = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < CB; c++)
#pragma unroll
            for (int j = 0; j < 16; j++) part[slot][c * 16 + j][lane] = O[c][j];
    };
    auto add = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < CB; c++)
#pragma unroll
            for (int j = 0; j < 16; j++) O[c][j] += part[slot][c * 16 + j][lane];
    };
    if (wave >= 2) put(wave - 2);
    __syncthreads();
    if (wave < 2) add(wave);
    __syncthreads();
    if (wave == 1) put(0);
    __syncthreads();
    if (wave != 0 || !write) return;
    add(0);
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            float4v o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = (BY4 ? O[c / 4 * 4 + e][4 * b + c % 4] : O[c][4 * b + e]) / den;
            *reinterpret_cast<float4v *>(op + (BY4 ? 128 * (c / 4) + 4 * (8 * b + 4 * half + c % 4) : 32 * c + 8 * b + 4 * half)) = o;
        }
}

// Attention in fp32 on the matrix cores (v_mfma_f32_32x32x2_f32), heads of 32 and 64.
// A workgroup serves 32 (token, query head) pairs of one key head -- row r of the key head is token r / G, head r % G of its
// group, so a tile spans few positions whatever G is -- and its four waves take the key tiles in turn, 32 keys each, with a
// running softmax of their own that the workgroup merges at the end: the chain of a wave is a quarter of the keys.  Scores are
// formed transposed (keys x rows): a row is a lane, and the accumulator that holds a row's probabilities is, register by
// register, the operand of the product with the values (the keys of a step are those the two lane halves hold), so nothing
// passes through LDS until the merge.
// An accumulator is rounded at every instruction, so no sum stays in one for long: a score is added up from parts of eight
// instructions (sixteen columns), a value sum from parts of four (eight keys), each part added while the next is multiplied.
// Per tile HD matrix instructions of 64 cycles, half for the scores: bound by them and by what stands between them (32-bit matrix and
// vector instructions of a SIMD's two waves do not run beside each other).
template <int HD>
__global__ __launch_bounds__(TB, 2) void k_prompt_attn(const float *__restrict__ Q, const float *__restrict__ Kc, const float *__restrict__ Vc,
                                                                       float *__restrict__ out, int M, int pos, int Hq, int G, int max_seq, float scale)
{
    constexpr int CB = HD / 32, HH = HD / 2;
    __shared__ float part[2][CB * 16][64];
    __shared__ float st[4][2][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5, col = lane & 31;
    const int kvh = blockIdx.y, rows = M * G, row0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * 32;      // the longest first
    const int r = min(row0 + col, rows - 1), m = r / G, head = kvh * G + r % G, qpos = pos + m;
    const int last = pos + min(row0 + 31, rows - 1) / G, tiles = last / 32 + 1;
    const float *Kh = Kc + (size_t)kvh * max_seq * HD, *Vh = Vc + (size_t)kvh * max_seq * HD;

    float4v q[HH / 4];                                     // columns half * HH .. of the lane's row
    const float *qp = Q + ((size_t)m * Hq + head) * HD + half * HH;
#pragma unroll
    for (int i = 0; i < HH / 4; i++) q[i] = *reinterpret_cast<const float4v *>(qp + 4 * i);

    float16v O[CB] = {};
    float mx = -3.0e38f, l = 0.f, bad = 0.f;
    for (int t = wave; t < tiles; t += 4) {
        // (a tile's part of every address is scalar, a lane's 32 bits)
        const float *Kt = Kh + (size_t)t * 32 * HD, *Vt = Vh + (size_t)t * 32 * HD;
        const uint32_t left = (uint32_t)(last - t * 32), k0 = min((uint32_t)col, left) * HD + half * HH;
        float16v S = {}, T[2];
        float4v k[2][4];                                   // sixteen columns while the sixteen before are multiplied
        auto keys = [&](int i) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 4; e++) k[i & 1][e] = *reinterpret_cast<const float4v *>(Kt + (k0 + 16 * i + 4 * e));
        };
        keys(0);
#pragma unroll
        for (int i = 0; i < HH / 16; i++) {
            if (i + 1 < HH / 16) keys(i + 1);
            __builtin_amdgcn_sched_barrier(0);             // (all of a tile's loads together spill)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                float16v &t8 = T[u];
                t8 = float16v{};
#pragma unroll
                for (int e = 0; e < 8; e++) t8 = __builtin_amdgcn_mfma_f32_32x32x2f32(k[i & 1][2 * u + (e >> 2)][e & 3], q[4 * i + 2 * u + (e >> 2)][e & 3], t8, 0, 0, 0);
                if (i + u > 0) S += T[u ^ 1];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        S += T[1];
        // value rows of four of the sixteen keys that the lane's half holds, keys 8 b + 4 half .. + 3 of the tile; the next
        // four are requested while these are multiplied
        float v[2][4][CB];
        auto values = [&](int b) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t v0 = min((uint32_t)(8 * b + 4 * half + e), left) * HD + col;
#pragma unroll
                for (int c = 0; c < CB; c++) v[b & 1][e][c] = Vt[v0 + 32 * c];
            }
        };
        values(0);
        float top = -3.0e38f;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const bool seen = t * 32 + 8 * (j >> 2) + 4 * half + (j & 3) <= qpos;
            S[j] = seen ? S[j] * scale : -INFINITY;
            if (seen) top = fmaxf(top, S[j]);
        }
        top = xor_max<32>(top);
        const float now = fmaxf(mx, top), keep = expf(mx - now);
        mx = now;
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < 16; j++) { S[j] = expf(S[j] - now); sum += S[j]; }       // (a key that is not seen: 0)
        l = fmaf(l, keep, sum);
        auto flush = [&](int n) __attribute__((always_inline)) {
            const int c = n % CB;
#pragma unroll
            for (int j = 0; j < 16; j++) O[c][j] = n < CB ? fmaf(O[c][j], keep, T[n & 1][j]) : O[c][j] + T[n & 1][j];
        };
#pragma unroll
        for (int b = 0; b < 4; b++) {
            if (b < 3) values(b + 1);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int c = 0; c < CB; c++) bad = fmaf(v[b & 1][e][c], 0.f, bad);     // (a branch for tiles that all rows see whole lets the sums below pile up behind it)
#pragma unroll
            for (int c = 0; c < CB; c++) {
                float16v &t4 = T[(b * CB + c) & 1];
                t4 = float16v{};
#pragma unroll
                for (int e = 0; e < 4; e++) t4 = __builtin_amdgcn_mfma_f32_32x32x2f32(v[b & 1][e][c], S[4 * b + e], t4, 0, 0, 0);
                if (b + c > 0) flush(b * CB + c - 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        flush(4 * CB - 1);
    }
    if (__syncthreads_or(bad != 0.f)) {                    // a probability of zero has met an infinity or NaN
        for (int i = wave; i < 32 && row0 + i < rows; i += 4) attend_plain<HD>(Q, Kh, Vh, out, (row0 + i) / G, kvh * G + (row0 + i) % G, pos + (row0 + i) / G, Hq, scale);
        return;
    }
    finish_rows<HD, false>(O, mx, l, part, st, out + ((size_t)m * Hq + head) * HD, row0 + col < rows);
}

// Eight values as three bf16 operands each, x = hi + mid + lo exactly (8 mantissa bits a piece, each rounded to nearest; not finite:
// mid and lo are NaN).  (Cut off instead of rounded, the parts have one sign and so has what the products below leave out: 2 to 5 % more error.)
struct Split3 { bf16x8 part[3]; };
__device__ __forceinline__ void split_pair(float x, float y, uint32_t (&to)[3])
{
    typedef float float2v __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 3; i++) {
        to[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v{x, y}), bf16x2));
        x -= __uint_as_float(to[i] << 16);
        y -= __uint_as_float(to[i] & 0xffff0000u);
    }
}
// c += A B of such operands, in six products from the smallest on (what is left out is 2^-24 of the largest)
__device__ __forceinline__ void mfma_split3(float16v &c, const Split3 &a, const Split3 &b)
{
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[2], b.part[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[0], b.part[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[1], b.part[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[1], b.part[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[0], b.part[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[0], b.part[0], c, 0, 0, 0);
}
// exp(x) for x <= 0 (0 far below; not finite: NaN): 2^(x log2 e) with what the product's rounding left put right behind
__device__ __forceinline__ float exp_below(float x)
{
    const float p = x * 1.44269502f, r = fmaf(x, 1.92596303e-8f, fmaf(x, 1.44269502f, -p)), e = __builtin_amdgcn_exp2f(p);
    return fmaf(e * r, 0.693147182f, e);
}

// The same for heads of 128 and 256, with 32-bit operands as three bf16 ones: six matrix instructions of 32 cycles stand for eight of 64,
// and they run beside the other wave's vector instructions.  Keys and values come to the waves through LDS, each wave's own ring of three
// stages of 4 KB, two of them on their way: straight to registers a load instruction touched 64 key rows, and there was room for one stage
// ahead.  The rows' operands are split once for the workgroup and lie in LDS (24 KB for heads of 128; two workgroups on a CU).  Scores are
// summed 32 columns at a time, values by the sixteen keys of an instruction.  Key heads are the fast grid dimension: of eight, each is
// read into one XCD's L2.
// Bound by the splits: some 1400 vector instructions per tile, 800 of them splits, beside 96 matrix ones; a wave that has a SIMD for itself
// takes 5.6 us for a tile, 7.4 in 32 bits.  32 heads of 128 over 8, 70 / 500 tokens 12.5 / 55 -> 10.5 / 28.2 us (ring and order of workgroups alone,
// still in 32 bits: 41); 4 heads of 256 over one 22.0 / 61 -> 18.0 / 43.7, 250 behind 777 121 -> 84.
// Error against 64 bits, units of 2^-24 of the result's norm, 70 / 500 tokens of normal keys: 128 1.99 / 2.04 -> 1.78 / 1.82, 256 2.06 / 2.05 -> 1.81 / 1.74;
// scores four times as wide 4.0 / 5.9 -> 3.6 / 5.2 and 4.9 / 6.4 -> 4.1 / 5.7.
template <int HD>
__global__ __launch_bounds__(TB, HD <= 128 ? 2 : 1) void k_prompt_attn_split(const float *__restrict__ Q, const float *__restrict__ Kc, const float *__restrict__ Vc,
                                                                             float *__restrict__ out, int M, int pos, int Hq, int G, int max_seq, float scale, int down)
{
    constexpr int CB = HD / 32, SLOTS = 3, SLOT = 4096, RING = 4 * SLOTS * SLOT, PART = 2 * CB * 16 * 64 * 4;
    constexpr int NK = HD / 32, NS = HD / 16;              // stages of a tile's keys, and of all of it
    __shared__ __attribute__((aligned(16))) char lds[RING > PART ? RING : PART];
    __shared__ bf16x8 qs[HD / 16][3][64];
    __shared__ float st[4][2][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), half = lane >> 5, col = lane & 31;
    const int kvh = blockIdx.x, rows = M * G, row0 = ((int)blockIdx.y < down ? (int)gridDim.y - 1 - (int)blockIdx.y : (int)blockIdx.y - down) * 32;
    const int r = min(row0 + col, rows - 1), m = r / G, head = kvh * G + r % G, qpos = pos + m;
    const int last = pos + min(row0 + 31, rows - 1) / G, tiles = last / 32 + 1;
    const float *Kh = Kc + (size_t)kvh * max_seq * HD, *Vh = Vc + (size_t)kvh * max_seq * HD;

    // Stage s of tile t on its way to a slot of the wave's own: 32 keys' columns 32 s .., or eight keys' values of 128 columns; a row
    // behind the last asks for the last again.  Key rows lie with their 16-byte parts turned by the row, so that lanes of sixteen
    // rows read from different banks.
    const uint32_t ring = (uint32_t)(uintptr_t)(lds_void *)lds + wave * (SLOTS * SLOT);
    const char *rd = lds + wave * (SLOTS * SLOT);
    auto ask = [&](int t, int s, uint32_t slot) __attribute__((always_inline)) {
        const uint32_t left = (uint32_t)(last - t * 32);
        const char *from = reinterpret_cast<const char *>((s < NK ? Kh : Vh) + (size_t)t * 32 * HD);
        const int v = s - NK, keys = 16 * (v / (HD / 64)) + 8 * (v % 2), cols = 128 * (v / 2 % (HD / 128));
        int ln = lane;
        asm volatile("" : "+v"(ln));                       // (the lane's share of every offset, kept over the loop, spills)
#pragma unroll
        for (int n = 0; n < 4; n++) {
            uint32_t off;
            if (s < NK) off = (min((uint32_t)(8 * n + (ln >> 3)), left) * HD + 32 * s + 4 * ((ln & 7) ^ (ln >> 3))) * 4;
            else off = (min((uint32_t)(keys + 2 * n + (ln >> 5)), left) * HD + cols + 4 * (ln & 31)) * 4;
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(off), "s"(from), "s"(ring + slot + 1024u * n) : "memory", "m0");
        }
    };
    // the stage that the wave goes on to is there once at most the eight loads of the two behind it are on their way; the second of them
    // goes where the stage before was read from (and multiplied: the products are ahead of the barrier)
    uint32_t now_slot = (SLOTS - 1) * SLOT;
    auto arrive = [&](int t, int s) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        if (s + 2 < NS) ask(t, s + 2, now_slot);
        else ask(t + 4 < tiles ? t + 4 : t, s + 2 - NS, now_slot);
        now_slot = now_slot == (SLOTS - 1) * SLOT ? 0 : now_slot + SLOT;
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // the rows' operands, a quarter by each wave: columns 32 (s / 2) + 16 half + 8 (s % 2) .. for step s
    {
        const float *qp = Q + ((size_t)m * Hq + head) * HD + 16 * half;
        float4v q[HD / 64][2];
#pragma unroll
        for (int i = 0; i < HD / 64; i++)
#pragma unroll
            for (int e = 0; e < 2; e++) q[i][e] = *reinterpret_cast<const float4v *>(qp + 32 * ((wave + 4 * i) >> 1) + 8 * (wave & 1) + 4 * e);
#pragma unroll
        for (int i = 0; i < HD / 64; i++) {
            u32x4 f[3];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                uint32_t w[3];
                split_pair(q[i][e >> 1][2 * (e & 1)], q[i][e >> 1][2 * (e & 1) + 1], w);
#pragma unroll
                for (int x = 0; x < 3; x++) f[x][e] = w[x];
            }
#pragma unroll
            for (int x = 0; x < 3; x++) qs[wave + 4 * i][x][lane] = __builtin_bit_cast(bf16x8, f[x]);
        }
    }
    __syncthreads();
    if (wave < tiles)
#pragma unroll
        for (int s = 0; s < 2; s++) ask(wave, s, s * SLOT);
    float16v O[CB] = {};
    float mx = -3.0e38f, before = -1.0e30f, l = 0.f, bad = 0.f;
    for (int t = wave; t < tiles; t += 4) {
        float16v S = {};
#pragma unroll
        for (int i = 0; i < NK; i++) {
            arrive(t, i);
            const char *at = rd + now_slot + col * 128;
            float4v k[4];
#pragma unroll
            for (int e = 0; e < 4; e++) k[e] = *reinterpret_cast<const float4v *>(at + 16 * ((4 * half + e) ^ (col & 7)));
            float16v T = {};
#pragma unroll
            for (int u = 0; u < 2; u++) {
                Split3 q, a;
#pragma unroll
                for (int x = 0; x < 3; x++) q.part[x] = qs[2 * i + u][x][lane];
                u32x4 f[3];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    uint32_t w[3];
                    split_pair(k[2 * u + (e >> 1)][2 * (e & 1)], k[2 * u + (e >> 1)][2 * (e & 1) + 1], w);
#pragma unroll
                    for (int x = 0; x < 3; x++) f[x][e] = w[x];
                }
#pragma unroll
                for (int x = 0; x < 3; x++) a.part[x] = __builtin_bit_cast(bf16x8, f[x]);
                mfma_split3(T, a, q);
            }
            S += T;
        }
        float top = -3.0e38f;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const bool seen = t * 32 + 8 * (j >> 2) + 4 * half + (j & 3) <= qpos;
            S[j] = seen ? S[j] * scale : -1.0e32f;
            if (seen) top = fmaxf(top, S[j]);
        }
        top = xor_max<32>(top);
        if (top < -1.0e29f && top > -3.0e38f) bad = 1.f;   // (below what the sums are taken relative to)
        mx = fmaxf(mx, top);
        const float now = fmaxf(mx, -1.0e30f), keep = exp_below(before - now);
        before = now;
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < 16; j++) { S[j] = exp_below(S[j] - now); sum += S[j]; }   // (a key that is not seen: 0)
        l = fmaf(l, keep, sum);
        // the two steps of sixteen keys: registers 8 n .. 8 n + 7 hold the half's eight
#pragma unroll
        for (int n = 0; n < 2; n++) {
            Split3 p;
            u32x4 f[3];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                uint32_t w[3];
                split_pair(S[8 * n + 2 * e], S[8 * n + 2 * e + 1], w);
#pragma unroll
                for (int x = 0; x < 3; x++) f[x][e] = w[x];
            }
#pragma unroll
            for (int x = 0; x < 3; x++) p.part[x] = __builtin_bit_cast(bf16x8, f[x]);
#pragma unroll
            for (int h = 0; h < HD / 128; h++) {           // columns 128 h + 4 col ..
                u32x4 a[4][3];
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    arrive(t, NK + n * (HD / 64) + 2 * h + b);
                    const char *at = rd + now_slot + half * 2048 + 16 * col;
                    float4v v[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = *reinterpret_cast<const float4v *>(at + 512 * e);
#pragma unroll
                    for (int c = 0; c < 4; c++)
#pragma unroll
                        for (int e = 0; e < 2; e++) {
                            uint32_t w[3];
                            split_pair(v[2 * e][c], v[2 * e + 1][c], w);
#pragma unroll
                            for (int x = 0; x < 3; x++) a[c][x][2 * b + e] = w[x];
                        }
                }
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    Split3 w;
#pragma unroll
                    for (int x = 0; x < 3; x++) w.part[x] = __builtin_bit_cast(bf16x8, a[c][x]);
                    float16v T = {};
                    mfma_split3(T, w, p);
#pragma unroll
                    for (int j = 0; j < 16; j++) O[4 * h + c][j] = n == 0 ? fmaf(O[4 * h + c][j], keep, T[j]) : O[4 * h + c][j] + T[j];
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (the slots become the merge's)
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
        for (int j = 0; j < 16; j++) bad = fmaf(O[c][j], 0.f, bad);
    if (__syncthreads_or(bad != 0.f)) {                    // an operand was not finite, or a sum grew beyond
        for (int i = wave; i < 32 && row0 + i < rows; i += 4) attend_plain<HD>(Q, Kh, Vh, out, (row0 + i) / G, kvh * G + (row0 + i) % G, pos + (row0 + i) / G, Hq, scale);
        return;
    }
    finish_rows<HD, true>(O, mx, l, reinterpret_cast<float (*)[CB * 16][64]>(lds), st, out + ((size_t)m * Hq + head) * HD, row0 + col < rows);
}

// The same for short contexts: one (token, query head) per wave, all in registers.  Sixteen lanes take a key, four columns each and 64
// apart, so four keys are read side by side, four such groups requested together; a score is a sum over sixteen lanes, a row of up to
// 64 scores sixteen registers, and the four lane groups' shares of the output meet at the end.  Up to 64 keys the tiles above are one
// or two, each the whole chain of HD matrix instructions of 64 cycles in one wave while others idle.  32 heads of 128 over 8 at 8 / 32 / 64
// tokens: 12.5 / 12.3 / 13.0 us, 4.0 / 4.9 / 7.6 so; 4 heads of 256 over one 21 / 21 / 22, 4.8 / 6.7 / 9.2.  The reads grow with the square
// of the tokens: 32 heads break even at some 100, so the line is at the sixteen registers.
constexpr int SHORT_KEYS = 64;
template <int HD>
__global__ __launch_bounds__(TB) void k_prompt_attn_short(const float *__restrict__ Q, const float *__restrict__ Kc, const float *__restrict__ Vc,
                                                          float *__restrict__ out, int M, int pos, int Hq, int G, int max_seq, float scale)
{
    constexpr int C = HD / 64, NI = SHORT_KEYS / 4;
    const int lane = threadIdx.x & 63, id = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (id >= M * Hq) return;
    const int m = id / Hq, head = id % Hq, qpos = pos + m, g = lane >> 4, c = 4 * (lane & 15);
    const float *Kh = Kc + (size_t)(head / G) * max_seq * HD, *Vh = Vc + (size_t)(head / G) * max_seq * HD, *q = Q + (size_t)id * HD;
    float4v qv[C];
#pragma unroll
    for (int i = 0; i < C; i++) qv[i] = *reinterpret_cast<const float4v *>(q + c + 64 * i);
    auto row = [&](const float *X, int it, float4v (&r)[C]) __attribute__((always_inline)) {       // (keys behind the query's repeat its own)
        const float *at = X + (uint32_t)(min(4 * it + g, qpos) * HD + c);
#pragma unroll
        for (int i = 0; i < C; i++) r[i] = *reinterpret_cast<const float4v *>(at + 64 * i);
    };
    float s[NI], mx = -3.0e38f;
#pragma unroll
    for (int i0 = 0; i0 < NI; i0 += 4) {
#pragma unroll
        for (int u = 0; u < 4; u++) s[i0 + u] = -INFINITY;
        if (4 * i0 > qpos) continue;                       // (uniform)
        float4v k[4][C];
#pragma unroll
        for (int u = 0; u < 4; u++) row(Kh, i0 + u, k[u]);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            float d = 0.f;
#pragma unroll
            for (int i = 0; i < C; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) d = fmaf(qv[i][e], k[u][i][e], d);
            d = xor_add<8>(xor_add<4>(xor_add<2>(xor_add<1>(d)))) * scale;
            if (4 * (i0 + u) + g <= qpos) { s[i0 + u] = d; mx = fmaxf(mx, d); }
        }
    }
    mx = xor_max<32>(xor_max<16>(mx));
    float l = 0.f;
#pragma unroll
    for (int i = 0; i < NI; i++) { s[i] = expf(s[i] - mx); l += s[i]; }
    l = xor_add<32>(xor_add<16>(l));
    float4v o[C] = {};
#pragma unroll
    for (int i0 = 0; i0 < NI; i0 += 4) {
        if (4 * i0 > qpos) continue;
        float4v v[4][C];
#pragma unroll
        for (int u = 0; u < 4; u++) row(Vh, i0 + u, v[u]);
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (4 * (i0 + u) + g <= qpos)
#pragma unroll
                for (int i = 0; i < C; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) o[i][e] = fmaf(s[i0 + u], v[u][i][e], o[i][e]);
    }
#pragma unroll
    for (int i = 0; i < C; i++) {
#pragma unroll
        for (int e = 0; e < 4; e++) o[i][e] = xor_add<32>(xor_add<16>(o[i][e])) / l;
        if (g == i % 4) *reinterpret_cast<float4v *>(out + (size_t)id * HD + c + 64 * i) = o[i];
    }
}

__global__ __launch_bounds__(TB) void k_planes_to_rows(SplitPlanes p, float *__restrict__ out, int N, int ldc)
{
    const int n = blockIdx.x * TB + threadIdx.x, m = blockIdx.y;
    if (n < N) out[(size_t)m * ldc + n] = planes_at(p, m, n);
}

// One workgroup per token, the gated row in registers (C chunks of four columns per thread): the planes are read once and the
// next product's operand leaves as two fp16 rows, where a gate kernel and a split kernel wrote and read the fp32 row between them.
// 500 rows of 9728: 20.7 us.  (A few rows leave most CUs without one: at eight, 11.8 us against 9.2 for the two kernels, which a
// batch's steps therefore keep.)
template <int C, int GELU>
__global__ __launch_bounds__(1024) void k_prompt_glu(SplitPlanes gu, half_t *__restrict__ a16, float *__restrict__ inv, int lo, int IS, int Kb)
{
    __shared__ float sm[16];
    const int m = blockIdx.x;
    float v[C][4];
    float amax = 0.f;
#pragma unroll
    for (int u = 0; u < C; u++) {
        const int n = (threadIdx.x + 1024 * u) * 4;
#pragma unroll
        for (int e = 0; e < 4; e++) v[u][e] = 0.f;
        if (n < IS) {
            const float4v g = planes4_at(gu, m, n), up = planes4_at(gu, m, IS + n);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float act = GELU ? 0.5f * g[e] * (1.0f + tanhf(gelu_inner(g[e]))) : g[e] / (1.0f + expf(-g[e]));
                v[u][e] = act * up[e];
                amax = fmaxf(amax, fabsf(v[u][e]));
            }
        }
    }
    amax = block_max(amax, sm);
    const float s = row_scale_for(amax), is = 1.0f / s;
#pragma unroll
    for (int u = 0; u < C; u++) {
        const int n = (threadIdx.x + 1024 * u) * 4;
        half4 h, l;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            h[e] = f2h(v[u][e] * s);
            l[e] = f2h((v[u][e] * s - h2f(h[e])) * PAIR_RESIDUAL_SCALE);
        }
        if (n < Kb * 64) {
            *reinterpret_cast<half4 *>(a16 + tiled_a_index(m, n, Kb)) = h;
            *reinterpret_cast<half4 *>(a16 + tiled_a_index(lo + m, n, Kb)) = l;
        }
    }
    if (threadIdx.x == 0) { inv[m] = is; inv[lo + m] = is / PAIR_RESIDUAL_SCALE; }
}

}  // namespace

namespace lmhip {

void launch_embed_ids(const float *emb, const int *ids, float scale, float *x, int M, int D)
{
    hipLaunchKernelGGL(k_embed_ids, dim3((D + TB - 1) / TB, M), dim3(TB), 0, stream(), emb, ids, scale, x, D);
}

void launch_copy_caches(float *k, float *v, int B, int Hkv, int max_seq, int hd, int len)
{
    if (B < 2) return;
    const size_t head = (size_t)max_seq * hd;
    hipLaunchKernelGGL(k_copy_caches, dim3((unsigned)(((size_t)len * hd + TB - 1) / TB), Hkv, 2 * (B - 1)), dim3(TB), 0, stream(), k, v, (size_t)Hkv * head, head, len * hd);
}

void launch_prompt_heads(const PromptHeads &a)
{
    if (a.M <= 0 || a.hd > 256 || (a.hd & 1) || a.R > 64 || a.pos < 0 || a.pos + a.M > a.max_seq) { fprintf(stderr, "[fast_hip] prompt_heads: unsupported shape\n"); abort(); }
    hipLaunchKernelGGL(k_prompt_heads, dim3((a.Hq + 2 * a.Hkv + 3) / 4, a.M), dim3(TB), 0, stream(), a);
}

bool prompt_attention_supported(int hd) { return hd == 32 || hd == 64 || hd == 128 || hd == 256; }

void launch_prompt_attention(const float *q, const float *kc, const float *vc, float *out, int M, int pos, int Hq, int Hkv, int hd, int max_seq)
{
    if (M <= 0 || pos < 0 || pos + M > max_seq || Hkv <= 0 || Hq % Hkv || (((uintptr_t)q | (uintptr_t)kc | (uintptr_t)(hd >= 128 ? vc : kc) | (uintptr_t)out) & 15)) {
        fprintf(stderr, "[fast_hip] prompt_attention: unsupported shape\n"); abort();
    }
    const int G = Hq / Hkv;
    const dim3 grid((M * G + 31) / 32, Hkv);
    const float scale = 1.0f / sqrtf((float)hd);
    if (pos + M <= SHORT_KEYS && (hd == 128 || hd == 256)) {
        const dim3 waves((M * Hq + 3) / 4);
        if (hd == 128) hipLaunchKernelGGL(k_prompt_attn_short<128>, waves, dim3(TB), 0, stream(), q, kc, vc, out, M, pos, Hq, G, max_seq, scale);
        else hipLaunchKernelGGL(k_prompt_attn_short<256>, waves, dim3(TB), 0, stream(), q, kc, vc, out, M, pos, Hq, G, max_seq, scale);
        return;
    }
    // longest first; where all workgroups are resident at once, two to a CU, those that come second to one are the shortest first: of 512 on 256 CUs
    // 16 + 1 tiles meet, 15 + 2 .., where 16 + 8 to 8 + 1 did
    const dim3 tall(Hkv, grid.x);
    const int cus = num_cus(), down = hd <= 128 && (int)(grid.x * grid.y) <= 2 * cus ? std::min<int>(grid.x, (cus + Hkv - 1) / Hkv) : (int)grid.x;
#define PA(HD_) hipLaunchKernelGGL(k_prompt_attn<HD_>, grid, dim3(TB), 0, stream(), q, kc, vc, out, M, pos, Hq, G, max_seq, scale)
#define PS(HD_) hipLaunchKernelGGL(k_prompt_attn_split<HD_>, tall, dim3(TB), 0, stream(), q, kc, vc, out, M, pos, Hq, G, max_seq, scale, down)
    if (hd == 32) PA(32); else if (hd == 64) PA(64); else if (hd == 128) PS(128); else if (hd == 256) PS(256);
    else { fprintf(stderr, "[fast_hip] prompt_attention: unsupported head size %d\n", hd); abort(); }
#undef PA
#undef PS
}

void launch_planes_to_rows(const SplitPlanes &p, float *out, int M, int N, int ldc)
{
    hipLaunchKernelGGL(k_planes_to_rows, dim3((N + TB - 1) / TB, M), dim3(TB), 0, stream(), p, out, N, ldc);
}

bool prompt_glu_supported(int IS) { return IS % 4 == 0 && tiled_kb(IS) * 64 <= 16384; }

void launch_prompt_glu(const SplitPlanes &gu, half_t *a16, float *inv, int M, int lo, int IS, int gelu)
{
    if (!prompt_glu_supported(IS) || lo < M || gu.N % 4 || gu.N < 2 * IS || (gu.plane | gu.plane2) % 4 || ((uintptr_t)gu.P | (uintptr_t)gu.P2) & 15) {
        fprintf(stderr, "[fast_hip] prompt_glu: unsupported shape %d\n", IS); abort();
    }
    const int Kb = tiled_kb(IS), C = (Kb * 16 + 1023) / 1024;
#define PG(C_) do { if (gelu) hipLaunchKernelGGL((k_prompt_glu<C_, 1>), dim3(M), dim3(1024), 0, stream(), gu, a16, inv, lo, IS, Kb); \
                    else hipLaunchKernelGGL((k_prompt_glu<C_, 0>), dim3(M), dim3(1024), 0, stream(), gu, a16, inv, lo, IS, Kb); } while (0)
    if (C == 1) PG(1); else if (C == 2) PG(2); else if (C == 3) PG(3); else PG(4);
#undef PG
}

}  // namespace lmhip
