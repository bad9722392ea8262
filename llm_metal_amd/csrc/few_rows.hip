// A batch's step or a short prompt reads every weight once for up to 32 rows: bound by the weights' bytes and by what stands between the launches, so
// its products take their operand as the kernels before leave it and leave what the kernels behind need (few_rows.h).
#include "backend.h"
#include "devutil.h"
#include "few_rows.h"
#include <stdio.h>
#include <algorithm>
#include <type_traits>

using namespace lmhip;

namespace {

constexpr float RESIDUAL = 2048.f;                         // a residual image is that many times what its value image left over

__device__ __forceinline__ float gated(float g, float u, int gelu)
{
    return (gelu ? 0.5f * g * (1.0f + tanhf(gelu_inner(g))) : g / (1.0f + expf(-g))) * u;
}

// The sums of a workgroup's waves for 32 weight rows (WT 2: gate and up rows) times the images of up to 16 MT vectors, acc[row block][image tile],
// meet in `part`, half of the waves at a time; value and residual images times their factors are added and the results stored.
// TOKENS: an accumulator's rows are the images and its columns the weight rows, else the other way round.
template <int MT, int WT, int WAVES, bool TOKENS>
__device__ __forceinline__ void few_finish(float *part, const float16v (&acc)[WT][MT], const float *__restrict__ inv, float *__restrict__ out, int ldo, int B, int N, int gelu)
{
    constexpr int HALF = WAVES / 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float *p = part + (size_t)(wave & (HALF - 1)) * WT * MT * 1024;
    if (wave >= HALF) {
#pragma unroll
        for (int q = 0; q < WT; q++)
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int i = 0; i < 16; i++) p[((q * MT + m) * 16 + i) * 64 + lane] = acc[q][m][i];
    }
    __syncthreads();
    if (wave < HALF) {
#pragma unroll
        for (int q = 0; q < WT; q++)
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int i = 0; i < 16; i++) p[((q * MT + m) * 16 + i) * 64 + lane] += acc[q][m][i];
    }
    __syncthreads();
    // row r of an accumulator is register 4 (r / 8) + r % 4 of the lanes of half (r / 4) % 2
    const int m = threadIdx.x & 31, n = blockIdx.x * 32 + m;
    if (n >= N) return;
    auto image = [&](int q, int row) __attribute__((always_inline)) {
        const int r = TOKENS ? row & 31 : m, c = TOKENS ? m : row & 31;
        const float *s = part + (q * MT + (MT > 1 ? row >> 5 : 0)) * 1024 + (4 * (r >> 3) + (r & 3)) * 64 + 32 * ((r >> 2) & 1) + c;
        float v = s[0];
#pragma unroll
        for (int h = 1; h < HALF; h++) v += s[h * WT * MT * 1024];
        return v * inv[row];
    };
    for (int b = threadIdx.x >> 5; b < B; b += 64 * WAVES / 32) {
        float v = image(0, b) + image(0, B + b);
        if (WT == 2) v = gated(v, image(WT - 1, b) + image(WT - 1, B + b), gelu);
        out[(size_t)b * ldo + n] = v;
    }
}

// WT 1: 32 weight rows of [N, K] per workgroup, WT 2: the 32 gate rows and the 32 up rows of as many FFN columns.  All of K in one
// workgroup, its waves taking the K tiles in turn with U of them requested at a time, straight into registers: a weight tile
// meets one operand tile, so there is nothing to share through LDS before the waves' sums meet there.  What leaves is the
// result itself: the kernels that added the planes of a K split, and for the gate a launch to form it, are not needed.
// MT: operand tiles of 32 rows (value and residual rows of up to 16 or 32 vectors).
// Weights are the first operand of the MFMA: a lane's column is a vector's image, its registers are weight rows.
// Eight vectors, 4B shape: Q|K|V 8.9 us (31 MB; the ring kernel 8.4 and 3.7 for its planes), gate|up 23.2 (100 MB; 20.0 and 4.8 for
// the gate), head of 32 768 rows 32.0 (27.3 and 4.2).  304 gate blocks fill 256 CUs unevenly: with four waves of up to four tiles in
// flight each 23.2, eight of two 24.2 (the operand tile of the next one then waits for registers).
// An accumulator is rounded at every instruction, so beyond sixteen vectors a K tile's four make a sum of their own: 20 tokens of one layer of width 2560
// are 4.2e-7 from 64 bits so, 5.0e-7 with up to forty instructions on one sum; steps of 17 sequences take 0.5 to 0.9 % more, of 32 no more.  Up to sixteen, where the matrix cores have half the work beside
// the same vector additions, that took 0.7 % of three sequences' steps and is left out.
template <int MT, int WT, int U, int WAVES>
__global__ __launch_bounds__(64 * WAVES, WT * MT == 4 || U > 3 ? 2 : 4) void k_few_full(const half8 *__restrict__ A, const float *__restrict__ inv, const half8 *__restrict__ W,
                                                                                float *__restrict__ out, int ldo, int B, int N, int Kb, int up_block, int gelu)
{
    constexpr int HALF = WAVES / 2;
    __shared__ float part[HALF * WT * MT * 16 * 64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const size_t up = (size_t)up_block * Kb * 256, second = (size_t)Kb * 256;      // (a tile's part of every address is scalar, a lane's 32 bits)
    uint32_t slot[MT];                                          // (rows past the last repeat it: no bytes of their own)
#pragma unroll
    for (int m = 0; m < MT; m++) slot[m] = a_lane((lane & 32) | (min(32 * m + (lane & 31), 2 * B - 1) & 31));
    float16v acc[WT][MT] = {};
    auto tiles = [&](auto count, int t0) __attribute__((always_inline)) {       // tiles t0, t0 + 8, ..: all of them asked for, then all multiplied
        constexpr int C = decltype(count)::value;
        constexpr int CA = U > 3 ? C : 1;                  // operand tiles in flight
        half8 w[C][WT][4], a[CA][MT][4];
        auto operand = [&](int u) __attribute__((always_inline)) {
            const half8 *at = A + (size_t)(t0 + WAVES * u) * 256;
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) a[u % CA][m][j] = (m ? at + second : at)[slot[m] + 64 * j];
        };
#pragma unroll
        for (int u = 0; u < C; u++) {
            const half8 *at = W + ((size_t)blockIdx.x * Kb + t0 + WAVES * u) * 256;
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                w[u][0][j] = __builtin_nontemporal_load(at + (uint32_t)(lane + 64 * j));
                if (WT == 2) w[u][WT - 1][j] = __builtin_nontemporal_load(at + up + (uint32_t)(lane + 64 * j));
            }
            if (u < CA) operand(u);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < C; u++) {
            if (MT == 1) {
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int q = 0; q < WT; q++) acc[q][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[u][q][j], a[u % CA][0][j], acc[q][0], 0, 0, 0);
            } else if (WAVES == 8) {                       // (128 registers: one tile's sum at a time)
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    float16v sum = {};
#pragma unroll
                    for (int j = 0; j < 4; j++) sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[u][0][j], a[u % CA][m][j], sum, 0, 0, 0);
                    acc[0][m] += sum;
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                float16v sum[WT][MT] = {};
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int q = 0; q < WT; q++)
#pragma unroll
                        for (int m = 0; m < MT; m++) sum[q][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[u][q][j], a[u % CA][m][j], sum[q][m], 0, 0, 0);
#pragma unroll
                for (int q = 0; q < WT; q++)
#pragma unroll
                    for (int m = 0; m < MT; m++) acc[q][m] += sum[q][m];
            }
            if (u + CA < C) operand(u + CA);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int t0 = wave, left = (Kb - wave + WAVES - 1) / WAVES;
    for (; left >= U; left -= U, t0 += WAVES * U) tiles(std::integral_constant<int, U>{}, t0);
    if (U > 4 && left == 4) tiles(std::integral_constant<int, U < 4 ? U : 4>{}, t0);
    if (U > 3 && left == 3) tiles(std::integral_constant<int, U < 3 ? U : 3>{}, t0);
    if (U > 2 && left == 2) tiles(std::integral_constant<int, U < 2 ? U : 2>{}, t0);
    if (left == 1) tiles(std::integral_constant<int, 1>{}, t0);
    few_finish<MT, WT, WAVES, false>(part, acc, inv, out, ldo, B, N, gelu);
}

// Eight codes of a Q8_0 row as fp16 integers, exactly: 1024 + (code + 128) is a half's bits, 1152 taken off
__device__ __forceinline__ half8 codes8(uint32_t a, uint32_t b)
{
    half8 r;
    const uint32_t w[2] = {a ^ 0x80808080u, b ^ 0x80808080u};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t p = __builtin_amdgcn_perm(0x64646464u, w[i >> 1], i & 1 ? 0x04030402u : 0x04010400u);
        const half2v h = __builtin_bit_cast(half2v, p) - half2v{(half_t)1152, (half_t)1152};
        r[2 * i] = h[0];
        r[2 * i + 1] = h[1];
    }
    return r;
}

// k_few_full over the rows of a Q8_0 matrix as they lie (codes [rows][K], a scale per 32 of them): 1.06 bytes per weight, and exact ones.
// A wave takes four blocks of its 32 rows at a time, a whole 128-byte line of each, the next ones on their way: read eight lanes to a
// line (a lane to a row made 32 lines of every load, which took the address unit 3.5 us a group) and turned through LDS of the
// wave's own.  Both lane halves multiply one block -- the operand's two column blocks, a lane half each, change places -- so
// that a block's two MFMAs multiply integers and its scale, one per lane with the weight rows as the accumulator's columns,
// goes onto their sum in fp32.  blockIdx.y: chunks of K (few_chunks), a plane of the result each.
// 4B shape, 8 / 32 vectors: Q|K|V 8.1 / 12.7 us, gate|up 21.8 / 29.4, O 7.4 / 10.5, down 12.4 / 20.6 (bound by the address unit and the
// trips, not by 1.06 bytes per weight); the two F16 images formed for every such product took 97 us a layer and their products 105.
// QUAD: a row's scales come in fours, in one load.
template <int MT, int WT, int WAVES, bool QUAD>
__global__ __launch_bounds__(64 * WAVES, MT * WT == 1 ? 4 : 2) void k_few_q8(const half8 *__restrict__ A, const float *__restrict__ inv, const int8_t *__restrict__ Wq,
                                                                            const half_t *__restrict__ Wd, float *__restrict__ out, int ldo, int B, int N, int K, int up_row, int gelu)
{
    constexpr int G = 4, LDR = 144;                        // bytes of a row's line in LDS
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    __shared__ float part[WAVES / 2 * WT * MT * 16 * 64];
    __shared__ u4 lines[WAVES][WT][32 * LDR / 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), h = lane >> 5;
    const int nb = K >> 5, Kb = tiled_kb(K), all = (nb + G - 1) / G, each = (all + (int)gridDim.y - 1) / (int)gridDim.y;
    const int first = blockIdx.y * each, groups = min(first + each, all), row0 = blockIdx.x * 32;
    struct Stage { u4 c[WT][G]; half4 d[WT]; };
    auto load = [&](Stage &w, int g) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < WT; q++) {
#pragma unroll
            for (int u = 0; u < G; u++) {                  // rows 8 u + lane / 8, sixteen codes of the line
                const size_t r = min(row0 + 8 * u + (lane >> 3), N - 1) + (q ? up_row : 0);
                w.c[q][u] = __builtin_nontemporal_load(reinterpret_cast<const u4 *>(Wq + r * K + min(g * 128 + 16 * (lane & 7), K - 16)));
            }
            const half_t *d = Wd + (size_t)(min(row0 + (lane & 31), N - 1) + (q ? up_row : 0)) * nb;
            if (QUAD) w.d[q] = *reinterpret_cast<const half4 *>(d + min(g, all - 1) * G);
            else
#pragma unroll
                for (int u = 0; u < G; u++) w.d[q][u] = d[min(g * G + u, nb - 1)];
        }
    };
    uint32_t slot[MT];                                     // (image rows past the last repeat it)
#pragma unroll
    for (int m = 0; m < MT; m++) slot[m] = a_lane((lane & 32) | (min(32 * m + (lane & 31), 2 * B - 1) & 31));
    float16v sum[WT][MT] = {};
    Stage w;
    load(w, first + wave);                                 // (a wave behind the last group asks for the last columns; nothing of it is used)
    for (int g = first + wave; g < groups; g += WAVES) {
        half8 a[MT][2][4];                                 // the group's two tiles
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const half8 *at = A + (size_t)min(2 * g + t, Kb - 1) * 256;
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) a[m][t][j] = (m ? at + (size_t)Kb * 256 : at)[slot[m] + 64 * j];
        }
        float d[WT][G];
#pragma unroll
        for (int q = 0; q < WT; q++)
#pragma unroll
            for (int u = 0; u < G; u++) {
                *reinterpret_cast<u4 *>(reinterpret_cast<char *>(lines[wave][q]) + (8 * u + (lane >> 3)) * LDR + 16 * (lane & 7)) = w.c[q][u];
                d[q][u] = (float)w.d[q][u];
            }
        load(w, g + WAVES);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");     // (a wave's own lines: no barrier)
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
        // column blocks 0 and 1 of a tile, a lane half each: slices 2 e and 2 e + 1 become block 0's and block 1's
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    u4 x = __builtin_bit_cast(u4, a[m][t][e]), y = __builtin_bit_cast(u4, a[m][t][e + 1]);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const auto r = __builtin_amdgcn_permlane32_swap(x[i], y[i], false, false);
                        x[i] = r[0];
                        y[i] = r[1];
                    }
                    a[m][t][e] = __builtin_bit_cast(half8, x);
                    a[m][t][e + 1] = __builtin_bit_cast(half8, y);
                }
#pragma unroll
        for (int u = 0; u < G; u++) {
            if (g * G + u >= nb) break;
#pragma unroll
            for (int q = 0; q < WT; q++) {
                const char *line = reinterpret_cast<const char *>(lines[wave][q]) + (lane & 31) * LDR + 32 * u + 8 * h;
                const u2 c0 = *reinterpret_cast<const u2 *>(line), c1 = *reinterpret_cast<const u2 *>(line + 16);
                const half8 w0 = codes8(c0[0], c0[1]), w1 = codes8(c1[0], c1[1]);
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    float16v acc = {};
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[m][u >> 1][u & 1], w0, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[m][u >> 1][2 + (u & 1)], w1, acc, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 16; i++) sum[q][m][i] = fmaf(acc[i], d[q][u], sum[q][m][i]);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    few_finish<MT, WT, WAVES, true>(part, sum, inv, out + (size_t)blockIdx.y * B * ldo, ldo, B, N, gelu);
}

// 128 weight rows and 2 T K tiles per workgroup: each of its eight waves holds the T weight tiles of one row block and one half of
// the K tiles, requested before anything else, and while they travel the waves turn the fp32 rows of the chunk into value and
// residual images in LDS, with a factor for each (row, K tile): no kernel in front has to know a row's maximum.  A tile's sum (four
// MFMAs) times its factors is added in fp32.  Planes [B, N], value and residual already together.
// Eight vectors, 4B shape: O 7.3 us, down 12.2; the ring kernel took 9.3 for either behind a launch of 4.2 and 4.7 that split the
// rows, and left twice the rows to add.
template <int MT, int T>
__global__ __launch_bounds__(512) void k_few_split(const float *__restrict__ X, const half8 *__restrict__ W, float *__restrict__ P, int B, int N, int K, int Kb)
{
    constexpr int TILES = 2 * T;
    __shared__ half_t img[(TILES * MT * 2048 > 8192 ? TILES * MT * 2048 : 8192)];       // later the sums of one half of the waves
    __shared__ float fac[TILES][16 * MT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int rt = wave & 3, kp = wave >> 2, rbs = (N + 31) >> 5;
    const int rb = blockIdx.x * 4 + rt, tile0 = blockIdx.y * TILES;
    half8 w[T][4];
    {
        const half8 *wp = W + (size_t)min(rb, rbs - 1) * Kb * 256 + lane;
#pragma unroll
        for (int u = 0; u < T; u++) {
            const size_t t = min(tile0 + kp * T + u, Kb - 1);
#pragma unroll
            for (int j = 0; j < 4; j++) w[u][j] = __builtin_nontemporal_load(wp + t * 256 + j * 64);
        }
    }
    for (int q = wave; q < TILES && tile0 + q < Kb; q += 8) {       // four lanes hold the 64 columns of a row
        half_t *at = img + q * MT * 2048;
        const int c = 16 * (lane & 3), k0 = (tile0 + q) * 64 + c;
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const int r = 16 * m + (lane >> 2);
            const float *x = X + (size_t)min(r, B - 1) * K + k0;
            float4v v[4];
            float top = 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = float4v{};
                if (k0 + 4 * e < K) v[e] = *reinterpret_cast<const float4v *>(x + 4 * e);
#pragma unroll
                for (int i = 0; i < 4; i++) top = fmaxf(top, fabsf(v[e][i]));
            }
            top = xor_max<2>(xor_max<1>(top));
            const float s = row_scale_for(top);
            half8 hi[2], lo[2];
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const float y = v[e >> 2][e & 3] * s;
                hi[e >> 3][e & 7] = f2h(y);
                lo[e >> 3][e & 7] = f2h((y - h2f(hi[e >> 3][e & 7])) * RESIDUAL);
            }
            const int row_lo = MT == 1 ? 16 + r : r;
            half_t *to_lo = at + (MT - 1) * 2048;
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int cc = c + 8 * e, piece = (cc & 31) >> 3, h = cc >> 5;
                *reinterpret_cast<half8 *>(at + (piece * 64 + 2 * r + h) * 8) = hi[e];
                *reinterpret_cast<half8 *>(to_lo + (piece * 64 + 2 * row_lo + h) * 8) = lo[e];
            }
            if ((lane & 3) == 0) fac[q][r] = 1.0f / s;
        }
    }
    __syncthreads();
    float16v sum = {};
#pragma unroll
    for (int u = 0; u < T; u++) {
        const int q = kp * T + u;
        if (tile0 + q >= Kb) break;
        const half8 *a = reinterpret_cast<const half8 *>(img + q * MT * 2048) + a_lane(lane);
        const float f = fac[q][lane & (16 * MT - 1)];
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float16v acc = {};
#pragma unroll
            for (int j = 0; j < 4; j++) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[u][j], a[m * 256 + j * 64], acc, 0, 0, 0);
            const float fm = (MT == 1 ? (lane & 16) != 0 : m == 1) ? f * (1.0f / RESIDUAL) : f;
#pragma unroll
            for (int i = 0; i < 16; i++) sum[i] = fmaf(acc[i], fm, sum[i]);
        }
    }
    __syncthreads();
    float *meet = reinterpret_cast<float *>(img) + rt * 1024 + lane;
    if (kp) {
#pragma unroll
        for (int i = 0; i < 16; i++) meet[i * 64] = sum[i];
    }
    __syncthreads();
    if (kp || rb >= rbs) return;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        sum[i] += meet[i * 64];
        if (MT == 1) sum[i] = xor_add<16>(sum[i]);
    }
    const int b = lane & (16 * MT - 1);
    if (b >= B || (MT == 1 && (lane & 16))) return;
    float *o = P + ((size_t)blockIdx.y * B + b) * N;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int n = rb * 32 + 8 * i + 4 * (lane >> 5);
        if (n < N) *reinterpret_cast<float4v *>(o + n) = float4v{sum[4 * i], sum[4 * i + 1], sum[4 * i + 2], sum[4 * i + 3]};
    }
}

// x += branch (br's planes added up; or its RMSNorm with g_branch); the RMSNorm of x with g as rows b and B + b of the next
// product's operand and, where ln is not null, as fp32.  One workgroup per row, four columns per thread, every load of it
// requested before the first sum: a chain of one trip to memory and one reduction (two with g_branch), which a workgroup per row
// can do no faster than that: 5.0 us at eight rows of 2560 or 1152 (5.9 and 6.6 with the residual's maximum and a round of loads
// more).  The residual image takes the value image's factor times 2^11, so that it needs no maximum of its own.
template <int C, bool AROUND>
__global__ __launch_bounds__(1024) void k_few_norm(float *__restrict__ x, FewPlanes br, const float *__restrict__ g_branch, const float *__restrict__ g,
                                                   float *__restrict__ ln, half_t *__restrict__ a16, float *__restrict__ inv_out, int B, int D, float eps)
{
    constexpr int Q = 20 / C;                              // planes in flight
    __shared__ float sm[32];
    const int b = blockIdx.x, Kb = tiled_kb(D);
    x += (size_t)b * D;
    float4v v[C], gv[C], gb[C], bv[C];
#pragma unroll
    for (int u = 0; u < C; u++) {
        const int i = 4 * (threadIdx.x + blockDim.x * u);
        v[u] = gv[u] = gb[u] = bv[u] = float4v{};
        if (i >= D) continue;
        v[u] = *reinterpret_cast<const float4v *>(x + i);
        gv[u] = *reinterpret_cast<const float4v *>(g + i);
        if (AROUND) gb[u] = *reinterpret_cast<const float4v *>(g_branch + i);
    }
    for (int s0 = 0; s0 < br.S; s0 += Q) {
        float4v t[C][Q];
#pragma unroll
        for (int u = 0; u < C; u++) {
            const int i = min(4 * (int)(threadIdx.x + blockDim.x * u), D - 4);
#pragma unroll
            for (int q = 0; q < Q; q++) t[u][q] = *reinterpret_cast<const float4v *>(br.P + (size_t)min(s0 + q, br.S - 1) * br.plane + (size_t)b * D + i);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < C; u++)
#pragma unroll
            for (int q = 0; q < Q; q++)
                if (s0 + q < br.S) bv[u] += t[u][q];
    }
    float inv_b = 1.f;
    if (AROUND) {
        float ss = 0.f;
#pragma unroll
        for (int u = 0; u < C; u++)
            if (4 * (int)(threadIdx.x + blockDim.x * u) < D)
#pragma unroll
                for (int e = 0; e < 4; e++) ss += bv[u][e] * bv[u][e];
        inv_b = rsqrtf(block_sum(ss, sm) / (float)D + eps);
    }
    float ss = 0.f, mxg = 0.f;
#pragma unroll
    for (int u = 0; u < C; u++) {
        const int i = 4 * (threadIdx.x + blockDim.x * u);
        if (i >= D) continue;
        if (br.S) {
            v[u] += AROUND ? bv[u] * inv_b * gb[u] : bv[u];
            *reinterpret_cast<float4v *>(x + i) = v[u];
        }
#pragma unroll
        for (int e = 0; e < 4; e++) { ss += v[u][e] * v[u][e]; mxg = fmaxf(mxg, fabsf(v[u][e] * gv[u][e])); }
    }
    block_sum_max(ss, mxg, sm);
    const float inv = rsqrtf(ss / (float)D + eps), s = row_scale_for(mxg * inv);
#pragma unroll
    for (int u = 0; u < C; u++) {
        const int i = 4 * (threadIdx.x + blockDim.x * u);
        v[u] = v[u] * inv * gv[u];
        if (ln && i < D) *reinterpret_cast<float4v *>(ln + (size_t)b * D + i) = v[u];
        half4 hi, lo;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float y = v[u][e] * s;
            hi[e] = f2h(y);
            lo[e] = f2h((y - h2f(hi[e])) * RESIDUAL);
        }
        if (i < Kb * 64) {
            *reinterpret_cast<half4 *>(a16 + tiled_a_index(b, i, Kb)) = hi;
            *reinterpret_cast<half4 *>(a16 + tiled_a_index(B + b, i, Kb)) = lo;
        }
    }
    if (threadIdx.x == 0) { inv_out[b] = 1.0f / s; inv_out[B + b] = 1.0f / s * (1.0f / RESIDUAL); }
}

// K tiles per wave: as many as leave the launch 200 workgroups (a chunk is a plane to add behind it).  Down of the 4B shape with eight
// instead of four: 12.7 against 12.2 us, and 0.25 us less in the norm behind it.
int split_tiles(int N, int K)
{
    const int groups = (tiled_rb(N) + 3) / 4;
    for (int T = 4; T > 1; T /= 2)
        if (groups * ((tiled_kb(K) + 2 * T - 1) / (2 * T)) >= 200) return T;
    return 1;
}

void check(bool ok, const char *what)
{
    if (!ok) { fprintf(stderr, "[fast_hip] %s: unsupported shape\n", what); abort(); }
}

}  // namespace

namespace lmhip {

void launch_few_full(const half_t *a16, const float *inv, const half_t *W, float *out, int ldo, int B, int N, int K)
{
    check(B >= 1 && B <= FEW_ROWS && N >= 1 && K >= 1 && ldo >= N, "few_full");
    const dim3 grid(tiled_rb(N));
    const half8 *A = reinterpret_cast<const half8 *>(a16), *w = reinterpret_cast<const half8 *>(W);
    const int Kb = tiled_kb(K);
    if (2 * B > 32) hipLaunchKernelGGL((k_few_full<2, 1, 2, 8>), grid, dim3(512), 0, stream(), A, inv, w, out, ldo, B, N, Kb, 0, 0);
    else hipLaunchKernelGGL((k_few_full<1, 1, 5, 8>), grid, dim3(512), 0, stream(), A, inv, w, out, ldo, B, N, Kb, 0, 0);
}

void launch_few_glu(const half_t *a16, const float *inv, const half_t *W, float *act, int B, int IS, int K, int gelu)
{
    check(B >= 1 && B <= FEW_ROWS && IS >= 32 && IS % 32 == 0 && K >= 1, "few_glu");
    const dim3 grid(IS / 32);
    const half8 *A = reinterpret_cast<const half8 *>(a16), *w = reinterpret_cast<const half8 *>(W);
    const int Kb = tiled_kb(K);
    if (2 * B > 32) hipLaunchKernelGGL((k_few_full<2, 2, 2, 4>), grid, dim3(256), 0, stream(), A, inv, w, act, IS, B, IS, Kb, IS / 32, gelu);
    else hipLaunchKernelGGL((k_few_full<1, 2, 4, 4>), grid, dim3(256), 0, stream(), A, inv, w, act, IS, B, IS, Kb, IS / 32, gelu);
}

void launch_few_norm(float *x, const FewPlanes &br, const float *g_branch, const float *g, float *ln, half_t *a16, float *inv, int B, int D, float eps)
{
    check(B >= 1 && B <= FEW_ROWS && D >= 4 && D % 4 == 0 && D <= 8192 && (!br.S || br.N == D) &&
          (((uintptr_t)x | (uintptr_t)br.P | (uintptr_t)g_branch | (uintptr_t)g | (uintptr_t)ln) & 15) == 0, "few_norm");
    const int pad = tiled_kb(D) * 64, nt = pad <= 4096 ? pad / 4 : 1024;      // (whole waves: pad is a multiple of 64, so nt of 16)
    const dim3 block((nt + 63) & ~63);
#define FN(C_, AROUND_) hipLaunchKernelGGL((k_few_norm<C_, AROUND_>), dim3(B), block, 0, stream(), x, br, g_branch, g, ln, a16, inv, B, D, eps)
    if (pad <= 4096) { if (br.S && g_branch) FN(1, true); else FN(1, false); }
    else { if (br.S && g_branch) FN(2, true); else FN(2, false); }
#undef FN
}

// K chunks of a product of [N, K] Q8_0 rows whose planes its consumer adds: 256 workgroups, at least two groups of columns per wave
int few_chunks(int N, int K)
{
    const int most = std::max(1, (K / 128) / 16);
    return std::min(most, (256 + tiled_rb(N) - 1) / tiled_rb(N));
}

#define FEW_Q8(MT_, WT_, WAVES_, OUT_, LDO_, UP_, GELU_) do { \
    if (K % 128 == 0 && ((uintptr_t)W.d & 7) == 0) hipLaunchKernelGGL((k_few_q8<MT_, WT_, WAVES_, true>), grid, dim3(64 * WAVES_), 0, stream(), A, inv, W.q, W.d, OUT_, LDO_, B, N, K, UP_, GELU_); \
    else hipLaunchKernelGGL((k_few_q8<MT_, WT_, WAVES_, false>), grid, dim3(64 * WAVES_), 0, stream(), A, inv, W.q, W.d, OUT_, LDO_, B, N, K, UP_, GELU_); } while (0)
FewPlanes launch_few_full_q8(const half_t *a16, const float *inv, const FewQ8 &W, float *out, int ldo, int B, int N, int K, int chunks)
{
    check(B >= 1 && B <= FEW_ROWS && N >= 1 && K >= 32 && K % 32 == 0 && ldo >= N && chunks >= 1 && chunks < 65536 && ((uintptr_t)W.q & 15) == 0, "few_full_q8");
    const dim3 grid(tiled_rb(N), chunks);
    const half8 *A = reinterpret_cast<const half8 *>(a16);
    if (2 * B > 32) FEW_Q8(2, 1, 8, out, ldo, 0, 0); else FEW_Q8(1, 1, 8, out, ldo, 0, 0);
    return FewPlanes{out, (size_t)B * ldo, chunks, ldo};
}

void launch_few_glu_q8(const half_t *a16, const float *inv, const FewQ8 &W, float *act, int B, int IS, int K, int gelu)
{
    check(B >= 1 && B <= FEW_ROWS && IS >= 32 && IS % 32 == 0 && K >= 32 && K % 32 == 0 && ((uintptr_t)W.q & 15) == 0, "few_glu_q8");
    const dim3 grid(IS / 32);
    const half8 *A = reinterpret_cast<const half8 *>(a16);
    const int N = IS;
    if (2 * B > 32) FEW_Q8(2, 2, 4, act, IS, IS, gelu); else FEW_Q8(1, 2, 4, act, IS, IS, gelu);
}
#undef FEW_Q8

int few_planes(int N, int K)
{
    const int T = split_tiles(N, K);
    return (tiled_kb(K) + 2 * T - 1) / (2 * T);
}

FewPlanes launch_few_split(const float *x, const half_t *W, float *P, int B, int N, int K)
{
    check(B >= 1 && B <= FEW_ROWS && N >= 4 && K >= 4 && N % 4 == 0 && K % 4 == 0 && (((uintptr_t)x | (uintptr_t)P) & 15) == 0, "few_split");
    const int T = split_tiles(N, K), S = few_planes(N, K), Kb = tiled_kb(K);
    const dim3 grid((tiled_rb(N) + 3) / 4, S);
    const half8 *w = reinterpret_cast<const half8 *>(W);
#define FS(MT_, T_) hipLaunchKernelGGL((k_few_split<MT_, T_>), grid, dim3(512), 0, stream(), x, w, P, B, N, K, Kb)
    if (2 * B > 32) { if (T == 4) FS(2, 4); else if (T == 2) FS(2, 2); else FS(2, 1); }
    else { if (T == 4) FS(1, 4); else if (T == 2) FS(1, 2); else FS(1, 1); }
#undef FS
    return FewPlanes{P, (size_t)B * N, S, N};
}

}  // namespace lmhip
