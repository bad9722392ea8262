// Large-M GEMM: C[M, N] = inv_scale[m] * A16[M, K] * W[N, K]^T for M of several hundred rows and more
// (batch * seq = 2048 in the Q8_0 configuration), where a weight tile is reused by enough activation rows
// that the matrix cores, not HBM, bound the product.  Same operands as the weight-streaming kernel
// (gemm.h: tiled fp16 activations with per-row power-of-two factors; F16 or Q8_0 weight tiles), fp16 products
// and fp32 accumulation, one launch; K chunks (planes) where the blocks leave CUs idle.  Q8_0 tiles and gemm_big_short multiply with
// v_mfma_f32_32x32x16_f16, F16 tiles (gemm_big_f16, gemm_big_pair) with v_mfma_f32_16x16x32_f16 on accumulators in place (acc_tiles.h).
//
// A workgroup of four waves owns a 128 x 256 block of C and walks K in steps of 64.  Per step every wave
// fetches one 32-row block of the activation tile and two of the weight tile from L2/HBM in the MFMA
// register layout, Q8_0 blocks are unpacked to fp16 there (int8 * fp16 scale, once per tile instead of once
// per consumer), and both go to LDS in the same [j][lane][8 halves] order, so a wave reads any row block back
// with conflict-free 16-byte loads.  LDS is double buffered and the operands travel three steps ahead in registers:
// during the MFMAs of step k the loads of step k+3 are issued and step k+1 is written to the other buffer; one
// barrier per step.  That is the kernel for Q8_0 tiles (gemm_big<1>, <2>); F16 tiles take gemm_big_f16 (the same block)
// or gemm_big_f16<256> (a 256 x 256 block) below, whose operands reach LDS without passing through registers, and
// launch_gemm_big chooses between the two block shapes, or gives each a part of the columns.
#include "backend.h"
#include "devutil.h"
#include "gemm.h"
#include "gemm_kernel.h"
#include "walk_k.h"
#include <hip/hip_ext.h>
#include <algorithm>

namespace lmhip {
namespace {

int g_big_split = 1;                  // 1: K chunks by the measured rule (big_gemm_chunks), 0: never, n > 1: always n
int g_big_block = 0;                  // F16 tiles: 0 block shape by the measured rule, 1 always 128 x 256, 2 always 256 x 256
constexpr int WPW = 2;               // weight row blocks each wave fetches per K step: the block is 128 x (WPW * 128)
constexpr int PF = 3;                // K steps whose operands are in flight in registers ahead of the one being multiplied

// What one thread holds of a K step that is still on its way to LDS: one row block of A and WPW of W, as loaded
// (Q8_0 stays packed until it is written to LDS, so nothing waits on a fresh load).
struct Stage {
    half8 a[4];
    half8 w16[WPW][4];               // F16 tile, or the column scales of a transposed Q8_0 tile
    uint4v q[WPW][2];                // Q8_0 int8
    uint32_t d[WPW];                 // Q8_0 row scale of this lane's weights: the fp16 bits in a register of their own (two halves
                                     // packed into one register would make the pack wait for the load that was just issued)
};

// kind of weight tile (uniform per wave): 0 F16, 1 Q8_0 row scales, 2 Q8_0 column scales
template <int WF>
__device__ __forceinline__ int tile_kind(const GemmKArgs &g, int nb, int kt)
{
    if (WF == 0) return 0;
    if (WF == 1) return nb < g.W.nbq ? 1 : 0;
    return kt < g.W.kbq ? 2 : 0;
}

template <int WF>
__device__ __forceinline__ void fetch(Stage &s, const GemmKArgs &g, int mb, const int (&nb)[WPW], int kt, int lane)
{
    const half8 *ap = g.A + ((size_t)mb * g.Kb + kt) * 256 + a_lane(lane);
#pragma unroll
    for (int j = 0; j < 4; j++) s.a[j] = ap[j * 64];
#pragma unroll
    for (int u = 0; u < WPW; u++) {
        const int kind = tile_kind<WF>(g, nb[u], kt);
        if (kind == 0) {
            if (WF == 0) load_w_f16(s.w16[u], g.W.w16, nb[u], g.Kb, kt, lane);
            else if (WF == 1) load_w_f16(s.w16[u], g.W.w16, nb[u] - g.W.nbq, g.Kb, kt, lane);
            else load_w_f16(s.w16[u], g.W.w16, nb[u], g.Kb - g.W.kbq, kt - g.W.kbq, lane);
        } else {
            const size_t tile = (size_t)nb[u] * (kind == 1 ? g.Kb : g.W.kbq) + kt;
            const uint4v *q = reinterpret_cast<const uint4v *>(g.W.q) + tile * 128 + lane;
            s.q[u][0] = __builtin_nontemporal_load(&q[0]);
            s.q[u][1] = __builtin_nontemporal_load(&q[64]);
            if (kind == 1) s.d[u] = reinterpret_cast<const uint16_t *>(g.W.d)[tile * 64 + lane];
            else {
                const half8 *sc = reinterpret_cast<const half8 *>(g.W.d + tile * 64 + (lane >> 5) * 32);
#pragma unroll
                for (int j = 0; j < 4; j++) s.w16[u][j] = sc[j];
            }
        }
    }
}

// fp16 weight registers of a fetched tile (Q8_0: int8 * scale, rounded once to fp16)
template <int WF>
__device__ __forceinline__ void unpack(half8 (&w)[4], const Stage &s, int u, int kind)
{
    if (kind == 0) {
#pragma unroll
        for (int j = 0; j < 4; j++) w[j] = s.w16[u][j];
        return;
    }
    const half8 q0 = q8_unpack8(s.q[u][0][0], s.q[u][0][1]), q1 = q8_unpack8(s.q[u][0][2], s.q[u][0][3]);
    const half8 q2 = q8_unpack8(s.q[u][1][0], s.q[u][1][1]), q3 = q8_unpack8(s.q[u][1][2], s.q[u][1][3]);
    if (kind == 1) { const half8 d = bcast8(__builtin_bit_cast(half_t, (uint16_t)s.d[u])); w[0] = q0 * d; w[1] = q1 * d; w[2] = q2 * d; w[3] = q3 * d; }
    else { w[0] = q0 * s.w16[u][0]; w[1] = q1 * s.w16[u][1]; w[2] = q2 * s.w16[u][2]; w[3] = q3 * s.w16[u][3]; }
}

// 1-D grid, block 256; LDS 2 x (4 + 4 WPW) row blocks x 4 KB.
// Wave (wm, wn) owns rows [64 wm, +64) and columns [64 WPW wn, +64 WPW) of the block.
//
// Which block a workgroup takes is chosen for the eight L2 caches: the hardware deals consecutive workgroup ids
// to the XCDs in turn, so id % 8 is the XCD.  Each XCD gets every eighth column of blocks, and the 32 workgroups
// that are resident on it together form an 8 x 4 patch (8 row blocks x 4 column blocks).  They walk K in step, so
// an activation slice fetched into that L2 serves 4 workgroups and a weight slice 8, instead of one each.
template <int WF>
__global__ __launch_bounds__(256) void gemm_big(GemmKArgs g)
{
    extern __shared__ half8 tiles[];                      // [buf][A blocks 0-3 | W blocks 0 .. 4 WPW - 1][j][lane]
    constexpr int NBLK = 4 + 4 * WPW, BUF = NBLK * 256, NW = 2 * WPW;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, h = lane >> 5;
    const int MT = (g.M + 127) >> 7, NT = (g.N + 128 * WPW - 1) / (128 * WPW);
    const int m_patches = (MT + 7) >> 3;
    const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3, patch = seq >> 5, in_patch = seq & 31;
    const int mt = (patch % m_patches) * 8 + (in_patch & 7);
    const int nt = ((patch / m_patches) * 4 + (in_patch >> 3)) * 8 + xcd;
    if (mt >= MT || nt >= NT) return;                     // padding of the patch grid; the whole workgroup leaves
    const int nb0 = nt * 4 * WPW, mb0 = mt * 4;
    const int wm = wave >> 1, wn = wave & 1;
    // the row blocks this wave fetches (clamped: rows past the end are computed and never stored)
    const int mb_ld = min(mb0 + wave, g.Mb - 1);
    int nb_ld[WPW];
#pragma unroll
    for (int u = 0; u < WPW; u++) nb_ld[u] = min(nb0 + wave * WPW + u, g.Nb - 1);

    float16v acc[2][NW];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NW; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    Stage st[PF];                                         // step s travels in st[s % PF]
    auto park = [&](const Stage &s, int kt, half8 *buf) {
#pragma unroll
        for (int j = 0; j < 4; j++) buf[(wave * 4 + j) * 64 + lane] = s.a[j];
#pragma unroll
        for (int u = 0; u < WPW; u++) {
            half8 w[4];
            unpack<WF>(w, s, u, tile_kind<WF>(g, nb_ld[u], kt));
#pragma unroll
            for (int j = 0; j < 4; j++) buf[((4 + wave * WPW + u) * 4 + j) * 64 + lane] = w[j];
        }
    };
    // Every fetch is issued unconditionally (past the end it asks for the last step again): with a fetch under a
    // condition the compiler cannot count how many younger loads are in flight when a stage is parked, and waits for
    // all of them -- the prefetch then hides nothing.
    const int last = g.Kb - 1;
#pragma unroll
    for (int p = 0; p < PF; p++) fetch<WF>(st[p], g, mb_ld, nb_ld, min(p, last), lane);
    park(st[0], 0, tiles);
    __syncthreads();
    // one K step: multiply step kt out of LDS buffer kt & 1 while step kt + 1 is unpacked and parked in the other one
    // and step kt + PF is requested into the slot that step kt left (u = kt % PF, a compile-time constant at every call)
    auto step = [&](int kt, int u) __attribute__((always_inline)) {
        const half8 *cur = tiles + (size_t)(kt & 1) * BUF;
        fetch<WF>(st[u], g, mb_ld, nb_ld, min(kt + PF, last), lane);
        // fp16 image of the next step's weight blocks: plain VALU work with no dependence on this step's MFMAs, placed in
        // the same block of code so that the two interleave (on the last step it unpacks a repeated step and the result
        // lands in the buffer nobody reads any more)
        const Stage &sn = st[(u + 1) % PF];
        half8 wnext[WPW][4];
#pragma unroll
        for (int x = 0; x < WPW; x++) unpack<WF>(wnext[x], sn, x, tile_kind<WF>(g, nb_ld[x], min(kt + 1, last)));
        // operands of K slice j + 1 are read from LDS before the MFMAs of slice j are issued, so the reads run under them
        half8 a[2][2], w[2][NW];
        auto read = [&](int j) {
#pragma unroll
            for (int i = 0; i < 2; i++) a[j & 1][i] = cur[((2 * wm + i) * 4 + j) * 64 + lane];
#pragma unroll
            for (int k = 0; k < NW; k++) w[j & 1][k] = cur[((4 + NW * wn + k) * 4 + j) * 64 + lane];
        };
        read(0);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j + 1 < 4) read(j + 1);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int k = 0; k < NW; k++)
                    acc[i][k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[j & 1][i], w[j & 1][k], acc[i][k], 0, 0, 0);
        }
        half8 *nxt = tiles + (size_t)((kt + 1) & 1) * BUF;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            nxt[(wave * 4 + j) * 64 + lane] = sn.a[j];
#pragma unroll
            for (int x = 0; x < WPW; x++) nxt[((4 + wave * WPW + x) * 4 + j) * 64 + lane] = wnext[x][j];
        }
        // Issue order of the step, one memory instruction in the shadow of each MFMA (a wave is the only one on its SIMD,
        // so whatever is not issued between two MFMAs is paid for on top of them): the 6 LDS reads of slice 0, then per
        // MFMA of slices 0-2 one LDS read of the next slice, the 12 global loads under slices 0-1, the 12 LDS writes
        // under slices 2-3.  Left to itself the scheduler sinks every read to just before its use.
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
        for (int i = 0; i < 32; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (i < 24 && (i & 7) < 6) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (i < 12) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            if (i >= 20) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
        __syncthreads();
    };
    const int full = g.Kb / PF * PF;
    for (int kt0 = 0; kt0 < full; kt0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; u++) step(kt0 + u, u);
    }
#pragma unroll
    for (int u = 0; u < PF - 1; u++) if (full + u < g.Kb) step(full + u, u);

    // D layout of v_mfma_f32_32x32x16: column = lane & 31, row = 8*(v/4) + 4*(lane/32) + v%4
    if (mb0 * 32 + 128 <= g.M && (nb0 + 4 * WPW) * 32 <= g.N) {
        // Block inside the matrix: no bounds tests, so the row factors are all requested at once and the stores follow
        // each other without a wait (a store under a condition makes the compiler drain the queue before every one).
        float sc[2][16];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) sc[i][v] = 1.0f;
        if (g.a_inv_scale) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int v = 0; v < 16; v++)
                    sc[i][v] = g.a_inv_scale[(mb0 + 2 * wm + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3)];
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = (mb0 + 2 * wm + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
                float *row = g.P + (size_t)m * g.ldp + (nb0 + NW * wn) * 32 + r;
#pragma unroll
                for (int k = 0; k < NW; k++) row[k * 32] = acc[i][k][v] * sc[i][v];
            }
        return;
    }
    // a block that reaches past the matrix (EdgeStore): the same stores, without a branch
    uint32_t col[NW];
#pragma unroll
    for (int k = 0; k < NW; k++) { const int n = (nb0 + NW * wn + k) * 32 + r; col[k] = EdgeStore::column(n < g.N, n * 4); }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        float sc[16];
#pragma unroll
        for (int v = 0; v < 16; v++)
            sc[v] = g.a_inv_scale ? g.a_inv_scale[min((mb0 + 2 * wm + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3), g.M - 1)] : 1.0f;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const EdgeStore edge(g.P, (mb0 + 2 * wm + i) * 32 + 8 * (v >> 2), g.M, g.ldp);
#pragma unroll
            for (int k = 0; k < NW; k++) edge.f32(4 * h + (v & 3), col[k], acc[i][k][v] * sc[v]);
        }
    }
}


// The product whose sums are of short parts (of a prompt's rows with what rounding a Q8_0 weight to F16 lost; value and residual rows take
// gemm_big_pair): no more than twelve MFMAs in one accumulator.  The matrix cores round an accumulator at every instruction, so a sum over K = 2560 in one is 2.5 times as far from the exact one as a
// matrix-vector product's (units of 2^-24 of the result's norm, 64 rows: 5.5 against 2.2; K = 9728: 10.5 against 3.9).  Two of the
// eight accumulators of a wave are added to sums of their own in each of four half steps out of six, under the MFMAs of the
// others, and start again from zero.  K goes in half steps of 32 through six buffers: half step hs is multiplied out of buffer hs % 6, in two
// slices of 16; the barrier that ends hs - 1 has found hs and hs + 1 in LDS, slice 0 of hs + 1 is read under the products of slice 1 of hs,
// and hs + 5 is requested into the buffer that hs - 1 left.
__global__ __launch_bounds__(256) void gemm_big_short(GemmKArgs g)
{
    constexpr int HB = 12 * 2 * 64;                       // half8 per buffer: [4 A + 8 W row blocks][2 slices][64 lanes]
    __shared__ half8 lb0[HB], lb1[HB], lb2[HB], lb3[HB], lb4[HB], lb5[HB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, h = lane >> 5;
    const int MT = (g.M + 127) >> 7, NT = (g.N + 255) >> 8;
    const int m_patches = (MT + 7) >> 3;
    int mt, nt, chunk = 0;
    if (g.m_tiles) {
        // few row blocks: those of one (column block, chunk) are consecutive workgroups of one XCD, so a weight tile comes
        // from memory once; the pairs are dealt to the XCDs in turn
        const int slot = blockIdx.x >> 3, pair = (slot / MT) * 8 + (blockIdx.x & 7);
        if (pair >= NT * g.S) return;
        mt = slot % MT; nt = pair % NT; chunk = pair / NT;
    } else if (g.S > 1) {
        const int t = blockIdx.x % (MT * NT);
        chunk = blockIdx.x / (MT * NT); mt = t % MT; nt = t / MT;
    } else {
        const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3, patch = seq >> 5, in_patch = seq & 31;
        mt = (patch % m_patches) * 8 + (in_patch & 7);
        nt = ((patch / m_patches) * 4 + (in_patch >> 3)) * 8 + xcd;
        if (mt >= MT || nt >= NT) return;
    }
    const int nb0 = nt * 8, mb0 = mt * 4;
    const int wm = wave >> 1, wn = wave & 1;
    const int k_beg = chunk * g.steps_per_chunk, nsteps = min(g.Kb, k_beg + g.steps_per_chunk) - k_beg;
    const int nhalf = 2 * nsteps, last = nhalf - 1;
    const half8 *src[3];
    src[0] = g.A + ((size_t)min(mb0 + wave, g.Mb - 1) * g.Kb + k_beg) * 256 + a_lane(lane);
    src[1] = reinterpret_cast<const half8 *>(g.W.w16) + ((size_t)min(nb0 + 2 * wave, g.Nb - 1) * g.Kb + k_beg) * 256 + lane;
    src[2] = reinterpret_cast<const half8 *>(g.W.w16) + ((size_t)min(nb0 + 2 * wave + 1, g.Nb - 1) * g.Kb + k_beg) * 256 + lane;
    const int dst[3] = {wave, 4 + 2 * wave, 5 + 2 * wave};
    float *const Cp = g.P + (size_t)chunk * g.plane_stride;

    float16v acc[2][4], sum[2][4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = sum[i][j][v] = 0.f;

    typedef __attribute__((address_space(3))) void lds_void;
    uint32_t loff[3][2];
#pragma unroll
    for (int u = 0; u < 3; u++)
#pragma unroll
        for (int j = 0; j < 2; j++) loff[u][j] = __builtin_amdgcn_readfirstlane((uint32_t)((dst[u] * 2 + j) * 64 * 16));
    constexpr int LOADS = 3 * 2, AHEAD = 5, LANDED = 2;   // copies per request and wave; requests in flight after a request; how many of them a barrier needs
    constexpr int WAIT = (AHEAD - LANDED) * LOADS;
    static_assert(WAIT == 18 && AHEAD * LOADS < 64, "the hand-written waits count this wave's LDS-direct loads; vmcnt has six bits");
    auto request = [&](half8 (&buf)[HB], int hs) __attribute__((always_inline)) {
        const size_t o = (size_t)(hs >> 1) * 256 + (hs & 1) * 128;
        const uint32_t base = (uint32_t)(uintptr_t)(lds_void *)buf;
#pragma unroll
        for (int u = 0; u < 3; u++)
#pragma unroll
            for (int j = 0; j < 2; j++)                    // LOADS of these
                asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(src[u] + o + j * 64), "s"(base + loff[u][j]) : "m0");
    };
    half8 a0[2], w0[4];
    auto read = [&](half8 (&a)[2], half8 (&w)[4], const half8 (&cur)[HB], int j) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; i++) a[i] = cur[((2 * wm + i) * 2 + j) * 64 + lane];
#pragma unroll
        for (int k = 0; k < 4; k++) w[k] = cur[((4 + 4 * wn + k) * 2 + j) * 64 + lane];
    };
    auto multiply = [&](const half8 (&a)[2], const half8 (&w)[4], int out) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (k == out) {
                    sum[i][k] += acc[i][k];
                    acc[i][k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], w[k], float16v{}, 0, 0, 0);
                } else acc[i][k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], w[k], acc[i][k], 0, 0, 0);
            }
    };
    // (out: the column of accumulators to add to the sums)
    auto step = [&](int hs, int out, const half8 (&cur)[HB], const half8 (&nxt)[HB], half8 (&free_buf)[HB]) __attribute__((always_inline)) {
        request(free_buf, min(hs + 5, last));
        half8 a1[2], w1[4];
        read(a1, w1, cur, 1);
        multiply(a0, w0, out);
        read(a0, w0, nxt, 0);
        multiply(a1, w1, -1);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (i < 4 || (i >= 8 && i < 14)) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        // In flight here: this wave's copies of half steps hs + 1 .. hs + 5, LOADS each, oldest first.  The barrier must find
        // hs + 1 and hs + 2 in LDS, so all but the newest three requests have to have retired (loads retire in order).
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(WAIT) : "memory");
    };
    request(lb0, 0); request(lb1, min(1, last)); request(lb2, min(2, last)); request(lb3, min(3, last)); request(lb4, min(4, last));
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(WAIT) : "memory");   // five requests out: the first two have landed
    read(a0, w0, lb0, 0);
    const int full = nhalf / 6 * 6;
    for (int h0 = 0; h0 < full; h0 += 6) {
        step(h0, 0, lb0, lb1, lb5);
        step(h0 + 1, 1, lb1, lb2, lb0);
        step(h0 + 2, 2, lb2, lb3, lb1);
        step(h0 + 3, 3, lb3, lb4, lb2);
        step(h0 + 4, 4, lb4, lb5, lb3);
        step(h0 + 5, 5, lb5, lb0, lb4);
    }
    if (full < nhalf) step(full, 0, lb0, lb1, lb5);
    if (full + 1 < nhalf) step(full + 1, 1, lb1, lb2, lb0);
    if (full + 2 < nhalf) step(full + 2, 2, lb2, lb3, lb1);
    if (full + 3 < nhalf) step(full + 3, 3, lb3, lb4, lb2);
    if (full + 4 < nhalf) step(full + 4, 4, lb4, lb5, lb3);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) acc[i][k] += sum[i][k];

    if (mb0 * 32 + 128 <= g.M && (nb0 + 8) * 32 <= g.N) {
        float sc[2][16];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int v = 0; v < 16; v++)
                sc[i][v] = g.a_inv_scale ? g.a_inv_scale[(mb0 + 2 * wm + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3)] : 1.0f;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = (mb0 + 2 * wm + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
                float *row = Cp + (size_t)m * g.ldp + (nb0 + 4 * wn) * 32 + r;
#pragma unroll
                for (int k = 0; k < 4; k++) row[k * 32] = acc[i][k][v] * sc[i][v];
            }
        return;
    }
    // a block that reaches past the matrix (EdgeStore): the same stores, without a branch
    uint32_t col[4];
#pragma unroll
    for (int k = 0; k < 4; k++) { const int n = (nb0 + 4 * wn + k) * 32 + r; col[k] = EdgeStore::column(n < g.N, n * 4); }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        float sc[16];
#pragma unroll
        for (int v = 0; v < 16; v++)
            sc[v] = g.a_inv_scale ? g.a_inv_scale[min((mb0 + 2 * wm + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3), g.M - 1)] : 1.0f;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const EdgeStore edge(Cp, (mb0 + 2 * wm + i) * 32 + 8 * (v >> 2), g.M, g.ldp);
#pragma unroll
            for (int k = 0; k < 4; k++) edge.f32(4 * h + (v & 3), col[k], acc[i][k][v] * sc[v]);
        }
    }
}


// F16 weight tiles need no unpacking, so their steps go from L2/HBM straight into LDS and never pass through registers or
// ds_write (walk_k).  BM x 256 outputs per workgroup, four waves of BM / 2 x 128; 256 rows: five buffers of 32 KB, all of a CU's
// 160 KB; 128 rows: six of 24 KB.
//
// What bounds it: the matrix cores' power.  On random operands the clock settles where the power limit is -- 1.5 to 1.75 GHz
// under this loop, 2.4 on constant operands -- so what counts is energy per flop as much as idle cycles.  v_mfma_f32_16x16x32
// takes the K = 32 of a half step at once and moves half the accumulator bytes per flop that 32x32x16 does; its sums are the same, bit for
// bit.  A half step's two slices hold exactly the two fragments of a row block: lane l of the fragment of rows 16 s .. 16 s + 15
// reads slice l >> 5, column half (l >> 4) & 1, row 16 s + (l & 15), conflict-free.  The MFMAs are assembly on accumulators in place (acc_tiles.h). With them pinned, one LDS read
// or one copy goes under every second or third MFMA instead of all copies behind the barrier, where the matrix cores waited for them (a
// K step of 64 took 2 800 cycles for 2 048 of MFMAs, now 2 370).  Random operands, alone: 2048 x 8192 x 9728 312 -> 241 us (1 045 -> 1 354 TFLOP/s), 2048 x 16384 x 2560 188 -> 148,
// 8192^3 988 -> 799 us (1 113 -> 1 375); 16x16x32 with the copies in one burst 264, 174 and 850 us, 32x32x16 with them spread 261, 151, 848.
//
// GROUPED: the row blocks of A belong to different weights of one shape, laid group.stride halves apart: block mt is
// multiplied with number group.of[mt]; only the first group.of[M / BM] blocks have rows.
struct GroupArgs { const int *of; size_t stride; };
template <int BM, bool GROUPED = false>
__global__ __launch_bounds__(256) void gemm_big_f16(GemmKArgs g, GroupArgs group)
{
    constexpr int AB = BM / 32, MI = BM / 32, AU = AB / 4;    // A row blocks of the block; 16-row tiles of a wave; A row blocks a wave fetches
    constexpr int NB = BM == 256 ? 5 : 6;                     // buffers
    __shared__ half8 lds[NB * walk_buffer(BM)];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int MT = (g.M + BM - 1) / BM, NT = (g.N + 255) >> 8;
    const int m_patches = (MT + 7) >> 3;
    int mt, nt, chunk = 0;
    if (GROUPED) {
        // the blocks that have rows, column blocks first, dealt to the XCDs in contiguous shares: the row blocks of a weight
        // meet in one L2, and few column blocks leave no XCD without work
        const int total = group.of[MT] * NT, share = (total + 7) >> 3, seq = blockIdx.x >> 3, t = (blockIdx.x & 7) * share + seq;
        if (seq >= share || t >= total) return;
        mt = t / NT; nt = t % NT;
    } else if (g.m_tiles) {
        // few row blocks: those of one (column block, chunk) are consecutive workgroups of one XCD, so a weight tile comes
        // from memory once; the pairs are dealt to the XCDs in turn
        const int slot = blockIdx.x >> 3, pair = (slot / MT) * 8 + (blockIdx.x & 7);
        if (pair >= NT * g.S) return;
        mt = slot % MT; nt = pair % NT; chunk = pair / NT;
    } else if (g.S > 1) {
        const int t = blockIdx.x % (MT * NT);
        chunk = blockIdx.x / (MT * NT); mt = t % MT; nt = t / MT;
    } else {
        const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3, patch = seq >> 5, in_patch = seq & 31;
        mt = (patch % m_patches) * 8 + (in_patch & 7);
        nt = ((patch / m_patches) * 4 + (in_patch >> 3)) * 8 + xcd;
        if (mt >= MT || nt >= NT) return;
    }
    const int nb0 = nt * 8, mb0 = mt * AB;
    if (GROUPED) g.W.w16 += (size_t)__builtin_amdgcn_readfirstlane(group.of[mt]) * group.stride;
    const int wm = wave >> 1, wn = wave & 1;
    const int k_beg = chunk * g.steps_per_chunk, nhalf = 2 * (min(g.Kb, k_beg + g.steps_per_chunk) - k_beg);
    float *const Cp = g.P + (size_t)chunk * g.plane_stride;
    // this wave's rows of C from m0 on, of which a lane ends with 16 j + mq .. + 3 and their factors; its columns from n0 on, 16 i + nr
    const int m0 = mb0 * 32 + wm * (BM / 2), n0 = (nb0 + 4 * wn) * 32, mq = 4 * (lane >> 4), nr = lane & 15;
    float sc[MI][4];
#pragma unroll
    for (int j = 0; j < MI; j++)
#pragma unroll
        for (int v = 0; v < 4; v++) sc[j][v] = 1.0f;
    if (g.a_inv_scale) {
#pragma unroll
        for (int j = 0; j < MI; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) sc[j][v] = g.a_inv_scale[min(m0 + 16 * j + mq + v, g.M - 1)];
    }

    // this wave's share of a half step: both slices of A row blocks w (, 4 + w) and of W row blocks w, 4 + w (clamped: rows past
    // the end are computed and never stored), as uniform bases and one lane offset per operand
    uint64_t src[AU + 2];
#pragma unroll
    for (int u = 0; u < AU; u++) src[u] = uniform_address(g.A + ((size_t)min(mb0 + 4 * u + wave, g.Mb - 1) * g.Kb + k_beg) * 256);
#pragma unroll
    for (int u = 0; u < 2; u++)
        src[AU + u] = uniform_address(reinterpret_cast<const half8 *>(g.W.w16) + ((size_t)min(nb0 + 4 * u + wave, g.Nb - 1) * g.Kb + k_beg) * 256);
    walk_k<BM, NB>(lds, src, a_lane(lane) * 16, nhalf);

    if (mb0 * 32 + BM <= g.M && (nb0 + 8) * 32 <= g.N) {      // a block inside the matrix: stores without tests
        unrolled<MI>([&](auto J) __attribute__((always_inline)) {
            float *const row = Cp + (size_t)(m0 + 16 * J + mq) * g.ldp + n0 + nr;
            unrolled<8>([&](auto I) __attribute__((always_inline)) {
                const float4v x = AccTile<I * MI + J>::take();
#pragma unroll
                for (int v = 0; v < 4; v++) row[(size_t)v * g.ldp + 16 * I] = x[v] * sc[J][v];
            });
        });
        return;
    }
    // a block that reaches past the matrix (EdgeStore): the same stores, without a branch
    unrolled<MI>([&](auto J) __attribute__((always_inline)) {
        const EdgeStore edge(Cp, m0 + 16 * J, g.M, g.ldp, 16);
        unrolled<8>([&](auto I) __attribute__((always_inline)) {
            const int n = n0 + 16 * I + nr;
            const uint32_t col = EdgeStore::column(n < g.N, n * 4);
            const float4v x = AccTile<I * MI + J>::take();
#pragma unroll
            for (int v = 0; v < 4; v++) edge.f32(mq + v, col, x[v] * sc[J][v]);
        });
    });
}

// The product of operands that hold more than fp16: row m of A as a value row m and a residual row lo + m that holds 2^11 times what
// rounding the value row lost, in units of the same factor (lo a multiple of 32).  A block of 128 rows and 256 columns is a 256 x 256
// block of gemm_big_f16 whose lower rows are the upper ones' residuals, so one wave ends with both products of an element and stores their
// sum times the row's factor: one value where two rows' planes went to memory and came back.
//
// The matrix cores round an accumulator at every instruction of K = 16 (this one rounds twice), so no sum of more than twelve such steps stays
// in one: in each of six half steps one or two of the eight columns of a wave's value tiles are added to sums in vector
// registers -- two instructions an entry, under the MFMAs before the tile begins anew -- and the residual's tiles, 2^-11 of the result, stay.
// (K = 2560, 64 rows, units of 2^-24 of the result's norm: 5.5 in one sum, 2.2 as a matrix-vector product forms it; K = 9728 10.5 and 3.9.)
// The K steps of all column blocks stand in one row, and each team of workgroups (one per row block) takes an equal run of them, so no last round
// of blocks is half empty: 304 blocks of 40 steps on 256 CUs are 48 steps for each instead of 80.  What a run holds of a column block is a piece
// of it, and the n-th piece goes to plane n (PairWalk): a column block has as many planes as teams had a part in it.
// The sums leave 96 registers for fragments: W is read in place behind the last MFMA that takes it, which keeps a half step's buffer in use
// while it is multiplied, so the ring runs a half step less ahead than gemm_big_f16's.
constexpr int PAIR_PERIOD = 6;
constexpr int pair_flush(int phase, int n) { constexpr int f[6][2] = {{0, -1}, {2, 4}, {1, -1}, {3, 6}, {5, -1}, {7, -1}}; return f[phase][n]; }
// the slot (MFMA of 64) ahead of which register u of the sixteen of a column's four value tiles is added to its sum: column f's tiles begin anew in
// the slots 8 f + 4 ..
constexpr int pair_slot(int f, int u) { return f == 0 ? u * 7 / 16 : (8 * f - 12 + u > 0 ? 8 * f - 12 + u : 0); }
__global__ __launch_bounds__(256) void gemm_big_pair(GemmKArgs g, int lo)
{
    constexpr int HB = 16 * 128, NB = 5;                      // half8 per buffer: [4 value A + 4 residual A + 8 W row blocks][2 slices][64]; buffers
    __shared__ half8 lds[NB * HB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // the row blocks of a team are consecutive workgroups of one XCD and walk K together, so a weight tile comes from memory once; the
    // teams are dealt to the XCDs in turn
    const int MT = (g.M + 127) >> 7, slot = blockIdx.x >> 3, team = (slot / MT) * 8 + (blockIdx.x & 7);
    const int mb0 = (slot % MT) * 4, wm = wave >> 1, wn = wave & 1;
    const int m0 = mb0 * 32 + wm * 64, mq = 4 * (lane >> 4), nr = lane & 15;
    const PairWalk walk{g.steps_per_chunk, g.Kb};
    const int begin = team * walk.steps;                      // of the K steps of all column blocks, one behind the other
    int at = begin;
    const int end = min(begin + walk.steps, ((g.N + 255) >> 8) * g.Kb);
    if (at >= end) return;

    // this wave's share of a half step: both slices of a value, its residual and two W row blocks (clamped: rows past the end
    // are computed and never stored), as uniform bases and one lane offset per operand
    const int ab = min(mb0 + wave, g.Mb - 1);
    const half8 *const w16 = reinterpret_cast<const half8 *>(g.W.w16);
    uint64_t src[4];
    const uint32_t a_off = a_lane(lane) * 16, w_off = lane * 16;
    typedef __attribute__((address_space(3))) void lds_void;
    const uint32_t place0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void *)lds + wave * 2048);
    constexpr int COPIES = 8;                                 // of 1 KB, per half step and wave
    constexpr int WAIT = (NB - 3) * COPIES;                   // all requests but the newest NB - 3 have landed (loads retire in order)
    static_assert((NB - 1) * COPIES < 64, "the hand-written waits count this wave's LDS-direct loads; vmcnt has six bits");
    auto copy = [&](uint32_t place, uint32_t koff, int c) __attribute__((always_inline)) {
        const int u = c >> 1;
        const uint32_t off = (u < 2 ? a_off : w_off) + koff;
        if (c & 1) asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024" :: "v"(off), "s"(src[u]), "s"(place), "n"(u * 8192) : "m0", "scc");
        else asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(off), "s"(src[u]), "s"(place), "n"(u * 8192) : "m0", "scc");
    };
    const half8 *const frag = lds + (lane >> 5) * 64 + ((lane >> 4) & 1) * 32 + (lane & 15);
    const half8 *const fa = frag + 2 * wm * 128, *const fw = frag + (8 + 4 * wn) * 128;
    auto read_a = [&](int t, int buf) __attribute__((always_inline)) { return fa[buf + (t >> 2) * 512 + ((t & 3) >> 1) * 128 + (t & 1) * 16]; };   // t < 4: values
    auto read_w = [&](int t, int buf) __attribute__((always_inline)) { return fw[buf + (t >> 1) * 128 + (t & 1) * 16]; };

    // the piece that begins at step `p`: column block, first step of it, half steps less one
    int nt = 0, k_beg = 0, last = 0;
    auto enter = [&](int p) __attribute__((always_inline)) {
        nt = p / g.Kb; k_beg = p - nt * g.Kb;
        last = 2 * min(g.Kb - k_beg, end - p) - 1;
        src[0] = uniform_address(g.A + ((size_t)ab * g.Kb + k_beg) * 256);
        src[1] = uniform_address(g.A + ((size_t)(ab + (lo >> 5)) * g.Kb + k_beg) * 256);
#pragma unroll
        for (int u = 0; u < 2; u++) src[2 + u] = uniform_address(w16 + ((size_t)min(nt * 8 + 4 * u + wave, g.Nb - 1) * g.Kb + k_beg) * 256);
#pragma unroll
        for (int h = 0; h < NB - 1; h++)
#pragma unroll
            for (int c = 0; c < COPIES; c++) copy(place0 + h * HB * 16, (uint32_t)min(h, last) * 2048, c);
    };
    float sum[8][4][4];
    half8 A0[8], A1[8], W[8];
    // Half step hs out of the buffer at `cur` (A in A, W but its last in W), the next one's fragments out of `nxt`; hs + NB - 1 goes to
    // `place`, the buffer of hs - 1.  Tile 8 i + j: value rows 16 j, W rows 16 i; 8 i + 4 + j: their residuals.
    auto step = [&](auto phase, const half8 (&A)[8], half8 (&An)[8], int hs, int cur, int nxt, uint32_t place) __attribute__((always_inline)) {
        constexpr int P = decltype(phase)::value;
        const uint32_t koff = (uint32_t)min(hs + NB - 1, last) * 2048;
        unrolled<64>([&](auto X) __attribute__((always_inline)) {
            constexpr int x = X, i = x / 8, jj = x % 8, j = jj % 4;
            if constexpr (jj == 1) { if constexpr (i > 0) W[i - 1] = read_w(i - 1, nxt); else W[7] = read_w(7, cur); __builtin_amdgcn_sched_barrier(0); }
            if constexpr (jj == 3) copy(place, koff, i);
            if constexpr (jj == 5) { An[i] = read_a(i, nxt); __builtin_amdgcn_sched_barrier(0); }
            unrolled<32>([&](auto U) __attribute__((always_inline)) {
                constexpr int f = pair_flush(P, U / 16), u = U % 16;
                if constexpr (f >= 0 && pair_slot(f, u) == x) sum[f][u / 4][u % 4] += AccTile<8 * f + u / 4>::template take_one<u % 4>();
            });
            if constexpr (jj < 4) AccTile<8 * i + 4 + j>::add(A[4 + j], W[i]);
            else if constexpr (i == pair_flush(P, 0) || i == pair_flush(P, 1)) AccTile<8 * i + j>::begin(A[j], W[i]);
            else AccTile<8 * i + j>::add(A[j], W[i]);
        });
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(WAIT) : "memory");   // (what was read of the buffer that goes next has been multiplied)
    };
    enter(at);
    for (;;) {
        const int nhalf = last + 1;
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) sum[i][j][v] = 0.f;
        unrolled<64>([](auto X) __attribute__((always_inline)) { AccTile<X>::clear(); });
        // NB - 1 requests are out and the first two have landed: in a later piece they are older than the 128 stores of the one before
        if (at == begin) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(WAIT) : "memory");
        else asm volatile("s_waitcnt vmcnt(63)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int t = 0; t < 8; t++) A0[t] = read_a(t, 0);
#pragma unroll
        for (int t = 0; t < 7; t++) W[t] = read_w(t, 0);
        int cur = 0, nxt = HB, hs = 0;
        uint32_t place = place0 + (NB - 1) * HB * 16;
        auto two = [&](auto phase) __attribute__((always_inline)) {
            auto advance = [&]() __attribute__((always_inline)) {
                cur = nxt;
                nxt = nxt == (NB - 1) * HB ? 0 : nxt + HB;
                place = place == place0 + (NB - 1) * HB * 16 ? place0 : place + HB * 16;
            };
            step(phase, A0, A1, hs, cur, nxt, place); advance();
            step(std::integral_constant<int, decltype(phase)::value + 1>{}, A1, A0, hs + 1, cur, nxt, place); advance();
            hs += 2;
        };
        const int full = nhalf / PAIR_PERIOD * PAIR_PERIOD;
        while (hs < full) { two(std::integral_constant<int, 0>{}); two(std::integral_constant<int, 2>{}); two(std::integral_constant<int, 4>{}); }
        if (hs < nhalf) two(std::integral_constant<int, 0>{});
        if (hs < nhalf) two(std::integral_constant<int, 2>{});
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        settle_tiles();

        float *const Cp = g.P + (size_t)walk.piece(team, nt) * g.plane_stride;
        const int nb0 = nt * 8, n0 = (nb0 + 4 * wn) * 32;
        int ld = g.ldp, mr = m0 + mq;
        asm volatile("" : "+s"(ld), "+v"(mr));                // (the addresses are formed here, not kept in registers that the loop has no room for)
        float sc[4][4];
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) sc[j][v] = g.a_inv_scale[min(mr + 16 * j + v, g.M - 1)];
#pragma unroll
        for (int j = 0; j < 4; j++) asm volatile("" : "+v"(sc[j][0]), "+v"(sc[j][1]), "+v"(sc[j][2]), "+v"(sc[j][3]));   // (here, ahead of the copies, which the compiler would wait for with them)
        // the next piece's operands come while this one's sums leave (every wave is behind the last barrier: the buffers are free)
        at += nhalf / 2;
        if (at < end) enter(at);
        auto value = [&](auto J, auto I, float (&y)[4]) __attribute__((always_inline)) {
            const float4v h = AccTile<8 * I + J>::take(), l = AccTile<8 * I + 4 + J>::take();
#pragma unroll
            for (int v = 0; v < 4; v++) y[v] = fmaf(l[v], 1.0f / PAIR_RESIDUAL_SCALE, sum[I][J][v] + h[v]) * sc[J][v];
        };
        if (mb0 * 32 + 128 <= g.M && (nb0 + 8) * 32 <= g.N) { // a block inside the matrix: stores without tests
            unrolled<4>([&](auto J) __attribute__((always_inline)) {
                float *const row = Cp + (size_t)(mr + 16 * J) * ld + n0 + nr;
                unrolled<8>([&](auto I) __attribute__((always_inline)) {
                    float y[4];
                    value(J, I, y);
#pragma unroll
                    for (int v = 0; v < 4; v++) row[(size_t)v * ld + 16 * I] = y[v];
                });
            });
        } else {                                              // a block that reaches past the matrix (EdgeStore): the same stores, without a branch
            unrolled<4>([&](auto J) __attribute__((always_inline)) {
                const EdgeStore edge(Cp, m0 + 16 * J, g.M, ld, 16);
                unrolled<8>([&](auto I) __attribute__((always_inline)) {
                    const int n = n0 + 16 * I + nr;
                    const uint32_t col = EdgeStore::column(n < g.N, n * 4);
                    float y[4];
                    value(J, I, y);
#pragma unroll
                    for (int v = 0; v < 4; v++) edge.f32(mq + v, col, y[v]);
                });
            });
        }
        if (at >= end) return;
    }
}

// The 256 x 256 block over Q8_0 weight tiles that stay quantised all the way into LDS: the dequant-fused product for
// many activation rows.  A half step of a weight row block is ONE 1 KB piece (16 int8 per lane: both 8-value slices), its
// 64 fp16 scales another 128 bytes, so a block's half step is 16 KB of activations + 8 KB of weights instead of 32 KB and
// six buffers fit; the copies are LDS-direct loads as in gemm_big_f16<256> (the scales as one dword per lane, lanes 32-63
// fetching the same 128 bytes again into the second half of a 256-byte slot, which keeps every lane active and inside
// the array).  A wave unpacks its fragments on the way from LDS to the MFMA: bytes to exact fp16 integers with
// v_perm_b32, times the scale with packed fp16 multiplies -- the values an F16 image of the dequantised weight holds.
// WF 1: scales per (row, 32 columns), all row blocks of the launch Q8_0 (the caller gives F16 row blocks to another
// launch).  WF 2: the transposed image, scales per (column, 32 rows); K steps from W.kbq on are F16 tiles (the adapter
// rows of the fused QKV weight): at most a step or two at the end of K, multiplied straight from memory after the loop.
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
// BM: rows of the block.  The launcher uses 256 (four waves of 128 x 128); with 128 (four waves of 64 x 128) a wave unpacks
// as many weight fragments for half as many MFMAs, and 192 such blocks took 68 us where the F16 kernel's take 45.
// TAIL (WF 1): the launch has a column block of F16 tiles at its end (only then does the loop carry that case).
template <int WF, int BM, bool TAIL = false>
__global__ __launch_bounds__(256) void gemm_big_q8(GemmKArgs g)
{
    constexpr int AB = BM / 32, MI = BM / 64, AU = BM / 128;  // A row blocks per block; accumulator tile rows and A pieces per wave
    // LDS-direct copies a wave issues per request (2 per A piece; 2 weight pieces + 2 scale pieces, or 4 F16 pieces), requests
    // in flight after a request (six buffers), and how many of them a barrier needs in LDS: the hand-written waits below
    constexpr int Q8_LOADS = 2 * AU + 4, Q8_AHEAD = 5, Q8_LANDED = 2, Q8_WAIT = (Q8_AHEAD - Q8_LANDED) * Q8_LOADS;
    static_assert(Q8_WAIT == (BM == 256 ? 24 : 18) && Q8_AHEAD * Q8_LOADS < 64, "the waits count this wave's LDS-direct loads; vmcnt has six bits");
    constexpr int HB = (2 * AB + 8) * 64;                 // 16-byte units per buffer: A [AB blocks][2 slices][64], Wq [8 blocks][64]
    __shared__ uint4v lb0[HB], lb1[HB], lb2[HB], lb3[HB], lb4[HB], lb5[HB];
    __shared__ half_t scl[6][8][128];                      // scales of the weight row blocks of the half step in buffer i
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, h = lane >> 5;
    const int MT = (g.M + BM - 1) / BM, NT = (g.N + 255) >> 8;
    const int m_patches = (MT + 7) >> 3;
    int mt, nt, chunk = 0;
    if (g.S > 1) {
        const int t = blockIdx.x % (MT * NT);
        chunk = blockIdx.x / (MT * NT); mt = t % MT; nt = t / MT;
    } else {
        const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3, patch = seq >> 5, in_patch = seq & 31;
        mt = (patch % m_patches) * 8 + (in_patch & 7);
        nt = ((patch / m_patches) * 4 + (in_patch >> 3)) * 8 + xcd;
        if (mt >= MT || nt >= NT) return;
    }
    const int nb0 = nt * 8, mb0 = mt * AB;
    const int wm = wave >> 1, wn = wave & 1;
    const int k_beg = chunk * g.steps_per_chunk, k_end = min(g.Kb, k_beg + g.steps_per_chunk);
    const int kq_end = WF == 2 ? min(k_end, g.W.kbq) : k_end;              // Q8_0 steps of this chunk: [k_beg, kq_end)
    const int nsteps = kq_end - k_beg, nhalf = 2 * nsteps, last = nhalf - 1;
    const int kstride = WF == 2 ? g.W.kbq : g.Kb;                           // K blocks per row block of the Q8_0 tile arrays
    // A column block from row block W.nbq on holds F16 tiles (WF 1: the adapter rows at the end of the fused QKV weight;
    // W.nbq is a multiple of 8 and at most one row block follows it, the rest of the block lies outside the matrix): its
    // one row block travels as two 1 KB slices per half step in the places of a piece and a scale copy.
    const bool f16_cols = TAIL && WF == 1 && nb0 >= g.W.nbq;
    // this wave's share of a half step: both slices of A row blocks w (, 4 + w); the piece and the scales of W row blocks w, 4 + w
    const uint4v *asrc[AU], *qsrc[2];
    const uint32_t *dsrc[2];
#pragma unroll
    for (int u = 0; u < AU; u++)
        asrc[u] = reinterpret_cast<const uint4v *>(g.A) + ((size_t)min(mb0 + 4 * u + wave, g.Mb - 1) * g.Kb + k_beg) * 256 + a_lane(lane);
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const size_t tile0 = (size_t)min(nb0 + 4 * u + wave, (WF == 1 ? min(g.Nb, g.W.nbq) : g.Nb) - 1) * kstride + k_beg;
        qsrc[u] = reinterpret_cast<const uint4v *>(g.W.q) + tile0 * 128 + lane;
        dsrc[u] = reinterpret_cast<const uint32_t *>(g.W.d + tile0 * 64) + (lane & 31);
    }
    const uint4v *fsrc = f16_cols ? reinterpret_cast<const uint4v *>(g.W.w16) + ((size_t)min(nb0 - g.W.nbq, g.Nb - g.W.nbq - 1) * g.Kb + k_beg) * 256 + lane : nullptr;
    float *const Cp = g.P + (size_t)chunk * g.plane_stride;

    float16v acc[MI][4];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    typedef __attribute__((address_space(3))) void lds_void;
    uint32_t aoff[AU][2], qoff[2], doff[2];                // byte offsets of this wave's pieces inside a buffer / a scale slot
#pragma unroll
    for (int u = 0; u < AU; u++)
#pragma unroll
        for (int j = 0; j < 2; j++) aoff[u][j] = __builtin_amdgcn_readfirstlane((uint32_t)((((4 * u + wave) * 2 + j) * 64) * 16));
#pragma unroll
    for (int u = 0; u < 2; u++) {
        qoff[u] = __builtin_amdgcn_readfirstlane((uint32_t)((2 * AB * 64 + (4 * u + wave) * 64) * 16));
        doff[u] = __builtin_amdgcn_readfirstlane((uint32_t)((4 * u + wave) * 256));
    }
    const uint32_t scl0 = (uint32_t)(uintptr_t)(lds_void *)&scl[0][0][0];
    auto request = [&](uint4v (&buf)[HB], int slot, int hs) __attribute__((always_inline)) {
        const int kt = hs >> 1, jh = hs & 1;
        const uint32_t base = (uint32_t)(uintptr_t)(lds_void *)buf, sbase = scl0 + (uint32_t)slot * (8 * 256);
#pragma unroll
        for (int u = 0; u < AU; u++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(asrc[u] + (size_t)kt * 256 + (2 * jh + j) * 64), "s"(base + aoff[u][j]) : "m0");
        if (f16_cols) {                                    // the same four copies: slice j of the F16 row block into W place w (j = 0) / 4 + w (j = 1)
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(fsrc + (size_t)kt * 256 + (2 * jh + j) * 64), "s"(base + qoff[j]) : "m0");
        } else {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(qsrc[u] + (size_t)kt * 128 + jh * 64), "s"(base + qoff[u]) : "m0");
                asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" :: "v"(dsrc[u] + (size_t)kt * 32), "s"(sbase + doff[u]) : "m0");
            }
        }
    };
    half8 a0[MI], w0[4];                                   // fragments of slice 0 of the half step about to be multiplied
    // slice j (0 / 1) of the half step in `cur` / scale slot `slot`: A as it lies, W unpacked
    auto read = [&](half8 (&a)[MI], half8 (&w)[4], const uint4v (&cur)[HB], int slot, int jh, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MI; i++) a[i] = __builtin_bit_cast(half8, cur[((MI * wm + i) * 2 + j) * 64 + lane]);
        if (f16_cols) {                                    // (wave 0's copies; every fragment of the block is that one row block)
#pragma unroll
            for (int k = 0; k < 4; k++) w[k] = __builtin_bit_cast(half8, cur[2 * AB * 64 + (j ? 4 : 0) * 64 + lane]);
            return;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int blk = 4 * wn + k;
            const uint2v q = reinterpret_cast<const uint2v *>(&cur[2 * AB * 64 + blk * 64 + lane])[j];
            half8 sc;
            if (WF == 1) sc = bcast8(scl[slot][blk][lane]);
            else sc = reinterpret_cast<const half8 *>(&scl[slot][blk][0])[h * 4 + 2 * jh + j];
            w[k] = q8_unpack8(q[0], q[1]) * sc;
        }
    };
    auto multiply = [&](const half8 (&a)[MI], const half8 (&w)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int k = 0; k < 4; k++) acc[i][k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], w[k], acc[i][k], 0, 0, 0);
    };
    // Half step hs is multiplied out of buffer hs % 6, as in gemm_big_short: the barrier that ends half step hs - 1 has
    // found hs and hs + 1 in LDS, slice 0 of hs + 1 is read and unpacked while slice 1 of hs is multiplied, hs + 5 is
    // requested into the buffer hs - 1 left.  Eight copies per wave and half step.
    auto step = [&](int hs, const uint4v (&cur)[HB], int slot, const uint4v (&nxt)[HB], int nslot, uint4v (&free_buf)[HB], int fslot)
        __attribute__((always_inline)) {
        request(free_buf, fslot, min(hs + 5, last));
        half8 a1[MI], w1[4];
        read(a1, w1, cur, slot, hs & 1, 1);
        multiply(a0, w0);
        read(a0, w0, nxt, nslot, (hs + 1) & 1, 0);
        multiply(a1, w1);
        // in flight: this wave's copies of hs + 1 .. hs + 5, Q8_LOADS each; hs + 1 and hs + 2 must have landed
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(Q8_WAIT) : "memory");
    };
    if (nhalf > 0) {
        request(lb0, 0, 0); request(lb1, 1, min(1, last)); request(lb2, 2, min(2, last)); request(lb3, 3, min(3, last));
        request(lb4, 4, min(4, last));
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(Q8_WAIT) : "memory");   // five requests out: the first two have landed
        read(a0, w0, lb0, 0, 0, 0);
        const int full = nhalf / 6 * 6;
        for (int h0 = 0; h0 < full; h0 += 6) {
            step(h0, lb0, 0, lb1, 1, lb5, 5);
            step(h0 + 1, lb1, 1, lb2, 2, lb0, 0);
            step(h0 + 2, lb2, 2, lb3, 3, lb1, 1);
            step(h0 + 3, lb3, 3, lb4, 4, lb2, 2);
            step(h0 + 4, lb4, 4, lb5, 5, lb3, 3);
            step(h0 + 5, lb5, 5, lb0, 0, lb4, 4);
        }
        if (full < nhalf) step(full, lb0, 0, lb1, 1, lb5, 5);
        if (full + 1 < nhalf) step(full + 1, lb1, 1, lb2, 2, lb0, 0);
        if (full + 2 < nhalf) step(full + 2, lb2, 2, lb3, 3, lb1, 1);
        if (full + 3 < nhalf) step(full + 3, lb3, 3, lb4, 4, lb2, 2);
        if (full + 4 < nhalf) step(full + 4, lb4, 4, lb5, 5, lb3, 3);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    if (WF == 2) {
        // the F16 K steps at the end of this chunk (adapter rows): operands straight from memory
        for (int kt = max(kq_end, k_beg); kt < k_end; kt++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                half8 a[MI], w[4];
#pragma unroll
                for (int i = 0; i < MI; i++) a[i] = g.A[((size_t)min(mb0 + MI * wm + i, g.Mb - 1) * g.Kb + kt) * 256 + j * 64 + a_lane(lane)];
#pragma unroll
                for (int k = 0; k < 4; k++)
                    w[k] = reinterpret_cast<const half8 *>(g.W.w16)[((size_t)min(nb0 + 4 * wn + k, g.Nb - 1) * (g.Kb - g.W.kbq) + kt - g.W.kbq) * 256 + j * 64 + lane];
                multiply(a, w);
            }
        }
    }

    if (mb0 * 32 + BM <= g.M && (nb0 + 8) * 32 <= g.N) {   // a block inside the matrix: stores without tests, factors first
        float sc[MI][16];
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int v = 0; v < 16; v++)
                sc[i][v] = g.a_inv_scale ? g.a_inv_scale[(mb0 + MI * wm + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3)] : 1.0f;
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = (mb0 + MI * wm + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
                float *row = Cp + (size_t)m * g.ldp + (nb0 + 4 * wn) * 32 + r;
#pragma unroll
                for (int k = 0; k < 4; k++) row[k * 32] = acc[i][k][v] * sc[i][v];
            }
        return;
    }
    // a block that reaches past the matrix (EdgeStore): the same stores, without a branch
    uint32_t col[4];
#pragma unroll
    for (int k = 0; k < 4; k++) { const int n = (nb0 + 4 * wn + k) * 32 + r; col[k] = EdgeStore::column(n < g.N, n * 4); }
#pragma unroll
    for (int i = 0; i < MI; i++) {
        float sc[16];
#pragma unroll
        for (int v = 0; v < 16; v++)
            sc[v] = g.a_inv_scale ? g.a_inv_scale[min((mb0 + MI * wm + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3), g.M - 1)] : 1.0f;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const EdgeStore edge(Cp, (mb0 + MI * wm + i) * 32 + 8 * (v >> 2), g.M, g.ldp);
#pragma unroll
            for (int k = 0; k < 4; k++) edge.f32(4 * h + (v & 3), col[k], acc[i][k][v] * sc[v]);
        }
    }
}

}  // namespace

// Products of 65 to 1023 rows on F16 tiles: which of the three kernels, and how many K chunks.  None of them wins over the
// whole range -- the streaming kernel pulls every activation tile through each CU's registers (1.65 us per GFLOP), the large-M
// blocks pay for their prologue, for CUs without a block and for rows a block does not have -- so the planner adds up what each
// would take and picks the least.  Microseconds, fitted on MI355X to 16 shapes (1152 .. 32768 columns, K 1024 .. 32768; Qwen3-4B and
// Gemma3-1B layers forward and backward) at 72 .. 1000 rows with cold weights, 5 to 8 % rms; a plane's bytes count once more for
// the consumer that reads them.  The choice is within 2 % of the best of all measured ones over these shapes, 34 % below the
// streaming kernel alone: 6176 x 2560 at 250 rows 26.7 -> 19.5 us, 19456 x 2560 64 -> 36, 2560 x 19456 at 500 rows 102 -> 56.
namespace {
struct MidPlan { int big, wide, chunks; };
double mid_big_us(int wide, int M, int N, int K, int S, int cus)
{
    const int bm = wide ? 256 : 128, Kb = tiled_kb(K), steps = (Kb + S - 1) / S;
    S = (Kb + steps - 1) / steps;
    const long mt = (M + bm - 1) / bm, nt = (N + 255) / 256, per_xcd = ((nt * S + 7) / 8) * mt;    // (the dealing of m_tiles below)
    const long rounds = (per_xcd + cus / 8 - 1) / (cus / 8);
    const double busy = (double)(mt * nt * S) / ((double)rounds * cus), plane_mb = (double)S * M * N * 4e-6;
    if (wide) return 1.6 + rounds * (7.5 + steps * (1.04 + 0.65 * busy)) + (0.144 + 0.2) * plane_mb;
    return 3.9 + rounds * (2.6 + steps * (0.73 + 0.23 * busy)) + (0.23 + 0.2) * plane_mb;
}
// the pair kernel with `steps` K steps per team: a step 1.0 to 1.5 us by how many CUs work, 6 us per piece of a team
double pair_us(int M, int N, int K, int steps, int cus)
{
    const int Kb = tiled_kb(K), mt = (M + 127) / 128, nt = (N + 255) / 256;
    const long teams = ((long)nt * Kb + steps - 1) / steps;
    const double busy = (double)teams * mt / cus, plane_mb = ((double)Kb / steps + (Kb % steps ? 1.0 : 0.0)) * M * N * 4e-6;
    return 1.6 + 6.0 * PairWalk{steps, Kb}.pieces() + steps * (1.04 + 0.45 * busy) + (0.144 + 0.2) * plane_mb;
}
MidPlan mid_plan(int M, int N, int K, bool one_plane)
{
    const int cus = num_cus() > 0 ? num_cus() : 256, Kb = tiled_kb(K);
    const GemmPlan t = plan_gemm(M, N, K);
    // (a single plane from a streaming product that leaves several: one more pass over them)
    double best = 5.1 + 0.152 * (2e-6 * N * K) + 1.65 * (2e-9 * M * N * K) + (0.115 + (one_plane && t.S == 1 ? 0.0 : 0.2)) * (4e-6 * t.S * M * N);
    MidPlan p{0, 0, 1};
    for (int wide = 0; wide < 2; wide++)
        for (int S = 1; S <= (one_plane ? 1 : 20) && S * 4 <= Kb; S++) {
            const double us = mid_big_us(wide, M, N, K, S, cus) - (one_plane ? 0.2 * (4e-6 * M * N) : 0.0);
            if (us < best) { best = us; p = MidPlan{1, wide, S}; }
        }
    return p;
}
bool mid_rows(int M, int fmt) { return fmt == 0 && M > 64 && M < 1024; }
}  // namespace
bool mid_takes_big(int M, int N, int K, bool one_plane) { return mid_plan(M, N, K, one_plane).big != 0; }

// How many K chunks the large-M kernel should cut a product with F16 tiles into: three when its 128 x 256 output blocks
// would leave a third of the CUs or more without work and K is at least 4096, else one.  Measured on MI355X at 2048
// rows: the products with 2560 output columns (160 blocks for 256 CUs) go from 66 / 140 / 281 / 93 us to 54 / 103 /
// 199 / 73 us (K = 4096 / 9728 / 19456 / 6176) with three chunks dealt evenly to the XCDs; two chunks change nothing
// (320 blocks are two rounds again) and every product with K = 2560 loses (13 K steps per workgroup).
int big_gemm_chunks(int M, int N, int K, int fmt)
{
    if (fmt != 0 || g_big_split == 0) return 1;
    if (g_big_split > 1) return g_big_split;
    if (mid_rows(M, fmt)) return mid_plan(M, N, K, false).chunks;
    const long blocks = (long)((M + 127) / 128) * ((N + 128 * WPW - 1) / (128 * WPW));
    const int cus = num_cus() > 0 ? num_cus() : 256;
    // a handful of blocks over a very long K (the LM head's backward at a few hundred rows: 25 blocks, K = 262 144): as
    // many chunks as it takes to give every CU a block, each still thousands of columns long (640 rows: 930 us on the
    // streaming kernel, 3 680 / 1 340 / 840 / 640 us with 1 / 3 / 5 / 8-10 chunks)
    if (blocks * 8 <= cus && K >= 65536) return (int)std::min<long>(std::min<long>(cus / blocks, K / 8192), 16);
    return (blocks * 3 <= cus * 2 && K >= 4096) ? 3 : 1;
}

// Whether a Q8_0 operand can run on gemm_big_q8: the row blocks of a row-scaled operand all quantised, or one F16 row
// block (the adapter rows of the fused QKV weight) that begins a column block of its own; at most two F16 K steps at the
// end of a column-scaled one.
bool q8_wide_ok(const WeightOp &W, int N, int K)
{
    if (g_big_block == 1) return false;
    if (W.fmt == 1) return W.nbq >= tiled_rb(N) || (W.nbq % 8 == 0 && tiled_rb(N) - W.nbq == 1 && W.w16);
    if (W.fmt == 2) return W.kbq >= 1 && tiled_kb(K) - W.kbq <= 2;
    return false;
}

// K chunks for any operand: big_gemm_chunks for F16 tiles; for Q8_0 tiles on the 256 x 256 block, two or three chunks
// where they fill at least half as many CUs again as one does (each chunk 20 K steps or more), else one.
int big_gemm_chunks_for(int M, int N, int K, const WeightOp &W)
{
    if (W.fmt == 0) return big_gemm_chunks(M, N, K, 0);
    if (g_big_split == 0 || !q8_wide_ok(W, N, K)) return 1;
    if (g_big_split > 1) return g_big_split;
    const int cus = num_cus() > 0 ? num_cus() : 256;
    const long blocks = (long)((M + 255) / 256) * ((N + 255) / 256);
    auto share = [&](int c) { return (double)(blocks * c) / (double)((blocks * c + cus - 1) / cus * cus); };
    int best = 1;
    for (int c = 2; c <= 3; c++)
        if (tiled_kb(K) / c >= 20 && share(c) >= 1.5 * share(1) && share(c) > share(best)) best = c;
    return best;
}

int launch_gemm_big(const half_t *A, const float *a_inv_scale, const WeightOp &W, float *C, int ldc, int M, int N, int K,
                    int chunks, size_t plane_stride)
{
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const int Kb = tiled_kb(K), Nb = tiled_rb(N), Mb = tiled_rb(M);
    bool ok = ldc >= N && W.fmt >= 0 && W.fmt <= 2;
    if (W.fmt == 0) ok = ok && W.w16;
    if (W.fmt == 1) ok = ok && W.q && W.d && W.nbq >= 0 && W.nbq <= Nb && (W.nbq == Nb || W.w16);
    if (W.fmt == 2) ok = ok && W.q && W.d && W.kbq >= 0 && W.kbq <= Kb && (W.kbq == Kb || W.w16);
    if (!ok) { fprintf(stderr, "[fast_hip] gemm_big: bad launch M=%d N=%d K=%d ldc=%d fmt=%d\n", M, N, K, ldc, W.fmt); abort(); }
    GemmKArgs g{};
    g.A = reinterpret_cast<const half8 *>(A); g.a_inv_scale = a_inv_scale; g.W = W;
    const bool q8_wide = W.fmt != 0 && q8_wide_ok(W, N, K);
    if (chunks < 1 || (chunks > 1 && W.fmt != 0 && !q8_wide)) { fprintf(stderr, "[fast_hip] gemm_big: K chunks need F16 tiles or the 256 x 256 Q8_0 kernel\n"); abort(); }
    g.P = C; g.ldp = ldc; g.plane_stride = plane_stride;
    g.M = M; g.N = N; g.Mb = Mb; g.Nb = Nb; g.Kb = Kb;
    g.steps_per_chunk = (Kb + chunks - 1) / chunks;
    g.S = (Kb + g.steps_per_chunk - 1) / g.steps_per_chunk;
    g.m_tiles = mid_rows(M, W.fmt) || (W.fmt == 0 && M <= 64);
    const dim3 block(256);
    hipEvent_t ev_a = nullptr, ev_b = nullptr;
    const bool prof = gemm_prof_begin(weight_stream_bytes(W, N, K), 2.0 * M * N * K, &ev_a, &ev_b);
    // grid of either block shape: with K chunks one workgroup per (chunk, block); else whole patches of 8 x 32 ids (see
    // the kernels), the ids past the matrix returning at once
    auto grid_of = [&](const GemmKArgs &a, int bm, int bn) {
        const int mt = (a.M + bm - 1) / bm, nt = (a.N + bn - 1) / bn;
        if (a.m_tiles) return dim3(8 * mt * ((nt * a.S + 7) / 8));
        return dim3(a.S > 1 ? mt * nt * a.S : 8 * 32 * ((mt + 7) / 8) * (((nt + 7) / 8 + 3) / 4));
    };
    if (W.fmt == 0 || q8_wide) {
        // 128 x 256 or 256 x 256 blocks, whichever keeps more of the GPU on useful work -- the share of the last round's
        // CUs that have a block times the share of the tiles' area that lies inside the matrix.  The wide block is faster
        // in its loop and wins from 0.9 of the other's share, given 20 K steps per block to win them in (below, its larger
        // prologue and epilogue take the gain back).  Measured at 2048 rows inside the step: 200 and 240 wide blocks win
        // against 400 and 480, 4752 against 9504; 608, 304 and 128 lose against 1216, 608 and 256.
        const int cus = num_cus() > 0 ? num_cus() : 256;
        auto share = [&](int bm, int bn) {
            const long tm = (M + bm - 1) / bm, tn = (N + bn - 1) / bn, blocks = tm * tn * g.S;
            return (double)M * N / ((double)tm * bm * tn * bn) * (double)blocks / (double)((blocks + cus - 1) / cus * cus);
        };
        const bool deep = g.steps_per_chunk >= 20;
        // (Q8_0 tiles: the wide block only, see gemm_big_q8)
        const bool mid = mid_rows(M, W.fmt);
        const bool wide = W.fmt != 0 || g_big_block == 2 || (g_big_block == 0 && mid && mid_big_us(1, M, N, K, g.S, cus) < mid_big_us(0, M, N, K, g.S, cus)) ||
                          (g_big_block == 0 && !mid && deep && share(256, 256) >= 0.9 * share(128, 128 * WPW));
        // A product of at least one full round of wide blocks whose last round would be half empty or less: the columns
        // of the full rounds go to wide blocks, the rest to 128 x 256 blocks in a launch of their own
        const int MX = (M + 255) / 256, NX = (N + 255) / 256, full = MX * NX / cus, rest = MX * NX % cus;
        const int wide_cols = full * cus / MX * 256;
        auto launch = [&](const GemmKArgs &a, bool w, hipEvent_t e0, hipEvent_t e1) {
            const dim3 grid = w ? grid_of(a, 256, 256) : grid_of(a, 128, 128 * WPW);
#define BIG_LAUNCH(KERNEL, ...) do { if (prof) hipExtLaunchKernelGGL(KERNEL, grid, block, 0, stream(), e0, e1, 0, __VA_ARGS__); \
                                     else hipLaunchKernelGGL(KERNEL, grid, block, 0, stream(), __VA_ARGS__); } while (0)
            if (W.fmt == 0) { if (w) BIG_LAUNCH((gemm_big_f16<256>), a, GroupArgs{}); else BIG_LAUNCH((gemm_big_f16<128>), a, GroupArgs{}); }
            else if (W.fmt == 1) { if (a.W.nbq < a.Nb) BIG_LAUNCH((gemm_big_q8<1, 256, true>), a); else BIG_LAUNCH((gemm_big_q8<1, 256>), a); }
            else BIG_LAUNCH((gemm_big_q8<2, 256>), a);
#undef BIG_LAUNCH
        };
        if (g_big_block == 0 && !wide && !mid && deep && g.S == 1 && full >= 1 && rest > 0 && rest * 2 <= cus && wide_cols < N) {
            GemmKArgs g1 = g, g2 = g;
            const int rb = wide_cols / 32;                 // weight row blocks that go to the wide launch
            g1.N = wide_cols; g1.Nb = rb;
            g2.N = N - wide_cols; g2.Nb = tiled_rb(g2.N);
            g2.P = C + wide_cols;
            g2.W.w16 = W.w16 + (size_t)rb * Kb * 2048;    // (F16 tiles: Q8_0 products are all wide)
            launch(g1, true, ev_a, nullptr);
            launch(g2, false, nullptr, ev_b);
        } else launch(g, wide, ev_a, ev_b);
        HIP_CHECK(hipGetLastError());
        return g.S;
    }
    const dim3 grid = grid_of(g, 128, 128 * WPW);
    const size_t lds = (size_t)2 * (4 + 4 * WPW) * 256 * sizeof(half8);
    static bool attr_set = false;
    if (!attr_set) {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_big<1>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_big<2>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        attr_set = true;
    }
    if (prof) {
        if (W.fmt == 1) hipExtLaunchKernelGGL(gemm_big<1>, grid, block, lds, stream(), ev_a, ev_b, 0, g);
        else hipExtLaunchKernelGGL(gemm_big<2>, grid, block, lds, stream(), ev_a, ev_b, 0, g);
    } else {
        if (W.fmt == 1) hipLaunchKernelGGL(gemm_big<1>, grid, block, lds, stream(), g);
        else hipLaunchKernelGGL(gemm_big<2>, grid, block, lds, stream(), g);
    }
    HIP_CHECK(hipGetLastError());
    return 1;
}

// The plan: the streaming kernel (its waves and planes in any case form short sums; at most four K steps per wave, sixteen MFMAs) or
// the 128 x 256 block, by the times of mid_plan at any number of rows.  Operands that are not F16 tiles: use_big_gemm's rule.
ShortPlan plan_short_sums(int M, int N, int K, int nbq, int fmt)
{
    ShortPlan p{0, 1, plan_gemm(M, N, K, nbq, fmt)};
    const int cus = num_cus() > 0 ? num_cus() : 256, Kb = tiled_kb(K);
    if (!p.t.ring && p.t.steps > 4 * p.t.nw) { p.t.steps = 4 * p.t.nw; p.t.S = (Kb + p.t.steps - 1) / p.t.steps; }
    const int policy = big_gemm_policy();
    if (policy < 0 || (policy == 0 && (M <= 64 || (fmt != 0 && !use_big_gemm(M, N, K, fmt))))) return p;
    double best = policy || fmt ? 1e30 : 5.1 + 0.152 * (2e-6 * N * K) + 1.65 * (2e-9 * M * N * K) + (0.115 + 0.2) * (4e-6 * p.t.S * M * N);
    for (int S = 1; S <= 20 && (S == 1 || S * 4 <= Kb); S++) {
        const double us = mid_big_us(0, M, N, K, S, cus);
        if (us < best) { best = us; p.big = 1; p.chunks = S; }
    }
    if (p.big && g_big_split != 1) p.chunks = std::min(std::max(1, g_big_split), Kb);
    return p;
}

int launch_short_sums(const half_t *A, const WeightOp &W, float *P, size_t plane_stride, int M, int N, int K, const ShortPlan &p)
{
    if (!p.big) { launch_gemm(A, nullptr, W, P, N, plane_stride, M, N, K, p.t, 0.f, true); return p.t.S; }
    if (W.fmt != 0) return launch_gemm_big(A, nullptr, W, P, N, M, N, K, 1, plane_stride);      // (Q8_0 tiles in the large-M kernel are asked for)
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    if (!W.w16 || p.chunks < 1) { fprintf(stderr, "[fast_hip] gemm_short: bad launch M=%d N=%d K=%d chunks=%d\n", M, N, K, p.chunks); abort(); }
    GemmKArgs g{};
    g.A = reinterpret_cast<const half8 *>(A); g.W = W;
    g.P = P; g.ldp = N; g.plane_stride = plane_stride;
    g.M = M; g.N = N; g.Mb = tiled_rb(M); g.Nb = tiled_rb(N); g.Kb = tiled_kb(K);
    g.steps_per_chunk = (g.Kb + p.chunks - 1) / p.chunks;
    g.S = (g.Kb + g.steps_per_chunk - 1) / g.steps_per_chunk;
    g.m_tiles = 1;
    const dim3 grid(8 * ((M + 127) / 128) * (((N + 255) / 256 * g.S + 7) / 8));
    hipEvent_t ev_a = nullptr, ev_b = nullptr;
    if (gemm_prof_begin(weight_stream_bytes(W, N, K), 2.0 * M * N * K, &ev_a, &ev_b))
        hipExtLaunchKernelGGL(gemm_big_short, grid, dim3(256), 0, stream(), ev_a, ev_b, 0, g);
    else hipLaunchKernelGGL(gemm_big_short, grid, dim3(256), 0, stream(), g);
    HIP_CHECK(hipGetLastError());
    return g.S;
}

// Value and residual rows: the pair kernel or the streaming kernel over all 2 M rows, by the same times; a block of 128 rows costs the pair kernel
// what one of 256 costs gemm_big_f16.  Q8_0 tiles that go through their F16 image (plan_short_sums' rule, and not asked to stay quantised)
// are the pair kernel's as well: a plan that says big for F16 tiles always has its steps.
ShortPlan plan_short_pair(int M, int N, int K, int nbq, int fmt)
{
    ShortPlan p = plan_short_sums(2 * M, N, K, nbq, fmt);
    p.lo = M;
    const int policy = big_gemm_policy();
    if (policy < 0 || (fmt != 0 && (!p.big || large_m_unpacks_q8()))) return p;
    if (M <= 32 && !policy) return p;
    const GemmPlan &t = p.t;
    p.big = 0;
    const int cus = num_cus() > 0 ? num_cus() : 256, Kb = tiled_kb(K);
    double best = policy || fmt ? 1e30 : 5.1 + 0.152 * (2e-6 * N * K) + 1.65 * (4e-9 * M * N * K) + (0.115 + 0.2) * (8e-6 * t.S * M * N);
    // one round: as many teams as the CUs of every XCD hold, or teams of a K-th part of a column block each, without pieces that share a team
    const int mt = (M + 127) / 128, nt = (N + 255) / 256, teams = 8 * std::max(1, cus / 8 / mt), least = std::max(1, (nt * Kb + teams - 1) / teams);
    for (int S = 0; S <= 20 && (S <= 1 || S * 4 <= Kb); S++) {
        const int steps = S ? std::max(least, (Kb + S - 1) / S) : least;
        const double us = pair_us(M, N, K, steps, cus);
        if (us < best) { best = us; p.big = 1; p.steps = steps; }
    }
    if (!p.big) return p;
    if (g_big_split != 1) p.steps = std::max(1, Kb / std::max(1, g_big_split));
    p.chunks = PairWalk{p.steps, Kb}.planes();
    p.lo = pair_row(M);
    return p;
}

PairPlanes launch_short_pair(const half_t *A, const float *inv, const WeightOp &W, float *P, int M, int N, int K, const ShortPlan &p)
{
    const int lo = p.lo;
    PairPlanes out{(size_t)(lo + M) * N, 0, false, {}};
    if (M <= 0 || N <= 0 || K <= 0) return out;
    if (lo < M || !inv) { fprintf(stderr, "[fast_hip] gemm_pair: bad rows M=%d lo=%d\n", M, lo); abort(); }
    if (!p.big || W.fmt != 0) { out.S = launch_short_sums(A, W, P, out.plane, lo + M, N, K, p); return out; }
    if (!W.w16 || p.steps < 1 || (lo & 31)) { fprintf(stderr, "[fast_hip] gemm_pair: bad launch M=%d lo=%d N=%d K=%d chunks=%d\n", M, lo, N, K, p.chunks); abort(); }
    GemmKArgs g{};
    g.A = reinterpret_cast<const half8 *>(A); g.W = W; g.a_inv_scale = inv;
    out.plane = (size_t)M * N;
    g.P = P; g.ldp = N; g.plane_stride = out.plane;
    g.M = M; g.N = N; g.Mb = tiled_rb(M); g.Nb = tiled_rb(N); g.Kb = tiled_kb(K);
    g.steps_per_chunk = p.steps;
    const int teams = ((N + 255) / 256 * g.Kb + p.steps - 1) / p.steps;
    const dim3 grid(8 * ((M + 127) / 128) * ((teams + 7) / 8));
    hipEvent_t ev_a = nullptr, ev_b = nullptr;
    if (gemm_prof_begin(weight_stream_bytes(W, N, K), 4.0 * M * N * K, &ev_a, &ev_b))
        hipExtLaunchKernelGGL(gemm_big_pair, grid, dim3(256), 0, stream(), ev_a, ev_b, 0, g, lo);
    else hipLaunchKernelGGL(gemm_big_pair, grid, dim3(256), 0, stream(), g, lo);
    HIP_CHECK(hipGetLastError());
    out.S = p.chunks;
    out.walk = PairWalk{p.steps, g.Kb};
    out.whole = true;
    return out;
}

void launch_gemm_groups(const half_t *A, const float *a_inv_scale, const half_t *W, size_t group_stride, const int *group_of, float *C, int ldc,
                        int M, int N, int K, int groups, hipStream_t s)
{
    if (M <= 0 || N <= 0 || K <= 0) return;
    if (ldc < N || (M & 127) || !A || !W || !group_of || group_stride < tiled_elems(N, K)) {
        fprintf(stderr, "[fast_hip] gemm_groups: bad launch M=%d N=%d K=%d ldc=%d\n", M, N, K, ldc);
        abort();
    }
    GemmKArgs g{};
    g.A = reinterpret_cast<const half8 *>(A); g.a_inv_scale = a_inv_scale; g.W = weight_f16(W);
    g.P = C; g.ldp = ldc; g.M = M; g.N = N; g.Mb = tiled_rb(M); g.Nb = tiled_rb(N); g.Kb = tiled_kb(K);
    g.steps_per_chunk = g.Kb; g.S = 1;
    const int mt = M / 128, nt = (N + 255) / 256;
    const dim3 grid(8 * ((mt * nt + 7) / 8));
    hipEvent_t ev_a = nullptr, ev_b = nullptr;
    if (gemm_prof_begin(2.0 * groups * N * K, 2.0 * M * N * K, &ev_a, &ev_b))
        hipExtLaunchKernelGGL((gemm_big_f16<128, true>), grid, dim3(256), 0, s, ev_a, ev_b, 0, g, GroupArgs{group_of, group_stride});
    else hipLaunchKernelGGL((gemm_big_f16<128, true>), grid, dim3(256), 0, s, g, GroupArgs{group_of, group_stride});
    HIP_CHECK(hipGetLastError());
}

void set_big_gemm_split(int mode) { g_big_split = mode; }
void set_big_gemm_block(int mode) { g_big_block = mode; }

}  // namespace lmhip
