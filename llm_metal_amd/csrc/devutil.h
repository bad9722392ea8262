// Device-side helpers shared by the kernels: wave64 / workgroup reductions,
// F16 <-> fp32 conversion with explicit rounding, vector types.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef _Float16 half_t;
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float    float16v __attribute__((ext_vector_type(16)));
typedef float    float4v __attribute__((ext_vector_type(4)));

#define WAVE 64

// v + (or max with) the value of lane ^ O, without the trip through LDS that __shfl_xor takes: DPP inside rows of sixteen lanes,
// gfx950's row and half swaps across them.  Every lane of the wave active.  The same operands meet in the same order as with
// __shfl_xor (a sum of products needs wave_sum_products for that); six dependent steps take some 50 cycles instead of 700 (Q8_0 head of
// 262 144 rows, one reduction per row: 86 -> 77 us; k_qkv_bwd_rows at 64 rows 9.6 -> 8.0; gated product with its norms 12.9 -> 11.7).
template <int CTRL, int BANKS = 0xF> __device__ __forceinline__ float dpp_move(float old, float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, v), CTRL, 0xF, BANKS, false));
}
struct LanePair { float a, b; };                           // v of this lane and of lane ^ O; in either order, the lower lane's first where O is 16 or 32
template <int O> __device__ __forceinline__ LanePair lane_pair(float v)
{
    static_assert(O == 1 || O == 2 || O == 4 || O == 8 || O == 16 || O == 32, "a power of two below 64");
    if constexpr (O == 1) return {v, dpp_move<0xB1>(v, v)};                          // quad_perm [1, 0, 3, 2]
    else if constexpr (O == 2) return {v, dpp_move<0x4E>(v, v)};                     // quad_perm [2, 3, 0, 1]
    else if constexpr (O == 4) return {v, dpp_move<0x114, 0xA>(dpp_move<0x104, 0x5>(v, v), v)};   // four up in the even quads, four down in the odd ones
    else if constexpr (O == 8) return {v, dpp_move<0x128>(v, v)};                    // rotated by eight of sixteen
    else {
        const unsigned u = __builtin_bit_cast(unsigned, v);
        unsigned x, y;                                     // (copies: a bit cast of a vector's element reads the first one)
        if constexpr (O == 16) { const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false); x = r[0]; y = r[1]; }
        else { const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false); x = r[0]; y = r[1]; }
        return {__builtin_bit_cast(float, x), __builtin_bit_cast(float, y)};
    }
}
template <int O> __device__ __forceinline__ float xor_add(float v) { const LanePair p = lane_pair<O>(v); return p.a + p.b; }
template <int O> __device__ __forceinline__ float xor_max(float v) { const LanePair p = lane_pair<O>(v); return fmaxf(p.a, p.b); }

__device__ __forceinline__ float wave_sum(float v)
{
    return xor_add<1>(xor_add<2>(xor_add<4>(xor_add<8>(xor_add<16>(xor_add<32>(v))))));
}

// The sum of a b over the wave.  Its first step adds the lane's own product, not yet rounded, to the rounded one of lane ^ 32:
// one fused operation, which `v += __shfl_xor(v, 32)` becomes when v is a product, and wave_sum(a * b), whose swap takes rounded
// products from both, does not.  (The last bit of a row's log-sum-exp turns roundings of its loss gradient to fp16: adapters after a
// step 1e-4 .. 2e-3 apart.)
__device__ __forceinline__ float wave_sum_products(float a, float b)
{
    const LanePair p = lane_pair<32>(__fmul_rn(a, b));     // a: of the lower half's lane, b: of the upper half's
    return xor_add<1>(xor_add<2>(xor_add<4>(xor_add<8>(xor_add<16>(fmaf(a, b, threadIdx.x & 32 ? p.a : p.b))))));
}

__device__ __forceinline__ float wave_max(float v)
{
    return xor_max<1>(xor_max<2>(xor_max<4>(xor_max<8>(xor_max<16>(xor_max<32>(v))))));
}

// Workgroup reductions for blocks of up to 1024 threads (16 waves).  `smem`
// must hold 16 floats; every thread gets the result.  Two barriers per call,
// so the same `smem` may be reused by the next call; AGAIN false: one, and this `smem` is not written again.
// NT: the workgroup's threads (whole waves), where the kernel knows them: the waves' values are then read together and not in a loop, which is one trip
// to LDS after the other, four for 256 threads; 0: blockDim.x.  The order is the same.  Row
// kernels of a training step so, and without a barrier behind their reductions: Gemma3-1B 1 x 64 (18 launches a layer) 3920 -> 3880 us, Qwen3-4B 6945 -> 6910,
// nine layers of it 1 x 250 3439 -> 3402, a tiny model 227 -> 223.
template <int NT, typename F> __device__ __forceinline__ void each_wave(const float *smem, F &&f)
{
    static_assert(NT % 64 == 0 && NT <= 1024, "whole waves");
    if constexpr (NT > 0) {
        float v[NT / 64];
#pragma unroll
        for (int i = 0; i < NT / 64; i++) v[i] = smem[i];
#pragma unroll
        for (int i = 0; i < NT / 64; i++) f(v[i]);
    } else
        for (int i = 0, nw = (blockDim.x + 63) >> 6; i < nw; i++) f(smem[i]);
}

template <int NT = 0, bool AGAIN = true> __device__ __forceinline__ float block_sum_waves(float v, float *smem)       // v: the sum of the thread's wave
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) smem[w] = v;
    __syncthreads();
    float r = 0.f;
    each_wave<NT>(smem, [&](float x) __attribute__((always_inline)) { r += x; });
    if (AGAIN) __syncthreads();
    return r;
}

template <int NT = 0, bool AGAIN = true> __device__ __forceinline__ float block_sum(float v, float *smem) { return block_sum_waves<NT, AGAIN>(wave_sum(v), smem); }
template <int NT = 0, bool AGAIN = true> __device__ __forceinline__ float block_sum_products(float a, float b, float *smem) { return block_sum_waves<NT, AGAIN>(wave_sum_products(a, b), smem); }

// Two sums for one pair of barriers; `smem` must hold 32 floats.  Each sum is formed in the order block_sum forms it.
template <int NT = 0, bool AGAIN = true> __device__ __forceinline__ void block_sum2_waves(float &a, float &b, float *smem)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) { smem[w] = a; smem[16 + w] = b; }
    __syncthreads();
    float ra = 0.f, rb = 0.f;
    each_wave<NT>(smem, [&](float x) __attribute__((always_inline)) { ra += x; });
    each_wave<NT>(smem + 16, [&](float x) __attribute__((always_inline)) { rb += x; });
    if (AGAIN) __syncthreads();
    a = ra; b = rb;
}
template <int NT = 0, bool AGAIN = true> __device__ __forceinline__ void block_sum2(float &a, float &b, float *smem) { a = wave_sum(a); b = wave_sum(b); block_sum2_waves<NT, AGAIN>(a, b, smem); }

// A sum and a maximum for one pair of barriers; `smem` must hold 32 floats.  The sum is formed in the order block_sum forms it.
template <int NT = 0, bool AGAIN = true> __device__ __forceinline__ void block_sum_max(float &a, float &m, float *smem)
{
    a = wave_sum(a); m = wave_max(m);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) { smem[w] = a; smem[16 + w] = m; }
    __syncthreads();
    float ra = 0.f, rm = smem[16];
    each_wave<NT>(smem, [&](float x) __attribute__((always_inline)) { ra += x; });
    each_wave<NT>(smem + 16, [&](float x) __attribute__((always_inline)) { rm = fmaxf(rm, x); });
    if (AGAIN) __syncthreads();
    a = ra; m = rm;
}

template <int NT = 0, bool AGAIN = true> __device__ __forceinline__ float block_max(float v, float *smem)
{
    v = wave_max(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) smem[w] = v;
    __syncthreads();
    float r = smem[0];
    each_wave<NT>(smem, [&](float x) __attribute__((always_inline)) { r = fmaxf(r, x); });
    if (AGAIN) __syncthreads();
    return r;
}

// Power-of-two scale s such that amax * s lies in [2^12, 2^13): the fp16 image of
// a row then keeps 11 significant bits for everything within 2^-26 of the row
// maximum and cannot overflow.  Exact to undo (inv = 1/s is a power of two).
__device__ __forceinline__ float row_scale_for(float amax)
{
    if (!(amax > 0.f) || !(amax < 3.0e38f)) return 1.0f;
    int e;
    frexpf(amax, &e);                 // amax = f * 2^e, f in [0.5, 1)
    int p = 13 - e;
    p = p > 120 ? 120 : (p < -120 ? -120 : p);
    return ldexpf(1.0f, p);
}

// Argument of the tanh in the GELU approximation, clamped as the reference clamps it (gelu_mul,
// shaders/q8_kernels.metal:349-362).
__device__ __forceinline__ float gelu_inner(float g)
{
    const float in = 0.7978845608f * (g + 0.044715f * g * g * g);
    return fminf(fmaxf(in, -15.0f), 15.0f);
}

__device__ __forceinline__ half_t f2h(float x) { return (half_t)x; }      // v_cvt_f16_f32: round to nearest even
__device__ __forceinline__ float  h2f(half_t x) { return (float)x; }

// Workgroup `wg` of `nwgs` reads its share of [base, base + bytes) with 16-byte loads, eight in flight per thread, and
// throws the values away: what a launch with spare CUs does for the weights of the product that follows it (the data then
// waits in the memory-side cache).  bytes % 16 == 0; block of 256 threads or more.
__device__ __forceinline__ void request_bytes_ahead(const char *base, size_t bytes, int wg, int nwgs)
{
    const size_t row = (size_t)blockDim.x * 16;
    const size_t per = ((bytes + nwgs - 1) / nwgs + row - 1) / row * row;
    const size_t beg = (size_t)wg * per, end = bytes < beg + per ? bytes : beg + per;
    unsigned sink = 0u;
    for (size_t o = beg + (size_t)threadIdx.x * 16; o < end; o += 8 * row) {
        uint4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = (o + u * row < end) ? *reinterpret_cast<const uint4 *>(base + o + u * row) : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int u = 0; u < 8; u++) sink ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
    }
    asm volatile("" :: "v"(sink));
}
