// One decoding step of one sequence in one launch: embedding, all layers, head and argmax.
//
// A token's products are short (Gemma3-1B Q8_0: 28 MB of weights per layer, 5.5 us of streaming) and each needs all of the vector
// before it, so that with a launch per product the step is a chain of ramps: 26 us per layer in five launches.  Here every CU holds
// one workgroup for the whole token, and what a product leaves passes from CU to CU as words of (value, tag): 64-bit device-scope
// atomics, relaxed, each of which carries its own proof of arrival, so no flag, no fence and no write-back of caches stands between
// the workgroup that wrote a value and the one that multiplies it.  A hand-over between all 256 workgroups takes 1.9 us for 1152 values
// and 2.4 for 6912, with its barrier and LDS trip.
//
// Workgroup: sixteen waves.  The weights that a wave multiplies, product after product from the first layer to the head, come into a ring
// in LDS of its own, RING slots ahead -- across products and layers, since weights depend on nothing.  A slot is 512 columns of R rows
// (half of them gate and half up rows in the gate|up product).  The slots of a product are dealt evenly to the waves, wherever that cuts a
// row; the parts of a row's sum meet in LDS.  Between products all threads poll the words of the next vector, form residual sum and norms
// (every workgroup for itself; the residual stays in registers from the first layer to the last), and after a product they finish
// the sums (norm factor, gate) and publish them.  Hq workgroups are the attention, which has its keys and values on the way while the query
// is awaited; they have no rows of O.
// What a layer takes is the sum of its five hand-overs and of the instructions between them, each of which the slowest wave sets.  Hence one piece
// of code for the slots of all products (with a copy per product, unrolled over stages in registers, the kernel was 118 KB, twice the instruction
// cache: 30 us per layer of Gemma3-1B), all waves at the slots (with eight that multiply and eight that form vectors 38 us; a slot is a chain of 0.5 us) and
// no more waves than it takes at everything else (sixteen share four issue slots).
// Per token, greedy, contexts of up to 128, in five launches per layer -> so: Gemma3-1B Q8_0 734 -> 617 us, nine layers of Qwen3-4B F16 with a head of
// 32 768 rows 480 -> 437.  Bound by the hand-overs and, Q8_0, by instructions (two per weight); F16 by the stream (5.5 TB/s while it flows).
//
// Words are reused layer after layer without a wait for readers: whoever writes one of a kind again has, through the vectors
// between, seen a word from every workgroup that it wrote after its last look at the kind (all workgroups have rows of gate|up and
// of down).
//
// All workgroups must be resident together: one per CU, on the library's one stream.  Should some be kept off the device (another
// process's kernel that waits in the same way), a wait ends at `ticks` of the 100 MHz clock: the kernel then runs to its end without
// waiting any more, leaves a mark for the host, and the host takes the step again in launches.
#include "backend.h"
#include "devutil.h"
#include "lds_copy.h"
#include "token.h"

using namespace lmhip;

namespace {

typedef unsigned long long u64;
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
#define AS_GLOBAL __attribute__((address_space(1)))

constexpr int WAVES = 16, TT = WAVES * 64;
constexpr int FW = 4, FT = FW * 64;                        // those that form the vector behind a norm: one on each SIMD (sixteen share its issue: 1.2 us, so 0.5)
constexpr int ROWS = 80;                                   // of a product that a workgroup has at most (the head takes more in turn)
template <int FMT> constexpr int R = FMT == 0 ? 2 : 4;     // rows of a slot
template <int FMT> constexpr int SLOT = FMT == 0 ? 2048 : 2304;              // its bytes: rows of 512 halves, or of 512 codes and then their scales
template <int FMT> constexpr int COPIES = FMT == 0 ? 2 : 3;                  // that fill it
template <int FMT, int SI> constexpr int RING = FMT == 1 && SI > 7 ? 2 : 3;  // slots that a wave has on their way (LDS)

__device__ __forceinline__ void wg_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// a lane's place behind an address that the whole wave has: stays a scalar base and a 32-bit offset
template <typename T> __device__ __forceinline__ const AS_GLOBAL T *global(u64 base, uint32_t bytes = 0) { return (const AS_GLOBAL T *)((const AS_GLOBAL char *)base + bytes); }

// v as if it were new: what follows from it is formed where it is used, instead of waiting in registers through all phases of a layer
template <typename T> __device__ __forceinline__ T anew(T v) { asm volatile("" : "+v"(v)); return v; }

// place of column c of a vector in LDS: a lane reads its eight (8 l .. 8 l + 7 of a 512-column step) in two pieces, each of which the wave
// reads whole
__device__ __forceinline__ int xs_at(int c) { return (c & ~511) | ((c & 4) << 6) | ((c >> 3) & 63) << 2 | (c & 3); }

__device__ __forceinline__ void publish(u64 *w, uint32_t tag, float v)
{
    __hip_atomic_store(w, ((u64)tag << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a wave's waits: until `ticks` have passed since the kernel began in this wave, after that none
struct Waits {
    u64 until;
    int *fail;
    bool over;
    uint32_t looks = 0;
    __device__ __forceinline__ bool expired()
    {
        if (!over && (looks++ & 15) == 0 && wall_clock64() >= until) { over = true; *fail = 1; }
        return over;
    }
};

// P x N words of each lane: N of them STRIDE apart from every place[p] on (words behind `words`)
template <int N, int STRIDE, int P>
__device__ __forceinline__ void await(const u64 *words, const uint32_t (&place)[P], uint32_t tag, float (&out)[P * N], Waits &w)
{
    u64 x[P * N];
    do {
        bool there = true;
#pragma unroll
        for (int i = 0; i < P * N; i++) x[i] = __hip_atomic_load(global<u64>((u64)words, 8 * place[i / N]) + STRIDE * (i % N), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < P * N; i++) there = there && (uint32_t)(x[i] >> 32) == tag;
        if (__ballot(!there) == 0) break;
    } while (!w.expired());
#pragma unroll
    for (int i = 0; i < P * N; i++) out[i] = __uint_as_float((uint32_t)x[i]);
}

// A product's rows as a workgroup sees them (bytes; scales follow at a sixteenth of the codes' offsets)
struct Rows {
    uint32_t row, odd, far;                                // of a row; from a slot's first row to the next, and to the second half of its rows
    uint32_t unit;                                         // from a unit of R rows to the next
    int cols, steps, units;
    int first;                                             // row of its first unit
    u64 begin;                                             // offset of its first unit
};
// of that a wave's share: its first slot and how many from there on
struct Share { int unit, step, left; };

template <int SI>
struct Shared {
    u64 layer[TOKEN_MAX_LAYERS * (sizeof(TokenLayer) / 8)];
    Rows rows[5];                                          // Q|K|V, O, gate|up, down, head
    Share share[WAVES][4];
    alignas(16) float part[2][FW];                         // sums of squares by wave: of the branch, of the vector
    alignas(16) float red[2][ROWS][WAVES];                 // parts of the rows' sums by wave, products in turn here and there
    float pm[WAVES], pl[WAVES];                            // attention: maximum and sum of each wave's keys (its values are in xs)
    alignas(16) float head[6][256];                        // its norm weights of query and key, (cos, sin) of the position; rows of the product
    float bv[WAVES];
    int bi[WAVES];
    alignas(16) float xs[SI * TT];                         // the vector of a product (behind a norm: times the norm's weight)
};

__device__ __forceinline__ u64 uniform(u64 v)
{
    return ((u64)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
#define LAYER_FIELD(L_, f_) uniform(sh.layer[(L_) * (int)(sizeof(TokenLayer) / 8) + (int)(offsetof(TokenLayer, f_) / 8)])

__device__ __forceinline__ Share share_of(int slots, int steps, int wave)
{
    const int begin = slots * wave / WAVES, unit = begin / steps;
    return {unit, begin - unit * steps, slots * (wave + 1) / WAVES - begin};
}

// What a wave requests: slots of a product
struct Asked {
    u64 W, scales;                                         // of the unit
    uint32_t odd, far, unit;
    int row, steps, step, left;                            // left: slots that are still to be requested
};
template <int FMT, int SI>
struct Stream {
    Asked p, next;                                         // next.left == 0: to be looked up
    int L, kind;                                           // of next: kinds 0 .. 3 of layer L, L = NL: part `kind` of the head
    uint32_t lds, slot;                                    // address of the ring, and of its next slot behind that

    // the product behind, if it has slots for the wave; behind the last one the head's first slot, again and again, which nobody reads
    __device__ __forceinline__ void look_up(const TokenArgs &a, Shared<SI> &sh, int wave, int head_parts)
    {
        while (next.left <= 0) {
            if (++kind == 4 && L < a.NL) { kind = 0; L++; }
            const bool head = L == a.NL;
            const Rows &r = sh.rows[head ? 4 : kind];
            Share s;
            if (head) {
                const int per = ROWS / R<FMT>;
                s = kind < head_parts ? share_of(min(per, uniform(r.units) - per * kind) * uniform(r.steps), uniform(r.steps), wave) : Share{0, 0, 1 << 30};
                if (kind < head_parts) s.unit += per * kind;
            } else s = Share{uniform(sh.share[wave][kind].unit), uniform(sh.share[wave][kind].step), uniform(sh.share[wave][kind].left)};
            next.row = uniform((int)r.row); next.odd = uniform((int)r.odd); next.far = uniform((int)r.far); next.unit = uniform((int)r.unit);
            next.steps = uniform(r.steps); next.step = s.step; next.left = s.left;
            const u64 from = uniform(r.begin) + (u64)next.unit * s.unit;
            const int at = head ? 0 : L * (int)(sizeof(TokenLayer) / 8) + 2 * kind;
            next.W = (head ? (u64)a.head : uniform(sh.layer[at])) + from;
            next.scales = (head ? (u64)a.head_d : uniform(sh.layer[at + 1])) + (from >> 4);
            if (head && kind >= head_parts) next.unit = 0;
        }
    }
    // false: the next product has not been looked up
    __device__ __forceinline__ bool ready()
    {
        if (p.left == 0) {
            if (next.left == 0) return false;
            p = next;
            next.left = 0;
        }
        return true;
    }
    __device__ __forceinline__ void request(int lane)
    {
        const uint32_t to = lds + slot;
        slot = slot + SLOT<FMT> == RING<FMT, SI> * SLOT<FMT> ? 0 : slot + SLOT<FMT>;
        // (columns behind the row's last are its last ones again: nobody counts them)
        if (FMT == 0) {
            const int at = min(1024 * p.step + 16 * lane, p.row - 16);
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" :: "v"(at), "s"(uniform((int)to)), "s"(uniform(p.W)) : "memory", "m0");
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" :: "v"(at), "s"(uniform((int)to + 1024)), "s"(uniform(p.W + p.far)) : "memory", "m0");
        } else {
            const uint32_t at = (uint32_t)min(512 * p.step + 16 * (lane & 31), p.row - 16) + (lane & 32 ? p.odd : 0u);
            const uint32_t sc = (uint32_t)min(32 * p.step + 4 * (lane & 7), (p.row >> 4) - 4) + (lane & 8 ? p.odd >> 4 : 0u) + (lane & 16 ? p.far >> 4 : 0u);
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" :: "v"(at), "s"(uniform((int)to)), "s"(uniform(p.W)) : "memory", "m0");
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" :: "v"(at), "s"(uniform((int)to + 1024)), "s"(uniform(p.W + p.far)) : "memory", "m0");
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, %2" :: "v"(sc), "s"(uniform((int)to + 2048)), "s"(uniform(p.scales)) : "memory", "m0");
        }
        if (++p.step == p.steps) { p.step = 0; p.W += p.unit; p.scales += p.unit >> 4; }
        p.left--;
    }
};

// a + its value of lane ^ O where bit O of the lane is clear, b + its value of lane ^ O where it is set
template <int O> __device__ __forceinline__ float both(float a, float b)
{
    unsigned x, y;
    if constexpr (O == 32) { const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false); x = r[0]; y = r[1]; }
    else { const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false); x = r[0]; y = r[1]; }
    return __uint_as_float(x) + __uint_as_float(y);
}

__device__ __forceinline__ float sum_lanes16(float v)
{
    v += dpp_move<0xB1>(v, v);
    v += dpp_move<0x4E>(v, v);
    v += dpp_move<0x141>(v, v);
    v += dpp_move<0x140>(v, v);
    return v;
}

// Attention of one head over the cached keys and the newest one, which is among the words of the Q|K|V product: k_attn_short by sixteen
// waves.  Keys go in turn to 64 groups of 16 lanes.  Everything of the cache that a group takes first is on its way before the product's words
// are awaited.
template <int HD, int SI>
__device__ __forceinline__ void attend(const TokenArgs &a, Shared<SI> &sh, int L, int hq, int tid, uint32_t tag, Waits &w)
{
    constexpr int C = HD / 64, U = HD == 256 ? 1 : 2, GROUPS = TT / 16;      // 16-byte pieces per lane and key; keys that a group has in flight
    tid = anew(tid);
    const int grp = tid >> 4, sub = tid & 15, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, pos = a.pos;
    const bool has_keys = 4 * wave < pos;
    const int hk = hq / (a.Hq / a.Hkv);
    const size_t head = (size_t)hk * a.max_seq * HD;
    const u64 Kh = LAYER_FIELD(L, kc) + 4 * head, Vh = LAYER_FIELD(L, vc) + 4 * head;
    const bool normed_q = LAYER_FIELD(L, g_q) != 0, normed_k = LAYER_FIELD(L, g_k) != 0;
    float4v k[U][C], v[U][C];
    auto keys = [&](int j0) __attribute__((always_inline)) {               // (past the newest cached key: the last one again)
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t at = (uint32_t)(max(min(j0 + GROUPS * u, pos - 1), 0) * HD + 4 * sub) * 4;
#pragma unroll
            for (int c = 0; c < C; c++) {
                k[u][c] = global<float4v>(Kh, at)[16 * c];
                v[u][c] = global<float4v>(Vh, at)[16 * c];
            }
        }
    };
    if (has_keys) keys(grp);
    __builtin_amdgcn_sched_barrier(0);
    auto lane_dot = [](const float4v (&x)[C], const float4v (&y)[C]) __attribute__((always_inline)) {
        float4v s = x[0] * y[0];
#pragma unroll
        for (int c = 1; c < C; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) s[e] = fmaf(x[c][e], y[c][e], s[e]);
        return (s[0] + s[1]) + (s[2] + s[3]);
    };
    // the head's rows of the product, a wave for each: RMSNorm and RoPE of query and newest key (columns d and d + HD / 2 of a rotary pair are in
    // the same lane), the newest value as it is
    if (wave < 3) {
        constexpr int N = HD / 64;
        uint32_t place[N];
        float f[N], norm[N], cs[N / 2], sn[N / 2];
#pragma unroll
        for (int i = 0; i < N; i++) {
            place[i] = (wave == 0 ? hq : a.Hq + (wave - 1) * a.Hkv + hk) * HD + lane + 64 * i;
            norm[i] = sh.head[wave & 1][lane + 64 * i];
            if (i < N / 2) { cs[i] = sh.head[2][2 * (lane + 64 * i)]; sn[i] = sh.head[2][2 * (lane + 64 * i) + 1]; }
        }
        await<1, 1>(a.qkv_w, place, tag, f, w);
        if (wave < 2) {
            if (wave ? normed_k : normed_q) {
                float ss = 0.f;
#pragma unroll
                for (int i = 0; i < N; i++) ss = fmaf(f[i], f[i], ss);
                const float inv = rsqrtf(wave_sum(ss) / (float)HD + a.eps);
#pragma unroll
                for (int i = 0; i < N; i++) f[i] *= inv * norm[i];
            }
#pragma unroll
            for (int i = 0; i < N / 2; i++) {
                const float p = f[i], q = f[i + N / 2];
                f[i] = p * cs[i] - q * sn[i]; f[i + N / 2] = p * sn[i] + q * cs[i];
            }
        }
#pragma unroll
        for (int i = 0; i < N; i++) sh.head[3 + wave][lane + 64 * i] = f[i];
    }
    wg_barrier();
    auto fetch = [&](float4v (&x)[C], int which) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < C; c++) x[c] = *reinterpret_cast<const float4v *>(&sh.head[3 + which][4 * sub + 64 * c]);
    };
    float4v q[C], o[C];
    if (!has_keys && wave) {         // (uniform)
#pragma unroll
        for (int i = 0; i < HD / 64; i++) sh.xs[wave * HD + lane + 64 * i] = 0.f;
        if (lane == 0) { sh.pm[wave] = -3.0e38f; sh.pl[wave] = 0.f; }
        return;
    }
    fetch(q, 0);
    float m = -3.0e38f, l = 0.f;
#pragma unroll
    for (int c = 0; c < C; c++) o[c] = float4v{};
    if (wave == 0) {                         // the newest key belongs to the first group
        float4v kn[C], vn[C];
        fetch(kn, 1);
        fetch(vn, 2);
        const float s0 = sum_lanes16(lane_dot(q, kn)) * a.scale;
        if (grp == 0) {
            if (hq % (a.Hq / a.Hkv) == 0) {                // for the launches to come
#pragma unroll
                for (int c = 0; c < C; c++) {
                    ((AS_GLOBAL float4v *)Kh)[(size_t)pos * (HD / 4) + sub + 16 * c] = kn[c];
                    ((AS_GLOBAL float4v *)Vh)[(size_t)pos * (HD / 4) + sub + 16 * c] = vn[c];
                }
            }
            m = s0; l = 1.f;
            if (!(s0 > -3.0e38f)) { m = -3.0e38f; l = __expf(s0 - m); }    // (not a number, or minus infinity)
#pragma unroll
            for (int c = 0; c < C; c++) o[c] = l * vn[c];
        }
    }
    for (int j0 = grp; j0 < pos; j0 += GROUPS * U) {
        float s[U], top = m;
#pragma unroll
        for (int u = 0; u < U; u++) {
            s[u] = sum_lanes16(lane_dot(q, k[u])) * a.scale;
            if (j0 + GROUPS * u < pos) top = fmaxf(top, s[u]);
        }
        const float keep = __expf(m - top);
        m = top;
        l *= keep;
#pragma unroll
        for (int c = 0; c < C; c++) o[c] *= keep;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool in = j0 + GROUPS * u < pos;
            const float p = in ? __expf(s[u] - m) : 0.f;
            l += p;
#pragma unroll
            for (int c = 0; c < C; c++)
#pragma unroll
                for (int e = 0; e < 4; e++) o[c][e] = fmaf(p, in ? v[u][c][e] : 0.f, o[c][e]);
        }
        if (j0 + GROUPS * U < pos) keys(j0 + GROUPS * U);
    }
    // the four groups of the wave together
    const float all = xor_max<16>(xor_max<32>(m)), e = __expf(m - all);
    l = xor_add<16>(xor_add<32>(l * e));
    float4v sum;                                           // of the 64 columns from 64 c on, c the lane's row of sixteen (HD 128: its half)
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (C == 4) sum[i] = both<16>(both<32>(o[0][i] * e, o[2 % C][i] * e), both<32>(o[1][i] * e, o[3 % C][i] * e));
        else sum[i] = xor_add<16>(both<32>(o[0][i] * e, o[1][i] * e));
    }
    if (C == 4 || (lane & 16) == 0) {
        *reinterpret_cast<float4v *>(&sh.xs[wave * HD + 4 * sub + 64 * (C == 4 ? lane >> 4 : lane >> 5)]) = sum;
        if (sub == 0) { sh.pm[wave] = all; sh.pl[wave] = l; }
    }
}

// what the waves left, merged
template <int HD, int SI>
__device__ __forceinline__ void merge_waves(const TokenArgs &a, Shared<SI> &sh, int hq, int tid, uint32_t tag)
{
    if (tid >= HD) return;
    float pm[WAVES], o[WAVES];
#pragma unroll
    for (int g = 0; g < WAVES; g++) { pm[g] = sh.pm[g]; o[g] = sh.xs[g * HD + tid]; }
    float all = pm[0];
#pragma unroll
    for (int g = 1; g < WAVES; g++) all = fmaxf(all, pm[g]);
    float den[4] = {}, num[4] = {};                        // (sums of four waves)
#pragma unroll
    for (int g = 0; g < WAVES; g++) {
        const float e = __expf(pm[g] - all);
        den[g & 3] = fmaf(sh.pl[g], e, den[g & 3]);
        num[g & 3] = fmaf(o[g], e, num[g & 3]);
    }
    const float n = (num[0] + num[1]) + (num[2] + num[3]), d = (den[0] + den[1]) + (den[2] + den[3]);
    publish(a.att_w + hq * HD + tid, tag, n / d);
}

// FMT 0 F16 rows, 1 Q8_0 codes and scales; a thread has S entries of a vector of D and SI of the feed-forward one
template <int FMT, int S, int SI, int HD, bool GEMMA>
__global__ __launch_bounds__(TT) void k_token(TokenArgs a)
{
    constexpr int RW = R<FMT>;
    __shared__ Shared<SI> sh;
    __shared__ alignas(16) char ring[WAVES][RING<FMT, SI> * SLOT<FMT>];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), wg = blockIdx.x, nwg = gridDim.x;
    const int D = a.D, heads = a.Hq, qd = a.Hq * HD;
    const bool attends = wg < heads;
    for (int i = t; i < a.NL * (int)(sizeof(TokenLayer) / 8); i += TT) sh.layer[i] = a.layers[i];
    if (t < 5) {                                           // units of R rows (gate|up: of R / 2 pairs)
        const int n = t == 0 ? (a.Hq + 2 * a.Hkv) * HD : t == 2 ? a.IS : t == 4 ? a.V : D, per = t == 2 ? RW / 2 : RW, all = n / per;
        const int i = t == 1 ? wg - heads : wg, of = t == 1 ? nwg - heads : nwg;
        const int begin = i < 0 ? 0 : (int)((long long)all * i / of);
        Rows p;
        p.cols = t == 1 ? qd : t == 3 ? a.IS : D;
        p.row = FMT == 0 ? 2 * p.cols : p.cols;
        p.odd = p.row;
        p.far = t == 2 ? p.row * a.IS : RW == 4 ? 2 * p.row : p.row;
        p.unit = per * p.row;
        p.steps = (p.cols + 511) >> 9;
        p.units = i < 0 ? 0 : (int)((long long)all * (i + 1) / of) - begin;
        p.first = begin * per;
        p.begin = (u64)p.first * p.row;
        sh.rows[t] = p;
    }
    __syncthreads();
    if (t < 4 * WAVES) sh.share[t >> 2][t & 3] = share_of(sh.rows[t & 3].units * sh.rows[t & 3].steps, sh.rows[t & 3].steps, t >> 2);
    __syncthreads();
    const int head_units = uniform(sh.rows[4].units), head_parts = max(1, (head_units + ROWS / RW - 1) / (ROWS / RW));

    Waits w{wall_clock64() + a.ticks, a.fail, false};
    float x[S];                                            // the residual, in the first waves: columns t + FT i
#pragma unroll
    for (int i = 0; i < S; i++) x[i] = wave < FW && t + FT * i < D ? global<float>((u64)a.emb_row, 4 * (t + FT * i))[0] * a.emb_scale : 0.f;

    Stream<FMT, SI> in;
    in.L = 0; in.kind = -1; in.slot = 0; in.p.left = in.next.left = 0;
    in.lds = uniform((int)(uint32_t)(uintptr_t)(lds_void *)ring[wave]);
    uint32_t slot = 0;
    int side = 0, waiting = RING<FMT, SI>;                 // slots of the ring that are to be requested
    auto refill = [&]() __attribute__((always_inline)) {
        for (; waiting > 0; waiting--) {
            if (!in.ready()) { in.look_up(a, sh, wave, head_parts); in.ready(); }
            in.request(lane);
        }
        in.look_up(a, sh, wave, head_parts);               // (with time to spare: a search through LDS)
    };

    // the parts of the sums that no wave will write
    auto clear = [&]() __attribute__((always_inline)) {
        side ^= 1;
        if (t < ROWS * WAVES / 4) reinterpret_cast<float4v *>(sh.red[side])[t] = float4v{};
    };
    // the wave's slots of a product
    auto run = [&](const Share &s, int steps, int cols) __attribute__((always_inline)) {
        int unit = s.unit, step = s.step;
        float acc[RW];
#pragma unroll
        for (int r = 0; r < RW; r++) acc[r] = 0.f;
        const int l = anew(lane);
        for (int left = s.left; left > 0; left--) {
            const int held = RING<FMT, SI> - waiting;      // slots on their way, this one among them
            if (held == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            else if (held == 2) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(COPIES<FMT>) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * COPIES<FMT>) : "memory");
            const char *at = ring[wave] + slot;
            half8 w16[RW];
            uint2v w8[RW];
            half_t d[RW];
#pragma unroll
            for (int r = 0; r < RW; r++) {
                if (FMT == 0) w16[r] = *reinterpret_cast<const half8 *>(at + 1024 * r + 16 * l);
                else {
                    w8[r] = *reinterpret_cast<const uint2v *>(at + 512 * r + 8 * l);
                    d[r] = *reinterpret_cast<const half_t *>(at + 2048 + 32 * r + 2 * (l >> 2));
                }
            }
            const float4v x0 = *reinterpret_cast<const float4v *>(&sh.xs[512 * step + 4 * l]), x1 = *reinterpret_cast<const float4v *>(&sh.xs[512 * step + 256 + 4 * l]);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");               // the slot has been read: it may be filled again
            // (F16, bound by the stream: the next product's slots not before this one's rows are out, 446 us per token of nine Qwen3-4B layers against
            // 473; Q8_0, bound by instructions: at once, 630 for 26 Gemma3-1B layers against 650)
            if (FMT == 0 ? in.p.left != 0 : in.ready()) in.request(l); else waiting++;
            slot = slot + SLOT<FMT> == RING<FMT, SI> * SLOT<FMT> ? 0 : slot + SLOT<FMT>;
            if (512 * step + 8 * l < cols) {
                float p[RW];
#pragma unroll
                for (int r = 0; r < RW; r++) p[r] = FMT == 0 ? acc[r] : 0.f;
#pragma unroll
                for (int e = 0; e < 8; e++)
#pragma unroll
                    for (int r = 0; r < RW; r++) p[r] = fmaf(FMT == 0 ? (float)w16[r][e] : (float)(int8_t)(w8[r][e >> 2] >> (8 * (e & 3))), e < 4 ? x0[e & 3] : x1[e & 3], p[r]);
#pragma unroll
                for (int r = 0; r < RW; r++) acc[r] = FMT == 0 ? p[r] : fmaf((float)d[r], p[r], acc[r]);
            }
            if (++step == steps || left == 1) {
                // the rows' sums together: halves of the wave swapped between rows, so that each step halves the rows as well
                float sum = both<32>(acc[0], acc[1]);
                int row = l >> 5;
                if (RW == 4) {
                    sum = both<16>(sum, both<32>(acc[2 % RW], acc[3 % RW]));
                    row += l >> 3 & 2;
                } else sum = xor_add<16>(sum);
                sum = xor_add<1>(xor_add<2>(xor_add<4>(xor_add<8>(sum))));
                if ((l & (RW == 4 ? 15 : 31)) == 0) sh.red[side][RW * unit + row][wave] = sum;
#pragma unroll
                for (int r = 0; r < RW; r++) acc[r] = 0.f;
                step = 0;
                unit++;
            }
        }
    };
    // sum of a row that the waves have just multiplied
    auto row_sum = [&](int r) __attribute__((always_inline)) {
        float4v p[WAVES / 4];
#pragma unroll
        for (int i = 0; i < WAVES / 4; i++) p[i] = *reinterpret_cast<const float4v *>(&sh.red[side][r][4 * i]);
        const float4v q = (p[0] + p[1]) + (p[2] + p[3]);
        return (q[0] + q[1]) + (q[2] + q[3]);
    };
    // the sum with a branch (Gemma3: its norm first), and the norm's weight times it into LDS
    auto form = [&](const u64 *words, uint32_t tag, u64 post, u64 gamma) __attribute__((always_inline)) {
        clear();
        if (wave >= FW) {
            if (GEMMA && words) wg_barrier();
            wg_barrier();
            return;
        }
        const int c = anew(t);
        float g[S], gb[S];
#pragma unroll
        for (int i = 0; i < S; i++) {
            g[i] = *global<float>(gamma, 4 * min(c + FT * i, D - 1));
            if (GEMMA && words) gb[i] = *global<float>(post, 4 * min(c + FT * i, D - 1));
        }
        __builtin_amdgcn_sched_barrier(0);
        if (words) {
            float b[S];
            uint32_t place[S];
#pragma unroll
            for (int i = 0; i < S; i++) place[i] = min(c + FT * i, D - 1);
            await<1, 1>(words, place, tag, b, w);
            if (GEMMA) {
                float ss[2] = {0.f, 0.f};
#pragma unroll
                for (int i = 0; i < S; i++) { b[i] = c + FT * i < D ? b[i] : 0.f; ss[i & 1] = fmaf(b[i], b[i], ss[i & 1]); }
                const float sum = wave_sum(ss[0] + ss[1]);
                if (lane == 0) sh.part[0][wave] = sum;
                wg_barrier();
                const float4v p = *reinterpret_cast<const float4v *>(sh.part[0]);
                const float inv = rsqrtf(((p[0] + p[1]) + (p[2] + p[3])) / (float)D + a.eps);
#pragma unroll
                for (int i = 0; i < S; i++) x[i] = fmaf(b[i] * inv, gb[i], x[i]);
            } else
#pragma unroll
                for (int i = 0; i < S; i++) x[i] += b[i];
        }
        float ss[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < S; i++) {
            const bool live = c + FT * i < D;
            x[i] = live ? x[i] : 0.f;
            ss[i & 1] = fmaf(x[i], x[i], ss[i & 1]);
            if (live) sh.xs[xs_at(c + FT * i)] = x[i] * g[i];
        }
        const float sum = wave_sum(ss[0] + ss[1]);
        if (lane == 0) sh.part[1][wave] = sum;
        wg_barrier();
    };
    auto norm_factor = [&]() __attribute__((always_inline)) {
        const float4v p = *reinterpret_cast<const float4v *>(sh.part[1]);
        return rsqrtf(((p[0] + p[1]) + (p[2] + p[3])) / (float)D + a.eps);
    };
    float best = -INFINITY;
    int idx = 0x7fffffff;
    auto pick = [&](float ob, int oi) __attribute__((always_inline)) { if (ob > best || (ob == best && oi < idx)) { best = ob; idx = oi; } };
    for (int L = 0, kind = 0;;) {
        const bool head = L == a.NL;                       // `kind` is a part of it then
        const uint32_t tag = a.tag + L;
        // the product
        const Rows &p = sh.rows[head ? 4 : kind];
        const int steps = uniform(p.steps), cols = uniform(p.cols);
        int units = uniform(p.units), first = uniform(p.first);
        Share s;
        if (head) {
            units = min(ROWS / RW, units - ROWS / RW * kind);
            first += ROWS * kind;
            s = share_of(units * steps, steps, wave);
        } else s = Share{uniform(sh.share[wave][kind].unit), uniform(sh.share[wave][kind].step), uniform(sh.share[wave][kind].left)};
        refill();
        // the product's vector
        if (head && kind) {
            clear();
            wg_barrier();
        } else if (!(kind & 1)) {
            float ahead[3] = {};                           // what the attention needs beside the cache
            const bool fetches = attends && kind == 0 && !head && t < HD;
            if (fetches) {
                const u64 g_q = LAYER_FIELD(L, g_q), g_k = LAYER_FIELD(L, g_k), rope = LAYER_FIELD(L, rope) + (u64)a.pos * (HD / 2) * 8;
                if (g_q) ahead[0] = *global<float>(g_q, 4 * t);
                if (g_k) ahead[1] = *global<float>(g_k, 4 * t);
                ahead[2] = *global<float>(rope, 4 * t);
            }
            const int before = max(L - 1, 0);
            if (kind == 0) form(L ? a.down_w : nullptr, tag - 1, LAYER_FIELD(before, g_post_ff), head ? (u64)a.g_final : LAYER_FIELD(head ? before : L, g_in));
            else form(a.o_w, tag, LAYER_FIELD(L, g_post_attn), LAYER_FIELD(L, g_ff));
            if (fetches)
#pragma unroll
                for (int i = 0; i < 3; i++) sh.head[i][t] = ahead[i];
        } else if (kind == 1) {
            if (attends) {
                attend<HD, SI>(a, sh, L, wg, t, tag, w);
                wg_barrier();
                merge_waves<HD, SI>(a, sh, wg, t, tag);
                kind = 2;
                continue;
            }
            const int c = anew(t);
            clear();
            constexpr int SA = HD == 256 ? 1 : 4;          // columns per thread
            float o[SA];
            uint32_t place[SA];
#pragma unroll
            for (int i = 0; i < SA; i++) place[i] = min(c + TT * i, qd - 1);
            await<1, 1>(a.att_w, place, tag, o, w);
#pragma unroll
            for (int i = 0; i < SA; i++)
                if (c + TT * i < qd) sh.xs[xs_at(c + TT * i)] = o[i];
            wg_barrier();
        } else {
            const int c = anew(t);
            clear();
            float h[SI];
            uint32_t place[SI];
#pragma unroll
            for (int i = 0; i < SI; i++) place[i] = min(c + TT * i, a.IS - 1);
            await<1, 1>(a.h_w, place, tag, h, w);
#pragma unroll
            for (int i = 0; i < SI; i++)
                if (c + TT * i < a.IS) sh.xs[xs_at(c + TT * i)] = h[i];
            wg_barrier();
        }
        const float inv = kind & 1 && !head ? 1.f : norm_factor();
        run(s, steps, cols);
        wg_barrier();
        // its rows
        if (head) {
            if (t < RW * units) {
                const int row = first + t;
                const float v = row_sum(t) * inv;
                a.logits[row] = v;
                if (a.logits_host) a.logits_host[row] = v;
                pick(v, row);
            }
            if (++kind == head_parts) break;
            continue;
        }
        if (kind == 2) {
            if (t < RW / 2 * units) {                      // a unit's rows: gate, then up
                const int r = RW == 2 ? 2 * t : 4 * (t >> 1) + (t & 1);
                const float g = row_sum(r) * inv, up = row_sum(r + RW / 2) * inv;
                publish(a.h_w + first + t, tag, (GEMMA ? 0.5f * g * (1.0f + tanhf(gelu_inner(g))) : g / (1.0f + expf(-g))) * up);
            }
        } else if (t < RW * units) {
            publish((kind == 0 ? a.qkv_w : kind == 1 ? a.o_w : a.down_w) + first + t, tag, row_sum(t) * inv);
        }
        if (++kind == 4) { kind = 0; L++; }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (nothing may arrive in LDS that is no longer ours)
    if (!a.best_host) return;
    auto pick_wave = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) { const float ob = __shfl_xor(best, o, 64); const int oi = __shfl_xor(idx, o, 64); pick(ob, oi); }
    };
    // the first maximum: of the wave, of the workgroup, of all of them
    pick_wave();
    if (lane == 0) { sh.bv[wave] = best; sh.bi[wave] = idx; }
    wg_barrier();
    if (wave) return;
    best = lane < WAVES ? sh.bv[lane] : -INFINITY;
    idx = lane < WAVES ? sh.bi[lane] : 0x7fffffff;
    pick_wave();
    const uint32_t tag = a.tag + a.NL;
    if (lane == 0) { publish(a.best_w + 2 * wg, tag, best); publish(a.best_w + 2 * wg + 1, tag, __int_as_float(idx)); }
    if (wg) return;
    best = -INFINITY; idx = 0x7fffffff;
    for (int i0 = 0; i0 < nwg; i0 += 64) {
        float f[2];
        const uint32_t place[1] = {2u * min(i0 + lane, nwg - 1)};
        await<2, 1>(a.best_w, place, tag, f, w);
        pick(f[0], __float_as_int(f[1]));
    }
    pick_wave();
    if (lane == 0) *a.best_host = idx == 0x7fffffff ? 0 : idx;
}

}  // namespace

namespace lmhip {

int token_workgroups(const TokenShape &s) { return std::min(num_cus(), std::min(s.D / 4, s.IS / 2)); }

// See the kernel: whole pieces of 64 columns (a Q8_0 step's scales in whole words), vectors that its threads hold, workgroups enough for the
// heads beside the O product, rows in whole units and no more than their sums in LDS hold
bool token_fits(const TokenShape &s)
{
    if (s.D % 64 || s.D > NORMED_COLS || s.IS % 64 || s.IS > 10 * TT || (s.hd != 128 && s.hd != 256)) return false;
    if (s.Hkv <= 0 || s.Hq % s.Hkv || s.Hq * s.hd > (s.hd == 256 ? 1 : 4) * TT || s.NL <= 0 || s.NL > TOKEN_MAX_LAYERS || s.V <= 0 || s.V % 4) return false;
    const int wgs = token_workgroups(s), heads = s.Hq;
    if (2 * heads > wgs) return false;
    auto rows = [](int n, int of) { return (n / 4 + of - 1) / of * 4; };
    return rows(s.D, wgs - heads) <= ROWS && rows(2 * s.IS, wgs) <= ROWS && rows((s.Hq + 2 * s.Hkv) * s.hd, wgs) <= ROWS;
}

// Whether the one launch is the faster way: an estimate in microseconds, behind which the launches' own time does not matter.  Measured, launches ->
// one launch, greedy, contexts of 10 and 230, models of 1 to 28 layers and 4096 to 262 144 rows of the head:
// - a step without its layers 38 -> 22 (chain of the head's norm, the argmax and the wait), of which a head of 64k rows takes eight back;
// - a layer, heads of 256, widths 384 / 640 / 1152 / 1536 F16 17.5 -> 17.4 / 20.1 -> 18.2 / 27.8 -> 23.0 / 31.0 -> 29.5, Q8_0 18.3 -> 18.7 / 20.4 -> 19.2 /
//   26.2 -> 20.7 / 28.5 -> 24.4; heads of 128, 640 / 1024 / 1536 F16 17.4 -> 16.1 / 18.9 -> 17.3 / 25.0 -> 23.5, Q8_0 17.5 -> 18.3 / 17.8 -> 19.4 /
//   22.7 -> 20.7; 2048 F16 with 16 / 32 of them 30.8 -> 31.6 / 40.0 -> 37.8, Q8_0 26.0 -> 24.6 / 32.6 -> 29.1, 2560 with 32 F16 51.6 -> 48.0, Q8_0 38.5 -> 36.5;
// - 64k rows of the head of widths 128 / 384 / 768 / 1152 / 2560, F16 2 -> 95 / 5 -> 33 / 14 -> 20 / 22 -> 28 / 51 -> 51, Q8_0 3 -> 105 / 4 -> 35 / 9 -> 20 /
//   12 -> 17 / 30 -> 41: here a workgroup takes 47 ns for a row and draws 22 GB/s (Q8_0: 18) and a narrow model has few of them (token_workgroups), a head's own
//   launch streams 6.5 TB/s with all CUs.
bool token_pays(const TokenShape &s, int q8)
{
    const float wgs = (float)token_workgroups(s), rows = (float)s.V, mb = rows * (float)s.D * (q8 ? 1.0625e-6f : 2e-6f);
    const float head = std::max(rows * 0.0465f / wgs, mb / (wgs * (q8 ? 0.018f : 0.0225f))) - mb / 6.5f;
    const float layer = s.hd == 256 ? (s.D >= 1024 ? 3.f : 1.5f) : q8 ? (s.D < 1280 ? -1.f : 1.5f) : s.Hq * s.hd > s.D ? 2.5f : s.D < 2048 ? 1.f : 0.f;
    return 15.f - 8.f * std::min(1.f, rows / 65536.f) + (float)s.NL * layer > head;
}

size_t token_words(const TokenShape &s, TokenArgs *a, u64 *base)
{
    auto padded = [](int n) { return (size_t)(n + 511) / 512 * 512; };
    size_t n = 0;
    auto take = [&](size_t k) { u64 *p = base ? base + n : nullptr; n += k; return p; };
    u64 *qkv = take(padded((s.Hq + 2 * s.Hkv) * s.hd)), *att = take(padded(s.Hq * s.hd)), *o = take(padded(s.D)), *h = take(padded(s.IS)), *down = take(padded(s.D));
    u64 *best = take(padded(2 * token_workgroups(s)));
    if (a) { a->qkv_w = qkv; a->att_w = att; a->o_w = o; a->h_w = h; a->down_w = down; a->best_w = best; }
    return n;
}

void launch_token(const TokenArgs &a, const TokenShape &s, int q8)
{
    const int wgs = token_workgroups(s);
    const bool wide = s.D > 5 * FT || s.IS > 7 * TT;
#define TOKEN_LAUNCH(F_, S_, I_, H_, G_) hipLaunchKernelGGL((k_token<F_, S_, I_, H_, G_>), dim3(wgs), dim3(TT), 0, stream(), a)
#define TOKEN_MODEL(F_, S_, I_) do { \
    if (s.hd == 256) { if (a.gemma) TOKEN_LAUNCH(F_, S_, I_, 256, true); else TOKEN_LAUNCH(F_, S_, I_, 256, false); } \
    else { if (a.gemma) TOKEN_LAUNCH(F_, S_, I_, 128, true); else TOKEN_LAUNCH(F_, S_, I_, 128, false); } } while (0)
#define TOKEN_WIDTH(F_) do { if (wide) TOKEN_MODEL(F_, 10, 10); else TOKEN_MODEL(F_, 5, 7); } while (0)
    if (q8) TOKEN_WIDTH(1); else TOKEN_WIDTH(0);
#undef TOKEN_WIDTH
#undef TOKEN_MODEL
#undef TOKEN_LAUNCH
    HIP_CHECK(hipGetLastError());
}

}  // namespace lmhip
