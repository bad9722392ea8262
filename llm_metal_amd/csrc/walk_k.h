// The walk of a workgroup of four waves through K that the products of many rows share: BM rows of an operand A against 256 rows of an
// operand W, both in the tiled layout, into accumulators of assembly (acc_tiles.h).
#pragma once
#include "acc_tiles.h"

namespace lmhip {

constexpr int walk_buffer(int BM) { return (BM / 32 + 8) * 128; }     // half8 per buffer of the ring: [BM / 32 A + 8 W row blocks][2 slices][64]

// an address that is the same in every lane, in scalar registers
__device__ __forceinline__ uint64_t uniform_address(const void *p)
{
    const uint64_t x = reinterpret_cast<uint64_t>(p);
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32;
}

// The steps go from L2/HBM straight into LDS (global_load_lds_dwordx4: a wave-uniform LDS base in M0, lane i's 16 bytes land at base + 16 i --
// the [j][lane] order of the tiles).  K goes in half steps of 32 (two of a tile's four 1 KB slices per row block) through a ring of
// NB buffers: half step h is multiplied out of registers while h + 1 is read from LDS and up to h + NB are on their way.  The barrier that
// ends half step h - 1 finds h and h + 1 in LDS (every wave has waited for its own copies of them), so the fragments of h + 1 are read under
// the MFMAs of h; h + NB is requested into the buffer that h has left.  The copies are assembly, outside the compiler's count of its own loads
// (it cannot tell which LDS bytes a pending copy writes and would wait for all of them before every LDS read), and so are the waits.
//
// src: this wave's share, the first tile of A row blocks w (, 4 + w) and of W row blocks w, 4 + w of the block; a_off: the lane's byte in a
// slice of A.  Wave (wm, wn) = (w / 2, w % 2) ends with rows wm BM / 2 .. of A and wn 128 .. of W in tiles i (BM / 32) + j: A rows 16 j, W rows 16 i;
// lane l has W row l & 15 and A rows 4 (l >> 4) .. + 3 of a tile.  nhalf is even and at least two; behind it the ring is free for other use.
template <int BM, int NB>
__device__ __forceinline__ void walk_k(half8 *const lds, const uint64_t (&src)[BM / 128 + 2], uint32_t a_off, int nhalf)
{
    constexpr int AB = BM / 32, MI = BM / 32, AU = AB / 4, HB = walk_buffer(BM);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave >> 1, wn = wave & 1, last = nhalf - 1;
    const uint32_t w_off = lane * 16;
    typedef __attribute__((address_space(3))) void lds_void;
    const uint32_t place0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void *)lds + wave * 2048);
    constexpr int COPIES = 2 * (AU + 2);                      // of 1 KB, per half step and wave
    static_assert(NB * COPIES < 64, "the hand-written waits count this wave's LDS-direct loads; vmcnt has six bits");
    // copy c of half step hs (koff = 2048 hs) into the buffer that this wave's first place `place` lies in
    auto copy = [&](uint32_t place, uint32_t koff, int c) __attribute__((always_inline)) {
        const int u = c >> 1;
        const uint32_t off = (u < AU ? a_off : w_off) + koff;
        if (c & 1) asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024" :: "v"(off), "s"(src[u]), "s"(place), "n"(u * 8192) : "m0", "scc");
        else asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(off), "s"(src[u]), "s"(place), "n"(u * 8192) : "m0", "scc");
    };
    const half8 *const frag = lds + (lane >> 5) * 64 + ((lane >> 4) & 1) * 32 + (lane & 15);
    const half8 *const fa = frag + MI / 2 * wm * 128, *const fw = frag + (AB + 4 * wn) * 128;
    auto read = [&](const half8 *f, int t, int buf) __attribute__((always_inline)) { return f[buf + (t >> 1) * 128 + (t & 1) * 16]; };

    half8 A0[MI], A1[MI], W0[8], W1[8];
    // the wait and barrier of a half step behind which `open` requests may still be under way
    auto meet = [&](int open) __attribute__((always_inline)) {
        if (NB > 5 && open >= 4) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((NB - 2) * COPIES) : "memory");
        else if (open >= 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(3 * COPIES) : "memory");
        else if (open == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(2 * COPIES) : "memory");
        else if (open == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(COPIES) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    // Half step hs: its fragments are in A and W; the next one's come out of the buffer at `nxt`; MORE: hs + NB goes into the buffer of
    // hs, at `place`.  (sched_barrier: the reads stay under the MFMAs where they are written.)
    auto step = [&](auto more, const half8 (&A)[MI], const half8 (&W)[8], half8 (&An)[MI], half8 (&Wn)[8], int hs, int nxt, uint32_t place) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more)::value;
        constexpr int READS = MI + 8, EVERY = MI == 8 ? 3 : 2;  // (256 rows: 16 reads under 48 of the 64 MFMAs; 128: 12 under 24 of 32)
        unrolled<8 * MI>([&](auto X) __attribute__((always_inline)) {
            constexpr int x = X, i = x / MI, j = x % MI, t = x / EVERY;
            if constexpr (x % EVERY == 0 && t < READS) {
                if constexpr (t < MI) An[t] = read(fa, t, nxt); else Wn[t - MI] = read(fw, t - MI, nxt);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (MORE && j == 3 && i < COPIES) copy(place, (uint32_t)(hs + NB) * 2048, i);
            AccTile<x>::add(A[j], W[i]);
        });
        __builtin_amdgcn_sched_barrier(0);
        if (MORE) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((NB - 2) * COPIES) : "memory");
        else meet(last - hs - 2);
    };
    auto request = [&](uint32_t place, int hs) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < COPIES; c++) copy(place, (uint32_t)hs * 2048, c);
    };
    // (nothing is requested past the end: a block's last half steps would wait for it -- five buffers, 3 us where all CUs do)
    request(place0, 0); request(place0 + HB * 16, 1);
#pragma unroll
    for (int h = 2; h < NB; h++) if (h <= last) request(place0 + h * HB * 16, h);
    unrolled<8 * MI>([](auto X) __attribute__((always_inline)) { AccTile<X>::clear(); });
    meet(min(NB, nhalf) - 2);                                 // the first two have landed
#pragma unroll
    for (int t = 0; t < MI; t++) A0[t] = read(fa, t, 0);
#pragma unroll
    for (int t = 0; t < 8; t++) W0[t] = read(fw, t, 0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // every wave has read buffer 0 before it is requested anew
    int nxt = HB, hs = 0;
    uint32_t place = place0;
    auto advance = [&]() __attribute__((always_inline)) {
        nxt = nxt == (NB - 1) * HB ? 0 : nxt + HB;
        place = place == place0 + (NB - 1) * HB * 16 ? place0 : place + HB * 16;
    };
    constexpr std::true_type more{};
    constexpr std::false_type done{};
    for (; hs + 1 + NB <= last; hs += 2) {
        step(more, A0, W0, A1, W1, hs, nxt, place); advance();
        step(more, A1, W1, A0, W0, hs + 1, nxt, place); advance();
    }
    if (NB % 2 && hs + NB <= last) request(place, hs + NB);   // (an odd ring: the last half step, nhalf being even)
    for (; hs < nhalf; hs += 2) {
        step(done, A0, W0, A1, W1, hs, nxt, place); advance();
        step(done, A1, W1, A0, W0, hs + 1, nxt, place); advance();
    }
    settle_tiles();
}

}  // namespace lmhip
