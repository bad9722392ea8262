// Accumulators that stay where they are: 64 tiles of v_mfma_f32_16x16x32_f16, four registers each, tile T in a[4 T : 4 T + 3].
//
// Written as assembly on named registers, because the compiler does not keep that many small tiles in place: with the builtin it gives
// a product's result other registers than its operand and copies whole tiles between the register files all through a loop (32x32
// tiles, which it cannot move so freely, it leaves), and as "+a" operands of assembly it still moves one now and then, next to an
// instruction whose result is not there yet -- it does not know what the assembly does.  Every instruction here names its tile
// as overwritten, so no value of the compiler's own lives in these registers across one; between them it takes them for free.  So a kernel that uses
// them has to give it no reason to: check_acc.py reads the assembly of every build and stops it where the compiler names an accumulation
// register, spills, or writes an MFMA's operand too short ahead of it (its hazard pass does not look inside assembly).  (Vector registers taken
// today: gemm_big_pair 254 of 256, gemm_big_f16<256> 156, k_wgrad_block<2> 106 of the 128 beside its tiles.)
// Who reads a tile (take) keeps it 18 cycles or more behind the last instruction that wrote it: settle_tiles().
#pragma once
#include "devutil.h"
#include <type_traits>
#include <utility>

namespace lmhip {

template <int T> struct AccTile;
#define LMHIP_ACC(T, R0, R1, R2, R3) \
    template <> struct AccTile<T> { \
        static __device__ __forceinline__ void clear() \
        { \
            asm volatile("v_accvgpr_write_b32 a" #R0 ", 0\n\tv_accvgpr_write_b32 a" #R1 ", 0\n\tv_accvgpr_write_b32 a" #R2 ", 0\n\tv_accvgpr_write_b32 a" #R3 ", 0" \
                         ::: "a" #R0, "a" #R1, "a" #R2, "a" #R3); \
        } \
        /* 16 rows of a x 16 rows of w over K = 32; lane l: column l & 15 (w), rows 4 (l >> 4) .. + 3 (a) */ \
        static __device__ __forceinline__ void add(half8 a, half8 w) \
        { \
            asm volatile("v_mfma_f32_16x16x32_f16 a[" #R0 ":" #R3 "], %0, %1, a[" #R0 ":" #R3 "]" :: "v"(a), "v"(w) : "a" #R0, "a" #R1, "a" #R2, "a" #R3); \
        } \
        /* the same on a tile that begins anew */ \
        static __device__ __forceinline__ void begin(half8 a, half8 w) \
        { \
            asm volatile("v_mfma_f32_16x16x32_f16 a[" #R0 ":" #R3 "], %0, %1, 0" :: "v"(a), "v"(w) : "a" #R0, "a" #R1, "a" #R2, "a" #R3); \
        } \
        /* register R of the tile */ \
        template <int R> static __device__ __forceinline__ float take_one() \
        { \
            float x; \
            if constexpr (R == 0) asm volatile("v_accvgpr_read_b32 %0, a" #R0 : "=v"(x)); \
            else if constexpr (R == 1) asm volatile("v_accvgpr_read_b32 %0, a" #R1 : "=v"(x)); \
            else if constexpr (R == 2) asm volatile("v_accvgpr_read_b32 %0, a" #R2 : "=v"(x)); \
            else asm volatile("v_accvgpr_read_b32 %0, a" #R3 : "=v"(x)); \
            return x; \
        } \
        static __device__ __forceinline__ float4v take() \
        { \
            float4v x; \
            float x0, x1, x2, x3; \
            asm volatile("v_accvgpr_read_b32 %0, a" #R0 "\n\tv_accvgpr_read_b32 %1, a" #R1 "\n\tv_accvgpr_read_b32 %2, a" #R2 "\n\tv_accvgpr_read_b32 %3, a" #R3 \
                         : "=v"(x0), "=v"(x1), "=v"(x2), "=v"(x3)); \
            x[0] = x0; x[1] = x1; x[2] = x2; x[3] = x3; \
            return x; \
        } \
    };
LMHIP_ACC(0, 0, 1, 2, 3) LMHIP_ACC(1, 4, 5, 6, 7) LMHIP_ACC(2, 8, 9, 10, 11) LMHIP_ACC(3, 12, 13, 14, 15)
LMHIP_ACC(4, 16, 17, 18, 19) LMHIP_ACC(5, 20, 21, 22, 23) LMHIP_ACC(6, 24, 25, 26, 27) LMHIP_ACC(7, 28, 29, 30, 31)
LMHIP_ACC(8, 32, 33, 34, 35) LMHIP_ACC(9, 36, 37, 38, 39) LMHIP_ACC(10, 40, 41, 42, 43) LMHIP_ACC(11, 44, 45, 46, 47)
LMHIP_ACC(12, 48, 49, 50, 51) LMHIP_ACC(13, 52, 53, 54, 55) LMHIP_ACC(14, 56, 57, 58, 59) LMHIP_ACC(15, 60, 61, 62, 63)
LMHIP_ACC(16, 64, 65, 66, 67) LMHIP_ACC(17, 68, 69, 70, 71) LMHIP_ACC(18, 72, 73, 74, 75) LMHIP_ACC(19, 76, 77, 78, 79)
LMHIP_ACC(20, 80, 81, 82, 83) LMHIP_ACC(21, 84, 85, 86, 87) LMHIP_ACC(22, 88, 89, 90, 91) LMHIP_ACC(23, 92, 93, 94, 95)
LMHIP_ACC(24, 96, 97, 98, 99) LMHIP_ACC(25, 100, 101, 102, 103) LMHIP_ACC(26, 104, 105, 106, 107) LMHIP_ACC(27, 108, 109, 110, 111)
LMHIP_ACC(28, 112, 113, 114, 115) LMHIP_ACC(29, 116, 117, 118, 119) LMHIP_ACC(30, 120, 121, 122, 123) LMHIP_ACC(31, 124, 125, 126, 127)
LMHIP_ACC(32, 128, 129, 130, 131) LMHIP_ACC(33, 132, 133, 134, 135) LMHIP_ACC(34, 136, 137, 138, 139) LMHIP_ACC(35, 140, 141, 142, 143)
LMHIP_ACC(36, 144, 145, 146, 147) LMHIP_ACC(37, 148, 149, 150, 151) LMHIP_ACC(38, 152, 153, 154, 155) LMHIP_ACC(39, 156, 157, 158, 159)
LMHIP_ACC(40, 160, 161, 162, 163) LMHIP_ACC(41, 164, 165, 166, 167) LMHIP_ACC(42, 168, 169, 170, 171) LMHIP_ACC(43, 172, 173, 174, 175)
LMHIP_ACC(44, 176, 177, 178, 179) LMHIP_ACC(45, 180, 181, 182, 183) LMHIP_ACC(46, 184, 185, 186, 187) LMHIP_ACC(47, 188, 189, 190, 191)
LMHIP_ACC(48, 192, 193, 194, 195) LMHIP_ACC(49, 196, 197, 198, 199) LMHIP_ACC(50, 200, 201, 202, 203) LMHIP_ACC(51, 204, 205, 206, 207)
LMHIP_ACC(52, 208, 209, 210, 211) LMHIP_ACC(53, 212, 213, 214, 215) LMHIP_ACC(54, 216, 217, 218, 219) LMHIP_ACC(55, 220, 221, 222, 223)
LMHIP_ACC(56, 224, 225, 226, 227) LMHIP_ACC(57, 228, 229, 230, 231) LMHIP_ACC(58, 232, 233, 234, 235) LMHIP_ACC(59, 236, 237, 238, 239)
LMHIP_ACC(60, 240, 241, 242, 243) LMHIP_ACC(61, 244, 245, 246, 247) LMHIP_ACC(62, 248, 249, 250, 251) LMHIP_ACC(63, 252, 253, 254, 255)
#undef LMHIP_ACC

// the last products' results, before take() reads them
__device__ __forceinline__ void settle_tiles() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// f(0) .. f(N - 1) with the number as a constant
template <int N, typename F, int... I> __device__ __forceinline__ void unrolled_(F &&f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F> __device__ __forceinline__ void unrolled(F &&f) { unrolled_<N>(f, std::make_integer_sequence<int, N>{}); }

}  // namespace lmhip
