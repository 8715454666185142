// fp32 contractions on the bf16 matrix pipe, with nothing lost from the fp32 operands.
//
// gfx950 multiplies bf16 sixteen times as fast as fp32 (v_mfma_f32_32x32x16_bf16: 32 clocks for sixteen k of a 32 x 32 block;
// v_mfma_f32_32x32x2_f32: 64 clocks for two). A float has 24 significant bits, a bf16 has 8, and
//   x = hi + mid + lo,  hi = bf16(x), mid = bf16(x - hi), lo = x - hi - mid
// is exact: rounding to nearest leaves |x - hi| <= 2^-8 of x's leading bit in at most 16 bits, of which mid takes 8 and leaves
// at most 6. A product of two such sums is nine bf16 products, each exact in fp32. Six of them are formed; the three left out
// (mid*lo, lo*mid, lo*lo) are together at most 2^-24 of the product, the unit roundoff of one fp32 multiplication. All sums are
// fp32, in the accumulators of the MFMA. Six sixteenths of the fp32 time per product remain: at the rates the pipes sustain on
// this part (1.82 PFLOP/s bf16, 155 TFLOP/s fp32, dense random operands) 303 against 155 TFLOP/s of fp32 work.
// Measured distance from float64 (2-norm; fp32 MFMA / these products): N(0,1) products of K = 90 on 256-wide tiles 1.70e-7 / 0.97e-7,
// 256 x 4096 x 4096 on 128-wide ones 5.75e-7 / 3.53e-7, 777 on 64-wide ones 4.98e-7 / 1.14e-7; layers behind a ReLU, forward, data
// and weight gradient: 64 -> 64 @56 3.03e-7 / 1.04e-7, 4.28e-7 / 1.35e-7, 2.71e-7 / 1.45e-7, 256 -> 256 @14 5.85e-7 / 2.20e-7, 8.31e-7 /
// 2.79e-7, 2.47e-7 / 1.15e-7. Sixteen k's share a rounding of the sum (weight gradients: two), or six where the parts share
// accumulators (products on tiles of 128 and 256, whose registers hold no second set). These six are not unbiased on the matrix
// pipe: 512 x 2048 x 4096 of U(0,1) is 6.2e-7 off, all of it one-sided (fp32 3.2e-7).
// An operand that is infinite, or beyond the range that is split (kSplitUp), has NaN among its parts, so it always shows
// as NaN in the sum. Sums that are not finite are formed once more from the fp32 operands and are those of an fp32 contraction
// (infinities keep their sign, large finite values stay finite). Convolutions: on the fp32 MFMA, straight from memory, by waves
// for their blocks (one infinity in 64 -> 64 @56 batch 32: 68 -> 109 us, a channel of infinities 269, its weight gradient 66 ->
// 709 and 757; element by element the forward pass took 3.2 and 7.2 ms). Products the same, by blocks (4096^3 overflowing
// throughout 0.65 -> 4.6 ms).
#pragma once
#include "crb_common.h"

namespace crb {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef u32 u32x4 __attribute__((ext_vector_type(4)));

constexpr int kSplit = 3;  // bf16 parts of a float

// The three parts of two floats, packed (x0 in the low half).
__device__ __forceinline__ void split_pair(float x0, float x1, u32 &hi, u32 &mid, u32 &lo) {
    const u32 h = __builtin_bit_cast(u32, __builtin_convertvector(f32x2{x0, x1}, bf16x2));
    const float r0 = x0 - __builtin_bit_cast(float, h << 16), r1 = x1 - __builtin_bit_cast(float, h & 0xffff0000u);
    const u32 m = __builtin_bit_cast(u32, __builtin_convertvector(f32x2{r0, r1}, bf16x2));
    const float s0 = r0 - __builtin_bit_cast(float, m << 16), s1 = r1 - __builtin_bit_cast(float, m & 0xffff0000u);
    hi = h, mid = m, lo = __builtin_bit_cast(u32, __builtin_convertvector(f32x2{s0, s1}, bf16x2));
}

// Operands are split at 2^16 times their value and the sums taken back by 2^-32 (both exact): the last part of a float under
// 2^-110 has bits below 2^-133, which a bf16 cannot hold; at 2^16 times the value it has none, down to the smallest float. What
// the scale moves out of range, operands from 2^112 and sums from 2^96 up, shows as a sum that is not finite and is formed again.
constexpr float kSplitUp = 65536.f, kSplitDown = 1.f / (65536.f * 65536.f);

// The three parts of eight floats, each a 16-byte MFMA fragment (element i in 16-bit slot i).
__device__ __forceinline__ void split8(const float *x, u32x4 (&part)[kSplit]) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        u32 h, m, l;
        split_pair(x[2 * p] * kSplitUp, x[2 * p + 1] * kSplitUp, h, m, l);
        part[0][p] = h, part[1][p] = m, part[2][p] = l;
    }
}

// A float at `voffset + soffset` bytes behind a uniform base, by a buffer load: the address needs no vector arithmetic beyond
// voffset, and an element that is to read as zero (halo, channels past the tensor) is named by kOutside, which the resource's
// range check turns into 0. Ranges are under 2 GiB, and `soffset` lies inside the range also where `voffset` does not: whether the check
// takes what is left behind `soffset` for a signed number or not is then all the same.
constexpr u32 kOutside = 0x80000000u;
typedef __amdgpu_buffer_rsrc_t BufferRange;
__device__ __forceinline__ BufferRange buffer_range(const float *base, size_t floats) {
    const size_t bytes = floats * 4;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, int(bytes < 0x7fffffffu ? bytes : 0x7fffffffu), 0x00020000);
}
__device__ __forceinline__ float buffer_load(BufferRange r, u32 voffset, u32 soffset) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, int(voffset), int(soffset), 0));
}

// Where there are registers for it, the five part products behind the leading one have accumulators of their own, 2^-8 of the
// others' size: the full sum is then rounded once per sixteen k instead of six times (forward 64 -> 64 @56 behind a ReLU 3.47e-7 ->
// 1.04e-7 from float64; 32 registers, times unchanged: 81 passes of random layers 0.99 of what they were in the mean).
template <class V, int TM, int TN>
__device__ __forceinline__ void add_small(V (&acc)[TM][TN], const V (&small)[TM][TN]) {
#pragma unroll
    for (int mi = 0; mi < TM; ++mi)
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mi][ni][r] += small[mi][ni][r];
}

// A lane's accumulators at their own scale; whether one of them is not finite.
template <class V, int TM, int TN>
__device__ __forceinline__ bool scale_down(V (&acc)[TM][TN]) {
    bool bad = false;
#pragma unroll
    for (int mi = 0; mi < TM; ++mi)
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mi][ni][r] *= kSplitDown, bad |= !__builtin_isfinite(acc[mi][ni][r]);
    return bad;
}

// The products that are formed: (part of A, part of B), the smallest first: where one term is most of a sum, the roundings before
// the last are then of its small parts (a sum of one product: off by 1.45 units in the last place at most, rms 0.39, or 0.95 and
// 0.30 with accumulators of their own for the small ones; the other way round 3.38 and 0.60; one fp32 multiplication 0.5 and 0.29). kPartOrder: the parts in the order in which they are needed.
constexpr int kTerms = 6;
constexpr int kTermA[kTerms] = {2, 0, 1, 1, 0, 0};
constexpr int kTermB[kTerms] = {0, 2, 1, 0, 1, 0};
constexpr int kPartOrderA[kSplit] = {2, 0, 1}, kPartOrderB[kSplit] = {0, 2, 1};

}  // namespace crb
