// fp32 products on the bf16 matrix pipes, at fp32 accuracy.
//
// A float is the sum of three bf16 numbers without a remainder (8 + 8 + 8 significand bits): x = h + m + l with
// h = bf16(x), m = bf16(x - h), l = x - h - m.  Of the nine products of two such sums, six are kept -- hh, hm, mh, mm, hl,
// lh; the other three are each at most 2^-25 of the product, together at most 2^-24 (2^-24.2 found over 2e6 pairs), and of either
// sign.  (The method is Henry, Tang and Heinecke's: "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019.)  The large products have one accumulator and the five small ones another, added at the end: errors
// against 64 bits over 64 x 1024 sums of normal numbers, v_mfma_f32_32x32x2_f32 / the six v_mfma_f32_32x32x16_bf16 that replace
// eight of it: 6.1e-7 / 2.0e-7 at 1152 terms, 1.2e-6 / 4.2e-7 at 4608; in one accumulator 5.2e-7 and 1.07e-6.
// The instruction adds eight products at a time and the two sums to the accumulator, each rounded to nearest; inside the
// eight what lies below the last place of the largest product is cut off, towards zero.  Sums of numbers of one sign come out no
// closer than on the fp32 pipe, and further off where a product's ranges are longer here: 2048^3 of positive numbers 2.1e-7 /
// 1.1e-7, 512 x 1000 x 784 5.9e-8 / 4.2e-8.
//
// Rate: 16 fp32 cycles against 6 * 16 / 16: 2.67 times the fp32 pipe's; a register-resident loop over random operands sustains
// 314 TFLOP/s of fp32 work (power-limited; 415 with constant operands), the fp32 instruction 153.
//
// A bf16 number has fewer places below the point than a float (2^-133 against 2^-149), so that the lower parts of numbers below
// 2^-110 would be lost.  Every number is multiplied by 2^16 before it is split, a sum by 2^-32 when it is finished: all floats
// are carried whole, subnormal ones too (the pipes keep subnormal operands and sums), and a sum is rounded below the smallest
// normal float as a float is.  Eight multiplications beside the 46 vector instructions that split eight numbers: 256 -> 256
// channels, 8 x 8 maps, 256 images, forward 105 us with and without.
//
// What the split does not carry are an infinity and a NaN (whose lower parts are not numbers), numbers from 2^112 and sums from
// 2^96 on.  They end in a sum that is not finite; the tile is then computed by a plain fp32 chain (split_sum_suspect): that
// convolution with an infinity in it 6.0 ms.  (Sums below 2^-90 went there too before the numbers were scaled, and one image
// classified without doubt -- errors of 2^-100 -- took a backward pass of AlexNet at 64 images from 1.9 to 58 ms.)
#pragma once
#include "gemm_engine.h"

namespace fitre {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t bf16_pair(float a, float b)
{
	bf16x2 r;
	r[0] = (__bf16)a, r[1] = (__bf16)b; // round to nearest even
	return __builtin_bit_cast(uint32_t, r);
}
constexpr float kSplitScale = 0x1p16f, kSplitSumScale = 0x1p-32f; // of what is split; of a sum of products of two such numbers
// two floats -> the three bf16 parts of their multiples, packed (a in the low half)
__device__ __forceinline__ void split_pair(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l)
{
	a *= kSplitScale, b *= kSplitScale;
	h = bf16_pair(a, b);
	const float ra = a - __builtin_bit_cast(float, h << 16), rb = b - __builtin_bit_cast(float, h & 0xffff0000u);
	m = bf16_pair(ra, rb);
	l = bf16_pair(ra - __builtin_bit_cast(float, m << 16), rb - __builtin_bit_cast(float, m & 0xffff0000u));
}
// eight floats, consecutive in the reduction -> one 16-byte fragment word per part
__device__ __forceinline__ void split_eight(const float (&x)[8], u32x4 (&part)[3])
{
#pragma unroll
	for (int q = 0; q < 4; q++) {
		uint32_t h, m, l;
		split_pair(x[2 * q], x[2 * q + 1], h, m, l);
		part[0][q] = h, part[1][q] = m, part[2][q] = l;
	}
}

__device__ __forceinline__ v16f mfma_bf16(u32x4 a, u32x4 b, v16f c)
{
	return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

typedef float quad4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ quad4f buffer_load4(__amdgpu_buffer_rsrc_t r, uint32_t byteOffset)
{
	return __builtin_bit_cast(quad4f, __builtin_amdgcn_raw_buffer_load_b128(r, (int)byteOffset, 0, 0));
}

// an offset that stays out of range with a few words added to it
constexpr uint32_t kSplitNowhere = 0xFFFFFF00u;

constexpr int kTileSplit = 10, kTileSplitCell = 11; // profile variants of these kernels

// a sum that the split may not have carried: not finite
__device__ __forceinline__ bool split_sum_suspect(float v) { return (__builtin_bit_cast(uint32_t, v) & 0x7f800000u) == 0x7f800000u; }

} // namespace fitre
