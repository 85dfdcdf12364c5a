// An fp32 value as three bf16 pieces that add up to it exactly, shared by the kernels that multiply fp32 operands on the
// bf16 matrix cores (the splitting of Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for
// higher-precision computations", ARITH 2019): 2^24 x = hi + mid + lo (24 significand bits in three times 8, each piece
// what is left rounded to nearest), and a product as the sum of its six piece products of weight 2^-16 and above, each
// exact, accumulated in fp32:
//   a b = ah bh + (ah bm + am bh) + (ah bl + am bm + al bh)     (am bl + al bm + al bl stay away: at most 2^-24 |a b|)
// The factor 2^24 puts the last bit of the smallest denormal (2^-149) at 2^-125, so that every piece of every value is zero
// or a normal bf16, however far its neighbours are from it.  The sums carry 2^48, which the kernels take off at their end.
// What has no such pieces or sums comes out as NaN or infinite: infinities, NaN, values from 2^103 on and sums that reach 2^80 on their way.
// The kernels compute such tiles again with the fp32 instructions.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace lten_hip {

typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// the order of the piece products of one k-step, the smallest first: piece of a, piece of b
constexpr int piece_a[6] = { 0, 2, 1, 0, 1, 0 }, piece_b[6] = { 2, 0, 1, 1, 0, 0 };
constexpr float pieces_scale = 0x1p24f, pieces_unscale = 0x1p-48f;

// The leading 8 significand bits of two values (rounded to nearest) as packed bf16; x becomes what is left, exactly.
__device__ __forceinline__ uint32_t split_off(float& x0, float& x1)
{
	const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){ x0, x1 }, bf16x2));
	x0 -= __builtin_bit_cast(float, u << 16);
	x1 -= __builtin_bit_cast(float, u & 0xffff0000u);
	return u;
}

// What is left of two values after two pieces, as packed bf16.
__device__ __forceinline__ uint32_t split_last(float x0, float x1)
{
	return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){ x0, x1 }, bf16x2));
}

// Eight values, scaled already, as their pieces, every step for all of them before the next one: a SIMD has one
// converting wavefront, and an instruction that waits for the one before it leaves it idle, one that waits for the fourth before it
// hardly (with this order and fewer cache lines a load the weight gradient of 32 x 32 x 128 x 128 -> 64 went from 115 to 99 us).
__device__ __forceinline__ void split8_scaled(float (&v)[8], uint4 (&piece)[3])
{
	uint32_t u[3][4];
#pragma unroll
	for (int k = 0; k < 3; k++) {
#pragma unroll
		for (int e = 0; e < 4; e++) u[k][e] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){ v[2 * e], v[2 * e + 1] }, bf16x2));
		__builtin_amdgcn_sched_barrier(0);
		if (k == 2) break;
		float h[8];
#pragma unroll
		for (int e = 0; e < 4; e++) {
			h[2 * e] = __builtin_bit_cast(float, u[k][e] << 16);
			h[2 * e + 1] = __builtin_bit_cast(float, u[k][e] & 0xffff0000u);
		}
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int e = 0; e < 8; e++) v[e] -= h[e];
		__builtin_amdgcn_sched_barrier(0);
	}
#pragma unroll
	for (int k = 0; k < 3; k++) piece[k] = make_uint4(u[k][0], u[k][1], u[k][2], u[k][3]);
}

// Eight values as their pieces.
__device__ __forceinline__ void split8(float (&v)[8], uint4 (&piece)[3])
{
#pragma unroll
	for (int e = 0; e < 8; e++) v[e] *= pieces_scale;
	__builtin_amdgcn_sched_barrier(0);
	split8_scaled(v, piece);
}

// The scale of value e of a group whose values that count are marked in `bits`, zero for the others (an infinity times it is a
// NaN, and what it reaches is computed again on the values themselves).
__device__ __forceinline__ float scale_where(uint32_t bits, int e)
{
	return __builtin_bit_cast(float, (uint32_t)((int)(bits << (31 - e)) >> 31) & __builtin_bit_cast(uint32_t, pieces_scale));
}

}  // namespace lten_hip
