// An fp32 value as two fp16 pieces, for the kernels that multiply fp32 operands on the fp16 matrix cores: s x = hi + lo / 2048,
// hi the leading 11 significand bits of s x and lo what is left, both rounded to nearest: 22 bits and the sign of lo, so
// that a value is off by 2^-23 of itself at most (a quarter of all values by that, the others by nothing).  A product is
//   a b = ah bh + (ah bl + al bh) / 2048     (al bl stays away: at most 2^-22 |a b|)
// with the corrections in sums of their own, which join the leading ones at the end.
//
// s is a power of two that every row of op(A) and column of op(B) has for itself: it puts the row's largest value into
// 2^14 .. 2^15, the top of fp16's range.  A value down to 2^-28 of that has both pieces whole; what a smaller one loses is at
// most 2^-36 on the scaled axis, as much as 2^-51 of the row's largest value.  Rows that hold such values are marked,
// and an output of a marked row or column counts only from 2^6 on (scaled): the products of what was lost, at most 2^-21 each,
// then stay below 2^-27 of it each, a quarter of what an fp32 sum may lose to rounding per term.  Rows with infinities or NaN are marked as
// not to be multiplied so at all.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "bf16_pieces.h"

namespace lten_hip {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr float pair_step = 2048.0f, pair_least = 64.0f;

// What is known of a row: the exponent of its scale (above the low byte) and the marks.
constexpr int row_small = 1;   // it holds values below 2^-14 on the scaled axis
constexpr int row_zero = 2;    // nothing but zeros
constexpr int row_not = 4;     // infinities or NaN
// The bits of the row's largest magnitude, and of its smallest but zero less one (0xffffffff: none).
__device__ __forceinline__ int row_info(uint32_t largest, uint32_t smallest)
{
	if (largest >= 0x7f800000u) return row_not;
	if (largest == 0) return row_zero;
	// largest in 2^e .. 2^(e + 1); denormal ones count as 2^-126 (they are scaled to less than the range then), and the scale
	// stays a normal number with 2048 times it in range
	const int e = max((int)(largest >> 23), 1) - 127, up = min(14 - e, 112);
	const float least = __builtin_bit_cast(float, smallest + 1) * __builtin_ldexpf(1.0f, up);
	return up * 256 + (least < 0x1p-14f ? row_small : 0);
}

// Eight values as their pieces.
__device__ __forceinline__ void pair8(const float (&v)[8], float scale, uint4& hi, uint4& lo)
{
	uint32_t h[4], l[4];
#pragma unroll
	for (int e = 0; e < 4; e++) {
		const float s0 = v[2 * e] * scale, s1 = v[2 * e + 1] * scale;
		const f16x2 lead = __builtin_convertvector((f2){ s0, s1 }, f16x2);
		const f2 rest = { __builtin_fmaf((float)lead.x, -pair_step, s0 * pair_step), __builtin_fmaf((float)lead.y, -pair_step, s1 * pair_step) };
		h[e] = __builtin_bit_cast(uint32_t, lead);
		l[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, f16x2));
	}
	hi = make_uint4(h[0], h[1], h[2], h[3]);
	lo = make_uint4(l[0], l[1], l[2], l[3]);
}

}  // namespace lten_hip
