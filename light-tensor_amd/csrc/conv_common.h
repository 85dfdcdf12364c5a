// Geometry of one Conv2d call and the entry points of the specialised convolution kernels.
#pragma once

#include "common.h"

#include <hip/hip_runtime.h>

namespace lten_hip {

struct ConvGeo {
	int N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw, dh, dw, Ho, Wo;
};

// Kernels for stride 1, dilation 1 that stage the input patch of an output tile in LDS (conv_patch.hip).
// *_takes: whether the kernel family covers this geometry and these pointers.
bool conv_patch_forward_takes(const ConvGeo& g, const float* x, const float* y);
int conv_patch_forward(const ConvGeo& g, const float* x, const float* w, const float* bias, float* y);
// the same tile with the LDS patch filled by direct global->LDS loads (conv_patch_fast.hip)
bool conv_patch_fast_forward_takes(const ConvGeo& g, const float* x, const float* w);
int conv_patch_fast_forward(const ConvGeo& g, const float* x, const float* w, const float* bias, float* y);
double conv_patch_fast_forward_us(const ConvGeo& g);  // what it is expected to take
bool conv_patch_wgrad_takes(const ConvGeo& g);
int conv_patch_wgrad_parts(const ConvGeo& g, bool upper_bound = false);  // partial [Cout x Cin*kh*kw] matrices the kernel writes
int conv_patch_wgrad(const ConvGeo& g, const float* x, const float* dy, float* partial, int parts);
// the same product with both LDS tiles filled by direct global->LDS loads (padding 1, W % 64 == 0, 16-byte aligned x and dy)
bool conv_patch_fast_wgrad_takes(const ConvGeo& g, const float* x, const float* dy);
int conv_patch_fast_wgrad(const ConvGeo& g, const float* x, const float* dy, float* partial, int parts);

// Forward and data gradient on the bf16 matrix cores (conv_split.hip): -1 when no tile takes the shape, its memory cannot be
// had or its estimated time is not below `limit_us`; forced: tile number (from 1) whatever the estimates, 0 the quickest.
int conv_split_forward(const ConvGeo& g, const float* x, const float* w, const float* bias, float* y, double limit_us, int forced);
int conv_split_dgrad(const ConvGeo& g, const float* w, const float* dy, float* dx, double limit_us, int forced);
int conv_split_wgrad(const ConvGeo& g, const float* x, const float* dy, float* dw, double limit_us);  // 3 x 3 (conv_split_wgrad.hip)

// 3x3, stride 1, at most four output channels: a stream over x on the vector ALUs (conv_fewout.hip).  dgrad: w is the
// weight array of the convolution whose data gradient is computed, read transposed and flipped in place.
bool conv_fewout_takes(const ConvGeo& g, const float* x, const float* y);
int conv_fewout_forward(const ConvGeo& g, const float* x, const float* w, const float* bias, float* y, bool dgrad);

// 3x3, stride 1, one or two input channels: a stream of y from registers, no LDS (conv_fewin.hip).
bool conv_fewin_takes(const ConvGeo& g, const float* x, const float* y);
int conv_fewin_forward(const ConvGeo& g, const float* x, const float* w, const float* bias, float* y);

// Kernels for stride 1, dilation 1 and Cin*kh*kw <= 32 (first layers): the whole reduction fits one MFMA tile
// dimension, the work is bound by the HBM traffic of y / dy (conv_smallk.hip).
bool conv_smallk_takes(const ConvGeo& g);
int conv_smallk_forward(const ConvGeo& g, const float* x, const float* w, const float* bias, float* y);
int conv_smallk_wgrad_parts(const ConvGeo& g);
int conv_smallk_wgrad(const ConvGeo& g, const float* x, const float* dy, float* partial, int parts);

// Sums `parts` partial matrices of `count` floats in a fixed order.
int conv_reduce_partials(const float* partial, int parts, int64_t count, float* out);

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Quotients of numbers below 2^31 by a divisor that a whole launch shares: n / d = (n ceil(2^(31 + s) / d)) >> (31 + s) for
// 2^(s - 1) < d <= 2^s (Granlund and Montgomery, "Division by invariant integers using multiplication", PLDI 1994).
struct Divisor {
	uint32_t mul, shift;
};
inline Divisor make_divisor(uint32_t d)
{
	Divisor r = { 0, 0 };
	while ((1ull << r.shift) < d) r.shift++;
	r.mul = (uint32_t)(((1ull << (31 + r.shift)) + d - 1) / d);
	return r;
}

#if defined(__HIPCC__)
__device__ __forceinline__ int quotient(int n, Divisor d) { return (int)(__umulhi((uint32_t)n << 1, d.mul) >> d.shift); }

// Four consecutive floats of a row starting at column gx; columns outside [0, limit) read as 0.  With VEC
// (limit % 4 == 0, gx % 4 == 0, 16-byte aligned row) the four are inside or outside together.
template <bool VEC>
__device__ __forceinline__ float4 load_row4(const float* row, int gx, int limit)
{
	float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	if (VEC) {
		if (gx >= 0 && gx + 3 < limit) v = *reinterpret_cast<const float4*>(row + gx);
	} else {
		if (gx >= 0 && gx < limit) v.x = row[gx];
		if (gx + 1 >= 0 && gx + 1 < limit) v.y = row[gx + 1];
		if (gx + 2 >= 0 && gx + 2 < limit) v.z = row[gx + 2];
		if (gx + 3 >= 0 && gx + 3 < limit) v.w = row[gx + 3];
	}
	return v;
}
#endif

}  // namespace lten_hip
