// Conv2d_q forward: uint8 input (NCHW) x uint8 weights -> int32 -> requantized uint8, for the whole batch.
//
// l-ten does this per image as a u8 im2col followed by quantized_matmul(false, false, Cout, Ho*Wo, Cin*kh*kw)
// with the weights as the left operand (l-ten/conv2d.cpp:355-372): element = sum_k w[co][k] * col[k][p]
//   - zpW * sum_k col[k][p] - zpIn * sum_k w[co][k] + K * zpW * zpIn (+ bias[p]), then the requantize of
// l-ten/math_fns.cpp:1474.  Positions outside the image hold the byte 0 in the column buffer (not the zero point).
//
// Windows of at most 64 taps for fewer than 48 output channels (the 1 -> 10 channel 5x5 layer of l-ten's quantized
// MNIST network has 25 taps) run in one launch without a column buffer: a thread owns one output position, gathers its window into 16 packed dwords,
// and takes the products with unsigned dot4 instructions against the weights of up to 64 output channels held in
// LDS; consecutive lanes are consecutive positions of a row, so loads and the byte stores of y run along rows.
// Longer windows also run in one launch where the weights fit LDS beside the image (small images, at most 64 output
// channels) or, a block of output channels at a time, beside the input rows of a band of output rows (any image):
// convq_image.hip.  Other longer
// windows run as three launches for the whole batch (the first also pads the weights): the patches of all output
// positions as rows of a
// [N * Ho * Wo][K] matrix (K padded to a multiple of 16 with the input zero point, the weights padded alike with
// theirs, so the padding multiplies to nothing), one int8 GEMM of qgemm.hip with the positions as rows (NT: both
// operands contiguous in K, the shape its MFMA tiles are built for) into int32 sums, and a pass that adds l-ten's
// per-position bias, requantizes and stores in NCHW order.  When the workspace that needs would exceed 2 GiB the
// call follows l-ten's own decomposition image by image: im2col_u8, then the GEMM with the weights on the left.
// Layers with more work than launches run as two: pixels of channels, then an implicit GEMM (convq_pixels.hip).
#include <algorithm>
#include <optional>
#include <type_traits>
#include "conv_common.h"
#include "qgemm_common.h"

namespace lten_hip {

constexpr int CQ_MAXK = 64, CQ_CO = 64;

// one launch for small images with windows above 64 taps (convq_image.hip); -1 = not a shape for it
int conv2dq_image_dispatch(const ConvGeo& g, const uint8_t* x, const uint8_t* w, const int32_t* bias, int zp_in, int zp_w, float mult,
                           float zp_out, void* y, bool out_acc);
// one launch for larger images, a band of output rows per workgroup (convq_image.hip); -1 = not a shape for it
int conv2dq_band_dispatch(const ConvGeo& g, const uint8_t* x, const uint8_t* w, const int32_t* bias, int zp_in, int zp_w, float mult,
                          float zp_out, void* y, bool out_acc);

bool conv2dq_image_takes(const ConvGeo& g, const uint8_t* w);
double conv2dq_band_estimate_us(const ConvGeo& g);
double conv2dq_band_us(const ConvGeo& g);
// two launches, any window: the input as pixels of channels, then an implicit GEMM (convq_pixels.hip); -1 = not a shape for it
int conv2dq_pixels_dispatch(const ConvGeo& g, const uint8_t* x, const uint8_t* w, const int32_t* bias, int zp_in, int zp_w, float mult,
                            float zp_out, uint8_t* y, void* memory, int forced);
double conv2dq_pixels_us(const ConvGeo& g, uint64_t& bytes);
int conv2dq_region_dispatch(const ConvGeo& g, const uint8_t* x, const uint8_t* w, const int32_t* bias, int zp_in, int zp_w, float mult, float zp_out,
                            uint8_t* y, double limit_us);

// Windows of at most 64 taps in rows of 3 to 8: a thread holds one position's window, a row of a channel in DPR dwords, and takes its
// dot products with the output channels.  NR = rows it holds, the smallest that covers Cin * kh.
//
// Bound by latency, and by its own instructions, which a launch this short fetches for the first time: so a row is one load (25 byte
// loads and their addresses were two thirds of a 5 x 5 window's kernel; those same loads all in flight at once: 7.6 -> 6.6 us), the
// weights' byte sums are taken once a workgroup (dot products issue at a quarter of the vector rate), and where the positions leave
// the chip idle `groups` of threads share them and take a part of the channels each.  64 x 1 x 28 x 28 -> 10 channels 5 x 5:
// 7.6 -> 4.6 us, 32 x 7 x 57 x 57 -> 24 3 x 3 stride 2 17.0 -> 6.1, 64 x 4 x 112 x 112 -> 47 3 x 3 60 -> 46.  Rows of one or two taps
// and of more than eight are read byte by byte below.
template <int OUT, int DPR, int NR>
__global__ __launch_bounds__(256) void conv2dq_direct_rows_kernel(ConvGeo g, const uint8_t* __restrict__ x, const uint8_t* __restrict__ w,
                                                                  const int32_t* __restrict__ bias, int zp_in, int zp_w, float mult,
                                                                  float zp_out, void* __restrict__ y, int groups)
{
	constexpr int ND = NR * DPR;
	using row_bits = std::conditional_t<DPR == 2, uint64_t, uint32_t>;
	typedef row_bits row_any __attribute__((aligned(1)));
	__shared__ __attribute__((aligned(16))) uint32_t s_w[CQ_CO][ND];
	__shared__ uint32_t s_sum[CQ_CO];  // the byte sum of a channel's weights
	const int tid = threadIdx.x;
	const int rows = g.Cin * g.kh, K = rows * g.kw, HW = g.Ho * g.Wo;
	const int co0 = blockIdx.y * CQ_CO, nco = min(CQ_CO, g.Cout - co0);
	if (tid < CQ_CO) s_sum[tid] = 0;
	__syncthreads();

	// N * HW < 2^31 (checked by the host): 32-bit divisions
	const uint32_t share = 256u / (uint32_t)groups;
	const int group = __builtin_amdgcn_readfirstlane((int)((uint32_t)tid / share));  // (a share is whole wavefronts)
	const uint32_t gid = blockIdx.x * share + ((uint32_t)tid - (uint32_t)group * share);
	const bool live = gid < (uint32_t)g.N * (uint32_t)HW;
	const int n = live ? (int)(gid / (uint32_t)HW) : 0, pos = live ? (int)(gid - (uint32_t)n * (uint32_t)HW) : 0;
	const int ho = (int)((uint32_t)pos / (uint32_t)g.Wo), wo = pos - ho * g.Wo;
	const int y0 = ho * g.sh - g.ph, x0 = wo * g.sw - g.pw;

	// Row (ci, i) of the window: the bytes from `base` + (ci H + i) W on (x is 4 DPR to 2^31 - 2^16 bytes, checked by the host), moved
	// back inside x where they reach past an end of it and shifted into place afterwards.  Rows past the last repeat it.
	const int base = n * (g.Cin * g.H * g.W) + y0 * g.W + x0, last = g.N * (g.Cin * g.H * g.W) - 4 * DPR;
	row_bits row[NR];
	int plane_row[NR];  // ci * H + i
	{
		int i = 0, at = 0;
#pragma unroll
		for (int r = 0; r < NR; r++) {
			plane_row[r] = at;
			row[r] = *reinterpret_cast<const row_any*>(x + (uint32_t)min(max(base + at * g.W, 0), last));
			const int more = r + 1 < rows ? 1 : 0, next = i + more == g.kh ? 1 : 0;
			i = next ? 0 : i + more;
			at += more + (next ? g.H - g.kh : 0);
			asm volatile("" : "+s"(at));  // (a load for every row: one under a condition is a branch, and waits for those before it)
		}
	}

	// weights of this block's output channels, laid out as the rows are, bytes past a row's taps and rows past the last zero
	for (int idx = tid; idx < nco * ND; idx += 256) {
		const int co = idx / ND, d = idx % ND, r = d / DPR, j0 = d % DPR * 4;
		const uint8_t* wr = w + (int64_t)(co0 + co) * K;
		uint32_t byte[4], v = 0;
#pragma unroll
		for (int b = 0; b < 4; b++) byte[b] = wr[min(r * g.kw + j0 + b, K - 1)];
		asm volatile("" : "+v"(byte[0]), "+v"(byte[1]), "+v"(byte[2]), "+v"(byte[3]));  // (four loads in flight)
#pragma unroll
		for (int b = 0; b < 4; b++) v |= (r < rows && j0 + b < g.kw ? byte[b] : 0u) << (8 * b);
		s_w[co][d] = v;
		atomicAdd(&s_sum[co], __builtin_amdgcn_udot4(v, 0x01010101u, 0u, false));
	}
	__syncthreads();

	if (__any(base < 0 || base + plane_row[NR - 1] * g.W > last)) {
#pragma unroll
		for (int r = 0; r < NR; r++) {
			const int off = base + plane_row[r] * g.W, moved = off - min(max(off, 0), last);
			row[r] = moved < 0 ? row[r] << (8 * min(-moved, 4 * DPR - 1)) : row[r] >> (8 * min(moved, 4 * DPR - 1));
		}
	}
	if (!live) return;

	// taps outside the image count as 0: columns alike in every row, rows by themselves
	const int from = max(-x0, 0), to = min(g.kw, g.W - x0);
	const row_bits below_to = to >= 4 * DPR ? ~(row_bits)0 : ((row_bits)1 << (8 * max(to, 0))) - 1;
	const row_bits columns = from >= 4 * DPR ? 0 : below_to & (~(row_bits)0 << (8 * from));
	uint32_t xk[ND], xsum = 0;
	{
		int i = 0;
#pragma unroll
		for (int r = 0; r < NR; r++) {
			const row_bits v = r < rows && (unsigned)(y0 + i) < (unsigned)g.H ? row[r] & columns : 0;
#pragma unroll
			for (int d = 0; d < DPR; d++) {
				xk[r * DPR + d] = (uint32_t)(v >> (32 * d * (DPR - 1)));
				xsum = __builtin_amdgcn_udot4(xk[r * DPR + d], 0x01010101u, xsum, false);
			}
			if (++i == g.kh) i = 0;
		}
	}
	// l-ten/math_fns.cpp:1362-1380,1433: row_vector[p] = -zpA * sum_k B[k][p] with A = weights; broadcast = K zpA zpB
	const int fixed = -zp_w * (int)xsum + K * zp_w * zp_in + (bias ? bias[pos] : 0);

	const int part = (nco + groups - 1) / groups, first_co = group * part, end_co = min(first_co + part, nco);
	const int64_t out = ((int64_t)n * g.Cout + co0) * HW + pos;
	for (int co = first_co; co < end_co; co++) {
		uint32_t dot = 0;
#pragma unroll
		for (int d = 0; d < ND; d++) dot = __builtin_amdgcn_udot4(s_w[co][d], xk[d], dot, false);
		const int v = (int)dot + fixed - zp_in * (int)s_sum[co];
		const int64_t o = out + (int64_t)co * HW;
		if (OUT == Q_OUT_ACC) static_cast<int*>(y)[o] = v;
		else static_cast<uint8_t*>(y)[o] = (uint8_t)requant<OUT>(v, mult, zp_out);
	}
}

template <int OUT>
static bool launch_conv2dq_direct_rows(const ConvGeo& g, const uint8_t* x, const uint8_t* w, const int32_t* bias, int zp_in, int zp_w,
                                       float mult, float zp_out, void* y)
{
	const int dpr = g.kw <= 4 ? 1 : 2, rows = g.Cin * g.kh;
	const int64_t bytes = (int64_t)g.N * g.Cin * g.H * g.W;
	// (offsets of windows that start above or left of the image, or end below it, stay within 32 bits too)
	if (g.kw < 3 || g.kw > 8 || rows < 1 || bytes < 4 * dpr || bytes + ((int64_t)g.ph + g.kh + 1) * g.W + g.pw >= (1ll << 31)) return false;
	// Threads that share positions load the same windows again: only up to two wavefronts a SIMD of them.
	const uint64_t positions = (uint64_t)g.N * g.Ho * g.Wo;
	int groups = 1;
	while (groups < 4 && positions * groups <= 65536 && g.Cout >= 4 * groups) groups *= 2;
	const dim3 grid((unsigned)ceil_div(positions, (uint64_t)(256 / groups)), (unsigned)ceil_div((uint64_t)g.Cout, CQ_CO));
	auto launch = [&](auto dpr_c, auto nr_c) {
		conv2dq_direct_rows_kernel<OUT, decltype(dpr_c)::value, decltype(nr_c)::value><<<grid, dim3(256), 0, stream()>>>(g, x, w, bias, zp_in, zp_w, mult, zp_out, y, groups);
	};
	using One = std::integral_constant<int, 1>;
	using Two = std::integral_constant<int, 2>;
	if (dpr == 1) {
		if (rows <= 4) launch(One{}, std::integral_constant<int, 4>{});
		else if (rows <= 9) launch(One{}, std::integral_constant<int, 9>{});
		else if (rows <= 15) launch(One{}, std::integral_constant<int, 15>{});
		else launch(One{}, std::integral_constant<int, 21>{});  // (64 taps in rows of 3)
	} else {
		if (rows <= 5) launch(Two{}, std::integral_constant<int, 5>{});
		else if (rows <= 8) launch(Two{}, std::integral_constant<int, 8>{});
		else launch(Two{}, std::integral_constant<int, 12>{});  // (64 taps in rows of 5)
	}
	return true;
}

// ND = dwords of packed taps a thread holds (4 taps each): 4, 8, 12 or 16, the smallest that covers K.
template <int OUT, int ND>
__global__ __launch_bounds__(256) void conv2dq_direct_kernel(ConvGeo g, const uint8_t* __restrict__ x, const uint8_t* __restrict__ w,
                                                             const int32_t* __restrict__ bias, int zp_in, int zp_w, float mult, float zp_out,
                                                             void* __restrict__ y)
{
	__shared__ __attribute__((aligned(16))) uint32_t s_w[CQ_CO][ND];
	const int tid = threadIdx.x;
	const int K = g.Cin * g.kh * g.kw, HW = g.Ho * g.Wo;
	const int co0 = blockIdx.y * CQ_CO, nco = min(CQ_CO, g.Cout - co0);

	// N * HW < 2^31 (checked by the host): 32-bit divisions
	const uint32_t gid = blockIdx.x * 256u + tid;
	const bool live = gid < (uint32_t)g.N * (uint32_t)HW;
	const int n = live ? (int)(gid / (uint32_t)HW) : 0, pos = live ? (int)(gid - (uint32_t)n * (uint32_t)HW) : 0;
	const int ho = (int)((uint32_t)pos / (uint32_t)g.Wo), wo = pos - ho * g.Wo;
	const int y0 = ho * g.sh - g.ph, x0 = wo * g.sw - g.pw;
	const uint8_t* xn = x + (int64_t)n * g.Cin * g.H * g.W + (int64_t)y0 * g.W + x0;  // tap (0, 0, 0) of this position's window

	// The window, tap k in byte k % 4 of dword k / 4; (ci, i, j) of tap k is the same for every thread and is stepped,
	// not divided out.  The loads are issued before the weights are staged, so that the two latencies overlap.
	uint8_t tap[4 * ND];
	{
		int i = 0, j = 0, plane_row = 0;  // plane_row = ci * H + i
#pragma unroll
		for (int k = 0; k < 4 * ND; k++) {
			tap[k] = 0;
			if (k < K) {
				const int yy = y0 + i, xx = x0 + j;
				if (live && yy >= 0 && yy < g.H && xx >= 0 && xx < g.W) tap[k] = xn[(int64_t)plane_row * g.W + j];
				if (++j == g.kw) {
					j = 0;
					plane_row++;
					if (++i == g.kh) {
						i = 0;
						plane_row += g.H - g.kh;
					}
				}
			}
		}
	}

	// weights of this block's output channels, four taps per dword, taps past K as zero bytes (every load issued, the
	// byte of a tap past K discarded)
	for (int idx = tid; idx < CQ_CO * ND; idx += 256) {
		const int co = idx / ND, d = idx % ND;
		uint32_t v = 0;
		if (co < nco && K > 0) {
			const uint8_t* wr = w + (int64_t)(co0 + co) * K;
#pragma unroll
			for (int b = 0; b < 4; b++) {
				const int k = 4 * d + b;
				const uint32_t byte = wr[min(k, K - 1)];
				v |= (k < K ? byte : 0u) << (8 * b);
			}
		}
		s_w[co][d] = v;
	}
	__syncthreads();
	if (!live) return;

	uint32_t xk[ND];
#pragma unroll
	for (int d = 0; d < ND; d++)
		xk[d] = (uint32_t)tap[4 * d] | (uint32_t)tap[4 * d + 1] << 8 | (uint32_t)tap[4 * d + 2] << 16 | (uint32_t)tap[4 * d + 3] << 24;
	uint32_t xsum = 0;
#pragma unroll
	for (int d = 0; d < ND; d++) xsum = __builtin_amdgcn_udot4(xk[d], 0x01010101u, xsum, false);
	// l-ten/math_fns.cpp:1362-1380,1433: row_vector[p] = -zpA * sum_k B[k][p] with A = weights; broadcast = K zpA zpB
	const int base = -zp_w * (int)xsum + K * zp_w * zp_in + (bias ? bias[pos] : 0);

	for (int co = 0; co < nco; co++) {
		// the byte sum of the channel's weights rides along: the dwords are in registers anyway
		uint32_t dot = 0, wsum = 0;
#pragma unroll
		for (int d = 0; d < ND; d++) {
			const uint32_t wd = s_w[co][d];
			dot = __builtin_amdgcn_udot4(wd, xk[d], dot, false);
			wsum = __builtin_amdgcn_udot4(wd, 0x01010101u, wsum, false);
		}
		const int v = (int)dot + base - zp_in * (int)wsum;
		const int64_t o = ((int64_t)n * g.Cout + co0 + co) * HW + pos;
		if (OUT == Q_OUT_ACC) static_cast<int*>(y)[o] = v;
		else static_cast<uint8_t*>(y)[o] = (uint8_t)requant<OUT>(v, mult, zp_out);
	}
}

template <int OUT>
static void launch_conv2dq_direct(const dim3& grid, int K, const ConvGeo& g, const uint8_t* x, const uint8_t* w, const int32_t* bias, int zp_in,
                                  int zp_w, float mult, float zp_out, void* y)
{
	if (K <= 16) conv2dq_direct_kernel<OUT, 4><<<grid, dim3(256), 0, stream()>>>(g, x, w, bias, zp_in, zp_w, mult, zp_out, y);
	else if (K <= 32) conv2dq_direct_kernel<OUT, 8><<<grid, dim3(256), 0, stream()>>>(g, x, w, bias, zp_in, zp_w, mult, zp_out, y);
	else if (K <= 48) conv2dq_direct_kernel<OUT, 12><<<grid, dim3(256), 0, stream()>>>(g, x, w, bias, zp_in, zp_w, mult, zp_out, y);
	else conv2dq_direct_kernel<OUT, 16><<<grid, dim3(256), 0, stream()>>>(g, x, w, bias, zp_in, zp_w, mult, zp_out, y);
}

// Row r = n * Ho * Wo + p of the patch matrix: the window of output position p of image n in l-ten's column order
// (ci, i, j).  Bytes outside the image are 0, as in l-ten's im2col (not the zero point); bytes from K on hold the input
// zero point.  A thread builds sixteen consecutive bytes of a row; the tap table (offset of the tap inside an image and
// its (i, j)) of the workgroup's 64 bytes of a row is built once per workgroup in LDS.  (Sixteen bytes and one 16-byte
// store per thread.)
__global__ __launch_bounds__(256) void conv2dq_rows_kernel(ConvGeo g, const uint8_t* __restrict__ x, uint8_t* __restrict__ rows, int Kp, int zp_in,
                                                           unsigned row_blocks, const uint8_t* __restrict__ w, uint8_t* __restrict__ wp, int Cp, int zp_w)
{
	__shared__ int s_tap[128];  // [64] offsets, then [64] i | j << 16
	const int K = g.Cin * g.kh * g.kw, HW = g.Ho * g.Wo;
	if (blockIdx.x >= row_blocks) {
		// the workgroups behind the rows pad the weights: wp[co][k] for co < Cp, k < Kp, with the weight zero point past K
		// and in the rows past Cout
		const int idx = (int)(blockIdx.x - row_blocks) * 256 + (int)threadIdx.x;
		if (idx < Cp * Kp) {
			const int co = idx / Kp, k = idx - co * Kp;
			wp[idx] = (co < g.Cout && k < K) ? w[(int64_t)co * K + k] : (uint8_t)zp_w;
		}
		return;
	}
	// A workgroup builds 64 consecutive rows x 64 bytes: a wavefront's lanes are 64 consecutive positions at one chunk, so
	// that each of its loads reads neighbouring bytes of the image (consecutive chunks of one row would read 64 channel
	// planes at once); the four wavefronts write the four chunks of the same 64 bytes of every row.
	const uint32_t chunks_per_row = (uint32_t)Kp / 16, groups = (chunks_per_row + 3) / 4;
	const uint32_t tile = blockIdx.x / groups, grp = blockIdx.x - tile * groups;
	const uint32_t r = tile * 64 + (threadIdx.x & 63), kc = grp * 4 + (threadIdx.x >> 6);
	if (threadIdx.x < 64) {  // the taps of this workgroup's 64 bytes of a row
		const int kt = min((int)grp * 64 + (int)threadIdx.x, K - 1);
		const int j = kt % g.kw, i = (kt / g.kw) % g.kh, ci = kt / (g.kw * g.kh);
		s_tap[threadIdx.x] = (ci * g.H + i) * g.W + j;
		s_tap[64 + threadIdx.x] = i | (j << 16);
	}
	__syncthreads();
	if (r >= (uint32_t)g.N * (uint32_t)HW || kc >= chunks_per_row) return;
	const int n = (int)(r / (uint32_t)HW), pos = (int)(r - (uint32_t)n * (uint32_t)HW);
	const int ho = pos / g.Wo, wo = pos - ho * g.Wo;
	const int y0 = ho * g.sh - g.ph, x0 = wo * g.sw - g.pw;
	const uint8_t* xn = x + (int64_t)n * g.Cin * g.H * g.W;
	const int base = y0 * g.W + x0;
	uint32_t bytes[16];
#pragma unroll
	for (int b = 0; b < 16; b++) {  // all sixteen loads first
		const int k = 16 * (int)kc + b, kl = 16 * (int)(threadIdx.x >> 6) + b;
		const int ij = s_tap[64 + kl];
		const int yy = y0 + (ij & 0xFFFF), xx = x0 + (ij >> 16);
		const bool inside = ((unsigned)yy < (unsigned)g.H) & ((unsigned)xx < (unsigned)g.W);
		const uint32_t byte = xn[(s_tap[kl] + base) & -(int)inside];  // offset 0 for taps outside: always a valid address
		bytes[b] = k < K ? (inside ? byte : 0u) : (uint32_t)zp_in;
	}
	uint4 out;
	out.x = bytes[0] | bytes[1] << 8 | bytes[2] << 16 | bytes[3] << 24;
	out.y = bytes[4] | bytes[5] << 8 | bytes[6] << 16 | bytes[7] << 24;
	out.z = bytes[8] | bytes[9] << 8 | bytes[10] << 16 | bytes[11] << 24;
	out.w = bytes[12] | bytes[13] << 8 | bytes[14] << 16 | bytes[15] << 24;
	reinterpret_cast<uint4*>(rows)[(uint64_t)r * chunks_per_row + kc] = out;
}

// y[n][co][p] = requantize(acc[n * HW + p][co] + bias[p]) (or the int32 sum itself): a workgroup takes 64 positions x 64
// channels, reads the sums along the channels and stores along the positions, through LDS.
template <int OUT>
__global__ __launch_bounds__(256) void conv2dq_finish_kernel(const int32_t* __restrict__ acc, const int32_t* __restrict__ bias, void* __restrict__ y,
                                                             int rows, int HW, int Cout, int Cp, float mult, float zp_out)
{
	__shared__ int s[64][65];
	const int r0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
	const int ncp = min(64, Cp - c0), nco = min(64, Cout - c0);  // columns of the sums to read, channels to store
	for (int e = threadIdx.x; e < 64 * ncp; e += 256) {
		const int rr = e / ncp, cc = e - rr * ncp;
		s[rr][cc] = acc[(int64_t)min(r0 + rr, rows - 1) * Cp + c0 + cc];
	}
	__syncthreads();
	// a thread keeps its position and walks the channels: the position is decomposed once
	const int rr = threadIdx.x & 63, r = r0 + rr;
	if (r >= rows) return;
	const int n = r / HW, pos = r - n * HW;
	const int b = bias ? bias[pos] : 0;
	for (int cc = threadIdx.x >> 6; cc < nco; cc += 4) {
		const int v = s[rr][cc] + b;
		const int64_t o = ((int64_t)n * Cout + c0 + cc) * HW + pos;
		if (OUT == Q_OUT_ACC) static_cast<int*>(y)[o] = v;
		else static_cast<uint8_t*>(y)[o] = (uint8_t)requant<OUT>(v, mult, zp_out);
	}
}

static int make_geo_q(ConvGeo& g, uint64_t N, uint64_t Cin, uint64_t H, uint64_t W, uint64_t Cout, int kh, int kw, int ph, int pw, int sh, int sw)
{
	LTEN_HIP_REQUIRE(kh > 0 && kw > 0 && sh > 0 && sw > 0 && ph >= 0 && pw >= 0, "conv2dq: bad kernel geometry");
	LTEN_HIP_REQUIRE(N < 65536 && Cin < (1u << 20) && Cout < (1u << 20) && H < (1u << 15) && W < (1u << 15), "conv2dq: dimension too large");
	LTEN_HIP_REQUIRE(Cin * H * W < (1ull << 31) && Cout * H * W < (1ull << 31), "conv2dq: one image must stay below 2^31 elements");
	const int64_t eh = (int64_t)H + 2 * ph - kh, ew = (int64_t)W + 2 * pw - kw;
	LTEN_HIP_REQUIRE(eh >= 0 && ew >= 0, "conv2dq: kernel larger than the padded image");
	LTEN_HIP_REQUIRE(Cin * (uint64_t)kh * kw * 255 * 255 < (1ull << 31), "conv2dq: Cin*kh*kw too large for an int32 accumulator");
	g.N = (int)N; g.Cin = (int)Cin; g.H = (int)H; g.W = (int)W; g.Cout = (int)Cout;
	g.kh = kh; g.kw = kw; g.ph = ph; g.pw = pw; g.sh = sh; g.sw = sw; g.dh = 1; g.dw = 1;
	g.Ho = (int)(eh / sh + 1);  // l-ten/conv2d.cpp:322-323
	g.Wo = (int)(ew / sw + 1);
	return 0;
}

static uint64_t align16(uint64_t v) { return (v + 15) & ~15ull; }
static uint64_t align256(uint64_t v) { return (v + 255) & ~255ull; }

// Workspace of the whole-batch route: patch rows, padded weights, int32 sums, the GEMM's zero-point terms.
struct BatchedPlan {
	bool ok;
	uint64_t rows, Kp, Cp, off_wp, off_acc, off_terms, bytes;
};

static BatchedPlan batched_plan(const ConvGeo& g)
{
	BatchedPlan b;
	const uint64_t K = (uint64_t)g.Cin * g.kh * g.kw;
	b.rows = (uint64_t)g.N * g.Ho * g.Wo;
	b.Kp = (K + 15) & ~15ull;
	b.Cp = ((uint64_t)g.Cout + 3) & ~3ull;
	b.off_wp = align256(b.rows * b.Kp);
	b.off_acc = b.off_wp + align256(b.Cp * b.Kp);
	b.off_terms = b.off_acc + align256(b.rows * b.Cp * 4);
	b.bytes = b.off_terms + 4 * (b.rows + b.Cp) + 16;
	b.ok = b.bytes <= (2ull << 30) && b.rows < (1ull << 31) && b.rows * b.Kp < (1ull << 32) && b.Cp * b.Kp < (1ull << 31);
	return b;
}

constexpr uint64_t LIBRARY_LIMIT = 512ull << 20;  // library memory that a call fills, unless one image takes more

// Library memory for the pixels of a call.  Where they about fill the L2s (4 MB in each of the eight XCDs, which all read some of
// the same lines) writing what the call before has read is slow: three places take turns then (call after call, 3 x 3, 32 x 64 x 56 x
// 56 -> 64 channels, 6.9 MB: 16.0 us in one place, 15.4 in two, 14.5 in three or more; 32 x 64 x 80 x 80 -> 64, 13.8 MB: 26.8 and
// 23.2; 1 x 1, 64 x 64 x 64 x 64 -> 96, 16.8 MB: 26.4 and 23.0; of 3.8 MB and less and of 28 MB all the same).
static void* pixels_memory(uint64_t bytes)
{
	constexpr unsigned places = 3;
	static unsigned turn = 0;
	const uint64_t place = align256(bytes);
	if (bytes > (4ull << 20) && bytes <= (24ull << 20)) {
		uint8_t* const all = static_cast<uint8_t*>(library_scratch(places * place));
		if (all != nullptr) return all + turn++ % places * place;
	}
	return library_scratch(bytes);
}

static int conv2dq_run(uint64_t N, uint64_t Cin, uint64_t H, uint64_t W, uint64_t Cout, int kh, int kw, int ph, int pw, int sh, int sw,
                       const uint8_t* x, const uint8_t* w, const int32_t* bias, const lten_hip_qparams* qp, void* y, bool out_acc,
                       void* workspace)
{
	ConvGeo g;
	if (int rc = make_geo_q(g, N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw)) return rc;
	LTEN_HIP_REQUIRE(qp != nullptr, "conv2dq: qparams is null");
	const int64_t HW = (int64_t)g.Ho * g.Wo, K = (int64_t)Cin * kh * kw;
	if (N == 0 || Cout == 0 || HW == 0) return 0;
	LTEN_HIP_REQUIRE(x && w && y, "conv2dq: null pointer");
	const int zp_in = qp[0].zero_point, zp_w = qp[1].zero_point;
	// l-ten/math_fns.cpp:1436 with qparams[0] = weights, [1] = input (l-ten/conv2d.cpp:347-349), left to right in fp32
	volatile float ab = qp[1].scale * qp[0].scale;
	const float mult = ab / qp[2].scale, zp_out = (float)qp[2].zero_point;

	const int variant = get_option(OPT_CONV_VARIANT);
	const BatchedPlan bp = batched_plan(g);
	// whether the three launches below are ahead of the band kernel (see there)
	const bool rows_ahead = variant == 0 && bp.ok && conv2dq_band_estimate_us(g) > 30.0 + 1.3e-6 * (double)bp.rows * (double)bp.Kp;
	// Bytes out of a layer with some work: pixels of channels and an implicit GEMM (convq_pixels.hip; int32 sums, which only
	// checks ask for, keep the kernels below).  Ahead of the three launches and of the decomposition image by image wherever
	// those were taken (1.6 to 5 times over 60 layers); ahead of the band kernel by the two estimates, with a margin for
	// their errors (8 x 116 x 24 x 24 -> 25 channels 3 x 3: 12.9 -> 8.0 us, 12 x 18 x 56 x 56 -> 144: 27.3 -> 11.4; 18 x 4 x 12 x 12 -> 61
	// stays, 5.3 against 6.8).  Option "conv_variant" 11 to 16 forces a tile.
	// Layers that one of the kernels of one launch could take leave the caller's workspace as it is, whatever they run as: the
	// header says so.  What they fill is memory of the library's; the others fill the workspace.
	// Before that the kernel that has a band of the input and its weights in LDS (convq_region.hip), one launch without memory of
	// its own, where it is ahead of both by the estimates with such margins: 32 x 64 x 56 x 56 -> 64 channels 3 x 3 16.1 -> 12.0 us (two
	// launches), 4 x 8 x 52 x 52 -> 149 9.8 -> 6.4 (bands) or 7.0; 59 x 37 x 16 x 16 -> 39 5 x 5 stays, 9.5 against 14.5, 8 x 138 x 27 x 27 ->
	// 117 1 x 1, 7.2 against 7.3, and 18 x 4 x 12 x 12 -> 61, 5.3 against 5.9.  Option "conv_variant" 20 forces it.
	if (!out_acc && (variant == 0 || variant > 10) && (variant > 10 || (K <= CQ_MAXK ? Cout >= 48 : !conv2dq_image_takes(g, w)))) {
		uint64_t bytes = 0;
		double here = conv2dq_pixels_us(g, bytes);
		if (bytes > lten_hip_conv2dq_workspace_bytes(N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw)) here = -1.0;  // (no more than the workspace would hold in any case)
		const double band_us = conv2dq_band_us(g), band = rows_ahead && K > CQ_MAXK ? -1.0 : band_us;
		const bool one_launch = K <= CQ_MAXK || band_us >= 0.0 || conv2dq_image_takes(g, w);
		if ((variant == 0 || variant == 20) && (one_launch || workspace != nullptr)) {  // (the other layers' contract wants a workspace, whatever they run as)
			const double limit_us = std::min(here < 0.0 ? 1e30 : 0.95 * here, band_us < 0.0 ? 1e30 : 0.95 * band_us);
			const int rc = conv2dq_region_dispatch(g, x, w, bias, zp_in, zp_w, mult, zp_out, static_cast<uint8_t*>(y), variant == 20 ? 1e30 : limit_us);
			if (rc >= 0) return rc;
		}
		if (variant != 20 && here >= 0.0 && (variant > 10 || (band < 0.0 ? K > CQ_MAXK : here < 0.93 * band))) {
			// images in groups whose pixels the library's memory holds, one at least
			ConvGeo part = g;
			if (one_launch && bytes > LIBRARY_LIMIT) {
				part.N = (int)std::max<uint64_t>(1, LIBRARY_LIMIT / ceil_div(bytes, N));
				conv2dq_pixels_us(part, bytes);
			}
			void* const memory = one_launch ? pixels_memory(bytes) : (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 ? workspace : nullptr;
			int rc = memory != nullptr ? 0 : -1;
			for (int n = 0; n < g.N && rc == 0; n += part.N) {
				ConvGeo now = g;
				now.N = std::min(part.N, g.N - n);
				rc = conv2dq_pixels_dispatch(now, x + (int64_t)n * g.Cin * g.H * g.W, w, bias, zp_in, zp_w, mult, zp_out, static_cast<uint8_t*>(y) + (int64_t)n * g.Cout * HW, memory,
				                             variant > 10 ? variant - 10 : 0);
			}
			if (rc >= 0) return rc;
		}
	}
	// Windows of at most 64 taps for 48 output channels and more: the band kernel's matrix cores are ahead of the dot
	// products below, which issue at a quarter of the vector rate (8 x 16 x 56 x 56 -> 64 channels 2 x 2, stride 2: 26.5
	// -> 6.9 us; 8 x 64 x 56 x 56 -> 256 channels 1 x 1: 30.0 -> 16.6 us; 64 x 3 x 224 x 224 -> 64 channels 3 x 3: 181 ->
	// 130 us), not for fewer (256 x 3 x 32 x 32 -> 32: 10.4 us below, 19.0 there; l-ten's MNIST conv1, 10 channels: 4.6
	// and 7.3).  Option "conv_variant" 2 keeps the kernel below.
	if (K <= CQ_MAXK && Cout >= 48 && (get_option(OPT_CONV_VARIANT) == 0 || get_option(OPT_CONV_VARIANT) == 3)) {
		const int rc = conv2dq_band_dispatch(g, x, w, bias, zp_in, zp_w, mult, zp_out, y, out_acc);
		if (rc >= 0) return rc;
	}
	if (K <= CQ_MAXK && (uint64_t)N * HW < (1ull << 31) && get_option(OPT_CONV_VARIANT) != 1) {
		const dim3 grid((unsigned)ceil_div((uint64_t)N * HW, 256), (unsigned)ceil_div(Cout, CQ_CO));
		set_kernel_name("conv2dq_direct");
		const bool fast = mult == mult && (mult < 0 ? -mult : mult) <= 0.99f;
		if (out_acc ? launch_conv2dq_direct_rows<Q_OUT_ACC>(g, x, w, bias, zp_in, zp_w, mult, zp_out, y)
		    : fast  ? launch_conv2dq_direct_rows<Q_OUT_U8_FAST>(g, x, w, bias, zp_in, zp_w, mult, zp_out, y)
		            : launch_conv2dq_direct_rows<Q_OUT_U8_EXACT>(g, x, w, bias, zp_in, zp_w, mult, zp_out, y)) {
			LTEN_HIP_LAUNCH_CHECK();
			return 0;
		}
		if (out_acc) launch_conv2dq_direct<Q_OUT_ACC>(grid, (int)K, g, x, w, bias, zp_in, zp_w, mult, zp_out, y);
		else if (fast)
			launch_conv2dq_direct<Q_OUT_U8_FAST>(grid, (int)K, g, x, w, bias, zp_in, zp_w, mult, zp_out, y);
		else launch_conv2dq_direct<Q_OUT_U8_EXACT>(grid, (int)K, g, x, w, bias, zp_in, zp_w, mult, zp_out, y);
		LTEN_HIP_LAUNCH_CHECK();
		return 0;
	}

	void* rows_memory = nullptr;
	// small images with a longer window (l-ten's quantized MNIST conv2): still one launch, no workspace (convq_image.hip;
	// option "conv_variant" 2 keeps such shapes on the three launches below, 3 skips the small-image kernel)
	if (get_option(OPT_CONV_VARIANT) == 0 || get_option(OPT_CONV_VARIANT) == 3) {
		int rc = get_option(OPT_CONV_VARIANT) == 3 ? -1 : conv2dq_image_dispatch(g, x, w, bias, zp_in, zp_w, mult, zp_out, y, out_acc);
		if (rc >= 0) return rc;
		// larger images or more channels: a band of output rows and a block of output channels per workgroup, the input rows
		// it needs in LDS -- unless long windows leave a workgroup so few pixels and channels that it stages more than it
		// computes and the three launches below are ahead, which take 30 us + 1.3 us per MB of patch rows (32 x 1024 x 14
		// x 14 -> 256 channels 1 x 1: 132 us on bands, 43 below; 32 x 128 x 28 x 28 -> 256 channels 3 x 3 stride 2: 55 and 44)
		if (rows_ahead && bp.bytes <= LIBRARY_LIMIT) rows_memory = library_scratch(bp.bytes);
		if (rows_memory == nullptr) rc = conv2dq_band_dispatch(g, x, w, bias, zp_in, zp_w, mult, zp_out, y, out_acc);
		if (rc >= 0) return rc;
	}

	LTEN_HIP_REQUIRE(workspace != nullptr || rows_memory != nullptr, "conv2dq: workspace is null");
	if (bp.ok && get_option(OPT_CONV_VARIANT) != 1) {
		std::optional<LibraryScratchHold> hold;  // (the GEMM may ask for memory of its own)
		if (rows_memory != nullptr) hold.emplace(bp.bytes);
		uint8_t* base = static_cast<uint8_t*>(rows_memory != nullptr ? rows_memory : workspace);
		uint8_t* rows = base;
		uint8_t* wp = base + bp.off_wp;
		int32_t* sums = reinterpret_cast<int32_t*>(base + bp.off_acc);
		int32_t* terms = reinterpret_cast<int32_t*>(base + bp.off_terms);
		const unsigned row_blocks = (unsigned)(ceil_div(bp.rows, 64) * ceil_div(bp.Kp / 16, 4)), weight_blocks = (unsigned)ceil_div(bp.Cp * bp.Kp, 256);
		conv2dq_rows_kernel<<<dim3(row_blocks + weight_blocks), dim3(256), 0, stream()>>>(g, x, rows, (int)bp.Kp, zp_in, row_blocks, w, wp,
		                                                                                                (int)bp.Cp, zp_w);
		LTEN_HIP_LAUNCH_CHECK();
		if (int rc = lten_hip_quantized_matmul_acc(0, 1, bp.rows, bp.Cp, bp.Kp, rows, wp, sums, qp, nullptr, terms)) return rc;
		const dim3 grid((unsigned)ceil_div(bp.rows, 64), (unsigned)ceil_div(Cout, 64));
		set_kernel_name("conv2dq_rows_gemm_finish");
		if (out_acc) conv2dq_finish_kernel<Q_OUT_ACC><<<grid, dim3(256), 0, stream()>>>(sums, bias, y, (int)bp.rows, (int)HW, (int)Cout, (int)bp.Cp, mult, zp_out);
		else if (mult == mult && (mult < 0 ? -mult : mult) <= 0.99f)
			conv2dq_finish_kernel<Q_OUT_U8_FAST><<<grid, dim3(256), 0, stream()>>>(sums, bias, y, (int)bp.rows, (int)HW, (int)Cout, (int)bp.Cp, mult, zp_out);
		else conv2dq_finish_kernel<Q_OUT_U8_EXACT><<<grid, dim3(256), 0, stream()>>>(sums, bias, y, (int)bp.rows, (int)HW, (int)Cout, (int)bp.Cp, mult, zp_out);
		LTEN_HIP_LAUNCH_CHECK();
		return 0;
	}

	// l-ten's own decomposition, image by image: column buffer, then C[Cout x HW] = W[Cout x K] * col[K x HW]
	uint8_t* col = static_cast<uint8_t*>(workspace);
	int32_t* terms = reinterpret_cast<int32_t*>(col + align16((uint64_t)K * HW));
	const lten_hip_qparams q3[3] = { qp[1], qp[0], qp[2] };
	for (uint64_t n = 0; n < N; n++) {
		if (int rc = lten_hip_im2col_u8(x + n * Cin * H * W, (int)Cin, (int)H, (int)W, kh, kw, ph, pw, sh, sw, 1, 1, col)) return rc;
		int rc;
		if (out_acc) rc = lten_hip_quantized_matmul_acc(0, 0, Cout, (uint64_t)HW, (uint64_t)K, w, col, static_cast<int32_t*>(y) + n * Cout * HW, q3, bias, terms);
		else rc = lten_hip_quantized_matmul(0, 0, Cout, (uint64_t)HW, (uint64_t)K, 1, w, col, 0, static_cast<uint8_t*>(y) + n * Cout * HW, q3, bias, terms);
		if (rc) return rc;
	}
	return 0;
}

}  // namespace lten_hip

using namespace lten_hip;

extern "C" {

uint64_t lten_hip_conv2dq_workspace_bytes(uint64_t N, uint64_t Cin, uint64_t H, uint64_t W, uint64_t Cout, int kh, int kw, int ph,
                                          int pw, int sh, int sw)
{
	ConvGeo g;
	if (make_geo_q(g, N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw)) return 0;
	const uint64_t HW = (uint64_t)g.Ho * g.Wo, K = Cin * kh * kw;
	const uint64_t per_image = align16(K * HW) + 4 * (Cout + HW) + 16;
	const BatchedPlan bp = batched_plan(g);
	return bp.ok ? std::max(per_image, bp.bytes) : per_image;
}

int lten_hip_conv2dq_forward(uint64_t N, uint64_t Cin, uint64_t H, uint64_t W, uint64_t Cout, int kh, int kw, int ph, int pw, int sh,
                             int sw, const uint8_t* x, const uint8_t* w, const int32_t* bias, const lten_hip_qparams* qparams_in_wt_out,
                             uint8_t* y, void* workspace)
{
	return conv2dq_run(N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw, x, w, bias, qparams_in_wt_out, y, false, workspace);
}

int lten_hip_conv2dq_forward_acc(uint64_t N, uint64_t Cin, uint64_t H, uint64_t W, uint64_t Cout, int kh, int kw, int ph, int pw,
                                 int sh, int sw, const uint8_t* x, const uint8_t* w, const int32_t* bias,
                                 const lten_hip_qparams* qparams_in_wt_out, int32_t* acc, void* workspace)
{
	return conv2dq_run(N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw, x, w, bias, qparams_in_wt_out, acc, true, workspace);
}

}  // extern "C"
