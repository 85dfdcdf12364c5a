// Conv2d_q forward of layers whose weights fit LDS beside a band of the input, in one launch (l-ten/conv2d.cpp:265-387;
// arithmetic as in convq_pixels.hip).
//
// A workgroup of eight wavefronts takes a band of output rows of one image and up to 64 output channels.  It stages the input
// rows under the band as pixels of channels ([row][column][16-byte chunks of channels], the padding written out) and the
// weights as rows of (tap, channel), both once, and walks the k-steps of (tap, 32 channels) on LDS alone: no barrier and no
// load from memory in the loop.  A wavefront owns blocks of 64 positions x 64 (or 32) channels.
// A channel's rows under the band are one run of bytes: a thread fetches 16 pixels of four channels in four loads, all under
// way before anything else is done, and turns them into 16 dwords of four channels.  The weights come in as they lie, 16 bytes
// a thread, and are put in order out of LDS (fetched in order, a load touched 64 cache lines).
//
// 32 x 64 x 56 x 56 -> 64 channels 3 x 3: 15.2 -> 11.4 us (two launches of 5.6 and 10.9 us on cold clocks, the pixels written and
// read again between them, against one of 13.5), in 44 thousand clocks of which 4 are matrix instructions'.  Bound by its parts one
// after the other: by the terms of the estimate below a launch 4.0, the stores 1.5, loads and LDS writes 2.0, the weights' order 0.6,
// the 18 k-steps of two wavefronts a SIMD 3.8.  16 x 32 x 28 x 28 -> 64 8.3 -> 6.2, 44 x 15 x 80 x 80 -> 29 16.1 -> 12.0, 24 x 24 x
// 48 x 48 -> 16 stride 2 11.4 -> 6.1, 1 x 249 x 28 x 28 -> 128 1 x 1 stride 2 11.8 -> 7.1.  With copies between the operand sets and
// the weights' sums in the loop the first took 11.7 us.
#include "conv_common.h"
#include "qgemm_common.h"

#include <algorithm>
#include <type_traits>

namespace lten_hip {

struct RegionPlan {
	int UC, PP, chunks, steps, wpitch;  // chunks of 16 channels in a pixel; bytes of a pixel; chunks of a window; k-steps; bytes of a weight row
	int TB, RH, RW, bands;              // output rows of a band; rows and columns of its region; bands of an image
	int pairs, rows;                    // blocks of 64 positions in a band; weight rows of a workgroup (32 or 64)
	int groups;                         // of output channels
	unsigned off_w, off_raw, off_tab, off_pos, off_row, off_sum, bytes;
};

struct RegionConv {
	int32_t konst, coef_a, coef_b;
	float mult, zp_c;
};

typedef v4i region_bytes16 __attribute__((aligned(1)));
typedef uint32_t region_bytes4 __attribute__((aligned(1)));

// The weights of a window of T taps out of LDS into (tap, channel) order, as int8, where the channels come in fours: four of
// them are T dwords of a row, and become T dwords of the new order, one per tap, in registers (byte by byte, as any other
// count takes it, the same took 2.2 times as long).
template <int T>
__device__ __forceinline__ void order_weights(const uint8_t* s_raw, uint8_t* s_w, int* s_sum, int cout_here, int quads_real, int Cp, int wpitch, int tid)
{
	for (int u = tid; u < cout_here * quads_real; u += 512) {
		const int co = u / quads_real, q = u - co * quads_real;
		const uint32_t* const src = reinterpret_cast<const uint32_t*>(s_raw) + u * T;
		uint32_t in[T];
#pragma unroll
		for (int i = 0; i < T; i++) in[i] = src[i];
		if (T > 1) {  // (the row's byte sum: where a thread has several dwords, an atomic of each is cheaper than a pass of its own, 11.2 against 12.2 us)
			uint32_t sum = 0;
#pragma unroll
			for (int i = 0; i < T; i++) sum = __builtin_amdgcn_sad_u8(in[i], 0u, sum);
			atomicAdd(s_sum + co, (int)sum);
		}
		uint8_t* const dst = s_w + co * wpitch + 4 * q;
#pragma unroll
		for (int t = 0; t < T; t++) {
			uint32_t v = 0;
#pragma unroll
			for (int b = 0; b < 4; b++) {
				const int pos = b * T + t;  // byte of the 4 T that holds (channel b, tap t)
				v |= ((in[pos >> 2] >> (8 * (pos & 3))) & 0xFFu) << (8 * b);
			}
			*reinterpret_cast<uint32_t*>(dst + t * Cp) = v ^ 0x80808080u;
		}
	}
}

// FN: blocks of 32 channels of a wavefront.  ROWSUM: the positions' byte sums are wanted (the region then holds l-ten's bytes).
template <int OUT, bool ROWSUM, int FN>
__global__ __launch_bounds__(512, 4) void conv2dq_region_kernel(ConvGeo g, RegionPlan pl, RegionConv c, const uint8_t* __restrict__ x,
                                                                const uint8_t* __restrict__ w, const int32_t* __restrict__ bias, uint8_t* __restrict__ y)
{
	extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
	constexpr uint32_t flip = ROWSUM ? 0u : 0x80808080u;
	constexpr int NW = 5;  // 16-byte pieces of the weights a thread has under way
	uint8_t* const s_rgn = smem;
	uint8_t* const s_w = smem + pl.off_w;
	uint8_t* const s_raw = smem + pl.off_raw;
	int* const s_tab = reinterpret_cast<int*>(smem + pl.off_tab);
	int* const s_pos = reinterpret_cast<int*>(smem + pl.off_pos);
	int* const s_sum = reinterpret_cast<int*>(smem + pl.off_sum);  // byte sums of the weight rows

	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int T = g.kh * g.kw, K = g.Cin * T, HWo = g.Ho * g.Wo, plane = g.H * g.W;
	// neighbouring bands, which share input rows, on one XCD
	const int nb = (int)gridDim.x, xcd = (int)blockIdx.x & 7;
	const int bid = xcd * (nb >> 3) + min(xcd, nb & 7) + ((int)blockIdx.x >> 3);
	const int n = bid / pl.bands, hb = (bid - n * pl.bands) * pl.TB;
	const int rows_here = min(pl.TB, g.Ho - hb), P = rows_here * g.Wo;
	const int co0 = (int)blockIdx.y * 64, cout_here = min(g.Cout - co0, 64);
	const int y_top = hb * g.sh - g.ph;                                                          // image row of the region's first
	const int ra = max(y_top, 0), rb = min(y_top + (rows_here - 1) * g.sh + g.kh, g.H);          // its rows inside the image
	const int run = (rb - ra) * g.W;                                                             // bytes of a channel, 16 at least
	const uint8_t* const xn = x + (int64_t)n * g.Cin * plane + (int64_t)ra * g.W;
	const uint8_t* const wn = w + (int64_t)co0 * K;
	const int w_total = cout_here * K;

	// ---- everything that comes from memory is asked for first
	const int runs16 = (run + 15) >> 4, quads = pl.UC * 4, tiles_c = (runs16 + 7) >> 3, tiles = tiles_c * ((quads + 7) >> 3);
	v4i d[4];
	int start = 0, quad = 0;
	bool live = false;
	auto fetch = [&](int tile) {  // 8 x 16 pixels of 8 x 4 channels
		const int tq = tile / tiles_c, piece = (tile - tq * tiles_c) * 8 + (lane & 7);
		quad = tq * 8 + (lane >> 3);
		live = piece < runs16 && quad < quads;
		start = min(piece * 16, run - 16);  // (the last piece repeats some pixels of the one before)
#pragma unroll
		for (int i = 0; i < 4; i++) d[i] = *reinterpret_cast<const region_bytes16*>(xn + (int64_t)min(quad * 4 + i, g.Cin - 1) * plane + start);
	};
	if (wave < tiles) fetch(wave);
	v4i wv[NW];
#pragma unroll
	for (int i = 0; i < NW; i++) {
		const int b = (i * 512 + tid) * 16;
		if (b + 16 <= w_total) wv[i] = *reinterpret_cast<const region_bytes16*>(wn + b);
	}

	// ---- meanwhile: where the chunks of a window lie, the positions' constants, the padding
	for (int k = tid; k < 2 * pl.steps; k += 512) {
		const int kc = min(k, pl.chunks - 1), t = kc / pl.UC, i = t / g.kw;
		s_tab[k] = (i * pl.RW + t - i * g.kw) * pl.PP + (kc - t * pl.UC) * 16;
	}
	if (tid < 64) s_sum[tid] = 0;
	for (int r = tid; r < pl.pairs * 64; r += 512) s_pos[r] = c.konst + (bias != nullptr ? bias[min(hb * g.Wo + r, HWo - 1)] : 0);
	{
		const int left = min(g.pw, pl.RW), right = max(0, pl.RW - g.pw - g.W);
		for (int r = wave; r < pl.RH; r += 8) {
			const bool outside = y_top + r < 0 || y_top + r >= g.H;
			const int count = (outside ? pl.RW : left + right) * pl.UC;
			for (int k = lane; k < count; k += 64) {
				const int q = k / pl.UC, cc = k - q * pl.UC, col = outside || q < left ? q : q - left + g.pw + g.W;
				v4i v;
#pragma unroll
				for (int e = 0; e < 4; e++) {
					const int real = min(max(g.Cin - cc * 16 - e * 4, 0), 4);  // real channels of the dword hold l-ten's byte 0, the others what counts as nothing
					v[e] = (int)((real == 4 ? 0u : 0x80808080u << (8 * real)) ^ flip);
				}
				*reinterpret_cast<v4i*>(s_rgn + (r * pl.RW + col) * pl.PP + cc * 16) = v;
			}
		}
	}

	const bool in_fours = (g.Cin & 3) == 0 && (T == 9 || T == 25 || T == 1);
	if (in_fours && ((g.Cin & 15) != 0 || (pl.chunks & 1) != 0 || cout_here < pl.rows))  // what no weight goes to
		for (int b = tid * 16; b < pl.rows * pl.wpitch; b += 512 * 16) *reinterpret_cast<v4i*>(s_w + b) = v4i{ 0, 0, 0, 0 };

	// ---- the weights as they lie
#pragma unroll
	for (int i = 0; i < NW; i++) {
		const int b = (i * 512 + tid) * 16;
		if (b + 16 <= w_total) *reinterpret_cast<v4i*>(s_raw + b) = wv[i];
	}
	for (int b = (NW * 512 + tid) * 16; b + 16 <= w_total; b += 512 * 16) *reinterpret_cast<v4i*>(s_raw + b) = *reinterpret_cast<const region_bytes16*>(wn + b);
	if (tid < (w_total & 15)) s_raw[(w_total & ~15) + tid] = wn[(w_total & ~15) + tid];

	// ---- the region
	for (int tile = wave; tile < tiles; tile += 8) {
		if (tile != wave) fetch(tile);
		uint32_t out[16];
#pragma unroll
		for (int q = 0; q < 4; q++) {
			uint32_t v[4];
#pragma unroll
			for (int i = 0; i < 4; i++) v[i] = quad * 4 + i < g.Cin ? (uint32_t)d[i][q] : 0x80808080u;
			const uint32_t lo01 = __builtin_amdgcn_perm(v[1], v[0], 0x05010400u), hi01 = __builtin_amdgcn_perm(v[1], v[0], 0x07030602u);
			const uint32_t lo23 = __builtin_amdgcn_perm(v[3], v[2], 0x05010400u), hi23 = __builtin_amdgcn_perm(v[3], v[2], 0x07030602u);
			out[4 * q] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u) ^ flip;
			out[4 * q + 1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u) ^ flip;
			out[4 * q + 2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u) ^ flip;
			out[4 * q + 3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u) ^ flip;
		}
		if (live) {
			int row = start / g.W, col = start - row * g.W;
			uint8_t* dst = s_rgn + ((ra - y_top + row) * pl.RW + g.pw + col) * pl.PP + quad * 4;
#pragma unroll
			for (int e = 0; e < 16; e++) {
				if (col + g.pw < pl.RW) *reinterpret_cast<uint32_t*>(dst) = out[e];
				dst += pl.PP;
				if (++col == g.W) {
					col = 0;
					dst += (pl.RW - g.W) * pl.PP;
				}
			}
		}
	}
	__syncthreads();

	// ---- the weight rows' byte sums, eight threads a row (rows start on any byte), where the next step does not add them up
	if (!in_fours || T == 1) {
		const int co = min(tid >> 3, cout_here - 1), begin = co * K, end = begin + K;
		uint32_t sum = 0;
#pragma unroll 4
		for (int b = (begin & ~3) + 4 * (tid & 7); b < end; b += 32) {
			uint32_t v = *reinterpret_cast<const uint32_t*>(s_raw + b);
			if (b < begin) v &= ~0u << (8 * (begin - b));
			if (b + 4 > end) v &= ~0u >> (8 * (b + 4 - end));
			sum = __builtin_amdgcn_sad_u8(v, 0u, sum);
		}
#pragma unroll
		for (int o = 1; o < 8; o <<= 1) sum += __shfl_xor(sum, o, 64);
		if ((tid & 7) == 0) s_sum[tid >> 3] = (int)sum;
	}
	// ---- the weights in (tap, channel) order
	if (in_fours && T == 9) order_weights<9>(s_raw, s_w, s_sum, cout_here, g.Cin / 4, pl.UC * 16, pl.wpitch, tid);
	else if (in_fours && T == 25) order_weights<25>(s_raw, s_w, s_sum, cout_here, g.Cin / 4, pl.UC * 16, pl.wpitch, tid);
	else if (in_fours) order_weights<1>(s_raw, s_w, s_sum, cout_here, g.Cin / 4, pl.UC * 16, pl.wpitch, tid);
	else {
		// a lane keeps its place in the row and goes down the channels
		for (int k = lane; k < pl.steps * 8; k += 64) {
			const int t = k / quads, q = k - t * quads;
			const bool real = t < T;
			const uint8_t* const src = s_raw + (real ? q * 4 * T + t : 0);
			uint8_t* const dst = s_w + k * 4;
			const int have = min(max(g.Cin - q * 4, 0), 4);
			const uint32_t keep = !real || have == 0 ? 0u : have == 4 ? ~0u : (1u << (8 * have)) - 1;
			const int t1 = have > 1 ? T : 0, t2 = have > 2 ? 2 * T : 0, t3 = have > 3 ? 3 * T : 0;
			const int safe = have > 0 ? 0 : -1;
#pragma unroll 4
			for (int co = wave; co < pl.rows; co += 8) {
				const uint8_t* const p = safe == 0 ? src + min(co, cout_here - 1) * K : s_raw;
				const uint32_t v = (uint32_t)p[0] | (uint32_t)p[t1] << 8 | (uint32_t)p[t2] << 16 | (uint32_t)p[t3] << 24;
				*reinterpret_cast<uint32_t*>(dst + co * pl.wpitch) = co < cout_here ? (v ^ 0x80808080u) & keep : 0u;
			}
		}
	}
	__syncthreads();

	// ---- the products: 64 positions x 32 FN channels at a time
	const int lrow = lane & 31, lgrp = lane >> 5;
	const int units = pl.pairs * (pl.rows / (32 * FN));
	for (int unit = wave; unit < units; unit += 8) {
		const int pair = unit % pl.pairs, cb = unit / pl.pairs * FN;
		if (pair * 64 >= P) continue;
		const uint8_t* a_at[2];
#pragma unroll
		for (int j = 0; j < 2; j++) {
			const int p = min(pair * 64 + j * 32 + lrow, P - 1), ho = p / g.Wo, wo = p - ho * g.Wo;
			a_at[j] = s_rgn + (ho * g.sh * pl.RW + wo * g.sw) * pl.PP;
		}
		const uint8_t* const b_at = s_w + (cb * 32 + lrow) * pl.wpitch + lgrp * 16;
		v16i acc[2][FN];
		unsigned rsum[2] = { 0, 0 };
#pragma unroll
		for (int i = 0; i < FN; i++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc[0][i][r] = acc[1][i][r] = 0;
		// a k-step's operands are read while the one before is multiplied, into the other of two sets
		const int last = pl.steps - 1;
		v4i fa[2][2], fb[2][FN];
		int off = s_tab[lgrp];
		auto operands = [&](auto set_c, int s) {
			constexpr int SET = decltype(set_c)::value;
#pragma unroll
			for (int j = 0; j < 2; j++) fa[SET][j] = *reinterpret_cast<const v4i*>(a_at[j] + off);
#pragma unroll
			for (int i = 0; i < FN; i++) fb[SET][i] = *reinterpret_cast<const v4i*>(b_at + i * 32 * pl.wpitch + s * 32);
			off = s_tab[2 * min(s + 1, last) + lgrp];
		};
		auto multiply = [&](auto set_c, int s) {
			constexpr int SET = decltype(set_c)::value;
			if (ROWSUM) {
				const bool real = 2 * s + lgrp < pl.chunks;
#pragma unroll
				for (int j = 0; j < 2; j++) {
					unsigned add = 0;
#pragma unroll
					for (int e = 0; e < 4; e++) add = __builtin_amdgcn_sad_u8((unsigned)fa[SET][j][e], 0u, add);
					rsum[j] += real ? add : 0u;
					fa[SET][j] = flip_sign_bits(fa[SET][j]);
				}
			}
#pragma unroll
			for (int i = 0; i < FN; i++)
#pragma unroll
				for (int j = 0; j < 2; j++) acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[SET][j], fb[SET][i], acc[j][i], 0, 0, 0);
		};
		using S0 = std::integral_constant<int, 0>;
		using S1 = std::integral_constant<int, 1>;
		operands(S0{}, 0);
		for (int s = 0; s < last; s += 2) {
			operands(S1{}, s + 1);
			multiply(S0{}, s);
			operands(S0{}, min(s + 2, last));  // (past the last step once more its own)
			multiply(S1{}, s + 1);
		}
		if ((pl.steps & 1) != 0) multiply(S0{}, last);
		int* const s_row = reinterpret_cast<int*>(smem + pl.off_row) + wave * 64;
		if (ROWSUM) {
#pragma unroll
			for (int j = 0; j < 2; j++) {
				const int both = (int)rsum[j] + __shfl_xor((int)rsum[j], 32, 64);
				if (lgrp == 0) s_row[j * 32 + lrow] = c.coef_a * both;
			}
			__builtin_amdgcn_wave_barrier();
		}
		// lane (lrow, lgrp), register 4q + e of block (j, i): position 64 pair + 32 j + 8 q + 4 lgrp + e of channel 32 (cb + i) + lrow
#pragma unroll
		for (int i = 0; i < FN; i++) {
			const int co = (cb + i) * 32 + lrow;
			const int ct = c.coef_b * s_sum[co];
#pragma unroll
			for (int j = 0; j < 2; j++) {
				const int p32 = pair * 64 + j * 32;
				unsigned word[4];
#pragma unroll
				for (int q = 0; q < 4; q++) {
					v4i v = *reinterpret_cast<const v4i*>(s_pos + p32 + 8 * q + 4 * lgrp);
					if (ROWSUM) v += *reinterpret_cast<const v4i*>(s_row + j * 32 + 8 * q + 4 * lgrp);
#pragma unroll
					for (int e = 0; e < 4; e++) v[e] += acc[j][i][q * 4 + e] + ct;
					word[q] = 0;
					if (OUT == Q_OUT_U8_FAST) {
						requant_into<0>(word[q], v.x, c.mult, c.zp_c);
						requant_into<1>(word[q], v.y, c.mult, c.zp_c);
						requant_into<2>(word[q], v.z, c.mult, c.zp_c);
						requant_into<3>(word[q], v.w, c.mult, c.zp_c);
					} else {
						word[q] = requant<OUT>(v.x, c.mult, c.zp_c) | requant<OUT>(v.y, c.mult, c.zp_c) << 8 | requant<OUT>(v.z, c.mult, c.zp_c) << 16 |
						          requant<OUT>(v.w, c.mult, c.zp_c) << 24;
					}
				}
				// the lane halves trade so that each holds 16 neighbouring positions
				const unsigned give0 = lgrp ? word[0] : word[2], give1 = lgrp ? word[1] : word[3];
				const unsigned got0 = (unsigned)__shfl_xor((int)give0, 32, 64), got1 = (unsigned)__shfl_xor((int)give1, 32, 64);
				const v4i out = lgrp ? v4i{ (int)got0, (int)word[2], (int)got1, (int)word[3] } : v4i{ (int)word[0], (int)got0, (int)word[1], (int)got1 };
				const int p = p32 + lgrp * 16;
				if (p >= P || co >= cout_here) continue;
				uint8_t* const dst = y + ((int64_t)n * g.Cout + co0 + co) * HWo + (int64_t)hb * g.Wo + p;
				if (p + 16 <= P) *reinterpret_cast<region_bytes16*>(dst) = out;
				else {
#pragma unroll
					for (int q = 0; q < 4; q++) {
						if (p + 4 * q + 4 <= P) *reinterpret_cast<region_bytes4*>(dst + 4 * q) = (uint32_t)out[q];
						else {
#pragma unroll
							for (int e = 0; e < 4; e++)
								if (p + 4 * q + e < P) dst[4 * q + e] = (uint8_t)((unsigned)out[q] >> (8 * e));
						}
					}
				}
			}
		}
	}
}

static int64_t align16(int64_t v) { return (v + 15) & ~15ll; }

// The band's height: the one whose launch is expected to be over first, if that is within limit_us; what is expected: a launch and
// the output; per round of 256 workgroups the region's bytes and the passes over it, the weights (as their channels come in fours or
// are gathered byte by byte) and the k-steps of a SIMD's wavefronts.  Fitted to 4700 layers of 1 to 256 images, 1 to 512 channels, 1 x
// 1 to 7 x 7 windows, strides 1 to 3 (9 % rms, 7 % in one round; a fit to 44 layers had sent 209 of 3485 here, or to a band of
// another height, that took up to 1.5 times as long as elsewhere).
static bool region_plan(const ConvGeo& g, RegionPlan& pl, double limit_us)
{
	const int64_t T = (int64_t)g.kh * g.kw, K = (int64_t)g.Cin * T;
	const double least = 4.0 + 0.23e-6 * (double)g.N * g.Ho * g.Wo * g.Cout;
	if (least >= limit_us) return false;
	if (g.dh != 1 || g.dw != 1 || g.ph >= g.kh || g.pw >= g.kw || T > 256 || g.Cin > 1024 || (int64_t)g.H * g.W >= (1 << 24) || (int64_t)g.Ho * g.Wo >= (1 << 24)) return false;
	pl.UC = (g.Cin + 15) / 16;
	pl.PP = 16 * (pl.UC | 1);  // an odd number of chunks: neighbouring pixels on different banks
	pl.chunks = (int)T * pl.UC;
	pl.steps = (pl.chunks + 1) / 2;
	pl.wpitch = pl.steps * 32 + 16;
	pl.rows = g.Cout > 32 ? 64 : 32;
	pl.groups = (g.Cout + 63) / 64;
	pl.RW = (g.Wo - 1) * g.sw + g.kw;
	const bool in_fours = g.Cin % 4 == 0 && (T == 9 || T == 25 || T == 1);
	const int64_t weights = (int64_t)pl.rows * pl.wpitch, raw = std::min(pl.rows, g.Cout) * K;
	const double order = in_fours ? 1.7e-5 * (double)raw : 1.6e-5 * (double)weights + 0.88 * ((pl.steps + 7) / 8) * (pl.rows / 64.0);
	if (least + order + 0.64 + 0.55 + 0.1 * pl.steps >= limit_us) return false;  // (one round of the shortest bands)
	double best = limit_us;
	// of the heights that cut an image into the same number of bands the least
	for (int tb = 1, bands = 0; tb <= g.Ho && (int64_t)tb * g.Wo <= 1024; tb = bands > 1 ? (g.Ho + bands - 2) / (bands - 1) : g.Ho + 1) {
		bands = (g.Ho + tb - 1) / tb;
		const int rh = (tb - 1) * g.sh + g.kh, pairs = (tb * g.Wo + 63) / 64;
		const int64_t region = (int64_t)rh * pl.RW * pl.PP;
		const int64_t bytes = align16(region) + weights + align16(raw) + 8 * pl.steps + 16 + pairs * 256 + 9 * 256;
		if (bytes > 160 * 1024) break;
		bool whole = true;  // every band has the 16 bytes of a channel that a load takes (the first and the last have the fewest rows inside the image)
		for (int b = 0; b < bands; b += std::max(bands - 1, 1)) {
			const int top = b * tb * g.sh - g.ph, rows = std::min(tb, g.Ho - b * tb);
			const int inside = std::min(top + (rows - 1) * g.sh + g.kh, g.H) - std::max(top, 0);
			whole = whole && inside > 0 && (int64_t)inside * g.W >= 16;
		}
		if (!whole || (int64_t)g.N * bands >= (1ll << 32) / 512) continue;  // (HIP launches fewer than 2^32 threads in a dimension)
		const int fn = pl.rows == 64 && pairs > 4 ? 2 : 1;
		const int units = pairs * (pl.rows / (32 * fn)), turns = (units + 7) / 8;
		const double rounds = (double)(((int64_t)g.N * bands * pl.groups + 255) / 256);
		const int passes = (int)((((int64_t)rh * g.W + 127) / 128 * ((pl.UC + 1) / 2) + 7) / 8);  // tiles of 8 x 16 pixels of 32 channels a wavefront stages
		const double t = least + rounds * (3.2e-5 * (double)region + 0.64 * passes + order + turns * (0.55 * fn + 0.05 * pl.steps * (fn + 1)));
		if (t < best) {
			best = t;
			pl.TB = tb; pl.RH = rh; pl.bands = bands; pl.pairs = pairs;
			pl.off_w = (unsigned)align16(region);
			pl.off_raw = pl.off_w + (unsigned)weights;
			pl.off_tab = pl.off_raw + (unsigned)align16(raw);
			pl.off_pos = pl.off_tab + (unsigned)align16(8 * pl.steps);
			pl.off_row = pl.off_pos + (unsigned)pairs * 256;
			pl.off_sum = pl.off_row + 8 * 256;
			pl.bytes = pl.off_sum + 256;
		}
	}
	return best < limit_us;
}

// 0 = launched; -1 = not a shape for this route, or not expected to be over within limit_us
int conv2dq_region_dispatch(const ConvGeo& g, const uint8_t* x, const uint8_t* w, const int32_t* bias, int zp_in, int zp_w, float mult, float zp_out, uint8_t* y,
                            double limit_us)
{
	RegionPlan pl;
	if (!region_plan(g, pl, limit_us)) return -1;
	RegionConv c;
	const int T = g.kh * g.kw, K = g.Cin * T;
	c.coef_a = 128 - zp_w;
	c.coef_b = 128 - zp_in;
	// (the channels past Cin count 128 each in a position's sum)
	c.konst = (int32_t)((uint32_t)K * (uint32_t)(zp_in * zp_w - 16384) - (uint32_t)c.coef_a * (uint32_t)(128 * T * (pl.UC * 16 - g.Cin)));
	c.mult = mult;
	c.zp_c = zp_out;
	const bool exact = !(mult == mult && (mult < 0 ? -mult : mult) <= 0.99f), rowsum = c.coef_a != 0, two = pl.rows == 64 && pl.pairs > 4;
	const dim3 grid((unsigned)(g.N * pl.bands), (unsigned)pl.groups), block(512);
	set_kernel_name("conv2dq_region");
#define LTEN_LAUNCH(OUTV, SUMS)                                                                                                    \
	if (two) conv2dq_region_kernel<OUTV, SUMS, 2><<<grid, block, pl.bytes, stream()>>>(g, pl, c, x, w, bias, y);               \
	else conv2dq_region_kernel<OUTV, SUMS, 1><<<grid, block, pl.bytes, stream()>>>(g, pl, c, x, w, bias, y);
	if (exact && rowsum) { LTEN_LAUNCH(Q_OUT_U8_EXACT, true) }
	else if (exact) { LTEN_LAUNCH(Q_OUT_U8_EXACT, false) }
	else if (rowsum) { LTEN_LAUNCH(Q_OUT_U8_FAST, true) }
	else { LTEN_LAUNCH(Q_OUT_U8_FAST, false) }
#undef LTEN_LAUNCH
	LTEN_HIP_LAUNCH_CHECK();
	return 0;
}

}  // namespace lten_hip
