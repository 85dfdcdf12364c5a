// Conv2d_q forward for layers with more than a little work, in two launches: the input turned to pixels of channels, then an
// implicit GEMM on the int8 matrix cores (l-ten/conv2d.cpp:265-387; arithmetic as in convq.hip and convq_image.hip).
//
// The first launch writes x as [n][row + padding][column + padding][channel], 16-byte chunks of 16 channels (channels past
// Cin hold the byte that counts as nothing, pixels of the padding hold l-ten's byte 0), and the weights as rows of
// (tap, channel) with their byte sums.  The second multiplies positions x channels tiles: the 16 bytes a lane loads for
// position p, tap (i, j) and chunk c lie at base(p) + (i, j, c), so the patches are gathered by the direct global->LDS
// loads themselves and never written anywhere.
//
// 32 x 64 x 56 x 56 -> 64 channels 3 x 3: 29.2 -> 16 us (4.3 + 9.7 by the profiler and the gap between them; the band
// kernel of convq_image.hip spends its time in phases that all its workgroups pass together).  Of the second launch's 9.7
// us 3.7 are a launch with one k-step and no store, 1.5 the stores, 1.4 the loads of the other eight k-steps, the rest the
// operand reads from LDS and the products; 3 or 4 tiles a CU (784 on 256) make the last wave.  Reading a k-step's operands
// while the one before is multiplied was slower (13.3 us: it takes the registers of a fourth wavefront).
// 36 x 127 x 47 x 47 -> 192 channels 5 x 5: 375 -> 114 us (three launches before).
#include <algorithm>
#include "conv_common.h"
#include "lds_async.h"
#include "qgemm_common.h"

namespace lten_hip {

struct PixelPlan {
	int Hp, Wp, Cp, UC, chunks, Kp;  // padded sides; channel bytes of a pixel, in chunks of 16; chunks of a window; bytes of a weight row
	uint64_t x_bytes, off_w, off_sums, bytes;
	int px_tiles, cgroups;           // first launch: blocks of 128 pixels, of 64 channels
	unsigned inner_blocks, border_blocks;
	int border;                      // pixels of padding in an image
};

struct PixelConv {
	const uint8_t* xp;
	const uint8_t* wp;
	const int32_t* wsum;
	const int32_t* bias;  // per position, or null
	uint8_t* y;
	int M, HW, Wo, Cout;
	uint32_t image, row, step_h, step_w;  // bytes of xp: an image, a row; from one output row / column to the next
	int Cp, UC, chunks, Kp, kw;
	unsigned inv_uc, inv_kw;
	int32_t konst, coef_a, coef_b;
	float mult, zp_c;
};

// loads and stores on any byte
typedef v4i bytes16 __attribute__((aligned(1)));
typedef uint32_t bytes4 __attribute__((aligned(1)));

__global__ __launch_bounds__(256) void conv2dq_pixels_kernel(ConvGeo g, PixelPlan pl, const uint8_t* __restrict__ x, const uint8_t* __restrict__ w,
                                                             uint8_t* __restrict__ xp, uint8_t* __restrict__ wp, int32_t* __restrict__ wsum, uint32_t flip)
{
	__shared__ __attribute__((aligned(16))) uint8_t s_px[128 * 80];
	__shared__ int s_sum[4];
	const int tid = threadIdx.x;
	unsigned blk = blockIdx.x;
	if (blk < pl.inner_blocks) {
		// 128 pixels x 64 channels: twice four pixels of four channels per thread, transposed in registers, through LDS into
		// runs of 64 bytes
		const unsigned per_image = (unsigned)pl.px_tiles * (unsigned)pl.cgroups;
		const int n = (int)(blk / per_image), rest = (int)(blk - (unsigned)n * per_image);
		const int cg = rest / pl.px_tiles, p0 = (rest - cg * pl.px_tiles) * 128;
		const int HW = g.H * g.W;
		const int pg = tid & 15, c4 = cg * 64 + (tid >> 4) * 4;
		const uint8_t* const xn = x + (int64_t)n * g.Cin * HW;
		uint32_t d[2][4];
#pragma unroll
		for (int h = 0; h < 2; h++) {
			const int p = p0 + h * 64 + pg * 4;
			if (p + 4 <= HW) {
#pragma unroll
				for (int i = 0; i < 4; i++) d[h][i] = *reinterpret_cast<const bytes4*>(xn + (int64_t)min(c4 + i, g.Cin - 1) * HW + p);
			} else {  // the image's last pixels
#pragma unroll
				for (int i = 0; i < 4; i++) {
					const uint8_t* const src = xn + (int64_t)min(c4 + i, g.Cin - 1) * HW;
					uint32_t b[3];
#pragma unroll
					for (int e = 0; e < 3; e++) b[e] = src[min(p + e, HW - 1)];
					d[h][i] = b[0] | b[1] << 8 | b[2] << 16;
				}
			}
		}
#pragma unroll
		for (int h = 0; h < 2; h++) {
#pragma unroll
			for (int i = 0; i < 4; i++)
				if (c4 + i >= g.Cin) d[h][i] = 0x80808080u;
			const uint32_t lo01 = __builtin_amdgcn_perm(d[h][1], d[h][0], 0x05010400u), hi01 = __builtin_amdgcn_perm(d[h][1], d[h][0], 0x07030602u);
			const uint32_t lo23 = __builtin_amdgcn_perm(d[h][3], d[h][2], 0x05010400u), hi23 = __builtin_amdgcn_perm(d[h][3], d[h][2], 0x07030602u);
			uint8_t* const dst = s_px + (h * 64 + pg * 4) * 80 + (tid >> 4) * 4;
			*reinterpret_cast<uint32_t*>(dst) = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u) ^ flip;
			*reinterpret_cast<uint32_t*>(dst + 80) = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u) ^ flip;
			*reinterpret_cast<uint32_t*>(dst + 160) = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u) ^ flip;
			*reinterpret_cast<uint32_t*>(dst + 240) = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u) ^ flip;
		}
		__syncthreads();
		const int chunk = cg * 4 + (tid & 3);
#pragma unroll
		for (int h = 0; h < 2; h++) {
			const int q = p0 + h * 64 + (tid >> 2);
			if (q < HW && chunk < pl.UC) {
				const int yy = q / g.W, xx = q - yy * g.W;
				const uint64_t at = ((uint64_t)((uint64_t)n * pl.Hp + yy + g.ph) * pl.Wp + xx + g.pw) * pl.Cp + chunk * 16;
				*reinterpret_cast<v4i*>(xp + at) = *reinterpret_cast<const v4i*>(s_px + (h * 64 + (tid >> 2)) * 80 + (tid & 3) * 16);
			}
		}
		return;
	}
	blk -= pl.inner_blocks;
	if (blk < pl.border_blocks) {
		const uint64_t idx = (uint64_t)blk * 256 + tid, per_image = (uint64_t)pl.border * pl.UC;
		if (idx >= per_image * g.N) return;
		const int n = (int)(idx / per_image);
		const uint32_t r = (uint32_t)(idx - (uint64_t)n * per_image);
		int b = (int)(r / (uint32_t)pl.UC);
		const int chunk = (int)r - b * pl.UC;
		int yy, xx;
		if (b < 2 * g.ph * pl.Wp) {  // the rows above and below the image
			const int row = b / pl.Wp;
			yy = row < g.ph ? row : row + g.H;
			xx = b - row * pl.Wp;
		} else {
			b -= 2 * g.ph * pl.Wp;
			const int row = b / (2 * g.pw), col = b - row * 2 * g.pw;
			yy = g.ph + row;
			xx = col < g.pw ? col : col + g.W;
		}
		v4i v;
#pragma unroll
		for (int d = 0; d < 4; d++) {
			const int live = min(max(g.Cin - chunk * 16 - d * 4, 0), 4);  // real channels of the dword hold 0, the others 0x80
			v[d] = (int)((live == 4 ? 0u : 0x80808080u << (8 * live)) ^ flip);
		}
		*reinterpret_cast<v4i*>(xp + ((uint64_t)((uint64_t)n * pl.Hp + yy) * pl.Wp + xx) * pl.Cp + chunk * 16) = v;
		return;
	}
	// an output channel's weights
	const int co = (int)(blk - pl.border_blocks), T = g.kh * g.kw, K = g.Cin * T;
	const uint8_t* const wr = w + (int64_t)co * K;
	unsigned sum = 0;
	for (int k = tid * 4; k < pl.Kp; k += 1024) {
		const int t = k / pl.Cp, c = k - t * pl.Cp;
		uint32_t v = 0x80808080u;
		if (t < T) {
#pragma unroll
			for (int e = 0; e < 4; e++) {
				const uint32_t raw = wr[min(c + e, g.Cin - 1) * T + t];
				if (c + e < g.Cin) v = (v & ~(0xFFu << (8 * e))) | raw << (8 * e);
			}
			sum = __builtin_amdgcn_sad_u8(v, 0u, sum) - 128u * (unsigned)(4 - min(max(g.Cin - c, 0), 4));
		}
		*reinterpret_cast<uint32_t*>(wp + (int64_t)co * pl.Kp + k) = v ^ 0x80808080u;
	}
#pragma unroll
	for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
	if ((tid & 63) == 0) s_sum[tid >> 6] = (int)sum;
	__syncthreads();
	if (tid == 0) wsum[co] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

template <int N>
__device__ __forceinline__ void wait_vm()
{
	asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// byte of xp at which the window of output position m starts
__device__ __forceinline__ uint32_t position_base(const PixelConv& p, int pos_all)
{
	const uint32_t m = (uint32_t)pos_all, n = m / (uint32_t)p.HW, pos = m - n * (uint32_t)p.HW, ho = pos / (uint32_t)p.Wo, wo = pos - ho * (uint32_t)p.Wo;
	return n * p.image + ho * p.step_h + wo * p.step_w;
}

// chunk of a window -> (tap row, tap column, 16 channels), as bytes from the window's start
__device__ __forceinline__ uint32_t chunk_offset(const PixelConv& p, int c)
{
	const int t = p.inv_uc == 0 ? c : (int)__umulhi((unsigned)c, p.inv_uc), cc = c - t * p.UC;
	const int i = p.inv_kw == 0 ? t : (int)__umulhi((unsigned)t, p.inv_kw), j = t - i * p.kw;
	return (uint32_t)i * p.row + (uint32_t)(j * p.Cp + cc * 16);
}

// 32 positions from m32 on by 32 channels, element [q][e] of a lane: position m32 + 8 q + 4 lgrp + e of channel co
template <int OUT>
__device__ __forceinline__ void store_block(const PixelConv& p, const v4i (&v)[4], int m32, int co, int lgrp)
{
	unsigned word[4];
#pragma unroll
	for (int q = 0; q < 4; q++) {
		word[q] = 0;
		if (OUT == Q_OUT_U8_FAST) {
			requant_into<0>(word[q], v[q].x, p.mult, p.zp_c);
			requant_into<1>(word[q], v[q].y, p.mult, p.zp_c);
			requant_into<2>(word[q], v[q].z, p.mult, p.zp_c);
			requant_into<3>(word[q], v[q].w, p.mult, p.zp_c);
		} else {
			word[q] = requant<OUT>(v[q].x, p.mult, p.zp_c) | requant<OUT>(v[q].y, p.mult, p.zp_c) << 8 | requant<OUT>(v[q].z, p.mult, p.zp_c) << 16 |
			          requant<OUT>(v[q].w, p.mult, p.zp_c) << 24;
		}
	}
	// the lane halves trade so that each holds 16 neighbouring positions: one store (on any byte) where they lie in one image
	const unsigned give0 = lgrp ? word[0] : word[2], give1 = lgrp ? word[1] : word[3];
	const unsigned got0 = (unsigned)__shfl_xor((int)give0, 32, 64), got1 = (unsigned)__shfl_xor((int)give1, 32, 64);
	const v4i out = lgrp ? v4i{ (int)got0, (int)word[2], (int)got1, (int)word[3] } : v4i{ (int)word[0], (int)got0, (int)word[1], (int)got1 };
	const int m = m32 + lgrp * 16;
	if (m >= p.M || co >= p.Cout) return;
	const int n = (int)((uint32_t)m / (uint32_t)p.HW);
	int pos = m - n * p.HW;
	uint8_t* dst = p.y + ((int64_t)n * p.Cout + co) * p.HW + pos;
	if (pos + 16 <= p.HW) {
		*reinterpret_cast<bytes16*>(dst) = out;
		return;
	}
#pragma unroll
	for (int d = 0; d < 4; d++) {
		const unsigned four = (unsigned)out[d];
		if (pos + 4 <= p.HW && m + 4 * d < p.M) {
			*reinterpret_cast<bytes4*>(dst) = four;
			pos += 4;
			dst += 4;
		} else {
#pragma unroll
			for (int e = 0; e < 4; e++) {
				if (m + 4 * d + e < p.M) *dst = (uint8_t)(four >> (8 * e));
				dst++;
				if (++pos == p.HW) {  // on to the next image
					pos = 0;
					dst += (int64_t)(p.Cout - 1) * p.HW;
				}
			}
		}
		if (pos == p.HW) {
			pos = 0;
			dst += (int64_t)(p.Cout - 1) * p.HW;
		}
	}
}

template <int BM, int BN, int WM, int WN, int S, int OUT, bool ROWSUM>
__global__ __launch_bounds__(WM* WN * 64) void conv2dq_implicit_kernel(PixelConv p)
{
	constexpr int W = WM * WN, BK = 64, CPR = BK / 16, RPL = 64 / CPR, STAGE = (BM + BN) * BK;
	constexpr int NA = BM / RPL / W, NBL = BN / RPL / W, LPW = NA + NBL;
	constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32;
	static_assert((BM / RPL) % W == 0 && (BN / RPL) % W == 0 && TM % 32 == 0 && TN % 32 == 0 && S >= 2 && S <= 4, "tile shape");
	__shared__ __attribute__((aligned(1024))) uint8_t smem[S * STAGE];
	__shared__ __attribute__((aligned(16))) int s_pos[BM];  // what a position adds to its sums: constant, bias, input sum

	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int wm = wave / WN, wn = wave % WN;
	// each XCD takes a contiguous run of tiles, the channel blocks of a block of positions together
	const int tiles_n = (p.Cout + BN - 1) / BN;
	const int nb = (int)gridDim.x, xcd = (int)blockIdx.x & 7;
	const int lid = xcd * (nb >> 3) + min(xcd, nb & 7) + ((int)blockIdx.x >> 3);
	const int m0 = (lid / tiles_n) * BM, n0 = (lid % tiles_n) * BN;

	// this lane's chunk of a k-step is the same in all its loads (rows 16 apart have the same swizzle)
	const int kcl = (lane % CPR) ^ swz<CPR>(lane / CPR);
	uint32_t abase[NA], bbase[NBL];
#pragma unroll
	for (int i = 0; i < NA; i++) abase[i] = position_base(p, min(m0 + (wave + i * W) * RPL + lane / CPR, p.M - 1));
#pragma unroll
	for (int i = 0; i < NBL; i++) bbase[i] = (uint32_t)min(n0 + (wave + i * W) * RPL + lane / CPR, p.Cout - 1) * (uint32_t)p.Kp + kcl * 16;
	const uint32_t smem_addr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
	auto issue = [&](int stage, int kt) {
		// (chunks past the last tap repeat it, their weights are zeros)
		const uint32_t off = chunk_offset(p, min(kt * CPR + kcl, p.chunks - 1));
#pragma unroll
		for (int q = 0; q < NA; q++) async_load16(smem_addr + stage * STAGE + (wave + q * W) * 1024, p.xp, abase[q] + off);
#pragma unroll
		for (int q = 0; q < NBL; q++) async_load16(smem_addr + stage * STAGE + BM * BK + (wave + q * W) * 1024, p.wp + kt * BK, bbase[q]);
	};
	const int lrow = lane & 31, lgrp = lane >> 5;
	for (int r = tid; r < BM; r += W * 64) s_pos[r] = p.konst + (p.bias != nullptr ? p.bias[(uint32_t)min(m0 + r, p.M - 1) % (uint32_t)p.HW] : 0);
	int ct[FN];
#pragma unroll
	for (int i = 0; i < FN; i++) ct[i] = p.coef_b * p.wsum[min(n0 + wn * TN + i * 32 + lrow, p.Cout - 1)];

	const int KT = p.Kp / BK;
#pragma unroll
	for (int st = 0; st < S - 1; st++)
		if (st < KT) issue(st, st);

	const int off_x = (wm * TM + lrow) * BK + ((lgrp ^ swz<CPR>(lrow)) << 4);
	const int off_w = BM * BK + (wn * TN + lrow) * BK + ((lgrp ^ swz<CPR>(lrow)) << 4);
	v16i acc[FM][FN];
	unsigned rsum[FM];
#pragma unroll
	for (int j = 0; j < FM; j++) {
		rsum[j] = 0;
#pragma unroll
		for (int i = 0; i < FN; i++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc[j][i][r] = 0;
	}
	int stage = 0;
	for (int kt = 0; kt < KT; kt++) {
		// k-step kt has landed (at most the S - 2 behind it are still on their way), and everybody has left the stage
		// before it, which is filled again
		if (S >= 4 && kt + 2 < KT) wait_vm<(S >= 4 ? 2 : 0) * LPW>();
		else if (S >= 3 && kt + 1 < KT) wait_vm<(S >= 3 ? 1 : 0) * LPW>();
		else wait_vm<0>();
		__syncthreads();
		if (kt + S - 1 < KT) issue(stage == 0 ? S - 1 : stage - 1, kt + S - 1);
		const uint8_t* const sb = smem + stage * STAGE;
		v4i fx[2][FM], fw[2][FN];
#pragma unroll
		for (int s = 0; s < 2; s++) {
#pragma unroll
			for (int j = 0; j < FM; j++) fx[s][j] = *reinterpret_cast<const v4i*>(sb + (off_x ^ (s << 5)) + j * 32 * BK);
#pragma unroll
			for (int i = 0; i < FN; i++) fw[s][i] = *reinterpret_cast<const v4i*>(sb + (off_w ^ (s << 5)) + i * 32 * BK);
		}
#pragma unroll
		for (int s = 0; s < 2; s++) {
			if (ROWSUM) {
				const bool real = kt * CPR + 2 * s + lgrp < p.chunks;
#pragma unroll
				for (int j = 0; j < FM; j++) {
					unsigned add = 0;
#pragma unroll
					for (int d = 0; d < 4; d++) add = __builtin_amdgcn_sad_u8((unsigned)fx[s][j][d], 0u, add);
					rsum[j] += real ? add : 0u;
					fx[s][j] = flip_sign_bits(fx[s][j]);
				}
			}
#pragma unroll
			for (int j = 0; j < FM; j++)
#pragma unroll
				for (int i = 0; i < FN; i++) acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx[s][j], fw[s][i], acc[j][i], 0, 0, 0);
		}
		stage = stage + 1 == S ? 0 : stage + 1;
	}
	if (ROWSUM) {
#pragma unroll
		for (int j = 0; j < FM; j++) {
			const int both = (int)rsum[j] + __shfl_xor((int)rsum[j], 32, 64);
			if (wn == 0 && lgrp == 0) s_pos[wm * TM + j * 32 + lrow] += p.coef_a * both;
		}
		__syncthreads();
	}
	// lane (lrow, lgrp), register 4q + e of block (j, i): position m0 + wm TM + 32 j + 8 q + 4 lgrp + e of channel n0 + wn TN + 32 i + lrow
#pragma unroll
	for (int j = 0; j < FM; j++)
#pragma unroll
		for (int i = 0; i < FN; i++) {
			v4i v[4];
#pragma unroll
			for (int q = 0; q < 4; q++) {
				const v4i pt = *reinterpret_cast<const v4i*>(&s_pos[wm * TM + j * 32 + 8 * q + 4 * lgrp]);
#pragma unroll
				for (int e = 0; e < 4; e++) v[q][e] = acc[j][i][q * 4 + e] + pt[e] + ct[i];
			}
			store_block<OUT>(p, v, m0 + wm * TM + j * 32, n0 + wn * TN + i * 32 + lrow, lgrp);
		}
}

// The same for few tiles and a long reduction: the wavefronts of a workgroup share the k-steps of one small tile, each out of a
// ring of its own (as qgemm_wave.hip does), and their sums meet in LDS.
template <int BM, int BN, int NW, int S, int OUT, bool ROWSUM>
__global__ __launch_bounds__(NW * 64) void conv2dq_implicit_wave_kernel(PixelConv p)
{
	constexpr int BK = 64, CPR = BK / 16, RPL = 64 / CPR, STAGE = (BM + BN) * BK;
	constexpr int NA = BM / RPL, NBL = BN / RPL, LPW = NA + NBL, FM = BM / 32, FN = BN / 32, NB = FM * FN;
	static_assert(S >= 2 && S <= 4 && (S - 1) * LPW < 64 && NB * 4096 <= S * STAGE, "pipeline shape");
	__shared__ __attribute__((aligned(1024))) uint8_t smem[NW * S * STAGE];
	__shared__ int row_sums[ROWSUM ? NW * BM : 1];
	__shared__ __attribute__((aligned(16))) int s_pos[BM];

	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int tiles_n = (p.Cout + BN - 1) / BN;
	const int nb = (int)gridDim.x, xcd = (int)blockIdx.x & 7;
	const int lid = xcd * (nb >> 3) + min(xcd, nb & 7) + ((int)blockIdx.x >> 3);
	const int m0 = (lid / tiles_n) * BM, n0 = (lid % tiles_n) * BN;
	const int kcl = (lane % CPR) ^ swz<CPR>(lane / CPR);
	uint32_t abase[NA], bbase[NBL];
#pragma unroll
	for (int i = 0; i < NA; i++) abase[i] = position_base(p, min(m0 + i * RPL + lane / CPR, p.M - 1));
#pragma unroll
	for (int i = 0; i < NBL; i++) bbase[i] = (uint32_t)min(n0 + i * RPL + lane / CPR, p.Cout - 1) * (uint32_t)p.Kp + kcl * 16;
	uint8_t* const ring = smem + wave * (S * STAGE);
	const uint32_t ring_addr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)ring;
	auto issue = [&](int stage, int kt) {
		const uint32_t off = chunk_offset(p, min(kt * CPR + kcl, p.chunks - 1));
#pragma unroll
		for (int q = 0; q < NA; q++) async_load16(ring_addr + stage * STAGE + q * 1024, p.xp, abase[q] + off);
#pragma unroll
		for (int q = 0; q < NBL; q++) async_load16(ring_addr + stage * STAGE + (NA + q) * 1024, p.wp + kt * BK, bbase[q]);
	};
	const int lrow = lane & 31, lgrp = lane >> 5;
	for (int r = tid; r < BM; r += NW * 64) s_pos[r] = p.konst + (p.bias != nullptr ? p.bias[(uint32_t)min(m0 + r, p.M - 1) % (uint32_t)p.HW] : 0);
	int ct[FN];
#pragma unroll
	for (int i = 0; i < FN; i++) ct[i] = p.coef_b * p.wsum[min(n0 + i * 32 + lrow, p.Cout - 1)];
	const int KT = p.Kp / BK, n_steps = wave < KT ? (KT - wave + NW - 1) / NW : 0;
#pragma unroll
	for (int st = 0; st < S; st++)
		if (st < n_steps) issue(st, wave + st * NW);
	const int off_x = lrow * BK + ((lgrp ^ swz<CPR>(lrow)) << 4), off_w = BM * BK + off_x;
	v16i acc[FM][FN];
	unsigned rsum[FM];
#pragma unroll
	for (int j = 0; j < FM; j++) {
		rsum[j] = 0;
#pragma unroll
		for (int i = 0; i < FN; i++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc[j][i][r] = 0;
	}
	int stage = 0;
	for (int t = 0; t < n_steps; t++) {
		const int ahead = min(S - 1, n_steps - 1 - t);  // k-steps behind this one that may still be on their way
		if (S >= 4 && ahead >= 3) wait_vm<(S >= 4 ? 3 : 0) * LPW>();
		else if (S >= 3 && ahead == 2) wait_vm<(S >= 3 ? 2 : 0) * LPW>();
		else if (ahead == 1) wait_vm<LPW>();
		else wait_vm<0>();
		const uint8_t* const sb = ring + stage * STAGE;
		v4i fx[2][FM], fw[2][FN];
#pragma unroll
		for (int s = 0; s < 2; s++) {
#pragma unroll
			for (int j = 0; j < FM; j++) fx[s][j] = *reinterpret_cast<const v4i*>(sb + (off_x ^ (s << 5)) + j * 32 * BK);
#pragma unroll
			for (int i = 0; i < FN; i++) fw[s][i] = *reinterpret_cast<const v4i*>(sb + (off_w ^ (s << 5)) + i * 32 * BK);
		}
		if (t + S < n_steps) {
			asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // the stage is in registers
			issue(stage, wave + (t + S) * NW);
		}
#pragma unroll
		for (int s = 0; s < 2; s++) {
			if (ROWSUM) {
				const bool real = (wave + t * NW) * CPR + 2 * s + lgrp < p.chunks;
#pragma unroll
				for (int j = 0; j < FM; j++) {
					unsigned add = 0;
#pragma unroll
					for (int d = 0; d < 4; d++) add = __builtin_amdgcn_sad_u8((unsigned)fx[s][j][d], 0u, add);
					rsum[j] += real ? add : 0u;
					fx[s][j] = flip_sign_bits(fx[s][j]);
				}
			}
#pragma unroll
			for (int j = 0; j < FM; j++)
#pragma unroll
				for (int i = 0; i < FN; i++) acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx[s][j], fw[s][i], acc[j][i], 0, 0, 0);
		}
		stage = stage + 1 == S ? 0 : stage + 1;
	}
	if (ROWSUM) {
#pragma unroll
		for (int j = 0; j < FM; j++) {
			const int both = (int)rsum[j] + __shfl_xor((int)rsum[j], 32, 64);
			if (lgrp == 0) row_sums[wave * BM + j * 32 + lrow] = both;
		}
	}
	__syncthreads();  // every wavefront has left its ring
#pragma unroll
	for (int j = 0; j < FM; j++)
#pragma unroll
		for (int i = 0; i < FN; i++)
#pragma unroll
			for (int q = 0; q < 4; q++)
				*reinterpret_cast<v4i*>(smem + (((wave * NB + i * FM + j) * 4 + q) * 64 + lane) * 16) =
				    v4i{ acc[j][i][q * 4], acc[j][i][q * 4 + 1], acc[j][i][q * 4 + 2], acc[j][i][q * 4 + 3] };
	if (ROWSUM) {
		for (int r = tid; r < BM; r += NW * 64) {
			int sum = 0;
#pragma unroll
			for (int w = 0; w < NW; w++) sum += row_sums[w * BM + r];
			s_pos[r] += p.coef_a * sum;
		}
	}
	__syncthreads();
#pragma unroll
	for (int b = 0; b < NB; b++) {
		if (b % NW != wave) continue;
		const int i = b / FM, j = b % FM;
		v4i v[4];
#pragma unroll
		for (int q = 0; q < 4; q++) {
			v[q] = *reinterpret_cast<const v4i*>(&s_pos[j * 32 + 8 * q + 4 * lgrp]) + v4i{ ct[i], ct[i], ct[i], ct[i] };
#pragma unroll
			for (int w = 0; w < NW; w++) v[q] += *reinterpret_cast<const v4i*>(smem + (((w * NB + b) * 4 + q) * 64 + lane) * 16);
		}
		store_block<OUT>(p, v, m0 + j * 32, n0 + i * 32 + lrow, lgrp);
	}
}

static uint64_t align256(uint64_t v) { return (v + 255) & ~255ull; }

static bool pixel_plan(const ConvGeo& g, PixelPlan& pl)
{
	const int64_t T = (int64_t)g.kh * g.kw;
	if (T > 1024 || g.Cin > 4096) return false;
	pl.Hp = g.H + 2 * g.ph;
	pl.Wp = g.W + 2 * g.pw;
	pl.Cp = (g.Cin + 15) & ~15;
	pl.UC = pl.Cp / 16;
	if (T * pl.UC > 4096) return false;  // (the reciprocals of the chunk's split are exact up to there)
	pl.chunks = (int)T * pl.UC;
	pl.Kp = (pl.chunks * 16 + 63) & ~63;
	pl.x_bytes = (uint64_t)g.N * pl.Hp * pl.Wp * pl.Cp;
	pl.off_w = align256(pl.x_bytes);
	pl.off_sums = pl.off_w + align256((uint64_t)g.Cout * pl.Kp);
	pl.bytes = pl.off_sums + 4ull * g.Cout;
	pl.px_tiles = (int)ceil_div((uint64_t)g.H * g.W, 128);
	pl.cgroups = (pl.Cp + 63) / 64;
	pl.border = pl.Hp * pl.Wp - g.H * g.W;
	const uint64_t inner = (uint64_t)g.N * pl.px_tiles * pl.cgroups, border = ceil_div((uint64_t)g.N * pl.border * pl.UC, 256);
	const uint64_t M = (uint64_t)g.N * g.Ho * g.Wo;
	if (pl.x_bytes >= (1ull << 32) || (uint64_t)g.Cout * pl.Kp >= (1ull << 32) || M >= (1ull << 31) || inner + border + g.Cout >= (1ull << 31)) return false;
	if ((uint64_t)pl.Hp * pl.Wp >= (1ull << 31) || (uint64_t)pl.border * pl.UC >= (1ull << 31)) return false;
	pl.inner_blocks = (unsigned)inner;
	pl.border_blocks = (unsigned)border;
	return true;
}

// What each tile is expected to take with the first launch (us): start and end, a k-step of 64 bytes where every CU has at most
// one tile and what each further tile adds to it, the store of a tile per CU, the megabytes of pixels.  Fitted to 260 layers
// of 1 to 64 images, 4 to 256 channels, 1 x 1 to 5 x 5 windows, strides 1 and 2 (6 % rms).
struct PixelTile {
	int number, bm, bn;
	double start, step, step_more, alone, store, megabyte;
};
static const PixelTile PIXEL_TILES[] = {
	{ 1, 128, 128, 6.3, 0.366, 0.207, 1.0, 1.05, 0.53 },
	{ 2, 128, 64, 5.1, 0.317, 0.134, 1.0, 0.74, 0.57 },
	{ 3, 64, 64, 4.65, 0.259, 0.090, 1.16, 0.46, 0.57 },
	{ 4, 64, 32, 4.35, 0.261, 0.054, 0.85, 0.30, 0.58 },
	{ 5, 32, 32, 4.65, 0.080, 0.035, 0.54, 1.84, 0.60 },  // wavefronts share K
	{ 6, 64, 32, 4.7, 0.111, 0.045, 0.59, 1.05, 0.65 },   // wavefronts share K
};

struct PixelChoice {
	int number;
	double us;
};

static PixelChoice pixel_tile(const ConvGeo& g, const PixelPlan& pl)
{
	PixelChoice best = { 0, 1e30 };
	for (const PixelTile& t : PIXEL_TILES) {
		const double per_cu = (double)(ceil_div((uint64_t)g.N * g.Ho * g.Wo, t.bm) * ceil_div((uint64_t)g.Cout, t.bn)) / 256.0;
		const double us = t.start + pl.Kp / 64 * (t.step + t.step_more * std::max(0.0, per_cu - t.alone)) + t.store * per_cu + t.megabyte * 1e-6 * (double)pl.x_bytes;
		if (us < best.us) best = { t.number, us };
	}
	best.us = std::max(best.us, 6.8);  // two launches in a row (6.6 to 7.4 us for eight of ten of 518 such layers)
	return best;
}

// What the route is expected to take, and the bytes of memory it fills; negative: not a shape for it
double conv2dq_pixels_us(const ConvGeo& g, uint64_t& bytes)
{
	PixelPlan pl;
	if (!pixel_plan(g, pl)) return -1.0;
	bytes = pl.bytes;
	return pixel_tile(g, pl).us;
}

template <int BM, int BN, int WM, int WN, int S>
static void launch_implicit(const PixelConv& p, bool exact, bool rowsum)
{
	const dim3 grid((unsigned)(ceil_div(p.M, BM) * ceil_div(p.Cout, BN))), block(WM * WN * 64);
	if (exact) {
		if (rowsum) conv2dq_implicit_kernel<BM, BN, WM, WN, S, Q_OUT_U8_EXACT, true><<<grid, block, 0, stream()>>>(p);
		else conv2dq_implicit_kernel<BM, BN, WM, WN, S, Q_OUT_U8_EXACT, false><<<grid, block, 0, stream()>>>(p);
	} else {
		if (rowsum) conv2dq_implicit_kernel<BM, BN, WM, WN, S, Q_OUT_U8_FAST, true><<<grid, block, 0, stream()>>>(p);
		else conv2dq_implicit_kernel<BM, BN, WM, WN, S, Q_OUT_U8_FAST, false><<<grid, block, 0, stream()>>>(p);
	}
}

template <int BM, int BN, int NW, int S>
static void launch_implicit_wave(const PixelConv& p, bool exact, bool rowsum)
{
	const dim3 grid((unsigned)(ceil_div(p.M, BM) * ceil_div(p.Cout, BN))), block(NW * 64);
	if (exact) {
		if (rowsum) conv2dq_implicit_wave_kernel<BM, BN, NW, S, Q_OUT_U8_EXACT, true><<<grid, block, 0, stream()>>>(p);
		else conv2dq_implicit_wave_kernel<BM, BN, NW, S, Q_OUT_U8_EXACT, false><<<grid, block, 0, stream()>>>(p);
	} else {
		if (rowsum) conv2dq_implicit_wave_kernel<BM, BN, NW, S, Q_OUT_U8_FAST, true><<<grid, block, 0, stream()>>>(p);
		else conv2dq_implicit_wave_kernel<BM, BN, NW, S, Q_OUT_U8_FAST, false><<<grid, block, 0, stream()>>>(p);
	}
}

// 0 = launched; -1 = not a shape for this route.  memory: the bytes conv2dq_pixels_us names, 16-byte aligned.  forced: tile number from 1,
// 0 the one expected to be quickest.
int conv2dq_pixels_dispatch(const ConvGeo& g, const uint8_t* x, const uint8_t* w, const int32_t* bias, int zp_in, int zp_w, float mult, float zp_out,
                            uint8_t* y, void* memory, int forced)
{
	PixelPlan pl;
	if (!pixel_plan(g, pl)) return -1;
	uint8_t* const base = static_cast<uint8_t*>(memory);
	uint8_t* const wp = base + pl.off_w;
	int32_t* const sums = reinterpret_cast<int32_t*>(base + pl.off_sums);
	PixelConv p;
	p.xp = base; p.wp = wp; p.wsum = sums; p.bias = bias; p.y = y;
	p.HW = g.Ho * g.Wo; p.Wo = g.Wo; p.Cout = g.Cout; p.M = g.N * p.HW;
	p.row = (uint32_t)pl.Wp * (uint32_t)pl.Cp;
	p.image = (uint32_t)pl.Hp * p.row;
	p.step_h = (uint32_t)g.sh * p.row;
	p.step_w = (uint32_t)g.sw * (uint32_t)pl.Cp;
	p.Cp = pl.Cp; p.UC = pl.UC; p.chunks = pl.chunks; p.Kp = pl.Kp; p.kw = g.kw;
	auto inverse = [](unsigned d) { return d <= 1 ? 0u : (unsigned)((0x100000000ull + d - 1) / d); };
	p.inv_uc = inverse((unsigned)pl.UC);
	p.inv_kw = inverse((unsigned)g.kw);
	const int K = g.Cin * g.kh * g.kw;
	p.coef_a = 128 - zp_w;
	p.coef_b = 128 - zp_in;
	// the channels past Cin count 128 each in a position's sum
	p.konst = (int32_t)((uint32_t)K * (uint32_t)(zp_in * zp_w - 16384) - (uint32_t)p.coef_a * (uint32_t)(128 * g.kh * g.kw * (pl.Cp - g.Cin)));
	p.mult = mult;
	p.zp_c = zp_out;
	const bool exact = !(mult == mult && (mult < 0 ? -mult : mult) <= 0.99f), rowsum = p.coef_a != 0;
	conv2dq_pixels_kernel<<<dim3(pl.inner_blocks + pl.border_blocks + (unsigned)g.Cout), dim3(256), 0, stream()>>>(g, pl, x, w, base, wp, sums,
	                                                                                                         rowsum ? 0u : 0x80808080u);
	LTEN_HIP_LAUNCH_CHECK();
	set_kernel_name("conv2dq_pixels");
	switch (forced != 0 ? forced : pixel_tile(g, pl).number) {
	case 1: launch_implicit<128, 128, 2, 2, 3>(p, exact, rowsum); break;
	case 2: launch_implicit<128, 64, 4, 1, 3>(p, exact, rowsum); break;
	case 3: launch_implicit<64, 64, 2, 2, 4>(p, exact, rowsum); break;
	case 4: launch_implicit<64, 32, 2, 1, 4>(p, exact, rowsum); break;
	case 5: launch_implicit_wave<32, 32, 8, 4>(p, exact, rowsum); break;
	default: launch_implicit_wave<64, 32, 4, 3>(p, exact, rowsum); break;
	}
	LTEN_HIP_LAUNCH_CHECK();
	return 0;
}

}  // namespace lten_hip
