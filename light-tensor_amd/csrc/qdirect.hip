// int8 FC for small outputs (a few hundred 16x16 tiles): one launch, operands straight from global memory.
//
// At these sizes (e.g. l-ten's 64 x 784 MNIST batch against a 512 x 784 weight matrix) the run time is launch
// and memory latency, not arithmetic, so the kernel is one dependent chain as short as possible: a workgroup
// owns one 16 x 16 output tile, its wavefronts split K in 64-byte steps (wavefront w takes steps w, w + WAVES,
// ...), the loads of U of its steps at once, and the zero-point byte sums come from the same registers with dot4
// instructions — no separate row-sum launch.  What bounds it is a CU's loads.  The 16x16x64 int8 MFMA wants 16 bytes of 16
// different rows on neighbouring lanes (row lane % 16, k-group lane / 16); loaded like that, rows a multiple of 128 bytes apart
// are slow.  There four lanes of a row load next to each other, and a pass through two KB of LDS brings the bytes into the
// operand layout (64 x 50 x 5760: 7.3 -> 5.2 us, 128 x 48 x 12288 12.7 -> 8.2, 300 x 1000 x 1024 6.8 -> 4.7, 400 x 400 x 2048 7.7 -> 5.1,
// 4096 x 50 x 5760 22.6 -> 17.9; a launch that does nothing: 3 to 4); qdirect_dispatch has the line.
// The partial tiles and sums meet in LDS and wavefront 0 applies the identity of qgemm.hip and the requantize of
// l-ten/math_fns.cpp:1469-1474.
//
// K only has to be a multiple of 16 (k-groups past K read as the zero of the signed domain).
#include "common.h"
#include "qgemm_common.h"

namespace lten_hip {

typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));

// The bytes of v from number `count` on (0 to 15, the same in every lane), the zero of the signed domain behind them.
__device__ __forceinline__ v4i drop_bytes(v4i v, int count)
{
	const uint32_t none = 0x80808080u;
	uint32_t w[5] = { (uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w, none };
	if (count & 8) { w[0] = w[2]; w[1] = w[3]; w[2] = w[3] = none; }
	if (count & 4) { w[0] = w[1]; w[1] = w[2]; w[2] = w[3]; w[3] = none; }
#pragma unroll
	for (int d = 0; d < 4; d++) w[d] = __builtin_amdgcn_alignbyte(w[d + 1], w[d], (uint32_t)count);
	return v4i{ (int)w[0], (int)w[1], (int)w[2], (int)w[3] };
}

// RAGGED: the rows of A as they lie, p.K - p.k_pad bytes long and one behind the other, where those of B are padded to p.K.
// U: steps in flight per wavefront and pass.  DIRECT: operands loaded as the matrix instruction takes them, not through LDS.
template <int WAVES, int U, int OUT, bool RAGGED = false, bool DIRECT = false>
__global__ __launch_bounds__(WAVES * 64) void qdirect_kernel(QProblem p, const int32_t* bias, int coef_a, int coef_b)
{
	__shared__ __attribute__((aligned(16))) uint8_t slabs[WAVES][2048];  // a step of A and of B; a wavefront's sums at the end
	__shared__ int sums_a[WAVES][16], sums_b[WAVES][16];

	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int lrow = lane & 15, lgrp = lane >> 4;
	const int tiles_n = (p.N + 15) / 16;
	const int m0 = (blockIdx.x / tiles_n) * 16, n0 = (blockIdx.x % tiles_n) * 16;
	// loads: in the operand layout, or four lanes to a row, 64 bytes next to each other
	const int ldrow = DIRECT ? lrow : lane >> 2, ldgrp = DIRECT ? lgrp : lane & 3;
	const bool a_ok = m0 + ldrow < p.M, b_ok = n0 + ldrow < p.N;
	const uint8_t* arow = p.A + (int64_t)(m0 + ldrow) * p.a_rs + ldgrp * 16;
	const uint8_t* brow = p.B + (int64_t)(n0 + ldrow) * p.b_rs + ldgrp * 16;
	// through LDS into the operand layout, the four chunks of a row turned so that neither side meets a bank twice
	uint8_t* const to = slabs[wave] + (ldrow * 4 + (ldgrp ^ (ldrow >> 2))) * 16;
	const uint8_t* const from = slabs[wave] + (lrow * 4 + (lgrp ^ (lrow >> 2))) * 16;
	const int steps = (p.K + 63) / 64, real = p.K - p.k_pad;
	const v4i zero = { (int)0x80808080, (int)0x80808080, (int)0x80808080, (int)0x80808080 };
	const v4i zero_b = { (int)p.b_flip, (int)p.b_flip, (int)p.b_flip, (int)p.b_flip };  // prepared weights: int8 zeros

	v4i acc = { 0, 0, 0, 0 };
	int sa = 0, sb = 0;
	auto fetch = [&](int s0, v4i (&fa)[U], v4i (&fb)[U]) {
#pragma unroll
		for (int u = 0; u < U; u++) {
			const int k = (s0 + u * WAVES) * 64 + ldgrp * 16;
			fa[u] = zero;
			fb[u] = zero_b;
			if (k < p.K) {
				const uint8_t* a = arow + (int64_t)(s0 + u * WAVES) * 64;
				if (RAGGED && a_ok) {
					// nothing may be read behind the last row: a row's last chunk is the 16 bytes up to its end, shifted below
					if (real >= 16) fa[u] = *reinterpret_cast<const v4i_any*>(k + 16 <= real ? a : a - p.k_pad);
					else if ((m0 + ldrow) * real + 16 <= p.M * real) {  // rows shorter than that: some of the next ones too, masked
						fa[u] = *reinterpret_cast<const v4i_any*>(a);
#pragma unroll
						for (int d = 0; d < 4; d++) {
							const int live = min(max(real - 4 * d, 0), 4);
							const uint32_t past = live == 4 ? 0u : ~0u << (8 * live);
							fa[u][d] = (int)(((uint32_t)fa[u][d] & ~past) | (0x80808080u & past));
						}
					} else {
#pragma unroll
						for (int d = 0; d < 4; d++) {
							uint32_t word = 0x80808080u;
#pragma unroll
							for (int e = 0; e < 4; e++)
								if (4 * d + e < real) word = (word & ~(0xffu << (8 * e))) | (uint32_t)a[4 * d + e] << (8 * e);
							fa[u][d] = (int)word;
						}
					}
				} else if (a_ok) fa[u] = *reinterpret_cast<const v4i*>(a);
				if (b_ok) fb[u] = *reinterpret_cast<const v4i*>(brow + (int64_t)(s0 + u * WAVES) * 64);
			}
		}
	};
	// A step's operands are asked for back from LDS before the step before is multiplied (LDS serves a wavefront in order, so one
	// slab does): with each step waiting for its own, the way through LDS stood in the chain once a step.
	auto multiply = [&](int s0, v4i (&fa)[U], v4i (&fb)[U]) {
		v4i ma[2], mb[2];
		auto exchange = [&](int u) {
			if (RAGGED && real >= 16 && (s0 + u * WAVES) * 64 + ldgrp * 16 == p.K - 16) fa[u] = drop_bytes(fa[u], p.k_pad);
			const v4i a = flip_sign_bits(fa[u]), b = flip_bits(fb[u], p.b_flip);
			if (DIRECT) {
				ma[u & 1] = a;
				mb[u & 1] = b;
			} else {
				*reinterpret_cast<v4i*>(to) = a;
				*reinterpret_cast<v4i*>(to + 1024) = b;
				__builtin_amdgcn_wave_barrier();
				ma[u & 1] = *reinterpret_cast<const v4i*>(from);
				mb[u & 1] = *reinterpret_cast<const v4i*>(from + 1024);
				__builtin_amdgcn_wave_barrier();
			}
			sa = __builtin_amdgcn_sdot4(a.x, 0x01010101, sa, false);
			sa = __builtin_amdgcn_sdot4(a.y, 0x01010101, sa, false);
			sa = __builtin_amdgcn_sdot4(a.z, 0x01010101, sa, false);
			sa = __builtin_amdgcn_sdot4(a.w, 0x01010101, sa, false);
			sb = __builtin_amdgcn_sdot4(b.x, 0x01010101, sb, false);
			sb = __builtin_amdgcn_sdot4(b.y, 0x01010101, sb, false);
			sb = __builtin_amdgcn_sdot4(b.z, 0x01010101, sb, false);
			sb = __builtin_amdgcn_sdot4(b.w, 0x01010101, sb, false);
		};
		exchange(0);
#pragma unroll
		for (int u = 0; u < U; u++) {
			if (u + 1 < U) exchange(u + 1);
			// lane (lrow, lgrp), register e holds out[m = 4*lgrp + e][n = lrow]
			acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(ma[u & 1], mb[u & 1], acc, 0, 0, 0);
		}
	};
	for (int s0 = wave; s0 < steps; s0 += WAVES * U) {
		v4i fa[U], fb[U];
		fetch(s0, fa, fb);
		multiply(s0, fa, fb);
	}
	// a lane holds the byte sums of its 16-byte k-groups only: fold the four lanes of a row
	constexpr int FOLD = DIRECT ? 16 : 1;
	sa += __shfl_xor(sa, FOLD, 64); sa += __shfl_xor(sa, 2 * FOLD, 64);
	sb += __shfl_xor(sb, FOLD, 64); sb += __shfl_xor(sb, 2 * FOLD, 64);
	if (ldgrp == 0) { sums_a[wave][ldrow] = sa; sums_b[wave][ldrow] = sb; }
	*reinterpret_cast<v4i*>(slabs[wave] + lane * 16) = acc;
	__syncthreads();
	if (wave != 0) return;

	v4i tot = { 0, 0, 0, 0 };
	int tsa[4] = { 0, 0, 0, 0 }, tsb = 0;
#pragma unroll
	for (int w = 0; w < WAVES; w++) {
		tot += *reinterpret_cast<const v4i*>(slabs[w] + lane * 16);
		tsb += sums_b[w][lrow];
#pragma unroll
		for (int e = 0; e < 4; e++) tsa[e] += sums_a[w][lgrp * 4 + e];
	}
	const int n = n0 + lrow;
	if (n >= p.N) return;
	// sum a'b' -> l-ten's element: + coef_a * sum_k a' + coef_b * sum_k b' + K * coef_a * coef_b (+ bias)
	//   with a' = a - 128, coef_a = 128 - zpB, coef_b = 128 - zpA
	const int base = coef_b * tsb + (p.K - p.k_pad) * coef_a * coef_b + (bias ? bias[n] : 0);
#pragma unroll
	for (int e = 0; e < 4; e++) {
		const int m = m0 + lgrp * 4 + e;
		if (m >= p.M) continue;
		const int v = tot[e] + base + coef_a * tsa[e];
		if (OUT == Q_OUT_ACC) static_cast<int*>(p.C)[(int64_t)m * p.N + n] = v;
		else static_cast<uint8_t*>(p.C)[(int64_t)m * p.N + n] = (uint8_t)requant<OUT>(v, p.mult, p.zp_c);
	}
}

// Whether the problem is a small NT product with 16-byte aligned rows that this kernel is the one for.
bool qdirect_takes(const QProblem& p)
{
	if (!(p.a_ks == 1 && p.b_ks == 1 && p.vec_ok && p.K % 16 == 0 && p.M >= 1 && p.N >= 1 && p.K >= 1)) return false;
	const int64_t tiles = (int64_t)ceil_div((uint64_t)p.M, 16) * ceil_div((uint64_t)p.N, 16);
	// Up to 8192 tiles, as long as this kernel is ahead of the 128 x 128 direct-to-LDS tiles where those apply (at least
	// 64 output columns, K >= 512 or at least 64 such tiles: qgemm_dispatch).  Its estimate is 2.3 us + 3 us per million
	// (tiles x K), 3.5 above a K of 1024.  From 64 tiles up it takes 0.6 to 1.9 times that (over 930 layers; 0.8 to 1.3 in the median of a
	// range of sizes).  Below, the chain over K counts, which has no term, and it takes up to four times that (8 us for one tile at K =
	// 16320): there they take longer still.  They take about 5.4 us + 0.33 us per k-step of 128 bytes of a workgroup's share of K while they run in one
	// round, 4 us more when workgroups share tiles (split K, as qgemm_dispatch picks it), 2 us more when N is no multiple
	// of 4 (rows of the output that start on any byte), 2.5 us more with a partial last k-step.  Raw weights, here and there: 851 x
	// 736 x 896 6.8 and 11.3 us, 393 x 1859 x 1040 12.9 and 16.3, 318 x 1338 x 2192 11.0 and 23.1, 463 x 440 x 5296 12.2 and
	// 39.1, 1135 x 191 x 6864 21.7 and 52.0, 45 x 2247 x 14160 24.4 and 97.2; 200 x 2000 x 256 4.3 (13.8 on the guarded kernel,
	// which took it before).  Prepared weights come here only where qgemm_wave_choose leaves them.  A few output
	// columns make poor use of 128-column tiles and stay here (4096 x 50 x 5760, l-ten's quantized MNIST layer at a large
	// batch: 18.1 us).
	if (tiles > 8192 || p.K > 16384) return false;
	const uint64_t tiles128 = ceil_div((uint64_t)p.M, 128) * ceil_div((uint64_t)p.N, 128);
	// (from 64 output columns on: half-empty 128-column tiles still beat this kernel on long or many rows, 4096 x 100 x 9216 58 -> 25
	// us, 16384 x 64 x 1024 17 -> 7.5 us; at 50 columns, l-ten's layer above, they are level)
	const bool tiles_apply = p.N >= 64 && (p.K >= 512 || (p.K >= 32 && tiles128 >= 64)) && (reinterpret_cast<uintptr_t>(p.C) & 15) == 0 &&
	                         (uint64_t)p.M * p.K < (1ull << 32) && (uint64_t)p.N * p.K < (1ull << 32);
	if (tiles_apply) {
		const int splits = (tiles128 <= 64 && p.K >= 8192) ? (tiles128 <= 32 ? 4 : 2) : (tiles128 <= 32 && p.K >= 4096) ? 2 : 1;
		const double here = 2.3 + (p.K <= 1024 ? 3.0e-6 : 3.5e-6) * (double)tiles * p.K;
		const double there = 5.4 + 0.0026 * p.K / splits + (splits > 1 ? 4.0 : 0.0) + (p.N % 4 != 0 ? 2.0 : 0.0) + (p.K % 128 != 0 ? 2.5 : 0.0);
		if (here >= there) return false;
	}
	return true;
}

template <int WAVES, int U, bool RAGGED = false, bool DIRECT = false>
static int launch_qdirect(const QProblem& p, int out, const int32_t* bias, int coef_a, int coef_b)
{
	const dim3 grid((unsigned)(ceil_div((uint64_t)p.M, 16) * ceil_div((uint64_t)p.N, 16))), block(WAVES * 64);
	if (out == Q_OUT_U8_FAST) qdirect_kernel<WAVES, U, Q_OUT_U8_FAST, RAGGED, DIRECT><<<grid, block, 0, stream()>>>(p, bias, coef_a, coef_b);
	else if (out == Q_OUT_U8_EXACT) qdirect_kernel<WAVES, U, Q_OUT_U8_EXACT, RAGGED, DIRECT><<<grid, block, 0, stream()>>>(p, bias, coef_a, coef_b);
	else qdirect_kernel<WAVES, U, Q_OUT_ACC, RAGGED, DIRECT><<<grid, block, 0, stream()>>>(p, bias, coef_a, coef_b);
	LTEN_HIP_LAUNCH_CHECK();
	return 0;
}

// Returns -1 when the problem is not one for this kernel.
int qdirect_dispatch(const QProblem& p, int out, const int32_t* bias, int zp_a, int zp_b)
{
	if (!qdirect_takes(p)) return -1;
	const int coef_a = 128 - zp_b, coef_b = 128 - zp_a;
	// Two steps of a wavefront in flight: places that a wavefront's share of K leaves empty cost more than what they hide (432 x 1406 x
	// 1056: 9.3 us with two, 11.0 with four).  A wavefront alone up to K = 256 (2000 x 200 x 256: 3.6, 4.1 with four wavefronts), four up to
	// 1024 (300 x 1000 x 1024: 4.7, 5.4 with eight; one 6.3), eight above (400 x 400 x 2048: 5.1, 5.3 with four).
	if (p.K <= 256) {
		set_kernel_name("qdirect_16x16_w1");
		return launch_qdirect<1, 2>(p, out, bias, coef_a, coef_b);
	}
	// Operands through LDS where rows lie a multiple of 128 bytes apart (300 x 1000 x 1024: 6.8 us in the operand layout, 4.7 through
	// LDS; 400 x 400 x 2048 7.5 and 5.1).  On other lengths the operand layout is as quick or quicker up to K = 2048 (219 x 2203 x 752:
	// 5.6 and 6.1; 432 x 1406 x 1056: 8.4 and 9.3) and slower above (53 x 1183 x 5392: 8.6 and 7.4; 145 x 861 x 5680 11.4 and 9.3), but
	// where one operand has few rows, whose loads are few accesses either way, the pass through LDS is a longer chain (3 x 15 x 4256:
	// 3.9 and 4.2; 2961 x 1 x 16336: 10.7 and 12.5).  Against the operand layout with four steps in flight everywhere, over 930 layers:
	// 0.915 of the time in the mean, 11 of them 3 to 6 % behind.
	const bool lines = p.K % 128 == 0, few = std::min(p.M, p.N) <= 12;
	const bool direct = lines ? few && p.K <= 4096 : few || p.K <= 2048;
	if (p.K <= 1024) {
		set_kernel_name("qdirect_16x16_w4");
		if (direct) return launch_qdirect<4, 2, false, true>(p, out, bias, coef_a, coef_b);
		return launch_qdirect<4, 2>(p, out, bias, coef_a, coef_b);
	}
	// (four steps in flight on the longest chains: 2961 x 1 x 16336 11.7 us with two, 10.7 with four; 4096 x 50 x 5760 18.9 and 17.9; not
	// through LDS on other lengths, 85 x 612 x 9168 9.3 and 9.9)
	set_kernel_name("qdirect_16x16_w8");
	if (direct && p.K > 8192) return launch_qdirect<8, 4, false, true>(p, out, bias, coef_a, coef_b);
	if (direct) return launch_qdirect<8, 2, false, true>(p, out, bias, coef_a, coef_b);
	if (lines && p.K > 4096) return launch_qdirect<8, 4>(p, out, bias, coef_a, coef_b);
	return launch_qdirect<8, 2>(p, out, bias, coef_a, coef_b);
}

// A with rows of K - k_pad bytes (RAGGED) where the padded problem would come here with at most four wavefronts: the copy that
// pads A is a launch of its own (64 x 10 x 50 7.0 -> 4.0 us, 96 x 512 x 1000 7.1 -> 4.1; with a row's last chunk loaded byte by byte
// large outputs were slower than with the copy, 64 x 8991 x 607 13.3 us and 9.6 where the shifted load takes 10.0, 300 x 1999 x 607
// 13.0, 9.7 and 10.4, 448 x 832 x 607 8.5, 7.7 and 7.3; over 180 shapes it is ahead of the copy by 28 % in the mean, 7 % behind at
// most.  Rows shorter than a chunk: 959 x 1568 x 12 11.2 us byte by byte, 9.6 masked, 9.2 with the copy; 500 x 500 x 12 4.2 and 5.2).
int qdirect_ragged_dispatch(const QProblem& p, int out, const int32_t* bias, int zp_a, int zp_b)
{
	if (p.K > 1024 || !qdirect_takes(p)) return -1;
	set_kernel_name("qdirect_16x16_w4");
	if (p.K <= 256) return launch_qdirect<4, 1, true>(p, out, bias, 128 - zp_b, 128 - zp_a);
	if (p.K <= 512) return launch_qdirect<4, 2, true>(p, out, bias, 128 - zp_b, 128 - zp_a);
	return launch_qdirect<4, 4, true>(p, out, bias, 128 - zp_b, 128 - zp_a);
}

}  // namespace lten_hip
