// int8 GEMM tiles for outputs that give the 128 x 128 tiles of qgemm_fast.hip too few workgroups: FullyConnected_q layers on
// prepared weights (NT: both operands contiguous in K, K a multiple of 16; M and N need not be multiples of the tile), 17
// rows up to a few hundred.
//
// A workgroup owns a BM x BN tile and its wavefronts share K, not the tile: wavefront w multiplies the whole tile over
// the k-steps w, w + NW, w + 2 NW, ... of 128 bytes, each out of a ring of S stages in LDS that no other wavefront
// touches.  Nothing in the main loop waits for another wavefront: no barrier, only the wavefront's own load counter.
// The partial tiles meet in LDS at the end, and the wavefronts share out the blocks of the epilogue.
//
// What bounds it: a CU's loads.  A 64 x 64 tile brings 128 rows x K bytes through the vector L1, 44 bytes a clock of them
// measured, 5.6 of the 9.9 us at 256 x 4096 x 4096 (18.4 us on 64 tiles of 128 x 128, which leave 192 CUs idle); the rest is
// the launch, the first round trip to memory and the exchange of the partial tiles.  Sharing K instead of the tile halves
// the LDS reads (a 64 x 64 tile in 32 x 32 pieces reads every staged byte twice) and needs no barrier; k-steps of 64 bytes
// in a deeper ring were no faster (10.2 us), nor 128 x 64 tiles, whose 192 rows a step take the longer (14.6 us), nor
// eight wavefronts a tile of 64 x 64 (10.6 us).
#include "common.h"
#include "qgemm_common.h"
#include "lds_async.h"

namespace lten_hip {

template <int N>
__device__ __forceinline__ void wait_loads()
{
	// as a statement that touches memory: no LDS read may be moved in front of it
	asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

template <int BM, int BN, int BK, int NW, int S, int OUT, bool ROWSUM>
__global__ __launch_bounds__(NW * 64) void qgemm_wave_kernel(QProblem p)
{
	constexpr int CPR = BK / 16;           // 16-byte chunks per tile row
	constexpr int RPL = 64 / CPR;          // tile rows covered by one wave-wide load
	constexpr int NS = BK / 32;            // k-slices per k-step
	constexpr int STAGE = (BM + BN) * BK;  // bytes
	constexpr int LOADS = STAGE / 1024;    // wave-wide loads per stage, the first NA of activation rows
	constexpr int NA = BM / RPL;
	constexpr int FM = BM / 32, FN = BN / 32, NB = FM * FN;
	static_assert(BM % RPL == 0 && BN % RPL == 0 && NS % 2 == 0 && S >= 2 && S <= 5 && (S - 1) * LOADS < 64, "pipeline shape");
	static_assert(NB * 4096 <= S * STAGE, "the partial tiles fit into the stages");
	__shared__ __attribute__((aligned(1024))) uint8_t smem[NW * S * STAGE];
	__shared__ int row_sums[ROWSUM ? NW * BM : 1];

	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

	// Workgroup -> tile.  Consecutive workgroups go round-robin to the 8 XCDs; each XCD takes a contiguous run of tiles,
	// down the rows first, so that the tiles that share weight rows share an L2.
	const int tiles_m = (p.M + BM - 1) / BM;
	const int nb = (int)gridDim.x, xcd = (int)blockIdx.x & 7;
	const int lid = xcd * (nb >> 3) + min(xcd, nb & 7) + ((int)blockIdx.x >> 3);
	const int m0 = (lid % tiles_m) * BM, n0 = (lid / tiles_m) * BN;

	uint32_t voff[LOADS];
	bool past[NA];  // this lane's activation chunk lies past K in the last k-step
	const int k_rest = p.K % BK;
#pragma unroll
	for (int q = 0; q < LOADS; q++) {
		const int r = q * RPL + lane / CPR;
		const int kc = (lane % CPR) ^ swz<CPR>(r);
		voff[q] = (q < NA ? (uint32_t)min(m0 + r, p.M - 1) : (uint32_t)min(n0 + r - BM, p.N - 1)) * (uint32_t)p.K + kc * 16;
		if (q < NA) past[q] = k_rest != 0 && kc * 16 >= k_rest;
	}
	uint8_t* const ring = smem + wave * (S * STAGE);
	const uint32_t ring_addr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)ring;
	const int steps = (p.K + BK - 1) / BK;
	const int n_steps = wave < steps ? (steps - wave + NW - 1) / NW : 0;

	// What each lane loads of the k-step with number t of this wavefront.  In a partial last k-step a lane whose chunk
	// lies past K loads the row's last chunk again: every k-step issues all LOADS loads, which is what the waits count.
	auto issue = [&](int stage, int t) {
		const int kt = wave + t * NW;
		const bool partial = k_rest != 0 && kt == steps - 1;
#pragma unroll
		for (int q = 0; q < LOADS; q++) {
			uint32_t off = voff[q];
			if (partial) {
				const int r = q * RPL + lane / CPR, kc = (lane % CPR) ^ swz<CPR>(r);
				if (kc * 16 >= k_rest) off -= (uint32_t)(kc * 16 - (k_rest - 16));
			}
			async_load16(ring_addr + stage * STAGE + q * 1024, (q < NA ? p.A : p.B) + (int64_t)kt * BK, off);
		}
	};
	// The chunks past K of a partial k-step, once it has landed: bytes of 0x80, zeros behind the sign flip, so whatever
	// the weights' chunks hold there is multiplied by 0.
	auto pad = [&](int stage, int t) {
		if (k_rest == 0 || wave + t * NW != steps - 1) return;
#pragma unroll
		for (int q = 0; q < NA; q++)
			if (past[q]) *reinterpret_cast<v4i*>(ring + stage * STAGE + q * 1024 + lane * 16) = v4i{ (int)0x80808080, (int)0x80808080, (int)0x80808080, (int)0x80808080 };
	};

	// MFMA operands: lane (lrow, lgrp) feeds row lrow of a 32-row block with the 16 bytes lgrp of a 32-byte k-slice
	const int lrow = lane & 31, lgrp = lane >> 5;
	const int off_x = lrow * BK + ((lgrp ^ swz<CPR>(lrow)) << 4), off_w = BM * BK + off_x;
	v16i acc[FN][FM];
#pragma unroll
	for (int i = 0; i < FN; i++)
#pragma unroll
		for (int j = 0; j < FM; j++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc[i][j][r] = 0;
	unsigned rsum[FM][2];
#pragma unroll
	for (int j = 0; j < FM; j++) rsum[j][0] = rsum[j][1] = 0;
	auto read = [&](v4i(&fw)[FN], v4i(&fx)[FM], int stage, int s) {
		const uint8_t* const b = ring + stage * STAGE;
#pragma unroll
		for (int j = 0; j < FM; j++) fx[j] = *reinterpret_cast<const v4i*>(b + (off_x ^ (s << 5)) + j * 32 * BK);
#pragma unroll
		for (int i = 0; i < FN; i++) fw[i] = *reinterpret_cast<const v4i*>(b + (off_w ^ (s << 5)) + i * 32 * BK);
	};
	auto multiply = [&](const v4i(&fw)[FN], v4i(&fx)[FM]) {
#pragma unroll
		for (int j = 0; j < FM; j++) {
			if (ROWSUM) {
#pragma unroll
				for (int d = 0; d < 4; d++) rsum[j][d & 1] = __builtin_amdgcn_sad_u8((unsigned)fx[j][d], 0u, rsum[j][d & 1]);
			}
			fx[j] = flip_sign_bits(fx[j]);
		}
#pragma unroll
		for (int i = 0; i < FN; i++)
#pragma unroll
			for (int j = 0; j < FM; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fw[i], fx[j], acc[i][j], 0, 0, 0);
	};
	// until at most n of this wavefront's youngest k-steps are still on their way
	auto wait_steps = [&](int n) {
		if (S >= 5 && n >= 4) wait_loads<(S >= 5 ? 4 : 0) * LOADS>();
		else if (S >= 4 && n == 3) wait_loads<(S >= 4 ? 3 : 0) * LOADS>();
		else if (S >= 3 && n == 2) wait_loads<(S >= 3 ? 2 : 0) * LOADS>();
		else if (n == 1) wait_loads<LOADS>();
		else wait_loads<0>();
	};

	// The column terms of the blocks this wavefront finishes: loaded here, where the operands are waited for anyway
	// (behind the main loop they cost a round trip to memory of their own).  A load past the last column fetches the last
	// one; what it is added to is not stored.
	constexpr int MINE = (NB + NW - 1) / NW;
	v4i ct[MINE][4], bt[MINE][4];
#pragma unroll
	for (int u = 0; u < MINE; u++) {
		const int nbase = n0 + min(wave + u * NW, NB - 1) / FM * 32 + lgrp * 4;
#pragma unroll
		for (int q = 0; q < 4; q++) {
			ct[u][q] = bt[u][q] = v4i{ 0, 0, 0, 0 };
			const int n = nbase + 8 * q;
			if ((p.N & 3) == 0 && (reinterpret_cast<uintptr_t>(p.bias) & 15) == 0) {
				if (p.wsum != nullptr) ct[u][q] = *reinterpret_cast<const v4i*>(p.wsum + min(n, p.N - 4));
				if (p.bias != nullptr) bt[u][q] = *reinterpret_cast<const v4i*>(p.bias + min(n, p.N - 4));
			} else {
#pragma unroll
				for (int e = 0; e < 4; e++) {
					const int col = min(n + e, p.N - 1);
					if (p.wsum != nullptr) ct[u][q][e] = p.wsum[col];
					if (p.bias != nullptr) bt[u][q][e] = p.bias[col];
				}
			}
		}
	}
	v4i fw0[FN], fx0[FM], fw1[FN], fx1[FM];
#pragma unroll
	for (int st = 0; st < S; st++)
		if (st < n_steps) issue(st, st);
	if (n_steps > 0) {
		wait_steps(min(S, n_steps) - 1);
		pad(0, 0);
		read(fw0, fx0, 0, 0);
	}
	int stage = 0;
	for (int t = 0; t < n_steps; t++) {
		const int next = stage + 1 == S ? 0 : stage + 1;
#pragma unroll
		for (int s = 0; s + 1 < NS; s++) {
			if (s & 1) { read(fw0, fx0, stage, s + 1); multiply(fw1, fx1); }
			else { read(fw1, fx1, stage, s + 1); multiply(fw0, fx0); }
		}
		// the last slice is on its way into the second register set; once it is there the stage can be filled again
		if (t + S < n_steps) {
			asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
			issue(stage, t + S);
		}
		if (t + 1 < n_steps) {
			wait_steps(min(S - 1, n_steps - 2 - t));
			pad(next, t + 1);
			read(fw0, fx0, next, 0);
		}
		multiply(fw1, fx1);
		stage = next;
	}

	// ---- the partial tiles meet: block b of wavefront w in register order at [w][b][quad of registers][lane]
	if (ROWSUM) {
#pragma unroll
		for (int j = 0; j < FM; j++) {
			const int mine = (int)(rsum[j][0] + rsum[j][1]);
			const int both = mine + __shfl_xor(mine, 32, 64);
			if (lgrp == 0) row_sums[wave * BM + j * 32 + lrow] = both;
		}
	}
	__syncthreads();  // every wavefront has left its ring
#pragma unroll
	for (int i = 0; i < FN; i++)
#pragma unroll
		for (int j = 0; j < FM; j++)
#pragma unroll
			for (int q = 0; q < 4; q++)
				*reinterpret_cast<v4i*>(smem + (((wave * NB + i * FM + j) * 4 + q) * 64 + lane) * 16) =
				    v4i{ acc[i][j][q * 4], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3] };
	__syncthreads();
#pragma unroll
	for (int u = 0; u < MINE; u++) {
		const int b = wave + u * NW;
		if (b >= NB) break;
		const int i = b / FM, j = b % FM;
		const int m = m0 + j * 32 + lrow, nbase = n0 + i * 32 + lgrp * 4;
		int rt = p.konst;
		if (ROWSUM) {
			int sum = -128 * (steps * BK - p.K);  // the bytes of a partial k-step past K counted 128 each
#pragma unroll
			for (int w = 0; w < NW; w++) sum += row_sums[w * BM + j * 32 + lrow];
			rt += p.coef_a * sum;
		}
		v4i v[4];
#pragma unroll
		for (int q = 0; q < 4; q++) {
			v[q] = v4i{ rt, rt, rt, rt };
#pragma unroll
			for (int w = 0; w < NW; w++) v[q] += *reinterpret_cast<const v4i*>(smem + (((w * NB + b) * 4 + q) * 64 + lane) * 16);
#pragma unroll
			for (int e = 0; e < 4; e++) v[q][e] += ct[u][q][e] * p.coef_b + bt[u][q][e];
		}
		// The sums as such, in registers: out of the exact form's selects and shifts the compiler otherwise takes them apart element
		// by element and holds all the partial tiles while it does (244 to 256 registers, of eight wavefronts 448 spilled ones:
		// 17 x 4096 x 4096 33.4 -> 8.3 us, 100 x 2000 x 2048 32.3 -> 5.6).
#pragma unroll
		for (int q = 0; q < 4; q++) asm volatile("" : "+v"(v[q]));
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
		uint8_t* const crow = static_cast<uint8_t*>(p.C) + (int64_t)m * p.N;
		if ((p.N & 15) == 0) {
			// the lane halves hold columns 8 q + 0..3 and 8 q + 4..7; traded so that each half has 16 neighbouring columns
			const unsigned give0 = lgrp ? word[0] : word[2], give1 = lgrp ? word[1] : word[3];
			const unsigned got0 = (unsigned)__shfl_xor((int)give0, 32, 64), got1 = (unsigned)__shfl_xor((int)give1, 32, 64);
			const v4i out = lgrp ? v4i{ (int)got0, (int)word[2], (int)got1, (int)word[3] } : v4i{ (int)word[0], (int)got0, (int)word[1], (int)got1 };
			const int n = n0 + i * 32 + lgrp * 16;
			if (m < p.M && n < p.N) *reinterpret_cast<v4i*>(crow + n) = out;
		} else if (m < p.M) {
#pragma unroll
			for (int q = 0; q < 4; q++) {
				const int n = nbase + 8 * q;
				if ((p.N & 3) == 0) {
					if (n < p.N) *reinterpret_cast<unsigned*>(crow + n) = word[q];
				} else {
#pragma unroll
					for (int e = 0; e < 4; e++)
						if (n + e < p.N) crow[n + e] = (uint8_t)(word[q] >> (8 * e));
				}
			}
		}
	}
}

template <int BM, int BN, int BK, int NW, int S>
static int launch_wave(const QProblem& p, int out, const char* name)
{
	const uint64_t tiles = ceil_div(p.M, BM) * ceil_div(p.N, BN);
	if (tiles >= (1ull << 31)) return -1;
	const dim3 grid((unsigned)tiles), block(NW * 64);
	const bool rowsum = p.wsum != nullptr && p.coef_a != 0;
	char full[96];
	snprintf(full, sizeof(full), "%s%s", name, rowsum ? "+zpcol+zprow" : p.wsum != nullptr ? "+zpcol" : "");
	set_kernel_name(full);
#define LTEN_LAUNCH(OUTV)                                                                                    \
	if (rowsum) qgemm_wave_kernel<BM, BN, BK, NW, S, OUTV, true><<<grid, block, 0, stream()>>>(p);            \
	else qgemm_wave_kernel<BM, BN, BK, NW, S, OUTV, false><<<grid, block, 0, stream()>>>(p);
	if (out == Q_OUT_U8_FAST) { LTEN_LAUNCH(Q_OUT_U8_FAST) }
	else { LTEN_LAUNCH(Q_OUT_U8_EXACT) }
#undef LTEN_LAUNCH
	LTEN_HIP_LAUNCH_CHECK();
	return 0;
}

// Prepared weights (whose entry point stores bytes), both operands contiguous in K on 16-byte boundaries; the zero-point
// terms come from the kept sums.
int qgemm_wave_dispatch(const QProblem& p, int out, int variant)
{
	const bool fits = out != Q_OUT_ACC && p.b_flip == 0 && p.rterm == nullptr && p.cterm == nullptr && p.a_ks == 1 && p.b_ks == 1 && p.vec_ok && p.K % 16 == 0 && p.K >= 16 &&
	                  (uint64_t)p.M * p.K < (1ull << 32) && (uint64_t)p.N * p.K < (1ull << 32) && (reinterpret_cast<uintptr_t>(p.C) & 15) == 0 &&
	                  (reinterpret_cast<uintptr_t>(p.wsum) & 15) == 0;
	if (!fits) return -1;
	switch (variant) {
	case 61: return launch_wave<64, 64, 128, 4, 2>(p, out, "qgemm_fast_64x64x128_k4_s2_wpre");
	case 62: return launch_wave<64, 32, 128, 4, 3>(p, out, "qgemm_fast_64x32x128_k4_s3_wpre");
	case 63: return launch_wave<32, 64, 128, 4, 3>(p, out, "qgemm_fast_32x64x128_k4_s3_wpre");
	case 64: return launch_wave<32, 32, 128, 8, 2>(p, out, "qgemm_fast_32x32x128_k8_s2_wpre");
	default: return -1;
	}
}

// What each tile is expected to take (us): a start and an end, a k-step's share of the loads (a CU's vector L1 hands over
// 40-odd bytes a clock; rows that start between cache lines take two lines a piece), more so the fuller the chip is, and
// what each further round of workgroups adds.  Fitted to 240 shapes of 17 to 2048 rows, K and N of 512 to 8192, the weights in the
// last-level cache (10 % rms).
struct WaveTile {
	int variant, bm, bn;
	double start, per_k1024, lone, unaligned, round;
};
static const WaveTile WAVE_TILES[] = {
	{ 61, 64, 64, 4.2, 1.83, 0.63, 1.15, 3.05 },
	{ 62, 64, 32, 3.8, 1.25, 0.67, 1.14, 2.5 },
	{ 63, 32, 64, 3.7, 1.26, 0.61, 1.18, 2.3 },
	{ 64, 32, 32, 3.5, 0.82, 0.57, 1.09, 2.2 },
};

int qgemm_wave_choose(const QProblem& p, bool direct_takes)
{
	// below 17 rows the streaming kernel reads the weights as fast; the model is fitted to 512 <= K and at most 2048 rows
	if (p.M <= 16 || p.M > 2048 || p.K < 512) return 0;
	const double kk = p.K / 1024.0;
	double best = 1e30;
	int variant = 0;
	for (const WaveTile& t : WAVE_TILES) {
		const double tiles = (double)(ceil_div(p.M, t.bm) * ceil_div(p.N, t.bn)), rounds = (double)ceil_div((uint64_t)tiles, 256);
		const double us = t.start + t.per_k1024 * kk * (p.K % 128 ? t.unaligned : 1.0) * (t.lone * rounds + (1 - t.lone) * tiles / 256) + t.round * (rounds - 1);
		if (us < best) {
			best = us;
			variant = t.variant;
		}
	}
	// 17 to 32 rows against weights of a megabyte and more, the streaming kernel's; pairs are its time and the one here, the weights in
	// the last-level cache / out of HBM.  Up to a K of 8192 in whole cache lines and 32768 columns these tiles are ahead (32 x 2048 x
	// 512 7.7 and 4.8; 17 x 1815 x 1024 1.33 / 1.19 times, 32 x 8192 x 8192 1.24 / 1.17, 32 x 1815 x 8192 1.34 / 0.89), up to 65536
	// on 65 of 70 shapes, by 6 % in the mean (32 x 65536 x 1024: 22.6 and 19.9); not where rows of so many outputs start on any byte
	// (17 x 50257 x 768: 17.8 and 22.3), nor with more columns (17 x 131072 x 720: 31.2 and 34.4).
	// A tile walks all of a K on one CU, and rows that start between cache lines take two lines a piece: from HBM that is slower from
	// a K of about 4608 on (17 x 1000 x 4112 1.64 / 1.11 times, 32 x 1000 x 4112 1.65 / 0.96, x 5008 1.57 / 0.85, x 7504 1.49 /
	// 0.70) unless there are tiles for most CUs (32 x 6000 x 6000 1.40 / 0.98, 17 x 6000 x 9232 1.54 / 1.29).  A K above 8192 is cut
	// into chunks there: in whole lines ahead here from about a tile for every third CU on (32 x 3173 x 16384 1.34 / 1.10, 32 x 1500 x 12288 1.38 / 0.85; 17 x 50 x 25088: 10.1 and 17.0 us).
	if (p.M <= 32 && (uint64_t)p.N * p.K >= (1ull << 20)) {
		const bool columns = p.N <= 32768 || (p.N <= 65536 && p.N % 4 == 0);
		const bool length = p.K % 128 == 0 ? p.K <= 8192 || p.N >= 3000 : p.K <= 4608 || p.N >= 6000;
		return columns && length ? variant : 0;
	}
	const double tiles16 = (double)(ceil_div(p.M, 16) * ceil_div(p.N, 16));
	if (direct_takes) {
		// the one-launch kernel of qdirect.hip (287 x 960 x 1456: 6.3 -> 4.9 us; 60 x 994 x 6000 stays, 6.3 against 7.4).  Its small
		// tiles hide the way to HBM better, which shows on a long K (64 x 1000 x 7504, weights from there: 10.3 and 14.6, by the
		// estimates 0.80; 128 x 490 x 6016 8.6 and 10.4; 128 x 1000 x 6000, 0.66, 1.2 times ahead).  The pairs are from before that
		// kernel's loads took four lanes a row; since then the line holds over 50 layers (95 x 1972 x 4976 7.0 here and 10.6 there, 467 x
		// 557 x 4880 9.2 and 16.3, 1368 x 194 x 2176 7.2 and 8.4; short K: 392 x 1825 x 704 7.7 and 7.4)
		const double direct = 1.5 + 2.1e-6 * tiles16 * p.K + 0.59 * kk + 0.55 * tiles16 / 1024;
		return best < (p.K > 6000 ? 0.79 : 0.85) * direct ? variant : 0;
	}
	// the 128 x 128 tiles of qgemm_fast.hip, K split where qgemm_dispatch splits it; outputs that give the chip 256-row tiles
	// are theirs (256 x 4096 x 4096: 18.4 -> 9.9 us, 64 x 4096 x 4096: 15.2 -> 6.1, 432 x 920 x 6416: 42 -> 11;
	// 784 x 2206 x 7040 stays, 28 against 32)
	if (ceil_div(p.M, 256) * ceil_div(p.N, 128) > 160) return 0;
	const double tiles128 = (double)(ceil_div(p.M, 128) * ceil_div(p.N, 128));
	const int splits = p.K % 128 != 0 ? 1 : (tiles128 <= 64 && p.K >= 8192) ? (tiles128 <= 32 ? 4 : 2) : (tiles128 <= 32 && p.K >= 4096) ? 2 : 1;
	const double large = 5.1 + 3.42 * kk / splits * (p.K % 128 ? 1.6 : 1.0) * (1 + 0.8 * (tiles128 > 64 ? tiles128 / 256 - 0.25 : 0.0)) + (splits > 1 ? 4.0 : 0.0);
	return best < 0.9 * large ? variant : 0;
}

}  // namespace lten_hip
