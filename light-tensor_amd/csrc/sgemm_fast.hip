// fp32 GEMM tiles on the bf16 matrix cores, in all four layouts, any size and any alignment of fp32 values.
//
// A bf16 matrix instruction does 16 times the work of an fp32 one in the same clocks.  So every operand value is taken
// apart into three bf16 pieces and a product is the sum of six piece products (bf16_pieces.h).  All tiles but the largest
// keep the leading products apart from the five corrections, so that a sum rounds once a k-step at its own last bit.
// 2-norm error against float64, the fp32 instructions' kernels -> here, 2048 x 2048 x K NT:
//   N(0,1)          K = 2 3.1e-8 -> 2.6e-8, 48 7.3e-8 -> 4.5e-8, 256 2.9e-7 -> 8.9e-8, 4096 1.14e-6 -> 2.7e-7
//   uniform (0, 1)  K = 2 2.9e-8 -> 2.6e-8, 48 4.6e-8 -> 4.1e-8, 256 2.2e-7 -> 8.4e-8, 4096 8.4e-7 -> 1.6e-7
// and over 95 products of ordinary sizes 0.37 of it in the mean, none larger on N(0,1); on uniform values up to 1.45 times (TN at
// K = 197: 7e-8) where eight wavefronts had shared K.  A single output of two products can be off by 1.5e-7 of their
// magnitudes where it was 1.2e-7 (the three piece products left away).  The 256 x 256 tile, whose registers are all taken
// (K >= 256 only): 1.01e-6 and 6.2e-7 at K = 4096, against 1.14e-6 and 9.9e-7.
// What has no such pieces or sums (infinities, NaN, values from 2^103 on, sums that reach 2^80) is computed again with the
// fp32 instructions at the end of the tile.
//
// Rate (4096^3, whichever layout): 545-590 us = 233-252 TFLOP/s where the fp32 instructions took 910-920 us (150); one
// tile per CU at the full clock has the matrix pipe busy 88 % of the time (256 x 4096 x 4096: 375 us), the whole chip is
// held back by its power limit (an MFMA-only loop on such pieces: 1850 TFLOP/s of bf16, 308 of products; here 1500).
//
// Tile: BM x BN, WM x WN wavefronts, k-steps of 16.  A thread loads fp32 values (16 bytes of a row that is contiguous in
// k, or GA (GB) values of four rows of k), converts them (5.5 vector instructions a value, once per workgroup) and writes the
// pieces to the LDS stage of the next k-step while the matrix instructions of this one run.
#include "bf16_pieces.h"
#include "common.h"
#include "gemm_f32_core.h"
#include "lds_async.h"
#include "sgemm_common.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace lten_hip {

typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));  // rows need not start on 16-byte boundaries
typedef float f2_any __attribute__((ext_vector_type(2), aligned(4)));

// WK groups of WM x WN wavefronts share a tile: group g takes every WK-th k-step in two LDS stages of its own, and the
// groups' sums are added at the end.
template <int BM, int BN, int WM, int WN, int WK, bool A_KC, bool B_KC>
__global__ __launch_bounds__(WM* WN* WK * 64, 2) void sgemm_fast_kernel(SProblem p)
{
	constexpr int NT = WM * WN * 64, BK = 16;
	constexpr int GA = BM * BK / NT / 4, GB = BN * BK / NT / 4, G = GA + GB;  // groups of four k of one row, per thread
	constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32;
	// LDS: [stage][operand][piece][octet of k][row][8 bf16].  Operands contiguous in k: the octets are set apart so that the
	// 8-byte writes of 16 lanes (four rows x four k groups) fall on different banks.  Contiguous along the row index, two
	// rows per thread: a block of 64 rows holds its even rows first, then the odd ones, so that the writes of 16 lanes are
	// 16 bytes apart; a 32-row operand block of the matrix instruction is then every other row of 64 (row_of, col_of).
	constexpr int OA = BM * 16 + (A_KC ? 64 : 0), OB = BN * 16 + (B_KC ? 64 : 0);
	constexpr bool A_PAIRS = !A_KC && GA == 2, B_PAIRS = !B_KC && GB == 2;
	constexpr int STAGE_A = 6 * OA, STAGE = STAGE_A + 6 * OB;
	static_assert((GA == 1 || GA == 2) && (GB == 1 || GB == 2), "a thread stages one or two groups of an operand");
	static_assert((!A_PAIRS || TM % 64 == 0) && (!B_PAIRS || TN % 64 == 0), "a wavefront's rows are whole blocks of 64");
	static_assert(WK == 1 || (WK - 1) * BM * BN * 4 <= 2 * WK * STAGE, "the groups' sums fit the stages");
	__shared__ __attribute__((aligned(1024))) uint8_t smem_all[2 * WK * STAGE];

	const int tid = threadIdx.x & (NT - 1), lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int grp = WK == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
	uint8_t* const smem = smem_all + grp * 2 * STAGE;
	const int wm = wave / WN, wn = wave % WN;
	const int lrow = lane & 31, lk = lane >> 5;

	// Workgroup -> tile.  Consecutive workgroup ids go round-robin to the 8 XCDs, each with its own L2; every
	// XCD gets compact 4 x 8 blocks of tiles so that its CUs stream the same rows of A and B.
	// A batch of small problems (problems_by_xcd): XCD x takes problems x, x + 8, ... whole, so that a problem's operands
	// cross one L2 only (the workgroups of the grid go round-robin to the XCDs in the order z * gridDim.x + x).
	const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
	int tm, tn, bz = blockIdx.z;
	{
		const int nb = tiles_m * tiles_n, bid = blockIdx.x;
		int lid = bid;
		if (p.problems_by_xcd) {
			const unsigned linear = blockIdx.z * (unsigned)nb + bid, j = linear >> 3;
			const unsigned prob = j / (unsigned)nb;  // (the division runs on the vector ALU: back to scalar registers)
			bz = __builtin_amdgcn_readfirstlane((int)prob * 8 + (int)(linear & 7));
			lid = __builtin_amdgcn_readfirstlane((int)(j - prob * (unsigned)nb));
		} else if ((nb & 7) == 0) lid = (bid & 7) * (nb >> 3) + (bid >> 3);
		constexpr int GM = 4, GN = 8;
		if (tiles_m % GM == 0 && tiles_n % GN == 0) {
			const int group = lid / (GM * GN), within = lid % (GM * GN), groups_n = tiles_n / GN;
			tm = (group / groups_n) * GM + within / GN;
			tn = (group % groups_n) * GN + within % GN;
		} else if (tiles_m < tiles_n && (nb & 7) == 0 && !p.problems_by_xcd) {
			// a wide product (few rows of tiles; tiles in a multiple of 8, so an XCD has a run of them): the run walks down the
			// columns of tiles, so that the XCD reads a narrow range of B and all of the smaller A (256 x 6272 x 2304, 4 x 98
			// tiles: B crossed the L2s 3.4 times with the run along a row of tiles)
			tn = lid / tiles_m;
			tm = lid % tiles_m;
		} else {
			tm = lid / tiles_n;
			tn = lid % tiles_n;
		}
	}
	// The last tile of a row or column of tiles is moved back inside the matrix where that has a whole tile's rows: nothing
	// is read past an edge, and what the tile before already stores is not stored again (m_first, n_first).
	const int m_first = tm * BM, n_first = tn * BN;
	const int m0 = p.M >= BM ? min(m_first, p.M - BM) : 0, n0 = p.N >= BN ? min(n_first, p.N - BN) : 0;
	const float* A = p.A + (int64_t)bz * p.stride_a + (A_KC ? (int64_t)m0 * p.lda : m0);
	const float* B = p.B + (int64_t)bz * p.stride_b + (B_KC ? (int64_t)n0 * p.ldb : n0);
	float* C = p.C + (int64_t)bz * p.stride_c;
	// (slices of one long reduction: the last may be shorter)
	const int K = p.k_total != 0 ? min(p.K, p.k_total - bz * p.K) : p.K;

	// ---- global -> registers.  Contiguous in k: thread -> (row tid / 4 (+ NT / 4), four k from 4 (tid % 4)), one 16-byte
	// load per group.  Contiguous along the row index: 16 neighbouring lanes -> 16 GA rows, lane / 16 -> four k, four loads of
	// GA floats (with the four k on neighbouring lanes the loads took four times as long: 128 x 128 tiles, 4096^3 TN, 905 us
	// against 715).
	const int qa = A_KC ? tid & 3 : lane >> 4, qb = B_KC ? tid & 3 : lane >> 4;
	const int srow = (tid >> 6) * 16 + (lane & 15);
	uint32_t va[GA], vb[GB];
	int ma = 0, mb = 0;
	if (A_KC) {
#pragma unroll
		for (int g = 0; g < GA; g++) va[g] = ((uint32_t)min((tid >> 2) + g * (NT / 4), p.M - 1 - m0) * (uint32_t)p.lda + 4 * qa) * 4;
	} else {
		ma = min(srow * GA, p.M - GA - m0);
		va[0] = ((uint32_t)(4 * qa) * (uint32_t)p.lda + ma) * 4;
	}
	if (B_KC) {
#pragma unroll
		for (int g = 0; g < GB; g++) vb[g] = ((uint32_t)min((tid >> 2) + g * (NT / 4), p.N - 1 - n0) * (uint32_t)p.ldb + 4 * qb) * 4;
	} else {
		mb = min(srow * GB, p.N - GB - n0);
		vb[0] = ((uint32_t)(4 * qb) * (uint32_t)p.ldb + mb) * 4;
	}
	constexpr int SETS = BM * BN < 256 * 256 ? 2 : 1;  // k-steps in flight behind the one being converted
	float ra[SETS][GA][4], rb[SETS][GB][4];
	auto load_a = [&](int set, int kt) {
		if (A_KC) {
			const char* base = reinterpret_cast<const char*>(A + kt * BK);
#pragma unroll
			for (int g = 0; g < GA; g++) {
				const f4_any v = *reinterpret_cast<const f4_any*>(base + va[g]);
				ra[set][g][0] = v.x; ra[set][g][1] = v.y; ra[set][g][2] = v.z; ra[set][g][3] = v.w;
			}
		} else {
			const float* base = A + (int64_t)kt * BK * p.lda;
#pragma unroll
			for (int t = 0; t < 4; t++) {
				const char* row = reinterpret_cast<const char*>(base + t * p.lda) + va[0];
				if (GA == 2) {
					const f2_any v = *reinterpret_cast<const f2_any*>(row);
					ra[set][0][t] = v.x; ra[set][GA - 1][t] = v.y;
				} else ra[set][0][t] = *reinterpret_cast<const float*>(row);
			}
		}
	};
	auto load_b = [&](int set, int kt) {
		if (B_KC) {
			const char* base = reinterpret_cast<const char*>(B + kt * BK);
#pragma unroll
			for (int g = 0; g < GB; g++) {
				const f4_any v = *reinterpret_cast<const f4_any*>(base + vb[g]);
				rb[set][g][0] = v.x; rb[set][g][1] = v.y; rb[set][g][2] = v.z; rb[set][g][3] = v.w;
			}
		} else {
			const float* base = B + (int64_t)kt * BK * p.ldb;
#pragma unroll
			for (int t = 0; t < 4; t++) {
				const char* row = reinterpret_cast<const char*>(base + t * p.ldb) + vb[0];
				if (GB == 2) {
					const f2_any v = *reinterpret_cast<const f2_any*>(row);
					rb[set][0][t] = v.x; rb[set][GB - 1][t] = v.y;
				} else rb[set][0][t] = *reinterpret_cast<const float*>(row);
			}
		}
	};
	// a partial k-step from k0 on: value by value, zeros past K
	auto load_guarded = [&](int k0) {
#pragma unroll
		for (int t = 0; t < 4; t++) {
			const int ka = k0 + 4 * qa + t, kca = min(ka, K - 1), kb = k0 + 4 * qb + t, kcb = min(kb, K - 1);
#pragma unroll
			for (int g = 0; g < GA; g++) {
				const float v = A_KC ? A[(int64_t)min((tid >> 2) + g * (NT / 4), p.M - 1 - m0) * p.lda + kca] : A[(int64_t)kca * p.lda + ma + g];
				ra[0][g][t] = ka < K ? v : 0.0f;
			}
#pragma unroll
			for (int g = 0; g < GB; g++) {
				const float v = B_KC ? B[(int64_t)min((tid >> 2) + g * (NT / 4), p.N - 1 - n0) * p.ldb + kcb] : B[(int64_t)kcb * p.ldb + mb + g];
				rb[0][g][t] = kb < K ? v : 0.0f;
			}
		}
	};

	// ---- registers -> LDS, a quarter of a group at a time: beat 0 the leading pieces, 1 the middle ones, 2 the last, 3 the writes.
	const int pair_pos = ((tid >> 7) << 6) + (tid >> 6 & 1) * 16 + (lane & 15);  // of the even row
	const int wa = (qa >> 1) * OA + (A_KC ? tid >> 2 : A_PAIRS ? pair_pos : srow) * 16 + (qa & 1) * 8;
	const int wb = STAGE_A + (qb >> 1) * OB + (B_KC ? tid >> 2 : B_PAIRS ? pair_pos : srow) * 16 + (qb & 1) * 8;
	uint2 ph, pm, pl;
	auto stage_part = [&](int part, int set, uint8_t* sbase) {
		const int g = part >> 2, beat = part & 3;
		const bool is_a = g < GA;
		float (&r)[4] = is_a ? ra[set][is_a ? g : 0] : rb[set][is_a ? 0 : g - GA];
		if (beat == 0) {
#pragma unroll
			for (int e = 0; e < 4; e++) r[e] *= pieces_scale;
			ph.x = split_off(r[0], r[1]);
			ph.y = split_off(r[2], r[3]);
		}
		if (beat == 1) { pm.x = split_off(r[0], r[1]); pm.y = split_off(r[2], r[3]); }
		if (beat == 2) {
			pl.x = split_last(r[0], r[1]);
			pl.y = split_last(r[2], r[3]);
		}
		if (beat == 3) {
			const int gg = is_a ? g : g - GA, step = (is_a ? A_KC : B_KC) ? NT / 4 * 16 : 512, plane = 2 * (is_a ? OA : OB);
			uint8_t* d = sbase + (is_a ? wa : wb) + gg * step;
			*reinterpret_cast<uint2*>(d) = ph;
			*reinterpret_cast<uint2*>(d + plane) = pm;
			*reinterpret_cast<uint2*>(d + 2 * plane) = pl;
		}
	};

	// ---- LDS -> MFMA operands: piece v of block i
	const int fa_off = lk * OA + (wm * TM + lrow) * 16, fb_off = STAGE_A + lk * OB + (wn * TN + lrow) * 16;
	auto frag_a = [&](const uint8_t* sbase, int i, int v) { return *reinterpret_cast<const bf16x8*>(sbase + fa_off + i * 512 + v * 2 * OA); };
	auto frag_b = [&](const uint8_t* sbase, int j, int v) { return *reinterpret_cast<const bf16x8*>(sbase + fb_off + j * 512 + v * 2 * OB); };

	// The products of the leading pieces in sums of their own where the registers allow it, so that those round once a k-step
	// at the last bit of the sum instead of six times.
	constexpr bool APART = FM * FN <= 4;
	v16f acc[FM][FN], low[APART ? FM : 1][APART ? FN : 1];
#pragma unroll
	for (int i = 0; i < FM; i++)
#pragma unroll
		for (int j = 0; j < FN; j++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc[i][j][r] = low[APART ? i : 0][APART ? j : 0][r] = 0.0f;

	// K = KF whole k-steps and perhaps a partial one, which comes first (behind steps of zeros that make the count a multiple
	// of the groups); past the last step the loads repeat it.
	const int KF = K / BK, rest = K % BK != 0 ? 1 : 0, steps = (KF + rest + WK - 1) / WK, first = grp - (steps * WK - KF);
	auto whole = [&](int s) { return min(s * WK + first, KF - 1); };
	bf16x8 fa[2][FM][3], fb[2][3];

	// One k-step (operand set PAR = its parity).  The matrix instructions of column block j, six piece products (the smallest
	// first) for each row block, and between them: the operands of the next column block; ahead of the barrier the
	// conversion of the next k-step into the other stage and the loads of a later one; behind it, under the last column
	// block, the first operands of the next k-step.
	constexpr int SLOTS = 6 * FM, BEFORE = FN > 1 ? SLOTS * (FN - 1) : SLOTS;
	auto k_step = [&](auto par_c, auto more_c, int next_load) {
		constexpr int PAR = decltype(par_c)::value, SET = SETS == 2 ? PAR ^ 1 : 0;
		constexpr bool MORE = decltype(more_c)::value;  // there is a next k-step
		const uint8_t* sbase = smem + PAR * STAGE;
		uint8_t* other = smem + (PAR ^ 1) * STAGE;
#pragma unroll
		for (int j = 0; j < FN; j++) {
			const bool last = j == FN - 1;
			const int bc = FN == 1 ? PAR : (j & 1);
			if (last && FN > 1 && MORE) {
				wait_vmcnt_lgkm0<63>();
				__syncthreads();
			}
#pragma unroll
			for (int s = 0; s < SLOTS; s++) {
				const int qq = s / FM, i = s % FM, n = j * SLOTS + s;
				v16f& sum = APART && qq < 5 ? low[APART ? i : 0][APART ? j : 0] : acc[i][j];
				sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[PAR][i][piece_a[qq]], fb[bc][piece_b[qq]], sum, 0, 0, 0);
				if (!last && s < 3) fb[(j + 1) & 1][s] = frag_b(sbase, j + 1, s);
				if (last && FN > 1 && MORE) {
#pragma unroll
					for (int e = s; e < 3 * FM + 3; e += SLOTS) {
						if (e < 3) fb[0][e] = frag_b(other, 0, e);
						else fa[PAR ^ 1][(e - 3) / 3][(e - 3) % 3] = frag_a(other, (e - 3) / 3, (e - 3) % 3);
					}
				}
				if (MORE && n < BEFORE) {
#pragma unroll
					for (int part = 0; part < 4 * G; part++)
						if (part * BEFORE / (4 * G) == n) {
							stage_part(part, SET, other);
							if (part == 4 * GA - 1) load_a(SET, next_load);
							if (part == 4 * G - 1) load_b(SET, next_load);
						}
				}
				__builtin_amdgcn_sched_barrier(0);
			}
		}
		if (FN == 1 && MORE) {
			wait_vmcnt_lgkm0<63>();
			__syncthreads();
#pragma unroll
			for (int v = 0; v < 3; v++) {
				fb[PAR ^ 1][v] = frag_b(other, 0, v);
#pragma unroll
				for (int i = 0; i < FM; i++) fa[PAR ^ 1][i][v] = frag_a(other, i, v);
			}
		}
	};
	using P0 = std::integral_constant<int, 0>;
	using P1 = std::integral_constant<int, 1>;

	if (first >= 0) { load_a(0, first); load_b(0, first); }
	else load_guarded(first == -1 && rest ? KF * BK : K);
#pragma unroll
	for (int part = 0; part < 4 * G; part++) stage_part(part, 0, smem);
	if (KF > 0) {
#pragma unroll
		for (int d = 1; d <= SETS; d++) {
			load_a(d & (SETS - 1), whole(d));
			load_b(d & (SETS - 1), whole(d));
		}
	}
	__syncthreads();
#pragma unroll
	for (int v = 0; v < 3; v++) {
		fb[0][v] = frag_b(smem, 0, v);
#pragma unroll
		for (int i = 0; i < FM; i++) fa[0][i][v] = frag_a(smem, i, v);
	}
	for (int s = 0; s + 1 < steps; s += 2) {
		k_step(P0{}, std::true_type{}, whole(s + 1 + SETS));
		k_step(P1{}, std::true_type{}, whole(s + 2 + SETS));
	}
	if (steps & 1) k_step(P0{}, std::false_type{}, 0);

	if (APART) {
#pragma unroll
		for (int i = 0; i < FM; i++)
#pragma unroll
			for (int j = 0; j < FN; j++)
#pragma unroll
				for (int r = 0; r < 16; r++) acc[i][j][r] += low[APART ? i : 0][APART ? j : 0][r];
	}
	if (WK > 1) {
		__syncthreads();  // (the sums go over the stages)
		float4* const sums = reinterpret_cast<float4*>(smem_all);
		if (grp != 0) {
#pragma unroll
			for (int i = 0; i < FM; i++)
#pragma unroll
				for (int j = 0; j < FN; j++)
#pragma unroll
					for (int e = 0; e < 4; e++)
						sums[((((grp - 1) * WM * WN + wave) * FM + i) * FN + j) * 256 + e * 64 + lane] =
						    make_float4(acc[i][j][4 * e], acc[i][j][4 * e + 1], acc[i][j][4 * e + 2], acc[i][j][4 * e + 3]);
		}
		__syncthreads();
		if (grp != 0) return;
#pragma unroll
		for (int g = 0; g < WK - 1; g++)
#pragma unroll
			for (int i = 0; i < FM; i++)
#pragma unroll
				for (int j = 0; j < FN; j++)
#pragma unroll
					for (int e = 0; e < 4; e++) {
						const float4 v = sums[(((g * WM * WN + wave) * FM + i) * FN + j) * 256 + e * 64 + lane];
						acc[i][j][4 * e] += v.x; acc[i][j][4 * e + 1] += v.y; acc[i][j][4 * e + 2] += v.z; acc[i][j][4 * e + 3] += v.w;
					}
	}

	// the row (column) of the wavefront's tile that row x of block i (column x of block j) stands for
	auto row_of = [&](int i, int x) { return A_PAIRS ? (i >> 1) * 64 + (i & 1) + 2 * x : i * 32 + x; };
	auto col_of = [&](int j, int x) { return B_PAIRS ? (j >> 1) * 64 + (j & 1) + 2 * x : j * 32 + x; };
	const int mw = m0 + wm * TM, nw = n0 + wn * TN;
	// one output, whatever the epilogue has to do with it
	auto put = [&](int m, int n, float sum) {
		if (m < m_first || m >= p.M || n < n_first || n >= p.N) return;
		if (p.col_group != 0) {
			const unsigned group = (unsigned)n / (unsigned)p.col_group;
			C[(int64_t)m * p.ldc + (int64_t)group * p.col_group_stride + (n - group * (unsigned)p.col_group)] = sum + (p.row_bias ? p.row_bias[m] : 0.0f);
			return;
		}
		float* c = C + (int64_t)m * p.ldc + n;
		float v = p.alpha * sum;
		if (p.beta != 0.0f) v += p.beta * *c;
		if (p.bias) v += p.bias[n];
		sgemm_store(p, c, v);
	};

	// Operands without three pieces, sums that are too large: the wavefront's tile once more on the values themselves.
	float finite = 0.0f;
#pragma unroll
	for (int i = 0; i < FM; i++)
#pragma unroll
		for (int j = 0; j < FN; j++)
#pragma unroll
			for (int r = 0; r < 16; r++) finite = fmaf(acc[i][j][r], 0.0f, finite);
	if (__any(finite != 0.0f)) {
#pragma unroll 1
		for (int b = 0; b < FM * FN; b++) {
			const int i = b / FN, j = b % FN;
			const int m = min(mw + row_of(i, lrow), p.M - 1) - m0, n = min(nw + col_of(j, lrow), p.N - 1) - n0;
			const float* ap = A + (A_KC ? (int64_t)m * p.lda : m);
			const float* bp = B + (B_KC ? (int64_t)n * p.ldb : n);
			v16f sum;
#pragma unroll
			for (int r = 0; r < 16; r++) sum[r] = 0.0f;
#pragma unroll 1
			for (int k = 0; k < K; k += 16) {
				float a[8], bb[8];
#pragma unroll
				for (int u = 0; u < 8; u++) {
					const int kk = k + 2 * u + lk, kc = min(kk, K - 1);
					a[u] = ap[A_KC ? kc : (int64_t)kc * p.lda];
					bb[u] = bp[B_KC ? kc : (int64_t)kc * p.ldb];
					if (kk >= K) a[u] = bb[u] = 0.0f;
				}
#pragma unroll
				for (int u = 0; u < 8; u++) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u], bb[u], sum, 0, 0, 0);
			}
#pragma unroll
			for (int r = 0; r < 16; r++) put(mw + row_of(i, (r >> 2) * 8 + 4 * lk + (r & 3)), nw + col_of(j, lrow), sum[r]);
		}
		return;
	}

#pragma unroll
	for (int i = 0; i < FM; i++)
#pragma unroll
		for (int j = 0; j < FN; j++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc[i][j][r] *= pieces_unscale;

	// Epilogue: register 4q + e of block (i, j) of lane (lrow, lk) is
	//   m = m0 + wm*TM + row_of(i, 8q + 4lk + e),  n = n0 + wn*TN + col_of(j, lrow).
	if (p.relu_in != nullptr || p.relu_out != nullptr) {
#pragma unroll
		for (int i = 0; i < FM; i++)
#pragma unroll
			for (int r = 0; r < 16; r++)
#pragma unroll
				for (int j = 0; j < FN; j++) put(mw + row_of(i, (r >> 2) * 8 + 4 * lk + (r & 3)), nw + col_of(j, lrow), acc[i][j][r]);
		return;
	}
	if (p.col_group != 0) {  // grouped columns (alpha = 1, beta = 0, a bias per row): the lane's columns are placed one by one
		int64_t coff[FN];
#pragma unroll
		for (int j = 0; j < FN; j++) {
			const unsigned n = (unsigned)(nw + col_of(j, lrow)), group = n / (unsigned)p.col_group;
			coff[j] = n >= (unsigned)n_first && n < (unsigned)p.N ? (int64_t)group * p.col_group_stride + (n - group * (unsigned)p.col_group) : -1;
		}
#pragma unroll
		for (int i = 0; i < FM; i++)
#pragma unroll
			for (int r = 0; r < 16; r++) {
				const int m = mw + row_of(i, (r >> 2) * 8 + 4 * lk + (r & 3));
				if (m < m_first || m >= p.M) continue;
				float* cr = C + (int64_t)m * p.ldc;
				const float row_bias = p.row_bias ? p.row_bias[m] : 0.0f;
#pragma unroll
				for (int j = 0; j < FN; j++)
					if (coff[j] >= 0) cr[coff[j]] = acc[i][j][r] + row_bias;
			}
		return;
	}
	float bv[FN];
#pragma unroll
	for (int j = 0; j < FN; j++) {
		const int n = nw + col_of(j, lrow);
		bv[j] = (p.bias && n < p.N) ? p.bias[n] : 0.0f;
	}
	// (an address is a part the wavefront shares plus a lane offset)
	float* cw = C + (int64_t)mw * p.ldc + nw;
	const unsigned c_lane = (unsigned)(row_of(0, 4 * lk) * p.ldc) + col_of(0, lrow);
	if (m_first + BM <= p.M && n_first + BN <= p.N) {
#pragma unroll
		for (int i = 0; i < FM; i++)
#pragma unroll
			for (int r = 0; r < 16; r++) {
				float* cr = cw + (int64_t)row_of(i, (r >> 2) * 8 + (r & 3)) * p.ldc;
				float v[FN];
#pragma unroll
				for (int j = 0; j < FN; j++) {
					v[j] = p.alpha * acc[i][j][r];
					if (p.beta != 0.0f) v[j] += p.beta * cr[c_lane + col_of(j, 0)];
					v[j] += bv[j];
				}
				// (C is written once and not read again here)
#pragma unroll
				for (int j = 0; j < FN; j++) {
					if (!B_PAIRS) __builtin_nontemporal_store(v[j], &cr[c_lane + col_of(j, 0)]);
					else if (!(j & 1)) __builtin_nontemporal_store((f2_any){ v[j], v[j + (B_PAIRS ? 1 : 0)] }, reinterpret_cast<f2_any*>(&cr[c_lane + col_of(j, 0)]));
				}
			}
		return;
	}
#pragma unroll
	for (int i = 0; i < FM; i++)
#pragma unroll
		for (int r = 0; r < 16; r++) {
			const int m = mw + row_of(i, (r >> 2) * 8 + 4 * lk + (r & 3));
			if (m < m_first || m >= p.M) continue;
			float* cr = cw + (int64_t)row_of(i, (r >> 2) * 8 + (r & 3)) * p.ldc;
#pragma unroll
			for (int j = 0; j < FN; j++) {
				const int n = nw + col_of(j, lrow);
				if (n < n_first || n >= p.N) continue;
				float v = p.alpha * acc[i][j][r];
				if (p.beta != 0.0f) v += p.beta * cr[c_lane + col_of(j, 0)];
				cr[c_lane + col_of(j, 0)] = v + bv[j];
			}
		}
}

// The tiles by number, with the rows of A and columns of B that a row-contiguous operand is read in groups of, and the
// constants of the time estimate.  A launch takes, in us,
//   start + rounds * edge + steps * per step,   rounds = tiles / 256 rounded up, steps = k-steps of a group,
//   per step = max(alone, rounds * busy), and with less than one tile per CU alone * (1 - power + power * tiles / 256):
// a CU works on its tiles side by side as far as LDS allows; `alone` is what a k-step takes when there is one tile on a CU,
// `busy` a tile's share when there are several, `edge` a tile's start and store, and `power` what the clock gives back
// when part of the chip is idle.  Fitted to 400 products of 64 to 4096 rows and columns (NT, NN and TN, stacks of up to
// 256 among them); picking by it costs 1 % on average over always knowing the best tile.
// With their second set of sums the 128 x 64 and 64 x 128 tiles are slower where a CU has several (848 x 2943 x 625 NN 36.4 -> 40.1
// and 33.5 -> 38.6 us; 31.0 on 128 x 128 in two groups): their `busy` is from six products of 230 to 644 tiles since then.
struct FastTile {
	const char* name;  // its size, the groups of wavefronts over K
	int number, BM, BN, WK, m_group, n_group;
	double start, alone, busy, edge, power;
};
static const FastTile fast_tiles[] = {
	{ "sgemm_fast_256x256_g1", 12, 256, 256, 1, 2, 2, 5.58, 1.954, 2.43, 8.5, 0.301 },
	{ "sgemm_fast_256x128_g1", 13, 256, 128, 1, 2, 1, 3.06, 1.049, 1.133, 5.46, 0.229 },
	{ "sgemm_fast_128x256_g1", 14, 128, 256, 1, 1, 2, 2.48, 1.038, 1.120, 5.47, 0.227 },
	{ "sgemm_fast_128x128_g1", 21, 128, 128, 1, 2, 2, 4.02, 0.688, 0.597, 2.30, 0.150 },
	{ "sgemm_fast_128x128_g2", 24, 128, 128, 2, 2, 2, 2.84, 1.182, 1.236, 5.10, 0.269 },
	{ "sgemm_fast_64x64_g1", 31, 64, 64, 1, 1, 1, 3.30, 0.356, 0.225, 0.50, 0.106 },
	{ "sgemm_fast_64x64_g2", 32, 64, 64, 2, 1, 1, 3.33, 0.471, 0.418, 0.96, 0.206 },
	{ "sgemm_fast_64x64_g4", 33, 64, 64, 4, 1, 1, 2.00, 0.824, 0.852, 3.07, 0.319 },
	{ "sgemm_fast_128x64_g2", 34, 128, 64, 2, 2, 1, 3.50, 0.736, 0.770, 1.90, 0.207 },
	{ "sgemm_fast_64x128_g2", 35, 64, 128, 2, 1, 2, 3.78, 0.722, 0.780, 1.81, 0.210 },
};

// What does not depend on the tile: 32-bit byte offsets inside the rows of one (an operand that is contiguous along the row
// index is read 16 rows of k at a time), and no sum over the rows of op(A).
static bool fast_takes(int tA, int tB, const SProblem& p)
{
	const uint64_t a_rows = tA ? 16 : (uint64_t)std::min(p.M, 256), b_rows = tB ? (uint64_t)std::min(p.N, 256) : 16;
	return a_rows * (uint64_t)p.lda <= (1ull << 30) && b_rows * (uint64_t)p.ldb <= (1ull << 30) && 4ull * (uint64_t)p.ldc + 256 < (1ull << 31) && p.rowsum == nullptr;
}
// Reads stay inside the rows whatever the shape: a row-contiguous operand with fewer rows than the tile is read in whole groups.
static bool tile_takes(const FastTile& t, int tA, int tB, uint64_t M, uint64_t N)
{
	return (!tA || M % t.m_group == 0 || M >= (uint64_t)t.BM) && (tB || N % t.n_group == 0 || N >= (uint64_t)t.BN);
}

double sgemm_fast_estimate(int tA, int tB, uint64_t M, uint64_t N, uint64_t K, uint64_t batch, int* variant)
{
	double best = 1e30;
	// K of at most 64 into many tiles is all store: the 128 x 128 tiles write 512-byte rows and read the operands half as often
	// (4096 x 4096 x 64: 21 us against 24 on the 64 x 64 ones, 12288 x 3072 x 48: 39 against 44; level at 192 to 256 tiles)
	auto up = [](uint64_t n, int t) { return (n + (uint64_t)t - 1) >> __builtin_ctz(t); };  // (by powers of two)
	const uint64_t tiles128 = ceil_div(M, 128) * ceil_div(N, 128) * batch;
	const bool store_bound = K <= 64 && M >= 1024 && N >= 1024 && tiles128 >= 512;
	for (const FastTile& t : fast_tiles) {
		if (!tile_takes(t, tA, tB, M, N)) continue;
		if (store_bound && t.number != 21 && tile_takes(fast_tiles[3], tA, tB, M, N)) continue;
		if (t.number == 12 && K < 256) continue;  // (a short reduction is all start and store: 4096 x 4096 x 64 31 against 22 us)
		const double tiles = (double)(up(M, t.BM) * up(N, t.BN)) * (double)batch, rounds = std::ceil(tiles / 256.0);
		const double steps = (double)up(up(K, 16), t.WK);
		// (the TN form of the 128 x 64 tile: 732 x 1408 x 320 13.3 -> 15.3 us with the second set of sums, NN and NT 14.7 -> 12.8)
		const double alone = t.number == 34 && tA && !tB ? 1.2 * t.alone : t.alone;
		const double per_step = tiles <= 256.0 ? alone * (1.0 - t.power + t.power * tiles / 256.0) : std::max(alone, rounds * t.busy);
		const double us = t.start + rounds * t.edge + steps * per_step;
		if (us < best) {
			best = us;
			if (variant) *variant = t.number;
		}
	}
	return best;
}

template <int BM, int BN, int WM, int WN, int WK>
static int launch_fast(const SProblem& q, int tA, int tB, uint64_t batch)
{
	SProblem p = q;
	const uint64_t nb = ceil_div(p.M, BM) * ceil_div(p.N, BN);
	// (problems of at most 64 tiles, a whole number of them per XCD; larger ones spread over the XCDs in compact blocks)
	p.problems_by_xcd = batch >= 8 && batch % 8 == 0 && nb <= 64 && nb * batch < (1ull << 31) ? 1 : 0;
	const dim3 grid((unsigned)nb, 1, (unsigned)batch), block(WM * WN * WK * 64);
	if (!tA && !tB) sgemm_fast_kernel<BM, BN, WM, WN, WK, true, false><<<grid, block, 0, stream()>>>(p);
	if (!tA && tB) sgemm_fast_kernel<BM, BN, WM, WN, WK, true, true><<<grid, block, 0, stream()>>>(p);
	if (tA && !tB) sgemm_fast_kernel<BM, BN, WM, WN, WK, false, false><<<grid, block, 0, stream()>>>(p);
	if (tA && tB) sgemm_fast_kernel<BM, BN, WM, WN, WK, false, true><<<grid, block, 0, stream()>>>(p);
	LTEN_HIP_LAUNCH_CHECK();
	return 0;
}

int sgemm_fast_dispatch(const SProblem& p, int tA, int tB, uint64_t batch, int variant)
{
	const FastTile* tile = nullptr;
	for (const FastTile& t : fast_tiles)
		if (t.number == variant) tile = &t;
	if (tile == nullptr || !tile_takes(*tile, tA, tB, (uint64_t)p.M, (uint64_t)p.N) || p.K < 1 || !fast_takes(tA, tB, p)) return -1;
	set_kernel_name(tile->name);
	switch (variant) {
	case 12: return launch_fast<256, 256, 4, 2, 1>(p, tA, tB, batch);
	case 13: return launch_fast<256, 128, 4, 2, 1>(p, tA, tB, batch);
	case 14: return launch_fast<128, 256, 2, 4, 1>(p, tA, tB, batch);
	case 21: return launch_fast<128, 128, 2, 2, 1>(p, tA, tB, batch);
	case 24: return launch_fast<128, 128, 2, 2, 2>(p, tA, tB, batch);
	case 31: return launch_fast<64, 64, 2, 2, 1>(p, tA, tB, batch);
	case 32: return launch_fast<64, 64, 2, 2, 2>(p, tA, tB, batch);
	case 33: return launch_fast<64, 64, 2, 2, 4>(p, tA, tB, batch);
	case 34: return launch_fast<128, 64, 2, 2, 2>(p, tA, tB, batch);
	default: return launch_fast<64, 128, 2, 2, 2>(p, tA, tB, batch);
	}
}

}  // namespace lten_hip
