// fp32 GEMM tiles of 128 x 128 on the fp16 matrix cores (fp16_pairs.h): three matrix products stand for one where the bf16 pieces
// of sgemm_fast.hip need six.
//
// Up to four launches: the range of every row of op(A) and column of op(B); their pieces, in the order in which the tiles want them in
// LDS (contiguous in k they come with the ranges); the tiles, which load them straight into LDS; and the bf16 tiles of the same size,
// for tiles that were marked as not to be multiplied so: all other workgroups of that launch end at once.
//
// What bounds it: the power limit.  A loop of nothing but matrix instructions on such pieces reaches 1180 TFLOP/s of fp16, 393 of
// products (bf16 pieces: 1883 and 314: the 11 significand bits cost 1.6 times the energy of 8), the tiles 1110 to 1200.  At 4096^3
// they take 343-370 us, ranges and pieces 43-45 (both operands contiguous in k) to 75, the last launch 2.6; together 394-412 us where
// the bf16 tiles took 575-613.
// 2-norm error against float64 on N(0,1): K = 1024 1.85e-7 -> 1.68e-7, 2048 2.72e-7 (128-wide tiles) and 7.0e-7 (256 x 256) -> 1.71e-7, 4096
// 3.96e-7 and 1.00e-6 -> 1.75e-7.  What the pieces themselves lose is 1.1e-7 of it; a product of two values is off by 2^-21 of itself at most.
#include "common.h"
#include "fp16_pairs.h"
#include "gemm_f32_core.h"
#include "lds_async.h"
#include "sgemm_common.h"

#include <algorithm>
#include <type_traits>

namespace lten_hip {

typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));  // rows need not start on 16-byte boundaries

// An operand: rows of op(A) or columns of op(B), both called rows here.
struct PackOperand {
	const float* values;
	int64_t ld, stride;
	int rows, K, batch;
	int along_k;      // a row's values lie one behind the other
	int* info;        // [batch][rows]
	uint8_t* images;
};

// The pieces: [problem][128 rows][16 of k][leading, rest][octet of k][row][8 fp16], zeros past the matrix: 8 KB for 128 rows and 16 of k.
constexpr int pair_tile = 128;
constexpr int image_rows = pair_tile, image_k = 16, image_bytes = image_rows * image_k * 4;
constexpr int fold_steps = 32;  // (even)

// The first launch: a workgroup of 16 wavefronts takes
//   16 rows that are contiguous in k, K of at most 4096: it holds them in registers, so their ranges and pieces cost one read of them;
//   16 rows contiguous in k, any K: their ranges, a wavefront a row;
//   32 rows contiguous along the row index (a line of memory): their ranges, 128 of k at a time.
// The second launch makes the pieces of what was not held.  All of it is bound by memory.  At 4096 x 4096 each: two operands
// contiguous in k 75 us in two launches, 45 in one; rows across (16 of them, 64 bytes a load) 75 and 91, so those take two.
constexpr int range_threads = 1024, held_k = 4096, rows_along = range_threads / 64, rows_across = 32;

static bool held(const PackOperand& o) { return o.along_k && o.K <= held_k; }
static uint64_t row_blocks(const PackOperand& o) { return ceil_div(o.rows, image_rows); }
static uint64_t range_blocks(const PackOperand& o)
{
	if (held(o)) return row_blocks(o) * (image_rows / rows_along) * o.batch;  // (the rows that fill the last image too)
	return o.along_k ? ceil_div((uint64_t)o.rows * o.batch, rows_along) : ceil_div(o.rows, rows_across) * o.batch;
}

// The bits of the largest magnitude among some values, and of the smallest but zero less one.
struct ValueRange {
	uint32_t largest = 0, smallest = ~0u;
	__device__ __forceinline__ void see(float v)
	{
		const uint32_t bits = __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
		largest = max(largest, bits);
		smallest = min(smallest, bits - 1u);
	}
	__device__ __forceinline__ void see(uint32_t l, uint32_t s)
	{
		largest = max(largest, l);
		smallest = min(smallest, s);
	}
	__device__ __forceinline__ void see_lane(int mask) { see((uint32_t)__shfl_xor((int)largest, mask, 64), (uint32_t)__shfl_xor((int)smallest, mask, 64)); }
};

__device__ __forceinline__ void range_along(const PackOperand& o, int block)
{
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int64_t row = (int64_t)block * rows_along + wave;
	if (row >= (int64_t)o.rows * o.batch) return;
	const int bz = (int)(row / o.rows), r = (int)(row - (int64_t)bz * o.rows);
	const float* v = o.values + bz * o.stride + (int64_t)r * o.ld;
	ValueRange range[4];
	int k = 4 * lane;
	for (; k + 3 * 256 + 3 < o.K; k += 4 * 256) {
		f4_any q[4];
#pragma unroll
		for (int u = 0; u < 4; u++) q[u] = *reinterpret_cast<const f4_any*>(v + k + u * 256);
#pragma unroll
		for (int u = 0; u < 4; u++)
#pragma unroll
			for (int e = 0; e < 4; e++) range[e].see(q[u][e]);
	}
	for (; k < o.K; k += 256)
#pragma unroll
		for (int e = 0; e < 4; e++) range[e].see(v[min(k + e, o.K - 1)]);
#pragma unroll
	for (int e = 1; e < 4; e++) range[0].see(range[e].largest, range[e].smallest);
#pragma unroll
	for (int d = 32; d > 0; d >>= 1) range[0].see_lane(d);
	if (lane == 0) o.info[row] = row_info(range[0].largest, range[0].smallest);
}

__device__ __forceinline__ void range_across(const PackOperand& o, int block, uint32_t (&seen)[2][16][rows_across])
{
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int blocks = (o.rows + rows_across - 1) / rows_across, bz = block / blocks, r0 = (block - bz * blocks) * rows_across;
	// (at least four rows; the last lanes' four rows are moved back inside and seen twice)
	const float* v = o.values + bz * o.stride + min(r0 + 4 * (lane & 7), o.rows - 4);
	constexpr int KS = range_threads / 8;
	ValueRange range[4];
	int k = wave * 8 + (lane >> 3);
	for (; k + 7 * KS < o.K; k += 8 * KS) {
		f4_any q[8];
#pragma unroll
		for (int u = 0; u < 8; u++) q[u] = *reinterpret_cast<const f4_any*>(v + (int64_t)(k + u * KS) * o.ld);
#pragma unroll
		for (int u = 0; u < 8; u++)
#pragma unroll
			for (int e = 0; e < 4; e++) range[e].see(q[u][e]);
	}
	for (; k < o.K; k += KS) {
		const f4_any q = *reinterpret_cast<const f4_any*>(v + (int64_t)k * o.ld);
#pragma unroll
		for (int e = 0; e < 4; e++) range[e].see(q[e]);
	}
#pragma unroll
	for (int e = 0; e < 4; e++) {
#pragma unroll
		for (int d = 32; d >= 8; d >>= 1) range[e].see_lane(d);
		if (lane < 8) {
			seen[0][wave][4 * lane + e] = range[e].largest;
			seen[1][wave][4 * lane + e] = range[e].smallest;
		}
	}
	__syncthreads();
	if (threadIdx.x >= rows_across) return;
	ValueRange all;
#pragma unroll
	for (int w = 0; w < 16; w++) all.see(seen[0][w][threadIdx.x], seen[1][w][threadIdx.x]);
	const int row = min(r0 + (int)(threadIdx.x & ~3u), o.rows - 4) + (int)(threadIdx.x & 3);
	o.info[(int64_t)bz * o.rows + row] = row_info(all.largest, all.smallest);
}

// lane -> (row lane / 4, octet of k lane % 4): a line of 16 rows a load, 512 of k a trip.
__device__ __forceinline__ void range_and_pieces(const PackOperand& o, int block, uint32_t (&seen)[2][16][rows_across], int (&infos)[rows_along])
{
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int RB = (o.rows + image_rows - 1) / image_rows, KB = (o.K + image_k - 1) / image_k, groups = RB * (image_rows / rows_along);
	const int bz = block / groups, r0 = (block - bz * groups) * rows_along, row = r0 + (lane >> 2);
	const float* const v = o.values + bz * o.stride + (int64_t)row * o.ld;
	constexpr int TRIPS = held_k / 512;
	float x[TRIPS][8];
#pragma unroll
	for (int j = 0; j < TRIPS; j++) {
		const int k = j * 512 + wave * 32 + (lane & 3) * 8;
		if (row < o.rows && k + 8 <= o.K) {
			const f4_any q0 = *reinterpret_cast<const f4_any*>(v + k), q1 = *reinterpret_cast<const f4_any*>(v + k + 4);
#pragma unroll
			for (int e = 0; e < 4; e++) {
				x[j][e] = q0[e];
				x[j][4 + e] = q1[e];
			}
		} else {
#pragma unroll
			for (int e = 0; e < 8; e++) x[j][e] = row < o.rows && k + e < o.K ? v[k + e] : 0.0f;
		}
	}
	ValueRange range[4];
#pragma unroll
	for (int j = 0; j < TRIPS; j++)
#pragma unroll
		for (int e = 0; e < 8; e++) range[e & 3].see(x[j][e]);
#pragma unroll
	for (int e = 1; e < 4; e++) range[0].see(range[e].largest, range[e].smallest);
	range[0].see_lane(1);
	range[0].see_lane(2);
	if ((lane & 3) == 0) {
		seen[0][wave][lane >> 2] = range[0].largest;
		seen[1][wave][lane >> 2] = range[0].smallest;
	}
	__syncthreads();
	if (threadIdx.x < rows_along) {
		ValueRange all;
#pragma unroll
		for (int w = 0; w < 16; w++) all.see(seen[0][w][threadIdx.x], seen[1][w][threadIdx.x]);
		const int info = row_info(all.largest, all.smallest);
		infos[threadIdx.x] = info;
		if (r0 + (int)threadIdx.x < o.rows) o.info[(int64_t)bz * o.rows + r0 + threadIdx.x] = info;
	}
	__syncthreads();
	const float scale = __builtin_ldexpf(1.0f, infos[lane >> 2] >> 8);
	uint8_t* const image = o.images + ((int64_t)bz * RB + r0 / image_rows) * KB * image_bytes + (r0 % image_rows + (lane >> 2)) * 16;
#pragma unroll
	for (int j = 0; j < TRIPS; j++) {
		const int k = j * 512 + wave * 32 + (lane & 3) * 8;
		if (k >= KB * image_k) continue;
		uint4 hi, lo;
		pair8(x[j], scale, hi, lo);
		uint4* to = reinterpret_cast<uint4*>(image + (int64_t)(k / image_k) * image_bytes + (k % image_k / 8) * (image_rows * 16));
		to[0] = hi;
		to[image_bytes / 2 / 16] = lo;
	}
}

__global__ __launch_bounds__(range_threads) void sgemm_pairs_range_kernel(PackOperand a, PackOperand b, int a_blocks)
{
	__shared__ uint32_t seen[2][16][rows_across];
	__shared__ int infos[rows_along];
	const bool is_a = (int)blockIdx.x < a_blocks;
	const PackOperand o = is_a ? a : b;
	const int block = is_a ? blockIdx.x : blockIdx.x - a_blocks;
	if (!o.along_k) range_across(o, block, seen);
	else if (o.K > held_k) range_along(o, block);
	else range_and_pieces(o, block, seen, infos);
}

// Contiguous in k: two lanes read 64 bytes of a row, a wavefront writes two pieces of 512 bytes twice.  Contiguous along the row index:
// the lanes of a wavefront read 64 rows of one k, and write 1 KB twice.
constexpr int pack_steps = 8;  // images that a workgroup makes one behind the other along k
static uint64_t pack_blocks(const PackOperand& o) { return held(o) ? 0 : row_blocks(o) * o.batch * ceil_div(ceil_div(o.K, image_k), pack_steps); }

__global__ __launch_bounds__(256) void sgemm_pairs_pack_kernel(PackOperand a, PackOperand b, int a_blocks)
{
	const bool is_a = (int)blockIdx.x < a_blocks;
	const PackOperand o = is_a ? a : b;
	const int block = is_a ? blockIdx.x : blockIdx.x - a_blocks;
	const int RB = (o.rows + image_rows - 1) / image_rows, KB = (o.K + image_k - 1) / image_k, KG = (KB + pack_steps - 1) / pack_steps;
	const int kg = block % KG, rb = (block / KG) % RB, bz = block / KG / RB;
	const float* v = o.values + bz * o.stride;
	const int* info = o.info + (int64_t)bz * o.rows;
	const int t = threadIdx.x;
	const int oct = o.along_k ? t & 1 : t >> 7, r = o.along_k ? t >> 1 : t & 127, row = rb * image_rows + r;
	const float scale = __builtin_ldexpf(1.0f, row < o.rows ? info[row] >> 8 : 0);
#pragma unroll 4
	for (int kb = kg * pack_steps; kb < min(KB, (kg + 1) * pack_steps); kb++) {
		const int k0 = kb * image_k + oct * 8;
		float x[8];
		if (row < o.rows && k0 + 8 <= o.K) {
			if (o.along_k) {
				const float* at = v + (int64_t)row * o.ld + k0;
				const f4_any q0 = *reinterpret_cast<const f4_any*>(at), q1 = *reinterpret_cast<const f4_any*>(at + 4);
				x[0] = q0.x; x[1] = q0.y; x[2] = q0.z; x[3] = q0.w; x[4] = q1.x; x[5] = q1.y; x[6] = q1.z; x[7] = q1.w;
			} else {
#pragma unroll
				for (int e = 0; e < 8; e++) x[e] = v[(int64_t)(k0 + e) * o.ld + row];
			}
		} else {
#pragma unroll
			for (int e = 0; e < 8; e++) {
				x[e] = 0.0f;
				if (row < o.rows && k0 + e < o.K) x[e] = o.along_k ? v[(int64_t)row * o.ld + k0 + e] : v[(int64_t)(k0 + e) * o.ld + row];
			}
		}
		uint4 hi, lo;
		pair8(x, scale, hi, lo);
		uint4* to = reinterpret_cast<uint4*>(o.images + (((int64_t)bz * RB + rb) * KB + kb) * image_bytes + oct * (image_rows * 16) + r * 16);
		to[0] = hi;
		to[image_bytes / 2 / 16] = lo;
	}
}

struct PairProblem {
	SProblem p;
	const uint8_t *a_images, *b_images;
	const int *a_info, *b_info;
	int64_t a_stride, b_stride;  // bytes of images per problem
	int64_t a_info_stride, b_info_stride;
	uint8_t* marks;  // a byte per tile: the bf16 tiles have to compute it
};

// 4 wavefronts in two rows and two columns, each FM x FN blocks of 32 x 32.  A ring of S stages of a k-step of 16 in LDS: 3 FM FN matrix
// instructions, and between them the reads of the next k-step's operands and the loads of the one S ahead.  One barrier a
// k-step: behind it the next k-step has landed and everybody holds this one's operands, whose stage is filled again.
// Two workgroups a CU: one multiplies while the other waits at its barrier (tiles of 256 x 128, one a CU with 128 x 64 a wavefront,
// read 40 % less LDS but had the matrix pipe busy 58 % of the time instead of 70 and took 388 us against 370).
__global__ __launch_bounds__(256, 2) void sgemm_pairs_kernel(PairProblem q)
{
	const SProblem& p = q.p;
	constexpr int FM = 2, FN = 2, S = 4, BM = pair_tile, BN = pair_tile, TM = BM / 2, TN = BN / 2;
	constexpr int STAGE = 2 * image_bytes;
	constexpr int LOADS = STAGE / 1024 / 4;  // per wavefront and stage
	constexpr int PLANE = image_bytes / 2, OCTET = image_rows * 16;
	__shared__ __attribute__((aligned(1024))) uint8_t smem[S * STAGE];
	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int wm = wave >> 1, wn = wave & 1, lrow = lane & 31, lk = lane >> 5;
	const int bz = blockIdx.z;

	// Workgroup -> tile, in compact blocks of tiles per XCD (as in sgemm_fast.hip)
	const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
	int tm, tn;
	{
		const int nb = tiles_m * tiles_n, bid = blockIdx.x;
		int lid = bid;
		if ((nb & 7) == 0) lid = (bid & 7) * (nb >> 3) + (bid >> 3);
		constexpr int GM = 4, GN = 8;
		if (tiles_m % GM == 0 && tiles_n % GN == 0) {
			const int group = lid / (GM * GN), within = lid % (GM * GN), groups_n = tiles_n / GN;
			tm = (group / groups_n) * GM + within / GN;
			tn = (group % groups_n) * GN + within % GN;
		} else if (tiles_m < tiles_n && (nb & 7) == 0) {
			tn = lid / tiles_m;
			tm = lid % tiles_m;
		} else {
			tm = lid / tiles_n;
			tn = lid % tiles_n;
		}
	}
	const int m0 = tm * BM, n0 = tn * BN;
	const int KT = (p.K + image_k - 1) / image_k;

	// ---- global -> LDS: the stage is the tile's images one behind the other, load i of a wavefront its kilobyte wave + 4 i
	const uint32_t smem_addr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
	const uint8_t* const image[2] = { q.a_images + bz * q.a_stride + (int64_t)tm * KT * image_bytes, q.b_images + bz * q.b_stride + (int64_t)tn * KT * image_bytes };
	const uint32_t voff = lane * 16;
	constexpr int PER_IMAGE = image_bytes / 1024 / 4;  // a wavefront's loads of an image
	auto load_one = [&](int i, uint32_t stage_at, int kt) {
		const int x = i / PER_IMAGE, part = wave + 4 * (i % PER_IMAGE);
		async_load16(smem_addr + stage_at + x * image_bytes + part * 1024, image[x] + (int64_t)kt * image_bytes + part * 1024, voff);
	};

	// ---- LDS -> MFMA operands
	const int a_off = (wm * TM + lrow) * 16 + lk * OCTET, b_off = image_bytes + (wn * TN + lrow) * 16 + lk * OCTET;
	f16x8 fa[2][FM][2], fb[2][FN][2];
	constexpr int READS = 2 * (FM + FN);
	// read r of k-step s of a stage into operand set `set`: the leading pieces and the rest of B, then of A
	auto read_one = [&](int r, int set, const uint8_t* stage) {
		const int v = r & 1, x = r >> 1;
		if (x < FN) fb[set][x][v] = *reinterpret_cast<const f16x8*>(stage + b_off + x * 512 + v * PLANE);
		else fa[set][x - FN][v] = *reinterpret_cast<const f16x8*>(stage + a_off + (x - FN) * 512 + v * PLANE);
	};

	v16f lead[FM][FN], low[FM][FN], sum[FM][FN];
#pragma unroll
	for (int i = 0; i < FM; i++)
#pragma unroll
		for (int j = 0; j < FN; j++)
#pragma unroll
			for (int r = 0; r < 16; r++) lead[i][j][r] = low[i][j][r] = sum[i][j][r] = 0.0f;

	constexpr int NM = 3 * FM * FN;
	static_assert(NM >= READS + 4 && NM > LOADS && S * LOADS < 64, "pipeline shape");
	// A k-step with operand set `set`; the next one's operands from `stage` into the other set; the loads of k-step kt into the stage at `to`.
	auto beat = [&](auto set_c, const uint8_t* stage, uint32_t to, int kt) {
		constexpr int set = decltype(set_c)::value;
#pragma unroll
		for (int n = 0; n < NM; n++) {
			const int piece = n / (FM * FN), i = n % (FM * FN) / FN, j = n % FN;
			if (piece == 0) low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[set][i][1], fb[set][j][0], low[i][j], 0, 0, 0);
			if (piece == 1) low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[set][i][0], fb[set][j][1], low[i][j], 0, 0, 0);
			if (piece == 2) lead[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[set][i][0], fb[set][j][0], lead[i][j], 0, 0, 0);
#pragma unroll
			for (int r = 0; r < READS; r++)
				if (r * (NM - 4) / READS == n) read_one(r, set ^ 1, stage);
#pragma unroll
			for (int h = 0; h < LOADS; h++)
				if (h * NM / LOADS + 1 == n) load_one(h, to, kt);
			__builtin_amdgcn_sched_barrier(0);
		}
	};

	// (past the last k-step the loads repeat it: the count of loads in flight stays the same, nothing reads them)
	for (int st = 0; st < S; st++)
#pragma unroll
		for (int i = 0; i < LOADS; i++) load_one(i, st * STAGE, min(st, KT - 1));
	wait_vmcnt<(S - 1) * LOADS>();
	__syncthreads();
#pragma unroll
	for (int r = 0; r < READS; r++) read_one(r, 0, smem);
	int at = 0;  // the stage of k-step kt
	int kt = 0;
	auto step = [&](auto set_c) {
		const int next = at + 1 == S ? 0 : at + 1;
		wait_vmcnt_lgkm0<(S - 2) * LOADS>();  // the next k-step's operands have landed, this one's are in registers
		__syncthreads();
		beat(set_c, smem + next * STAGE, at * STAGE, min(kt + S, KT - 1));
		at = next;
		kt++;
	};
	using P0 = std::integral_constant<int, 0>;
	using P1 = std::integral_constant<int, 1>;
	for (;;) {
		const int end = min(kt + fold_steps, KT);
#pragma unroll 1
		while (kt + 1 < end) {
			step(P0{});
			step(P1{});
		}
		if (kt < end) step(P0{});
		// (sums of 512 of K each lose less to rounding than one of all K, which pays for what the pieces lose)
#pragma unroll
		for (int i = 0; i < FM; i++)
#pragma unroll
			for (int j = 0; j < FN; j++)
#pragma unroll
				for (int r = 0; r < 16; r++) {
					sum[i][j][r] += lead[i][j][r];
					lead[i][j][r] = 0.0f;
				}
		if (kt == KT) break;
	}
	wait_vmcnt_lgkm0<0>();  // no load may be on its way into LDS that is used for something else now, or by another workgroup
	__syncthreads();

	// ---- what is known of the tile's rows and columns, and off with the scales
	int* const infos = reinterpret_cast<int*>(smem);
	int* const failed_any = infos + BM + BN;
	for (int x = tid; x < BM + BN; x += 256)
		infos[x] = x < BM ? q.a_info[bz * q.a_info_stride + min(m0 + x, p.M - 1)] : q.b_info[bz * q.b_info_stride + min(n0 + x - BM, p.N - 1)];
	if (tid == 0) *failed_any = 0;
	__syncthreads();
	int cinfo[FN], seen = 0;
#pragma unroll
	for (int j = 0; j < FN; j++) seen |= cinfo[j] = infos[BM + wn * TN + j * 32 + lrow];
	for (int x = lane; x < TM; x += 64) seen |= infos[wm * TM + x];
	const bool look = __any((seen & (row_small | row_not)) != 0);
	bool failed = false;
#pragma unroll
	for (int i = 0; i < FM; i++)
#pragma unroll
		for (int r = 0; r < 16; r++) {
			const int rinfo = infos[wm * TM + i * 32 + (r >> 2) * 8 + 4 * lk + (r & 3)];
#pragma unroll
			for (int j = 0; j < FN; j++) {
				const float v = sum[i][j][r] + low[i][j][r] * (1.0f / pair_step);
				if (look) {
					const int both = rinfo | cinfo[j];
					failed |= (both & row_not) != 0 || ((both & row_small) != 0 && (both & row_zero) == 0 && !(fabsf(v) >= pair_least));
				}
				sum[i][j][r] = __builtin_ldexpf(v, -(rinfo >> 8) - (cinfo[j] >> 8));
			}
		}
	if (failed) *failed_any = 1;
	__syncthreads();
	const bool mark = *failed_any != 0;
	if (tid == 0) q.marks[((int64_t)bz * tiles_m + tm) * tiles_n + tn] = mark ? 1 : 0;
	if (mark) return;

	// Epilogue: register 4 u + e of block (i, j) of lane (lrow, lk) is row i*32 + 8u + 4lk + e, column j*32 + lrow of the wavefront's tile.
	float* C = p.C + (int64_t)bz * p.stride_c;
	const int mw = m0 + wm * TM, nw = n0 + wn * TN;
	const bool relu = p.relu_in != nullptr || p.relu_out != nullptr;
	float bv[FN];
#pragma unroll
	for (int j = 0; j < FN; j++) bv[j] = p.bias && nw + j * 32 + lrow < p.N ? p.bias[nw + j * 32 + lrow] : 0.0f;
	float* cw = C + (int64_t)mw * p.ldc + nw;
	const unsigned c_lane = (unsigned)(4 * lk * p.ldc) + lrow;
	const bool whole = m0 + BM <= p.M && n0 + BN <= p.N;
#pragma unroll
	for (int i = 0; i < FM; i++)
#pragma unroll
		for (int r = 0; r < 16; r++) {
			float* cr = cw + (int64_t)(i * 32 + (r >> 2) * 8 + (r & 3)) * p.ldc;
			const int m = mw + i * 32 + (r >> 2) * 8 + 4 * lk + (r & 3);
#pragma unroll
			for (int j = 0; j < FN; j++) {
				if (!whole && (m >= p.M || nw + j * 32 + lrow >= p.N)) continue;
				float* c = &cr[c_lane + j * 32];
				float v = p.alpha * sum[i][j][r];
				if (p.beta != 0.0f) v += p.beta * *c;
				v += bv[j];
				if (relu) sgemm_store(p, c, v);
				else __builtin_nontemporal_store(v, c);  // (C is written once and not read again here)
			}
		}
}

static uint64_t align256(uint64_t n) { return (n + 255) & ~255ull; }

uint64_t sgemm_pairs_bytes(uint64_t M, uint64_t N, uint64_t K, uint64_t batch)
{
	const uint64_t tiles = ceil_div(M, pair_tile) * ceil_div(N, pair_tile);
	return batch * (ceil_div(M, image_rows) + ceil_div(N, image_rows)) * ceil_div(K, image_k) * image_bytes + align256(4 * M * batch) + align256(4 * N * batch) +
	       align256(tiles * batch);
}

// What the four launches take, in us (as for the tiles of sgemm_fast.hip: a start, a tile's edge, a k-step of 16 of a CU's tiles, the clock
// that comes back when part of the chip is idle; and the operands' way through the first two launches).  Fitted to 47 products of 256 to
// 6000 rows and columns and a K of 1024 to 6000; off by 4 % in the mean.
double sgemm_pairs_estimate(int tA, int tB, uint64_t M, uint64_t N, uint64_t K, uint64_t batch)
{
	const double tiles = (double)(ceil_div(M, pair_tile) * ceil_div(N, pair_tile) * batch), rounds = std::ceil(tiles / 256.0), steps = (double)ceil_div(K, image_k);
	const double per_step = tiles <= 256.0 ? 0.324 * (0.61 + 0.39 * tiles / 256.0) : std::max(0.324, 0.31 * rounds);
	auto value = [&](bool along_k) { return along_k && K <= (uint64_t)held_k ? 0.9e-6 : 1.6e-6; };
	return 19.5 + 3.5 * rounds + steps * per_step + (value(!tA) * (double)M + value(tB) * (double)N) * (double)K * (double)batch;
}

int sgemm_pairs_dispatch(const SProblem& p, int tA, int tB, uint64_t batch, void* scratch)
{
	if (scratch == nullptr || p.M < 4 || p.N < 4 || p.K < 1 || p.k_total != 0 || p.col_group != 0 || !sgemm_fast_takes(p, tA, tB, 21)) return -1;
	char* at = static_cast<char*>(scratch);
	auto take = [&](uint64_t bytes) {
		char* here = at;
		at += align256(bytes);
		return here;
	};
	const int64_t KB = (int64_t)ceil_div(p.K, image_k);
	PackOperand a = { p.A, p.lda, p.stride_a, p.M, p.K, p.stride_a == 0 ? 1 : (int)batch, !tA, nullptr, nullptr };
	PackOperand b = { p.B, p.ldb, p.stride_b, p.N, p.K, p.stride_b == 0 ? 1 : (int)batch, tB, nullptr, nullptr };
	PairProblem q = {};
	q.p = p;
	const int64_t a_bytes = (int64_t)row_blocks(a) * KB * image_bytes, b_bytes = (int64_t)row_blocks(b) * KB * image_bytes;
	q.a_images = a.images = reinterpret_cast<uint8_t*>(take(a_bytes * a.batch));
	q.b_images = b.images = reinterpret_cast<uint8_t*>(take(b_bytes * b.batch));
	q.a_info = a.info = reinterpret_cast<int*>(take(4ull * p.M * a.batch));
	q.b_info = b.info = reinterpret_cast<int*>(take(4ull * p.N * b.batch));
	q.a_stride = a.batch > 1 ? a_bytes : 0;
	q.b_stride = b.batch > 1 ? b_bytes : 0;
	q.a_info_stride = a.batch > 1 ? p.M : 0;
	q.b_info_stride = b.batch > 1 ? p.N : 0;
	q.marks = reinterpret_cast<uint8_t*>(at);

	const uint64_t a_range = range_blocks(a), b_range = range_blocks(b), a_pack = pack_blocks(a), b_pack = pack_blocks(b);
	const uint64_t tiles = ceil_div(p.M, pair_tile) * ceil_div(p.N, pair_tile);
	if (a_range + b_range >= (1ull << 31) || a_pack + b_pack >= (1ull << 31) || tiles >= (1ull << 31)) return -1;
	sgemm_pairs_range_kernel<<<dim3((unsigned)(a_range + b_range)), dim3(range_threads), 0, stream()>>>(a, b, (int)a_range);
	LTEN_HIP_LAUNCH_CHECK();
	if (a_pack + b_pack != 0) {
		sgemm_pairs_pack_kernel<<<dim3((unsigned)(a_pack + b_pack)), dim3(256), 0, stream()>>>(a, b, (int)a_pack);
		LTEN_HIP_LAUNCH_CHECK();
	}
	sgemm_pairs_kernel<<<dim3((unsigned)tiles, 1, (unsigned)batch), dim3(256), 0, stream()>>>(q);
	LTEN_HIP_LAUNCH_CHECK();
	SProblem left = p;
	left.marks = q.marks;
	const int rc = sgemm_fast_dispatch(left, tA, tB, batch, 21);
	set_kernel_name("sgemm_fast_128x128_pairs");
	return rc;
}

}  // namespace lten_hip
