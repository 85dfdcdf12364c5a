// Conv2d forward and data gradient on the bf16 matrix cores: the input patch of a tile in LDS as bf16 pieces.
//
// fp32 values are taken apart into three bf16 pieces and multiplied as six piece products (bf16_pieces.h).  A tile is BM
// output channels x BN output pixels; the pixels are consecutive in (image, row, column) of one column strip of the maps, so
// tiles cross rows and images and none is padded but the last.  The reduction runs over chunks of 16 input channels, and
// inside a chunk over the taps of the window, one k-step of 16 channels each:
//   LDS holds, for one chunk, every input position the tile's windows touch (the rows with their padding), as
//   [octet of channels][piece][position][8 channels]: a matrix operand is the 16 bytes of (octet, piece) at a lane's own
//   position, and another tap is another position.  So a value is loaded and converted once per tile and used under all taps
//   (a column matrix holds it once per tap), whatever the window, the stride and the map.
//   The rows of the patch are whole quads of positions: a staging thread loads 16 bytes, four positions of a row, for four
//   channels (one position of eight channels took four times the load instructions, which cost 16 clocks each whatever their
//   width).  Position 4 q + e lies in slot e Q + q of its plane, Q = 2 modulo 8: the writes of neighbouring quads are next to each
//   other, and any eight consecutive positions, or eight that are two apart, fall on different banks.
//   The weights are packed into pieces in operand order by a small launch before, [32 channels][chunk][tap][piece][lane][8],
//   and go from the cache straight into registers, D k-steps ahead.
// Half of the eight wavefronts of a workgroup (one per SIMD) only multiply, the other half only loads, converts and fills the
// LDS stage of the next chunk while the matrix instructions of this one run; loads are a chunk further ahead.  (In one
// wavefront the loads of the patch would stand between the loads of the weights, which complete in order.)  One workgroup
// per CU walks over tiles, the chunks of the next tile staged under the last of this one.
//
// Measured (forward; fp32 matrix instructions or column matrices -> here): 32 x 32 x 128 x 128 -> 64 channels 3 x 3
// 155 -> 111 us (174 TFLOP/s), 32 x 256 x 14 x 14 -> 256 81 -> 50, 16 x 64 x 57 x 57 -> 128 at stride 2 40 -> 22, 17 x 352 x
// 50 x 50 -> 48 427 -> 90, 30 x 176 x 14 x 14 -> 320 5 x 5 205 -> 88.  One wavefront to a SIMD multiplies, so what stands
// between two of its matrix instructions is lost.  With the nine taps of a 3 x 3 window written out (not counted between k-steps),
// loads and reads each behind a matrix instruction, operands read two blocks ahead and staging by quads, 32 x 256 x 14 x 14 -> 256
// went from 60 to 50 us (its kernel from 114 to 88 thousand clocks, 42 of them in matrix instructions), 40 x 50 x 28 x 28 -> 150
// 46 -> 40, 64 x 256 x 7 x 7 -> 512 58 -> 51.
// Bound by the matrix cores (49 to 59 % of a whole launch's clocks at 32 x 32 x 128 x 128 -> 64, at about 2 GHz); then the stores at
// the end of a tile, which all CUs reach together (32 KB to 128 KB a CU: 2 to 8 us at 4.2 TB/s), and the first chunk (3 to 4.5 us).
//
// 2-norm error against float64 over 22 layers each way, the routes before -> here: 0.31 to 0.5 of it in the tiles of four or
// fewer blocks of 32 x 32, whose registers leave room for sums of their own (below), 0.8 to 0.9 in the tiles of eight; up to
// 2.2 times, 1.3e-7, where column matrices had summed the window's taps apart (8 x 16 x 68 x 89 <- 48 channels, N(0,1): 9.3e-8
// -> 1.16e-7).
//
// The data gradient is the same sum over dy with the weights transposed and flipped by their packing.  With a stride of two
// the pixels of dx fall into four classes (y mod 2, x mod 2), each a convolution of stride one with its own taps: the tiles
// of all classes are one launch.
#include "bf16_pieces.h"
#include "common.h"
#include "conv_common.h"
#include "gemm_f32_core.h"

#include <algorithm>
#include <type_traits>

namespace lten_hip {

typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));  // quads need not start on 16-byte boundaries

namespace {

constexpr int MAX_CLASSES = 4;

// One convolution of stride S = (sh, sw): output pixel (oy, ox) and tap (a, b) meet input position (oy sh - ph + a, ox sw - pw + b).
struct SplitClass {
	int kh, kw, ph, pw, Ho, Wo;
	int strip_w, strips;   // the columns of the map in strips, a tile lies in one
	int patch_q;           // quads of positions in a row of the patch
	int pixels, tiles_n;   // output pixels of a strip of the batch, their tiles
	int step;              // pixels of a tile, at most BN
	int first_tile;        // of the launch
	int out_y, out_x;      // output pixel (oy, ox) is stored at (oy out_s + out_y, ox out_s + out_x)
	int w0, wa, wb;        // tap (a, b) is weight w0 + a wa + b wb of its channels
	int64_t packed;        // where its packed weights start, in bytes
};

struct SplitConv {
	const float* x;
	const float* w;
	const float* src;   // what is staged: x, or a copy whose planes have four values
	int plane;          // of src
	const uint8_t* wp;
	const float* bias;
	float* y;
	int N, C, H, W, M;     // C input, M output channels
	int sh, sw, chunks, tiles, tiles_m;
	int out_s, out_w;      // output rows are out_w long, every out_s-th pixel is written
	int64_t out_plane;
	int w_co, w_ci;        // strides of the weights
	int classes;
	SplitClass cls[MAX_CLASSES];
};

}  // namespace

// w -> pieces in operand order, channels past the end zero: grid (chunks, blocks of 32 output channels, classes x groups of
// four taps), a tap per wavefront.
__global__ __launch_bounds__(256) void conv_split_pack_kernel(SplitConv p, uint8_t* wp)
{
	const SplitClass& c = p.cls[blockIdx.z % p.classes];
	const int lane = threadIdx.x & 63, co = blockIdx.y * 32 + (lane & 31), ci0 = blockIdx.x * 16 + (lane >> 5) * 8;
	const int taps = c.kh * c.kw, t = (int)(blockIdx.z / p.classes) * 4 + (threadIdx.x >> 6);
	if (t >= taps) return;
	uint8_t* out = wp + c.packed + (((int64_t)blockIdx.y * p.chunks + blockIdx.x) * taps + t) * 3072 + lane * 16;
	const int a = t / c.kw, b = t - a * c.kw;
	const float* src = p.w + c.w0 + a * c.wa + b * c.wb + (int64_t)min(co, p.M - 1) * p.w_co;
	float v[8];
#pragma unroll
	for (int e = 0; e < 8; e++) v[e] = src[(int64_t)min(ci0 + e, p.C - 1) * p.w_ci];
#pragma unroll
	for (int e = 0; e < 8; e++)
		if (co >= p.M || ci0 + e >= p.C) v[e] = 0.0f;
	uint4 piece[3];
	split8(v, piece);
#pragma unroll
	for (int q = 0; q < 3; q++) *reinterpret_cast<uint4*>(out + q * 1024) = piece[q];
}

// Planes of fewer than four values, a quad each (the last values repeat).
__global__ __launch_bounds__(256) void pad_planes_kernel(const float* x, float* out, int planes, int hw)
{
	const int i = blockIdx.x * 256 + threadIdx.x;
	if (i >= planes) return;
#pragma unroll
	for (int e = 0; e < 4; e++) out[4 * (int64_t)i + e] = x[(int64_t)i * hw + min(e, hw - 1)];
}

// Q: quads of positions that the patch holds (2 modulo 8, see the header).
// T3: every class has 3 x 3 taps.
template <int BM, int BN, int WM, int WN, int Q, bool T3>
__global__ __launch_bounds__(512, 2) void conv_split_kernel(SplitConv p)
{
	constexpr int PLANE = 4 * Q * 16, STAGE = 6 * PLANE, U = (Q + 63) / 64;  // U: quads of a staging thread
	constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32;
	static_assert(WM * WN == 4 && FN % 2 == 0, "four multiplying wavefronts, column blocks in pairs");
	static_assert(Q % 8 == 2, "the four groups of quads lie 32 bytes apart modulo 128");
	constexpr int D = FM * FN == 8 ? 1 : T3 || FM * FN == 4 ? 2 : 3;  // k-steps the weights are loaded ahead
	__shared__ __attribute__((aligned(1024))) uint8_t smem[2 * STAGE];

	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	// XCD x (workgroups x, x + 8, ...) has a run of tiles: neighbours in it read the same rows, or the same pixels for other channels
	const int per_xcd = (p.tiles + 7) / 8, stride = (int)(gridDim.x >> 3);
	const int tile0 = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3), tile_end = min((int)(blockIdx.x & 7) * per_xcd + per_xcd, p.tiles);
	if (tile0 >= tile_end) return;
	const int my_tiles = (tile_end - tile0 + stride - 1) / stride, items = my_tiles * p.chunks;

	// tile -> class, first output channel, strip, first pixel
	struct Place { int cls, m0, strip, p0, n0, ho0; };
	auto place_of = [&](int tile) {
		Place t;
		t.cls = 0;
		for (int c = 1; c < p.classes; c++)
			if (tile >= p.cls[c].first_tile) t.cls = c;
		const SplitClass& c = p.cls[t.cls];
		unsigned r = (unsigned)(tile - c.first_tile);
		t.m0 = (int)(r % (unsigned)p.tiles_m) * BM;
		r /= (unsigned)p.tiles_m;
		t.strip = (int)(r / (unsigned)c.tiles_n);
		t.p0 = (int)(r - (unsigned)t.strip * c.tiles_n) * c.step;
		const unsigned row = (unsigned)t.p0 / (unsigned)c.strip_w;
		t.n0 = (int)(row / (unsigned)c.Ho);
		t.ho0 = (int)row - t.n0 * c.Ho;
		return t;
	};

	if (wave >= 4) {
		// ---- the staging half: wavefront -> octet of channels; thread -> four channels of it, quads quad0 + 64 u of positions
		const int oct = wave >> 1 & 1, half = lane & 1, quad0 = (wave & 1) * 32 + (lane >> 1), ch0 = oct * 8 + half * 4;
		uint32_t off[U];           // of the item being loaded: byte offset of the quad in channel 0
		float raw[U][4][4];        // [channel][position]
		unsigned inside = 0, inside_next = 0, turn = 0, turn_next = 0;
		int quads = 0, quads_next = 0;  // of the tile's patch
		auto place_loads = [&](int tile) {
			const Place t = place_of(tile);
			const SplitClass& c = p.cls[t.cls];
			const int last = min(t.p0 + c.step, c.pixels) - 1;
			const int row_l = last / c.strip_w, n_l = row_l / c.Ho, ho_l = row_l - n_l * c.Ho;
			const int first_rows = (c.Ho - 1 - t.ho0) * p.sh + c.kh, full_rows = (c.Ho - 1) * p.sh + c.kh;
			const int rows = n_l == t.n0 ? (ho_l - t.ho0) * p.sh + c.kh : first_rows + (n_l - t.n0 - 1) * full_rows + ho_l * p.sh + c.kh;
			quads_next = rows * c.patch_q;
			inside_next = turn_next = 0;
			const int x0 = t.strip * c.strip_w * p.sw - c.pw, y0 = t.ho0 * p.sh - c.ph;
#pragma unroll
			for (int u = 0; u < U; u++) {
				const unsigned quad = (unsigned)quad0 + 64 * u;
				const unsigned r = quad / (unsigned)c.patch_q, q = quad - r * c.patch_q;
				int n = t.n0, yy = y0 + (int)r;
				if ((int)r >= first_rows) {
					const unsigned k = (r - (unsigned)first_rows) / (unsigned)full_rows;
					n += 1 + (int)k;
					yy = (int)(r - first_rows - k * full_rows) - c.ph;
				}
				const int xx = x0 + 4 * (int)q;
				unsigned in = 0;
				if ((int)quad < quads_next && (unsigned)yy < (unsigned)p.H && n < p.N) {
#pragma unroll
					for (int e = 0; e < 4; e++) in |= (unsigned)((unsigned)(xx + e) < (unsigned)p.W) << e;
				}
				// a quad that reaches past the ends of the map's plane is loaded from the plane's first or last four values and
				// turned in registers
				const int at = yy * p.W + xx, clamped = min(max(at, 0), p.plane - 4);
				off[u] = in ? ((unsigned)n * p.C * (unsigned)p.plane + (unsigned)clamped) * 4u : 0u;
				inside_next |= in << (4 * u);
				turn_next |= (in ? (unsigned)(at - clamped) & 3u : 0u) << (2 * u);
			}
		};
		// (every load is issued whatever the position: a load under a condition would make each wait one for all)
		auto load = [&](int u, int chunk) {
#pragma unroll
			for (int e = 0; e < 4; e++) {
				const char* base = reinterpret_cast<const char*>(p.src + (int64_t)min(chunk * 16 + ch0 + e, p.C - 1) * p.plane);
				const f4_any v = *reinterpret_cast<const f4_any*>(base + off[u]);
				raw[u][e][0] = v.x; raw[u][e][1] = v.y; raw[u][e][2] = v.z; raw[u][e][3] = v.w;
			}
		};
		// (channels past the end repeat the last one: their weights are zero)
		auto convert = [&](int u, int stage) {
			const int quad = quad0 + 64 * u;
			if (quad >= quads) return;
			if (__any(turn >> (2 * u) & 3u)) {
				const bool by1 = turn >> (2 * u) & 1u, by2 = turn >> (2 * u) & 2u;
#pragma unroll
				for (int e = 0; e < 4; e++) {
					float(&r)[4] = raw[u][e];
					const float a0 = by1 ? r[1] : r[0], a1 = by1 ? r[2] : r[1], a2 = by1 ? r[3] : r[2], a3 = by1 ? r[0] : r[3];
					r[0] = by2 ? a2 : a0; r[1] = by2 ? a3 : a1; r[2] = by2 ? a0 : a2; r[3] = by2 ? a1 : a3;
				}
			}
			uint8_t* d = smem + stage * STAGE + oct * 3 * PLANE + quad * 16 + half * 8;
#pragma unroll
			for (int e = 0; e < 4; e += 2) {
				const float scale0 = scale_where(inside, 4 * u + e), scale1 = scale_where(inside, 4 * u + e + 1);  // (a position outside the map counts as zeros)
				float v[8];
#pragma unroll
				for (int k = 0; k < 4; k++) {
					v[k] = raw[u][k][e] * scale0;
					v[4 + k] = raw[u][k][e + 1] * scale1;
				}
				uint4 piece[3];
				split8_scaled(v, piece);
#pragma unroll
				for (int k = 0; k < 3; k++) {
					*reinterpret_cast<uint2*>(d + k * PLANE + e * Q * 16) = make_uint2(piece[k].x, piece[k].y);
					*reinterpret_cast<uint2*>(d + k * PLANE + (e + 1) * Q * 16) = make_uint2(piece[k].z, piece[k].w);
				}
			}
		};
		int ld_tile = tile0, ld_chunk = 0;
		place_loads(tile0);
#pragma unroll
		for (int u = 0; u < U; u++) load(u, 0);
		for (int it = -1; it < items; it++) {
			// convert item it + 1, load item it + 2 (past the last one: loaded again, not converted)
			const bool have = it + 1 < items;
			quads = have ? quads_next : 0;
			inside = inside_next;
			turn = turn_next;
			if (it + 2 < items) {
				if (++ld_chunk == p.chunks) {
					ld_chunk = 0;
					ld_tile += stride;
					place_loads(ld_tile);
				}
			}
			const int stage = (it + 1) & 1;
#pragma unroll
			for (int u = 0; u < U; u++) {
				convert(u, stage);
				load(u, ld_chunk);
			}
			__syncthreads();
		}
		return;
	}

	// ---- the multiplying half
	__builtin_amdgcn_s_setprio(1);
	const int wm = wave / WN, wn = wave % WN, lrow = lane & 31, lk = lane >> 5;
	const uint32_t lane16 = lane * 16, lk3 = lk * 3 * PLANE;
	__syncthreads();  // stage 0 holds the first chunk

	int stage = 0;
	for (int tile = tile0; tile < tile_end; tile += stride) {
		const Place t = place_of(tile);
		const SplitClass& c = p.cls[t.cls];
		// (through readfirstlane: kept in registers instead of loaded again in the loop)
		const int kh = __builtin_amdgcn_readfirstlane(c.kh), kw = __builtin_amdgcn_readfirstlane(c.kw);
		const int row_step = __builtin_amdgcn_readfirstlane((4 * c.patch_q - c.kw) * 4);
		const int total = p.chunks * kh * kw;
		const int first_rows = (c.Ho - 1 - t.ho0) * p.sh + c.kh, full_rows = (c.Ho - 1) * p.sh + c.kh;
		// the lane's column of each block: four times its position in the patch, place in the output (-1: none)
		uint32_t vb[FN];
		int out[FN];
#pragma unroll
		for (int j = 0; j < FN; j++) {
			const int px = t.p0 + wn * TN + j * 32 + lrow;
			const int end = min(t.p0 + c.step, c.pixels);
			const unsigned pc = (unsigned)min(px, end - 1), row = pc / (unsigned)c.strip_w, wo = pc - row * c.strip_w;
			const unsigned n = row / (unsigned)c.Ho, ho = row - n * c.Ho;
			const int r = (int)n == t.n0 ? ((int)ho - t.ho0) * p.sh : first_rows + ((int)n - t.n0 - 1) * full_rows + (int)ho * p.sh;
			vb[j] = (uint32_t)((r * 4 * c.patch_q + (int)wo * p.sw) * 4);
			const int ox = t.strip * c.strip_w + (int)wo;
			out[j] = px < end && ox < c.Wo ? (int)(((int64_t)n * p.M + t.m0 + wm * TM) * p.out_plane) + ((int)ho * p.out_s + c.out_y) * p.out_w + ox * p.out_s + c.out_x : -1;
		}
		const uint8_t* wb[FM];
		const int64_t packed = (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)c.packed) | (uint64_t)__builtin_amdgcn_readfirstlane((int)(c.packed >> 32)) << 32);
#pragma unroll
		for (int i = 0; i < FM; i++) {
			// (blocks of 32 channels past the last one: read the last one again, never stored)
			const int block = __builtin_amdgcn_readfirstlane(min(t.m0 / 32 + wm * FM + i, (p.M + 31) / 32 - 1));
			wb[i] = p.wp + packed + (int64_t)block * total * 3072;
		}

		// register 4q + e of block (i, j) of lane (lrow, lk): channel i * 32 + 8q + 4 lk + e, column j * 32 + lrow of the
		// wavefront's.  The bias is added to the finished sum (sums that start at a large one round at its last bit in every
		// k-step); lane l has loaded channel l's by then (loaded behind the last product it cost 1 to 2 us a tile).
		const int mw = t.m0 + wm * TM;
		const float bias = p.bias ? p.bias[min(mw + (lane & (TM - 1)), p.M - 1)] : 0.0f;
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

		// Operands of column blocks are read DB blocks ahead: with one row block to a column block its six matrix instructions are
		// over before an LDS read that queues behind the staging half's writes has come back.
		constexpr int DB = FM == 1 ? 2 : 1, SETS = FM == 2 ? 2 : D == 2 ? 3 : 4;
		static_assert(!T3 || 9 % (D + 1) == 0, "a k-step's weights are the same in every chunk");
		static_assert((T3 ? 9 : D + 1) * FN % SETS == 0 && SETS > DB, "a block's operand set is the same in every round of k-steps");
		bf16x8 fa[D + 1][FM][3], fb[SETS][3];
		// (the loads run up to D k-steps past a block: into the next one, or what the buffer has behind the last one)
		uint32_t a_at = 0;
		auto load_a = [&](int set, int i, int v) { fa[set][i][v] = *reinterpret_cast<const bf16x8*>(wb[i] + (uint32_t)(lane16 + a_at) + v * 1024); };
		auto next_a = [&]() {
			a_at += 3072;
			asm volatile("" : "+s"(a_at));  // (a scalar, not a pointer of every lane)
		};
		// position 4 q + e lies in slot e Q + q of its plane; tap4: four times the tap's place in the patch, at: the stage
		auto slot_of = [&](int j, uint32_t tap4, uint32_t at) {
			const uint32_t t = vb[j] + tap4;
			uint32_t slot = __umul24(t & 12u, 4 * Q - 1) + t + at + lk3;
			asm volatile("" : "+v"(slot));  // (a multiple of 16, which its parts are not)
			return slot;
		};
		auto read_b = [&](int set, uint32_t slot, int v) { fb[set][v] = *reinterpret_cast<const bf16x8*>(smem + slot + v * PLANE); };
#pragma unroll
		for (int d = 0; d < D; d++) {
#pragma unroll
			for (int i = 0; i < FM; i++)
#pragma unroll
				for (int v = 0; v < 3; v++) load_a(d, i, v);
			next_a();
		}
		if constexpr (T3) {
			// Nine k-steps to a chunk, written out.  (With the taps counted at run time the scalar instructions between two k-steps
			// leave the pipe empty.)  Where registers are left, the addresses of a row's taps are kept.
			constexpr bool KEPT = FM * FN == 2;
			uint32_t slot3[KEPT ? FN : 1][3];
			if (KEPT) {
#pragma unroll
				for (int j = 0; j < FN; j++)
#pragma unroll
					for (int b = 0; b < 3; b++) {
						slot3[KEPT ? j : 0][b] = slot_of(j, 4 * b, 0);
						asm volatile("" : "+v"(slot3[KEPT ? j : 0][b]));
					}
			}
			const uint32_t row_bytes = 16 * (uint32_t)__builtin_amdgcn_readfirstlane(c.patch_q);
			auto opaque = [](uint32_t v) {  // (what hangs on it is worked out where it is used, not kept in registers)
				asm volatile("" : "+s"(v));
				return v;
			};
			auto slot_at = [&](int j, int tap, uint32_t at) { return KEPT ? slot3[KEPT ? j : 0][tap % 3] + (at + tap / 3 * row_bytes) : slot_of(j, opaque(4 * (tap % 3)), at + tap / 3 * row_bytes); };
			uint32_t stage_at = stage * STAGE;
#pragma unroll
			for (int b = 0; b < DB; b++)
#pragma unroll
				for (int v = 0; v < 3; v++) read_b(b, slot_at(b, 0, stage_at), v);
			auto k_step = [&](auto tap_c) {
				constexpr int TAP = decltype(tap_c)::value, NEXT = (TAP + 1) % 9, SET = TAP % (D + 1), FIRST = TAP * FN;
#pragma unroll
				for (int j = 0; j < FN; j++) {
					const bool ahead = j >= FN - DB;  // the block that is read is of the next k-step
					uint32_t slot = 0;
#pragma unroll
					for (int q = 0; q < 6 * FM; q++) {
						const int i = q % FM, qq = q / FM;
						v16f& sum = APART && qq < 5 ? low[APART ? i : 0][APART ? j : 0] : acc[i][j];
						sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[SET][i][piece_a[qq]], fb[(FIRST + j) % SETS][piece_b[qq]], sum, 0, 0, 0);
						__builtin_amdgcn_sched_barrier(0);
						if (q == 0) {
							if (TAP == 8 && j == FN - DB) {  // the next k-step is the next chunk's
								__syncthreads();
								stage_at = STAGE - stage_at;
							}
							slot = slot_at(ahead ? j + DB - FN : j + DB, ahead ? NEXT : TAP, stage_at);
						}
						if (q >= 1 && q < 4) read_b((FIRST + j + DB) % SETS, slot, q - 1);
						if (j < FM && q >= 3 && q < 6) load_a((SET + D) % (D + 1), j, q - 3);
						if (j == FN - 1 && q == 6 * FM - 2) next_a();
						__builtin_amdgcn_sched_barrier(0);
					}
				}
			};
			for (int left = p.chunks;;) {
				k_step(std::integral_constant<int, 0>{});
				k_step(std::integral_constant<int, 1>{});
				k_step(std::integral_constant<int, 2>{});
				k_step(std::integral_constant<int, 3>{});
				k_step(std::integral_constant<int, 4>{});
				k_step(std::integral_constant<int, 5>{});
				k_step(std::integral_constant<int, 6>{});
				k_step(std::integral_constant<int, 7>{});
				k_step(std::integral_constant<int, 8>{});
				if (--left == 0) break;
			}
			stage = stage_at != 0;
		} else {
#pragma unroll
			for (int b = 0; b < DB; b++)
#pragma unroll
				for (int v = 0; v < 3; v++) read_b(b, slot_of(b, 0, stage * STAGE), v);
			// The tap of this k-step and of the next one, and whether that is the next chunk's: worked out under the matrix
			// instructions of the k-step before.
			int tb = 0, ta = 0, s = 0;
			uint32_t tap4 = 0, next_tap4 = 0;
			bool chunk_end = false;
			auto advance = [&]() {
				const bool row_end = tb == kw - 1;
				chunk_end = row_end & (ta == kh - 1);
				next_tap4 = chunk_end ? 0u : tap4 + 4 + (row_end ? (uint32_t)row_step : 0u);
				ta = chunk_end ? 0 : ta + (int)row_end;
				tb = row_end ? 0 : tb + 1;
			};
			advance();
			// One k-step: the matrix instructions of every column block, the operands of a later block read under them, those of the
			// next k-step's first blocks behind a barrier where that is the next chunk's.  Everything else stands behind a matrix
			// instruction too: between two k-steps it would leave the pipe empty.
			auto k_step = [&](auto par_c) {
				constexpr int PAR = decltype(par_c)::value, FIRST = PAR * FN;
#pragma unroll
				for (int j = 0; j < FN; j++) {
					const bool ahead = j >= FN - DB;  // the block that is read is of the next k-step
					uint32_t slot = 0;
#pragma unroll
					for (int q = 0; q < 6 * FM; q++) {
						const int i = q % FM, qq = q / FM;
						v16f& sum = APART && qq < 5 ? low[APART ? i : 0][APART ? j : 0] : acc[i][j];
						sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[PAR][i][piece_a[qq]], fb[(FIRST + j) % SETS][piece_b[qq]], sum, 0, 0, 0);
						__builtin_amdgcn_sched_barrier(0);
						if (q == 0) {
							if (j == FN - DB && chunk_end) {
								__syncthreads();
								stage ^= 1;
							}
							slot = slot_of(ahead ? j + DB - FN : j + DB, ahead ? next_tap4 : tap4, stage * STAGE);
						}
						if (q >= 1 && q < 4) read_b((FIRST + j + DB) % SETS, slot, q - 1);
						if (j < FM && q >= 3 && q < 6) load_a((PAR + D) % (D + 1), j, q - 3);
						if (j == FN - 1 && q == 6 * FM - 2) {
							next_a();
							tap4 = next_tap4;
							advance();
							s++;
						}
						__builtin_amdgcn_sched_barrier(0);
					}
				}
			};
			using S0 = std::integral_constant<int, 0>;
			using S1 = std::integral_constant<int, 1>;
			using S2 = std::integral_constant<int, D >= 2 ? 2 : 0>;
			using S3 = std::integral_constant<int, D >= 3 ? 3 : 0>;
			while (s + D < total) {
				k_step(S0{});
				k_step(S1{});
				if (D >= 2) k_step(S2{});
				if (D >= 3) k_step(S3{});
			}
			if (s < total) {
				k_step(S0{});
				if (D >= 2 && s < total) {
					k_step(S1{});
					if (D >= 3 && s < total) k_step(S2{});
				}
			}
		}

		if (APART) {
#pragma unroll
			for (int i = 0; i < FM; i++)
#pragma unroll
				for (int j = 0; j < FN; j++)
#pragma unroll
					for (int r = 0; r < 16; r++) acc[i][j][r] += low[APART ? i : 0][APART ? j : 0][r];
		}

		// Values without three pieces, sums that are too large: the wavefront's tile once more on the values themselves.
		float finite[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
		for (int i = 0; i < FM; i++)
#pragma unroll
			for (int j = 0; j < FN; j++)
#pragma unroll
				for (int r = 0; r < 16; r++) finite[r & 3] = fmaf(acc[i][j][r], 0.0f, finite[r & 3]);
		if (__any((finite[0] + finite[1]) + (finite[2] + finite[3]) != 0.0f)) {
#pragma unroll 1
			for (int ij = 0; ij < FM * FN; ij++) {
				const int i = ij / FN, j = ij % FN, px = t.p0 + wn * TN + j * 32 + lrow;
				const int end = min(t.p0 + c.step, c.pixels);
				const unsigned pc = (unsigned)min(px, end - 1), row = pc / (unsigned)c.strip_w, n = row / (unsigned)c.Ho;
				const int oy = (int)(row - n * c.Ho), ox = t.strip * c.strip_w + (int)(pc - row * c.strip_w);
				const int yy = oy * p.sh - c.ph, xx = ox * p.sw - c.pw, co = t.m0 + wm * TM + i * 32;
				const float* wr = p.w + c.w0 + (int64_t)min(co + lrow, p.M - 1) * p.w_co;
				v16f sum;
#pragma unroll
				for (int r = 0; r < 16; r++) sum[r] = 0.0f;
#pragma unroll 1
				for (int ch = 0; ch < p.C; ch += 8) {  // (four loads of either operand in flight)
#pragma unroll 1
					for (int a = 0; a < c.kh; a++)
#pragma unroll 1
						for (int b = 0; b < c.kw; b++) {
							const bool at = (unsigned)(yy + a) < (unsigned)p.H && (unsigned)(xx + b) < (unsigned)p.W;
							float xv[4], wv[4];
#pragma unroll
							for (int u = 0; u < 4; u++) {
								const int cu = ch + 2 * u + lk, ci = min(cu, p.C - 1);
								xv[u] = p.x[((int64_t)n * p.C + ci) * p.H * p.W + (at ? (yy + a) * p.W + xx + b : 0)];
								wv[u] = wr[(int64_t)ci * p.w_ci + a * c.wa + b * c.wb];
								if (cu >= p.C) wv[u] = 0.0f;
								if (cu >= p.C || !at) xv[u] = 0.0f;
							}
#pragma unroll
							for (int u = 0; u < 4; u++) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[u], xv[u], sum, 0, 0, 0);
						}
				}
#pragma unroll
				for (int r = 0; r < 16; r++) {
					const int m = co + (r >> 2) * 8 + 4 * lk + (r & 3);
					if (m < p.M && px < end && ox < c.Wo)
						p.y[((int64_t)n * p.M + m) * p.out_plane + (oy * p.out_s + c.out_y) * p.out_w + ox * p.out_s + c.out_x] = sum[r] + (p.bias ? p.bias[m] : 0.0f);
				}
			}
			continue;
		}

#pragma unroll
		for (int i = 0; i < FM; i++)
#pragma unroll
			for (int r = 0; r < 16; r++) {
				const float b = p.bias ? __shfl(bias, i * 32 + (r >> 2) * 8 + 4 * lk + (r & 3)) : 0.0f;
#pragma unroll
				for (int j = 0; j < FN; j++) acc[i][j][r] = fmaf(acc[i][j][r], pieces_unscale, b);
			}
		const bool all_rows = mw + TM <= p.M;
#pragma unroll
		for (int j = 0; j < FN; j++) {
			if (out[j] < 0) continue;
			const unsigned at_lane = (unsigned)out[j] + (unsigned)(4 * lk * (int)p.out_plane);
#pragma unroll
			for (int i = 0; i < FM; i++)
#pragma unroll
				for (int r = 0; r < 16; r++) {
					const int m = i * 32 + (r >> 2) * 8 + (r & 3);
					if (all_rows || mw + m + 4 * lk < p.M) __builtin_nontemporal_store(acc[i][j][r], &p.y[m * p.out_plane + at_lane]);
				}
		}
	}
}

namespace {

// The tiles, with what a k-step of a wavefront multiplies (blocks of 32 x 32), the quads of positions a patch may have, and what
// a matrix instruction and the rest of a round of tiles take (fitted to 28 convolutions each, which it meets within 15 %).
struct SplitTile {
	int BM, BN, blocks, quads;
	double mfma_ns, round_us;
};
const SplitTile split_tiles[] = {
	{ 64, 512, 8, 210, 15.1, 16.0 }, { 32, 512, 4, 210, 15.8, 7.5 }, { 128, 256, 8, 162, 15.0, 12.0 }, { 64, 256, 4, 162, 17.9, 8.2 },
	{ 32, 256, 2, 162, 20.7, 2.7 }, { 64, 128, 2, 98, 19.2, 3.3 }, { 64, 128, 2, 210, 20.3, 3.3 },
};
constexpr int SPLIT_TILES = sizeof(split_tiles) / sizeof(split_tiles[0]);

template <int BM, int BN, int WM, int WN, int Q>
void launch_split(const SplitConv& p, bool t3)
{
	const unsigned per_xcd = (unsigned)((p.tiles + 7) / 8);
	const dim3 grid(8 * std::min(32u, per_xcd));
	constexpr bool T3 = BM / WM / 32 * (BN / WN / 32) < 8;  // (with eight blocks the registers do not hold out)
	if (T3 && t3) conv_split_kernel<BM, BN, WM, WN, Q, T3><<<grid, dim3(512), 0, stream()>>>(p);
	else conv_split_kernel<BM, BN, WM, WN, Q, false><<<grid, dim3(512), 0, stream()>>>(p);
}

// The most consecutive pixels of a strip w columns wide whose patch the tile's quads hold, at most BN (tiles start at multiples of it).
int split_step(const SplitClass& c, const SplitConv& p, const SplitTile& t, int w, int patch_q)
{
	const int budget = t.quads / patch_q, window = std::max(c.kh, p.sh), all_rows = p.N * c.Ho;
	if (budget < window) return 0;
	// rows that lie anywhere touch up to (rows - 2 + Ho) / Ho + 1 images, each with the rest of a window
	auto images = [&](int rows) { return std::min(p.N, (rows - 2 + c.Ho) / c.Ho + 1); };
	const int most = std::min(all_rows, (budget - window) / p.sh + 1);
	auto fits = [&](int rows) { return rows * p.sh + images(rows) * (window - p.sh) <= budget; };
	const int cap = std::min(most, (t.BN - 2 + w) / w + 1);
	int any = cap;
	if (!fits(any)) {
		any = std::max(1, (budget - images(any) * (window - p.sh)) / p.sh);  // (with as many images as that: then up)
		while (any < cap && fits(any + 1)) any++;
	}
	if (any == all_rows) return t.BN;
	// whole rows of the strip: those, whole images, or a divisor of an image's rows
	int whole = std::min(any, t.BN / w);
	const int per_image = (c.Ho - 1) * p.sh + window, full = std::min({ p.N, budget / per_image, t.BN / w / c.Ho });
	whole = std::max(whole, full * c.Ho);
	for (int rows = std::min({ most, t.BN / w, c.Ho }); rows > whole; rows--)
		if (c.Ho % rows == 0) whole = rows;
	if (whole == all_rows) return t.BN;
	// ((rows - 1) w + 1 pixels lie in up to `rows`)
	return std::max(whole * w, std::min(t.BN, (any - 1) * w + 1));
}

// Lays the classes out in strips and tiles of the given kind; false when a patch would not fit.
bool split_layout(SplitConv& p, const SplitTile& t)
{
	p.tiles_m = (int)ceil_div((uint64_t)p.M, (uint64_t)t.BM);
	uint64_t tiles = 0;
	for (int k = 0; k < p.classes; k++) {
		SplitClass& c = p.cls[k];
		// strips of at most 128 columns; where a patch would not fit, up to three more, and tiles of fewer pixels: of these the
		// fewest tiles
		const int first = (int)ceil_div((uint64_t)c.Wo, 128);
		int64_t pixels = 0, least = INT64_MAX;
		for (int strips = first; strips < first + 4; strips++) {
			const int strip_w = (int)ceil_div((uint64_t)c.Wo, (uint64_t)strips), patch_q = ((strip_w - 1) * p.sw + c.kw + 3) / 4;
			const int64_t strip_pixels = (int64_t)p.N * c.Ho * strip_w;
			if (strip_pixels >= (1ll << 30)) return false;
			const int step = split_step(c, p, t, strip_w, patch_q);
			if (step < t.BN / 2) continue;
			const int64_t tiles_here = (int64_t)((strip_pixels + step - 1) / step) * strips;
			if (tiles_here < least) {
				least = tiles_here;
				c.step = step; c.strips = strips; c.strip_w = strip_w; c.patch_q = patch_q;
				pixels = strip_pixels;
			}
			if (step == t.BN) break;
		}
		if (least == INT64_MAX) return false;
		c.pixels = (int)pixels;
		c.tiles_n = (int)ceil_div((uint64_t)pixels, (uint64_t)c.step);
		if (tiles > (1ull << 28)) return false;
		c.first_tile = (int)tiles;
		tiles += (uint64_t)c.tiles_n * c.strips * p.tiles_m;
	}
	if (tiles > (1ull << 28)) return false;
	p.tiles = (int)tiles;
	return true;
}

bool split_t3(const SplitConv& p)
{
	for (int k = 0; k < p.classes; k++)
		if (p.cls[k].kh != 3 || p.cls[k].kw != 3) return false;
	return true;
}

// What a launch takes, in us: the two launches, rounds of tiles on 256 CUs; a chunk as long as its matrix instructions (where taps are
// counted at run time 10 % more; the tiles of eight blocks, which never have them written out, have the nine taps' time in theirs) or
// its staging (9.5 ns a quad); the start and the store of a tile.  Where CUs stay idle the others run at a higher clock (32 x 64 x 32 x
// 32 -> 32 5 x 5: 32.3 us in 128 tiles of 32 x 256, 38.4 in 256 of 64 x 128, half of them padding).  Classes of one to four taps switch
// between the two limits and store every other pixel.  Over 4300 layers and 25 thousand (layer, tile) pairs it is 10 % above the time,
// 12 to 16 % rms, and the tile it picks 1.2 % behind the quickest in the mean.
double split_us(const SplitConv& p, const SplitTile& t)
{
	const double rounds = (double)ceil_div(ceil_div((uint64_t)p.tiles, 8), 32), slower = split_t3(p) ? 1.0 : 1.1, clock = 0.8 + 0.2 * p.tiles / (256.0 * rounds);
	double chunk_us = 0;
	for (int k = 0; k < p.classes; k++) chunk_us += std::max(p.cls[k].kh * p.cls[k].kw * 6e-3 * t.blocks * t.mfma_ns * slower * clock, t.quads * 9.5e-3) / p.classes;
	if (p.classes > 1) return 0.95 * (9.0 + rounds * (p.chunks * chunk_us * (t.blocks == 8 ? 1.6 : 1.25) + t.round_us * 1.4));
	return 9.0 + rounds * (p.chunks * chunk_us + t.round_us);
}

// Fills in the sizes that are common to all classes, packs the weights and launches; -1 when no tile takes the shape, the
// library memory cannot be had or the estimate is above `limit_us`.
int split_run(SplitConv& p, double limit_us, int forced)
{
	const uint64_t in_elems = (uint64_t)p.N * p.C * p.H * p.W, out_elems = (uint64_t)p.N * p.M * (uint64_t)p.out_plane;
	if (in_elems >= (1ull << 30) || out_elems >= (1ull << 30) || p.C < 1 || p.M < 1) return -1;
	p.chunks = (int)ceil_div((uint64_t)p.C, 16);
	const uint64_t cobs = ceil_div((uint64_t)p.M, 32);
	if (cobs >= 65536) return -1;
	int best = -1;
	double best_us = limit_us;
	for (int k = 0; k < SPLIT_TILES; k++) {
		if (forced > 0 && k != forced - 1) continue;
		if (!split_layout(p, split_tiles[k])) continue;
		const double us = split_us(p, split_tiles[k]);
		if (us < best_us) {
			best_us = us;
			best = k;
		}
	}
	if (best < 0) return -1;
	int64_t packed = 0;
	for (int k = 0; k < p.classes; k++) {
		p.cls[k].packed = packed;
		packed += (int64_t)cobs * p.chunks * p.cls[k].kh * p.cls[k].kw * 3072;
		if (p.cls[k].kh * p.cls[k].kw * (int64_t)p.chunks * 3072 >= (1ll << 31)) return -1;
	}
	int tap_groups = 1;
	for (int k = 0; k < p.classes; k++) tap_groups = std::max(tap_groups, (p.cls[k].kh * p.cls[k].kw + 3) / 4);
	packed += 3 * 3072;  // (read, not used, where the last block's loads run ahead)
	// Planes of less than a quad are staged from a copy with a quad each, of as many images at a time as 512 MB hold: a load's offset
	// is a 32-bit number of bytes, in the copy as in the tensor.
	const int hw = p.H * p.W;
	const int group = hw < 4 ? (int)std::min<uint64_t>((uint64_t)p.N, std::max<uint64_t>(1, (512ull << 20) / (16ull * p.C))) : p.N;
	p.plane = std::max(hw, 4);
	uint8_t* scratch = static_cast<uint8_t*>(library_scratch((uint64_t)packed + (hw < 4 ? 16ull * group * p.C : 0)));
	if (scratch == nullptr) return -1;
	conv_split_pack_kernel<<<dim3((unsigned)p.chunks, (unsigned)cobs, (unsigned)(p.classes * tap_groups)), dim3(256), 0, stream()>>>(p, scratch);
	LTEN_HIP_LAUNCH_CHECK();
	p.wp = scratch;
	const bool t3 = split_t3(p);
	const float* const x = p.x;
	float* const y = p.y;
	for (int n = 0, N = p.N; n < N; n += group) {
		p.N = std::min(group, N - n);
		p.x = p.src = x + (int64_t)n * p.C * hw;
		p.y = y + (int64_t)n * p.M * p.out_plane;
		split_layout(p, split_tiles[best]);
		if (hw < 4) {
			float* copy = reinterpret_cast<float*>(scratch + packed);
			pad_planes_kernel<<<dim3((unsigned)ceil_div((uint64_t)p.N * p.C, 256)), dim3(256), 0, stream()>>>(p.x, copy, p.N * p.C, hw);
			LTEN_HIP_LAUNCH_CHECK();
			p.src = copy;
		}
		switch (best) {
		case 0: launch_split<64, 512, 1, 4, 210>(p, t3); break;
		case 1: launch_split<32, 512, 1, 4, 210>(p, t3); break;
		case 2: launch_split<128, 256, 2, 2, 162>(p, t3); break;
		case 3: launch_split<64, 256, 1, 4, 162>(p, t3); break;
		case 4: launch_split<32, 256, 1, 4, 162>(p, t3); break;
		case 5: launch_split<64, 128, 2, 2, 98>(p, t3); break;
		default: launch_split<64, 128, 2, 2, 210>(p, t3); break;
		}
		LTEN_HIP_LAUNCH_CHECK();
	}
	return 0;
}

}  // namespace

int conv_split_forward(const ConvGeo& g, const float* x, const float* w, const float* bias, float* y, double limit_us, int forced)
{
	if (g.dh != 1 || g.dw != 1 || g.sh > g.kh || g.sw > g.kw || (uint64_t)g.Cout * g.Cin * g.kh * g.kw >= (1ull << 31)) return -1;
	SplitConv p = {};
	p.x = x; p.w = w; p.bias = bias; p.y = y;
	p.N = g.N; p.C = g.Cin; p.H = g.H; p.W = g.W; p.M = g.Cout;
	p.sh = g.sh; p.sw = g.sw;
	p.out_s = 1; p.out_w = g.Wo; p.out_plane = (int64_t)g.Ho * g.Wo;
	p.w_co = g.Cin * g.kh * g.kw; p.w_ci = g.kh * g.kw;
	p.classes = 1;
	SplitClass& c = p.cls[0];
	c.kh = g.kh; c.kw = g.kw; c.ph = g.ph; c.pw = g.pw; c.Ho = g.Ho; c.Wo = g.Wo;
	c.wa = g.kw; c.wb = 1;
	return split_run(p, limit_us, forced);
}

// dx[Y][X] = sum over the taps (i, j) with Y + ph - i = sh oy of dy[oy][ox] w[i][j].  For the pixels Y = s q + y, tap rows
// i = i0 + s a of i0 = (y + ph) mod s reach oy = q + e - a with e = (y + ph - i0) / s: with the taps in reverse order a
// convolution of stride one of Na tap rows and padding Na - 1 - e (which may be negative).
int conv_split_dgrad(const ConvGeo& g, const float* w, const float* dy, float* dx, double limit_us, int forced)
{
	if (g.dh != 1 || g.dw != 1 || g.sh != g.sw || g.sh > 2 || g.sh > g.kh || g.sw > g.kw || (uint64_t)g.Cout * g.Cin * g.kh * g.kw >= (1ull << 31)) return -1;
	const int s = g.sh;
	if (g.H < s || g.W < s) return -1;
	SplitConv p = {};
	p.x = dy; p.w = w; p.y = dx;
	p.N = g.N; p.C = g.Cout; p.H = g.Ho; p.W = g.Wo; p.M = g.Cin;
	p.sh = p.sw = 1;
	p.out_s = s; p.out_w = g.W; p.out_plane = (int64_t)g.H * g.W;
	p.w_co = g.kh * g.kw; p.w_ci = g.Cin * g.kh * g.kw;
	p.classes = s * s;
	for (int k = 0; k < s * s; k++) {
		SplitClass& c = p.cls[k];
		const int y = k / s, x = k % s, i0 = (y + g.ph) % s, j0 = (x + g.pw) % s;
		c.kh = (g.kh - i0 + s - 1) / s; c.kw = (g.kw - j0 + s - 1) / s;
		c.ph = c.kh - 1 - (y + g.ph - i0) / s; c.pw = c.kw - 1 - (x + g.pw - j0) / s;
		c.Ho = (g.H - y + s - 1) / s; c.Wo = (g.W - x + s - 1) / s;
		c.out_y = y; c.out_x = x;
		c.w0 = (i0 + s * (c.kh - 1)) * g.kw + j0 + s * (c.kw - 1); c.wa = -s * g.kw; c.wb = -s;
	}
	return split_run(p, limit_us, forced);
}

}  // namespace lten_hip
