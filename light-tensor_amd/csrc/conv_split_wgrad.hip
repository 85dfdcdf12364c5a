// Conv2d weight gradient, 3 x 3 windows, on the bf16 matrix cores: dw[co][ci][i][j] = sum over the pixels of dy[co] x[ci]
// shifted by the tap, operands as three bf16 pieces in LDS (bf16_pieces.h).
//
// A workgroup sums a slice of the pixels into 64 output x 32 input channels x nine taps.  It walks chunks of OCT octets of
// pixels, an octet being eight neighbours in one output row, OC octets of a row to a strip of columns; rows are counted
// through the batch, so chunks cross images.  LDS holds a chunk twice:
//   dy  [piece][octet][64 channels][8 pixels]: a matrix operand is 16 bytes of a lane's channel
//   x   [column mod stride][piece][slot][32 channels][8 columns], slot = (input row, octet of columns), the rows the
//       chunk's windows touch, one octet more than OC
// A tap row's operands for all three tap columns are the 16 bytes of a slot and the first four of the next: the shift by
// one column is four vector instructions a piece, and a value is converted once however many taps use it.
//
// Half of the eight wavefronts load, convert and fill the stage of the next chunk (loads are a chunk further ahead), the other
// half multiplies: two blocks of 32 channels x two halves of the chunk's k-steps of 16 pixels, nine accumulators each, added at
// the end.  Measured (patch kernels, column matrices -> here): 32 x 32 x 128 x 128 -> 64 channels 171 -> 107 us (180 TFLOP/s),
// 32 x 256 x 14 x 14 -> 256 120 -> 51, 27 x 124 x 35 x 35 -> 32 86 -> 38; at stride two a chunk's staging is the longer half (16
// x 64 x 57 x 57 -> 128: 32.3 us against the implicit GEMM's 44).  Staging had bound stride one too: loads
// that touched 64 cache lines each, divisions, conversions of two values at a time, in which every instruction waits for the one
// before.  Without them the first kernel takes 175 thousand clocks, not 230, of which 111 are matrix instructions' (the second 87,
// not 109, of which 48; 57, not 67, at stride two), and slower ones, for the power limit: 120 -> 107, 59 -> 51, 97 -> 86 us
// at 64 x 128 x 28 x 28.  Shifting the operands of the next tap
// between the products of this one instead of ahead of them made no difference.  The sums of the slices go to memory
// of the library as [slice][tap][co][ci] and are added in order by a second launch.
// 2-norm error against float64 over 16 layers, the routes before -> here: 0.07 to 0.95 of it on uniform values, 0.24 to 1.3 on
// N(0,1) up to 120 thousand pixels, 1.8 times (4.5e-7) at 128 thousand and 2.3 times at 524 thousand (32 x 32 x 128 x 128 -> 64:
// 5.8e-7 -> 1.30e-6), where a slice is a chain of 128 k-steps.  The leading products in sums of their own, as the other kernels on
// pieces have them, want 144 registers more; sums from zero per k-step, added on the vector ALU, spilled.
#include "bf16_pieces.h"
#include "common.h"
#include "conv_common.h"
#include "gemm_f32_core.h"

#include <algorithm>
#include <type_traits>

namespace lten_hip {

namespace {

typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));

struct SplitWgrad {
	const float* x;
	const float* dy;
	float* partial;
	int N, C, H, W, M, Ho, Wo, ph;
	int oc_log2;                       // OC = octets of a row in a strip
	int rows;                          // output rows of the batch
	int row_chunks, chunks;            // chunks of a strip, of all strips
	int tiles_m, tiles, slices, per_slice;
	int x_last4, dy_last4;             // the last element four values can be read from
	Divisor by_Ho, by_full_rows, by_row_chunks;
};

template <int S>
struct WgradTile {
	static constexpr int OCT = S == 1 ? 8 : 4, SLOTS = S == 1 ? 32 : 20;
	// (slots and octets set apart so that the 8-byte writes of 32 lanes, two to a slot or octet, fall on different banks)
	static constexpr int X_SLOT = 512 + 16, X_PIECE = SLOTS * X_SLOT, X_PLANE = 3 * X_PIECE, X_BYTES = S * X_PLANE;
	static constexpr int DY_OCT = 1024 + (OCT == 8 ? 32 : 64), DY_PIECE = OCT * DY_OCT, DY_BYTES = 3 * DY_PIECE, STAGE = X_BYTES + DY_BYTES;
	static constexpr int X_UNITS = S == 1 ? 8 : 5, DY_LANES = 32 / OCT, DY_UNITS = 16 / DY_LANES;  // of a staging thread; channels of dy to a wavefront
	static constexpr int STEPS = OCT / 4;     // k-steps of a wavefront in a chunk
	static_assert(2 * STAGE + 64 <= 160 * 1024 && 2 * STAGE >= 2 * 9 * 16 * 64 * 4, "two stages fit LDS, and the halves' sums fit them");
};

}  // namespace

// S: stride both ways, PW: column padding (0 or 1)
template <int S, int PW>
__global__ __launch_bounds__(512, 2) void conv_split_wgrad_kernel(SplitWgrad p)
{
	typedef WgradTile<S> T;
	__shared__ __attribute__((aligned(1024))) uint8_t smem[2 * T::STAGE + 64];
	int* const again = reinterpret_cast<int*>(smem + 2 * T::STAGE);

	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	// XCD x (workgroups x, x + 8, ...) has a run of (slice, tile): the tiles of a slice read the same pixels
	const int total = p.tiles * p.slices, per_xcd = (total + 7) / 8;
	const int id = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
	if ((int)(blockIdx.x >> 3) >= per_xcd || id >= total) return;
	const int slice = id / p.tiles, tile = id - slice * p.tiles;
	const int m0 = (tile % p.tiles_m) * 64, c0 = (tile / p.tiles_m) * 32;
	const int begin = slice * p.per_slice, end = min(begin + p.per_slice, p.chunks);
	const int OC = 1 << p.oc_log2, XO = OC + 1, chunk_rows = T::OCT >> p.oc_log2;
	const int full_rows = (p.Ho - 1) * S + 3;

	if (threadIdx.x == 0) *again = 0;
	__syncthreads();

	if (wave >= 4) {
		// ---- the staging half
		// x: two lanes to a slot.  A wavefront takes eight channels: all 32 slots of one at a time, at stride two 16 slots of two at a
		// time and then the other four slots of all eight.  dy: two lanes to an octet, all octets of DY_LANES channels at a time.  So the
		// lanes of a load read rows that lie next to each other (with 16 channels of four slots to a wavefront every lane had a cache
		// line of its own).
		const int w = wave & 3, h = lane & 1;
		constexpr int COLS = 4 * S, KINDS = S;    // columns of a lane; kinds of slots it takes: its first, its second
		constexpr int DY_STEP = 4 * T::DY_LANES;  // channels from one unit to the next
		int slot_row[KINDS], slot_oct[KINDS], x_lds[KINDS], x_channel[T::X_UNITS], dy_channel[T::DY_UNITS];
		const int x_plane = p.H * p.W, x_image = p.C * x_plane, dy_plane = p.Ho * p.Wo, dy_image = p.M * dy_plane;
#pragma unroll
		for (int k = 0; k < KINDS; k++) {
			const int slot = S == 1 ? lane >> 1 : k == 0 ? lane >> 1 & 15 : 16 + (lane >> 1 & 3);
			slot_row[k] = slot / XO;
			slot_oct[k] = slot - slot_row[k] * XO;
			x_lds[k] = slot * T::X_SLOT + (8 * w + (S == 1 ? 0 : k == 0 ? lane >> 5 : lane >> 3)) * 16 + h * 8;
		}
		// (channels past the end repeat the last one, and what they add up to is not read)
#pragma unroll
		for (int u = 0; u < T::X_UNITS; u++) x_channel[u] = min(c0 + 8 * w + (S == 1 ? u : u < 4 ? 2 * u + (lane >> 5) : lane >> 3), p.C - 1) * x_plane;
		const int dy_oct = (lane >> 1) & (T::OCT - 1), dy_co = w * T::DY_LANES + (lane >> 1) / T::OCT;
#pragma unroll
		for (int u = 0; u < T::DY_UNITS; u++) dy_channel[u] = min(m0 + dy_co + DY_STEP * u, p.M - 1) * dy_plane;
		float rx[T::X_UNITS][COLS], rd[T::DY_UNITS][4];
		// of a lane's loads: where they start in channel 0, which columns exist, whether a load could leave the tensor
		struct Held { int x_at[KINDS], dy_at; unsigned x_bits[KINDS], dy_bits; bool edge; };
		Held held = {}, next = {};
		auto place_loads = [&](int chunk) {
			const int strip = quotient(chunk, p.by_row_chunks), g0 = (chunk - strip * p.row_chunks) * chunk_rows;
			const int n0 = quotient(g0, p.by_Ho), ho0 = g0 - n0 * p.Ho, g_last = min(g0 + chunk_rows, p.rows) - 1;
			const int first_rows = (p.Ho - 1 - ho0) * S + 3;
			const int n_last = quotient(g_last, p.by_Ho), ho_last = g_last - n_last * p.Ho;
			const int rows = n_last == n0 ? (ho_last - ho0) * S + 3 : first_rows + (n_last - n0 - 1) * full_rows + ho_last * S + 3;
			next.edge = false;
#pragma unroll
			for (int k = 0; k < KINDS; k++) {
				int image = n0 * x_image, yy = ho0 * S - p.ph + slot_row[k];
				if (slot_row[k] >= first_rows) {
					const int i = quotient(slot_row[k] - first_rows, p.by_full_rows);
					image += (1 + i) * x_image;
					yy = slot_row[k] - first_rows - i * full_rows - p.ph;
				}
				// (the column left of a row is the value before it, which does not count)
				const int col = (strip * OC + slot_oct[k]) * 8 * S - PW + h * COLS;
				const bool there = slot_row[k] < rows && (unsigned)yy < (unsigned)p.H;
				next.x_bits[k] = there ? ((1u << min(max(p.W - col, 0), COLS)) - 1) & ~(unsigned)(PW != 0 && col < 0) : 0u;
				next.x_at[k] = next.x_bits[k] != 0 ? image + yy * p.W + col : 0;
				next.edge |= next.x_at[k] < 0 || next.x_at[k] + (p.C - 1) * x_plane + COLS - 4 > p.x_last4;
			}
			const int g = g0 + (dy_oct >> p.oc_log2), dcol = (strip * OC + (dy_oct & (OC - 1))) * 8 + 4 * h;
			const int dn = quotient(g, p.by_Ho), dho = g - dn * p.Ho;
			next.dy_bits = g < p.rows ? (1u << min(max(p.Wo - dcol, 0), 4)) - 1 : 0u;
			next.dy_at = next.dy_bits != 0 ? dn * dy_image + dho * p.Wo + dcol : 0;
			next.edge |= next.dy_at + (p.M - 1) * dy_plane > p.dy_last4;
		};
		auto kind = [](int u) { return S == 2 && u == 4 ? 1 : 0; };
		auto load4 = [&](const float* from, int at, float* r) {
			const f4_any v = *reinterpret_cast<const f4_any*>(reinterpret_cast<const char*>(from) + (uint32_t)at * 4u);
			r[0] = v.x; r[1] = v.y; r[2] = v.z; r[3] = v.w;
		};
		// (loads under no condition: each wait is for all behind one)
		auto load_x = [&](int u) {
#pragma unroll
			for (int q = 0; q < S; q++) load4(p.x, min(max(next.x_at[kind(u) < KINDS ? kind(u) : 0] + x_channel[u] + 4 * q, 0), p.x_last4), &rx[u][4 * q]);
		};
		auto load_dy = [&](int u) { load4(p.dy, min(next.dy_at + dy_channel[u], p.dy_last4), rd[u]); };
		// four values that were read `by` elements early because the tensor ends behind them, or one late because it starts with the second
		auto move = [&](float* r, int by) {
			const float v0 = r[0], v1 = r[1], v2 = r[2], v3 = r[3];
			r[0] = by == 1 ? v1 : by == 2 ? v2 : by == 3 ? v3 : v0;
			r[1] = by == -1 ? v0 : by == 1 ? v2 : by == 2 ? v3 : v1;
			r[2] = by == -1 ? v1 : by == 1 ? v3 : v2;
			r[3] = by == -1 ? v2 : v3;
		};
		// eight values, the first four for `a`, the others for `b`
		auto put = [&](float (&v)[8], uint8_t* a, uint8_t* b, int step) {
			uint4 piece[3];
			split8_scaled(v, piece);
#pragma unroll
			for (int q = 0; q < 3; q++) *reinterpret_cast<uint2*>(a + q * step) = make_uint2(piece[q].x, piece[q].y);
#pragma unroll
			for (int q = 0; q < 3; q++) *reinterpret_cast<uint2*>(b + q * step) = make_uint2(piece[q].z, piece[q].w);
		};
		place_loads(begin);
#pragma unroll
		for (int u = 0; u < T::X_UNITS; u++) load_x(u);
#pragma unroll
		for (int u = 0; u < T::DY_UNITS; u++) load_dy(u);
		for (int chunk = begin - 1; chunk < end; chunk++) {  // converts chunk + 1, loads chunk + 2 (the last one again past the end)
			if (chunk + 1 < end) {
				held = next;
				place_loads(min(chunk + 2, end - 1));
				if (__any(held.edge)) {
#pragma unroll
					for (int u = 0; u < T::X_UNITS; u++)
#pragma unroll
						for (int q = 0; q < S; q++) {
							const int want = held.x_at[kind(u) < KINDS ? kind(u) : 0] + x_channel[u] + 4 * q;
							move(&rx[u][4 * q], want - min(max(want, 0), p.x_last4));
						}
#pragma unroll
					for (int u = 0; u < T::DY_UNITS; u++) {
						const int want = held.dy_at + dy_channel[u];
						move(rd[u], want - min(want, p.dy_last4));
					}
				}
				uint8_t* const st = smem + ((chunk + 1 - begin) & 1) * T::STAGE;
				float scale[COLS], v[8];
#pragma unroll
				for (int e = 0; e < COLS; e++) scale[e] = scale_where(held.x_bits[0], e);
				if constexpr (S == 1) {
					uint8_t* const sx = st + x_lds[0];
#pragma unroll
					for (int u = 0; u < T::X_UNITS; u += 2) {
#pragma unroll
						for (int e = 0; e < 8; e++) v[e] = rx[u + e / 4][e % 4] * scale[e % 4];
						load_x(u);
						load_x(u + 1);
						put(v, sx + u * 16, sx + u * 16 + 16, T::X_PIECE);
					}
				} else {
#pragma unroll
					for (int u = 0; u < T::X_UNITS; u++) {
						if (u == 4) {
#pragma unroll
							for (int e = 0; e < COLS; e++) scale[e] = scale_where(held.x_bits[KINDS - 1], e);
						}
#pragma unroll
						for (int e = 0; e < 8; e++) v[e] = rx[u][e < 4 ? 2 * e : 2 * e - 7] * scale[e < 4 ? 2 * e : 2 * e - 7];  // the even ones, the odd ones
						load_x(u);
						uint8_t* const sx = st + x_lds[u == 4 ? KINDS - 1 : 0] + (u < 4 ? u * 32 : 0);
						put(v, sx, sx + T::X_PLANE, T::X_PIECE);
					}
				}
#pragma unroll
				for (int e = 0; e < 4; e++) scale[e] = scale_where(held.dy_bits, e);
				uint8_t* const sd = st + T::X_BYTES + dy_oct * T::DY_OCT + dy_co * 16 + h * 8;
#pragma unroll
				for (int u = 0; u < T::DY_UNITS; u += 2) {
#pragma unroll
					for (int e = 0; e < 8; e++) v[e] = rd[u + e / 4][e % 4] * scale[e % 4];
					load_dy(u);
					load_dy(u + 1);
					put(v, sd + u * DY_STEP * 16, sd + (u + 1) * DY_STEP * 16, T::DY_PIECE);
				}
			}
			__syncthreads();
		}
		__syncthreads();  // (the multiplying half exchanges its sums)
		return;
	}

	// ---- the multiplying half
	__builtin_amdgcn_s_setprio(1);
	const int mt = wave & 1, khalf = wave >> 1, lrow = lane & 31, lk = lane >> 5;
	v16f acc[9];
#pragma unroll
	for (int t = 0; t < 9; t++)
#pragma unroll
		for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;

	// k-step t of this wavefront: octets 2 (khalf + 2 t) + lk of the chunk; where they lie in the stage
	uint32_t xb[T::STEPS], db[T::STEPS];
#pragma unroll
	for (int t = 0; t < T::STEPS; t++) db[t] = (uint32_t)(T::X_BYTES + (2 * (khalf + 2 * t) + lk) * T::DY_OCT + (mt * 32 + lrow) * 16);
	auto place = [&](int chunk) {
		const int strip = quotient(chunk, p.by_row_chunks), g0 = (chunk - strip * p.row_chunks) * chunk_rows;
		const int n0 = quotient(g0, p.by_Ho), ho0 = g0 - n0 * p.Ho, first_rows = (p.Ho - 1 - ho0) * S + 3;
#pragma unroll
		for (int t = 0; t < T::STEPS; t++) {
			const int oct = 2 * (khalf + 2 * t) + lk;
			const int g = min(g0 + (oct >> p.oc_log2), p.rows - 1);  // (rows past the last: their dy is zero)
			const int n = quotient(g, p.by_Ho), ho = g - n * p.Ho;
			const int r = n == n0 ? (ho - ho0) * S : first_rows + (n - n0 - 1) * full_rows + ho * S;
			xb[t] = (uint32_t)((r * XO + (oct & (OC - 1))) * T::X_SLOT + lrow * 16);
		}
	};
	// a window: eight columns in four words and two more in the fifth; at stride two the eight odd ones behind them
	constexpr int WORDS = S == 1 ? 5 : 9;
	uint32_t win[2][3][WORDS];
	bf16x8 fa[2][3];
	auto read_window = [&](int set, uint32_t base, int i) {
#pragma unroll
		for (int v = 0; v < 3; v++) {
			const uint8_t* at = smem + base + i * XO * T::X_SLOT + v * T::X_PIECE;
			const uint4 a = *reinterpret_cast<const uint4*>(at);
			win[set][v][0] = a.x; win[set][v][1] = a.y; win[set][v][2] = a.z; win[set][v][3] = a.w;
			win[set][v][4] = *reinterpret_cast<const uint32_t*>(at + T::X_SLOT);
			if (S == 2) {
				const uint4 o = *reinterpret_cast<const uint4*>(at + T::X_PLANE);
				win[set][v][WORDS - 4] = o.x; win[set][v][WORDS - 3] = o.y; win[set][v][WORDS - 2] = o.z; win[set][v][WORDS - 1] = o.w;
			}
		}
	};
	auto read_a = [&](int set, uint32_t base) {
#pragma unroll
		for (int v = 0; v < 3; v++) fa[set][v] = *reinterpret_cast<const bf16x8*>(smem + base + v * T::DY_PIECE);
	};
	typedef uint32_t u4 __attribute__((ext_vector_type(4)));
	// the operand of tap column j
	auto tap = [&](int set, int v, int j) {
		uint32_t f[4];
#pragma unroll
		for (int e = 0; e < 4; e++) {
			const uint32_t w0 = win[set][v][e], w1 = win[set][v][e + 1];
			f[e] = j == 0 ? w0 : S == 2 && j == 1 ? win[set][v][WORDS - 4 + e] : S == 1 && j == 2 ? w1 : __builtin_amdgcn_alignbit(w1, w0, 16);
		}
		return __builtin_bit_cast(bf16x8, (u4){ f[0], f[1], f[2], f[3] });
	};

	place(begin);
	__syncthreads();  // stage 0 holds the first chunk
	read_a(0, db[0]);
	read_window(0, xb[0], 0);
	// A chunk from stage ST: the operands of the next (k-step, tap row) are read under the products of this one, those of the
	// next chunk behind the barrier, under the last tap's.  (PAR: the operand set the chunk starts with)
	auto run_chunk = [&](auto par_c, int chunk, int stage) {
		constexpr int PAR = decltype(par_c)::value;
		const uint32_t base = stage * T::STAGE, other = (stage ^ 1) * T::STAGE;
#pragma unroll
		for (int t = 0; t < T::STEPS; t++) {
			constexpr int A0 = T::STEPS == 1 ? PAR : 0;
			const int a_set = T::STEPS == 1 ? A0 : (t & 1);
#pragma unroll
			for (int i = 0; i < 3; i++) {
				const int set = (PAR + t * 3 + i) & 1;
				const bool last_row = i == 2, last = last_row && t == T::STEPS - 1;
#pragma unroll
				for (int j = 0; j < 3; j++) {
					bf16x8 fb[3];
#pragma unroll
					for (int v = 0; v < 3; v++) fb[v] = tap(set, v, j);
					if (last && j == 2) {
						place(min(chunk + 1, end - 1));
						__syncthreads();
						read_a(a_set ^ 1, other + db[0]);
						read_window(set ^ 1, other + xb[0], 0);
					}
					if (!last && j == 0) {
						if (last_row) read_a(a_set ^ 1, base + db[t + 1 < T::STEPS ? t + 1 : 0]);
						read_window(set ^ 1, base + xb[last_row && t + 1 < T::STEPS ? t + 1 : t], last_row ? 0 : i + 1);
					}
#pragma unroll
					for (int q = 0; q < 6; q++) {
						acc[i * 3 + j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a_set][piece_a[q]], fb[piece_b[q]], acc[i * 3 + j], 0, 0, 0);
					}
					__builtin_amdgcn_sched_barrier(0);
				}
			}
		}
	};
	using P0 = std::integral_constant<int, 0>;
	using P1 = std::integral_constant<int, T::STEPS & 1>;  // three tap rows a k-step: an odd count of steps changes the set
	int chunk = begin;
	for (; chunk + 1 < end; chunk += 2) {
		run_chunk(P0{}, chunk, 0);
		run_chunk(P1{}, chunk + 1, 1);
	}
	if (chunk < end) run_chunk(P0{}, chunk, 0);

	// Values without three pieces, sums that are too large: the slice once more on the values themselves.
	float finite[3] = { 0.0f, 0.0f, 0.0f };
#pragma unroll
	for (int t = 0; t < 9; t++)
#pragma unroll
		for (int r = 0; r < 16; r++) finite[t % 3] = fmaf(acc[t][r], 0.0f, finite[t % 3]);
	if (__any(finite[0] + finite[1] + finite[2] != 0.0f) && lane == 0) *again = 1;
	float4* const sums = reinterpret_cast<float4*>(smem);
	if (khalf == 1) {
#pragma unroll
		for (int t = 0; t < 9; t++)
#pragma unroll
			for (int e = 0; e < 4; e++)
				sums[((mt * 9 + t) * 4 + e) * 64 + lane] = make_float4(acc[t][4 * e], acc[t][4 * e + 1], acc[t][4 * e + 2], acc[t][4 * e + 3]);
	}
	__syncthreads();
	if (khalf == 1) return;
	const int Mp = p.tiles_m * 64, Cp = p.tiles / p.tiles_m * 32;
	float* out = p.partial + (int64_t)slice * 9 * Mp * Cp + (int64_t)(m0 + mt * 32 + 4 * lk) * Cp + c0 + lrow;
	if (*again != 0) {
		const float* dyc = p.dy + (int64_t)min(m0 + mt * 32 + lrow, p.M - 1) * p.Ho * p.Wo;
		const float* xc = p.x + (int64_t)min(c0 + lrow, p.C - 1) * p.H * p.W;
#pragma unroll 1
		for (int t = 0; t < 9; t++) {
			v16f sum;
#pragma unroll
			for (int r = 0; r < 16; r++) sum[r] = 0.0f;
#pragma unroll 1
			for (int c = begin; c < end; c++) {
				const int strip = c / p.row_chunks, g0 = (c - strip * p.row_chunks) * chunk_rows, last = min((strip + 1) * OC * 8, p.Wo);
#pragma unroll 1
				for (int g = g0; g < min(g0 + chunk_rows, p.rows); g++) {
					const int n = g / p.Ho, ho = g - n * p.Ho, yy = ho * S - p.ph + t / 3;
#pragma unroll 1
					for (int first = strip * OC * 8; first < last; first += 2) {
						const int wo = first + lk, xx = wo * S - PW + t % 3;
						const bool in = wo < last, there = in && (unsigned)yy < (unsigned)p.H && (unsigned)xx < (unsigned)p.W;
						const float a = dyc[((int64_t)n * p.M * p.Ho + ho) * p.Wo + (in ? wo : 0)];
						const float b = xc[(int64_t)n * p.C * p.H * p.W + (there ? yy * p.W + xx : 0)];
						sum = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? a : 0.0f, there ? b : 0.0f, sum, 0, 0, 0);
					}
				}
			}
#pragma unroll
			for (int r = 0; r < 16; r++) out[((int64_t)t * Mp + (r >> 2) * 8 + (r & 3)) * Cp] = sum[r];
		}
		return;
	}
#pragma unroll
	for (int t = 0; t < 9; t++) {
#pragma unroll
		for (int e = 0; e < 4; e++) {
			const float4 v = sums[((mt * 9 + t) * 4 + e) * 64 + lane];
			const float half[4] = { v.x, v.y, v.z, v.w };
			// (unscaled one by one: the halves are finite, their sum need not be)
#pragma unroll
			for (int f = 0; f < 4; f++) acc[t][4 * e + f] = fmaf(half[f], pieces_unscale, acc[t][4 * e + f] * pieces_unscale);
		}
#pragma unroll
		for (int r = 0; r < 16; r++) out[((int64_t)t * Mp + (r >> 2) * 8 + (r & 3)) * Cp] = acc[t][r];
	}
}

// dw[co][ci][tap] = sum of partial[slice][tap][co][ci] over the slices: a workgroup takes 32 input channels of one (tap, co),
// eight threads to a value, each a run of slices, added in order.
__global__ __launch_bounds__(256) void conv_split_wgrad_sum_kernel(const float* __restrict__ partial, float* __restrict__ dw, int slices, int M, int C, int Mp, int Cp)
{
	__shared__ float part[8][33];
	const int ci = blockIdx.x * 32 + (threadIdx.x & 31), part_of = threadIdx.x >> 5, co = blockIdx.y, tap = blockIdx.z;
	const int per = (slices + 7) / 8, first = part_of * per, last = min(first + per, slices);
	const float* src = partial + ((int64_t)tap * Mp + co) * Cp + ci;
	const int64_t step = (int64_t)9 * Mp * Cp;
	float sum = 0.0f;
	int s = first;
	for (; s + 8 <= last; s += 8) {
		float v[8];
#pragma unroll
		for (int e = 0; e < 8; e++) v[e] = src[(s + e) * step];
#pragma unroll
		for (int e = 0; e < 8; e++) sum += v[e];
	}
	for (; s < last; s++) sum += src[s * step];
	part[part_of][threadIdx.x & 31] = sum;
	__syncthreads();
	if (part_of != 0 || ci >= C) return;
#pragma unroll
	for (int k = 1; k < 8; k++) sum += part[k][threadIdx.x & 31];
	dw[((int64_t)co * C + ci) * 9 + tap] = sum;
}

// The same sums, in the same order, for up to 16 slices of a wide layer: a workgroup takes 32 input channels of WIDE_CO output channels, a thread
// four channels of one tap over all slices, and the 288 values of an output channel leave in one run.  Bound by the read of the slices
// (with eight threads to a value and a workgroup per (tap, channel) it was the 18432 workgroups: 256 x 256 x 3 x 3 of 8 slices 10.6
// us, 5.7 here).
constexpr int WIDE_CO = 3, WIDE_SLICES = 16;
__global__ __launch_bounds__(256) void conv_split_wgrad_sum_wide_kernel(const float* __restrict__ partial, float* __restrict__ dw, int slices, int M, int C, int Mp, int Cp)
{
	__shared__ float out[WIDE_CO][288];
	const int tid = threadIdx.x, of = tid / 72, at = tid % 72, tap = at >> 3, ci = (at & 7) * 4, co = blockIdx.y * WIDE_CO + of, ci0 = blockIdx.x * 32;
	if (of < WIDE_CO && co < M) {
		const float* src = partial + ((int64_t)tap * Mp + co) * Cp + ci0 + ci;
		const int64_t step = (int64_t)9 * Mp * Cp;
		const int per = (slices + 7) / 8;  // 1 or 2: the others' runs
		float4 v[WIDE_SLICES];
#pragma unroll
		for (int s = 0; s < WIDE_SLICES; s++) v[s] = *reinterpret_cast<const float4*>(src + min(s, slices - 1) * step);
		float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
		for (int s = 0; s < WIDE_SLICES; s++) {
			float4 run = v[s];
			if (per == 2) {
				if (s & 1) continue;
				if (s + 1 < slices) { run.x += v[s + 1].x; run.y += v[s + 1].y; run.z += v[s + 1].z; run.w += v[s + 1].w; }
			}
			if (s < slices) { sum.x += run.x; sum.y += run.y; sum.z += run.z; sum.w += run.w; }
		}
		out[of][(ci + 0) * 9 + tap] = sum.x;
		out[of][(ci + 1) * 9 + tap] = sum.y;
		out[of][(ci + 2) * 9 + tap] = sum.z;
		out[of][(ci + 3) * 9 + tap] = sum.w;
	}
	__syncthreads();
	const int have = min(C - ci0, 32) * 9;
	for (int i = tid; i < WIDE_CO * 288; i += 256) {
		const int k = i / 288, j = i - k * 288, m = blockIdx.y * WIDE_CO + k;
		if (m < M && j < have) dw[((int64_t)m * C + ci0) * 9 + j] = out[k][j];
	}
}

// -1: not taken (another window, stride or padding, sizes, no memory, or expected to take `limit_us` or more)
int conv_split_wgrad(const ConvGeo& g, const float* x, const float* dy, float* dw, double limit_us)
{
	const uint64_t in_elems = (uint64_t)g.N * g.Cin * g.H * g.W, out_elems = (uint64_t)g.N * g.Cout * g.Ho * g.Wo;
	if (g.kh != 3 || g.kw != 3 || g.dh != 1 || g.dw != 1 || g.sh != g.sw || g.sh > 2 || g.pw > 1 || g.ph > 2 || in_elems >= (1ull << 30) || out_elems >= (1ull << 30) ||
	    in_elems < 4 || out_elems < 4 || (uint64_t)g.Cout >= 65536) return -1;
	if (in_elems < 16 && g.W < 3) return -1;  // (a handful of values: the other routes')
	const int S = g.sh, oct = S == 1 ? 8 : 4, slots = S == 1 ? 32 : 20;
	SplitWgrad p = {};
	p.x = x; p.dy = dy;
	p.N = g.N; p.C = g.Cin; p.H = g.H; p.W = g.W; p.M = g.Cout; p.Ho = g.Ho; p.Wo = g.Wo; p.ph = g.ph;
	p.x_last4 = (int)in_elems - 4; p.dy_last4 = (int)out_elems - 4;
	p.rows = g.N * g.Ho;
	p.by_Ho = make_divisor((uint32_t)g.Ho);
	p.by_full_rows = make_divisor((uint32_t)((g.Ho - 1) * S + 3));
	p.tiles_m = (int)ceil_div((uint64_t)g.Cout, 64);
	p.tiles = p.tiles_m * (int)ceil_div((uint64_t)g.Cin, 32);
	// Strips of OC octets: the fewest chunks, then the fewest slots staged (a chunk's rows with their halo, of every image they
	// can touch).
	int64_t best = INT64_MAX, best_used = 0;
	int best_log2 = -1;
	for (int l = 0; (1 << l) <= oct; l++) {
		const int64_t OC = 1 << l, rows = std::min<int64_t>(p.rows, oct / OC), images = std::min<int64_t>(g.N, g.Ho % rows == 0 && oct / OC == rows ? 1 : (rows - 2 + g.Ho) / g.Ho + 1);
		const int64_t used = ((rows - images) * S + images * std::max(3, S)) * (OC + 1);
		if (used > slots) continue;
		const int64_t chunks = (int64_t)ceil_div((uint64_t)p.rows, (uint64_t)(oct / OC)) * (int64_t)ceil_div((uint64_t)g.Wo, (uint64_t)(8 * OC));
		const int64_t cost = chunks * (100 + used);
		if (cost < best) {
			best = cost;
			best_used = used;
			best_log2 = l;
		}
	}
	if (best_log2 < 0) return -1;
	p.oc_log2 = best_log2;
	p.row_chunks = (int)ceil_div((uint64_t)p.rows, (uint64_t)(oct >> best_log2));
	p.chunks = p.row_chunks * (int)ceil_div((uint64_t)g.Wo, (uint64_t)(8 << best_log2));
	p.by_row_chunks = make_divisor((uint32_t)p.row_chunks);
	// slices that give every CU a workgroup
	const uint64_t want = std::max<uint64_t>(1, 256 / (uint64_t)p.tiles);
	p.per_slice = (int)ceil_div((uint64_t)p.chunks, want);
	p.slices = (int)ceil_div((uint64_t)p.chunks, (uint64_t)p.per_slice);
	const uint64_t Mp = (uint64_t)p.tiles_m * 64, Cp = (uint64_t)(p.tiles / p.tiles_m) * 32, bytes = (uint64_t)p.slices * 9 * Mp * Cp * 4;
	if (bytes > (1ull << 29) || (uint64_t)p.tiles * p.slices >= (1u << 24)) return -1;
	// a chunk: two k-steps of 54 products (32 clocks each; 41 and, at stride two, the staging's 3900 with 15 slots are fitted to times);
	// a start and an end; the launches and the sums
	const double rounds = (double)ceil_div((uint64_t)p.tiles * p.slices, 256), chunk_clocks = S == 1 ? 2 * 54 * 41.0 : 3900.0 + 200.0 * (double)std::max<int64_t>(0, best_used - 16);
	if (10.0 + rounds * (p.per_slice * chunk_clocks + 8000.0) / 1850.0 + 1.2 * (double)bytes / 4e6 >= limit_us) return -1;
	p.partial = static_cast<float*>(library_scratch(bytes));
	if (p.partial == nullptr) return -1;
	const dim3 grid((unsigned)(8 * ceil_div((uint64_t)p.tiles * p.slices, 8)));
	if (S == 1 && g.pw == 0) conv_split_wgrad_kernel<1, 0><<<grid, dim3(512), 0, stream()>>>(p);
	if (S == 1 && g.pw == 1) conv_split_wgrad_kernel<1, 1><<<grid, dim3(512), 0, stream()>>>(p);
	if (S == 2 && g.pw == 0) conv_split_wgrad_kernel<2, 0><<<grid, dim3(512), 0, stream()>>>(p);
	if (S == 2 && g.pw == 1) conv_split_wgrad_kernel<2, 1><<<grid, dim3(512), 0, stream()>>>(p);
	LTEN_HIP_LAUNCH_CHECK();
	if (p.slices <= WIDE_SLICES)
		conv_split_wgrad_sum_wide_kernel<<<dim3((unsigned)ceil_div((uint64_t)g.Cin, 32), (unsigned)ceil_div((uint64_t)g.Cout, WIDE_CO)), dim3(256), 0, stream()>>>(
		    p.partial, dw, p.slices, g.Cout, g.Cin, (int)Mp, (int)Cp);
	else conv_split_wgrad_sum_kernel<<<dim3((unsigned)ceil_div((uint64_t)g.Cin, 32), (unsigned)g.Cout, 9), dim3(256), 0, stream()>>>(p.partial, dw, p.slices, g.Cout, g.Cin, (int)Mp, (int)Cp);
	LTEN_HIP_LAUNCH_CHECK();
	return 0;
}

}  // namespace lten_hip
