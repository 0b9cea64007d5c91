// The weight gemvs on either side of nnc's attention (reference
// src/libnnc/nn_ops.h:95-180; model.cpp:1189-1210 picks one by tensor type):
// Y[t][r] = sum_k W[r][k] X[t][k], W in BF16, in the Q8_0 split layout (int8 q,
// one BF16 scale per 32-column block) or the Q4_S split layout (nibble q, BF16
// scale and bias per block; reference docs/design.md:141-193).
//
// One vector (gemv_vec_kernel): x in LDS, fp32 products on the VALU, a
// wavefront per pair of rows. More than one: MFMA products
// (v_mfma_f32_16x16x32_bf16), 16 weight rows x 16 vectors, one 32-column block
// per k-step. A = the rows' weights of the block as bf16, exact for BF16 and
// for the integer q of Q8_0 (|q| <= 127) and Q4_S (0..15). B = X^T split into
// bf16 hi + lo (x ~= hi + lo to about 16 bits), so the product against the
// exact A is near-fp32 and the accumulation fp32. A quantised block's product
// starts from zero and is scaled into the row's sum with the block's scale;
// Q4_S adds bias * (block sum of x) in a second sum. Three kernels:
//   gemv_kernel        2 to 16 vectors of wide and of narrow matrices
//                      (gemv_stages_x has the lines). Grid: (row groups of kGemvRows = 128, K splits).
//                      A work-group of 8 wavefronts (two work-groups per CU)
//                      stages its K range of X^T (hi, lo, and for Q4_S the
//                      block sums) in LDS once; each wavefront then streams
//                      the weights of its own 16 rows block by block over the
//                      whole range, kAhead<F> blocks of loads in flight (BF16:
//                      every block of its split, at most 16, issued before X^T
//                      is staged). With one K split the rows go straight to Y;
//                      with several, each split writes a partial and a second
//                      kernel adds the splits in split order;
//   gemv_batch_kernel  the other 2 to 16 vectors, and up to 64. X is put into
//                      operand order once by gemv_stage_x_kernel; a work-group
//                      takes a few row tiles, its wavefronts share the columns,
//                      and their sums meet in LDS: no partials in memory;
//   gemv_tile_kernel   more vectors than that: tiles of rows x vectors over all
//                      the columns, W and X through LDS.
// The sums' orders are fixed, so results are the same run to run.
#include "device_common.h"
#include "kernels.h"

#include <algorithm>
#include <type_traits>

namespace nnchip
{
	namespace
	{
		// Blocks of weights in flight per wavefront of the batch kernel, per
		// layout (a 16-vector Qwen3-4B layer, us, at 8 / 4 / 3 / 2: BF16 91.6 /
		// 87.5 / 87.6 / 89.6, Q8_0 97.6 / 88.9 / 89.5 / 85.7, Q4_S 96.5 / 90.2 /
		// 90.3 / 87.7; 12 was slower still than 8).
		template <int F>
		constexpr int kAhead = F == kGemvBf16 ? 4 : 2;
		// BF16 instead issues every weight load of its K split (at most
		// kGemvBf16Blocks blocks, 16 bytes per lane each) before X^T is staged, and
		// runs its blocks unrolled with no load left to wait for (a 16-vector
		// Qwen3-4B layer 86.9 -> 77.8 us; the quantised layouts, whose loads are
		// 8 and 4 bytes, ran 8 % slower that way: 92.1 and 94.5 us).
		constexpr int kGemvBf16Blocks = 16;
		// The quantised layouts' blocks per K split, what gemv_batch_lds holds
		// of 16 vectors.
		constexpr int kGemvQuantBlocks = 18;
		// 16-byte loads in flight per lane of the one-vector kernel, per layout
		// (a one-vector Qwen3-4B layer, us, at 8 / 6 / 4: BF16 55.7 / 56.1 /
		// 59.2, Q8_0 48.7 / 48.9 / 48.4, Q4_S 51.5 / 50.9 / 48.4; 16 slower).
		template <int F>
		constexpr int kVecAhead = F == kGemvQ4S ? 4 : 8;

		// The matrix holding stacked row `row` and the row's index in it (row
		// uniform over the caller's rows: a row pair or a 16-row tile).
		struct mat_row
		{
			gemv_mat m;
			int r;
		};
		__device__ __forceinline__ mat_row locate(const gemv_params& p, int row)
		{
			const int k = (row >= p.mrow[1]) + (row >= p.mrow[2]);
			const gemv_mat& m = k == 0 ? p.mats[0] : (k == 1 ? p.mats[1] : p.mats[2]);
			return {m, row - (k == 0 ? 0 : (k == 1 ? p.mrow[1] : p.mrow[2]))};
		}

		// MFMA k-slots of a 32-column block: a lane of k-group g holds slots
		// 8 g .. 8 g + 7. For BF16 and Q8_0 slot s is column s. Q4_S packs
		// elements i and i + 16 into byte i, so a lane reading bytes 4 g .. 4 g + 3
		// holds columns 4 g .. 4 g + 3 (low nibbles, slots 8 g .. 8 g + 3) and
		// 16 + 4 g .. 16 + 4 g + 3 (high nibbles, slots 8 g + 4 .. 8 g + 7); X^T is
		// staged in the same slot order.

		// Two fp32 values whose bf16 is exact (integers below 256 in magnitude)
		// -> one packed bf16 pair: the upper halves of their bit patterns.
		__device__ __forceinline__ uint32_t pack_hi16(float lo, float hi)
		{
			return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
		}

		// Eight int8 q (two dwords) -> bf16: u = q + 128 as unsigned bytes,
		// float(u) - 128 = q exactly.
		__device__ __forceinline__ bf16x8 q8_to_bf16x8(uint32_t w0, uint32_t w1)
		{
			u32x4 r;
			const uint32_t u0 = w0 ^ 0x80808080u, u1 = w1 ^ 0x80808080u;
			auto byte = [](uint32_t u, int i) { return static_cast<float>((u >> (8 * i)) & 0xffu) - 128.0f; };
			r[0] = pack_hi16(byte(u0, 0), byte(u0, 1));
			r[1] = pack_hi16(byte(u0, 2), byte(u0, 3));
			r[2] = pack_hi16(byte(u1, 0), byte(u1, 1));
			r[3] = pack_hi16(byte(u1, 2), byte(u1, 3));
			return as_bf16x8(r);
		}

		// Four Q4_S bytes -> bf16 slots: low nibbles then high nibbles.
		__device__ __forceinline__ bf16x8 q4_to_bf16x8(uint32_t w)
		{
			u32x4 r;
			const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;
			auto byte = [](uint32_t u, int i) { return static_cast<float>((u >> (8 * i)) & 0xffu); };
			r[0] = pack_hi16(byte(lo, 0), byte(lo, 1));
			r[1] = pack_hi16(byte(lo, 2), byte(lo, 3));
			r[2] = pack_hi16(byte(hi, 0), byte(hi, 1));
			r[3] = pack_hi16(byte(hi, 2), byte(hi, 3));
			return as_bf16x8(r);
		}

		template <int F>
		struct a_block
		{
			u32x4 v; // BF16: 8 weights; Q8_0: 8 int8 in v[0..1]; Q4_S: 4 bytes in v[0]
		};

		// Row `row` of W (cols columns), block blk, the lane's k-group grp.
		template <int F>
		__device__ __forceinline__ a_block<F> load_a(const void* W, int cols, int row, int blk, int grp)
		{
			a_block<F> a;
			const size_t base = static_cast<size_t>(row) * cols + 32 * blk;
			if constexpr (F == kGemvBf16)
				a.v = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(W) + base + 8 * grp);
			else if constexpr (F == kGemvQ8_0)
			{
				const u32x2 w = *reinterpret_cast<const u32x2*>(static_cast<const int8_t*>(W) + base + 8 * grp);
				a.v = u32x4{w.x, w.y, 0u, 0u};
			}
			else
				a.v = u32x4{*reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(W) + base / 2 + 4 * grp), 0u,
				            0u, 0u};
			return a;
		}

		template <int F>
		__device__ __forceinline__ bf16x8 a_operand(const a_block<F>& a)
		{
			if constexpr (F == kGemvBf16)
				return as_bf16x8(a.v);
			else if constexpr (F == kGemvQ8_0)
				return q8_to_bf16x8(a.v[0], a.v[1]);
			else
				return q4_to_bf16x8(a.v[0]);
		}

		template <int F>
		__global__ __launch_bounds__(4 * kGemvRows) void gemv_kernel(const gemv_params p)
		{
			// Dynamic LDS: X^T hi and lo [block][token][32 slots] (bf16), the 16
			// rows' scales (and biases) [block][16], and the wavefronts' sums.
			extern __shared__ __attribute__((aligned(16))) unsigned char s_raw[];
			const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
			const int col = lane & 15, grp = lane >> 4;
			const int nt = p.n_batch;
			const int split = blockIdx.y;
			const int b0 = split * p.split_blocks;
			const int nblk = min(p.split_blocks, p.cols / 32 - b0); // >= 1
			uint16_t* s_xh = reinterpret_cast<uint16_t*>(s_raw);
			uint16_t* s_xl = s_xh + static_cast<size_t>(p.split_blocks) * nt * 32;
			uint16_t* s_sc = s_xl + static_cast<size_t>(p.split_blocks) * nt * 32;
			uint16_t* s_bi = s_sc + p.split_blocks * kGemvRows;
			float* s_xs = reinterpret_cast<float*>(s_bi + p.split_blocks * kGemvRows); // Q4_S: [block][token] sums of x

			// The work-group's kGemvRows rows; wavefront w takes rows 16 w .. 16 w + 15
			// over every block of the range, kAhead blocks in flight, the first
			// ones while X^T is staged.
			const int row0 = blockIdx.x * kGemvRows + 16 * wave;
			// The tile's matrix (one for all 16 rows) and its rows in it (a tile
			// past the last row has none and only helps stage X^T).
			const int m_rows = max(0, min(16, p.rows - row0)); // (only the last matrix's last tile is short)
			const mat_row mr = locate(p, min(row0, p.rows - 1));
			const int ra = mr.r + min(col, max(m_rows - 1, 0)); // this lane's A row in the matrix (clamped; not stored)
			const int n_mine = m_rows > 0 ? nblk : 0; // blocks of this wavefront
			auto my_block = [&](int i) { return b0 + min(i, max(n_mine - 1, 0)); };
			constexpr int NA = F == kGemvBf16 ? kGemvBf16Blocks : kAhead<F>; // loads in flight
			a_block<F> ab[NA];
#pragma unroll
			for (int j = 0; j < NA; ++j) ab[j] = load_a<F>(mr.m.w, p.cols, ra, min(my_block(j), p.cols / 32 - 1), grp);

			// X^T of the range, four columns per piece (consecutive threads read
			// consecutive 16 bytes of a token's row), loads issued eight at a time.
			const int n_pieces = nblk * nt * 8;
			for (int i0 = 0; i0 < n_pieces; i0 += 4 * kGemvRows * 8)
			{
				float4 xv[8];
#pragma unroll
				for (int u = 0; u < 8; ++u)
				{
					const int i = i0 + threadIdx.x + 4 * kGemvRows * u;
					const int q = i & 7, b = (i >> 3) % nblk, t = (i >> 3) / nblk;
					xv[u] = i < n_pieces ? *reinterpret_cast<const float4*>(p.x + t * p.x_stride + 32 * (b0 + b) + 4 * q)
					                     : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
				}
#pragma unroll
				for (int u = 0; u < 8; ++u)
				{
					const int i = i0 + threadIdx.x + 4 * kGemvRows * u;
					if (i >= n_pieces) continue;
					const int q = i & 7, b = (i >> 3) % nblk, t = (i >> 3) / nblk;
					// The piece's first k-slot; its four columns take four consecutive slots.
					const int slot0 = F == kGemvQ4S ? (q < 4 ? 8 * q : 8 * (q - 4) + 4) : 4 * q;
					const uint32_t h0 = cvt_pk_bf16(xv[u].x, xv[u].y), h1 = cvt_pk_bf16(xv[u].z, xv[u].w);
					const uint32_t l0 = cvt_pk_bf16(xv[u].x - bf16_lo(h0), xv[u].y - bf16_hi(h0));
					const uint32_t l1 = cvt_pk_bf16(xv[u].z - bf16_lo(h1), xv[u].w - bf16_hi(h1));
					const size_t at = (static_cast<size_t>(b) * nt + t) * 32 + slot0;
					*reinterpret_cast<u32x2*>(s_xh + at) = u32x2{h0, h1};
					*reinterpret_cast<u32x2*>(s_xl + at) = u32x2{l0, l1};
				}
			}
			const int nb_all = p.cols / 32;
			if constexpr (F == kGemvQ4S)
			{
				// Block sums of x: the caller's, or as the reference evaluates them
				// (reference nn_ops.cpp:1305-1316 under its -ffast-math build:
				// lane j = (x[j] + x[8 + j]) + (x[16 + j] + x[24 + j]), then the
				// lanes pairwise).
				for (int i = threadIdx.x; i < nblk * nt; i += 4 * kGemvRows)
				{
					const int b = i % nblk, t = i / nblk;
					float sum;
					if (p.xsum)
						sum = p.xsum[t * p.xsum_stride + b0 + b];
					else
					{
						const float4* x4 = reinterpret_cast<const float4*>(p.x + t * p.x_stride + 32 * (b0 + b));
						float x[32];
#pragma unroll
						for (int u = 0; u < 8; ++u)
						{
							const float4 v = x4[u];
							x[4 * u] = v.x;
							x[4 * u + 1] = v.y;
							x[4 * u + 2] = v.z;
							x[4 * u + 3] = v.w;
						}
						float l[8];
#pragma unroll
						for (int j = 0; j < 8; ++j) l[j] = (x[j] + x[8 + j]) + (x[16 + j] + x[24 + j]);
						sum = ((l[0] + l[4]) + (l[1] + l[5])) + ((l[2] + l[6]) + (l[3] + l[7]));
					}
					s_xs[b * nt + t] = sum;
				}
			}
			if constexpr (F != kGemvBf16)
			{
				// The work-group's rows' scales (and biases) of the range, [block][row], so
				// a lane reads its four rows with one 8-byte read.
				for (int i = threadIdx.x; i < nblk * kGemvRows; i += 4 * kGemvRows)
				{
					const int r = i / nblk, b = i % nblk;
					const int sr = min(blockIdx.x * kGemvRows + r, p.rows - 1); // stacked row (clamped; not used past the end)
					const mat_row sm = locate(p, sr);
					const size_t src = static_cast<size_t>(sm.r) * nb_all + b0 + b;
					s_sc[b * kGemvRows + r] = sm.m.scales[src];
					if constexpr (F == kGemvQ4S) s_bi[b * kGemvRows + r] = sm.m.biases[src];
				}
			}
			__syncthreads();

			f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, acc_b = {0.0f, 0.0f, 0.0f, 0.0f};
			const bf16x8 zero8 = as_bf16x8(u32x4{0u, 0u, 0u, 0u});
			for (int i0 = 0; i0 < n_mine; i0 += NA)
			{
#pragma unroll
				for (int j = 0; j < NA; ++j)
				{
					const int i = i0 + j;
					const int bl = my_block(i) - b0; // block within the range
					const bf16x8 a = a_operand<F>(ab[j]);
					// The next load into this slot, kAhead blocks on (clamped: a
					// load is never under a branch); BF16 has all of its loads out.
					if constexpr (F != kGemvBf16)
						ab[j] = load_a<F>(mr.m.w, p.cols, ra, min(my_block(i + kAhead<F>), nb_all - 1), grp);
					if (i < n_mine) // uniform
					{
						const size_t at = (static_cast<size_t>(bl) * nt + col) * 32 + 8 * grp;
						const bf16x8 xh = col < nt ? *reinterpret_cast<const bf16x8*>(s_xh + at) : zero8;
						const bf16x8 xl = col < nt ? *reinterpret_cast<const bf16x8*>(s_xl + at) : zero8;
						if constexpr (F == kGemvBf16)
						{
							acc = mfma16x16x32(a, xh, acc);
							acc = mfma16x16x32(a, xl, acc);
						}
						else
						{
							f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
							d = mfma16x16x32(a, xh, d);
							d = mfma16x16x32(a, xl, d);
							const u32x2 sc = *reinterpret_cast<const u32x2*>(s_sc + bl * kGemvRows + 16 * wave + 4 * grp);
							acc[0] = fmaf(bf16_lo(sc.x), d[0], acc[0]);
							acc[1] = fmaf(bf16_hi(sc.x), d[1], acc[1]);
							acc[2] = fmaf(bf16_lo(sc.y), d[2], acc[2]);
							acc[3] = fmaf(bf16_hi(sc.y), d[3], acc[3]);
							if constexpr (F == kGemvQ4S)
							{
								// The bias term: bias * (block sum of x).
								const u32x2 bi = *reinterpret_cast<const u32x2*>(s_bi + bl * kGemvRows + 16 * wave + 4 * grp);
								const float xs = col < nt ? s_xs[bl * nt + col] : 0.0f;
								acc_b[0] = fmaf(bf16_lo(bi.x), xs, acc_b[0]);
								acc_b[1] = fmaf(bf16_hi(bi.x), xs, acc_b[1]);
								acc_b[2] = fmaf(bf16_lo(bi.y), xs, acc_b[2]);
								acc_b[3] = fmaf(bf16_hi(bi.y), xs, acc_b[3]);
							}
						}
					}
				}
			}

			// Lane (grp, col) holds rows 4 grp + i of token col.
#pragma unroll
			for (int i = 0; i < 4; ++i)
			{
				const int r = 4 * grp + i, t = col;
				const float v = F == kGemvQ4S ? acc[i] + acc_b[i] : acc[i];
				if (r < m_rows && t < nt)
				{
					if (p.n_split == 1)
						mr.m.y[t * mr.m.y_stride + mr.r + r] = v;
					else
						p.part[(static_cast<size_t>(split) * nt + t) * p.rows + row0 + r] = v;
				}
			}
		}

		// ---- gemv_batch_kernel and gemv_tile_kernel ----
		//
		// X is split into bf16 hi + lo once per call (gemv_stage_x_kernel) and
		// the products go the other way round: A = X (16 vectors x 32 columns),
		// B = the rows' weights, so D holds vectors 4 (l / 16) + i of row
		// l % 16: a row's scale is one value per lane and Y's rows are
		// consecutive lanes. (512 vectors ran 16 at a time through gemv_kernel
		// before, the weights read 32 times over: 6144 x 2560 BF16 448 us, now
		// 47.)

		// 64 bytes of each of 16 weight rows per wavefront load (a "piece", 16
		// bytes per lane: row l % 16, bytes 16 (l / 16) ..): this many 32-column
		// blocks.
		template <int F>
		constexpr int kPieceBlocks = F == kGemvBf16 ? 1 : (F == kGemvQ8_0 ? 2 : 4);

		__device__ __forceinline__ u32x2 swap32(uint32_t a, uint32_t b)
		{
			const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
			return u32x2{r[0], r[1]};
		}
		__device__ __forceinline__ u32x2 swap16(uint32_t a, uint32_t b)
		{
			const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
			return u32x2{r[0], r[1]};
		}

		// The B operands (16 rows x 32 columns each) of a piece's blocks. The
		// columns that lane group g = l / 16 holds of a block (and so must hold
		// of X): BF16 8 g .. 8 g + 7; Q8_0 16 (g % 2) + 8 (g / 2) .. + 7; Q4_S
		// 4 g .. 4 g + 3 and 16 + 4 g .. + 3.
		template <int F>
		__device__ __forceinline__ void batch_operands(const u32x4& w, bf16x8 (&b)[kPieceBlocks<F>])
		{
			if constexpr (F == kGemvBf16)
				b[0] = as_bf16x8(w);
			else if constexpr (F == kGemvQ8_0)
			{
				// The piece holds block 0 in lane groups 0, 1 and block 1 in 2, 3:
				// exchanging halves gives each block to all four groups.
				const u32x2 d0 = swap32(w[0], w[2]), d1 = swap32(w[1], w[3]);
				b[0] = q8_to_bf16x8(d0.x, d1.x);
				b[1] = q8_to_bf16x8(d0.y, d1.y);
			}
			else
			{
				// Lane group g holds block g's four dwords; block j wants dword g
				// in group g: a 4 x 4 transpose.
				const u32x2 s02 = swap32(w[0], w[2]), s13 = swap32(w[1], w[3]);
				const u32x2 b01 = swap16(s02.x, s13.x), b23 = swap16(s02.y, s13.y);
				b[0] = q4_to_bf16x8(b01.x);
				b[1] = q4_to_bf16x8(b01.y);
				b[2] = q4_to_bf16x8(b23.x);
				b[3] = q4_to_bf16x8(b23.y);
			}
		}

		// The sum of a block's 32 x on every lane of a vector (lane l: vector
		// l % 16, x[0..3] columns 4 g .. and x[4..7] columns 16 + 4 g .., g =
		// l / 16), added as the reference does (reference nn_ops.cpp:1305-1316
		// under its -ffast-math build: l_j = (x_j + x_8+j) + (x_16+j + x_24+j),
		// then ((l0 + l4) + (l1 + l5)) + ((l2 + l6) + (l3 + l7))).
		__device__ __forceinline__ float batch_block_sum(const float (&x)[8])
		{
			float u[4];
#pragma unroll
			for (int j = 0; j < 4; ++j)
				u[j] = add_with_other_row(add_with_other_half(x[j]) + add_with_other_half(x[4 + j]));
			return (u[0] + u[1]) + (u[2] + u[3]);
		}

		// The first of a lane's columns in a block, and where its second four are.
		template <int F>
		__device__ __forceinline__ int x_first_col(int grp)
		{
			return F == kGemvBf16 ? 8 * grp : (F == kGemvQ8_0 ? 16 * (grp & 1) + 8 * (grp >> 1) : 4 * grp);
		}
		template <int F>
		constexpr int kXSecond = F == kGemvQ4S ? 16 : 4;

		// X^T of a 32-column block and a tile of 16 vectors as the A operand (lane
		// l: vector l % 16, its columns of the block), split into bf16 hi + lo,
		// from the lane's eight values as loaded.
		__device__ __forceinline__ void x_operands(const u32x4& a, const u32x4& b, bf16x8& hi, bf16x8& lo)
		{
			const float4 f = __builtin_bit_cast(float4, a), g = __builtin_bit_cast(float4, b);
			const float o[8] = {f.x, f.y, f.z, f.w, g.x, g.y, g.z, g.w};
			split_bf16x8(o, hi, lo);
		}

		// X of a whole call as operands in memory (p.xs, written by
		// gemv_stage_x_kernel): per (block, tile of 16 vectors) 1 KB of hi and
		// 1 KB of lo in lane order, so a wavefront's load is 1 KB of consecutive
		// addresses, where the vectors themselves lie cols * 4 bytes apart (16
		// lines per load, for many widths on one L2 channel). For Q4_S then the
		// block sums as operands of a product over blocks: per (32 blocks,
		// tile) 1 KB each of hi, mid and lo, the three bf16 that hold a sum's
		// 24 bits (lane l: vector l % 16, blocks 8 (l / 16) .. + 7).
		__device__ __forceinline__ u32x4* x_staged(const gemv_params& p, int blk, int tile)
		{
			return static_cast<u32x4*>(p.xs) + (static_cast<size_t>(blk) * p.x_tiles + tile) * 128;
		}
		// A descriptor of the staged X from block blk on, to its end (at most
		// kGemvStagedMax bytes).
		__device__ __forceinline__ __amdgpu_buffer_rsrc_t x_from(const gemv_params& p, int blk)
		{
			return __builtin_amdgcn_make_buffer_rsrc(x_staged(p, blk, 0), 0, (p.cols / 32 - blk) * p.x_tiles * 2048, 0x00020000);
		}
		__device__ __forceinline__ uint16_t* x_sums(const gemv_params& p, int step, int tile)
		{
			const size_t n = static_cast<size_t>(p.cols / 32) * p.x_tiles;
			return reinterpret_cast<uint16_t*>(static_cast<u32x4*>(p.xs) + n * 128) +
			       (static_cast<size_t>(step) * p.x_tiles + tile) * 1536;
		}

		// One wavefront per (block, tile); Q4_S: also the blocks that fill up the
		// last 32 (sums of zero). Vectors past the last one repeat it.
		template <int F>
		__global__ __launch_bounds__(256) void gemv_stage_x_kernel(const gemv_params p)
		{
			const int lane = threadIdx.x & 63, item = blockIdx.x * 4 + (threadIdx.x >> 6);
			const int nb = p.cols / 32, blk = item / p.x_tiles, tile = item % p.x_tiles;
			if (blk >= (F == kGemvQ4S ? (nb + 31) & ~31 : nb)) return; // the whole wavefront
			const int t = min(16 * tile + (lane & 15), p.n_batch - 1);
			const float* x = p.x + static_cast<size_t>(t) * p.x_stride + 32 * min(blk, nb - 1) + x_first_col<F>(lane >> 4);
			const u32x4 a = *reinterpret_cast<const u32x4*>(x), b = *reinterpret_cast<const u32x4*>(x + kXSecond<F>);
			if (blk < nb)
			{
				bf16x8 hi, lo;
				x_operands(a, b, hi, lo);
				u32x4* o = x_staged(p, blk, tile) + lane;
				o[0] = __builtin_bit_cast(u32x4, hi);
				o[64] = __builtin_bit_cast(u32x4, lo);
			}
			if constexpr (F == kGemvQ4S)
			{
				const float4 f = __builtin_bit_cast(float4, a), g = __builtin_bit_cast(float4, b);
				const float v[8] = {f.x, f.y, f.z, f.w, g.x, g.y, g.z, g.w};
				float s = batch_block_sum(v);
				if (blk >= nb)
					s = 0.0f;
				else if (p.xsum)
					s = p.xsum[static_cast<size_t>(t) * p.xsum_stride + blk];
				if (lane < 16)
				{
					uint16_t* o = x_sums(p, blk >> 5, tile) + (lane + 16 * ((blk & 31) >> 3)) * 8 + (blk & 7);
					// (the first part at most the largest finite bf16; an infinite
					// sum or NaN is every part)
					const float big = bf16_bits_to_f32(0x7f7f);
					const bool finite = fabsf(s) < INFINITY;
					if (s != s) s = __uint_as_float(0x7fc00000u); // (whose rounding stays NaN)
					const uint32_t h = f32_to_bf16_bits(finite ? fminf(fmaxf(s, -big), big) : s);
					const float r = finite ? s - bf16_bits_to_f32(h) : s;
					const uint32_t m = f32_to_bf16_bits(r);
					o[0] = static_cast<uint16_t>(h);
					o[512] = static_cast<uint16_t>(m);
					o[1024] = static_cast<uint16_t>(f32_to_bf16_bits(finite ? r - bf16_bits_to_f32(m) : s));
				}
			}
		}

		// 16 rows of each of RT tiles (rows past the last one repeat it; they are
		// not stored), read through one buffer descriptor per tile. A piece goes
		// to LDS by LDS-DMA with four lanes on each row's 64 bytes (row l / 4),
		// and comes back one 16-byte read per lane in the operand's order (row
		// l % 16): loads in that order straight to registers put 16 rows in each
		// quarter wavefront, 64 line lookups per KB, and held a CU to 16 bytes
		// per clock whatever their depth. The 16-byte slots of a row are XORed
		// with row / 4, so a quarter wavefront's reads fall on distinct banks.
		// What lies past a row's end or the wavefront's pieces is loaded from an
		// offset past the descriptor's, which gives zeros without a memory
		// access, so no load (and no product) is under a branch: the counts of
		// loads in flight stay exact.
		constexpr uint32_t kDeadOffset = 0x80000000u;
		template <int F, int RT>
		struct batch_rows
		{
			__amdgpu_buffer_rsrc_t w[RT], sc[RT];
			uint32_t off[RT], s_off[RT]; // this lane's row and its 16 bytes of a piece; its scale
			const uint16_t* bi[RT];
			int nb;
			uint32_t row_bytes, lane_bytes;
			__device__ __forceinline__ batch_rows(const gemv_params& p, int row0)
			{
				const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
				nb = p.cols / 32;
				row_bytes = static_cast<uint32_t>(nb) * (64 / kPieceBlocks<F>);
				lane_bytes = 16u * ((lane & 3) ^ grp);
#pragma unroll
				for (int r = 0; r < RT; ++r)
				{
					const int t0 = min(row0 + 16 * r, (p.rows - 1) & ~15), n = min(16, p.rows - t0);
					const mat_row mr = locate(p, t0);
					w[r] = __builtin_amdgcn_make_buffer_rsrc(
						const_cast<char*>(static_cast<const char*>(mr.m.w) + static_cast<size_t>(mr.r) * row_bytes), 0,
						static_cast<int>(n * row_bytes), 0x00020000);
					off[r] = static_cast<uint32_t>(min(lane >> 2, n - 1)) * row_bytes + lane_bytes;
					const uint32_t row = min(col, n - 1);
					if constexpr (F != kGemvBf16)
					{
						sc[r] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(mr.m.scales + static_cast<size_t>(mr.r) * nb),
						                                          0, n * nb * 2, 0x00020000);
						s_off[r] = (row * nb + (grp & (kPieceBlocks<F> - 1))) * 2;
					}
					bi[r] = F == kGemvQ4S ? mr.m.biases + (static_cast<size_t>(mr.r) + row) * nb : nullptr;
				}
			}
			// Piece i of tile r into 1 KB of LDS if it is one of the caller's
			// (below end), and the scale of block (l / 16) % kPieceBlocks of it.
			__device__ __forceinline__ void load(unsigned char* dst, uint32_t& scale, int r, int i, int end) const
			{
				const bool live = i < end && 64u * i + lane_bytes < row_bytes;
				dma_lds16(w[r], dst, live ? off[r] + 64u * i : kDeadOffset, 0);
				if constexpr (F != kGemvBf16)
				{
					const int grp = (threadIdx.x & 63) >> 4;
					const bool ok = i < end && kPieceBlocks<F> * i + (grp & (kPieceBlocks<F> - 1)) < nb;
					scale = __builtin_amdgcn_raw_buffer_load_b16(sc[r], ok ? s_off[r] + 2u * kPieceBlocks<F> * i : kDeadOffset, 0, 0);
				}
			}
			// The piece's 16 bytes of row l % 16, quarter l / 16.
			static __device__ __forceinline__ u32x4 read(const unsigned char* piece)
			{
				const int col = threadIdx.x & 15, grp = (threadIdx.x & 63) >> 4;
				return *reinterpret_cast<const u32x4*>(piece + 64 * col + 16 * (grp ^ (col >> 2)));
			}
		};

		// A piece's scales, each on every lane, from load()'s.
		template <int F>
		__device__ __forceinline__ void batch_scales(uint32_t scale, float (&s)[4])
		{
			const uint32_t x = scale << 16;
			if constexpr (F == kGemvQ8_0)
			{
				const u32x2 v = swap16(x, x); // rows 0 1 0 1
				s[0] = __uint_as_float(v.x);
				s[1] = __uint_as_float(v.y);
			}
			else if constexpr (F == kGemvQ4S)
			{
				const u32x2 h = swap32(x, x); // rows 0 1 0 1, rows 2 3 2 3
				const u32x2 lo = swap16(h.x, h.x), hi = swap16(h.y, h.y);
				s[0] = __uint_as_float(lo.x);
				s[1] = __uint_as_float(lo.y);
				s[2] = __uint_as_float(hi.x);
				s[3] = __uint_as_float(hi.y);
			}
		}

		// acc += one block's products of a 16-row tile and a 16-vector tile.
		template <int F>
		__device__ __forceinline__ void batch_product(f32x4& acc, const bf16x8& xh, const bf16x8& xl, const bf16x8& w, float s)
		{
			if constexpr (F == kGemvBf16)
			{
				acc = mfma16x16x32(xh, w, acc);
				acc = mfma16x16x32(xl, w, acc);
			}
			else
			{
				f32x4 d = mfma16x16x32(xh, w, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
				d = mfma16x16x32(xl, w, d);
#pragma unroll
				for (int i = 0; i < 4; ++i) acc[i] = fmaf(s, d[i], acc[i]);
			}
		}

		// s_waitcnt vmcnt(n), the other counters not waited on (gfx9 encoding:
		// vmcnt[3:0], expcnt[6:4] = 7, lgkmcnt[11:8] = 0xf, vmcnt[5:4] at
		// bits 15:14). Nothing is scheduled across it.
		template <int N>
		__device__ __forceinline__ void wait_loads()
		{
			static_assert(N < 64, "vmcnt");
			__builtin_amdgcn_sched_barrier(0);
			__builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
			__builtin_amdgcn_sched_barrier(0);
		}

		// Eight biases of a row from block b0 on as a B operand (zero past the
		// row's end).
		__device__ __forceinline__ bf16x8 bias_operand(const uint16_t* bi, int b0, int nb)
		{
			uint32_t h[8];
#pragma unroll
			for (int i = 0; i < 8; ++i)
			{
				const uint32_t v = bi[min(b0 + i, nb - 1)];
				h[i] = b0 + i < nb ? v : 0u;
			}
			return as_bf16x8(u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)});
		}

		constexpr int kBatchWaves = 8;
		// Y[t][r] for 16 RT rows per work-group and TT = p.x_tiles tiles of 16
		// vectors (every tile that is read is staged), W streamed once. The wavefronts split the columns (contiguous runs of
		// whole pieces, the same whatever RT and the number of rows, so a row
		// gets the same bits in any group) and run without a barrier until
		// their sums meet in LDS, added in wavefront order: no K splits over
		// work-groups, no partials in memory and no second launch. A = X (16
		// vectors x 32 columns, bf16 hi + lo), B = the rows' weights, so D holds
		// vectors 4 (l / 16) + i of row l % 16: a row's scale is one value per
		// lane, and Y's rows are consecutive lanes. X comes as operands
		// (gemv_stage_x_kernel). Bound by latency at small sizes and by the
		// wavefronts' short lives at large ones, so one piece at a time and many
		// wavefronts: rings of 2, 4 and 6 pieces ran 16 vectors of 6144 x 2560
		// (BF16 / Q8_0 / Q4_S) in 14.2 / 13.2 / 14.3, 14.7 / 16.0 / 23.1 and 15.0 /
		// 15.0 / - us against 13.0 / 12.4 / 13.2, and 16 wavefronts in 14.8 / 13.2 /
		// 13.5.
		template <int F, int RT, int TT>
		__global__ __launch_bounds__(64 * kBatchWaves) void gemv_batch_kernel(const gemv_params p)
		{
			constexpr int PB = kPieceBlocks<F>;
			extern __shared__ __attribute__((aligned(16))) unsigned char s_raw[];
			const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
			const int grp = lane >> 4;
			const int nb = p.cols / 32, np = (nb + PB - 1) / PB;
			const int i_lo = wave * np / kBatchWaves, i_hi = (wave + 1) * np / kBatchWaves;
			const int row0 = blockIdx.x * 16 * RT;
			const batch_rows<F, RT> rows(p, row0);
			unsigned char* const s_w = s_raw + wave * RT * 1024; // [RT] pieces of this wavefront

			u32x4 xh[PB][TT], xl[PB][TT];
			uint32_t scale[RT];
			const uint32_t xs_block = static_cast<uint32_t>(p.x_tiles) * 2048u;
			const __amdgpu_buffer_rsrc_t rx = x_from(p, min(i_lo * PB, nb - 1));
			auto load = [&](int i) __attribute__((always_inline))
			{
#pragma unroll
				for (int j = 0; j < PB; ++j)
				{
					const int b = i * PB + j;
					const bool live = i < i_hi && b < nb; // uniform
					const uint32_t o = live ? (b - i_lo * PB) * xs_block + 16u * lane : kDeadOffset;
#pragma unroll
					for (int t = 0; t < TT; ++t)
					{
						xh[j][t] = __builtin_amdgcn_raw_buffer_load_b128(rx, o, 2048 * t, 0);
						xl[j][t] = __builtin_amdgcn_raw_buffer_load_b128(rx, o, 2048 * t + 1024, 0);
					}
				}
#pragma unroll
				for (int r = 0; r < RT; ++r) rows.load(s_w + r * 1024, scale[r], r, i, i_hi);
			};

			f32x4 acc[RT][TT];
#pragma unroll
			for (int r = 0; r < RT; ++r)
#pragma unroll
				for (int t = 0; t < TT; ++t) acc[r][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

			load(i_lo);
			for (int i = i_lo; i < i_hi; ++i)
			{
				wait_loads<0>();
				bf16x8 wb[RT][PB];
				float sc[RT][4];
#pragma unroll
				for (int r = 0; r < RT; ++r)
				{
					batch_operands<F>(rows.read(s_w + r * 1024), wb[r]);
					batch_scales<F>(scale[r], sc[r]);
				}
#pragma unroll
				for (int j = 0; j < PB; ++j)
#pragma unroll
					for (int t = 0; t < TT; ++t)
#pragma unroll
						for (int r = 0; r < RT; ++r)
							batch_product<F>(acc[r][t], as_bf16x8(xh[j][t]), as_bf16x8(xl[j][t]), wb[r][j], sc[r][j]);
				// (the piece's LDS reads have returned: the products took them)
				__builtin_amdgcn_sched_barrier(0);
				load(i + 1);
				__builtin_amdgcn_sched_barrier(0);
			}
			wait_loads<0>(); // (zeros on their way to LDS)
			__syncthreads(); // the sums take the pieces' place
			f32x4* s_sum = reinterpret_cast<f32x4*>(s_raw); // [wavefront][RT][TT][64]
			if constexpr (F == kGemvQ4S)
			{
				// The bias term, bias . (block sums of x), 32 blocks per product,
				// the products in turn over the wavefronts.
				for (int st = wave; st < (nb + 31) / 32; st += kBatchWaves)
#pragma unroll
					for (int r = 0; r < RT; ++r)
					{
						const bf16x8 b = bias_operand(rows.bi[r], 32 * st + 8 * grp, nb);
#pragma unroll
						for (int t = 0; t < TT; ++t)
						{
							const u32x4* xs = reinterpret_cast<const u32x4*>(x_sums(p, st, t)) + lane;
#pragma unroll
							for (int i = 2; i >= 0; --i) acc[r][t] = mfma16x16x32(as_bf16x8(xs[64 * i]), b, acc[r][t]);
						}
					}
			}

#pragma unroll
			for (int r = 0; r < RT; ++r)
#pragma unroll
				for (int t = 0; t < TT; ++t) s_sum[((wave * RT + r) * TT + t) * 64 + lane] = acc[r][t];
			__syncthreads();
			const float* s_f = reinterpret_cast<const float*>(s_raw);
			for (int i = threadIdx.x; i < RT * TT * 256; i += 64 * kBatchWaves)
			{
				const int rl = i & 15, tl = (i >> 4) & 15, tile = i >> 8; // tile = r * TT + t
				const int row = row0 + 16 * (tile / TT) + rl, tok = 16 * (tile % TT) + tl;
				const float* f = s_f + tile * 256 + 4 * (rl + 16 * (tl >> 2)) + (tl & 3);
				float v[kBatchWaves], sum = 0.0f;
#pragma unroll
				for (int w = 0; w < kBatchWaves; ++w) v[w] = f[w * RT * TT * 256];
#pragma unroll
				for (int w = 0; w < kBatchWaves; ++w) sum = w == 0 ? v[0] : sum + v[w];
				if (row < p.rows && tok < p.n_batch)
				{
					const mat_row mr = locate(p, row);
					mr.m.y[tok * mr.m.y_stride + mr.r] = sum;
				}
			}
		}

		// ---- many vectors: gemv_tile_kernel ----

		// Y of 16 RT WR rows and 16 TT vectors per work-group: WR groups of 16 RT
		// rows for each of two groups over the columns, one wavefront each. X's
		// operands arrive in LDS by LDS-DMA as they lie staged, one block a
		// slot, in a ring of SLOTS slots per column group, shared by the row
		// groups; a wavefront's own weights in a ring of NPW pieces. The column
		// groups' sums meet in LDS at the end. Work-groups of one row tile run
		// on one XCD, so a weight comes from HBM once and from that XCD's L2 for
		// the other vectors.
		template <int F, int RT, int TT, int WR, int SLOTS, int NPW>
		struct tile_shape
		{
			static constexpr int PB = kPieceBlocks<F>;
			static constexpr int WB = NPW * PB; // blocks of W in flight
			static constexpr int U = SLOTS > WB ? SLOTS : WB; // blocks per loop pass (a multiple of both)
			static constexpr int kSlot = TT * 2048;
			static constexpr int DX = TT * 2 / WR; // X's DMAs per wavefront and block
			static constexpr int NW = RT * (F == kGemvBf16 ? 1 : 2); // weight and scale loads per piece
			static constexpr int kLdsX = 2 * SLOTS * kSlot;
			static constexpr int kLds = kLdsX + 2 * WR * NPW * RT * 1024;
			static_assert(TT * 2 % WR == 0 && (U == 2 || U == 4 || U == 8) && U % SLOTS == 0 && U % WB == 0, "tile shape");
			static_assert(WR * RT * TT * 1024 <= kLds, "the sums reuse the rings");
			// Loads a wavefront may have in flight at the top of block j with X
			// and W of block j landed: those asked for after both. Block b asks
			// for X of block b + SLOTS - 1 at its top, and at its end, if it is
			// a piece's last, for the piece WB blocks on.
			static constexpr int in_flight(int j)
			{
				int n = 0, since = 0; // since the later of the two
				for (int b = j - 2 * U; b < j; ++b)
				{
					n += DX;
					if (b + SLOTS - 1 == j) since = n;
					if ((b + 4 * U + 1) % PB == 0)
					{
						n += NW;
						const int first = b + 1 - PB + WB;
						if (first <= j && j < first + PB) since = n;
					}
				}
				return n - since;
			}
		};

		template <int F, int RT, int TT, int WR, int SLOTS, int NPW>
		__global__ __launch_bounds__(128 * WR) void gemv_tile_kernel(const gemv_params p)
		{
			using S = tile_shape<F, RT, TT, WR, SLOTS, NPW>;
			constexpr int PB = S::PB, U = S::U, WB = S::WB;
			extern __shared__ __attribute__((aligned(16))) unsigned char s_raw[];
			const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
			const int col = lane & 15, grp = lane >> 4;
			const int wr = wave % WR, kg = wave / WR;
			const int nb = p.cols / 32;
			const int n_tt = (p.x_tiles + TT - 1) / TT, n_rt = (p.rows + 16 * RT * WR - 1) / (16 * RT * WR);
			// (row tile, vector tile): the vector tiles of a row tile consecutive on one XCD
			int rt, tt;
			{
				const int xcd = blockIdx.x & 7, i = blockIdx.x >> 3;
				rt = 8 * (i / n_tt) + xcd;
				tt = i % n_tt;
			}
			if (rt >= n_rt) return; // the whole work-group
			const int row0 = (rt * WR + wr) * 16 * RT;
			const batch_rows<F, RT> rows(p, row0);

			// Column group kg takes blocks b_lo .. b_lo + h - 1 (whole pieces),
			// as far as there are any.
			const int np = (nb + PB - 1) / PB, h = (np + 1) / 2 * PB;
			const int b_lo = kg * h, p_hi = min(np, (kg + 1) * (h / PB));

			const uint32_t xs_block = static_cast<uint32_t>(p.x_tiles) * 2048u;
			const __amdgpu_buffer_rsrc_t rx = x_from(p, min(b_lo, nb - 1));
			unsigned char* const s_x = s_raw + kg * SLOTS * S::kSlot;
			unsigned char* const s_w = s_raw + S::kLdsX + wave * NPW * RT * 1024; // [NPW][RT] pieces of this wavefront
			uint32_t x_off[S::DX]; // DMA u: 1 KB (hi or lo of a tile) to its place [tile][hi, lo] in the slot
#pragma unroll
			for (int u = 0; u < S::DX; ++u)
			{
				const int e = u * WR + wr;
				x_off[u] = 2048u * min(tt * TT + e / 2, p.x_tiles - 1) + 1024u * (e & 1) + 16u * lane;
			}
			// X of block i of the group into slot i % SLOTS.
			auto load_x = [&](int i, int slot) __attribute__((always_inline))
			{
				const bool live = i < h && b_lo + i < nb; // uniform
#pragma unroll
				for (int u = 0; u < S::DX; ++u)
					dma_lds16(rx, s_x + slot * S::kSlot + 1024 * (u * WR + wr), live ? x_off[u] : kDeadOffset,
					          live ? i * xs_block : 0u);
			};
			uint32_t scale[NPW][RT];
			f32x4 acc[RT][TT];
#pragma unroll
			for (int r = 0; r < RT; ++r)
#pragma unroll
				for (int t = 0; t < TT; ++t) acc[r][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

			// The loop's order of loads, begun before its first block.
#pragma unroll
			for (int b = -U; b < 0; ++b)
			{
				if (b >= 1 - SLOTS) load_x(b + SLOTS - 1, (b + SLOTS - 1) % SLOTS);
				__builtin_amdgcn_sched_barrier(0);
				if (b >= -WB && (b + WB + 1) % PB == 0)
				{
					const int q = (b + WB) / PB; // the piece's slot, and its number in the group
#pragma unroll
					for (int r = 0; r < RT; ++r) rows.load(s_w + (q * RT + r) * 1024, scale[q][r], r, b_lo / PB + q, p_hi);
				}
				__builtin_amdgcn_sched_barrier(0);
			}
			for (int i0 = 0; i0 < h; i0 += U)
			{
				auto block = [&](auto j_tag) __attribute__((always_inline))
				{
					constexpr int j = decltype(j_tag)::value, q = (j % WB) / PB;
					wait_loads<S::in_flight(j)>();
					// Everyone's X of block j, and everyone is done with the slot
					// reused next (its reads have returned: the products took
					// them). The bare barrier: __syncthreads() would wait for
					// the loads in flight.
					__builtin_amdgcn_s_barrier();
					__builtin_amdgcn_sched_barrier(0);
					load_x(i0 + j + SLOTS - 1, (j + SLOTS - 1) % SLOTS);
					__builtin_amdgcn_sched_barrier(0);
					u32x4 wv[RT];
#pragma unroll
					for (int r = 0; r < RT; ++r) wv[r] = rows.read(s_w + (q * RT + r) * 1024);
					const u32x4* xs = reinterpret_cast<const u32x4*>(s_x + (j % SLOTS) * S::kSlot) + lane;
					bf16x8 xh[TT], xl[TT];
#pragma unroll
					for (int t = 0; t < TT; ++t)
					{
						xh[t] = as_bf16x8(xs[t * 128]);
						xl[t] = as_bf16x8(xs[t * 128 + 64]);
					}
					__builtin_amdgcn_sched_barrier(0);
					bf16x8 wb[RT];
					float sb[RT];
#pragma unroll
					for (int r = 0; r < RT; ++r)
					{
						bf16x8 all[PB];
						float sc[4];
						batch_operands<F>(wv[r], all);
						batch_scales<F>(scale[q][r], sc);
						wb[r] = all[j % PB];
						sb[r] = sc[j % PB];
					}
#pragma unroll
					for (int t = 0; t < TT; ++t)
#pragma unroll
						for (int r = 0; r < RT; ++r) batch_product<F>(acc[r][t], xh[t], xl[t], wb[r], sb[r]);
					__builtin_amdgcn_sched_barrier(0);
					if constexpr ((j + 1) % PB == 0)
					{
#pragma unroll
						for (int r = 0; r < RT; ++r)
							rows.load(s_w + (q * RT + r) * 1024, scale[q][r], r, (b_lo + i0 + j + 1 - PB + WB) / PB, p_hi);
					}
					__builtin_amdgcn_sched_barrier(0);
				};
				block(std::integral_constant<int, 0>{});
				block(std::integral_constant<int, 1>{});
				if constexpr (U >= 4)
				{
					block(std::integral_constant<int, 2>{});
					block(std::integral_constant<int, 3>{});
				}
				if constexpr (U == 8)
				{
					block(std::integral_constant<int, 4>{});
					block(std::integral_constant<int, 5>{});
					block(std::integral_constant<int, 6>{});
					block(std::integral_constant<int, 7>{});
				}
			}
			if constexpr (F == kGemvQ4S)
			{
				for (int st = kg; st < (nb + 31) / 32; st += 2)
#pragma unroll
					for (int r = 0; r < RT; ++r)
					{
						const bf16x8 b = bias_operand(rows.bi[r], 32 * st + 8 * grp, nb);
#pragma unroll
						for (int t = 0; t < TT; ++t)
						{
							const u32x4* xs = reinterpret_cast<const u32x4*>(
								                  x_sums(p, st, min(tt * TT + t, p.x_tiles - 1))) + lane;
#pragma unroll
							for (int i = 2; i >= 0; --i) acc[r][t] = mfma16x16x32(as_bf16x8(xs[64 * i]), b, acc[r][t]);
						}
					}
			}

			// (the blocks after the last are in flight, as zeros, into LDS)
			wait_loads<0>();
			__syncthreads();
			f32x4* s_sum = reinterpret_cast<f32x4*>(s_raw) + wr * RT * TT * 64 + lane;
			if (kg == 1)
			{
#pragma unroll
				for (int r = 0; r < RT; ++r)
#pragma unroll
					for (int t = 0; t < TT; ++t) s_sum[(r * TT + t) * 64] = acc[r][t];
			}
			__syncthreads();
			if (kg == 0)
			{
#pragma unroll
				for (int r = 0; r < RT; ++r)
				{
					const int row = row0 + 16 * r + col;
					if (row >= p.rows) continue;
					const mat_row mr = locate(p, row);
#pragma unroll
					for (int t = 0; t < TT; ++t)
					{
						const f32x4 v = acc[r][t] + s_sum[(r * TT + t) * 64];
#pragma unroll
						for (int i = 0; i < 4; ++i)
						{
							const int tok = (tt * TT + t) * 16 + 4 * grp + i;
							if (tok < p.n_batch) mr.m.y[tok * mr.m.y_stride + mr.r] = v[i];
						}
					}
				}
			}
		}

		// One activation vector (the decode gemv) on the VALU: every load is 16
		// contiguous bytes of a weight row (a wavefront reads 1 KB of one row
		// per instruction), x sits in LDS, and each wavefront streams pairs of
		// rows with kVecAhead<F> loads in flight across row boundaries; a row's
		// lane sums meet through DPP and lane swaps.
		template <int F>
		struct vec_shape
		{
			static constexpr int CPL = F == kGemvBf16 ? 8 : (F == kGemvQ8_0 ? 16 : 32); // columns per lane per load
			static constexpr int CW = 64 * CPL; // columns per wavefront load
		};

		// Whether a row pair's last chunk is one item for both rows: when it is at
		// most half full, an item being as much work whatever its lanes hold
		// (Q4_S, 2560 columns: three items per pair instead of four; 19456 rows
		// 17.4 -> 14.9 us per launch of a graph, with the byte masks of vec_dot).
		// Only Q4_S, whose VALU work bounds it: Q8_0 was no faster with it (17.3 ->
		// 17.7 us).
		template <int F>
		bool vec_joint(int cols)
		{
			constexpr int CW = vec_shape<F>::CW;
			return F == kGemvQ4S && (cols - 1) % CW < CW / 2;
		}

		template <int F>
		struct vec_item
		{
			u32x4 w; // 16 bytes of the row
			float sc, bi; // the block's scale (Q8_0, Q4_S) and bias (Q4_S)
		};

		// x in LDS for the one-vector kernels. Q4_S (a lane's 32 columns per
		// load, its reads 128 bytes apart in column order: 8-way bank
		// conflicts) keeps it in the order the lanes read it: the four
		// consecutive columns 4 g .. 4 g + 3 of lane l's CPL columns of a
		// CW-column chunk sit at chunk * CW + 256 g + 4 l, so each of a
		// wavefront's 16-byte LDS reads covers 1 KB of consecutive addresses
		// (Qwen3-4B layer, one vector: 58.3 -> 51.6 us), the chunks padded to
		// CW columns and the block sums after them. BF16 and Q8_0 keep column
		// order (the same layout measured no faster for BF16, 6 % slower for
		// Q8_0).
		template <int F>
		constexpr bool kVecLaneOrder = F == kGemvQ4S;

		template <int F>
		__host__ __device__ constexpr int vec_x_floats(int cols)
		{
			return kVecLaneOrder<F> ? (cols + vec_shape<F>::CW - 1) / vec_shape<F>::CW * vec_shape<F>::CW : cols;
		}

		// A lane's dot product of one item (16 bytes of a row at columns c0 ..,
		// those of lane `lane` of a chunk) with x in LDS.
		template <int F>
		__device__ __forceinline__ float vec_dot(const vec_item<F>& it, int c0, int lane, const float* s_x, int cols)
		{
			constexpr int CPL = vec_shape<F>::CPL;
			if (c0 >= cols) return 0.0f;
			// columns c0 + 4 g .. + 3 at xq + GS g
			constexpr int GS = kVecLaneOrder<F> ? 256 : 4;
			const float* xq = kVecLaneOrder<F> ? s_x + (c0 - lane * CPL) + 4 * lane : s_x + c0;
			if constexpr (F == kGemvBf16)
			{
				const float4 x0 = *reinterpret_cast<const float4*>(xq);
				const float4 x1 = *reinterpret_cast<const float4*>(xq + GS);
				float d = 0.0f;
				d = fmaf(bf16_lo(it.w[0]), x0.x, d);
				d = fmaf(bf16_hi(it.w[0]), x0.y, d);
				d = fmaf(bf16_lo(it.w[1]), x0.z, d);
				d = fmaf(bf16_hi(it.w[1]), x0.w, d);
				d = fmaf(bf16_lo(it.w[2]), x1.x, d);
				d = fmaf(bf16_hi(it.w[2]), x1.y, d);
				d = fmaf(bf16_lo(it.w[3]), x1.z, d);
				d = fmaf(bf16_hi(it.w[3]), x1.w, d);
				return d;
			}
			else if constexpr (F == kGemvQ8_0)
			{
				float d = 0.0f;
#pragma unroll
				for (int u = 0; u < 4; ++u)
				{
					const float4 x = *reinterpret_cast<const float4*>(xq + GS * u);
					const uint32_t b = it.w[u] ^ 0x80808080u; // q + 128 per byte
					d = fmaf(static_cast<float>(b & 0xffu) - 128.0f, x.x, d);
					d = fmaf(static_cast<float>((b >> 8) & 0xffu) - 128.0f, x.y, d);
					d = fmaf(static_cast<float>((b >> 16) & 0xffu) - 128.0f, x.z, d);
					d = fmaf(static_cast<float>(b >> 24) - 128.0f, x.w, d);
				}
				return it.sc * d;
			}
			else
			{
				// Byte i of the block: element i (low nibble), i + 16 (high).
				float d = 0.0f;
#pragma unroll
				for (int u = 0; u < 4; ++u)
				{
					const float4 xl = *reinterpret_cast<const float4*>(xq + GS * u); // columns 4 u ..
					const float4 xh = *reinterpret_cast<const float4*>(xq + GS * (4 + u)); // columns 16 + 4 u ..
					// (a byte per nibble: 19 instructions for eight weights with the
					// byte conversions, against 24 with a bit-field extract per
					// nibble, into which the compiler folds the masks unless it
					// cannot see them)
					uint32_t lo = it.w[u] & 0x0f0f0f0fu, hi = (it.w[u] >> 4) & 0x0f0f0f0fu;
					asm("" : "+v"(lo), "+v"(hi));
					d = fmaf(static_cast<float>(lo & 0xffu), xl.x, d);
					d = fmaf(static_cast<float>((lo >> 8) & 0xffu), xl.y, d);
					d = fmaf(static_cast<float>((lo >> 16) & 0xffu), xl.z, d);
					d = fmaf(static_cast<float>(lo >> 24), xl.w, d);
					d = fmaf(static_cast<float>(hi & 0xffu), xh.x, d);
					d = fmaf(static_cast<float>((hi >> 8) & 0xffu), xh.y, d);
					d = fmaf(static_cast<float>((hi >> 16) & 0xffu), xh.z, d);
					d = fmaf(static_cast<float>(hi >> 24), xh.w, d);
				}
				return fmaf(it.bi, s_x[vec_x_floats<F>(cols) + c0 / 32], it.sc * d);
			}
		}

		// 16 bytes of row r0 (second: r0 + 1) of matrix m at columns c0 ..
		// (lanes past the row's end re-read its last bytes; their sums are not
		// used), with the block's scale and bias.
		template <int F>
		__device__ __forceinline__ vec_item<F> vec_load(const gemv_mat& m, int r0, int second, int c0, int cols)
		{
			constexpr int CPL = vec_shape<F>::CPL;
			const int cc = min(c0, cols - CPL);
			vec_item<F> it;
			const size_t off = static_cast<size_t>(r0) * cols + (second ? cols : 0) + cc;
			if constexpr (F == kGemvBf16)
				it.w = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(m.w) + off);
			else if constexpr (F == kGemvQ8_0)
				it.w = *reinterpret_cast<const u32x4*>(static_cast<const int8_t*>(m.w) + off);
			else
				it.w = *reinterpret_cast<const u32x4*>(static_cast<const uint8_t*>(m.w) + off / 2);
			if constexpr (F != kGemvBf16)
			{
				const size_t si = static_cast<size_t>(r0) * (cols / 32) + (second ? cols / 32 : 0) + cc / 32;
				it.sc = bf16_bits_to_f32(m.scales[si]);
				if constexpr (F == kGemvQ4S) it.bi = bf16_bits_to_f32(m.biases[si]);
			}
			return it;
		}

		// x into LDS (in the lanes' order for Q4_S, vec_x_floats), and for Q4_S
		// its block sums after it; the caller's barrier follows. Thread t takes elements 4 t .. 4 t + 3
		// of each 1024. Q4_S without the caller's block sums: the eight threads
		// of a block hold its quarters q = t % 8, and three lane exchanges add
		// them in the reference's order (reference nn_ops.cpp:1305-1316 under
		// its -ffast-math build: l_j = (x_j + x_8+j) + (x_16+j + x_24+j), then
		// ((l0 + l4) + (l1 + l5)) + ((l2 + l6) + (l3 + l7))), so x is read once.
		template <int F>
		__device__ __forceinline__ void vec_stage_x(const gemv_params& p, float* s_x)
		{
			constexpr int CW = vec_shape<F>::CW, CPL = vec_shape<F>::CPL;
			const int nb_all = p.cols / 32;
			const int xs = vec_x_floats<F>(p.cols); // the block sums' offset
			const bool own_sums = F == kGemvQ4S && p.xsum == nullptr; // uniform
			for (int i0 = 0; i0 < p.cols; i0 += 1024)
			{
				const int i = i0 + 4 * threadIdx.x;
				const bool ok = i < p.cols; // a block's eight threads agree (cols % 32 == 0)
				const float4 v = ok ? *reinterpret_cast<const float4*>(p.x + i) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
				const int rem = i % CW; // lane rem / CPL, group (rem % CPL) / 4 of chunk i / CW
				const int dst = kVecLaneOrder<F> ? (i - rem) + 256 * ((rem % CPL) / 4) + 4 * (rem / CPL) : i;
				if (ok) *reinterpret_cast<float4*>(s_x + dst) = v;
				if (own_sums)
				{
					auto add_from = [](const float4& a, int m) __attribute__((always_inline)) -> float4
					{
						return make_float4(a.x + __shfl_xor(a.x, m), a.y + __shfl_xor(a.y, m), a.z + __shfl_xor(a.z, m),
						                   a.w + __shfl_xor(a.w, m));
					};
					const float4 a = add_from(v, 2); // q = 0: x_j + x_8+j; q = 4: x_16+j + x_24+j (j < 4)
					const float4 l = add_from(a, 4); // q = 0: l_0..3; q = 1: l_4..7
					const float4 u = add_from(l, 1); // q = 0: l_k + l_k+4
					if (ok && (threadIdx.x & 7) == 0) s_x[xs + i / 32] = (u.x + u.y) + (u.z + u.w);
				}
			}
			if (F == kGemvQ4S && !own_sums)
				for (int b = threadIdx.x; b < nb_all; b += 256) s_x[xs + b] = p.xsum[b];
		}

		// The argmax order: (v, r) beats (bv, br) when v is above -inf (NaN never
		// is) and larger, or equal with a smaller row; br = -1 is "none". The
		// smallest row of the largest value wins whatever order rows are met in.
		__device__ __forceinline__ bool argmax_better(float v, int r, float bv, int br)
		{
			return r >= 0 && v > -INFINITY && (br < 0 || v > bv || (v == bv && r < br));
		}

		// ARGMAX (BF16 only): no y; each wavefront keeps its best row and the
		// work-group writes its best (value, row) to p.best[blockIdx.x].
		// JOINT: vec_joint.
		template <int F, bool ARGMAX = false, bool JOINT = false>
		__global__ __launch_bounds__(256) void gemv_vec_kernel(const gemv_params p)
		{
			static_assert(!ARGMAX || F == kGemvBf16, "argmax of a BF16 gemv only");
			using V = vec_shape<F>;
			constexpr int CPL = V::CPL, CW = V::CW, NA = kVecAhead<F>;
			extern __shared__ __attribute__((aligned(16))) float s_x[]; // x, then (Q4_S) its block sums
			// (wave uniform: every row index below, and the matrix lookup, stays scalar)
			const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

			// Items: for each of this wavefront's row pairs, chunk c of row 0,
			// then of row 1, for every chunk c of CW columns; where the last
			// chunk is at most half full (JOINT), one item for both rows, row
			// 1's in the upper half of the lanes. Two cursors walk
			// them, the loads' (kVecAhead<F> ahead) and the sums': (pair, item within
			// the pair), stepped by one item at a time (no division per item);
			// a pair's matrix is looked up when the load cursor enters it.
			const int nch = (p.cols + CW - 1) / CW;
			const int per_pair = 2 * nch - JOINT;
			const int gw = blockIdx.x * 4 + wave, n_gw = gridDim.x * 4;
			const int n_pairs = (p.rows + 1) / 2;
			const int my_pairs = gw < n_pairs ? (n_pairs - 1 - gw) / n_gw + 1 : 0;
			const int n_items = my_pairs * per_pair;
			// (A wavefront without rows still takes part in staging x.)
			int l_pi = 0, l_rem = 0; // the next load's pair and item
			gemv_mat l_m = p.mats[0];
			int l_r0 = 0, l_two = 0; // the pair's first row in its matrix; whether it has a second row
			auto enter_pair = [&]() __attribute__((always_inline))
			{
				const int row0 = 2 * (gw + min(l_pi, max(my_pairs - 1, 0)) * n_gw);
				const mat_row mr = locate(p, min(row0, p.rows - 1));
				l_m = mr.m;
				l_r0 = mr.r;
				l_two = row0 + 1 < p.rows;
			};
			enter_pair();
			// The next item's load (past the wavefront's last item: its last item
			// again, so no load is under a branch), then the cursor steps on.
			auto load = [&]() __attribute__((always_inline)) -> vec_item<F>
			{
				const bool past = l_pi >= my_pairs;
				const int rem = past ? per_pair - 1 : l_rem;
				const bool both = JOINT && rem == per_pair - 1;
				const int sub = both ? lane & 31 : lane;
				const int row = both ? lane >> 5 : rem & 1;
				// (where an item holds one row its index stays scalar: as a lane's
				// selection Q8_0 took 18.5 us for 19456 x 2560 instead of 17.3)
				const vec_item<F> it = JOINT
					? vec_load<F>(l_m, l_r0, row & l_two, (rem >> 1) * CW + sub * CPL, p.cols)
					: vec_load<F>(l_m, l_r0 + ((rem & 1) & l_two), 0, (rem >> 1) * CW + lane * CPL, p.cols);
				if (!past && ++l_rem == per_pair)
				{
					l_rem = 0;
					++l_pi;
					if (l_pi < my_pairs) enter_pair();
				}
				return it;
			};

			// The first loads go out before x is staged.
			vec_item<F> ring[NA];
#pragma unroll
			for (int j = 0; j < NA; ++j) ring[j] = load();

			vec_stage_x<F>(p, s_x);
			__syncthreads();

			float acc[2] = {0.0f, 0.0f};
			float best_v = -INFINITY; // ARGMAX: this wavefront's best row so far (lane 0)
			int best_r = -1;
			int u_pi = 0, u_rem = 0; // the next sum's pair and item
			for (int k0 = 0; k0 < n_items; k0 += NA)
			{
#pragma unroll
				for (int j = 0; j < NA; ++j)
				{
					const int k = k0 + j;
					const vec_item<F> it = ring[j];
					ring[j] = load(); // past the end: a repeat, never under a branch
					if (k < n_items) // uniform
					{
						if constexpr (JOINT)
						{
							const bool both = u_rem == per_pair - 1;
							const int sub = both ? lane & 31 : lane;
							const float d = vec_dot<F>(it, (u_rem >> 1) * CW + sub * CPL, sub, s_x, p.cols);
							const bool second = both ? lane > 31 : (u_rem & 1) != 0;
							acc[0] += second ? 0.0f : d;
							acc[1] += second ? d : 0.0f;
						}
						else
							acc[j & 1] += vec_dot<F>(it, (u_rem >> 1) * CW + lane * CPL, lane, s_x, p.cols);
						if (u_rem == per_pair - 1) // the pair's last item: both rows are complete
						{
							const float y0 = wave_sum_dpp(acc[0]), y1 = wave_sum_dpp(acc[1]);
							const int r0 = 2 * (gw + u_pi * n_gw);
							if constexpr (ARGMAX)
							{
								if (r0 == 0 && lane == 0) p.argmax[1] = __builtin_isnan(y0);
								if (argmax_better(y0, r0, best_v, best_r))
								{
									best_v = y0;
									best_r = r0;
								}
								if (r0 + 1 < p.rows && argmax_better(y1, r0 + 1, best_v, best_r))
								{
									best_v = y1;
									best_r = r0 + 1;
								}
							}
							else if (lane == 0)
							{
								const mat_row mr = locate(p, r0); // the pair's matrix (pairs never span two)
								mr.m.y[mr.r] = y0;
								if (r0 + 1 < p.rows) mr.m.y[mr.r + 1] = y1;
							}
							acc[0] = acc[1] = 0.0f;
						}
						if (++u_rem == per_pair)
						{
							u_rem = 0;
							++u_pi;
						}
					}
				}
			}
			if constexpr (ARGMAX)
			{
				// The work-group's best: the four wavefronts' (lane 0's), after x
				// in LDS, then one (value, row) pair per work-group.
				float* s_best = s_x + vec_x_floats<F>(p.cols);
				if (lane == 0)
				{
					s_best[2 * wave] = best_v;
					s_best[2 * wave + 1] = __int_as_float(best_r);
				}
				__syncthreads();
				if (threadIdx.x == 0)
				{
					float bv = -INFINITY;
					int br = -1;
#pragma unroll
					for (int w = 0; w < 4; ++w)
					{
						const float wv = s_best[2 * w];
						const int wr = __float_as_int(s_best[2 * w + 1]);
						if (argmax_better(wv, wr, bv, br))
						{
							bv = wv;
							br = wr;
						}
					}
					p.best[blockIdx.x] = make_float2(bv, __int_as_float(br));
				}
			}
		}

		// The argmax over the work-groups' best pairs: one work-group of 256.
		__global__ __launch_bounds__(256) void gemv_argmax_final_kernel(const gemv_params p, int n_best)
		{
			__shared__ float s_v[256];
			__shared__ int s_r[256];
			float bv = -INFINITY;
			int br = -1;
			for (int i = threadIdx.x; i < n_best; i += 256)
			{
				const float2 b = p.best[i];
				if (argmax_better(b.x, __float_as_int(b.y), bv, br))
				{
					bv = b.x;
					br = __float_as_int(b.y);
				}
			}
			s_v[threadIdx.x] = bv;
			s_r[threadIdx.x] = br;
			__syncthreads();
			for (int h = 128; h > 0; h >>= 1)
			{
				if (static_cast<int>(threadIdx.x) < h && argmax_better(s_v[threadIdx.x + h], s_r[threadIdx.x + h], s_v[threadIdx.x],
				                                     s_r[threadIdx.x]))
				{
					s_v[threadIdx.x] = s_v[threadIdx.x + h];
					s_r[threadIdx.x] = s_r[threadIdx.x + h];
				}
				__syncthreads();
			}
			if (threadIdx.x == 0) p.argmax[0] = s_r[0] >= 0 && !(p.first_sticks && p.argmax[1]) ? s_r[0] : 0;
		}

		// The argmax's first pass over a float vector: each work-group's best
		// (value, row) pair; y[0]'s NaN flag.
		__global__ __launch_bounds__(256) void argmax_part_kernel(const gemv_params p)
		{
			__shared__ float s_v[256];
			__shared__ int s_r[256];
			float bv = -INFINITY;
			int br = -1;
			for (int i = blockIdx.x * 256 + threadIdx.x; i < p.rows; i += gridDim.x * 256)
			{
				const float v = p.mats[0].y[i];
				if (i == 0) p.argmax[1] = __builtin_isnan(v);
				if (argmax_better(v, i, bv, br))
				{
					bv = v;
					br = i;
				}
			}
			s_v[threadIdx.x] = bv;
			s_r[threadIdx.x] = br;
			__syncthreads();
			for (int h = 128; h > 0; h >>= 1)
			{
				if (static_cast<int>(threadIdx.x) < h && argmax_better(s_v[threadIdx.x + h], s_r[threadIdx.x + h], s_v[threadIdx.x],
				                                     s_r[threadIdx.x]))
				{
					s_v[threadIdx.x] = s_v[threadIdx.x + h];
					s_r[threadIdx.x] = s_r[threadIdx.x + h];
				}
				__syncthreads();
			}
			if (threadIdx.x == 0) p.best[blockIdx.x] = make_float2(s_v[0], __int_as_float(s_r[0]));
		}

		// Y[t][r] = the splits' partials summed in split order.
		__global__ void gemv_reduce_kernel(const gemv_params p)
		{
			const size_t n = static_cast<size_t>(p.n_batch) * p.rows;
			for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
			     i += static_cast<size_t>(gridDim.x) * blockDim.x)
			{
				// Eight splits' loads in flight at a time, added in split order.
				float s = 0.0f;
				for (int k0 = 0; k0 < p.n_split; k0 += 8)
				{
					float v[8];
#pragma unroll
					for (int u = 0; u < 8; ++u)
						v[u] = k0 + u < p.n_split ? p.part[static_cast<size_t>(k0 + u) * n + i] : 0.0f;
#pragma unroll
					for (int u = 0; u < 8; ++u)
						if (k0 + u < p.n_split) s = k0 + u == 0 ? v[u] : s + v[u];
				}
				const int t = static_cast<int>(i / p.rows);
				const mat_row mr = locate(p, static_cast<int>(i % p.rows));
				mr.m.y[t * mr.m.y_stride + mr.r] = s;
			}
		}

		// p.x_tiles tiles of vectors: 1 to 4. (Q4_S with four: one row tile, since
		// two spilled 61 registers: 64 vectors of 19456 x 2560 103 us, of 10240 x
		// 9728 243; with one 63 and 110.)
		template <int F, int RT, int TT = 1>
		void launch_batch(const gemv_params& p, hipStream_t stream)
		{
			if constexpr (TT < 4)
				if (p.x_tiles != TT) return launch_batch<F, RT, TT + 1>(p, stream);
			if constexpr (F == kGemvQ4S && RT == 2 && TT == 4) return launch_batch<F, 1, TT>(p, stream);
			else
				gemv_batch_kernel<F, RT, TT><<<(p.rows + 16 * RT - 1) / (16 * RT), 64 * kBatchWaves,
				                               kBatchWaves * RT * TT * 1024, stream>>>(p);
		}

		template <int F, int RT, int TT, int WR, int SLOTS, int NPW>
		void launch_tile(const gemv_params& p, hipStream_t stream)
		{
			using S = tile_shape<F, RT, TT, WR, SLOTS, NPW>;
			const int n_tt = (p.x_tiles + TT - 1) / TT, n_rt = (p.rows + 16 * RT * WR - 1) / (16 * RT * WR);
			gemv_tile_kernel<F, RT, TT, WR, SLOTS, NPW><<<(n_rt + 7) / 8 * 8 * n_tt, 128 * WR, S::kLds, stream>>>(p);
		}

		// The calls with staged X. A row's sums do not depend on the choices by
		// `rows` below, only on the columns and the number of vectors, so the
		// matrices of a group get the bits of their own calls.
		template <int F>
		void launch_wide(const gemv_params& p, hipStream_t stream)
		{
			const int nb = p.cols / 32, items = (F == kGemvQ4S ? (nb + 31) & ~31 : nb) * p.x_tiles;
			gemv_stage_x_kernel<F><<<(items + 3) / 4, 256, 0, stream>>>(p);
			if (p.n_batch <= kGemvBatchMax)
			{
				// Two 16-row tiles per work-group halve the reads of X; one
				// fills more CUs (from 160 work-groups on, two).
				p.rows >= 32 * 160 ? launch_batch<F, 2>(p, stream) : launch_batch<F, 1>(p, stream);
				return;
			}
			// rows x vectors per work-group, by what fills the 256 CUs (us, BF16 /
			// Q8_0): 128 x 128 moves the fewest bytes per product but takes one
			// CU each (6144 x 2560, 512 vectors, 192 of them: 48.1 / 61.3 against
			// 54.5 / 63.8 in 128 x 64; 19456 x 2560, 608 of them: 133 / 161
			// against 131 / 154); 64 x 64 for few (6144 x 2560, 128 vectors, 96
			// work-groups of 128 x 64: 31.0 / 34.0 against 34.8 / 40.7); and for
			// BF16 the deeper rings, one work-group per CU, where there is no
			// second one to cover the waits (2560 x 4096, 512 vectors: 45.4
			// against 49.5; with 384 work-groups 62.0 against 54.5).
			const long long w128 = 1LL * ((p.rows + 127) / 128) * ((p.x_tiles + 7) / 8);
			const long long w64 = 1LL * ((p.rows + 127) / 128) * ((p.x_tiles + 3) / 4);
			if (w128 >= 128 && w128 <= 256)
				launch_tile<F, 2, 8, 4, 2, 2>(p, stream);
			else if (w64 <= 128)
				launch_tile<F, 2, 4, 2, 2, 2>(p, stream);
			else if (F == kGemvBf16 && w64 <= 256)
				launch_tile<kGemvBf16, 2, 4, 4, 4, 4>(p, stream);
			else
				launch_tile<F, 2, 4, 4, 2, 2>(p, stream);
		}
	}

	void gemv_plan(int cols, int n_batch, int format, int& n_split, int& split_blocks)
	{
		const int nb = cols / 32;
		// As few K splits as the LDS copy of X^T of 16 vectors allows, the
		// splits equal in size (fewer vectors leave room for longer splits,
		// whose few work-groups ran 2 vectors of 2560 x 9728 in 38 us where 16
		// took 23).
		int max_blocks = 1;
		const int cap = format == kGemvBf16 ? kGemvBf16Blocks : kGemvQuantBlocks;
		while (max_blocks < std::min(nb, cap) && gemv_lds_bytes(max_blocks + 1, n_batch) <= gemv_batch_lds(format))
			++max_blocks;
		n_split = (nb + max_blocks - 1) / max_blocks;
		split_blocks = (nb + n_split - 1) / n_split;
	}

	// Up to 16 vectors run either kernel. Graph replays of one stream, us, 2 and 16
	// vectors, gemv_kernel / gemv_batch_kernel (with its staging): BF16 2560 x
	// 1024 10.9 / 6.7 and 12.2 / 6.8, 2560 x 2048 11.1 / 8.8 and 12.3 / 9.1, 6144 x
	// 2048 12.3 / 12.2 and 14.3 / 12.4, 6144 x 2560 12.6 / 13.9 and 14.5 / 14.2 (and
	// 14336 x 2048 18.4 / 20.4 and 21.3 / 20.7, the price of a line at columns);
	// Q8_0 2560 x 2048 12.4 / 7.7 and 13.5 / 7.7, 6144 x 4096 18.8 / 17.1 and 22.1 /
	// 17.2, 2560 x 6144 16.6 / 16.2 and 17.9 / 16.4, 2560 x 7168 17.5 / 18.2 and
	// 19.1 / 18.5, 2560 x 9728, 16 vectors, 23.3 / 23.5 (X is read once per 16 rows
	// there, four times the weights' bytes); Q4_S 6144 x 2048 13.1 / 10.5 and
	// 14.5 / 10.5, 2560 x 6144 15.0 / 13.9 and 16.5 / 14.1, 2560 x 7168 15.5 / 16.2
	// and 17.8 / 16.3. With three streams at once, which calls from one thread
	// bound by their launches, two each, both take 7 to 8 us up to about 4096
	// columns, and at 6144 two Q8_0 vectors 7.8 / 9.7 and sixteen 8.9 / 9.3. A
	// narrow matrix takes gemv_kernel one launch and no scratch, 4.6 us of host
	// time against 7.4: eager calls of one stream, 2 and 16 vectors, BF16 640 x 128
	// 7.0 / 7.7 and 7.9 / 7.8, 4096 x 320 7.6 / 7.6 and 8.8 / 7.8; Q8_0 640 x 256
	// 5.5 / 7.9 and 6.4 / 7.7, 4096 x 384 8.1 / 7.7 and 9.3 / 8.0; Q4_S 640 x 384
	// 7.3 / 8.1 and 8.4 / 8.4, 2048 x 448 8.2 / 8.3 and 9.6 / 7.9 (replays of a graph,
	// where the launch is cheap, 6.9 / 4.2 for BF16 640 x 128, 6.5 / 4.6 for Q8_0
	// 640 x 384). BF16 matrices of many rows give gemv_kernel work-groups enough,
	// and up to eight vectors leave it little besides the weights: eager calls of
	// one stream and of three, 2 and 8 vectors, 151 936 x 1024 60 / 75 and 71 / 79,
	// 50 / 59 and 55 / 61; x 1536 91 / 111 and 108 / 115, 76 / 94 and 88 / 96;
	// 32 000 x 1024 17.5 / 20.2 and 18.9 / 20.4 (12 vectors 20.4 / 20.5, 16 22.1 /
	// 20.6); but x 640 52.8 / 49.7 and 60.7 / 51.6; and where one K split takes
	// all the columns, up to 512, for any number: 50 000 x 448, 2 and 12 vectors,
	// 22 and 12 % faster. Of fewer rows, two matrices in a group (gate and up) of
	// 8704 to 10 752 rows leave gemv_batch_kernel a short last round (9216 x 1280,
	// x 1440, x 1536, 2 vectors: 16 to 21 % faster in gemv_kernel, 8 vectors 12 to
	// 18; 11 264 x 1280 5 % slower), and from 1664 columns on so do most (6144 x
	// 1792 11 %, 8192 x 2048 2 and with three streams 12 %). The rows are one
	// matrix's; see gemv_launch_vectors.
	bool gemv_stages_x(int rows, int cols, int n_batch, int format)
	{
		if (gemv_vec_fits(cols, n_batch, format)) return false;
		if (n_batch > kGemvMaxBatch) return true;
		if (format == kGemvBf16 && rows >= 20000 && cols <= 512) return false;
		if (format == kGemvBf16 && n_batch <= 8 && rows >= 6144)
		{
			const int most = rows >= 20000 ? 863 : (rows >= 8704 && rows <= 10752 ? 1151 : 1663);
			return cols > 256 && cols <= most;
		}
		return format == kGemvBf16 ? cols > 256 && cols <= 2048 : cols > 384 && cols <= 6144;
	}

	// One launch takes all the vectors up to kGemvWideBatch, but where the kernel
	// of that number leaves most of the chip idle: a work-group walks all the
	// columns, so few rows of many columns are a long chain on few CUs. 65 and
	// more vectors then run 64 at a time through gemv_batch_kernel, whose
	// wavefronts share the columns, and 17 and more of the widest matrices 16 at
	// a time through gemv_kernel, whose K splits give more work-groups. Graph
	// replays of one stream, us, 16 at a time / 64 at a time / all in
	// gemv_tile_kernel, 80 and 96 vectors: BF16 1024 x 9728 67 / 59 / 90 and 80 /
	// 69 / 90, 2048 x 8192 67 / 53 / 77 and 81 / 59 / 77; Q8_0 1024 x 9728 69 /
	// 58 / 108 and 82 / 72 / 108, 2560 x 9728 106 / 68 / 110 and 127 / 76 / 111;
	// Q4_S 1024 x 7168 72 / 45 / 82 and 86 / 48 / 83. Three streams at once fill
	// the CUs that one leaves idle: 64 at a time is then slower than all at once
	// (BF16 2048 x 8192, 80 and 96 vectors, 32 / 28 and 37 / 30; quantised at 128
	// vectors, 2560 x 9728 53 / 45), so the lines are where all at once is also
	// slower than 16 at a time for one stream. 16 at a time / all at once: BF16
	// 640 x 9728 26 / 30 (32 vectors), 640 x 14336 70 / 131 (80), Q8_0 1024 x
	// 14336 33 / 43 (32). The rows are those of one matrix, and the matrices of a
	// group that differ here run by themselves: a matrix gets the same bits
	// alone and in a group.
	int gemv_launch_vectors(int rows, int cols, int n_batch, int format)
	{
		const bool bf16 = format == kGemvBf16;
		const int widest = bf16 ? 7680 : (format == kGemvQ8_0 ? 12288 : 16384);
		if (gemv_staged_bytes(cols, std::min(n_batch, kGemvWideBatch), format) > kGemvStagedMax) return kGemvMaxBatch;
		if (rows <= 1024 && n_batch > kGemvMaxBatch && n_batch <= (cols - widest) / 64) return kGemvMaxBatch;
		if (rows <= (bf16 ? 2048 : 3072) && cols >= (bf16 ? 7168 : 6144) && n_batch > kGemvBatchMax &&
		    n_batch <= (!bf16 ? 112 : (rows <= 1024 ? 96 : 80)))
			return kGemvBatchMax;
		return kGemvWideBatch;
	}

	size_t gemv_staged_bytes(int cols, int n_batch, int format)
	{
		const size_t nb = cols / 32, tiles = (n_batch + 15) / 16;
		return tiles * (nb * 2048 + (format == kGemvQ4S ? (nb + 31) / 32 * 3072 : 0));
	}

	int gemv_vec_groups(int rows)
	{
		const int n_pairs = (rows + 1) / 2;
		return std::max(1, std::min((n_pairs + 3) / 4, 512));
	}

	// LDS of the one-vector kernel: x in the lanes' order (padded to whole
	// chunks), then Q4_S's block sums, or the argmax's eight floats.
	static size_t gemv_vec_lds(int cols, int format)
	{
		const int xf = format == kGemvBf16   ? vec_x_floats<kGemvBf16>(cols)
		               : format == kGemvQ8_0 ? vec_x_floats<kGemvQ8_0>(cols)
		                                     : vec_x_floats<kGemvQ4S>(cols);
		return static_cast<size_t>(xf + std::max(cols / 32, 8)) * 4;
	}

	bool gemv_vec_fits(int cols, int n_batch, int format)
	{
		return n_batch == 1 && gemv_vec_lds(cols, format) <= kGemvLdsBudget;
	}

	bool launch_gemv(const gemv_params& p, hipStream_t stream)
	{
		if (gemv_vec_fits(p.cols, p.n_batch, p.format))
		{
			const size_t lds = gemv_vec_lds(p.cols, p.format);
			const dim3 grid(gemv_vec_groups(p.rows));
			switch (p.format)
			{
			case kGemvBf16: gemv_vec_kernel<kGemvBf16><<<grid, 256, lds, stream>>>(p); return true;
			case kGemvQ8_0: gemv_vec_kernel<kGemvQ8_0><<<grid, 256, lds, stream>>>(p); return true;
			case kGemvQ4S:
				if (vec_joint<kGemvQ4S>(p.cols))
					gemv_vec_kernel<kGemvQ4S, false, true><<<grid, 256, lds, stream>>>(p);
				else
					gemv_vec_kernel<kGemvQ4S><<<grid, 256, lds, stream>>>(p);
				return true;
			default: return false;
			}
		}
		if (p.xs)
		{
			switch (p.format)
			{
			case kGemvBf16: launch_wide<kGemvBf16>(p, stream); return true;
			case kGemvQ8_0: launch_wide<kGemvQ8_0>(p, stream); return true;
			case kGemvQ4S: launch_wide<kGemvQ4S>(p, stream); return true;
			default: return false;
			}
		}
		const dim3 grid((p.rows + kGemvRows - 1) / kGemvRows, p.n_split);
		const size_t lds = gemv_lds_bytes(p.split_blocks, p.n_batch);
		switch (p.format)
		{
		case kGemvBf16: gemv_kernel<kGemvBf16><<<grid, 4 * kGemvRows, lds, stream>>>(p); break;
		case kGemvQ8_0: gemv_kernel<kGemvQ8_0><<<grid, 4 * kGemvRows, lds, stream>>>(p); break;
		case kGemvQ4S: gemv_kernel<kGemvQ4S><<<grid, 4 * kGemvRows, lds, stream>>>(p); break;
		default: return false;
		}
		if (p.n_split > 1)
		{
			const size_t n = static_cast<size_t>(p.n_batch) * p.rows;
			const unsigned g = static_cast<unsigned>(std::min<size_t>((n + 255) / 256, 4096));
			gemv_reduce_kernel<<<g, 256, 0, stream>>>(p);
		}
		return true;
	}

	bool launch_gemv_argmax(const gemv_params& p, hipStream_t stream)
	{
		if (p.format != kGemvBf16 || !gemv_vec_fits(p.cols, 1, kGemvBf16)) return false;
		const int groups = gemv_vec_groups(p.rows);
		const size_t lds = gemv_vec_lds(p.cols, kGemvBf16); // x, then the wavefronts' best pairs
		gemv_vec_kernel<kGemvBf16, true><<<groups, 256, lds, stream>>>(p);
		gemv_argmax_final_kernel<<<1, 256, 0, stream>>>(p, groups);
		return true;
	}

	bool launch_argmax(const gemv_params& p, hipStream_t stream)
	{
		const int groups = std::max(1, std::min((p.rows + 1023) / 1024, kArgmaxGroups));
		argmax_part_kernel<<<groups, 256, 0, stream>>>(p);
		gemv_argmax_final_kernel<<<1, 256, 0, stream>>>(p, groups);
		return true;
	}
}
