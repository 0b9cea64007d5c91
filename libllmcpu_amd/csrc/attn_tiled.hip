// Tiled attention for the batches the MFMA prefill kernel does not take: F32
// K/V, and head shapes outside mfma_shape (head_dim a multiple of 16 up to
// 512, any group up to 16). nnc runs these through the same attention core
// as every batch (reference src/libnnc/model.cpp:1750-1757); its embedding
// call (model.cpp:2355-2368) is one such batch: the whole input over an F32
// cache, bidirectional.
//
// Rows are (token, query head) pairs of one KV head, token major. Grid:
// (row blocks of 64, KV heads, key splits of the block's keys). A work-group
// of four wavefronts owns 64 rows, 16 per wavefront, and walks its split's
// keys in steps of 16:
// the step's K and V rows are loaded by all 256 threads (F32 as is, BF16
// widened by a 16-bit shift) into LDS, double-buffered, the next step's
// loads in flight in registers while the current one is computed. Every
// product is fp32 on the matrix cores (v_mfma_f32_16x16x4_f32: exact fp32
// products, fp32 sums):
//   S^T = K . Q^T    16 keys x 16 rows, head_dim / 4 MFMAs. Lane l's row is
//                    l % 16; its Q elements sit in registers, element
//                    (l / 16) * (head_dim / 4) + s in MFMA s (any fixed
//                    permutation of d gives the same dot product), so the
//                    K rows are read from LDS 16 bytes at a time;
//   softmax          per row, in fp32 and log2 units (Q pre-scaled by
//                    scale * log2(e)): weights exp2(s - m) against the row's
//                    offset m, raised only when a score passes it by more
//                    than kTileLazy, and their running sum; keys outside the
//                    row's span weigh exactly 0;
//   O^T += V^T . P^T head_dim / 16 tiles of 16 elements x 4 MFMAs of 4 keys;
//                    P^T comes straight from the score registers (key
//                    4 (l / 16) + s in MFMA s), so the row stays in the lane
//                    and the rescale is in-lane.
// A split writes its partial (o, m, l per row, o and l relative to the
// offset m) and a merge kernel combines each row's splits in order; with one
// split per block the kernel writes o * (1 / l) (0 when l == 0, reference
// nn_ops.cpp:492) directly. Splits are relative to the block's first key, so
// only splits that hold keys of the block exist (the windows of a
// bidirectional or sliding layer, the short spans of a causal chunk's first
// tokens), and the partials take n_tok * n_kv * (largest split count) rows.
#include "device_common.h"
#include "kernels.h"

namespace nnchip
{
	namespace
	{
		constexpr int kTileRows = 16; // rows per wavefront
		constexpr int kTileWaves = 4;
		constexpr int kTileBlock = kTileRows * kTileWaves; // rows per work-group
		constexpr int kTileKeys = 16; // keys per step
		constexpr float kTileLazy = 8.0f; // max growth of a row's scores over its offset (log2 units)

		__device__ __forceinline__ f32x4 mfma_f32(float a, float b, const f32x4& c)
		{
			return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
		}

		// max / sum of x over the four lanes l % 16 + 16 j (one row's lanes).
		__device__ __forceinline__ float row4_max(float x)
		{
			const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
			x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
			return max_with_other_half(x);
		}

		__device__ __forceinline__ float row4_sum(float x) { return add_with_other_half(add_with_other_row(x)); }

		// Four elements of K or V row `row` at element e (a multiple of 4) of
		// this head, as fp32.
		template <bool BF16>
		__device__ __forceinline__ float4 load4(const void* base, size_t elem)
		{
			if constexpr (BF16)
			{
				const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(base) + elem);
				return make_float4(bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y));
			}
			else
				return *reinterpret_cast<const float4*>(static_cast<const float*>(base) + elem);
		}

		// The keys of row block `blk` of BLOCK rows (its rows' spans together:
		// both ends of a span move forward with the position; the first key
		// rounded down to a multiple of ALIGN) and its splits: split z covers
		// keys b_lo + z * split_keys .. + split_keys - 1, relative to the block's
		// first key, so a block has (b_hi - b_lo) / split_keys + 1 of them and
		// the grid's z extent is the largest such count.
		template <int BLOCK = kTileBlock, int ALIGN = 1>
		__device__ __forceinline__ void tiled_block_keys(const decode_params& p, int G, int blk, int& b_lo, int& b_hi)
		{
			const int n_rows = p.n_tok * G, r0 = blk * BLOCK, r1 = min(r0 + BLOCK, n_rows) - 1;
			int unused;
			attn_span(p.causal, p.window, p.pos0 + r0 / G, p.n_seq, b_lo, unused);
			attn_span(p.causal, p.window, p.pos0 + r1 / G, p.n_seq, unused, b_hi);
			b_lo = b_lo / ALIGN * ALIGN;
		}

		__device__ __forceinline__ int tiled_block_splits(int b_lo, int b_hi, int split_keys)
		{
			return b_lo <= b_hi ? (b_hi - b_lo) / split_keys + 1 : 0;
		}

		// Row (t, h)'s partial of its block's split z: [token][KV head][z][group][head_dim + 4]
		// (o, then m and l), z below n_split, the grid's z extent.
		__device__ __forceinline__ float* tiled_partial(const decode_params& p, int G, int hd, int t, int kvh, int z, int h)
		{
			const size_t PL = static_cast<size_t>(hd) + 4;
			return p.part + ((static_cast<size_t>(t) * p.n_kv + kvh) * p.n_split + z) * G * PL + static_cast<size_t>(h) * PL;
		}

		// HD: the head_dim when it is fixed at compile time (the common sizes:
		// no runtime bounds inside the MFMA loops), else 0 and head_dim_arg
		// up to HDMAX.
		template <int HD, int HDMAX, bool BF16>
		__global__ __launch_bounds__(64 * kTileWaves)
		__attribute__((amdgpu_waves_per_eu(HDMAX <= 256 ? 2 : 1))) void tiled_kernel(const decode_params p,
		                                                                              int head_dim_arg, int G)
		{
			const int hd = HD ? HD : head_dim_arg;
			constexpr int PMAX = HDMAX + 4; // LDS row pitch (floats) bound
			constexpr int QV = HDMAX / 4; // Q registers per lane
			constexpr int DT = HDMAX / 16; // 16-element tiles of O^T
			constexpr int LPT = (4 * HDMAX + 255) / 256; // float4 loads per thread per tensor and step
			__shared__ __attribute__((aligned(16))) float s_k[2][kTileKeys * PMAX];
			__shared__ __attribute__((aligned(16))) float s_v[2][kTileKeys * PMAX];

			const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
			const int c = lane >> 4, r16 = lane & 15;
			const int kvh = blockIdx.y, split = blockIdx.z;
			const int pitch = hd + 4, q4 = hd / 4, n_dt = hd / 16, n_f4 = 4 * hd; // float4 slots of a step's K
			const int n_rows = p.n_tok * G;
			const int row0 = blockIdx.x * kTileBlock;
			const int row = row0 + wave * kTileRows + r16;
			const bool row_ok = row < n_rows;
			const int t = row_ok ? row / G : 0, h = row_ok ? row % G : 0;
			const size_t qo = (static_cast<size_t>(t) * p.n_head + static_cast<size_t>(kvh) * G + h) * hd;

			// This split's keys: the row's, and the work-group's (the union over
			// its tokens; both ends of a span move forward with the position).
			int b_lo, b_hi;
			tiled_block_keys(p, G, blockIdx.x, b_lo, b_hi);
			if (split >= tiled_block_splits(b_lo, b_hi, p.split_keys)) return; // the whole work-group: no split here
			const int w_lo = b_lo + split * p.split_keys, w_hi = min(b_hi, w_lo + p.split_keys - 1);
			int first, last;
			attn_span(p.causal, p.window, p.pos0 + t, p.n_seq, first, last);
			const int r_lo = row_ok ? max(first, w_lo) : 1, r_hi = row_ok ? min(last, w_hi) : 0;
			const int n_steps = (w_hi - w_lo) / kTileKeys + 1;

			// Q: element (lane / 16) * (hd / 4) + s in register s, log2 units.
			float q[QV];
#pragma unroll
			for (int s4 = 0; s4 < QV / 4; ++s4)
			{
				float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
				if (row_ok && s4 < q4 / 4) v = *reinterpret_cast<const float4*>(p.q + qo + c * q4 + 4 * s4);
				q[4 * s4] = v.x * p.qscale;
				q[4 * s4 + 1] = v.y * p.qscale;
				q[4 * s4 + 2] = v.z * p.qscale;
				q[4 * s4 + 3] = v.w * p.qscale;
			}

			// A step's K and V rows into registers: thread slot i = tid + 256 j
			// is key i / (hd / 4), elements 4 (i % (hd / 4)) .. + 3; keys past
			// the work-group's range are zeros.
			const size_t head_off = static_cast<size_t>(kvh) * hd;
			float4 pk[LPT], pv[LPT];
			auto load_step = [&](int st) __attribute__((always_inline))
			{
				const int k0 = w_lo + st * kTileKeys;
#pragma unroll
				for (int j = 0; j < LPT; ++j)
				{
					const int i = tid + 256 * j;
					const int key = i / q4, e = 4 * (i % q4);
					pk[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
					pv[j] = pk[j];
					if (i < n_f4 && k0 + key <= w_hi)
					{
						const size_t el = static_cast<size_t>((k0 + key) % p.rows) * p.kv_dim + head_off + e;
						pk[j] = load4<BF16>(p.K, el);
						pv[j] = load4<BF16>(p.V, el);
					}
				}
			};
			auto store_step = [&](int buf) __attribute__((always_inline))
			{
#pragma unroll
				for (int j = 0; j < LPT; ++j)
				{
					const int i = tid + 256 * j;
					if (i < n_f4)
					{
						const int off = (i / q4) * pitch + 4 * (i % q4);
						*reinterpret_cast<float4*>(&s_k[buf][off]) = pk[j];
						*reinterpret_cast<float4*>(&s_v[buf][off]) = pv[j];
					}
				}
			};

			f32x4 acc[DT];
#pragma unroll
			for (int d = 0; d < DT; ++d) acc[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
			float m_run = -INFINITY, l_run = 0.0f;

			if (n_steps > 0)
			{
				load_step(0);
				store_step(0);
			}
			__syncthreads();
			for (int st = 0; st < n_steps; ++st)
			{
				const int buf = st & 1;
				if (st + 1 < n_steps) load_step(st + 1);
				const int k0 = w_lo + st * kTileKeys;

				// S^T: lane holds keys k0 + 4 c + i of row r16.
				f32x4 sc = {0.0f, 0.0f, 0.0f, 0.0f};
				const float* kp = &s_k[buf][r16 * pitch + c * q4];
#pragma unroll
				for (int s4 = 0; s4 < QV / 4; ++s4)
				{
					if (s4 < q4 / 4)
					{
						const float4 kv = *reinterpret_cast<const float4*>(kp + 4 * s4);
						sc = mfma_f32(kv.x, q[4 * s4], sc);
						sc = mfma_f32(kv.y, q[4 * s4 + 1], sc);
						sc = mfma_f32(kv.z, q[4 * s4 + 2], sc);
						sc = mfma_f32(kv.w, q[4 * s4 + 3], sc);
					}
				}

				// Online softmax of the row.
				float cmax = -INFINITY;
#pragma unroll
				for (int i = 0; i < 4; ++i)
				{
					const int k = k0 + 4 * c + i;
					sc[i] = (k >= r_lo && k <= r_hi) ? sc[i] : -INFINITY;
					cmax = fmaxf(cmax, sc[i]);
				}
				cmax = row4_max(cmax);
				// The row's offset m is raised (to the step's max) only when a
				// score passes it by more than kTileLazy: weights stay in
				// (0, 2^kTileLazy] and the O rescale is rare (a wavefront-wide
				// branch).
				const bool raise = cmax > m_run + kTileLazy;
				if (__builtin_amdgcn_ballot_w64(raise))
				{
					const float alpha = raise && m_run != -INFINITY ? fast_exp2(m_run - cmax) : 1.0f;
					m_run = raise ? cmax : m_run;
					l_run *= alpha;
#pragma unroll
					for (int d = 0; d < DT; ++d) acc[d] *= alpha;
				}
				const float m_use = m_run == -INFINITY ? 0.0f : m_run;
				float pw[4], ls = 0.0f;
#pragma unroll
				for (int i = 0; i < 4; ++i)
				{
					pw[i] = fast_exp2(sc[i] - m_use);
					ls += pw[i];
				}
				l_run += row4_sum(ls);

				// O^T: tile d holds elements 16 d + 4 c + i of row r16.
				const float* vp = &s_v[buf][(4 * c) * pitch + r16];
#pragma unroll
				for (int d = 0; d < DT; ++d)
				{
					if (d < n_dt)
					{
#pragma unroll
						for (int s = 0; s < 4; ++s) acc[d] = mfma_f32(vp[s * pitch + 16 * d], pw[s], acc[d]);
					}
				}

				if (st + 1 < n_steps) store_step(buf ^ 1);
				__syncthreads();
			}

			if (!row_ok) return;
			if (p.n_split > 1)
			{
				float* gp = tiled_partial(p, G, hd, t, kvh, split, h);
#pragma unroll
				for (int d = 0; d < DT; ++d)
					if (d < n_dt) *reinterpret_cast<f32x4*>(gp + 16 * d + 4 * c) = acc[d];
				if (c == 0) *reinterpret_cast<float2*>(gp + hd) = make_float2(m_run, l_run);
			}
			else
			{
				const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
#pragma unroll
				for (int d = 0; d < DT; ++d)
				{
					if (d < n_dt)
					{
						const size_t oi = qo + 16 * d + 4 * c;
						float4 o;
						o.x = gated(acc[d][0] * inv, p.gate, oi);
						o.y = gated(acc[d][1] * inv, p.gate, oi + 1);
						o.z = gated(acc[d][2] * inv, p.gate, oi + 2);
						o.w = gated(acc[d][3] * inv, p.gate, oi + 3);
						*reinterpret_cast<float4*>(p.out + oi) = o;
					}
				}
			}
		}

		// The merge of row (t, h)'s splits: those of its block that its own
		// span reaches, in order; M = the largest offset m, o = sum o_z
		// 2^(m_z - M), l likewise; out = o * (1 / l), 0 when l == 0. Four rows
		// per work-group, 64 threads per row, four elements per thread and
		// pass.
		template <int BLOCK, int ALIGN>
		__global__ __launch_bounds__(256) void tiled_merge_kernel(const decode_params p, int hd, int G)
		{
			const int n_rows = p.n_tok * G, r = blockIdx.x * 4 + (threadIdx.x >> 6), kvh = blockIdx.y;
			if (r >= n_rows) return;
			const int lane = threadIdx.x & 63, t = r / G, h = r % G;
			int b_lo, b_hi, first, last;
			tiled_block_keys<BLOCK, ALIGN>(p, G, r / BLOCK, b_lo, b_hi);
			attn_span(p.causal, p.window, p.pos0 + t, p.n_seq, first, last);
			const int z0 = first <= last ? (first - b_lo) / p.split_keys : 0;
			const int z1 = first <= last ? (last - b_lo) / p.split_keys : -1;
			float M = -INFINITY;
			for (int z = z0; z <= z1; ++z) M = fmaxf(M, tiled_partial(p, G, hd, t, kvh, z, h)[hd]);
			const float m_use = M == -INFINITY ? 0.0f : M;
			const size_t oi0 = (static_cast<size_t>(t) * p.n_head + static_cast<size_t>(kvh) * G + h) * hd;
			for (int d = 4 * lane; d < hd; d += 256)
			{
				float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
				float L = 0.0f;
				for (int z = z0; z <= z1; ++z)
				{
					const float* gp = tiled_partial(p, G, hd, t, kvh, z, h);
					const float f = fast_exp2(gp[hd] - m_use);
					const float4 v = *reinterpret_cast<const float4*>(gp + d);
					acc.x = fmaf(v.x, f, acc.x);
					acc.y = fmaf(v.y, f, acc.y);
					acc.z = fmaf(v.z, f, acc.z);
					acc.w = fmaf(v.w, f, acc.w);
					L = fmaf(gp[hd + 1], f, L);
				}
				const float inv = L > 0.0f ? 1.0f / L : 0.0f;
				const size_t oi = oi0 + d;
				float4 o;
				o.x = gated(acc.x * inv, p.gate, oi);
				o.y = gated(acc.y * inv, p.gate, oi + 1);
				o.z = gated(acc.z * inv, p.gate, oi + 2);
				o.w = gated(acc.w * inv, p.gate, oi + 3);
				*reinterpret_cast<float4*>(p.out + oi) = o;
			}
		}

		// ---- F32 caches at head_dim 64, 128 and 256, long batches: tiled3_kernel ----
		//
		// fp32 products as sums of bf16 ones: x = x1 + x2 + x3, three bf16 that
		// hold fp32's 24 bits, and x . y = x1y1 + (x1y2 + x2y1) + (x1y3 + x2y2 +
		// x3y1); the three products left out are below 2^-25 of x . y, half of
		// one fp32 rounding. Six bf16 MFMAs of 32 deep take 96 clocks where the
		// fp32 ones take 256 (v_mfma_f32_16x16x4_f32: 157 TFLOP/s on this part,
		// and the kernel above is bound by them). Sums stay fp32, and a 32-deep
		// MFMA rounds its sum less often than eight 4-deep ones: against 64 bits
		// (relative, 2-norm) a 2048-token embedding call is off by 4.6e-7 (fp32
		// MFMAs: 5.7e-7), 1000 causal tokens of 4 x 256 by 4.7e-7 (5.8e-7), 300
		// over 1500 keys of 16 x 128 by 4.4e-7 (4.6e-7).
		//
		// tiled3_split_kernel first writes the span's K and V as operands (kept
		// for the call; every row block reads them): per 32-key group and KV head
		// 1 KB fragments in lane order, K [16-key tile][32 elements][part], V
		// [16 elements][part] with the keys in the score registers' order. A
		// work-group takes 128 rows; Q (three parts) and O stay in registers. A
		// group's K and V have one LDS buffer each: the next K loads (LDS-DMA)
		// during this group's P . V, the next V during the next scores. us, one
		// stream / three at once, tiled_kernel -> this: six layers of a 2048-token
		// embedding call (five windowed) 408 / 318 -> 345 / 222, four of 1000
		// causal tokens of 4 x 256 244 / 171 -> 197 / 123, two of 300 tokens over
		// 1500 keys of 16 x 128 133 / 90 -> 119 / 63. Bound by the matrix cores,
		// and in a windowed layer (four groups per work-group) by Q's staging,
		// the operands' kernel and the merge around them.
		constexpr int kT3Block = kTiled3Block, kT3Keys = kTiled3Keys;

		// x as bf16 parts, x = out[0] + out[1] + out[2] to 24 bits (fewer below
		// 2^-109, where the last is subnormal). Parts are at most the largest
		// finite bf16: the first for K and V, which are finite wherever the parts
		// are used; for Q the second too, so an infinite x is (largest, largest,
		// x), whose products with elements below 2^8 are infinite of the right
		// sign or finite. NaN stays in the last part. (The weights: at most 2^8.)
		enum t3_operand { kT3KV, kT3Q, kT3P };
		template <t3_operand OF>
		__device__ __forceinline__ void split3(const float (&x)[8], u32x4 (&out)[3])
		{
			const float big = __uint_as_float(0x7f7f0000u);
			auto lim = [&](bool on, float v) __attribute__((always_inline)) { return on ? __builtin_amdgcn_fmed3f(v, -big, big) : v; };
#pragma unroll
			for (int j = 0; j < 4; ++j)
			{
				const float a = x[2 * j], b = x[2 * j + 1];
				const uint32_t h = cvt_pk_bf16(lim(OF != kT3P, a), lim(OF != kT3P, b));
				const float a1 = a - bf16_lo(h), b1 = b - bf16_hi(h);
				const uint32_t m = cvt_pk_bf16(lim(OF == kT3Q, a1), lim(OF == kT3Q, b1));
				out[0][j] = h;
				out[1][j] = m;
				out[2][j] = cvt_pk_bf16(a1 - bf16_lo(m), b1 - bf16_hi(m));
			}
		}

		// z stays 0 while every x is finite, and is NaN once one is not.
		__device__ __forceinline__ void add_zeros(const float (&x)[8], float& z)
		{
#pragma unroll
			for (int j = 0; j < 8; ++j) z = fmaf(x[j], 0.0f, z);
		}

		// Bytes of a group's K (or V) of one head.
		template <int HD>
		constexpr uint32_t kT3Bytes = HD * kT3Keys * 6;

		// After the operands: per (head, group) whether K or V holds an infinite
		// or NaN element, one word for each wavefront of tiled3_split_kernel.
		template <int HD>
		__device__ __forceinline__ uint4* t3_flags(char* split, int n_kv, int n_g, int kvh)
		{
			return reinterpret_cast<uint4*>(split + static_cast<size_t>(n_kv) * n_g * 2 * kT3Bytes<HD>) + static_cast<size_t>(kvh) * n_g;
		}

		// Group g0 + blockIdx.x of head blockIdx.y; keys outside k_lo .. k_hi as
		// zeros.
		template <int HD>
		__global__ __launch_bounds__(256) void tiled3_split_kernel(const decode_params p, char* split, int k_lo, int k_hi, int g0)
		{
			const int kvh = blockIdx.y, key0 = (g0 + static_cast<int>(blockIdx.x)) * kT3Keys;
			char* dst = split + (static_cast<size_t>(kvh) * gridDim.x + blockIdx.x) * 2 * kT3Bytes<HD>;
			const size_t head_off = static_cast<size_t>(kvh) * HD;
			auto row = [&](int k) { return static_cast<size_t>(k % p.rows) * p.kv_dim + head_off; };
			const float* K = static_cast<const float*>(p.K);
			const float* V = static_cast<const float*>(p.V);
			float z = 0.0f;
			for (int i = threadIdx.x; i < HD * 4; i += 256) // (8 elements each)
			{
				const int lane = i & 63, f = i >> 6, r = lane & 15, g = lane >> 4;
				float x[8];
				u32x4 o[3];
				{
					const int t = f / (HD / 32), kk = f % (HD / 32), k = key0 + 16 * t + r;
					float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f), b = a;
					if (k >= k_lo && k <= k_hi)
					{
						const float* s = K + row(k) + 32 * kk + 8 * g;
						a = *reinterpret_cast<const float4*>(s);
						b = *reinterpret_cast<const float4*>(s + 4);
					}
					x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
					x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
					add_zeros(x, z);
					split3<kT3KV>(x, o);
#pragma unroll
					for (int c = 0; c < 3; ++c) *reinterpret_cast<u32x4*>(dst + (f * 3 + c) * 1024 + 16 * lane) = o[c];
				}
				{
#pragma unroll
					for (int j = 0; j < 8; ++j)
					{
						const int k = key0 + 16 * (j >> 2) + 4 * g + (j & 3);
						x[j] = k >= k_lo && k <= k_hi ? V[row(k) + 16 * f + r] : 0.0f;
					}
					add_zeros(x, z);
					split3<kT3KV>(x, o);
#pragma unroll
					for (int c = 0; c < 3; ++c)
						*reinterpret_cast<u32x4*>(dst + kT3Bytes<HD> + (f * 3 + c) * 1024 + 16 * lane) = o[c];
				}
			}
			const bool any = __builtin_amdgcn_ballot_w64(z != 0.0f) != 0;
			if ((threadIdx.x & 63) == 0)
				reinterpret_cast<uint32_t*>(t3_flags<HD>(split, p.n_kv, gridDim.x, kvh) + blockIdx.x)[threadIdx.x >> 6] = any;
		}

		// At most N of this wavefront's loads in flight (s_waitcnt vmcnt(N), the
		// other counters not waited on), then everyone's.
		template <int N>
		__device__ __forceinline__ void t3_wait_barrier()
		{
			static_assert(N < 16, "vmcnt");
			__builtin_amdgcn_sched_barrier(0);
			__builtin_amdgcn_s_waitcnt(0x0F70 | N);
			__builtin_amdgcn_s_barrier();
			__builtin_amdgcn_sched_barrier(0);
		}

		// This wavefront's LDS reads have returned (lgkmcnt(0)), then everyone's.
		__device__ __forceinline__ void t3_read_barrier()
		{
			__builtin_amdgcn_sched_barrier(0);
			__builtin_amdgcn_s_waitcnt(0xC07F);
			__builtin_amdgcn_s_barrier();
			__builtin_amdgcn_sched_barrier(0);
		}

		// c[y][x] += a[x] . b[y] of three-part operands, the smallest products
		// first, the sums in turn (a sum's next product waits for its last).
		template <int NA>
		__device__ __forceinline__ void mfma3(const u32x4 (&a)[2][3], const u32x4 (&b)[NA][3], f32x4 (&c)[NA][2])
		{
			constexpr int A[6] = {2, 0, 1, 1, 0, 0}, B[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
			for (int u = 0; u < 6; ++u)
#pragma unroll
				for (int x = 0; x < 2; ++x)
#pragma unroll
					for (int y = 0; y < NA; ++y) c[y][x] = mfma16x16x32(as_bf16x8(a[x][A[u]]), as_bf16x8(b[y][B[u]]), c[y][x]);
		}

		// Rows row .. end - 1 (one wavefront's) over keys w_lo .. w_hi of their own
		// spans, in fp32, a row at a time: the work-groups whose keys hold an
		// infinite or NaN element of K or V. In the matrix products a key that
		// weighs 0 in a row makes it NaN all the same, and the parts of an
		// infinite operand have no right products with the other's lower parts.
		template <int HD>
		__device__ void t3_rows_fp32(const decode_params& p, int G, int kvh, int z, int row, int end, int w_lo, int w_hi)
		{
			constexpr int E = HD / 64;
			const int e0 = E * (threadIdx.x & 63);
			const float* K = static_cast<const float*>(p.K) + static_cast<size_t>(kvh) * HD + e0;
			const float* V = static_cast<const float*>(p.V) + static_cast<size_t>(kvh) * HD + e0;
			for (; row < end; ++row)
			{
				const int t = row / G, h = row % G;
				const size_t qo = (static_cast<size_t>(t) * p.n_head + static_cast<size_t>(kvh) * G + h) * HD + e0;
				int first, last;
				attn_span(p.causal, p.window, p.pos0 + t, p.n_seq, first, last);
				float q[E], o[E], m = -INFINITY, l = 0.0f;
#pragma unroll
				for (int e = 0; e < E; ++e)
				{
					q[e] = p.q[qo + e] * p.qscale;
					o[e] = 0.0f;
				}
				for (int k = max(first, w_lo); k <= min(last, w_hi); ++k)
				{
					const size_t at = static_cast<size_t>(k % p.rows) * p.kv_dim;
					float s = 0.0f;
#pragma unroll
					for (int e = 0; e < E; ++e) s = fmaf(q[e], K[at + e], s);
					s = wave_sum_dpp(s);
					if (s > m + kTileLazy)
					{
						const float alpha = m == -INFINITY ? 1.0f : fast_exp2(m - s);
						m = s;
						l *= alpha;
#pragma unroll
						for (int e = 0; e < E; ++e) o[e] *= alpha;
					}
					const float w = fast_exp2(s - (m == -INFINITY ? 0.0f : m));
					l += w;
#pragma unroll
					for (int e = 0; e < E; ++e) o[e] = fmaf(w, V[at + e], o[e]);
				}
				if (p.n_split > 1)
				{
					float* gp = tiled_partial(p, G, HD, t, kvh, z, h);
#pragma unroll
					for (int e = 0; e < E; ++e) gp[e0 + e] = o[e];
					if (e0 == 0) *reinterpret_cast<float2*>(gp + HD) = make_float2(m, l);
				}
				else
				{
					const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
					for (int e = 0; e < E; ++e) p.out[qo + e] = gated(o[e] * inv, p.gate, qo + e);
				}
			}
		}

		// Row tiles per wavefront: two at head_dim 64 and 128 (a fragment read
		// from LDS serves two products; four wavefronts, two work-groups per
		// CU), one at 256, where two tiles' Q and O left one wavefront per SIMD and
		// spilled (417 / 278 us for the embedding call above; eight wavefronts,
		// two per SIMD, 340 / 220).
		template <int HD>
		constexpr int kT3Tiles = HD == 256 ? 1 : 2;

		template <int HD>
		__global__ __launch_bounds__(512 / kT3Tiles<HD>) __attribute__((amdgpu_waves_per_eu(2, 2))) void tiled3_kernel(
			const decode_params p, const char* split, int G, int g0, int n_g)
		{
			constexpr int NA = kT3Tiles<HD>, NWV = 8 / NA;
			constexpr int KK = HD / 32, DT = HD / 16, ND = kT3Bytes<HD> / 1024 / NWV; // DMAs per wavefront per K (or V)
			__shared__ __attribute__((aligned(16))) unsigned char s_k[kT3Bytes<HD>];
			__shared__ __attribute__((aligned(16))) unsigned char s_v[kT3Bytes<HD>];
			const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
			const int c = lane >> 4, r16 = lane & 15;
			const int kvh = blockIdx.y, z = blockIdx.z, n_rows = p.n_tok * G;

			int b_lo, b_hi;
			tiled_block_keys<kT3Block, kT3Keys>(p, G, blockIdx.x, b_lo, b_hi);
			if (z >= tiled_block_splits(b_lo, b_hi, p.split_keys)) return; // the whole work-group: no split here
			const int w_lo = b_lo + z * p.split_keys, w_hi = min(b_hi, w_lo + p.split_keys - 1);
			const int n_steps = (w_hi - w_lo) / kT3Keys + 1;

			const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
				const_cast<char*>(split) + static_cast<size_t>(kvh) * n_g * 2 * kT3Bytes<HD>, 0,
				static_cast<int>(static_cast<uint32_t>(n_g) * 2 * kT3Bytes<HD>), 0x00020000);
			// K (v = 0) or V (1) of step st; a step past the last loads nothing
			// (zeros), so that the counts of loads in flight stay the same.
			auto load = [&](int st, int v, unsigned char* dst) __attribute__((always_inline))
			{
				const uint32_t o = st < n_steps ? (static_cast<uint32_t>(w_lo / kT3Keys - g0 + st) * 2 + v) * kT3Bytes<HD> : 0u;
				const uint32_t lo = st < n_steps ? 16u * lane + 1024u * wave : 0x80000000u;
#pragma unroll
				for (int u = 0; u < ND; ++u) dma_lds16(rs, dst + 1024 * (NWV * u + wave), lo, o + 1024 * NWV * u);
			};
			load(0, 0, s_k);
			load(0, 1, s_v);

			uint32_t bad = 0; // of a lane, not 0: an infinite or NaN element in these keys' K or V
			{
				const uint4* flags = t3_flags<HD>(const_cast<char*>(split), p.n_kv, n_g, kvh) + (w_lo / kT3Keys - g0);
				for (int i = lane; i < n_steps; i += 64)
				{
					const uint4 f = flags[i];
					bad |= f.x | f.y | f.z | f.w;
				}
			}

			// This lane's row of each of the wavefront's tiles.
			int r_lo[NA], r_hi[NA];
			size_t qo[NA];
			u32x4 q[KK][NA][3];
#pragma unroll
			for (int a = 0; a < NA; ++a)
			{
				const int row = blockIdx.x * kT3Block + 16 * (NA * wave + a) + r16;
				const bool ok = row < n_rows;
				const int t = ok ? row / G : 0, h = ok ? row % G : 0;
				int first, last;
				attn_span(p.causal, p.window, p.pos0 + t, p.n_seq, first, last);
				r_lo[a] = ok ? max(first, w_lo) : 1;
				r_hi[a] = ok ? min(last, w_hi) : 0;
				qo[a] = (static_cast<size_t>(t) * p.n_head + static_cast<size_t>(kvh) * G + h) * HD;
#pragma unroll
				for (int kk = 0; kk < KK; ++kk)
				{
					const float4 u = *reinterpret_cast<const float4*>(p.q + qo[a] + 32 * kk + 8 * c);
					const float4 v = *reinterpret_cast<const float4*>(p.q + qo[a] + 32 * kk + 8 * c + 4);
					const float x[8] = {u.x * p.qscale, u.y * p.qscale, u.z * p.qscale, u.w * p.qscale,
					                    v.x * p.qscale, v.y * p.qscale, v.z * p.qscale, v.w * p.qscale};
					split3<kT3Q>(x, q[kk][a]);
				}
			}

			f32x4 acc[DT / 2][NA][2]; // elements 32 d + 16 x + 4 c + i
			float m_run[NA], l_run[NA];
#pragma unroll
			for (int a = 0; a < NA; ++a)
			{
				m_run[a] = -INFINITY;
				l_run[a] = 0.0f;
#pragma unroll
				for (int d = 0; d < DT / 2; ++d) acc[d][a][0] = acc[d][a][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
			}
			// (Q's loads came after the first DMAs: none of this is counted on)
			__builtin_amdgcn_sched_barrier(0);
			__builtin_amdgcn_s_waitcnt(0x0F70);
			if (__builtin_amdgcn_ballot_w64(bad != 0)) // (the same in every wavefront)
			{
				const int row = blockIdx.x * kT3Block + 16 * NA * wave;
				t3_rows_fp32<HD>(p, G, kvh, z, row, min(row + 16 * NA, n_rows), w_lo, w_hi);
				return;
			}

			for (int st = 0; st < n_steps; ++st)
			{
				const int k0 = w_lo + st * kT3Keys;
				t3_wait_barrier<ND>(); // K has landed; V may be in flight
				// S^T: tile t's keys k0 + 16 t + 4 c + i of row r16.
				f32x4 sc[NA][2];
#pragma unroll
				for (int a = 0; a < NA; ++a) sc[a][0] = sc[a][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
				// (the next fragments are read before the current ones' products)
				u32x4 f[2][2][3];
				auto read_k = [&](int kk, u32x4 (&o)[2][3]) __attribute__((always_inline))
				{
#pragma unroll
					for (int t = 0; t < 2; ++t)
#pragma unroll
						for (int u = 0; u < 3; ++u)
							o[t][u] = *reinterpret_cast<const u32x4*>(s_k + ((t * KK + kk) * 3 + u) * 1024 + 16 * lane);
				};
				read_k(0, f[0]);
#pragma unroll
				for (int kk = 0; kk < KK; ++kk)
				{
					if (kk + 1 < KK) read_k(kk + 1, f[(kk + 1) & 1]);
					__builtin_amdgcn_sched_barrier(0);
					mfma3<NA>(f[kk & 1], q[kk], sc);
					__builtin_amdgcn_sched_barrier(0);
				}
				t3_read_barrier(); // everyone is done with K
				load(st + 1, 0, s_k);

				// Online softmax of each row (offset, weights and their sum as in
				// tiled_kernel); P as the B operand: k-slot 4 t + i.
				u32x4 pw[NA][3];
#pragma unroll
				for (int a = 0; a < NA; ++a)
				{
					float cmax = -INFINITY;
#pragma unroll
					for (int t = 0; t < 2; ++t)
#pragma unroll
						for (int i = 0; i < 4; ++i)
						{
							const int k = k0 + 16 * t + 4 * c + i;
							sc[a][t][i] = (k >= r_lo[a] && k <= r_hi[a]) ? sc[a][t][i] : -INFINITY;
							cmax = fmaxf(cmax, sc[a][t][i]);
						}
					cmax = row4_max(cmax);
					const bool raise = cmax > m_run[a] + kTileLazy;
					if (__builtin_amdgcn_ballot_w64(raise))
					{
						const float alpha = raise && m_run[a] != -INFINITY ? fast_exp2(m_run[a] - cmax) : 1.0f;
						m_run[a] = raise ? cmax : m_run[a];
						l_run[a] *= alpha;
#pragma unroll
						for (int d = 0; d < DT / 2; ++d)
						{
							acc[d][a][0] *= alpha;
							acc[d][a][1] *= alpha;
						}
					}
					const float m_use = m_run[a] == -INFINITY ? 0.0f : m_run[a];
					float w[8], ls = 0.0f;
#pragma unroll
					for (int j = 0; j < 8; ++j)
					{
						w[j] = fast_exp2(sc[a][j >> 2][j & 3] - m_use);
						ls += w[j];
					}
					l_run[a] += row4_sum(ls);
					split3<kT3P>(w, pw[a]);
				}

				t3_wait_barrier<ND>(); // V has landed; the next K may be in flight
				auto read_v = [&](int d, u32x4 (&o)[2][3]) __attribute__((always_inline))
				{
#pragma unroll
					for (int t = 0; t < 2; ++t)
#pragma unroll
						for (int u = 0; u < 3; ++u)
							o[t][u] = *reinterpret_cast<const u32x4*>(s_v + ((d + t) * 3 + u) * 1024 + 16 * lane);
				};
				read_v(0, f[0]);
#pragma unroll
				for (int d = 0; d < DT; d += 2)
				{
					if (d + 2 < DT) read_v(d + 2, f[(d / 2 + 1) & 1]);
					__builtin_amdgcn_sched_barrier(0);
					mfma3<NA>(f[(d / 2) & 1], pw, acc[d / 2]);
					__builtin_amdgcn_sched_barrier(0);
				}
				t3_read_barrier(); // everyone is done with V
				load(st + 1, 1, s_v);
			}
			__builtin_amdgcn_sched_barrier(0);
			__builtin_amdgcn_s_waitcnt(0x0F70); // (zeros on their way to LDS)

#pragma unroll
			for (int a = 0; a < NA; ++a)
			{
				const int row = blockIdx.x * kT3Block + 16 * (NA * wave + a) + r16;
				if (row >= n_rows) continue;
				if (p.n_split > 1)
				{
					float* gp = tiled_partial(p, G, HD, row / G, kvh, z, row % G);
#pragma unroll
					for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4*>(gp + 16 * d + 4 * c) = acc[d / 2][a][d & 1];
					if (c == 0) *reinterpret_cast<float2*>(gp + HD) = make_float2(m_run[a], l_run[a]);
				}
				else
				{
					const float inv = l_run[a] > 0.0f ? 1.0f / l_run[a] : 0.0f;
#pragma unroll
					for (int d = 0; d < DT; ++d)
					{
						const size_t oi = qo[a] + 16 * d + 4 * c;
						float4 o;
						o.x = gated(acc[d / 2][a][d & 1][0] * inv, p.gate, oi);
						o.y = gated(acc[d / 2][a][d & 1][1] * inv, p.gate, oi + 1);
						o.z = gated(acc[d / 2][a][d & 1][2] * inv, p.gate, oi + 2);
						o.w = gated(acc[d / 2][a][d & 1][3] * inv, p.gate, oi + 3);
						*reinterpret_cast<float4*>(p.out + oi) = o;
					}
				}
			}
		}

		template <int HD>
		void launch_t3(const decode_params& p, int G, void* split, int k_lo, int k_hi, int g0, dim3 sgrid, dim3 grid,
		               hipStream_t stream)
		{
			tiled3_split_kernel<HD><<<sgrid, 256, 0, stream>>>(p, static_cast<char*>(split), k_lo, k_hi, g0);
			tiled3_kernel<HD><<<grid, 512 / kT3Tiles<HD>, 0, stream>>>(p, static_cast<const char*>(split), G, g0, sgrid.x);
		}

		template <int HD, int HDMAX>
		void launch_hd(const decode_params& p, int n_tok, int head_dim, int group, bool bf16, hipStream_t stream)
		{
			const dim3 grid((n_tok * group + kTileBlock - 1) / kTileBlock, p.n_kv, p.n_split);
			if (bf16)
				tiled_kernel<HD, HDMAX, true><<<grid, 64 * kTileWaves, 0, stream>>>(p, head_dim, group);
			else
				tiled_kernel<HD, HDMAX, false><<<grid, 64 * kTileWaves, 0, stream>>>(p, head_dim, group);
		}
	}

	bool launch_tiled(const decode_params& p, int n_tok, int head_dim, int group, bool bf16, hipStream_t stream)
	{
		if (!tiled_shape_ok(head_dim, group)) return false;
		switch (head_dim)
		{
		case 64: launch_hd<64, 64>(p, n_tok, head_dim, group, bf16, stream); break;
		case 80: launch_hd<80, 80>(p, n_tok, head_dim, group, bf16, stream); break;
		case 96: launch_hd<96, 96>(p, n_tok, head_dim, group, bf16, stream); break;
		case 128: launch_hd<128, 128>(p, n_tok, head_dim, group, bf16, stream); break;
		case 256: launch_hd<256, 256>(p, n_tok, head_dim, group, bf16, stream); break;
		case 512: launch_hd<512, 512>(p, n_tok, head_dim, group, bf16, stream); break;
		default:
			if (head_dim <= 128)
				launch_hd<0, 128>(p, n_tok, head_dim, group, bf16, stream);
			else if (head_dim <= 256)
				launch_hd<0, 256>(p, n_tok, head_dim, group, bf16, stream);
			else
				launch_hd<0, 512>(p, n_tok, head_dim, group, bf16, stream);
		}
		if (p.n_split > 1)
			tiled_merge_kernel<kTileBlock, 1><<<dim3((n_tok * group + 3) / 4, p.n_kv), 256, 0, stream>>>(p, head_dim, group);
		return true;
	}

	bool launch_tiled3(const decode_params& p, int n_tok, int head_dim, int group, void* split, int k_lo, int k_hi,
	                   hipStream_t stream)
	{
		const int g0 = k_lo / kT3Keys, n_g = k_hi / kT3Keys - g0 + 1;
		const dim3 sgrid(n_g, p.n_kv), grid((n_tok * group + kT3Block - 1) / kT3Block, p.n_kv, p.n_split);
		switch (head_dim)
		{
		case 64: launch_t3<64>(p, group, split, k_lo, k_hi, g0, sgrid, grid, stream); break;
		case 128: launch_t3<128>(p, group, split, k_lo, k_hi, g0, sgrid, grid, stream); break;
		case 256: launch_t3<256>(p, group, split, k_lo, k_hi, g0, sgrid, grid, stream); break;
		default: return false;
		}
		if (p.n_split > 1)
			tiled_merge_kernel<kT3Block, kT3Keys><<<dim3((n_tok * group + 3) / 4, p.n_kv), 256, 0, stream>>>(p, head_dim, group);
		return true;
	}
}
