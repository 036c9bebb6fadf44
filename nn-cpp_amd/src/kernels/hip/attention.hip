// attention.hip - nn::attention's forward (src/autograd/ops.cpp:1226-1261) as one kernel for head width 64.
//
// A workgroup owns 32 query rows of one (sample, head) pair and runs the reference's three steps for them
// with the score rows resident in LDS:
//   1. S = Q_h K_h^T: each element the fma chain over d = 0..63 from +0 (sgemm F,T, ops.cpp:1256). A wave takes 64
//      keys against the 32 queries, computing S^T (the product fma(k, q, acc) is the reference's fma(q, k, acc)).
//   2. masked_softmax_row (ops.cpp:1183-1204) over the 32 rows: scale and mask, std::max's scan, glibc's
//      expf, the sum over live keys in key order, the division; the probabilities go to `probs` (kept for the
//      backward pass) and stay in LDS.
//   3. O_h = P V_h: each element the fma chain over the keys j = 0..Tk-1 from +0 (sgemm F,F, ops.cpp:1259),
//      every key included (a zero probability still meets its V entry). Wave w takes output columns 16w..16w+15;
//      P comes from LDS, V from global memory 16 steps of four keys ahead.
// Same bits as the three-launch path (batched GEMM, row softmax, batched GEMM): both sgemm shapes are below
// nn-cpp's depth cut (k = 64 and k = Tk <= 256), so every element is a single chain.
// What bounds the forward: the vector ALUs and the matrix cores in turn (a third of the issue cycles each) and the
// waits between the phases. Four workgroups share a CU (34 KB of LDS each at Tk = 256, 128 registers a lane), so one's
// MFMA phases overlap another's VALU phases. Measured at 32 x 8 heads x 256 x 64 (us): 64 rows a workgroup and two
// workgroups a CU 85, 32 rows 81, and 74 with a third of the vector instructions taken out (rows summed by one wave
// for 32 rows at once, V's addresses kept uniform, no division by Tk, one test for 16 exponentials' special cases).
#include "attention.hpp"

#include <algorithm>

#include "gemm.hpp"

#include "gemm_tile.hpp"
#include "softmax_row.hpp"

namespace nnh {

namespace {

constexpr int kRows = 32;          // query rows per workgroup
constexpr int kDh = 64;            // head width
constexpr int kMaxKeys = 256;     // four waves of 64 keys
constexpr int64_t kMaxGrid = ((int64_t)1 << 24) - 1;  // workgroups of 256 threads: below 2^32 work-items a launch

struct FusedArgs {
	const float* q;
	const float* k;
	const float* v;
	float* out;
	float* probs;
	const float* pad;  // {N, Tk}, 0 marks a padded key; or null
	int heads, tq, tk, d;
	int qblocks, total;
	int causal;
	float scale;
};

// LDS row stride of the scores: whole groups of 16 keys (four steps of the 16x16x4 product for each lane group) and
// four floats more, so that the 16-byte reads of 16 rows hit distinct banks.
__host__ __device__ constexpr int score_stride(int tk) { return (tk + 15) / 16 * 16 + 4; }

static_assert(4 * kRows * score_stride(kMaxKeys) <= 64 * 1024, "no launch asks for more LDS than the default limit");

// The 64-float rows' operand of the 16x16x4 product from 16-byte loads: lane (g, i) loads floats 16c + 4g .. + 3 of
// its row i and needs floats 16c + 4s + g (s = 0..3), the transpose of four registers over the four lane groups.
__device__ __forceinline__ f32x4 lane_groups_transposed(const f32x4& x) {
	auto bits = [](float v) { return __builtin_bit_cast(unsigned, v); };
	auto flt = [](unsigned v) { return __builtin_bit_cast(float, v); };
	const auto a = __builtin_amdgcn_permlane32_swap(bits(x[0]), bits(x[2]), false, false);
	const auto b = __builtin_amdgcn_permlane32_swap(bits(x[1]), bits(x[3]), false, false);
	const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
	const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
	return f32x4{flt(c[0]), flt(c[1]), flt(d[0]), flt(d[1])};
}

// Phase 1, shared by the forward and the backward: (R K^T)^T for the 32 rows of R (row stride d, nr of them valid)
// against keys key0 .. key0 + 63 of K (row stride d, tk valid): s[t][u] of lane (g, i) holds keys key0 + 16t + 4g ..
// + 3 of row 16u + i, each element the fma chain over d = 0..63 from +0 on the 16x16x4 MFMA (two independent chains a
// wave). Tiles of 16 keys from `limit` on stay +0. Both operands come straight from global memory, 64 bytes of 16 rows
// a load instruction; a lane holding one key row whole would load 16 bytes of 64 rows at a time (the dS kernel 49 us
// against 45 so).
using M4 = Mfma<kMf16x4>;
constexpr int kTiles = kRows / 16, kKeyTiles = 4;

__device__ __forceinline__ void rows_times_keys(const float* rp, int nr, const float* kp, int tk, int key0, int limit,
                                                int d, M4::Acc (&s)[kKeyTiles][kTiles]) {
	const int lane = threadIdx.x & 63, g = lane >> 4, il = lane & 15;
#pragma unroll
	for (int t = 0; t < kKeyTiles; ++t)
#pragma unroll
		for (int u = 0; u < kTiles; ++u) s[t][u] = M4::Acc{0.0f, 0.0f, 0.0f, 0.0f};
	if (key0 >= limit) return;  // uniform
	// loads are unconditional (indices clamped into range) so that they are in flight together; values past the end
	// are never used
	auto load = [&](f32x4 (&dst)[kDh / 16], const float* base, int row) {
#pragma unroll
		for (int c = 0; c < kDh / 16; ++c) dst[c] = *reinterpret_cast<const f32x4*>(base + (int64_t)row * d + 16 * c + 4 * g);
	};
	f32x4 q[kTiles][kDh / 16], k[2][kDh / 16];
#pragma unroll
	for (int u = 0; u < kTiles; ++u) load(q[u], rp, min(16 * u + il, nr - 1));
	load(k[0], kp, min(key0 + il, tk - 1));
#pragma unroll
	for (int u = 0; u < kTiles; ++u)
#pragma unroll
		for (int c = 0; c < kDh / 16; ++c) q[u][c] = lane_groups_transposed(q[u][c]);
#pragma unroll
	for (int t = 0; t < kKeyTiles; ++t) {
		if (key0 + 16 * t >= limit) return;  // uniform
		if (t + 1 < kKeyTiles) load(k[(t + 1) & 1], kp, min(key0 + 16 * (t + 1) + il, tk - 1));
#pragma unroll
		for (int c = 0; c < kDh / 16; ++c) {
			const f32x4 kc = lane_groups_transposed(k[t & 1][c]);
#pragma unroll
			for (int e = 0; e < 4; ++e)
#pragma unroll
				for (int u = 0; u < kTiles; ++u) s[t][u] = M4::mma(kc[e], q[u][c][e], s[t][u]);
		}
	}
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) attention_fused_kernel(const FusedArgs a) {
	extern __shared__ __align__(16) float sm[];
	__shared__ unsigned long long table[32];
	__shared__ float rowmax[kRows], rowsum[kRows];
	__shared__ double rowinv[kRows];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int lid = xcd_remap(blockIdx.x, a.total);  // the query blocks of one head share an XCD's L2
	const int nh = lid / a.qblocks, qb = lid - nh * a.qblocks;
	const int n = nh / a.heads, h = nh - n * a.heads;
	const int i0 = qb * kRows, nq = min(kRows, a.tq - i0);
	const int tk = a.tk, ldp = score_stride(tk);
	const float* qp = a.q + ((int64_t)n * a.tq + i0) * a.d + h * kDh;
	const float* kp = a.k + (int64_t)n * tk * a.d + h * kDh;
	const float* vp = a.v + (int64_t)n * tk * a.d + h * kDh;
	const float* padrow = a.pad ? a.pad + (int64_t)n * tk : nullptr;
	if (tid < 32) table[tid] = kExp2Table[tid];

	// 1. S^T (fma(k, q, acc) is the reference's fma(q, k, acc)). Scores past the block's causal limit are replaced
	// below whatever they are and not computed; the waves' key blocks rotate over the workgroups, so that every SIMD
	// gets short and long ones.
	const int kw = (wave + lid) & 3, g = lane >> 4, il = lane & 15;
	const int block_live = a.causal ? min(tk, i0 + nq) : tk;  // keys any row of the block reaches
	M4::Acc s[kKeyTiles][kTiles];
	rows_times_keys(qp, nq, kp, tk, 64 * kw, block_live, a.d, s);

	// 2a. scaled and masked scores into LDS (ops.cpp:1186-1191): four consecutive keys of one query a 16-byte store
	f32x4* sm4 = reinterpret_cast<f32x4*>(sm);
	const int ldp4 = ldp / 4;
	{
		const bool masked = padrow != nullptr || a.causal;
#pragma unroll
		for (int t = 0; t < kKeyTiles; ++t) {
			const int j = 64 * kw + 16 * t + 4 * g;
#pragma unroll
			for (int u = 0; u < kTiles; ++u) {
				const int row = 16 * u + il;
				f32x4 val;
#pragma unroll
				for (int c = 0; c < 4; ++c) val[c] = s[t][u][c] * a.scale;
				if (masked) {  // uniform
					const f32x4 pd = padrow ? *reinterpret_cast<const f32x4*>(padrow + min(j, tk - 4)) : f32x4{1, 1, 1, 1};
#pragma unroll
					for (int c = 0; c < 4; ++c) {
						val[c] = pd[c] == 0.0f ? -1e9f : val[c];
						val[c] = a.causal && j + c > i0 + row ? -2e9f : val[c];
					}
				}
				if (row < nq && j < tk) sm4[row * ldp4 + j / 4] = val;  // tk % 4 == 0: the quad is whole
			}
		}
	}
	__syncthreads();

	// 2b. the row maxima: std::max's scan is v_0 when v_0 is NaN, else the largest non-NaN value, which fmaxf
	// gives in any order (a zero maximum's sign cannot change v - m or its exp). Eight lanes per row.
	{
		const int row = 8 * wave + (lane >> 3), q = lane & 7;
		float m = __builtin_nanf("");
		if (row < nq) {
			const float* o = sm + row * ldp;
			for (int j = 4 * q; j < tk; j += 32) {
				const f32x4 x = *reinterpret_cast<const f32x4*>(o + j);
				m = fmaxf(m, fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
			}
		}
		m = fmaxf(m, __shfl_xor(m, 1));
		m = fmaxf(m, __shfl_xor(m, 2));
		m = fmaxf(m, __shfl_xor(m, 4));
		if (row < nq && q == 0) {
			const float first = sm[row * ldp];
			rowmax[row] = first != first ? first : m;
		}
	}
	__syncthreads();

	// 2c. p_j = exp(v_j - m) for the live keys, exact zeros past the causal limit (ops.cpp:1197-1201). Half wave h of
	// the eight takes the quads of keys h, h + 8, ... of its lanes' 32 rows, kExpQuads of them at a time so that their
	// table reads and double-precision chains overlap. Keys past a row's causal limit take exp(0) in place of
	// exp(-2e9 - m), whose result is replaced by an exact zero, which keeps waves out of exp's special-case path (padded
	// keys stay live and go through exp). Quads past the block's last live key are zero for every row: they are stored
	// without computing anything.
	{
		constexpr int kExpQuads = 4, kHalves = 8;
		const int row = lane & 31, nq4 = tk / 4;
		const float m = rowmax[min(row, nq - 1)];
		const int live = a.causal ? min(tk, i0 + row + 1) : tk;
		f32x4* orow = sm4 + row * ldp4;
		for (int q0 = 2 * wave + (lane >> 5); q0 < nq4; q0 += kHalves * kExpQuads) {
			if (4 * q0 >= block_live) {  // this and every later quad of the half wave is dead for all rows
				if (row < nq) {
#pragma unroll
					for (int h2 = 0; h2 < kExpQuads; ++h2)
						if (q0 + kHalves * h2 < nq4) orow[q0 + kHalves * h2] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
				}
				continue;
			}
			f32x4 x[kExpQuads];
			float ex[4 * kExpQuads];
#pragma unroll
			for (int h2 = 0; h2 < kExpQuads; ++h2) x[h2] = orow[min(q0 + kHalves * h2, nq4 - 1)];
			// uniform: no key of the wave's quads is past any row's limit
			const bool whole = !a.causal || 4 * (q0 + kHalves * (kExpQuads - 1) + 1) + 3 <= i0;
			if (__all(whole)) {
#pragma unroll
				for (int e = 0; e < 4 * kExpQuads; ++e) ex[e] = x[e / 4][e % 4] - m;
				expf_glibc_n(ex, table);
			} else {
#pragma unroll
				for (int e = 0; e < 4 * kExpQuads; ++e)
					ex[e] = 4 * (q0 + kHalves * (e / 4)) + e % 4 < live ? x[e / 4][e % 4] - m : 0.0f;
				expf_glibc_n(ex, table);
#pragma unroll
				for (int e = 0; e < 4 * kExpQuads; ++e)
					ex[e] = 4 * (q0 + kHalves * (e / 4)) + e % 4 < live ? ex[e] : 0.0f;
			}
			if (row < nq) {
#pragma unroll
				for (int h2 = 0; h2 < kExpQuads; ++h2) {
					const int q = q0 + kHalves * h2;
					if (q < nq4) orow[q] = f32x4{ex[4 * h2], ex[4 * h2 + 1], ex[4 * h2 + 2], ex[4 * h2 + 3]};
				}
			}
		}
	}
	__syncthreads();

	// 2d. the sum over the live keys in key order from +0, one lane per row (ops.cpp:1198-1200): all rows in one wave,
	// whose adds issue once for 32 rows, another wave for another workgroup
	if (wave == ((lid >> 2) & 3)) {
		const int row = lane;
		if (row < nq) {
			const float* o = sm + row * ldp;
			const int live = a.causal ? min(tk, i0 + row + 1) : tk;
			float sum = 0.0f;
			int j = 0;
			for (; j + 16 <= live; j += 16) {
				f32x4 x[4];
#pragma unroll
				for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const f32x4*>(o + j + 4 * u);
#pragma unroll
				for (int u = 0; u < 4; ++u) {
					sum += x[u][0];
					sum += x[u][1];
					sum += x[u][2];
					sum += x[u][3];
				}
			}
			for (; j < live; ++j) sum += o[j];
			rowsum[row] = sum;
			rowinv[row] = 1.0 / (double)sum;
		}
	}
	__syncthreads();

	// 2e. p_j / sum into probs (ops.cpp:1203) and back into LDS as the 16x16x4 product below reads its rows: key j at
	// (j % 4) q4 + j / 4, q4 = Tk / 4 rounded up to 4. Every quad is read and divided first, then, after a barrier,
	// written back in that order. A thread has quads il, il + 16, ... of rows 4g + w and 16 + 4g + w: 256-byte pieces
	// of a row in memory, and the four rows of a wave's 4-byte LDS stores 16 banks apart.
	const int steps = tk >> 2, q4 = (steps + 3) & ~3;
	{
		float* pr = a.probs + ((int64_t)nh * a.tq + i0) * tk;
		constexpr int kPer = kMaxKeys / 64;
		f32x4 yv[kTiles][kPer];
#pragma unroll
		for (int u = 0; u < kTiles; ++u) {
			const int row = 16 * u + 4 * g + wave;
			if (row < nq) {
				const float sum = rowsum[row];
				const double inv = rowinv[row];
#pragma unroll
				for (int x = 0; x < kPer; ++x) {
					const int jq = il + 16 * x;
					if (jq < steps) {
						const f32x4 v = sm4[row * ldp4 + jq];
						float y[4] = {v[0], v[1], v[2], v[3]};
						div_n_by_row_sum(y, sum, inv);
						yv[u][x] = f32x4{y[0], y[1], y[2], y[3]};
						*reinterpret_cast<f32x4*>(pr + row * tk + 4 * jq) = yv[u][x];
					}
				}
			}
		}
		__syncthreads();
#pragma unroll
		for (int u = 0; u < kTiles; ++u) {
			const int row = 16 * u + 4 * g + wave;
#pragma unroll
			for (int x = 0; x < kPer; ++x) {
				const int jq = il + 16 * x;
				if (row < nq && jq < steps)
#pragma unroll
					for (int c = 0; c < 4; ++c) sm[row * ldp + c * q4 + jq] = yv[u][x][c];
			}
		}
	}
	__syncthreads();

	// 3. O columns 16w .. 16w+15 for the 32 rows on the 16x16x4 MFMA (Mfma<kMf16x4>: four keys per instruction,
	// bit for bit four fmas in key order): two 16-row tiles, two independent chains over every key. At step s
	// lane (g, i) supplies P[16 t + i][4 s + g], read four steps at a time from the permuted rows (positions
	// g q4 + s; steps past the last one are read, never used, and rows past nq hold stale values, never stored), and
	// V[4 s + g][16 w + i], loaded 16 steps ahead.
	M4::Acc acc4[kTiles];
#pragma unroll
	for (int t = 0; t < kTiles; ++t) acc4[t] = M4::Acc{0.0f, 0.0f, 0.0f, 0.0f};
	// V's row of a step: a uniform address (the step's first key) and the lane's offset, one key a lane group
	const unsigned vlane = (unsigned)g * (unsigned)a.d + (unsigned)(16 * wave + il);
	auto v_at = [&](int step) { return (vp + (int64_t)(4 * min(step, steps - 1)) * a.d)[vlane]; };
	const float* pbase = sm + il * ldp + g * q4;
	auto load_v = [&](float (&dst)[16], int s0) {  // steps s0 .. s0 + 15 (clamped rows are loaded, never used)
#pragma unroll
		for (int u = 0; u < 16; ++u) dst[u] = v_at(s0 + u);
	};
	auto load_p = [&](f32x4 (&dst)[kTiles], int s0) {  // steps s0 .. s0 + 3 of the tiles
#pragma unroll
		for (int t = 0; t < kTiles; ++t) dst[t] = *reinterpret_cast<const f32x4*>(pbase + 16 * t * ldp + min(s0, q4 - 4));
	};
	float v0[16], v1[16];
	f32x4 pa[kTiles], pb[kTiles];
	auto chunk = [&](const float (&v)[16], int s0) {  // 16 steps from s0, P one group of four steps ahead
		load_p(pa, s0);
#pragma unroll
		for (int h4 = 0; h4 < 4; ++h4) {
			f32x4 (&cur)[kTiles] = (h4 & 1) ? pb : pa;
			f32x4 (&nxt)[kTiles] = (h4 & 1) ? pa : pb;
			if (h4 < 3) load_p(nxt, s0 + 4 * (h4 + 1));
#pragma unroll
			for (int e = 0; e < 4; ++e)
#pragma unroll
				for (int t = 0; t < kTiles; ++t) acc4[t] = M4::mma(cur[t][e], v[4 * h4 + e], acc4[t]);
		}
	};
	load_v(v0, 0);  // chunks of 16 steps, V two chunks ahead
	load_v(v1, 16);
	int s0 = 0;
	for (; s0 + 32 <= steps; s0 += 32) {
		chunk(v0, s0);
		load_v(v0, s0 + 32);
		chunk(v1, s0 + 16);
		load_v(v1, s0 + 48);
	}
	// the rest: fewer than 32 steps, in groups of four, of which the last may be partial
	for (; s0 < steps; s0 += 4) {
		float vv[4];
		f32x4 pp[kTiles];
		load_p(pp, s0);
#pragma unroll
		for (int e = 0; e < 4; ++e) vv[e] = v_at(s0 + e);
#pragma unroll
		for (int e = 0; e < 4; ++e)
			if (s0 + e < steps) {  // uniform
#pragma unroll
				for (int t = 0; t < kTiles; ++t) acc4[t] = M4::mma(pp[t][e], vv[e], acc4[t]);
			}
	}
	float* op = a.out + ((int64_t)n * a.tq + i0) * a.d + h * kDh + 16 * wave + il;
#pragma unroll
	for (int t = 0; t < kTiles; ++t)
#pragma unroll
		for (int r = 0; r < 4; ++r) {
			const int row = 16 * t + 4 * g + r;
			if (row < nq) op[(int64_t)row * a.d] = acc4[t][r];
		}
}

struct DScoresArgs {
	const float* g;      // upstream gradient {N, Tq, D}
	const float* v;
	const float* probs;  // the forward's {N, heads, Tq, Tk}
	float* ds;           // {N, heads, Tq, Tk}
	const float* pad;
	int heads, tq, tk, d;
	int qblocks, total;
	int causal;
	float scale;
};

// The first half of nn::attention's backward for 32 query rows of one (sample, head) pair (ops.cpp:1286-1290):
//   dP = G_h V_h^T                     each element the fma chain over d = 0..63 from +0 (sgemm F,T)
//   dot_i = sum_j dP_ij * y_ij         the products rounded, then added in key order from +0
//   dS_ij = masked ? 0 : scale * (y_ij * (dP_ij - dot_i)) + 0     (masked_softmax_row_backward, ops.cpp:1216-1224)
// dP stays in the MFMA accumulators (wave w holds keys 64w..64w+63 of the 32 rows, four consecutive keys per
// four registers); y is loaded in the same layout; only the products dP y go through LDS, where one lane per
// row adds them in key order. dS is written to HBM for the dQ and dK products.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) attention_dscores_kernel(const DScoresArgs a) {
	extern __shared__ __align__(16) float sm[];
	__shared__ float rowdot[kRows];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int lid = xcd_remap(blockIdx.x, a.total);
	const int nh = lid / a.qblocks, qb = lid - nh * a.qblocks;
	const int n = nh / a.heads, h = nh - n * a.heads;
	const int i0 = qb * kRows, nq = min(kRows, a.tq - i0);
	const int tk = a.tk, ldp4 = score_stride(tk) / 4;
	const float* gp = a.g + ((int64_t)n * a.tq + i0) * a.d + h * kDh;
	const float* vp = a.v + (int64_t)n * tk * a.d + h * kDh;
	const float* yp = a.probs + ((int64_t)nh * a.tq + i0) * tk;
	float* dsp = a.ds + ((int64_t)nh * a.tq + i0) * tk;
	const float* padrow = a.pad ? a.pad + (int64_t)n * tk : nullptr;
	f32x4* sm4 = reinterpret_cast<f32x4*>(sm);

	// dP^T; y in the accumulators' layout: y[t][u] is row 16u + i, keys key0 + 16t + 4g .. + 3 (rows and keys clamped
	// into range; values outside are never used)
	const int key0 = 64 * wave, g = lane >> 4, il = lane & 15;
	M4::Acc s[kKeyTiles][kTiles];
	rows_times_keys(gp, nq, vp, tk, key0, tk, a.d, s);
	f32x4 y[kKeyTiles][kTiles];
	if (key0 < tk) {
#pragma unroll
		for (int t = 0; t < kKeyTiles; ++t)
#pragma unroll
			for (int u = 0; u < kTiles; ++u)
				y[t][u] = *reinterpret_cast<const f32x4*>(yp + (int64_t)min(16 * u + il, nq - 1) * tk +
				                                          min(key0 + 16 * t + 4 * g, tk - 4));
		// the products dP y, rounded, into LDS (tk % 4 == 0: every quad is whole)
#pragma unroll
		for (int t = 0; t < kKeyTiles; ++t) {
			const int j = key0 + 16 * t + 4 * g;
#pragma unroll
			for (int u = 0; u < kTiles; ++u) {
				const int row = 16 * u + il;
				f32x4 prod;
#pragma unroll
				for (int c = 0; c < 4; ++c) prod[c] = s[t][u][c] * y[t][u][c];
				if (row < nq && j < tk) sm4[row * ldp4 + j / 4] = prod;
			}
		}
	}
	__syncthreads();

	// dot_i: one lane per row, every key in order from +0
	{
		const int r = lane;
		if (wave == ((lid >> 2) & 3) && r < nq) {
			const f32x4* o = sm4 + r * ldp4;
			float dot = 0.0f;
			int q = 0;
			for (; q + 4 <= tk / 4; q += 4) {
				f32x4 x[4];
#pragma unroll
				for (int u = 0; u < 4; ++u) x[u] = o[q + u];
#pragma unroll
				for (int u = 0; u < 4; ++u) {
					dot += x[u][0];
					dot += x[u][1];
					dot += x[u][2];
					dot += x[u][3];
				}
			}
			for (; q < tk / 4; ++q) {
				const f32x4 x = o[q];
				dot += x[0];
				dot += x[1];
				dot += x[2];
				dot += x[3];
			}
			rowdot[r] = dot;
		}
	}
	__syncthreads();

	// dS from the registers
	if (key0 < tk) {
		const bool masked = padrow != nullptr || a.causal;
#pragma unroll
		for (int u = 0; u < kTiles; ++u) {
			const int row = 16 * u + il;
			const float dot = rowdot[min(row, nq - 1)];
#pragma unroll
			for (int t = 0; t < kKeyTiles; ++t) {
				const int j = key0 + 16 * t + 4 * g;
				f32x4 r;
#pragma unroll
				for (int c = 0; c < 4; ++c) r[c] = a.scale * (y[t][u][c] * (s[t][u][c] - dot)) + 0.0f;
				if (masked) {  // uniform
					const f32x4 pd = padrow ? *reinterpret_cast<const f32x4*>(padrow + min(j, tk - 4)) : f32x4{1, 1, 1, 1};
#pragma unroll
					for (int c = 0; c < 4; ++c)
						r[c] = pd[c] == 0.0f || (a.causal && j + c > i0 + row) ? 0.0f : r[c];
				}
				if (row < nq && j < tk) *reinterpret_cast<f32x4*>(dsp + (int64_t)row * tk + j) = r;
			}
		}
	}
}

}  // namespace

bool attention_fused_ok(int64_t tq, int64_t tk, int64_t dh, int64_t d, const void* q, const void* k, const void* v,
                        const void* out, const void* probs, const void* pad) {
	auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
	// the kernel runs S = Q K^T and O = P V as whole-depth chains: products that take the depth cut go elsewhere
	if (depth_cut(tq, tk, dh) || depth_cut(tq, dh, tk)) return false;
	// one sample's blocks in a launch
	if (dh != kDh || d / kDh * ((tq + kRows - 1) / kRows) > kMaxGrid) return false;
	return tk >= 1 && tk <= kMaxKeys && tk % 4 == 0 && d % 4 == 0 && tq >= 1 && tq < (1 << 24) &&
	       al(q) && al(k) && al(v) && al(out) && al(probs) && (pad == nullptr || al(pad));
}

hipError_t attention_fused_forward(const float* q, const float* k, const float* v, int64_t n, int64_t tq, int64_t tk,
                                   int64_t d, int64_t heads, const float* pad, int causal, float scale, float* out,
                                   float* probs, hipStream_t s) {
	const int64_t qblocks = (tq + kRows - 1) / kRows, total = n * heads * qblocks;
	if (total == 0) return hipSuccess;
	if (total >= ((int64_t)1 << 31) || n * heads * tq * tk >= ((int64_t)1 << 62)) return hipErrorInvalidValue;
	FusedArgs a;
	a.heads = (int)heads;
	a.tq = (int)tq;
	a.tk = (int)tk;
	a.d = (int)d;
	a.qblocks = (int)qblocks;
	a.causal = causal ? 1 : 0;
	a.scale = scale;
	const int lds = 4 * kRows * score_stride((int)tk);
	const int64_t most = kMaxGrid / (heads * qblocks);  // samples of a launch
	for (int64_t n0 = 0; n0 < n; n0 += most) {
		const int64_t q0 = n0 * tq * d, k0 = n0 * tk * d, cnt = std::min(most, n - n0);
		a.q = q + q0;
		a.k = k + k0;
		a.v = v + k0;
		a.out = out + q0;
		a.probs = probs + n0 * heads * tq * tk;
		a.pad = pad ? pad + n0 * tk : nullptr;
		a.total = (int)(cnt * heads * qblocks);
		hipLaunchKernelGGL(attention_fused_kernel, dim3((unsigned)a.total), dim3(256), lds, s, a);
		const hipError_t e = hipGetLastError();
		if (e != hipSuccess) return e;
	}
	return hipSuccess;
}

hipError_t attention_fused_dscores(const float* g, const float* v, const float* probs, int64_t n, int64_t tq, int64_t tk,
                                   int64_t d, int64_t heads, const float* pad, int causal, float scale, float* ds,
                                   hipStream_t s) {
	const int64_t qblocks = (tq + kRows - 1) / kRows, total = n * heads * qblocks;
	if (total == 0) return hipSuccess;
	if (total >= ((int64_t)1 << 31) || n * heads * tq * tk >= ((int64_t)1 << 62)) return hipErrorInvalidValue;
	DScoresArgs a;
	a.heads = (int)heads;
	a.tq = (int)tq;
	a.tk = (int)tk;
	a.d = (int)d;
	a.qblocks = (int)qblocks;
	a.causal = causal ? 1 : 0;
	a.scale = scale;
	const int lds = 4 * kRows * score_stride((int)tk);
	const int64_t most = kMaxGrid / (heads * qblocks);  // samples of a launch
	for (int64_t n0 = 0; n0 < n; n0 += most) {
		const int64_t p0 = n0 * heads * tq * tk, cnt = std::min(most, n - n0);
		a.g = g + n0 * tq * d;
		a.v = v + n0 * tk * d;
		a.probs = probs + p0;
		a.ds = ds + p0;
		a.pad = pad ? pad + n0 * tk : nullptr;
		a.total = (int)(cnt * heads * qblocks);
		hipLaunchKernelGGL(attention_dscores_kernel, dim3((unsigned)a.total), dim3(256), lds, s, a);
		const hipError_t e = hipGetLastError();
		if (e != hipSuccess) return e;
	}
	return hipSuccess;
}

}  // namespace nnh
