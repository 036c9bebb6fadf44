// gemm_ring.hpp - the fp32 tile GEMM with its operands streamed straight from global memory into a ring of LDS stages.
//
// Same numbers as gemm_tile.hpp: every output is one fused multiply-add chain over the whole depth in increasing k from
// +0, advanced four steps per 16x16x4 MFMA, old C joining after the first min(K, 256) steps when accumulating, steps
// past the depth padded with A = +0 and B = -0. Results are a pure function of the inputs.
//
// What bounds it: the matrix cores (32 cycles a 16x16x4 MFMA per SIMD), so everything else has to hide behind them.
//   * global_load_lds writes the operands into LDS without passing through registers: a stage costs a wave a handful
//     of load instructions, no register ring and no LDS stores, and up to ST - 1 stages are in flight.
//   * One barrier a stage. At the barrier of stage kt every wave has waited (by count) for its own loads of stage
//     kt + 1, so during stage kt the next stage is already readable and its first fragments are read behind the last
//     MFMAs of this one: no wave waits for LDS after a barrier.
//   * LDS cannot be padded (a load writes 64 lanes' data back to back), so the bank conflicts are taken out by
//     permuting what each lane loads: a k-contiguous tile ([row][BK]) stores the 4-float chunk c of a row at chunk
//     c ^ swizzle(row), an m/n-contiguous tile ([BK][rows]) stores row block b (16 rows) of depth k at b ^ (k & 3). The
//     64 lanes of a fragment read (16 rows x 4 depths) then hit 64 different banks.
//   * The MFMA is issued with the operands exchanged (C^T = B^T A^T, the same products and the same chain), so a lane
//     holds four consecutive columns of a row of C and stores them as one 16-byte word, with no transpose through LDS.
//   * V = 1 loads one float per lane instead of four, for rows that are not 16-byte aligned or whose length is not a
//     multiple of four: four times the load instructions, still far below the MFMAs' issue time.
// The depth is at least one (ring_ok). Rows and columns past the edge are read from the last valid ones (their outputs are not stored); depth past k is
// read from the last valid depth and then overwritten in LDS with the padding.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gelu_math.hpp"
#include "gemm_tile.hpp"

namespace nnh {

template <int BM, int BN, int BK, int WM, int WN, int ST, bool TA, bool TB, int V>
struct RingShape {
	static constexpr int kWavesN = BN / WN;
	static constexpr int kWaves = (BM / WM) * (BN / WN);
	static constexpr int kThreads = 64 * kWaves;
	static constexpr int I = WM / 16, J = WN / 16;
	static constexpr int kA = BM * BK, kB = BN * BK, kStage = kA + kB;
	// k-contiguous operands stored in fragment order (ring::kc_index), where one float a lane is loaded anyway. Loading
	// single floats for its sake cost more than its quarter of the reads gave (512^3 A B on 32 x 32 tiles 7.1 -> 7.7 us).
	static constexpr bool kFrag = V == 1;
	static constexpr int kPer = 64 * V;  // floats a load instruction moves
	static constexpr int LA = kA / (kPer * kWaves), LB = kB / (kPer * kWaves);
	static constexpr int L = LA + LB;        // load instructions of a wave per stage
	static constexpr int kLdsBytes = ST * kStage * 4;
	static_assert(LA * kPer * kWaves == kA && LB * kPer * kWaves == kB, "a stage splits evenly over the waves");
	static_assert(WM % 16 == 0 && WN % 16 == 0 && BM % WM == 0 && BN % WN == 0, "whole 16 x 16 blocks");
	static_assert(BK % 32 == 0 && kAccAfter % BK == 0, "an even number of 16-deep groups; 256 on a stage boundary");
	static_assert(ST >= 3 && ST <= 5, "the tail is written out for 5 stages");
	// the wait that leaves `stages` whole stages outstanding (a wave counts at most 63 loads: then it waits for more)
	static constexpr int waits(int stages) { return stages * L < 63 ? stages * L : 63; }
	static_assert(kLdsBytes <= 160 * 1024, "gfx950 has 160 KiB of LDS per CU");
};

namespace ring {

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void global_void;

// Waits until at most N of the wave's loads into LDS are outstanding and its LDS reads have returned, then meets the
// other waves. The memory clobber keeps every LDS access of the program on its side.
template <int N>
__device__ __forceinline__ void wait_and_meet() {
	asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// The swizzle of a row of a k-contiguous tile: chunk c of the row lives at c ^ swz(row).
template <int BK>
__device__ __forceinline__ int swz(int row) {
	constexpr int kRowsPerBankLine = BK >= 64 ? 1 : 64 / BK;
	return (row / kRowsPerBankLine) & ((BK >= 64 ? 16 : BK / 4) - 1);
}

// The same for an m/n-contiguous tile of R rows: the offset XORed onto the row index at depth k (a multiple of 16).
template <int R>
__device__ __forceinline__ int kswz(int k) {
	return R >= 64 ? 16 * (k & 3) : R == 32 ? 16 * ((k >> 1) & 1) : 0;
}

// Where row `row`, depth k of a k-contiguous tile lives. FRAG (fragment order): every 16 depths are stored lane group
// by lane group, depth 4 t + g at position 4 g + t, so that a lane's operands of four MFMAs are one 16-byte read.
template <int BK, bool FRAG>
__device__ __forceinline__ int kc_index(int row, int k) {
	const int c = FRAG ? (k / 16) * 4 + k % 4 : k / 4, e = FRAG ? (k / 4) % 4 : k % 4;
	return row * BK + 4 * (c ^ swz<BK>(row)) + e;
}

// Float offset, from the tile's first element, of what lane `lane` loads with the load instruction that fills LDS
// floats [64 V q, 64 V (q + 1)) of the tile. KC: k-contiguous (rows of BK, FRAG as above), else depth rows of R. rows:
// valid rows of the tile (>= 1; with V = 4 and !KC a multiple of 4), depth: valid depth of the stage (>= 1; with V = 4
// and KC a multiple of 4).
template <bool KC, bool FRAG, int R, int BK, int V>
__device__ __forceinline__ unsigned src_offset(int q, int lane, int64_t ld, int rows, int depth) {
	static_assert(V == 1 || !KC || !FRAG, "fragment order moves single floats");
	const int pos = (q * 64 + lane) * V;
	if (KC) {
		const int row = pos / BK, e = pos % BK;
		const int c = (e / 4) ^ swz<BK>(row);
		const int k = FRAG ? 16 * (c / 4) + 4 * (e % 4) + c % 4 : 4 * c + (V == 1 ? e % 4 : 0);
		return (unsigned)min(row, rows - 1) * (unsigned)ld + (unsigned)min(k, depth - V);
	}
	const int k = pos / R, e = pos % R;
	const int row = e ^ kswz<R>(k);
	return (unsigned)min(k, depth - 1) * (unsigned)ld + (unsigned)min(row, rows - V);
}

}  // namespace ring

// What a kernel does beyond the product and its element-wise epilogue.
enum RingExtra : int { kRingPlain = 0, kRingRowSums = 1, kRingGelu = 2 };

template <int BM, int BN, int BK, int WM, int WN, int ST, bool TA, bool TB, int V, int EXTRA>
__device__ __forceinline__ void ring_tile(const GemmArgs& p, int block) {
	using S = RingShape<BM, BN, BK, WM, WN, ST, TA, TB, V>;
	constexpr int I = S::I, J = S::J, NG = BK / 16;
	constexpr bool RS = EXTRA == kRingRowSums;
	static_assert(!RS || (TA && !TB && BM <= S::kThreads), "row sums: the weight-gradient layout, one thread a row");
	extern __shared__ __align__(16) float lds[];
	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int wm0 = (wave / S::kWavesN) * WM, wn0 = (wave % S::kWavesN) * WN;
	const int lr = lane & 15, g = lane >> 4;

	// ---- which tile and batch matrix (the order of gemm_tile.hpp) ----
	const int tiles = p.tiles_m * p.tiles_n;
	const int lid = xcd_remap(block, tiles * p.batch_count);
	const int t0 = lid % tiles, bi = lid / tiles;
	constexpr int G = 8;
	const int group = t0 / (G * p.tiles_n);
	const int gsize = min(G, p.tiles_m - group * G);
	const int in_group = t0 % (G * p.tiles_n);
	const int tm = group * G + in_group % gsize, tn = in_group / gsize;
	const int m0 = tm * BM, n0 = tn * BN;
	int64_t oa = 0, ob = 0, oc = 0;
	if (p.batch.ndim > 0) batch_offsets(p.batch, bi, oa, ob, oc);

	const int nkt = (p.k + BK - 1) / BK;
	const int krem = p.k - (nkt - 1) * BK;  // depth of the last stage
	const int rows_a = p.m - m0, rows_b = p.n - n0;
	const float* a_next = p.a + oa + (TA ? (int64_t)m0 : (int64_t)m0 * p.lda);  // the next stage's first element
	const float* b_next = p.b + ob + (TB ? (int64_t)n0 * p.ldb : (int64_t)n0);
	const int64_t a_step = TA ? (int64_t)BK * p.lda : BK, b_step = TB ? BK : (int64_t)BK * p.ldb;

	unsigned offa[S::LA], offb[S::LB];
#pragma unroll
	for (int q = 0; q < S::LA; ++q)
		offa[q] = ring::src_offset<!TA, S::kFrag, BM, BK, V>(wave * S::LA + q, lane, p.lda, rows_a, BK);
#pragma unroll
	for (int q = 0; q < S::LB; ++q)
		offb[q] = ring::src_offset<TB, S::kFrag, BN, BK, V>(wave * S::LB + q, lane, p.ldb, rows_b, BK);

	auto dma = [&](const float* src, unsigned off, float* dst) {
		if constexpr (V == 4)
			__builtin_amdgcn_global_load_lds((ring::global_void*)(src + off), (ring::lds_void*)dst, 16, 0, 0);
		else
			__builtin_amdgcn_global_load_lds((ring::global_void*)(src + off), (ring::lds_void*)dst, 4, 0, 0);
	};
	// The wave's load instruction q (0 .. L - 1) of the next stage, whole, into ring slot `slot`; advance() follows the
	// last. Stages are issued in order.
	auto issue_one = [&](int q, int slot) {
		float* As = lds + slot * S::kStage + wave * S::LA * S::kPer;
		float* Bs = lds + slot * S::kStage + S::kA + wave * S::LB * S::kPer;
		if (q < S::LA) dma(a_next, offa[q < S::LA ? q : 0], As + q * S::kPer);
		else dma(b_next, offb[q >= S::LA ? q - S::LA : 0], Bs + (q - S::LA) * S::kPer);
	};
	auto advance = [&]() {
		a_next += a_step;
		b_next += b_step;
	};
	// All of stage kt at once; a partial last stage loads nothing past the depth.
	auto issue = [&](int kt, int slot) {
		if (krem != BK && kt == nkt - 1) {
			float* As = lds + slot * S::kStage + wave * S::LA * S::kPer;
			float* Bs = lds + slot * S::kStage + S::kA + wave * S::LB * S::kPer;
#pragma unroll
			for (int q = 0; q < S::LA; ++q)
				dma(a_next, ring::src_offset<!TA, S::kFrag, BM, BK, V>(wave * S::LA + q, lane, p.lda, rows_a, krem),
				    As + q * S::kPer);
#pragma unroll
			for (int q = 0; q < S::LB; ++q)
				dma(b_next, ring::src_offset<TB, S::kFrag, BN, BK, V>(wave * S::LB + q, lane, p.ldb, rows_b, krem),
				    Bs + q * S::kPer);
			return;
		}
#pragma unroll
		for (int q = 0; q < S::L; ++q) issue_one(q, slot);
		advance();
	};
	// Called by every wave once stage kt is in LDS: gives a partial last stage its padding.
	auto ready = [&](int kt, int slot) {
		if (krem == BK || kt != nkt - 1) return;
		float* As = lds + slot * S::kStage;
		float* Bs = As + S::kA;
		for (int e = tid; e < BM * (BK - krem); e += S::kThreads) {
			const int r = e % BM, k = krem + e / BM;
			As[TA ? k * BM + (r ^ ring::kswz<BM>(k)) : ring::kc_index<BK, S::kFrag>(r, k)] = 0.0f;
		}
		for (int e = tid; e < BN * (BK - krem); e += S::kThreads) {
			const int r = e % BN, k = krem + e / BN;
			Bs[TB ? ring::kc_index<BK, S::kFrag>(r, k) : k * BN + (r ^ ring::kswz<BN>(k))] = -0.0f;
		}
		ring::wait_and_meet<63>();
	};

	// ---- fragments: element t of lane (g, lr) is depth kk + 4 t + g of row (column) lr of a 16-wide block ----
	// k-contiguous: chunk c is at koff ^ 4 c (fragment order: the lane's chunk of the 16 depths from kk is c = kk / 4 + g)
	const int koff = lr * BK + 4 * ring::swz<BK>(lr) + (S::kFrag ? 0 : g);
	int moffa[I], moffb[J];
#pragma unroll
	for (int i = 0; i < I; ++i) moffa[i] = g * BM + ((wm0 + 16 * i) ^ ring::kswz<BM>(g)) + lr;
#pragma unroll
	for (int j = 0; j < J; ++j) moffb[j] = g * BN + ((wn0 + 16 * j) ^ ring::kswz<BN>(g)) + lr;
	// element t of the group of 16 depths from kk (fragment order: all four elements of every fourth block instead)
	auto read_frags = [&](int slot, int kk, int t, f32x4* af, f32x4* bf) {
		const float* As = lds + slot * S::kStage;
		const float* Bs = As + S::kA;
#pragma unroll
		for (int i = 0; i < I; ++i) {
			if (TA) af[i][t] = As[(kk + 4 * t) * BM + moffa[i]];
			else if (!S::kFrag) af[i][t] = As[(wm0 + 16 * i) * BK + (koff ^ (kk + 4 * t))];
			else if (i % 4 == t) af[i] = *reinterpret_cast<const f32x4*>(As + (wm0 + 16 * i) * BK + (koff ^ (kk + 4 * g)));
		}
#pragma unroll
		for (int j = 0; j < J; ++j) {
			if (!TB) bf[j][t] = Bs[(kk + 4 * t) * BN + moffb[j]];
			else if (!S::kFrag) bf[j][t] = Bs[(wn0 + 16 * j) * BK + (koff ^ (kk + 4 * t))];
			else if (j % 4 == t) bf[j] = *reinterpret_cast<const f32x4*>(Bs + (wn0 + 16 * j) * BK + (koff ^ (kk + 4 * g)));
		}
	};

	f32x4 acc[I][J];
#pragma unroll
	for (int i = 0; i < I; ++i)
#pragma unroll
		for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
	f32x4 af[2][I], bf[2][J];
	// Row sums of op(A) (GemmArgs::rowsum): the first column tile's thread tid folds row tid in depth order. Depth past
	// k was filled with +0, which leaves a sum from +0 unchanged. With one or four chains a wave, four adds stand at each
	// step's MFMAs, their operands read with the group's fragments, in whole waves (a tile of 32 rows: the upper lanes repeat the
	// lower ones'): ahead of a stage's MFMAs its chain of adds took longer than they (4096 rows of a 512 -> 512 layer's
	// dW and db 61 us, 45 so, and 27 without db; 65536 rows of 64 -> 1088 930, 670, 370). Larger tiles have no registers for
	// that, and 2048 or more cycles of MFMAs a stage beside the adds.
	constexpr bool kSpread = I * J <= 4;
	float rsum = 0.0f, sums[RS && kSpread ? 2 : 1][16];
	const bool summing = RS && p.rowsum != nullptr && tn == 0 && 64 * wave < BM;  // uniform
	const int srow = tid & (BM - 1);
	auto read_sums = [&](int slot, int k, float* v) {  // depths k .. k + 3 of the stage in `slot`
		const float* As = lds + slot * S::kStage;
#pragma unroll
		for (int e = 0; e < 4; ++e) v[e] = As[(k + e) * BM + (srow ^ ring::kswz<BM>(k + e))];
	};

	// The MFMAs of the stage in `slot`, the fragments of its first group being in set 0; each group's reads are issued
	// among the MFMAs of the group before, the last group reading the first of the stage in `after` (with has_next). With
	// `issuing` the loads of the next stage to fetch, into ring slot `fill`, are spread over the whole stage too: issued
	// in one burst they would stall the wave at the memory unit's rate with the matrix core idle.
	auto compute_stage = [&](int slot, int after, auto has_next, auto issuing, int fill, auto with_sums) {
		constexpr int kSteps = BK / 4;
#pragma unroll
		for (int gi = 0; gi < NG; ++gi) {
			const int cur = gi & 1;
#pragma unroll
			for (int t = 0; t < 4; ++t) {
				const int step = 4 * gi + t;
				if constexpr (decltype(with_sums)::value) {
#pragma unroll
					for (int e = 0; e < 4; ++e) rsum = rsum + sums[cur][4 * t + e];
				}
				if constexpr (decltype(issuing)::value) {
#pragma unroll
					for (int q = 0; q < S::L; ++q)
						if (q * kSteps / S::L == step) issue_one(q, fill);
				}
				// one chain a wave: the whole group's reads ahead of its first MFMA, so that the last of them does not
				// meet the barrier half done
				constexpr bool kBurst = I * J == 1;
#pragma unroll
				for (int tt = 0; tt < 4; ++tt) {
					if (kBurst ? t != 0 : tt != t) continue;
					if (gi + 1 < NG) {
						read_frags(slot, 16 * (gi + 1), tt, af[cur ^ 1], bf[cur ^ 1]);
						if (decltype(with_sums)::value) read_sums(slot, 16 * (gi + 1) + 4 * tt, sums[cur ^ 1] + 4 * tt);
					} else if (decltype(has_next)::value) {
						read_frags(after, 0, tt, af[cur ^ 1], bf[cur ^ 1]);
						if (decltype(with_sums)::value) read_sums(after, 4 * tt, sums[cur ^ 1] + 4 * tt);
					}
				}
#pragma unroll
				for (int i = 0; i < I; ++i)
#pragma unroll
					for (int j = 0; j < J; ++j)
						acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[cur][j][t], af[cur][i][t], acc[i][j], 0, 0, 0);
				// a read or a load between every two or so MFMAs
				constexpr int kOther = I + J + 1, kPer = (I * J) / kOther > 0 ? (I * J) / kOther : 1;
#pragma unroll
				for (int x = 0; x < I * J / kPer; ++x) {
					__builtin_amdgcn_sched_group_barrier(0x008, kPer, 0);
					__builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
					__builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
				}
				__builtin_amdgcn_sched_barrier(0);
			}
		}
		if constexpr (decltype(issuing)::value) advance();
	};
	auto compute = [&](int slot, int after, auto has_next, auto issuing, int fill) {
		if constexpr (RS && kSpread) {
			if (summing) return compute_stage(slot, after, has_next, issuing, fill, std::true_type{});
		} else if (RS && summing) {
			const float* As = lds + slot * S::kStage;
#pragma unroll 8
			for (int k = 0; k < BK; ++k) rsum = rsum + As[k * BM + (tid ^ ring::kswz<BM>(k))];
		}
		compute_stage(slot, after, has_next, issuing, fill, std::false_type{});
	};
	auto next = [](int slot) { return slot + 1 == ST ? 0 : slot + 1; };

	// ---- the depth loop ----
	const bool acc_mode = p.accumulate != 0;
	const int c_row0 = m0 + wm0 + lr, c_col0 = n0 + wn0 + 4 * g;  // this lane's first row and its four columns
	float* __restrict__ Cp = p.c + oc;
	auto add_old = [&]() {  // old C joins the chain after the first 256 steps
#pragma unroll
		for (int i = 0; i < I; ++i)
#pragma unroll
			for (int j = 0; j < J; ++j)
#pragma unroll
				for (int e = 0; e < 4; ++e) {
					const int row = c_row0 + 16 * i, col = c_col0 + 16 * j + e;
					if (row < p.m && col < p.n) acc[i][j][e] = Cp[(int64_t)row * p.ldc + col] + acc[i][j][e];
				}
	};
	// always so; without the test the compiler's code is 2% slower (1000 x 1000 x 100 8.56 us against 8.34)
	if (nkt > 0) {
		int fill = 0, slot = 0;  // the slots the next issued and the next computed stage take
		const int first = min(ST - 1, nkt);
		for (; fill < first; ++fill) issue(fill, fill);
		if (first == ST - 1) ring::wait_and_meet<S::waits(ST - 2)>();
		else ring::wait_and_meet<0>();
		ready(0, 0);
#pragma unroll
		for (int t = 0; t < 4; ++t) read_frags(0, 0, t, af[0], bf[0]);
		if (RS && kSpread && summing) {
#pragma unroll
			for (int t = 0; t < 4; ++t) read_sums(0, 4 * t, sums[0] + 4 * t);
		}
		int kt = 0;
		// whole iterations up to stage `end`, each issuing the (whole) stage ST - 1 ahead
		auto run = [&](int end) {
			for (; kt < end; ++kt) {
				const int after = next(slot);
				ring::wait_and_meet<S::waits(ST - 3)>();
				compute(slot, after, std::true_type{}, std::true_type{}, fill);
				fill = next(fill);
				slot = after;
			}
		};
		const int whole = krem == BK ? nkt : nkt - 1;           // whole stages
		const int last_issue = max(0, nkt - (ST - 1));          // from this stage on nothing is left to issue
		const int last_whole = max(0, whole - (ST - 1));        // up to this one the stage to issue is whole
		const int mid = (acc_mode && p.k > kAccAfter) ? kAccAfter / BK : -1;
		bool added = mid < 0;
		auto add_at_mid = [&]() {
			if (added || kt != mid) return;
			add_old();
			added = true;
		};
		if (!added && mid <= last_whole) run(mid);
		add_at_mid();
		run(last_whole);
		if (kt < last_issue) {  // the partial stage's loads
			const int after = next(slot);
			ring::wait_and_meet<S::waits(ST - 3)>();
			issue(kt + ST - 1, fill);
			compute(slot, after, std::true_type{}, std::false_type{}, 0);
			slot = after;
			++kt;
			add_at_mid();
		}
		auto tail = [&](auto beyond) {  // nothing left to issue, `beyond` stages in flight past the next one
			constexpr int r = decltype(beyond)::value;
			if (kt + 2 + r != nkt) return;
			const int after = next(slot);
			ring::wait_and_meet<S::waits(r)>();
			ready(kt + 1, after);
			compute(slot, after, std::true_type{}, std::false_type{}, 0);
			slot = after;
			++kt;
			add_at_mid();
		};
		if constexpr (ST >= 5) tail(std::integral_constant<int, 2>{});
		if constexpr (ST >= 4) tail(std::integral_constant<int, 1>{});
		tail(std::integral_constant<int, 0>{});
		compute(slot, slot, std::false_type{}, std::false_type{}, 0);
	}
	if (RS && summing && tid < BM && m0 + tid < p.m) {
		float* d = p.rowsum + m0 + tid;
		*d = p.rowsum_combine == 0 ? rsum : (p.rowsum_combine == 1 ? rsum + 0.0f : *d + rsum);
	}

	// ---- the store: accumulate, bias, residual, GELU, ReLU per element, in the reference's order ----
	const bool old_at_end = acc_mode && p.k <= kAccAfter;
	const bool c_vec = p.c_vec != 0;
	unsigned char* alive = p.ep.alive ? p.ep.alive + oc : nullptr;
	const float* res = p.ep.res ? p.ep.res + oc : nullptr;
	float* gy = p.ep.gelu_y ? p.ep.gelu_y + oc : nullptr;
	float* gt = p.ep.gelu_t ? p.ep.gelu_t + oc : nullptr;
	int row0 = c_row0, col0 = c_col0;
	asm volatile("" : "+v"(row0), "+v"(col0));  // keeps the store addresses from being computed before the loop
#pragma unroll
	for (int i = 0; i < I; ++i) {
		const int row = row0 + 16 * i;
#pragma unroll
		for (int j = 0; j < J; ++j) {
			const int col = col0 + 16 * j;
			const int nc = row < p.m ? min(4, p.n - col) : 0;  // valid columns of the lane's four
			if (nc <= 0) continue;
			const int64_t off = (int64_t)row * p.ldc + col;
			f32x4 v = acc[i][j];
			if (c_vec && nc == 4) {
				if (old_at_end) {
					const f32x4 old = *reinterpret_cast<const f32x4*>(Cp + off);
#pragma unroll
					for (int e = 0; e < 4; ++e) v[e] = old[e] + v[e];
				}
				if (p.ep.bias_mode == kBiasCol) {
#pragma unroll
					for (int e = 0; e < 4; ++e) v[e] = v[e] + p.ep.bias[col + e];
				} else if (p.ep.bias_mode == kBiasRow) {
					const float b = p.ep.bias[row];
#pragma unroll
					for (int e = 0; e < 4; ++e) v[e] = v[e] + b;
				}
				if (res) {
#pragma unroll
					for (int e = 0; e < 4; ++e) v[e] = res[off + e] + v[e];
				}
				if constexpr (EXTRA == kRingGelu) {
					f32x4 y, t;
#pragma unroll
					for (int e = 0; e < 4; ++e) {
						float te;
						y[e] = gelu_math::gelu_one(v[e], te);
						t[e] = te;
					}
					*reinterpret_cast<f32x4*>(gy + off) = y;
					*reinterpret_cast<f32x4*>(gt + off) = t;
				}
				if (p.ep.relu) {
#pragma unroll
					for (int e = 0; e < 4; ++e) {
						const bool on = v[e] > 0.0f;
						if (alive) alive[off + e] = on ? 1 : 0;
						v[e] = on ? v[e] : 0.0f;
					}
				}
				*reinterpret_cast<f32x4*>(Cp + off) = v;
				continue;
			}
#pragma unroll
			for (int e = 0; e < 4; ++e) {
				if (e >= nc) continue;
				float x = v[e];
				if (old_at_end) x = Cp[off + e] + x;
				if (p.ep.bias_mode == kBiasCol) x = x + p.ep.bias[col + e];
				else if (p.ep.bias_mode == kBiasRow) x = x + p.ep.bias[row];
				if (res) x = res[off + e] + x;
				if constexpr (EXTRA == kRingGelu) {
					float t;
					gy[off + e] = gelu_math::gelu_one(x, t);
					gt[off + e] = t;
				}
				if (p.ep.relu) {
					const bool on = x > 0.0f;
					if (alive) alive[off + e] = on ? 1 : 0;
					x = on ? x : 0.0f;
				}
				Cp[off + e] = x;
			}
		}
	}
}

template <int BM, int BN, int BK, int WM, int WN, int ST, int WPE, bool TA, bool TB, int V, int EXTRA>
__global__ void __launch_bounds__((RingShape<BM, BN, BK, WM, WN, ST, TA, TB, V>::kThreads))
__attribute__((amdgpu_waves_per_eu(WPE, WPE))) sgemm_ring_kernel(const GemmArgs p) {
	ring_tile<BM, BN, BK, WM, WN, ST, TA, TB, V, EXTRA>(p, (int)blockIdx.x);
}

// Two products in one grid on the same tile: A B or A B^T (workgroups 0 .. blocks0 - 1) and an A^T B, with or without
// row sums.
template <int BM, int BN, int BK, int WM, int WN, int ST, int WPE, bool TB0, int V0, int V1, int EXTRA1>
__global__ void __launch_bounds__((RingShape<BM, BN, BK, WM, WN, ST, false, TB0, V0>::kThreads))
__attribute__((amdgpu_waves_per_eu(WPE, WPE))) sgemm_ring_pair_kernel(const GemmArgs p0, const GemmArgs p1, int blocks0) {
	const int block = (int)blockIdx.x;
	if (block < blocks0) ring_tile<BM, BN, BK, WM, WN, ST, false, TB0, V0, kRingPlain>(p0, block);
	else ring_tile<BM, BN, BK, WM, WN, ST, true, false, V1, EXTRA1>(p1, block - blocks0);
}

// One compiled tile shape of the ring kernel: its kernels by layout (ta * 2 + tb) and by the load width.
struct RingConfig {
	const char* name;
	int bm, bn, threads, lds_bytes;
	void (*fn[4][2])(const GemmArgs);  // [layout][0: one float a lane, 1: four]
	void (*rowsum_fn[2])(const GemmArgs);  // A transposed, B not, with row sums of op(A)
	void (*gelu_fn[2])(const GemmArgs);    // A not transposed, B transposed, with the GELU epilogue
};

template <int BM, int BN, int BK, int WM, int WN, int ST, int WPE>
RingConfig make_ring_config(const char* name) {
	using S = RingShape<BM, BN, BK, WM, WN, ST, false, false, 4>;  // threads and LDS are the same for every layout
	RingConfig c{};
	c.name = name;
	c.bm = BM;
	c.bn = BN;
	c.threads = S::kThreads;
	c.lds_bytes = S::kLdsBytes;
#define NNH_RING(TA, TB, V, EXTRA) sgemm_ring_kernel<BM, BN, BK, WM, WN, ST, WPE, TA, TB, V, EXTRA>
	c.fn[0][0] = NNH_RING(false, false, 1, kRingPlain);
	c.fn[0][1] = NNH_RING(false, false, 4, kRingPlain);
	c.fn[1][0] = NNH_RING(false, true, 1, kRingPlain);
	c.fn[1][1] = NNH_RING(false, true, 4, kRingPlain);
	c.fn[2][0] = NNH_RING(true, false, 1, kRingPlain);
	c.fn[2][1] = NNH_RING(true, false, 4, kRingPlain);
	c.fn[3][0] = NNH_RING(true, true, 1, kRingPlain);
	c.fn[3][1] = NNH_RING(true, true, 4, kRingPlain);
	c.rowsum_fn[0] = NNH_RING(true, false, 1, kRingRowSums);
	c.rowsum_fn[1] = NNH_RING(true, false, 4, kRingRowSums);
	c.gelu_fn[0] = NNH_RING(false, true, 1, kRingGelu);
	c.gelu_fn[1] = NNH_RING(false, true, 4, kRingGelu);
#undef NNH_RING
	return c;
}

using RingPairFn = void (*)(const GemmArgs, const GemmArgs, int);
RingPairFn ring_pair_32x32(int kind, int v0, int v1);  // kind 0: A B, 1: A B with row sums of the other, 2: A B^T

RingConfig ring_config_256x128();
RingConfig ring_config_128x128();
RingConfig ring_config_64x64();
RingConfig ring_config_32x32();

}  // namespace nnh
