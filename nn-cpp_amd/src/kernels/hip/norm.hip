// norm.hip - nn::batchnorm (training mode, optionally with its folded ReLU) and nn::layernorm, forward and backward
// (src/autograd/ops.cpp:900-1078), with the reference's summation orders.
//
// Batch norm. The reference gives each channel to one thread: for n = 0..N-1 in order it adds, in double, the
// lane_sum of row (n, c) (eight float partial sums over the row, combined as ((a0+a1)+(a2+a3))+((a4+a5)+(a6+a7)),
// then the tail), divides by N*S, and does the same with lane_sq around the mean. Here:
//   * bn_rows_kernel computes the per-row float sums (lane_sum, lane_sq, or the backward's masked lane_sum and
//     lane_dot): a workgroup owns 4, 8 or 32 rows of one channel; all its threads form the terms from wide coalesced
//     loads and put them in LDS, and the reference's eight lane chains per row run over LDS (thread 8r + k is
//     partial a[k] of row r), combine and add the tail in order.
//   * The channel-level double sums over n run in order in one thread of every workgroup that needs them (the
//     rows' sums are staged in LDS first), so the channel's statistics come with each workgroup's own prologue
//     instead of a launch of their own.
//   * bn_norm_kernel (forward) and bn_dx_kernel (backward) are elementwise over a channel's N*S elements in 4096-
//     element chunks, 16-byte loads and stores where the rows allow.
// Layer norm. Each row's sums are single float chains (ops.cpp:1017-1026): a workgroup holds some rows in registers, all
// its threads form the chains' terms and put them in LDS, and one thread a chain adds them there. The gamma/beta
// gradient sums run down columns in row order (ops.cpp:1063-1075): chains over LDS again, beside dx in the same launch.
// Longer rows than a workgroup's registers hold take one thread a row and one a column.
#include "norm.hpp"

#include <algorithm>
#include <mutex>

#include "fastdiv.hpp"

namespace nnh {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Workgroups of 256 threads in one launch: HIP takes fewer than 2^32 work-items a dimension.
constexpr int64_t kMaxGrid = ((int64_t)1 << 24) - 1;

// acc + v[0] + v[1] + ... + v[n - 1] in order; v is 16-byte aligned LDS.
__device__ __forceinline__ float lds_chain(const float* v, int n, float acc = 0.0f) {
	const f32x4* q = reinterpret_cast<const f32x4*>(v);
	const int nb = n / 16;
	if (nb > 0) {
		f32x4 t[3][4];
#pragma unroll
		for (int e = 0; e < 4; ++e) t[0][e] = q[e];
#pragma unroll
		for (int e = 0; e < 4; ++e) t[1][e] = q[4 * min(1, nb - 1) + e];
		for (int b = 0; b < nb; b += 3) {
#pragma unroll
			for (int k = 0; k < 3; ++k) {
				// past the end a redundant read of the last block: no branch around a read
#pragma unroll
				for (int e = 0; e < 4; ++e) t[(k + 2) % 3][e] = q[4 * min(b + k + 2, nb - 1) + e];
				__builtin_amdgcn_sched_barrier(0);  // keeps the reads ahead of the adds they run beside
				if (b + k < nb) {
#pragma unroll
					for (int e = 0; e < 4; ++e)
#pragma unroll
						for (int i = 0; i < 4; ++i) acc = acc + t[k][e][i];
				}
			}
		}
	}
	for (int j = 16 * nb; j < n; ++j) acc = acc + v[j];
	return acc;
}

// bn_rows_kernel: rows a workgroup owns, elements of each staged per step, and the LDS layout: partial k's elements
// k, k + 8, k + 16, ... of a row lie back to back (kPart apart), so that its lane adds them from 16-byte reads. kPart is 8
// mod 16: both the staging's four-byte stores (two partials, 32 positions) and the chains' reads (eight partials) then use
// different banks.
template <int ROWS, int CHUNK>
struct BnRowShape {
	static constexpr int kRows = ROWS, kChunk = CHUNK;
	static constexpr int kPart = (CHUNK / 8 + 7) / 16 * 16 + 8, kRowLds = 8 * kPart;
	static constexpr int kRowTail = 8;  // a row's last S mod 8 terms, after the partials
	static constexpr int kRowSet = ROWS * (kRowLds + kRowTail);
	static_assert(CHUNK % 8 == 0 && kPart >= CHUNK / 8 && 8 * ROWS <= 256, "eight partials a row, a thread each");
};
using BnLong = BnRowShape<4, 2304>;
using BnMedium = BnRowShape<8, 1024>;
using BnShort = BnRowShape<32, 128>;

enum BnRowMode { kSum = 0, kSq = 1, kBwd = 2 };

struct BnRowArgs {
	const float* x;
	const float* g;               // kBwd: the upstream gradient
	const unsigned char* alive;   // kBwd: the folded ReLU's flags, or null
	const float* rowsum;          // kSq: the rows' lane sums, source of the channel mean
	const float* mean;            // kBwd: the forward's channel means
	float* out0;                  // per row (n * C + c): kSum lane_sum, kSq lane_sq, kBwd lane_sum of masked g
	float* out1;                  // kBwd: lane_dot of masked g with x - mean
	float* mean_out;              // kSq: the channel mean, written by the channel's first workgroup
	int64_t N, C, S;
	int64_t groups;               // workgroups per channel: ceil(N / rows)
	int64_t first_block;          // of this launch
	double dm;
	FastDiv whole, last;          // units of a row in a whole chunk and in the last one
};

// Sums in double of v0[n * C + c] (and v1's) for n = 0..N-1 in order, as the reference adds a channel's row sums
// (ops.cpp:927-929, 973-978): the values are staged 256 at a time in LDS and one thread adds them. Every thread
// of the block receives the sums.
template <int NSUM>
__device__ void channel_dsums(const float* v0, const float* v1, int64_t N, int64_t C, int64_t c, float (*buf)[256],
                              double* out, double* res) {
	const int tid = threadIdx.x;
	double s0 = 0.0, s1 = 0.0;
	for (int64_t n0 = 0; n0 < N; n0 += 256) {
		const int64_t n = n0 + tid;
		if (n < N) {
			buf[0][tid] = v0[n * C + c];
			if (NSUM == 2) buf[1][tid] = v1[n * C + c];
		}
		__syncthreads();
		if (tid == 0) {
			const int cnt = (int)(N - n0 < 256 ? N - n0 : 256);
			int i = 0;
			for (; i + 16 <= cnt; i += 16) {  // sixteen LDS reads ahead of the dependent adds
				float t0[16], t1[16];
#pragma unroll
				for (int u = 0; u < 16; ++u) {
					t0[u] = buf[0][i + u];
					if (NSUM == 2) t1[u] = buf[1][i + u];
				}
#pragma unroll
				for (int u = 0; u < 16; ++u) {
					s0 += (double)t0[u];
					if (NSUM == 2) s1 += (double)t1[u];
				}
			}
			for (; i < cnt; ++i) {
				s0 += (double)buf[0][i];
				if (NSUM == 2) s1 += (double)buf[1][i];
			}
		}
		__syncthreads();
	}
	if (tid == 0) {
		out[0] = s0;
		out[1] = s1;
	}
	__syncthreads();
	res[0] = out[0];
	res[1] = out[1];
}

// lane_sum (ops.cpp:804-812), lane_sq (824-834), and the backward's lane_sum / lane_sum_masked with lane_dot /
// lane_dot_masked (848-897) of SH::kRows rows of channel c per workgroup. All threads load the rows (16-byte
// loads with VEC: S % 4 == 0, aligned rows), form the terms the chains add (x, (x - mean)^2, or the masked g and g (x -
// mean)) and put them in LDS; thread 8 r + k (the backward's second sum: those after the first sum's, or the same one where
// they fill the workgroup) adds partial k of row r, about 7 cycles a term, then the eight partials combine and the row's
// tail follows in order. Rows longer than kChunk go chunk by chunk, the next chunk's loads in flight during the chains.
// Measured at [64, 16, 48, 48] (9.4 MB): sums 9.4 -> 6.3 us, squares 10.4 -> 7.4, backward 27.3 -> 7.6, against eight rows
// a workgroup (128 of them), element-wise work in the chain lanes and three exposed chunk loads.
template <int MODE, bool VEC, class SH>
__global__ void __launch_bounds__(256) bn_rows_kernel(const BnRowArgs a) {
	constexpr int kRows = SH::kRows, kChunk = SH::kChunk, kPart = SH::kPart, kRowLds = SH::kRowLds;
	constexpr int kRowTail = SH::kRowTail, kRowSet = SH::kRowSet;
	extern __shared__ __align__(16) float lds[];  // a set of terms, and with kBwd a second one
	__shared__ float buf[2][256];
	__shared__ double bcast[2];
	constexpr int kW = VEC ? 4 : 1;                        // floats of a unit
	constexpr int kPer = kRows * kChunk / kW / 256;        // units a thread holds
	constexpr int kBatch = VEC ? kPer : kPer % 18 == 0 ? 18 : 16;  // of them in flight at once
	static_assert(kPer * 256 * kW == kRows * kChunk && kPer % kBatch == 0, "a chunk splits evenly over the threads");
	constexpr int kSets = MODE == kBwd ? 2 : 1, kSetThreads = 8 * kRows;
	constexpr int kMine = kSets * kSetThreads <= 256 ? 1 : kSets;  // chains of a thread
	const int tid = threadIdx.x;
	const int64_t blk = a.first_block + blockIdx.x;
	const int64_t c = blk / a.groups, j = blk - c * a.groups;
	const int64_t n0 = j * kRows;
	const int nrows = (int)(a.N - n0 < kRows ? (a.N > n0 ? a.N - n0 : 0) : kRows);
	const int64_t row0 = n0 * a.C + c;  // row index of (n0, c); rows of one channel are C apart
	const int64_t full = a.S & ~(int64_t)7;
	const bool masked = MODE == kBwd && a.alive != nullptr;

	float xv[kBatch][kW], gv[kBatch][kW];
	unsigned fv[kBatch];
	// units u0 .. u0 + kBatch - 1 (times 256 threads) of the chunk from s0: loads at clamped indices, then the terms
	auto load = [&](int64_t s0, int u0, int tot, const FastDiv& dv) {
#pragma unroll
		for (int u = 0; u < kBatch; ++u) {
			const int i = min(tid + 256 * (u0 + u), tot - 1);
			const int r = (int)fdiv((unsigned)i, dv), q = i - r * (int)dv.d;
			const int64_t at = (row0 + r * a.C) * a.S + s0 + kW * q;
			if constexpr (VEC) {
				const f32x4 x4 = *reinterpret_cast<const f32x4*>(a.x + at);
#pragma unroll
				for (int e = 0; e < 4; ++e) xv[u][e] = x4[e];
				if (MODE == kBwd) {
					const f32x4 g4 = *reinterpret_cast<const f32x4*>(a.g + at);
#pragma unroll
					for (int e = 0; e < 4; ++e) gv[u][e] = g4[e];
					if (masked) fv[u] = *reinterpret_cast<const unsigned*>(a.alive + at);
				}
			} else {
				xv[u][0] = a.x[at];
				if (MODE == kBwd) {
					gv[u][0] = a.g[at];
					if (masked) fv[u] = a.alive[at];
				}
			}
		}
	};
	float mu = 0.0f;
	auto put = [&](int64_t s0, int u0, int tot, const FastDiv& dv) {
#pragma unroll
		for (int u = 0; u < kBatch; ++u) {
			const int i = tid + 256 * (u0 + u);
			if (i >= tot) continue;
			const int r = (int)fdiv((unsigned)i, dv), l = kW * (i - r * (int)dv.d);
#pragma unroll
			for (int e = 0; e < kW; ++e) {
				float t0, t1 = 0.0f;
				if (MODE == kSum) {
					t0 = xv[u][e];
				} else if (MODE == kSq) {
					const float d = xv[u][e] - mu;
					t0 = d * d;
				} else {
					t0 = masked && !((fv[u] >> (8 * e)) & 0xffu) ? 0.0f : gv[u][e];
					t1 = t0 * (xv[u][e] - mu);
				}
				const int at = s0 + l + e < full ? r * kRowLds + ((l + e) & 7) * kPart + ((l + e) >> 3)
				                                 : kRows * kRowLds + r * kRowTail + (int)(s0 + l + e - full);
				lds[at] = t0;
				if (MODE == kBwd) lds[kRowSet + at] = t1;
			}
		}
	};
	auto chunk_len = [&](int64_t s0) { return (int)(a.S - s0 < kChunk ? a.S - s0 : kChunk); };
	auto units = [&](int64_t s0) { return nrows * (chunk_len(s0) / kW); };
	auto div_of = [&](int64_t s0) -> const FastDiv& { return s0 + kChunk < a.S ? a.whole : a.last; };
	// With VEC a whole chunk is one batch, loaded before the channel's mean is known
	const bool any = nrows > 0 && a.S > 0;
	if (VEC && any) load(0, 0, units(0), div_of(0));
	if (MODE == kSq) {
		double s[2];
		channel_dsums<1>(a.rowsum, nullptr, a.N, a.C, c, buf, bcast, s);
		mu = (float)(s[0] / a.dm);
		if (j == 0 && tid == 0) a.mean_out[c] = mu;
	} else if (MODE == kBwd) {
		mu = a.mean[c];
	}
	if (nrows <= 0) return;
	const int which = kMine == 1 ? tid / kSetThreads : 0, r = (tid % kSetThreads) >> 3, k = tid & 7;
	const bool adds = which < kSets && r < nrows;
	const float* set = lds + which * kRowSet;
	float acc[kMine] = {};
	for (int64_t s0 = 0; s0 < a.S; s0 += kChunk) {
		const int tot = units(s0);
		if constexpr (VEC) {
			put(s0, 0, tot, div_of(s0));
		} else {
			for (int u0 = 0; u0 < kPer; u0 += kBatch) {
				load(s0, u0, tot, div_of(s0));
				put(s0, u0, tot, div_of(s0));
			}
		}
		__syncthreads();
		if (VEC && s0 + kChunk < a.S) load(s0 + kChunk, 0, units(s0 + kChunk), div_of(s0 + kChunk));
		if (adds) {
			const int64_t left = full - s0;
			const int n = (int)(left < kChunk ? (left > 0 ? left : 0) : kChunk) / 8;
#pragma unroll
			for (int i = 0; i < kMine; ++i) acc[i] = lds_chain(set + i * kRowSet + r * kRowLds + k * kPart, n, acc[i]);
		}
		__syncthreads();
	}
	// the partials combine as ((a0 + a1) + (a2 + a3)) + ((a4 + a5) + (a6 + a7)), then the tail in order
#pragma unroll
	for (int i = 0; i < kMine; ++i) {
		float p[8];
#pragma unroll
		for (int u = 0; u < 8; ++u) p[u] = __shfl(acc[i], (tid & 56) + u);
		if (!adds || k != 0) continue;
		float t = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
		const float* tail = set + i * kRowSet + kRows * kRowLds + r * kRowTail;
		for (int l = 0; l < (int)(a.S - full); ++l) t = t + tail[l];
		(which + i == 0 ? a.out0 : a.out1)[row0 + r * a.C] = t;
	}
}

constexpr int kElemChunk = 4096;  // channel elements per workgroup in the elementwise kernels (16 per thread)

struct BnElemArgs {
	const float* x;
	const float* g;               // backward: upstream gradient
	const unsigned char* alive_in;  // backward: the folded ReLU's flags, or null
	const float* w;
	const float* b;
	const float* rowv0;           // forward: rows' lane_sq; backward: rows' lane sums of masked g
	const float* rowv1;           // backward: rows' lane_dot
	const float* mean;
	const float* inv_in;          // backward: inv_std from the forward
	float* y;                     // forward output / backward dx
	unsigned char* alive;         // forward: flags out (relu), may be null
	float* var_out;
	float* inv_out;
	float* dw;
	float* db;
	int64_t N, C, S;
	int64_t chunks;               // workgroups per channel
	double dm;
	float fm, eps;
	int relu, vec, first, dw_first, db_first;
	FastDiv sdiv;                 // S, when N * S < 2^31
};

// Channel element e (0 <= e < N*S) -> its offset (n * C + c) * S + s.
template <bool FAST>
__device__ __forceinline__ int64_t channel_offset(int64_t e, const BnElemArgs& a, int64_t c) {
	int64_t n;
	if (FAST) n = (int64_t)fdiv((unsigned)e, a.sdiv);
	else n = e / a.S;
	return (n * a.C + c) * a.S + (e - n * a.S);
}

// y = (x - mean) * (weight * inv_std) + bias (ops.cpp:931-957), alive and clipping with relu. The prologue turns the
// rows' lane_sq into the channel's variance and inv_std; the channel's first workgroup stores them.
template <bool FAST>
__global__ void __launch_bounds__(256) bn_norm_kernel(const BnElemArgs a) {
	__shared__ float buf[2][256];
	__shared__ double bcast[2];
	const int tid = threadIdx.x;
	const int64_t c = blockIdx.x / a.chunks;
	const int64_t j = blockIdx.x - c * a.chunks;
	const int64_t total = a.N * a.S;
	const int64_t e0 = j * kElemChunk;
	// the chunk's elements are loaded ahead of the channel's sums (clamped: past the end the last group again)
	f32x4 xs[kElemChunk / 1024];
	int64_t offs[kElemChunk / 1024];
	if (a.vec && total > 0) {
#pragma unroll
		for (int u = 0; u < kElemChunk / 1024; ++u) {
			const int64_t e = e0 + 4 * (tid + 256 * u);
			offs[u] = channel_offset<FAST>(e < total ? e : total - 4, a, c);
			xs[u] = *reinterpret_cast<const f32x4*>(a.x + offs[u]);
		}
	}
	double s[2];
	channel_dsums<1>(a.rowv0, nullptr, a.N, a.C, c, buf, bcast, s);
	const float mu = a.mean[c];
	const float v = (float)(s[0] / a.dm);
	const float inv = 1.0f / sqrtf(v + a.eps);
	if (j == 0 && tid == 0) {
		if (a.var_out) a.var_out[c] = v;
		a.inv_out[c] = inv;
	}
	const float scale = a.w[c] * inv, bc = a.b[c];
	if (a.vec) {
#pragma unroll
		for (int u = 0; u < kElemChunk / 1024; ++u) {
			if (e0 + 4 * (tid + 256 * u) >= total) continue;
			const int64_t off = offs[u];
			const f32x4 xv = xs[u];
			f32x4 o;
			unsigned fl = 0;
#pragma unroll
			for (int i = 0; i < 4; ++i) {
				const float t = (xv[i] - mu) * scale + bc;
				if (a.relu) {
					fl |= (t > 0.0f ? 1u : 0u) << (8 * i);
					o[i] = t > 0.0f ? t : 0.0f;
				} else {
					o[i] = t;
				}
			}
			*reinterpret_cast<f32x4*>(a.y + off) = o;
			if (a.relu && a.alive) *reinterpret_cast<unsigned*>(a.alive + off) = fl;
		}
	} else {
		for (int u = 0; u < kElemChunk / 256; ++u) {
			const int64_t e = e0 + tid + 256 * u;
			if (e >= total) break;
			const int64_t off = channel_offset<FAST>(e, a, c);
			const float t = (a.x[off] - mu) * scale + bc;
			if (a.relu) {
				if (a.alive) a.alive[off] = t > 0.0f;
				a.y[off] = t > 0.0f ? t : 0.0f;
			} else {
				a.y[off] = t;
			}
		}
	}
}

// The backward rule's per-channel part (ops.cpp:970-999): the prologue adds the rows' sums in double, the
// channel's first workgroup adds sdy into db and sdg * inv_std into dw, and every workgroup writes its chunk of
// dx = k * (M * g' - a - ((x - mean) * inv_std) * b) with k = weight * inv_std / M, g' masked by alive.
// AHEAD: the chunk's elements are loaded ahead of the channel's sums, which takes 88 registers (5 waves a SIMD) against 44
// (8): a few percent faster while the sums are short, but with thousands of samples the sums are the time and all of a
// channel's workgroups have to be resident at once ([4096, 8, 16 x 16] 164 us with it, 118 without; [512, 16, 14 x 14] 24.5
// and 25.2; [1024, 8, 28 x 28] 55 and 46).
template <bool FAST, bool AHEAD>
__global__ void __launch_bounds__(256) bn_dx_kernel(const BnElemArgs a) {
	__shared__ float buf[2][256];
	__shared__ double bcast[2];
	const int tid = threadIdx.x;
	const int64_t c = blockIdx.x / a.chunks;
	const int64_t j = blockIdx.x - c * a.chunks;
	const int64_t total = a.N * a.S;
	const int64_t e0 = j * kElemChunk;
	const bool masked = a.alive_in != nullptr;
	f32x4 gs[kElemChunk / 1024], xs[kElemChunk / 1024];
	unsigned fls[kElemChunk / 1024];
	int64_t offs[kElemChunk / 1024];
	auto load = [&](int u) {  // past the end the last group again
		const int64_t e = e0 + 4 * (tid + 256 * u);
		offs[u] = channel_offset<FAST>(e < total ? e : total - 4, a, c);
		gs[u] = *reinterpret_cast<const f32x4*>(a.g + offs[u]);
		xs[u] = *reinterpret_cast<const f32x4*>(a.x + offs[u]);
		fls[u] = masked ? *reinterpret_cast<const unsigned*>(a.alive_in + offs[u]) : 0x01010101u;
	};
	if (AHEAD && a.y && a.vec && total > 0) {
#pragma unroll
		for (int u = 0; u < kElemChunk / 1024; ++u) load(u);
	}
	double s[2];
	channel_dsums<2>(a.rowv0, a.rowv1, a.N, a.C, c, buf, bcast, s);
	const float mu = a.mean[c], inv = a.inv_in[c];
	const double sdy = s[0], sdyx = s[1] * (double)inv;
	if (j == 0 && tid == 0) {
		if (a.db) a.db[c] = a.db_first ? 0.0f + (float)sdy : a.db[c] + (float)sdy;
		if (a.dw) a.dw[c] = a.dw_first ? 0.0f + (float)sdyx : a.dw[c] + (float)sdyx;
	}
	if (!a.y) return;
	const float kk = a.w[c] * inv / a.fm, fm = a.fm, av = (float)sdy, bb = (float)sdyx;
	if (a.vec) {
#pragma unroll
		for (int u = 0; u < kElemChunk / 1024; ++u) {
			if (e0 + 4 * (tid + 256 * u) >= total) continue;
			if (!AHEAD) load(u);
			const int64_t off = offs[u];
			const f32x4 gv = gs[u], xv = xs[u];
			const unsigned fl = fls[u];
			f32x4 old = a.first ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : *reinterpret_cast<const f32x4*>(a.y + off);
			f32x4 o;
#pragma unroll
			for (int i = 0; i < 4; ++i) {
				const float gm = masked ? (((fl >> (8 * i)) & 0xffu) ? gv[i] : 0.0f) : gv[i];
				const float term = kk * (fm * gm - av - ((xv[i] - mu) * inv) * bb);
				o[i] = a.first ? term + 0.0f : old[i] + term;
			}
			*reinterpret_cast<f32x4*>(a.y + off) = o;
		}
	} else {
		for (int u = 0; u < kElemChunk / 256; ++u) {
			const int64_t e = e0 + tid + 256 * u;
			if (e >= total) break;
			const int64_t off = channel_offset<FAST>(e, a, c);
			const float gm = masked ? (a.alive_in[off] ? a.g[off] : 0.0f) : a.g[off];
			const float term = kk * (fm * gm - av - ((a.x[off] - mu) * inv) * bb);
			a.y[off] = a.first ? term + 0.0f : a.y[off] + term;
		}
	}
}

// layernorm forward, one thread per row (ops.cpp:1017-1030): the row's sum and its sum of squared deviations are
// single float chains in column order.
__global__ void __launch_bounds__(256) ln_forward_kernel(const float* __restrict__ x, const float* __restrict__ gm,
                                                         const float* __restrict__ bt, int64_t R, int D, float fd,
                                                         float eps, float* __restrict__ y, float* __restrict__ mean,
                                                         float* __restrict__ inv_std, int vec) {
	const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
	if (r >= R) return;
	const float* row = x + r * D;
	float* out = y + r * D;
	float sum = 0.0f;
	if (vec) {
		for (int j = 0; j < D; j += 4) {
			const f32x4 v = *reinterpret_cast<const f32x4*>(row + j);
			sum = sum + v[0];
			sum = sum + v[1];
			sum = sum + v[2];
			sum = sum + v[3];
		}
	} else {
		for (int j = 0; j < D; ++j) sum = sum + row[j];
	}
	const float mu = sum / fd;
	float sq = 0.0f;
	if (vec) {
		for (int j = 0; j < D; j += 4) {
			const f32x4 v = *reinterpret_cast<const f32x4*>(row + j);
#pragma unroll
			for (int i = 0; i < 4; ++i) sq = sq + (v[i] - mu) * (v[i] - mu);
		}
	} else {
		for (int j = 0; j < D; ++j) sq = sq + (row[j] - mu) * (row[j] - mu);
	}
	const float inv = 1.0f / sqrtf(sq / fd + eps);
	mean[r] = mu;
	inv_std[r] = inv;
	if (vec) {
		for (int j = 0; j < D; j += 4) {
			const f32x4 v = *reinterpret_cast<const f32x4*>(row + j);
			const f32x4 g = *reinterpret_cast<const f32x4*>(gm + j);
			const f32x4 b = *reinterpret_cast<const f32x4*>(bt + j);
			f32x4 o;
#pragma unroll
			for (int i = 0; i < 4; ++i) o[i] = (v[i] - mu) * inv * g[i] + b[i];
			*reinterpret_cast<f32x4*>(out + j) = o;
		}
	} else {
		for (int j = 0; j < D; ++j) out[j] = (row[j] - mu) * inv * gm[j] + bt[j];
	}
}

struct LnBwdArgs {
	const float* g;
	const float* x;
	const float* gm;
	const float* mean;
	const float* inv;
	float* dx;
	float* dgamma;
	float* dbeta;
	int64_t R;
	int D;
	float fd;
	int dx_first, dg_first, db_first;
	unsigned row_blocks;  // blocks [0, row_blocks) own rows (dx), the rest own columns (dgamma, dbeta)
};

// layernorm backward: blocks below row_blocks give each thread a row of dx (ops.cpp:1043-1060), the others each
// thread a column of dgamma and dbeta, summed over the rows in order (ops.cpp:1061-1076).
__global__ void __launch_bounds__(256) ln_backward_kernel(const LnBwdArgs a) {
	if (blockIdx.x < a.row_blocks) {
		const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
		if (r >= a.R) return;
		const float* gr = a.g + r * a.D;
		const float* xr = a.x + r * a.D;
		float* dr = a.dx + r * a.D;
		const float mu = a.mean[r], inv = a.inv[r];
		float sa = 0.0f, sb = 0.0f;
		for (int j = 0; j < a.D; ++j) {
			const float dxhat = gr[j] * a.gm[j];
			sa = sa + dxhat;
			sb = sb + dxhat * ((xr[j] - mu) * inv);
		}
		const float k = inv / a.fd, fd = a.fd;
		for (int j = 0; j < a.D; ++j) {
			const float dxhat = gr[j] * a.gm[j];
			const float term = k * (fd * dxhat - sa - ((xr[j] - mu) * inv) * sb);
			dr[j] = a.dx_first ? term + 0.0f : dr[j] + term;
		}
		return;
	}
	const int64_t col = (int64_t)(blockIdx.x - a.row_blocks) * 256 + threadIdx.x;
	if (col >= a.D) return;
	float sg = 0.0f, sb = 0.0f;
	int64_t r = 0;
	for (; r + 8 <= a.R; r += 8) {
		float gv[8], xv[8], mv[8], iv[8];
#pragma unroll
		for (int u = 0; u < 8; ++u) {
			gv[u] = a.g[(r + u) * a.D + col];
			xv[u] = a.x[(r + u) * a.D + col];
			mv[u] = a.mean[r + u];
			iv[u] = a.inv[r + u];
		}
#pragma unroll
		for (int u = 0; u < 8; ++u) {
			sg = sg + gv[u] * ((xv[u] - mv[u]) * iv[u]);
			sb = sb + gv[u];
		}
	}
	for (; r < a.R; ++r) {
		const float gv = a.g[r * a.D + col];
		sg = sg + gv * ((a.x[r * a.D + col] - a.mean[r]) * a.inv[r]);
		sb = sb + gv;
	}
	if (a.dgamma) a.dgamma[col] = a.dg_first ? 0.0f + sg : a.dgamma[col] + sg;
	if (a.dbeta) a.dbeta[col] = a.db_first ? 0.0f + sb : a.dbeta[col] + sb;
}

// ---- layernorm, a few rows per workgroup ----
// A workgroup of 256 threads owns `rw` consecutive rows (a contiguous block of rw * D floats) and keeps them in
// registers from the load to the store. Only the row chains (one dependent add per element, the reference's order) run
// over LDS: all threads put the terms there, element-wise, and one lane per chain adds them in order, sixteen at a time
// from 16-byte reads two blocks ahead, about 7 cycles an add (4.3 from registers; the reads take the rest). The rows of
// LDS are an odd number of 16-byte words apart, so that the lanes of a read (one row each) use different banks.
// What bounds it: the two (forward) or one (backward) chain of D adds, 1.5 us at D = 512, between the load and the store;
// rw is chosen so that 2 to 4 workgroups share a CU and one's chain runs beside another's memory traffic. Measured
// over [8192, 512]: forward 22.8 -> 12.4 us, dx alone 37.2 -> 12.0, against a version that also ran the element-wise
// passes in the chain lanes.
// PER: 16-byte groups (VEC) or quadruples of floats a thread holds: rw * D <= 1024 PER.

// Chains of one kind: in the forward a thread each; in the backward lanes 0 .. 31 of wave 0, the second kind lanes 32 .. 63.
constexpr int kLnMaxRows = 256, kLnMaxDxRows = 32;

__device__ __host__ __forceinline__ int ln_pitch(int D) { return 4 * (((D + 3) >> 2) | 1); }

struct LnArgs {
	const float* x;
	const float* g;       // backward: upstream gradient
	const float* gm;
	const float* bt;
	const float* mean_in;  // backward
	const float* inv_in;   // backward
	float* y;              // forward: y; backward: dx
	float* mean;           // forward
	float* inv;            // forward
	int64_t R;
	int D, rw, first;
	float fd, eps;
	FastDiv dq;            // D / 4 (VEC) or D
};

// The workgroup's elements as units of four consecutive floats of a row (VEC) or single floats (four to a slot): unit
// e of slot u. Calls f(slot, element in the slot, row, column, index in the block) for every element of the block, and
// with 16-byte units the elements of a slot share a row.
template <int PER, bool VEC, class F>
__device__ __forceinline__ void ln_each(int total, int D, const FastDiv& dq, F&& f) {
	const int tid = threadIdx.x;
#pragma unroll
	for (int u = 0; u < PER; ++u) {
		if constexpr (VEC) {
			const int q = tid + 256 * u;
			if (4 * q < total) {
				const int r = (int)fdiv((unsigned)q, dq), c = 4 * (q - r * (D >> 2));
				f(u, r, c, 4 * q);
			}
		} else {
#pragma unroll
			for (int i = 0; i < 4; ++i) {
				const int e = tid + 256 * (4 * u + i);
				if (e < total) {
					const int r = (int)fdiv((unsigned)e, dq);
					f(4 * u + i, r, e - r * D, e);
				}
			}
		}
	}
}

// The block's elements into registers, every load issued at an index clamped into the block.
template <int PER, bool VEC>
__device__ __forceinline__ void ln_load(const float* __restrict__ src, int total, f32x4 (&v)[PER]) {
	const int tid = threadIdx.x;
#pragma unroll
	for (int u = 0; u < PER; ++u) {
		if constexpr (VEC) {
			v[u] = *reinterpret_cast<const f32x4*>(src + 4 * min(tid + 256 * u, total / 4 - 1));
		} else {
#pragma unroll
			for (int i = 0; i < 4; ++i) v[u][i] = src[min(tid + 256 * (4 * u + i), total - 1)];
		}
	}
}

// layernorm forward (ops.cpp:1017-1030) on rw rows per workgroup.
template <int PER, bool VEC>
__global__ void __launch_bounds__(256) ln_forward_rows_kernel(const LnArgs a) {
	extern __shared__ __align__(16) float lds[];
	const int D = a.D, pitch = ln_pitch(D), tid = threadIdx.x;
	float* st = lds + a.rw * pitch;  // per row: mean, inv_std
	const int64_t r0 = (int64_t)blockIdx.x * a.rw;
	const int nr = (int)(a.R - r0 < a.rw ? a.R - r0 : a.rw), total = nr * D;
	f32x4 v[PER];
	ln_load<PER, VEC>(a.x + r0 * D, total, v);
	ln_each<PER, VEC>(total, D, a.dq, [&](int s, int r, int c, int) {
		if constexpr (VEC) *reinterpret_cast<f32x4*>(lds + r * pitch + c) = v[s];
		else lds[r * pitch + c] = v[s / 4][s % 4];
	});
	__syncthreads();
	if (tid < nr) st[2 * tid] = lds_chain(lds + tid * pitch, D) / a.fd;
	__syncthreads();
	ln_each<PER, VEC>(total, D, a.dq, [&](int s, int r, int c, int) {
		const float mu = st[2 * r];
		if constexpr (VEC) {
			f32x4 sq;
#pragma unroll
			for (int i = 0; i < 4; ++i) sq[i] = (v[s][i] - mu) * (v[s][i] - mu);
			*reinterpret_cast<f32x4*>(lds + r * pitch + c) = sq;
		} else {
			lds[r * pitch + c] = (v[s / 4][s % 4] - mu) * (v[s / 4][s % 4] - mu);
		}
	});
	__syncthreads();
	if (tid < nr) {
		const float inv = 1.0f / sqrtf(lds_chain(lds + tid * pitch, D) / a.fd + a.eps);
		st[2 * tid + 1] = inv;
		a.mean[r0 + tid] = st[2 * tid];
		a.inv[r0 + tid] = inv;
	}
	__syncthreads();
	float* out = a.y + r0 * D;
	ln_each<PER, VEC>(total, D, a.dq, [&](int s, int r, int c, int e) {
		const float mu = st[2 * r], inv = st[2 * r + 1];
		if constexpr (VEC) {
			f32x4 o;
#pragma unroll
			for (int i = 0; i < 4; ++i) o[i] = (v[s][i] - mu) * inv * a.gm[c + i] + a.bt[c + i];
			*reinterpret_cast<f32x4*>(out + e) = o;
		} else {
			out[e] = (v[s / 4][s % 4] - mu) * inv * a.gm[c] + a.bt[c];
		}
	});
}

// layernorm backward's dx (ops.cpp:1043-1060) on rw rows per workgroup: the terms g gamma and (g gamma) ((x - mean)
// inv_std) go to LDS for the row's two chains and stay in registers, as dxhat and xhat, for
// dx = k (D dxhat - sa - xhat sb).
template <int PER, bool VEC>
__device__ __forceinline__ void ln_dx_body(const LnArgs& a, int block, float* lds) {
	const int D = a.D, pitch = ln_pitch(D), tid = threadIdx.x;
	float* la = lds;
	float* lb = la + a.rw * pitch;
	float* st = lb + a.rw * pitch;  // per row: mean, inv_std, sa, sb
	const int64_t r0 = (int64_t)block * a.rw;
	const int nr = (int)(a.R - r0 < a.rw ? a.R - r0 : a.rw), total = nr * D;
	f32x4 dxh[PER], xh[PER];
	ln_load<PER, VEC>(a.g + r0 * D, total, dxh);
	ln_load<PER, VEC>(a.x + r0 * D, total, xh);
	if (tid < nr) {
		st[4 * tid] = a.mean_in[r0 + tid];
		st[4 * tid + 1] = a.inv_in[r0 + tid];
	}
	__syncthreads();
	ln_each<PER, VEC>(total, D, a.dq, [&](int s, int r, int c, int) {
		const float mu = st[4 * r], iv = st[4 * r + 1];
		if constexpr (VEC) {
			f32x4 p;
#pragma unroll
			for (int i = 0; i < 4; ++i) {
				dxh[s][i] = dxh[s][i] * a.gm[c + i];
				xh[s][i] = (xh[s][i] - mu) * iv;
				p[i] = dxh[s][i] * xh[s][i];
			}
			*reinterpret_cast<f32x4*>(la + r * pitch + c) = dxh[s];
			*reinterpret_cast<f32x4*>(lb + r * pitch + c) = p;
		} else {
			float& d = reinterpret_cast<float(&)[4 * PER]>(dxh)[s];
			float& h = reinterpret_cast<float(&)[4 * PER]>(xh)[s];
			d = d * a.gm[c];
			h = (h - mu) * iv;
			la[r * pitch + c] = d;
			lb[r * pitch + c] = d * h;
		}
	});
	__syncthreads();
	if (tid < 64 && (tid & (kLnMaxDxRows - 1)) < nr) {
		const int r = tid & (kLnMaxDxRows - 1), second = tid / kLnMaxDxRows;
		st[4 * r + 2 + second] = lds_chain((second ? lb : la) + r * pitch, D);
	}
	__syncthreads();
	const float fd = a.fd;
	float* dst = a.y + r0 * D;
	ln_each<PER, VEC>(total, D, a.dq, [&](int s, int r, int, int e) {
		const float k = st[4 * r + 1] / fd, sa = st[4 * r + 2], sb = st[4 * r + 3];
		if constexpr (VEC) {
			f32x4 o;
			if (!a.first) o = *reinterpret_cast<const f32x4*>(dst + e);
#pragma unroll
			for (int i = 0; i < 4; ++i) {
				const float term = k * (fd * dxh[s][i] - sa - xh[s][i] * sb);
				o[i] = a.first ? term + 0.0f : o[i] + term;
			}
			*reinterpret_cast<f32x4*>(dst + e) = o;
		} else {
			const float term = k * (fd * dxh[s / 4][s % 4] - sa - xh[s / 4][s % 4] * sb);
			dst[e] = a.first ? term + 0.0f : dst[e] + term;
		}
	});
}

struct LnColArgs {
	const float* g;
	const float* x;
	const float* mean;
	const float* inv;
	int64_t R;
	int D;
	float* dgamma;
	int dg_first;
	float* dbeta;
	int db_first;
	int blocks;  // workgroups of the column chains
};

// layernorm backward's dgamma and dbeta (ops.cpp:1061-1076): each is a chain down a column in row order, so the
// columns are the only parallelism, and about 7 cycles a row (24 us for 8192 rows) the least time. A workgroup of
// four waves, one a SIMD, owns 16 columns: waves 1-3 load the rows in chunks of 192, three chunks ahead in a register
// ring, form g * ((x - mean) * inv_std) exactly as the reference does and write it and g to LDS column by column (a
// column's rows back to back); wave 0, one chunk behind, adds: lanes 0-15 the products down their column (dgamma),
// lanes 16-31 g (dbeta), four rows per 16-byte read. One barrier a chunk, two buffers. 16 columns a workgroup keep the
// loads (64 bytes a row) at a third of what a CU can take. Measured for 8192 rows of 512: 37 us, and 39 with dx beside it
// (52 and 90 in two launches with 32 columns and fifteen producer waves, where the chain wave shared its SIMD with three
// producers and read one row at a time); of 64: 30 us against 51. Wide rows are bound by memory, so the two blocks that share
// a 128-byte line run on one XCD: 8192 rows of 4096 without dx 81 us in launch order, 50 so (32 columns a workgroup: 54).
constexpr int kLnCols = 16, kLnAhead = 3, kLnWaveRows = 64, kLnChunk = 3 * kLnWaveRows;
constexpr int kLnColPitch = kLnChunk + 4;  // 4 mod 64: the chain lanes' 16-byte reads use different banks
constexpr int kLnColBuf = 2 * kLnCols * kLnColPitch;
constexpr size_t kLnColLds = 2 * kLnColBuf * sizeof(float);

template <bool VEC>
__device__ __forceinline__ void ln_columns_body(const LnColArgs& d, int block, float* lds) {
	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int per = d.blocks / 8;  // neighbouring blocks share the rows' cache lines: a contiguous range for each XCD
	const int c0 = (block < per * 8 ? (block % 8) * per + block / 8 : block) * kLnCols, D = d.D;
	const int64_t R = d.R, chunks = (R + kLnChunk - 1) / kLnChunk;
	// a producer's slot u of a chunk: VEC row 16 u + lane / 4, columns 4 (lane % 4) ..; else row 4 u + lane / 16, column
	// lane % 16 (columns past D read a clamped address: their chains are not stored)
	constexpr int kSlots = VEC ? kLnWaveRows / 16 : kLnWaveRows / 4, kW = VEC ? 4 : 1;
	constexpr int kRowStep = VEC ? 16 : 4;
	const int cl = VEC ? 4 * (lane & 3) : lane & 15, rl = VEC ? lane >> 2 : lane >> 4;
	const int col = min(c0 + cl, D - kW);
	if (wave > 0) {
		float gv[kLnAhead][kSlots][kW], xv[kLnAhead][kSlots][kW], mv[kLnAhead][kSlots], iv[kLnAhead][kSlots];
		// a slot's offsets from its chunk's first row; the last chunk's rows past R read the last row
		const int row0 = (wave - 1) * kLnWaveRows + rl, left = (int)(R - (chunks - 1) * kLnChunk) - 1;
		unsigned off[kSlots], offl[kSlots];
#pragma unroll
		for (int u = 0; u < kSlots; ++u) {
			off[u] = (unsigned)(row0 + kRowStep * u) * (unsigned)D + (unsigned)col;
			offl[u] = (unsigned)min(row0 + kRowStep * u, left) * (unsigned)D + (unsigned)col;
		}
		auto load = [&](int64_t ch, int slot) {
			const float* gp = d.g + ch * kLnChunk * D;
			const float* xp = d.x + ch * kLnChunk * D;
			const float* mp = d.mean + ch * kLnChunk;
			const float* ip = d.inv + ch * kLnChunk;
			const bool last = ch == chunks - 1;
#pragma unroll
			for (int u = 0; u < kSlots; ++u) {
				const unsigned o = last ? offl[u] : off[u];
				const unsigned r = last ? (unsigned)min(row0 + kRowStep * u, left) : (unsigned)(row0 + kRowStep * u);
				if constexpr (VEC) {
					const f32x4 g4 = *reinterpret_cast<const f32x4*>(gp + o);
					const f32x4 x4 = *reinterpret_cast<const f32x4*>(xp + o);
#pragma unroll
					for (int i = 0; i < 4; ++i) {
						gv[slot][u][i] = g4[i];
						xv[slot][u][i] = x4[i];
					}
				} else {
					gv[slot][u][0] = gp[o];
					xv[slot][u][0] = xp[o];
				}
				mv[slot][u] = mp[r];
				iv[slot][u] = ip[r];
			}
		};
#pragma unroll
		for (int k = 0; k < kLnAhead; ++k) load(min((int64_t)k, chunks - 1), k);
		auto step = [&](int64_t ch, int k) {
			float* pr = lds + (ch & 1) * kLnColBuf;
			float* gg = pr + kLnCols * kLnColPitch;
#pragma unroll
			for (int u = 0; u < kSlots; ++u) {
				const int row = (wave - 1) * kLnWaveRows + kRowStep * u + rl;
#pragma unroll
				for (int i = 0; i < kW; ++i) {
					pr[(cl + i) * kLnColPitch + row] = gv[k][u][i] * ((xv[k][u][i] - mv[k][u]) * iv[k][u]);
					gg[(cl + i) * kLnColPitch + row] = gv[k][u][i];
				}
			}
			load(min(ch + kLnAhead, chunks - 1), k);
			__syncthreads();
		};
		// whole rounds without a branch, so that the compiler waits for each slot's loads by count, then the rest
		int64_t ch = 0;
		for (; ch + kLnAhead <= chunks; ch += kLnAhead) {
#pragma unroll
			for (int k = 0; k < kLnAhead; ++k) step(ch + k, k);
		}
#pragma unroll
		for (int k = 0; k < kLnAhead - 1; ++k)
			if (ch + k < chunks) step(ch + k, k);
		return;
	}
	// wave 0: at barrier ch chunk ch is whole; it is added before the producers, two barriers on, reuse its buffer
	float acc = 0.0f;
	const float* mine = lds + (lane & 31) * kLnColPitch;
	__syncthreads();
	for (int64_t ch = 0; ch < chunks; ++ch) {
		const float* v = mine + (ch & 1) * kLnColBuf;
		if (ch + 1 < chunks) {
			const f32x4* q = reinterpret_cast<const f32x4*>(v);
			constexpr int kB = kLnChunk / 16;
			f32x4 t[3][4];
#pragma unroll
			for (int b = 0; b < 2; ++b)
#pragma unroll
				for (int e = 0; e < 4; ++e) t[b][e] = q[4 * b + e];
#pragma unroll
			for (int b = 0; b < kB; ++b) {
				if (b + 2 < kB) {
#pragma unroll
					for (int e = 0; e < 4; ++e) t[(b + 2) % 3][e] = q[4 * (b + 2) + e];
				}
				__builtin_amdgcn_sched_barrier(0);  // keeps the reads ahead of the adds they run beside
#pragma unroll
				for (int e = 0; e < 4; ++e)
#pragma unroll
					for (int i = 0; i < 4; ++i) acc = acc + t[b % 3][e][i];
			}
			__syncthreads();
		} else {
			acc = lds_chain(v, (int)(R - ch * kLnChunk), acc);
		}
	}
	const int j = c0 + (lane & 15);
	if (lane >= 32 || j >= D) return;
	if (lane < 16) {
		if (d.dgamma) d.dgamma[j] = d.dg_first ? 0.0f + acc : d.dgamma[j] + acc;
	} else {
		if (d.dbeta) d.dbeta[j] = d.db_first ? 0.0f + acc : d.dbeta[j] + acc;
	}
}

// dgamma and dbeta for at most 1024 rows (transformer_tiny's 16 x 64 tokens): the same chains, one pass. A
// workgroup owns a few columns (four with 1024 threads alone, one with 256 threads beside dx, so that the loads
// spread over many CUs); every thread loads its share of a column's rows (g, x, the rows' mean and inv_std, all in
// flight at once) and parks g * ((x - mean) * inv_std) and g in LDS, column by column; then one lane per column adds
// the products down it in row order (dgamma) and one the gradients (dbeta), four rows per 16-byte LDS read. Rows
// past R are parked as +0: a chain from +0 never holds -0 (x + (-x) rounds to +0, and no sum of finite floats
// underflows to zero), so adding +0 leaves it unchanged.
constexpr int kLnSmallRows = 1024, kLnSmallThreads = 1024;
constexpr int kLnSmallCols = 4;     // columns of a workgroup of the standalone kernel
constexpr int kLnMergedCols = 1;    // columns of a 256-thread workgroup beside dx
constexpr int kLnSmallPitch = kLnSmallRows + 4;  // a column's rows, padded against bank conflicts of the stores
constexpr size_t kLnMergedLds = 2 * kLnMergedCols * kLnSmallPitch * sizeof(float);

// block: the workgroup's index among the chains' workgroups; THREADS its size, COLS its columns; buf:
// 2 COLS kLnSmallPitch floats of LDS.
template <int THREADS, int COLS>
__device__ __forceinline__ void ln_dgamma_small_body(const LnColArgs& d, int block, float* buf) {
	constexpr int kRowStep = THREADS / COLS;
	constexpr int kPer = kLnSmallRows / kRowStep;
	const int R = (int)d.R, D = d.D;
	const int tid = threadIdx.x;
	const int c = tid % COLS, r0 = tid / COLS;  // rows r0 + kRowStep u
	const int c0 = block * COLS;
	const int col = min(c0 + c, D - 1);
	float gv[kPer], xv[kPer], mv[kPer], iv[kPer];
#pragma unroll
	for (int u = 0; u < kPer; ++u) {
		const int64_t r = min(r0 + kRowStep * u, R - 1);
		gv[u] = d.g[r * D + col];
		xv[u] = d.x[r * D + col];
		mv[u] = d.mean[r];
		iv[u] = d.inv[r];
	}
	// the chains read whole blocks of 32 rows
	const int rpad = (R + 31) & ~31;
#pragma unroll
	for (int u = 0; u < kPer; ++u) {
		const int r = r0 + kRowStep * u;
		if (r < rpad) {
			const bool in = r < R;
			buf[c * kLnSmallPitch + r] = in ? gv[u] * ((xv[u] - mv[u]) * iv[u]) : 0.0f;
			buf[(COLS + c) * kLnSmallPitch + r] = in ? gv[u] : 0.0f;
		}
	}
	__syncthreads();
	if (tid >= 2 * COLS) return;
	// lane c: column c's products (dgamma); lane COLS + c: its gradients (dbeta). Rows in order, 32 at a time; the
	// reads of the next two blocks are in flight while one is added (a dependent add takes about six cycles).
	const f32x4* v = reinterpret_cast<const f32x4*>(buf + tid * kLnSmallPitch);
	const int nb = rpad / 32;
	float acc = 0.0f;
	f32x4 t[3][8];
#pragma unroll
	for (int e = 0; e < 8; ++e) t[0][e] = v[e];
	if (nb > 1) {
#pragma unroll
		for (int e = 0; e < 8; ++e) t[1][e] = v[8 + e];
	}
	for (int b = 0; b < nb; b += 3) {
#pragma unroll
		for (int k = 0; k < 3; ++k) {
			if (b + k >= nb) break;
			if (b + k + 2 < nb) {
#pragma unroll
				for (int e = 0; e < 8; ++e) t[(k + 2) % 3][e] = v[8 * (b + k + 2) + e];
			}
#pragma unroll
			for (int e = 0; e < 8; ++e)
#pragma unroll
				for (int q = 0; q < 4; ++q) acc = acc + t[k][e][q];
		}
	}
	if (c0 + c >= D) return;
	const int j = c0 + c;
	if (tid < COLS) {
		if (d.dgamma) d.dgamma[j] = d.dg_first ? 0.0f + acc : d.dgamma[j] + acc;
	} else {
		if (d.dbeta) d.dbeta[j] = d.db_first ? 0.0f + acc : d.dbeta[j] + acc;
	}
}

__global__ void __launch_bounds__(kLnSmallThreads) ln_dgamma_small_kernel(const LnColArgs d) {
	__shared__ __align__(16) float buf[2 * kLnSmallCols * kLnSmallPitch];
	ln_dgamma_small_body<kLnSmallThreads, kLnSmallCols>(d, (int)blockIdx.x, buf);
}

// One layernorm backward in one launch: the workgroups of the column chains first, since theirs is the longest work,
// then the dx row blocks beside them on the other CUs. COLS: no chains (0), those of at most 1024 rows, a column a
// workgroup (1), or of any number of rows, 16 columns a workgroup (2).
template <int PER, bool VEC, int COLS>
__global__ void __launch_bounds__(256) ln_backward_rows_kernel(const LnArgs a, const LnColArgs d) {
	extern __shared__ __align__(16) float lds[];
	if (COLS != 0 && (int)blockIdx.x < d.blocks) {
		if constexpr (COLS == 1) ln_dgamma_small_body<256, kLnMergedCols>(d, (int)blockIdx.x, lds);
		if constexpr (COLS == 2) ln_columns_body<VEC>(d, (int)blockIdx.x, lds);
		return;
	}
	ln_dx_body<PER, VEC>(a, (int)blockIdx.x - d.blocks, lds);
}

constexpr int kLnMaxPer = 16;
constexpr int kLnMaxD = 1024 * kLnMaxPer;  // longest row a workgroup holds in registers

using LnForwardFn = void (*)(const LnArgs);
using LnBackwardFn = void (*)(const LnArgs, const LnColArgs);
// [PER 2, 8, 16][VEC]
const LnForwardFn kLnForward[3][2] = {{ln_forward_rows_kernel<2, false>, ln_forward_rows_kernel<2, true>},
                                      {ln_forward_rows_kernel<8, false>, ln_forward_rows_kernel<8, true>},
                                      {ln_forward_rows_kernel<16, false>, ln_forward_rows_kernel<16, true>}};
// [PER 16][VEC][COLS]
const LnBackwardFn kLnBackward[2][2][3] = {
    {{ln_backward_rows_kernel<8, false, 0>, ln_backward_rows_kernel<8, false, 1>, ln_backward_rows_kernel<8, false, 2>},
     {ln_backward_rows_kernel<8, true, 0>, ln_backward_rows_kernel<8, true, 1>, ln_backward_rows_kernel<8, true, 2>}},
    {{ln_backward_rows_kernel<16, false, 0>, ln_backward_rows_kernel<16, false, 1>, ln_backward_rows_kernel<16, false, 2>},
     {ln_backward_rows_kernel<16, true, 0>, ln_backward_rows_kernel<16, true, 1>, ln_backward_rows_kernel<16, true, 2>}}};

// Raises the kernels' dynamic LDS limit once per device (a row of kLnMaxD floats and its product: 131 KB).
hipError_t prepare_norm() {
	static std::mutex mu;
	static bool done[64] = {};
	int dev = 0;
	hipError_t e = hipGetDevice(&dev);
	if (e != hipSuccess) return e;
	if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
	std::lock_guard<std::mutex> lock(mu);
	if (done[dev]) return hipSuccess;
	auto raise = [&](const void* fn) {
		if (e == hipSuccess) e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
	};
	raise(reinterpret_cast<const void*>(bn_rows_kernel<kBwd, false, BnLong>));  // two sets of terms: 76 KB
	raise(reinterpret_cast<const void*>(bn_rows_kernel<kBwd, true, BnLong>));
	raise(reinterpret_cast<const void*>(bn_rows_kernel<kBwd, false, BnMedium>));
	raise(reinterpret_cast<const void*>(bn_rows_kernel<kBwd, true, BnMedium>));
	for (int v = 0; v < 2; ++v) {
		for (int p = 0; p < 3; ++p) raise(reinterpret_cast<const void*>(kLnForward[p][v]));
		for (int p = 0; p < 2; ++p)
			for (int c = 0; c < 3; ++c) raise(reinterpret_cast<const void*>(kLnBackward[p][v][c]));
	}
	done[dev] = e == hipSuccess;
	return e;
}

// Rows per workgroup: as many as its registers and chain lanes hold, but few enough for about `blocks` workgroups, and
// enough that every thread has an element.
int ln_rows(int64_t R, int D, int blocks, int max_rows) {
	const int64_t most = std::max<int64_t>(1, std::min<int64_t>(max_rows, (D <= 8192 ? 8192 : kLnMaxD) / D));
	return (int)std::max<int64_t>(1, std::min(std::min(most, R), std::max<int64_t>((R + blocks - 1) / blocks, (255 + D) / D)));
}

inline bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

template <int MODE, class SH>
hipError_t launch_rows_as(BnRowArgs& a, bool vec, hipStream_t s) {
	const hipError_t e = prepare_norm();
	if (e != hipSuccess) return e;
	a.groups = std::max<int64_t>(1, (a.N + SH::kRows - 1) / SH::kRows);
	const int per = vec ? 4 : 1;
	const int64_t last = a.S > 0 ? (a.S - 1) % SH::kChunk + 1 : per;
	a.whole = make_fastdiv((unsigned)(SH::kChunk / per));
	a.last = make_fastdiv((unsigned)(last / per));
	const int64_t blocks = a.C * a.groups;
	for (a.first_block = 0; a.first_block < blocks; a.first_block += kMaxGrid) {
		hipLaunchKernelGGL((vec ? bn_rows_kernel<MODE, true, SH> : bn_rows_kernel<MODE, false, SH>),
		                   dim3((unsigned)std::min(kMaxGrid, blocks - a.first_block)), dim3(256),
		                   (MODE == kBwd ? 2 : 1) * SH::kRowSet * sizeof(float), s, a);
		const hipError_t err = hipGetLastError();
		if (err != hipSuccess) return err;
	}
	return hipSuccess;
}

// Rows a workgroup. Every workgroup of the squares repeats the channel's double sum over N rows (about 8 cycles a row), and
// issues its loads for a whole chunk, so short rows go 32 to a workgroup, and rows of up to 1024 go 8 as long as 256
// workgroups are left. Forward and backward with four rows a workgroup against this (us): [256, 256] 243 -> 30 and 171 ->
// 21, [4096, 128] 5707 -> 644 and 1339 -> 146, [64, 576, 7 x 7] 141 -> 29 and 115 -> 28, [27, 60] 19.9 -> 15.5, [64, 128, 14 x
// 14] 25.8 -> 22.5 and 22.5 -> 18.0, [128, 64, 28 x 28] 32 -> 30 and 35 -> 32. The backward's two sets of terms fill LDS with
// 1024 long rows: from 900 on four rows are faster ([32, 64, 32 x 32] 13.5 against 16.9), as for a few aligned rows from 64
// ([32, 8, 10 x 10] 10.7 against 11.6).
template <int MODE>
hipError_t launch_rows(BnRowArgs& a, bool vec, hipStream_t s) {
	auto fills = [&](int rows) { return a.C * ((a.N + rows - 1) / rows) >= 256; };
	if (a.S <= BnShort::kChunk && (MODE != kBwd || !vec || a.S <= 64 || fills(BnShort::kRows)))
		return launch_rows_as<MODE, BnShort>(a, vec, s);
	if (a.S <= (MODE == kBwd ? 768 : BnMedium::kChunk) && fills(BnMedium::kRows))
		return launch_rows_as<MODE, BnMedium>(a, vec, s);
	return launch_rows_as<MODE, BnLong>(a, vec, s);
}

hipError_t launch_elem(bool fwd, BnElemArgs& a, hipStream_t s) {
	const int64_t total = a.N * a.S;
	a.chunks = total > 0 ? (total + kElemChunk - 1) / kElemChunk : 1;
	const bool fast = total < ((int64_t)1 << 31) && a.S > 0 && a.S < ((int64_t)1 << 31);
	if (fast) a.sdiv = make_fastdiv((unsigned)a.S);
	const dim3 grid((unsigned)(a.C * a.chunks));
	if (fwd) {
		if (fast) hipLaunchKernelGGL(bn_norm_kernel<true>, grid, dim3(256), 0, s, a);
		else hipLaunchKernelGGL(bn_norm_kernel<false>, grid, dim3(256), 0, s, a);
	} else {
		const bool ahead = a.N <= 512;
		const auto fn = fast ? (ahead ? bn_dx_kernel<true, true> : bn_dx_kernel<true, false>)
		                     : (ahead ? bn_dx_kernel<false, true> : bn_dx_kernel<false, false>);
		hipLaunchKernelGGL(fn, grid, dim3(256), 0, s, a);
	}
	return hipGetLastError();
}

}  // namespace

hipError_t batchnorm_forward(const float* x, const float* w, const float* b, const BnGeom& g, float eps, int relu,
                             float* y, unsigned char* alive, float* mean, float* var, float* inv_std, float* scratch,
                             hipStream_t s) {
	if (g.C == 0) return hipSuccess;
	const bool vec = g.S % 4 == 0 && aligned16(x) && aligned16(y) && (!alive || reinterpret_cast<uintptr_t>(alive) % 4 == 0);
	float* rowsum = scratch;
	float* rowsq = scratch + g.N * g.C;
	BnRowArgs r{};
	r.x = x;
	r.out0 = rowsum;
	r.N = g.N;
	r.C = g.C;
	r.S = g.S;
	r.dm = g.dm;
	const bool row_vec = g.S % 4 == 0 && aligned16(x);
	hipError_t e = hipSuccess;
	if (g.N > 0) {
		e = launch_rows<kSum>(r, row_vec, s);
		if (e != hipSuccess) return e;
	}
	r.rowsum = rowsum;
	r.out0 = rowsq;
	r.mean_out = mean;
	e = launch_rows<kSq>(r, row_vec, s);  // also writes the channel means (a workgroup per channel when N is 0)
	if (e != hipSuccess) return e;
	BnElemArgs a{};
	a.x = x;
	a.w = w;
	a.b = b;
	a.rowv0 = rowsq;
	a.mean = mean;
	a.y = y;
	a.alive = alive;
	a.var_out = var;
	a.inv_out = inv_std;
	a.N = g.N;
	a.C = g.C;
	a.S = g.S;
	a.dm = g.dm;
	a.fm = g.fm;
	a.eps = eps;
	a.relu = relu;
	a.vec = vec;
	return launch_elem(true, a, s);
}

hipError_t batchnorm_backward(const float* gy, const float* x, const unsigned char* alive, const float* w,
                              const float* mean, const float* inv_std, const BnGeom& g, float* dx, int dx_first,
                              float* dw, int dw_first, float* db, int db_first, float* scratch, hipStream_t s) {
	if (g.C == 0 || (!dx && !dw && !db)) return hipSuccess;
	float* rowdy = scratch;
	float* rowdg = scratch + g.N * g.C;
	if (g.N > 0) {
		BnRowArgs r{};
		r.x = x;
		r.g = gy;
		r.alive = alive;
		r.mean = mean;
		r.out0 = rowdy;
		r.out1 = rowdg;
		r.N = g.N;
		r.C = g.C;
		r.S = g.S;
		r.dm = g.dm;
		const bool row_vec =
		    g.S % 4 == 0 && aligned16(x) && aligned16(gy) && (!alive || reinterpret_cast<uintptr_t>(alive) % 4 == 0);
		const hipError_t e = launch_rows<kBwd>(r, row_vec, s);
		if (e != hipSuccess) return e;
	}
	BnElemArgs a{};
	a.x = x;
	a.g = gy;
	a.alive_in = alive;
	a.w = w;
	a.rowv0 = rowdy;
	a.rowv1 = rowdg;
	a.mean = mean;
	a.inv_in = inv_std;
	a.y = dx;
	a.dw = dw;
	a.db = db;
	a.N = g.N;
	a.C = g.C;
	a.S = g.S;
	a.dm = g.dm;
	a.fm = g.fm;
	a.first = dx_first;
	a.dw_first = dw_first;
	a.db_first = db_first;
	a.vec = g.S % 4 == 0 && aligned16(x) && aligned16(gy) && aligned16(dx) &&
	        (!alive || reinterpret_cast<uintptr_t>(alive) % 4 == 0);
	return launch_elem(false, a, s);
}

hipError_t layernorm_forward(const float* x, const float* gamma, const float* beta, int64_t R, int D, float fd,
                             float eps, float* y, float* mean, float* inv_std, hipStream_t s) {
	if (R == 0) return hipSuccess;
	const bool vec = D % 4 == 0 && aligned16(x) && aligned16(y);
	// Short rows in workgroups of 2048 floats, two 16-byte groups a thread: with more, each thread issues eight groups (or 32
	// single floats) however few the rows are, and 32 rows of a few floats are no work for a workgroup. Against 32 rows a
	// workgroup and eight groups (us): [8192, 5] 4.2 -> 3.2, [262144, 5] 35 -> 5.7, [262144, 32] 22 -> 12.5, unaligned [32768,
	// 65] 12.3 -> 8.1. Aligned rows above 64 are as fast in larger blocks, all rows above 256 faster ([8192, 1537] 67 against
	// 95, [1024, 2048] 30.7 against 32.8).
	const int rw = ln_rows(R, D, 1024, D <= (vec ? 64 : 256) ? std::min(2048 / D, kLnMaxRows) : kLnMaxRows);
	if (D <= kLnMaxD && R / rw < kMaxGrid) {
		LnArgs a{};
		a.x = x;
		a.gm = gamma;
		a.bt = beta;
		a.y = y;
		a.mean = mean;
		a.inv = inv_std;
		a.R = R;
		a.D = D;
		a.rw = rw;
		a.fd = fd;
		a.eps = eps;
		a.dq = make_fastdiv((unsigned)(vec ? D / 4 : D));
		const hipError_t e = prepare_norm();
		if (e != hipSuccess) return e;
		const int per = D <= 256 && rw * D <= 2048 ? 0 : D <= 8192 ? 1 : 2;
		hipLaunchKernelGGL(kLnForward[per][vec ? 1 : 0], dim3((unsigned)((R + rw - 1) / rw)), dim3(256),
		                   (size_t)rw * (ln_pitch(D) + 2) * sizeof(float), s, a);
		return hipGetLastError();
	}
	hipLaunchKernelGGL(ln_forward_kernel, dim3((unsigned)((R + 255) / 256)), dim3(256), 0, s, x, gamma, beta, R, D, fd,
	                   eps, y, mean, inv_std, vec && aligned16(gamma) && aligned16(beta) ? 1 : 0);
	return hipGetLastError();
}

hipError_t layernorm_backward(const float* gy, const float* x, const float* gamma, const float* mean,
                              const float* inv_std, int64_t R, int D, float fd, float* dx, int dx_first,
                              float* dgamma, int dgamma_first, float* dbeta, int dbeta_first, hipStream_t s) {
	if (R == 0 && !dgamma && !dbeta) return hipSuccess;
	const int rw = ln_rows(std::max<int64_t>(R, 1), D, 512, kLnMaxDxRows);
	const bool cols = dgamma || dbeta;
	// Column sums alone of up to 1024 wide rows: a thread a column, coalesced, without LDS. The small kernel's four columns a
	// workgroup read 16 bytes a row: 1 row of 8192 10.1 us against 2.1, 512 rows of 4096 27.5 against 20, 1024 rows 58 against
	// 50, of 2048 17.5 against 20.
	const bool wide_cols = !dx && R <= kLnSmallRows && D >= 4096;
	if (D <= kLnMaxD && R > 0 && !wide_cols) {
		LnArgs a{};
		a.gm = gamma;
		a.D = D;
		a.rw = rw;
		a.fd = fd;
		a.first = dx_first;
		const bool vec = D % 4 == 0 && aligned16(x) && aligned16(gy) && (!dx || aligned16(dx));
		a.dq = make_fastdiv((unsigned)(vec ? D / 4 : D));
		LnColArgs d{gy, x, mean, inv_std, R, D, dgamma, dgamma_first, dbeta, dbeta_first, 0};
		const bool small = cols && R <= kLnSmallRows;
		hipError_t e = prepare_norm();
		if (e != hipSuccess) return e;
		if (small && !dx) {
			d.blocks = (D + kLnSmallCols - 1) / kLnSmallCols;
			hipLaunchKernelGGL(ln_dgamma_small_kernel, dim3((unsigned)d.blocks), dim3(kLnSmallThreads), 0, s, d);
			return hipGetLastError();
		}
		if (cols) d.blocks = small ? (D + kLnMergedCols - 1) / kLnMergedCols : (D + kLnCols - 1) / kLnCols;
		const size_t lds_dx = dx ? (size_t)rw * (2 * ln_pitch(D) + 4) * sizeof(float) : 0;
		const size_t lds_cols = !cols ? 0 : small ? kLnMergedLds : kLnColLds;
		const auto* fns = kLnBackward[D > 8192 ? 1 : 0][vec ? 1 : 0];
		// the columns and the rows of one launch, then the rows that are left
		const int64_t most = (kMaxGrid - kLnMaxD) * rw;
		for (int64_t r0 = 0; r0 < R && (r0 == 0 || dx); r0 += most) {
			a.g = gy + r0 * D;
			a.x = x + r0 * D;
			a.mean_in = mean + r0;
			a.inv_in = inv_std + r0;
			a.y = dx ? dx + r0 * D : nullptr;
			a.R = std::min(most, R - r0);
			const int64_t blocks = d.blocks + (dx ? (a.R + rw - 1) / rw : 0);
			hipLaunchKernelGGL(fns[d.blocks == 0 ? 0 : small ? 1 : 2], dim3((unsigned)blocks), dim3(256),
			                   std::max(lds_dx, lds_cols), s, a, d);
			e = hipGetLastError();
			if (e != hipSuccess) return e;
			d.blocks = 0;
		}
		return hipSuccess;
	}
	LnBwdArgs a{};
	a.g = gy;
	a.x = x;
	a.gm = gamma;
	a.mean = mean;
	a.inv = inv_std;
	a.dx = dx;
	a.dgamma = dgamma;
	a.dbeta = dbeta;
	a.R = R;
	a.D = D;
	a.fd = fd;
	a.dx_first = dx_first;
	a.dg_first = dgamma_first;
	a.db_first = dbeta_first;
	a.row_blocks = dx ? (unsigned)((R + 255) / 256) : 0u;
	const unsigned col_blocks = (dgamma || dbeta) ? (unsigned)((D + 255) / 256) : 0u;
	if (a.row_blocks + col_blocks == 0) return hipSuccess;
	hipLaunchKernelGGL(ln_backward_kernel, dim3(a.row_blocks + col_blocks), dim3(256), 0, s, a);
	return hipGetLastError();
}

}  // namespace nnh
