// batchnorm.hip - nn::batchnorm (training mode, optionally with its folded ReLU), forward and backward
// (src/autograd/ops.cpp:900-1000), with the reference's summation orders.
//
// The reference gives each channel to one thread: for n = 0..N-1 in order it adds, in double, the
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
// These kernels are a few microseconds each and run in turn, so their code is kept together, apart from the layer norm's:
// with both in one code object a pass over [64, 16, 48, 48] took 42 us, and 39 so.
#include <algorithm>
#include <mutex>

#include "fastdiv.hpp"
#include "norm.hpp"
#include "norm_common.hpp"

namespace nnh {

namespace {

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

// Raises the kernels' dynamic LDS limit once per device (two sets of terms: 76 KB).
hipError_t prepare_batchnorm() {
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
	raise(reinterpret_cast<const void*>(bn_rows_kernel<kBwd, false, BnLong>));
	raise(reinterpret_cast<const void*>(bn_rows_kernel<kBwd, true, BnLong>));
	raise(reinterpret_cast<const void*>(bn_rows_kernel<kBwd, false, BnMedium>));
	raise(reinterpret_cast<const void*>(bn_rows_kernel<kBwd, true, BnMedium>));
	done[dev] = e == hipSuccess;
	return e;
}

template <int MODE, class SH>
hipError_t launch_rows_as(BnRowArgs& a, bool vec, hipStream_t s) {
	const hipError_t e = prepare_batchnorm();
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
		if (!fast) hipLaunchKernelGGL((bn_dx_kernel<false, false>), grid, dim3(256), 0, s, a);
		else if (a.N <= 512) hipLaunchKernelGGL((bn_dx_kernel<true, true>), grid, dim3(256), 0, s, a);
		else hipLaunchKernelGGL((bn_dx_kernel<true, false>), grid, dim3(256), 0, s, a);
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

}  // namespace nnh
