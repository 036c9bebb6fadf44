// norm.hip - nn::layernorm, forward and backward (src/autograd/ops.cpp:1002-1078), with the reference's summation orders.
//
// Each row's sums are single float chains (ops.cpp:1017-1026): a workgroup holds some rows in registers, all
// its threads form the chains' terms and put them in LDS, and one thread a chain adds them there. The gamma/beta
// gradient sums run down columns in row order (ops.cpp:1063-1075): chains over LDS again, beside dx in the same launch.
// Longer rows than a workgroup's registers hold take one thread a row and one a column.
#include "norm.hpp"

#include <algorithm>
#include <mutex>

#include "fastdiv.hpp"
#include "norm_common.hpp"

namespace nnh {

namespace {

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
hipError_t prepare_layernorm() {
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

}  // namespace

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
		const hipError_t e = prepare_layernorm();
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
		hipError_t e = prepare_layernorm();
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
