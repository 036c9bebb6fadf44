// gemm_ring.hip - which products run on the ring kernel (gemm_ring.hpp), on which tile, and their launch.
#include "gemm_ring.hpp"

#include <cmath>
#include <mutex>

#include "gemm.hpp"
#include "gemm_valu.hpp"

namespace nnh {

namespace {

enum { kRing256x128 = 0, kRing128x128 = 1, kRing64x64 = 2, kRing32x32 = 3 };

const RingConfig* ring_configs() {
	static const RingConfig table[kRingConfigs] = {ring_config_256x128(), ring_config_128x128(), ring_config_64x64(),
	                                               ring_config_32x32()};
	return table;
}

// Raises the kernels' dynamic LDS limit once per device.
hipError_t prepare_ring() {
	static std::mutex mu;
	static bool done[64] = {};
	int dev = 0;
	hipError_t e = hipGetDevice(&dev);
	if (e != hipSuccess) return e;
	if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
	std::lock_guard<std::mutex> lock(mu);
	if (done[dev]) return hipSuccess;
	for (int i = 0; i < kRingConfigs; ++i) {
		const RingConfig& c = ring_configs()[i];
		for (int v = 0; v < 2; ++v)
			for (int f = 0; f < 6; ++f) {
				const auto fn = f < 4 ? c.fn[f][v] : f == 4 ? c.rowsum_fn[v] : c.gelu_fn[v];
				e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
				                        c.lds_bytes);
				if (e != hipSuccess) return e;
			}
	}
	for (int i = 0; i < 12; ++i) {
		e = hipFuncSetAttribute(reinterpret_cast<const void*>(ring_pair_32x32(i / 4, (i / 2) & 1, i & 1)),
		                        hipFuncAttributeMaxDynamicSharedMemorySize, ring_configs()[kRing32x32].lds_bytes);
		if (e != hipSuccess) return e;
	}
	done[dev] = true;
	return hipSuccess;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// 16-byte operand loads: aligned rows whose contiguous length is whole chunks of four, so that no chunk crosses it.
bool ring_vec(const GemmCall& g) {
	bool ok = aligned16(g.a) && aligned16(g.b) && g.lda % 4 == 0 && g.ldb % 4 == 0 && (g.ta ? g.m : g.k) % 4 == 0 &&
	          (g.tb ? g.k : g.n) % 4 == 0;
	for (int d = 0; d < g.batch.ndim; ++d) ok = ok && g.batch.sa[d] % 4 == 0 && g.batch.sb[d] % 4 == 0;
	return ok;
}

// The time of `tiles` workgroups on a chip of 256 CUs, in cycles, for `steps` 32-deep steps. Measured per step: 256 x 128
// 8790 cycles (8192 of them MFMAs), 128 x 128 4610 (4096), 64 x 64 2380 for the two workgroups a CU holds (2048) and
// 1450 for one alone (1024), 32 x 32 830 for two with A transposed and B not (512; 960 for the other layouts, whose
// k-contiguous rows are a large stride apart and crowd a few L2 channels) and 490 (600) for one alone, whose waves have one
// dependent MFMA chain each. A workgroup's start and end (first loads, stores) add the constants.
double ring_cost(const GemmCall& g, double tiles, double steps, int config) {
	const double rounds = tiles / 256;
	auto pairs = [&](double two, double one, double ends) {  // two workgroups a CU
		const double full = std::floor(rounds / 2), rest = std::ceil(rounds - 2 * full);
		return full * (two * steps + ends) + (rest > 1 ? two * steps + ends : rest > 0 ? one * steps + ends : 0);
	};
	switch (config) {
		case kRing256x128: return std::ceil(rounds) * (8790 * steps + 12000);
		case kRing128x128: return std::ceil(rounds) * (4610 * steps + 9000);
		case kRing64x64: return pairs(2380, 1450, 5000);
		default: return g.ta && !g.tb ? pairs(830, 490, 4500) : pairs(960, 600, 4500);
	}
}

bool narrow(const GemmCall& g) {
	return g.m >= 128 && g.n < 128 && (double)g.m * (double)g.n * (double)g.batch_count >= 512.0 * 128 * 64;
}

int ring_pick(const GemmCall& g) {
	const double steps = (double)((g.k + 31) / 32);
	int best = kRing64x64;
	double cost = 0;
	for (int i = 0; i < kRingConfigs; ++i) {
		// one float a lane takes the 256 x 128 tile's load addresses past its registers
		if (i == kRing256x128 && !ring_vec(g)) continue;
		const RingConfig& c = ring_configs()[i];
		const double tiles = (double)((g.m + c.bm - 1) / c.bm) * (double)((g.n + c.bn - 1) / c.bn) * (double)g.batch_count;
		const double t = ring_cost(g, tiles, steps, i);
		if (i == 0 || cost == 0 || t < cost) {
			cost = t;
			best = i;
		}
	}
	return best;
}

// A launch holds fewer than 2^32 work-items.
bool ring_grid_ok(const GemmCall& g) {
	const RingConfig& c = ring_configs()[ring_pick(g)];
	return (double)((g.m + c.bm - 1) / c.bm) * (double)((g.n + c.bn - 1) / c.bn) * (double)g.batch_count * c.threads < 4294967296.0;
}

}  // namespace

bool ring_ok(const GemmCall& g) {
	// the offsets of a tile's rows are 32-bit byte counts: 256 rows of 2^21 floats stay below 2^31
	constexpr int64_t kMaxLd = int64_t(1) << 21;
	if (g.gather || g.k <= 0 || depth_cut(g.m, g.n, g.k) || g.lda >= kMaxLd || g.ldb >= kMaxLd ||
	    g.batch_count >= (int64_t(1) << 31))
		return false;
	return !g.rowsum || (g.ta && !g.tb && g.rowsum_outer == 0 && g.batch_count == 1 && g.batch.ndim == 0);
}

bool ring_takes_large(const GemmCall& g) {
	// Products with a 64 x 64 tile for two thirds of the CUs or more, and a depth of a few stages. Measured against the
	// tile kernels (us): 4096^3 NN 1106 -> 974, 2048^3 157 -> 137, 1024^3 28.8 -> 23.9, 8192 x 512 x 2048 NT 152 -> 136,
	// 2048 x 512 x 8192 TN 205 -> 150, 1021 x 771 x 1533 NN (one float a lane) 79 -> 39, 300 x 3000 x 500 24 -> 14.
	// With fewer tiles the tile kernels' three 32 x 32 workgroups a CU win (768^3, 144 tiles: 16.7 us against 18.4), and
	// products narrower than 128 with 2^22 outputs or more (attention's 256 x 64 per head) keep their 128 x 64 tiles
	// (256 of them, 256 deep: 26 to 31 us against 29 to 33).
	if (!ring_ok(g) || g.k < 96) return false;
	if (narrow(g)) return false;
	const double tiles = (double)((g.m + 63) / 64) * (double)((g.n + 63) / 64) * (double)g.batch_count;
	return tiles >= 176;
}

namespace {

// Where the ring wins over the tile kernels.
bool ring_fits(const GemmCall& g) {
	if (ring_takes_large(g)) return ring_grid_ok(g);
	// Smaller products, where the 32 x 32 tile's chains are the time. A^T B (a weight gradient) is faster here at every
	// size: 512 x 512 x 8192 67 -> 52 us, 1024 x 512 x 4096 66 -> 46, 512 x 784 x 256 7.7 -> 5.9 (chain kernel), 256 x 256 x
	// 300 7.0 -> 5.4 (VALU kernel). The other layouts where the tile kernel would check bounds (200 x 2000 x 1000 23 -> 17,
	// 300 x 1000 x 512 NT 13.5 -> 10.4), and A B with a tile a CU at most (64 x 4096 x 4096 33.8 -> 32.4, 256 x 784 x 512 9.6 ->
	// 7.1); whole aligned A B^T tiles stay where they are (512^3 7.3 us against 8.0, 64 x 4096 x 4096 33.6 against 38).
	if (!ring_ok(g) || g.k < 128 || narrow(g)) return false;
	const double tiles = (double)((g.m + 31) / 32) * (double)((g.n + 31) / 32) * (double)g.batch_count;
	// few outputs with row sums have no other pipelined kernel (the backward of a 256 -> 10 layer at 256 rows, its dX 4 us of
	// it: 13.2 us with dW on the tile kernel, 11.1 here)
	if (tiles < 64) return g.rowsum != nullptr;
	if (g.ta && !g.tb) return ring_grid_ok(g);
	const bool whole = ring_vec(g) && g.m % 32 == 0 && g.n % 32 == 0 && g.k % 64 == 0 && g.ldc % 4 == 0 && aligned16(g.c);
	return (!whole || (!g.ta && !g.tb && tiles <= 256)) && ring_grid_ok(g);
}

}  // namespace

bool ring_takes(const GemmCall& g) {
	if (!ring_fits(g)) return false;
	if (g.rowsum) return true;  // the kernels below have none
	// Where another kernel than the tiles takes the product, or most of a 32 x 32 tile is padding, as products of a few rows
	// or columns and batches of small ones have it. Two 32 x 32 workgroups share a CU, so past 512 of them a product takes
	// another round, while the chain kernel needs no LDS and the VALU kernel's blocks are 16 x 16; a depth that leaves the
	// chain kernel a remainder, or single floats to load, favours the ring. The lines are fitted to 29000 products of 1 to 8192
	// rows and columns, 96 to 4096 deep, up to 1024 of them; each with examples, the other kernel's us against the ring's.
	const double m = (double)g.m, n = (double)g.n, batch = (double)g.batch_count;
	const double tiles = (double)((g.m + 31) / 32) * (double)((g.n + 31) / 32) * batch;
	const double blocks = (double)((g.m + 15) / 16) * (double)((g.n + 15) / 16) * batch;  // of the VALU kernel
	const double padded = tiles * 1024 / (m * n * batch);
	const bool vec = ring_vec(g), one_round = tiles <= 512;
	if (chain4_takes(g)) {
		// A^T B: 512 x 784 x 256 8.1, 6.2; 512 x 2048 x 200 11.0, 9.5; 354 x 1744 x 208 8.3, 10.0
		if (g.ta && !g.tb)
			return (g.k >= 248 && (one_round || tiles > 768)) || (vec && g.k >= 172 && tiles > 768) ||
			       (g.k > 100 && one_round && blocks <= 1024 && batch > 1);
		if (g.ta) return one_round && g.n > 15 && (vec || g.k < 128);
		// A B^T: 64 x 1500 x 128 5.1, 4.6; 200 of 1 x 128 x 128 7.6, 9.0; 111 of 64 x 126 x 103 17.4, 11.3
		if (g.tb) return vec ? padded <= 2 && (one_round || (g.m > 32 && g.n > 32)) : (g.k > 112 || padded <= 4) && (g.m > 16 || g.n > 16);
		// A B: 64 x 1500 x 128 4.6, 4.4; 4 of 2 x 4032 x 112 4.8, 5.5; 11 of 5 x 5553 x 112 12.9, 20.2
		return one_round && g.m > 20 && (vec || (g.k > 112 && g.k < 128));
	}
	if (!g.ta && valu_takes(g)) {
		// A B^T, 16-byte loads: 256 x 512 x 784 10.6, 11.4; 16 x 2930 x 456 7.1, 9.1; 20 x 5352 x 640 10.8, 9.0
		if (g.tb && vec) return 2.9 * tiles <= blocks && blocks > 512;
		// one float a lane: 215 of 2 x 168 x 2693 129, 169; 768 x 132 x 3670 39, 32
		if (g.tb) return (g.k > 480 && 2.9 * tiles <= blocks) || (g.k > 800 && 5 * tiles <= 3 * blocks && tiles >= 160 && one_round);
		// A B: 256 x 512 x 300 7.5, 6.4; 6 x 2976 x 256 4.5, 5.4; 549 of 4 x 2 x 464 9.1, 18.7
		return g.n > 16 && g.k > 272 && (blocks > 256 || g.k > 800);
	}
	// the tile kernels: 260 of 2 x 1269 x 257 A B^T 145, 201; 435 of 2 x 2874 x 107 A B 297, 368; 300 x 1000 x 512 A B^T 13.8,
	// 10.6; 200 x 2000 x 1000 A B 22.7, 16.7
	if (one_round || g.ta) return true;
	if (g.tb) return padded <= 4;
	return (g.m > 16 || g.n > 16) && (g.m > 3 || g.k >= 176);
}

bool ring_takes_gelu(const GemmCall& g) {
	// The other kernel with the epilogue is the chain kernel, at home where 16-byte loads feed it and its few chunks are in
	// flight at once: 768 x 399 x 208 9.1 us against 11.1, 187 x 981 x 228 7.5 against 8.9; 8192 x 2048 x 512 far slower.
	if (!ring_fits(g)) return false;
	const double tiles = (double)((g.m + 31) / 32) * (double)((g.n + 31) / 32);
	return !ring_vec(g) || g.k >= 256 || (tiles <= 512 ? tiles > 256 : (double)g.m * (double)g.n > 1.5e6);
}

namespace {

GemmArgs ring_args(const GemmCall& g, const RingConfig& c) {
	GemmArgs p{};
	p.a = g.a;
	p.b = g.b;
	p.c = g.c;
	p.lda = g.lda;
	p.ldb = g.ldb;
	p.ldc = g.ldc;
	p.m = (int)g.m;
	p.n = (int)g.n;
	p.k = (int)g.k;
	p.accumulate = g.accumulate;
	p.tiles_m = (int)((g.m + c.bm - 1) / c.bm);
	p.tiles_n = (int)((g.n + c.bn - 1) / c.bn);
	p.batch_count = (int)g.batch_count;
	p.batch = g.batch;
	p.ep = g.ep;
	p.pieces = 1;
	p.piece_k = (int)g.k;
	p.rowsum = g.rowsum;
	p.rowsum_combine = g.rowsum_combine;
	bool c_vec = g.ldc % 4 == 0 && aligned16(g.c) && (!g.ep.gelu_y || (aligned16(g.ep.gelu_y) && aligned16(g.ep.gelu_t)));
	for (int d = 0; d < g.batch.ndim; ++d) c_vec = c_vec && g.batch.sc[d] % 4 == 0;
	p.c_vec = c_vec ? 1 : 0;
	return p;
}

}  // namespace

hipError_t gemm_ring_launch(const GemmCall& g, hipStream_t s, int config) {
	if (!ring_ok(g)) return hipErrorInvalidValue;
	hipError_t e = prepare_ring();
	if (e != hipSuccess) return e;
	const RingConfig& c = ring_configs()[config >= 0 ? config : ring_pick(g)];
	const GemmArgs p = ring_args(g, c);
	const int64_t blocks = (int64_t)p.tiles_m * p.tiles_n * p.batch_count;
	if (blocks * c.threads > 0xffffffff) return hipErrorInvalidConfiguration;
	if (g.ep.gelu_y && (g.ta || !g.tb || g.rowsum)) return hipErrorInvalidValue;
	const int v = ring_vec(g) ? 1 : 0;
	const auto fn = g.ep.gelu_y ? c.gelu_fn[v] : g.rowsum ? c.rowsum_fn[v] : c.fn[(g.ta ? 2 : 0) + (g.tb ? 1 : 0)][v];
	hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3((unsigned)c.threads), (size_t)c.lds_bytes, s, p);
	return hipGetLastError();
}

bool ring_pair_takes(const GemmCall& g0, const GemmCall& g1) {
	// A product's dX (or dA) and dW (or dB), each with fewer 64 x 64 tiles than the chip takes: on 32 x 32 tiles side by
	// side, one's workgroups fill the CUs that the other leaves idle. Backward passes over M rows of a K -> N layer (us, two
	// launches or the tile kernel's pair before): matmul 512, 512, 512 14.1 -> 10.6, 256, 512, 256 9.9 -> 6.4, 300, 900, 130 15.4 ->
	// 9.3, 640, 640, 256 13.9 -> 12.9; linear with its bias 512, 512, 512 18.6 -> 13.6, 256, 784, 512 13.4 -> 11.3, 200, 300, 500
	// 11.6 -> 8.1. Below 64 tiles of a product or 128 deep the chain kernels' pairs and the tile pair stay.
	if (g0.ta || !g1.ta || g1.tb || !ring_ok(g0) || !ring_ok(g1) || g0.rowsum || g0.ep.gelu_y || g1.ep.gelu_y) return false;
	if (g0.tb && g1.rowsum) return false;  // not compiled: a linear layer's dX is an A B
	if (g0.batch_count != 1 || g1.batch_count != 1 || g0.batch.ndim != 0 || g1.batch.ndim != 0) return false;
	if (g0.k < 128 || g1.k < 128 || ring_takes_large(g0) || ring_takes_large(g1)) return false;
	auto tiles = [](const GemmCall& g) { return (double)((g.m + 31) / 32) * (double)((g.n + 31) / 32); };
	// A narrow dX (2^22 outputs and more, but fewer than 128 columns) counts as small here: beside a weight gradient of few
	// tiles and a long depth it pays to start both at once (33056, 127, 520 580 -> 307). With row sums its deep aligned form is
	// better off on its 128 x 64 tiles (48384, 96, 1216 645 us against 745, 40000, 120, 1000 541 against 633).
	if (narrow(g0) && g1.rowsum && ring_vec(g0) && g0.k >= 1000) return false;
	return tiles(g0) >= 64 && tiles(g1) >= 64 && tiles(g0) + tiles(g1) < 16777216.0;  // 2^32 work-items
}

hipError_t gemm_ring_pair_launch(const GemmCall& g0, const GemmCall& g1, hipStream_t s) {
	if (!ring_pair_takes(g0, g1)) return hipErrorInvalidValue;
	hipError_t e = prepare_ring();
	if (e != hipSuccess) return e;
	const RingConfig& c = ring_configs()[kRing32x32];
	const GemmArgs p0 = ring_args(g0, c), p1 = ring_args(g1, c);
	const int b0 = p0.tiles_m * p0.tiles_n, b1 = p1.tiles_m * p1.tiles_n;
	const auto fn = ring_pair_32x32(g0.tb ? 2 : g1.rowsum ? 1 : 0, ring_vec(g0) ? 1 : 0, ring_vec(g1) ? 1 : 0);
	hipLaunchKernelGGL(fn, dim3((unsigned)(b0 + b1)), dim3((unsigned)c.threads), (size_t)c.lds_bytes, s, p0, p1, b0);
	return hipGetLastError();
}

const char* ring_config_name(int config) { return ring_configs()[config].name; }

}  // namespace nnh
