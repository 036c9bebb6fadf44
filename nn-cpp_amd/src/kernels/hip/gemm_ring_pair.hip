// The ring kernel's pair launches on 32 x 32 tiles (the tile shape of gemm_ring_32x32.hip).
#include "gemm_ring.hpp"

namespace nnh {

RingPairFn ring_pair_32x32(int kind, int v0, int v1) {
#define NNH_PAIR(TB0, V0, V1, EXTRA1) sgemm_ring_pair_kernel<32, 32, 64, 16, 16, 5, 2, TB0, V0, V1, EXTRA1>
	static const RingPairFn fns[3][2][2] = {
	    {{NNH_PAIR(false, 1, 1, kRingPlain), NNH_PAIR(false, 1, 4, kRingPlain)},
	     {NNH_PAIR(false, 4, 1, kRingPlain), NNH_PAIR(false, 4, 4, kRingPlain)}},
	    {{NNH_PAIR(false, 1, 1, kRingRowSums), NNH_PAIR(false, 1, 4, kRingRowSums)},
	     {NNH_PAIR(false, 4, 1, kRingRowSums), NNH_PAIR(false, 4, 4, kRingRowSums)}},
	    {{NNH_PAIR(true, 1, 1, kRingPlain), NNH_PAIR(true, 1, 4, kRingPlain)},
	     {NNH_PAIR(true, 4, 1, kRingPlain), NNH_PAIR(true, 4, 4, kRingPlain)}}};
#undef NNH_PAIR
	return fns[kind][v0][v1];
}

}  // namespace nnh
