// Ring kernel 64x64_deep (workgroup 64 x 64, 4 waves of 32 x 32, 3 stages of 64: one workgroup a CU, half the barriers).
#include "gemm_ring.hpp"

namespace nnh {
RingConfig ring_config_64x64_deep() { return make_ring_config<64, 64, 64, 32, 32, 3, 1>("ring 64x64_deep"); }
}  // namespace nnh
