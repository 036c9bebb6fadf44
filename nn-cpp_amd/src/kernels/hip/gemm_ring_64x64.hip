// Ring kernel 64x64 (workgroup 64 x 64, 4 waves of 32 x 32, 5 stages of 32: two workgroups fill a CU's LDS).
#include "gemm_ring.hpp"

namespace nnh {
RingConfig ring_config_64x64() { return make_ring_config<64, 64, 32, 32, 32, 5, 2>("ring 64x64"); }
}  // namespace nnh
