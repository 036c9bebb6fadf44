// Ring kernel 32x32 (workgroup 32 x 32, 4 waves of one 16 x 16 block each, 5 stages of 64: two workgroups a CU).
#include "gemm_ring.hpp"

namespace nnh {
RingConfig ring_config_32x32() { return make_ring_config<32, 32, 64, 16, 16, 5, 2>("ring 32x32"); }
}  // namespace nnh
