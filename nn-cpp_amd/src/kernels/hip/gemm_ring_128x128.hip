// Ring kernel 128x128 (workgroup 128 x 128, 8 waves of 64 x 32, 4 stages of 32).
#include "gemm_ring.hpp"

namespace nnh {
RingConfig ring_config_128x128() { return make_ring_config<128, 128, 32, 64, 32, 4, 2>("ring 128x128"); }
}  // namespace nnh
