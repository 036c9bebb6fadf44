// Ring kernel 256x128 (workgroup 256 x 128, 8 waves of 64 x 64, 3 stages of 32).
#include "gemm_ring.hpp"

namespace nnh {
RingConfig ring_config_256x128() { return make_ring_config<256, 128, 32, 64, 64, 3, 2>("ring 256x128"); }
}  // namespace nnh
