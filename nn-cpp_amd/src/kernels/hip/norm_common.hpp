// norm_common.hpp - what the batch and layer norm kernels share: the ordered sum over LDS and the launches' limits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nnh {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Workgroups of 256 threads in one launch: HIP takes fewer than 2^32 work-items a dimension.
constexpr int64_t kMaxGrid = ((int64_t)1 << 24) - 1;

inline bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

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

}  // namespace nnh
