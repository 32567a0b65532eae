/*
 * buffer_loads.hpp — loads through buffer descriptors, straight into registers: an address is a lane's offset and the wavefront's, and a
 * lane without an operand is given an offset beyond the buffer instead of a branch.
 */
#ifndef CATTLE_HIP_BUFFER_LOADS_HPP_
#define CATTLE_HIP_BUFFER_LOADS_HPP_

#include <hip/hip_runtime.h>

namespace cattle_hip {
namespace buffer_loads {

/* A byte offset beyond any buffer (below 2 GiB): such a load returns zero. Loads are to be in range by the lane's own choice between its
 * offset and this one; none counts on the range check for a sum of its two offsets, and the wavefront's alone lies inside the buffer. */
constexpr unsigned OUTSIDE = 0x80000000u;
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, unsigned bytes) {
	return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int) bytes, 0x00020000);
}
__device__ __forceinline__ float load_1(__amdgpu_buffer_rsrc_t b, unsigned lane_off, unsigned wave_off) {
	return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, (int) lane_off, (int) wave_off, 0));
}
__device__ __forceinline__ f32x2 load_2(__amdgpu_buffer_rsrc_t b, unsigned lane_off, unsigned wave_off) {
	return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(b, (int) lane_off, (int) wave_off, 0));
}
__device__ __forceinline__ f32x4 load_4(__amdgpu_buffer_rsrc_t b, unsigned lane_off, unsigned wave_off) {
	return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(b, (int) lane_off, (int) wave_off, 0));
}

/* Operands of 32 samples a row that turn in LDS: where 16-byte unit c (four samples) of row r lies, shifted by the row, so that the eight
 * rows that a read of 64 lanes takes at a time lie on different banks. */
constexpr int UNITS = 8;
__device__ __forceinline__ int unit_of(int r, int c) {
	return r * UNITS + (c ^ (r % UNITS));
}

} /* namespace buffer_loads */
} /* namespace cattle_hip */

#endif /* CATTLE_HIP_BUFFER_LOADS_HPP_ */
