// Device helpers for subset tests on the matrix cores.  Internal to the match
// kernels.
//
// f is a subset of q exactly when f and ~q share no bit, that is when the
// dot product of their bits is zero.  The bits of a 32-bit word spread over
// 32 4-bit floats (E2M1) with a few ANDs and shifts, in any order as long as
// both operands use the same one; so one v_mfma_f32_32x32x64_f8f6f4 tests 64
// bits of 32 filters against 32 queries, and three of them test the pairs
// whole.  A shared bit adds 1 or more, the accumulators start at -0.5 or -1:
// the sign bit is set exactly where the filter is a subset.  Sums are
// multiples of 0.5 up to 4 * 192: exact in FP32.
//
// Lane l = 32 h + n holds words 2 k + h (k = 0, 1, 2) of row or column n of
// an operand, and of a result column n and the rows 8 (i / 4) + 4 h + i % 4.
#pragma once

#include <hip/hip_runtime.h>

namespace tmx {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// 32 bits as 32 E2M1 values: bit b as 0.5, 1, 2, 2 for b mod 4 = 0, 1, 2, 3
// (0x8 would be -0).
__device__ inline v8i spread(uint32_t w) {
	v8i r = {0, 0, 0, 0, 0, 0, 0, 0};
	r[0] = (int)(w & 0x11111111u);
	r[1] = (int)(w & 0x22222222u);
	r[2] = (int)(w & 0x44444444u);
	r[3] = (int)((w >> 1) & 0x44444444u);
	return r;
}
// The other operand's: 2, 1, 2, 2, so that no product is below 1.
__device__ inline v8i spread_up(uint32_t w) {
	v8i r = spread(w);
	r[0] = (int)((w << 2) & 0x44444444u);
	return r;
}

// What a pair's accumulators start from: two values, since a constant of one
// use stays in the instruction, and one of more takes 16 moves each time.
__device__ inline v16f start_lo() { return (v16f)(-0.5f); }
__device__ inline v16f start_hi() { return (v16f)(-1.0f); }

__device__ inline v16f mfma(const v8i & a, const v8i & b, const v16f & c) {
	return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 4, 4, 0, 0, 0, 0);
}

// Bit r set where register r of lo (r < 16) or r - 16 of hi is negative: one
// instruction a register (zero tests of packed halves took 1.5, compares and
// carries 2 and wait states).
__device__ inline uint32_t subset_mask(const v16f & lo, const v16f & hi) {
	uint32_t m = 0;
#pragma unroll
	for (int i = 15; i >= 0; --i) m = __builtin_amdgcn_alignbit(m, __float_as_uint(hi[i]), 31);
#pragma unroll
	for (int i = 15; i >= 0; --i) m = __builtin_amdgcn_alignbit(m, __float_as_uint(lo[i]), 31);
	return m;
}

// Wave-level ordering of LDS traffic between lanes.
__device__ inline void wave_fence() {
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline uint32_t uniform(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

// Inclusive prefix sum over the wave's lanes.
__device__ inline uint32_t wave_prefix(uint32_t x) {
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);   // row_shr:1
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);   // row_bcast:15
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);   // row_bcast:31
	return x;
}

// A mask of 64 rows (lo's, then hi's) in subset_mask's order, for half h.
__device__ inline uint32_t half_mask(uint64_t lm, uint32_t h) {
	if (lm == ~0ULL) return ~0u;
	uint64_t x = (lm >> (4 * h)) & 0x0F0F0F0F0F0F0F0FULL;
	x = (x | (x >> 4)) & 0x00FF00FF00FF00FFULL;
	x = (x | (x >> 8)) & 0x0000FFFF0000FFFFULL;
	return (uint32_t)x | (uint32_t)(x >> 16);
}

} // namespace tmx
