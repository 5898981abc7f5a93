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
// Of 64 rows in two tiles, row_of says which each lane holds, so that bit b
// of a lane's subset_mask is row 32 h + b; or, for rows in memory, near_row,
// which keeps each tile to 32 rows that lie together, and near_bit.
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

// The signs of both accumulators, one bit each.  A conversion to 6-bit floats
// takes all 32 at once and leaves their signs 6 bits apart: those of words 0
// to 2 at different odd bits, those of words 3 to 5 at the same ones.  88
// cycles of the vector unit; a funnel shift per register took 128, zero
// tests of packed halves 192.
typedef uint32_t v6u __attribute__((ext_vector_type(6)));
__device__ inline uint32_t subset_mask(const v16f & lo, const v16f & hi) {
	constexpr uint32_t A = 0x20820820u, B = 0x08208208u, ODD = 0xAAAAAAAAu;
	const v6u r = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(lo, hi, 1.0f);
	const uint32_t x = (A & r[0]) | (~A & ((B & r[1]) | (~B & r[2])));
	const uint32_t y = (A & r[3]) | (~A & ((B & r[4]) | (~B & r[5])));
	return (ODD & x) | (~ODD & (y >> 1));
}
// Its bit of register i of lo (mt = 0) or hi (1): the conversion alternates
// between them.
__host__ __device__ constexpr uint32_t mask_bit(uint32_t mt, uint32_t i) {
	return (6 * ((2 * i + mt) % 16) + 5) % 32 - (2 * i + mt) / 16;
}
// The row, of 64, that lane n holds of tile mt.
__device__ inline uint32_t row_of(uint32_t mt, uint32_t n) {
	return 32 * (n / 4 % 2) + mask_bit(mt, n / 8 * 4 + n % 4);
}

// Bit 1 of a mask's bit tells the tile; the row that bit b of half h is then,
// and the one that lane n holds of tile mt.  (Tiles of rows that alternate
// between two lines of memory cost a step of 1000 queries 36 us instead of
// 26.)
__host__ __device__ constexpr uint32_t near_bit(uint32_t b, uint32_t h) {
	return (b & 2) * 16 + h * 16 + b / 4 * 2 + (b & 1);
}
__device__ inline uint32_t near_row(uint32_t mt, uint32_t n) {
	return near_bit(mask_bit(mt, n / 8 * 4 + n % 4), n / 4 % 2);
}
// A mask of 64 such rows as half h has them.
__device__ inline uint32_t near_mask(uint64_t lm, uint32_t h) {
	if (lm == ~0ULL) return ~0u;
	uint32_t m[2];
#pragma unroll
	for (uint32_t mt = 0; mt < 2; ++mt) {   // 16 bits as eight pairs, four bits apart
		uint32_t x = (uint32_t)(lm >> (32 * mt + 16 * h)) & 0xFFFFu;
		x = (x | (x << 8)) & 0x00FF00FFu;
		x = (x | (x << 4)) & 0x0F0F0F0Fu;
		m[mt] = (x | (x << 2)) & 0x33333333u;
	}
	return m[0] | (m[1] << 2);
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

} // namespace tmx
