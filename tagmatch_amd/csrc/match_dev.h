// Device helpers shared by the match kernels.  Internal to
// libtagmatch_amd.so.
#pragma once

#include "fib.h"

namespace tmx {

__device__ inline uint32_t mbcnt64(uint64_t m) {
	return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// The overflow list a slot points to, bounded by the table's overflow words:
// whatever a slot holds, nothing outside the table is read (n = 0 then).
__device__ inline uint32_t ovf_list(uint64_t kv, const uint32_t * __restrict__ ovf, uint32_t ovf_n, uint32_t & off) {
	off = (uint32_t)(kv >> 16);
	if (off >= ovf_n) return 0;
	const uint32_t n = ovf[off];
	return n < ovf_n - off ? n : 0;
}

// Number of keys in a slot (inline ids or an overflow list).
__device__ inline uint32_t key_count(uint64_t kv, const uint32_t * __restrict__ ovf, uint32_t ovf_n) {
	uint32_t off;
	if ((kv & 0xFFFFu) == KEY_NONE) return ovf_list(kv, ovf, ovf_n, off);
	uint32_t n = 0;
	for (int x = 0; x < 4; ++x) n += ((kv >> (16 * x)) & 0xFFFFu) != KEY_NONE;
	return n;
}

// Uniform loads through the constant address space compile to scalar
// loads (s_load) into SGPRs; used for data that no thread writes during the
// kernel (FIB block info, partition info, inverted query words).
typedef const __attribute__((address_space(4))) uint32_t cu32_t;

__device__ inline uint4 sld4(const uint32_t * p) {
	cu32_t * c = (cu32_t *)(p);
	return make_uint4(c[0], c[1], c[2], c[3]);
}
__device__ inline uint2 sld2(const uint32_t * p) {
	cu32_t * c = (cu32_t *)(p);
	return make_uint2(c[0], c[1]);
}
__device__ inline uint32_t sld1(const uint32_t * p) { return *(cu32_t *)(p); }

// Four words, not aligned: rows begin at any word.
typedef uint32_t quad __attribute__((ext_vector_type(4), aligned(4)));

// Words w .. w + 3 of a row of kw words.
__device__ inline void store_words(uint32_t * row, uint32_t w, uint32_t kw, const quad & v) {
	if (w + 4 <= kw) {
		*reinterpret_cast<quad *>(row + w) = v;
		return;
	}
#pragma unroll
	for (uint32_t k = 0; k < 4; ++k)
		if (w + k < kw) row[w + k] = v[k];
}
__device__ inline quad load_words(const uint32_t * row, uint32_t w, uint32_t kw) {
	if (w + 4 <= kw) return *reinterpret_cast<const quad *>(row + w);
	quad v = {0, 0, 0, 0};
#pragma unroll
	for (uint32_t k = 0; k < 4; ++k)
		if (w + k < kw) v[k] = row[w + k];
	return v;
}
} // namespace tmx
