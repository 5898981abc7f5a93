// The launch interface of the kernel that runs before the match of a step.
// Internal to libtagmatch_amd.so.
#pragma once

#include "fib.h"

namespace tmx {

struct front_args {
	const uint32_t * __restrict__ q;            // words of each query, 8 apart
	uint32_t nq;
	uint32_t chunk;                             // queries per workgroup (front_launch sets it)
	const uint32_t * __restrict__ part_info;    // partition masks
	uint32_t P;
	uint32_t * pcount;                          // adds the queries of each partition (NULL: no count)
	const uint32_t * __restrict__ rich_words;   // rich filters, those that hold every key first
	const uint32_t * __restrict__ rich_bm;      // their key bitmaps
	uint32_t n_rich, n_full;                    // their number (0: counts only)
	uint32_t kw, last_mask;                     // words of a key row, valid bits of the last
	uint32_t * gbm;                             // key rows
	uint32_t * qfull;                           // 2 where a row holds every key, else 0
	uint32_t * active;                          // the other queries, in any order (NULL: not listed),
	uint32_t * qact;                            // their words
	uint32_t * n_active;                        // and their number, zero at the start
};

void front_launch(front_args a, hipStream_t s);

} // namespace tmx
