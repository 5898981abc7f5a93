// The matrix-core match kernel's launch interface.  Internal to
// libtagmatch_amd.so.
#pragma once

#include "fib.h"

namespace tmx {

// What a launch does with its hits:
//   MX_KEYS      their keys into rows in HBM (which hold most keys already);
//   MX_KEYS_LDS  the same through rows in local memory (rows that start empty);
//   MX_COUNT, MX_COUNT_KEYS   values per query and segment (filter ids; keys);
//   MX_WRITE, MX_WRITE_KEYS   the values, behind those of earlier segments.
enum mx_mode { MX_KEYS, MX_KEYS_LDS, MX_COUNT, MX_COUNT_KEYS, MX_WRITE, MX_WRITE_KEYS, MX_MODES };

constexpr uint32_t MX_LDS_KW = 64;      // MX_KEYS_LDS: words of a row with the most queries per item
constexpr uint32_t MX_ROW_WORDS = 192 * MX_LDS_KW;   // MX_KEYS_LDS: words of an item's rows, at most
constexpr uint32_t MX_QUEUES = 8;       // work queues, one per XCD
constexpr uint32_t MX_QPAD = 32;        // queue cursors 256 B apart
constexpr uint32_t MX_MAX_SEG = 16384;  // blocks per work item, at most
constexpr uint32_t MX_MAX_GROUPS = 2048;   // workgroups of a launch, at most
constexpr uint32_t MX_LONG_LIST = 64;  // MX_WRITE_KEYS: keys of a list that is written apart, at least
constexpr uint32_t MX_VISITS = 1024;    // blocks of a pass, at most

constexpr int MX_WAVES = 8;             // waves per workgroup

// Queries per work item, at most, and the words of the candidate masks (an
// odd number of words per block, two for 64 queries and one).  Two
// workgroups of 8 waves share a CU's 160 KB of local memory; within that,
// more queries per item mean more candidates for each block whose filters
// are loaded and spread.  Rows in local memory (48 KB for 192 queries at
// 2048 keys) leave room for fewer: match times of the uneven units (541k
// queries) 3.06 ms with 192, 3.73 with 128; with 448 and one workgroup of 16
// waves per CU 4 % more than with 192.
__host__ __device__ constexpr uint32_t mx_super(int mode) {
	return mode == MX_KEYS ? 2048u : mode == MX_KEYS_LDS ? 192u : 1536u;
}
// The same for rows of kw words: wider ones leave room for fewer (128 KB of
// rows and one workgroup per CU took longer at every width up to 1024 words
// but 256: 4096 keys 552 and 691 us, 16384 keys 1067 and 1593).
__host__ __device__ inline uint32_t mx_super_of(int mode, uint32_t kw) {
	const uint32_t most = mx_super(mode);
	return mode != MX_KEYS_LDS || kw * most <= MX_ROW_WORDS ? most : MX_ROW_WORDS / kw;
}
__host__ __device__ constexpr uint32_t mx_mask_words(int mode) {
	return mode == MX_KEYS ? 64u * 65u : mode == MX_KEYS_LDS ? 128u * 7u : 64u * 49u;
}
__host__ __device__ constexpr uint32_t mx_visits(int mode) { return mode == MX_KEYS_LDS ? 128u : MX_VISITS; }

// Work items of a launch over nq queries and nblk blocks: item = segment *
// nsuper + super, supers of sq queries, segments of about seg blocks: every
// nseg-th tile of 32, so that the blocks with many matches, which lie
// together, are spread over all segments (against runs of blocks: 100k
// queries on 1M filters 0.63 and 0.74 ms, the uneven units 3.52 and 3.95).
// Work for at most five items of 64 blocks per workgroup: one item each (10M
// filters: 1000 queries 31 us against 52, 10k 75 against 85; 1M filters, 16
// queries 13 against 17 for two rounds).  One super: as many items of up to
// 512 blocks (43.6M filters: 1000 queries 39 us, 83 with 128 blocks, 16k 99
// and 135).  Otherwise 128 blocks: between 64
// and 256 it is the fastest or within 4 % of it (1M filters, 300k queries,
// for 64, 128, 256: 1.58, 1.52, 1.65 ms; 10M, 1M queries: 1.00, 0.98, 1.00;
// 65k without the full-row exit: 11.7, 11.4, 11.4); up to 512 for wide rows
// in local memory, cleared and merged for each item, at four items per
// workgroup (4096 keys, no long list, 1M filters, 20k queries: 2.37 ms with
// 128, 1.98 with 512; 4M, 5k: 2.06, 1.72).  seg_min: least blocks
// per segment (a bound on the segments), 0: none.
struct mx_shape {
	uint32_t sq, nsuper, seg, nseg;
};
__host__ __device__ inline mx_shape mx_shape_of(int mode, uint32_t kw, uint32_t nq, uint32_t nblk, uint32_t resident,
												uint32_t seg_fixed, uint32_t seg_min) {
	uint32_t sq = mx_super_of(mode, kw);
	if (nq < sq) {
		const uint32_t some = nq > 64 ? (nq + 63) & ~63u : 64u;
		if (some < sq) sq = some;
	}
	// few blocks: fewer queries per item (20k queries, 8.8k blocks: 0.70
	// instead of 1.30 ms; KEYS_ALL, 1000 queries on 20 blocks: 77 instead of
	// 129 us)
	while (sq > 256 && (uint64_t)((nq + sq - 1) / sq) * ((nblk + 63) / 64) < 4ull * resident) sq = (sq / 2 + 63) & ~63u;
	while (sq > 64 && 4ull * ((nq + sq - 1) / sq) * ((nblk + 31) / 32) < resident) sq = (sq / 2 + 63) & ~63u;
	const uint32_t nsuper = (nq + sq - 1) / sq;
	uint32_t seg = 128;
	if (nsuper == 1 || (uint64_t)nsuper * ((nblk + 63) / 64) <= 5ull * resident) {
		const uint64_t per = ((uint64_t)nblk * nsuper + resident - 1) / resident;   // blocks of a workgroup
		const uint64_t rounds = (per + 511) / 512;
		seg = per == 0 ? 32u : (uint32_t)((per + rounds - 1) / rounds + 31) & ~31u;
	} else if (mode == MX_KEYS_LDS && kw > MX_LDS_KW) {
		const uint64_t per = (uint64_t)nblk * nsuper / (4ull * resident);
		seg = per < 128 ? 128u : per > 512 ? 512u : (uint32_t)per & ~31u;
	}
	// a configured size holds where it leaves an item for each workgroup (50k
	// queries, 4.4k blocks in segments of 4096: 4.28 ms otherwise, 1.25 so)
	if (seg_fixed && (seg_fixed < seg || (uint64_t)nsuper * ((nblk + seg_fixed - 1) / seg_fixed) >= resident)) seg = seg_fixed;
	if (seg < seg_min) seg = seg_min;
	if (seg > MX_MAX_SEG) seg = MX_MAX_SEG;
	const uint32_t tiles = (nblk + 31) / 32, per = (seg + 31) / 32;
	mx_shape h;
	h.sq = sq;
	h.nsuper = nsuper;
	h.seg = seg;
	h.nseg = (tiles + per - 1) / per;
	return h;
}

struct mx_args {
	dev_fib_view f;
	const uint32_t * __restrict__ q;       // words of each local query, 8 apart
	const uint32_t * __restrict__ qmap;    // query (result row) of each local query (NULL: identity)
	uint32_t nq;                           // local queries
	const uint32_t * __restrict__ nq_dev;  // device count of local queries (NULL: nq)
	uint32_t nblk;                         // blocks of the table
	uint32_t seg_fixed;                    // configured blocks per item (0: by the launch's size)
	uint32_t seg_min;                      // least blocks per item (0: any)
	uint32_t resident;                     // workgroups of the launch
	const uint32_t * __restrict__ units;   // explicit units, 8 words each: partition, first query,
	                                       // queries, supers, segments, blocks per segment, first
	                                       // block, end block
	const uint32_t * __restrict__ uprefix; // n_units + 1: first work item of each unit
	uint32_t n_units;
	uint32_t unit_sq;                      // queries of a unit's items, at most mx_super_of()
	unsigned long long * qnext;            // MX_QUEUES cursors, MX_QPAD apart, zero at the start
	uint32_t * gbm;                        // key rows
	const uint32_t * __restrict__ qfull;   // flags of rows that hold every key (NULL: none known)
	const uint32_t * __restrict__ rich_bm; // key bitmaps of the rich filters
	uint32_t n_rich;
	uint32_t rich_done;                    // the rows already hold the rich filters' keys
	uint32_t * hcnt;                       // MX_COUNT..: values of each query, one row of nq per segment;
	                                       // MX_WRITE..: values of earlier segments
	const uint64_t * __restrict__ off;     // MX_WRITE..: first value of each query
	uint32_t * vals;
	uint64_t vcap;
	uint4 * lists;                         // MX_WRITE_KEYS: long key lists to write (first value, 64
	                                       // bits; list; keys), lists_cap of them at most
	uint64_t lists_cap;
	unsigned long long * n_lists;          // their number, zero at the start
	uint64_t * wg_stats;                   // per workgroup: hits, block visits, subset tests, tests
	                                       // with hits
	uint64_t * n_items;                    // receives the launch's work items
	const uint32_t * __restrict__ slot_epoch;
	uint32_t epoch;
	const uint32_t * __restrict__ step_vals;   // replayed steps: [0] epoch, [1] valid overflow words
};

// hcnt's rows (segments) to each query's values of earlier segments, and the
// queries' totals.
void mx_prefix(uint32_t * hcnt, uint32_t rows, uint32_t nq, uint32_t * total, hipStream_t s);

// MX_WRITE_KEYS: the lists it recorded.
void mx_write_lists(const mx_args & a, hipStream_t s);

// Workgroups that fit the GPU at once.
uint32_t mx_resident(int mode);
void mx_launch(const mx_args & a, int mode, uint32_t grid, hipStream_t s);

} // namespace tmx
