// GPU balanced partitioning of a filter table.
//
// Restates the reference's recursive balanced partitioning
// (reference partitioning.cc:230-411) level-synchronously: every pending
// candidate ("segment") of the current level is processed at once.
//
//   * A BALANCE segment (size > maxp) is split on the bit whose frequency is
//     nearest half its size, searching from its first unused pivot bit
//     (balancing_pivot, partitioning.cc:262-278).  The 0-side keeps the
//     segment's pivot mask, the 1-side adds the pivot (:307-312).  A child
//     larger than maxp stays BALANCE; a smaller child is finished if its
//     pivot mask is non-empty, else it goes to NONZERO (:314-357).
//   * A NONZERO segment is split on its most frequent bit until all its
//     filters share a bit (nonzero_mask_partitioning, :251-271): the 1-side
//     is finished, the 0-side continues.  A segment of all-zero filters is
//     finished with an empty mask (the reference does not terminate there).
//   * Splits are stable: zeros first, then ones, each in input order
//     (std::stable_partition, :165).
//
// Because every decision depends only on the members of a segment, this
// produces the same partitions (as sets, with the same member order) as the
// reference's thread pool, whatever order the reference finishes them in.
//
// Per BALANCE level: a bit histogram per segment, one device-to-host copy of
// the histograms, the pivot decisions on the host (a few hundred segments at
// most), per-tile split offsets, and a stable scatter (ballot + mbcnt) of all
// positions into the other buffer.
//
// A NONZERO segment needs up to 192 splits in a row, each on what the last
// one left: one workgroup makes them all without the host (k_nonzero), on
// lists of positions instead of the records.  Segments of more filters than
// NZ_MAX, or of more set bits than NZ_BITS, are split level by level until
// they fit.
#include "hip_util.h"

#include <algorithm>
#include <cstring>
#include <vector>

using namespace tmx;

namespace {

constexpr uint32_t TILE = 1024;
// A workgroup takes about 0.5 us per 1024 filters left and split: a million
// would keep one CU busy for milliseconds, where the levels use them all.
// Each filter it moves also has its set bits counted out, 0.2 us per 1024:
// segments of more set bits than NZ_BITS are split by the levels, too (whole
// calls on 200k filters with half, an eighth, a fiftieth of their bits set:
// 5.2, 4.7, 11.7 ms without this bound, 1.4, 3.9, 11.6 with 4M, 1.07, 1.9, 8.7
// with 0.5M).
constexpr uint32_t NZ_MAX = 256 * 1024;
constexpr uint64_t NZ_BITS = 500000;
constexpr uint32_t NZ_ROUNDS = 193;   // splits of a NONZERO segment (a pivot bit is gone after its split) + 1
constexpr int NO_PIVOT = -1;

enum seg_mode : uint8_t { BALANCE = 0, NONZERO = 1, DONE = 2 };

struct seg_t {
	uint32_t begin, end;
	uint64_t bits;          // set bits of its filters, at most
	uint32_t used[6];       // pivot bits used on the path (BALANCE only)
	uint8_t mode;
	uint8_t mask_nonempty;  // some 1-side pivot on the path
};

// tile: [begin, end) positions of one segment
struct tile_t {
	uint32_t begin, end, seg, pad;
};

__device__ inline uint32_t mbcnt(uint64_t m) {
	return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Adds `by` (1 or -1) to the counts of a filter's bits.
__device__ inline void count_bits(uint32_t * h, const uint4 & a, const uint2 & c, uint32_t by) {
	const uint32_t w[6] = {a.x, a.y, a.z, a.w, c.x, c.y};
#pragma unroll
	for (int j = 0; j < 6; ++j) {
		uint32_t v = w[j];
		while (v) {
			const uint32_t b = (uint32_t)__builtin_ctz(v);
			v &= v - 1;
			atomicAdd(&h[j * 32 + b], by);
		}
	}
}

// Each filter record: 6 words, input index, pad (32 bytes).
__global__ void __launch_bounds__(256)
k_pack(const uint32_t * __restrict__ w, uint32_t n, uint32_t * __restrict__ rec) {
	uint32_t i = blockIdx.x * 256 + threadIdx.x;
	if (i >= n) return;
	uint32_t * r = rec + (size_t)i * 8;
	for (int j = 0; j < 6; ++j) r[j] = w[(size_t)i * 6 + j];
	r[6] = i;
	r[7] = 0;
}

// Bit counts of each tile, and of its segment (tile.pad: the segment's row).
__global__ void __launch_bounds__(256)
k_tile_hist(const uint32_t * __restrict__ rec, const tile_t * __restrict__ tiles,
			uint32_t * __restrict__ tile_hist, uint32_t * __restrict__ freq) {
	__shared__ uint32_t h[192];
	const tile_t t = tiles[blockIdx.x];
	for (uint32_t b = threadIdx.x; b < 192; b += 256) h[b] = 0;
	__syncthreads();
	for (uint32_t i = t.begin + threadIdx.x; i < t.end; i += 256) {
		const uint4 a = *reinterpret_cast<const uint4 *>(rec + (size_t)i * 8);
		const uint2 c = *reinterpret_cast<const uint2 *>(rec + (size_t)i * 8 + 4);
		count_bits(h, a, c, 1u);
	}
	__syncthreads();
	for (uint32_t b = threadIdx.x; b < 192; b += 256) {
		const uint32_t v = h[b];
		tile_hist[(size_t)blockIdx.x * 192 + b] = v;
		if (v) atomicAdd(&freq[(size_t)t.pad * 192 + b], v);
	}
}

// One wave per split segment: zero/one base of each of its tiles, 64 tiles
// at a time.  piv[s] is the pivot of split segment s; its tiles are
// [tb[s], tb[s+1]).  hidx[t] is the histogram row of tile t.
__global__ void __launch_bounds__(64)
k_tile_bases(const uint32_t * __restrict__ tile_hist, const uint32_t * __restrict__ hidx,
			 const tile_t * __restrict__ tiles,
			 const uint32_t * __restrict__ tb, const int32_t * __restrict__ piv,
			 const uint32_t * __restrict__ seg_zeros, uint32_t * __restrict__ zbase,
			 uint32_t * __restrict__ obase) {
	const uint32_t s = blockIdx.x, lane = threadIdx.x;
	const int32_t p = piv[s];
	const uint32_t first = tiles[tb[s]].begin, nz = seg_zeros[s], end = tb[s + 1];
	uint32_t z = 0, o = 0;
	for (uint32_t t0 = tb[s]; t0 < end; t0 += 64) {
		const uint32_t t = t0 + lane;
		uint32_t ones = 0, size = 0;
		if (t < end) {
			ones = tile_hist[(size_t)hidx[t] * 192 + p];
			size = tiles[t].end - tiles[t].begin;
		}
		uint32_t po = ones, ps = size;
		for (int d = 1; d < 64; d <<= 1) {
			const uint32_t yo = __shfl_up(po, d, 64), ys = __shfl_up(ps, d, 64);
			if ((int)lane >= d) {
				po += yo;
				ps += ys;
			}
		}
		if (t < end) {
			zbase[t] = first + z + (ps - size) - (po - ones);
			obase[t] = first + nz + o + po - ones;
		}
		o += __shfl(po, 63, 64);
		z += __shfl(ps, 63, 64) - __shfl(po, 63, 64);
	}
}

// A NONZERO segment: its range, and the row of its bit counts.
struct nz_seg {
	uint32_t begin, end, row, pad;
};

// All splits of a NONZERO segment by one workgroup: the most frequent bit of
// the filters left (first of equal ones) moves the filters that have it to
// the end of the range still open, both sides in their order; until every
// filter left has that bit, or none has any.  ord[begin..end) receives the
// positions in the final order; counts[0] the filters left at the end (the
// segment's first partition), counts[r] those of split r (its partitions
// lie last split first), rounds the splits.  Bound by one CU's latency (a
// gather and a barrier per 4096 filters, three barriers per split): 1.5 ms for
// the 1M-filter table's segment of about 64k filters and 75 splits (2.6 ms
// with 1024 filters at a time), 1.08 for what is left of it after the five that
// the levels make down to NZ_BITS; split level by level over all the records,
// each with its round trips to the host, they took 17 ms.
__global__ void __launch_bounds__(1024)
k_nonzero(const uint32_t * __restrict__ rec, const nz_seg * __restrict__ segs, const uint32_t * __restrict__ freq,
		  uint32_t * __restrict__ list0, uint32_t * __restrict__ list1, uint32_t * __restrict__ ord,
		  uint32_t * __restrict__ counts, uint32_t * __restrict__ rounds) {
	__shared__ uint32_t s_freq[192], s_best[3], s_z[2][64];
	const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const nz_seg g = segs[blockIdx.x];
	uint32_t left = g.end - g.begin, tail = g.end, r = 0;
	uint32_t * cnt = counts + (size_t)blockIdx.x * NZ_ROUNDS;
	if (tid < 192) s_freq[tid] = freq[(size_t)g.row * 192 + tid];
	__syncthreads();
	const uint32_t * cur = nullptr;   // the positions left (NULL: all, in order)
	uint32_t * next = list0;
	for (; r + 1 < NZ_ROUNDS; ++r) {
		if (tid < 192) {
			// counts are below 2^24 (NZ_MAX filters): the first of the largest
			uint32_t k = (s_freq[tid] << 8) | (255u - tid);
			for (int d = 32; d > 0; d >>= 1) k = max(k, (uint32_t)__shfl_xor(k, d, 64));
			if (lane == 0) s_best[wave] = k;
		}
		__syncthreads();
		const uint32_t best = max(max(s_best[0], s_best[1]), s_best[2]);
		const uint32_t mf = best >> 8, p = 255u - (best & 255u);
		if (mf == left || mf == 0) break;
		tail -= mf;
		// 4096 filters at a time, four in flight per thread; a filter's
		// rank among the ones is its rank in the list less the zeros before
		// it, so the zeros of each 64 suffice
		uint32_t zeros = 0;
		for (uint32_t c = 0, par = 0; c < left; c += 4096, par ^= 1) {
			uint32_t at[4], w[4];
			uint64_t zm[4];
#pragma unroll
			for (int k = 0; k < 4; ++k) {
				const uint32_t i = c + k * 1024 + tid;
				at[k] = i < left ? (cur ? cur[g.begin + i] : g.begin + i) : g.begin;
			}
#pragma unroll
			for (int k = 0; k < 4; ++k) w[k] = rec[(size_t)at[k] * 8 + (p >> 5)];
#pragma unroll
			for (int k = 0; k < 4; ++k) {
				zm[k] = __ballot(c + k * 1024 + tid < left && ((w[k] >> (p & 31)) & 1u) == 0);
				if (lane == 0) s_z[par][k * 16 + wave] = (uint32_t)__popcll(zm[k]);
			}
			__syncthreads();   // (the other parity's counts may still be read)
			const uint32_t own = s_z[par][lane];
			uint32_t pre = own;
			for (int d = 1; d < 64; d <<= 1) {
				const uint32_t y = __shfl_up(pre, d, 64);
				if ((int)lane >= d) pre += y;
			}
			const uint32_t all = __shfl(pre, 63, 64);
			pre -= own;
#pragma unroll
			for (int k = 0; k < 4; ++k) {
				const uint32_t i = c + k * 1024 + tid;
				const uint32_t z = zeros + __shfl(pre, k * 16 + (int)wave, 64) + mbcnt(zm[k]);
				if (i >= left) continue;
				if ((zm[k] >> lane) & 1) {
					next[g.begin + z] = at[k];
				} else {
					ord[tail + i - z] = at[k];
					const uint4 a = *reinterpret_cast<const uint4 *>(rec + (size_t)at[k] * 8);
					const uint2 b = *reinterpret_cast<const uint2 *>(rec + (size_t)at[k] * 8 + 4);
					count_bits(s_freq, a, b, ~0u);
				}
			}
			zeros += all;
		}
		left -= mf;
		if (tid == 0) cnt[r + 1] = mf;
		cur = next;
		next = cur == list0 ? list1 : list0;
		__syncthreads();
	}
	for (uint32_t i = tid; i < left; i += 1024) ord[g.begin + i] = cur ? cur[g.begin + i] : g.begin + i;
	if (tid == 0) {
		cnt[0] = left;
		rounds[blockIdx.x] = r;
	}
}

__global__ void __launch_bounds__(256)
k_identity(uint32_t * __restrict__ ord, uint32_t n) {
	const uint32_t i = blockIdx.x * 256 + threadIdx.x;
	if (i < n) ord[i] = i;
}

// Stable split of a tile on its pivot (the tile's whole 1024 records in
// flight, a quarter for each wave), or a plain copy of a longer one.  Moves
// 64 bytes per record: 14 us for 1M records (4.6 TB/s); one wave per tile,
// 64 records at a time, took 75 us.
__global__ void __launch_bounds__(256)
k_scatter(const uint32_t * __restrict__ src, uint32_t * __restrict__ dst,
		  const tile_t * __restrict__ tiles, const int32_t * __restrict__ tile_piv,
		  const uint32_t * __restrict__ zbase, const uint32_t * __restrict__ obase) {
	__shared__ uint32_t s_z[4];
	const tile_t t = tiles[blockIdx.x];
	const int32_t p = tile_piv[blockIdx.x];
	const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
	const uint4 * a = reinterpret_cast<const uint4 *>(src);
	uint4 * d = reinterpret_cast<uint4 *>(dst);
	if (p < 0) {
		for (size_t i = (size_t)t.begin * 2 + tid; i < (size_t)t.end * 2; i += 256) d[i] = a[i];
		return;
	}
	const uint32_t pw = (uint32_t)p >> 5, pb = (uint32_t)p & 31, first = t.begin + wave * 256 + lane;
	uint4 a0[4], a1[4];
	uint64_t zm[4], om[4];
	uint32_t nz = 0;
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		const uint32_t i = first + k * 64;
		a0[k] = a1[k] = make_uint4(0, 0, 0, 0);
		if (i < t.end) {
			a0[k] = a[(size_t)i * 2];
			a1[k] = a[(size_t)i * 2 + 1];
		}
	}
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		const bool valid = first + k * 64 < t.end;
		const uint32_t w = pw == 0 ? a0[k].x : pw == 1 ? a0[k].y : pw == 2 ? a0[k].z : pw == 3 ? a0[k].w
						   : pw == 4 ? a1[k].x : a1[k].y;
		const bool one = (w >> pb) & 1;
		zm[k] = __ballot(valid && !one);
		om[k] = __ballot(valid && one);
		nz += (uint32_t)__popcll(zm[k]);
	}
	if (lane == 0) s_z[wave] = nz;
	__syncthreads();
	uint32_t zpos = zbase[blockIdx.x];
	for (uint32_t w = 0; w < wave; ++w) zpos += s_z[w];
	uint32_t opos = obase[blockIdx.x] + wave * 256 - (zpos - zbase[blockIdx.x]);
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		if (first + k * 64 < t.end) {
			const size_t to = (zm[k] >> lane) & 1 ? zpos + mbcnt(zm[k]) : opos + mbcnt(om[k]);
			d[to * 2] = a0[k];
			d[to * 2 + 1] = a1[k];
		}
		zpos += (uint32_t)__popcll(zm[k]);
		opos += (uint32_t)__popcll(om[k]);
	}
}

// AND of the members of each finished partition; all-ones if empty.
__global__ void __launch_bounds__(1024)
k_part_masks(const uint32_t * __restrict__ rec, const uint32_t * __restrict__ ord, const uint32_t * __restrict__ ranges,
			 uint32_t * __restrict__ masks) {
	__shared__ uint32_t s[16][6];
	const uint32_t p = blockIdx.x, b = ranges[p], e = ranges[p + 1];
	uint32_t m[6] = {~0u, ~0u, ~0u, ~0u, ~0u, ~0u};
	for (uint32_t i = b + threadIdx.x; i < e; i += 1024) {
		const size_t at = (size_t)ord[i] * 8;
		const uint4 x = *reinterpret_cast<const uint4 *>(rec + at);
		const uint2 y = *reinterpret_cast<const uint2 *>(rec + at + 4);
		m[0] &= x.x; m[1] &= x.y; m[2] &= x.z; m[3] &= x.w; m[4] &= y.x; m[5] &= y.y;
	}
	for (int j = 0; j < 6; ++j) {
		for (int d = 32; d > 0; d >>= 1) m[j] &= (uint32_t)__shfl_xor(m[j], d, 64);
		if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6][j] = m[j];
	}
	__syncthreads();
	if (threadIdx.x < 6) {
		uint32_t v = ~0u;
		for (int w = 0; w < 16; ++w) v &= s[w][threadIdx.x];
		masks[(size_t)p * 6 + threadIdx.x] = v;
	}
}

__global__ void __launch_bounds__(256)
k_extract_perm(const uint32_t * __restrict__ rec, const uint32_t * __restrict__ ord, uint32_t n,
			   uint32_t * __restrict__ perm) {
	uint32_t i = blockIdx.x * 256 + threadIdx.x;
	if (i < n) perm[i] = rec[(size_t)ord[i] * 8 + 6];
}

inline bool used_bit(const seg_t & s, int b) { return (s.used[b >> 5] >> (b & 31)) & 1; }

uint32_t dist(uint32_t a, uint32_t b) { return a > b ? a - b : b - a; }

// balancing_pivot (reference partitioning.cc:262-278)
int balancing_pivot(const seg_t & s, const uint32_t * f) {
	const uint32_t size = s.end - s.begin, half = size / 2;
	int pivot = 0;
	while (pivot < 192 && used_bit(s, pivot)) ++pivot;
	if (pivot >= 192) return NO_PIVOT;
	uint32_t min_d = dist(half, f[pivot]);
	for (int b = pivot + 1; b < 192; ++b) {
		uint32_t d = dist(half, f[b]);
		if (d < min_d) {
			pivot = b;
			if (d == 0) break;
			min_d = d;
		}
	}
	return pivot;
}

struct dev_buf {
	void * p = nullptr;
	~dev_buf() { if (p) (void)hipFree(p); }
};

template <typename T>
int ensure(dev_buf & b, size_t & cap, size_t need) {
	if (need <= cap && b.p) return TM_OK;
	if (b.p) (void)hipFree(b.p);
	b.p = nullptr;
	size_t n = std::max<size_t>(need, 1) * 2;
	TM_HIP(hipMalloc(&b.p, n * sizeof(T)));
	cap = n;
	return TM_OK;
}

} // namespace

extern "C" int tm_partition(const uint32_t * words, uint32_t n, uint32_t maxp, uint32_t * perm,
							uint32_t * part_offsets, uint32_t * part_masks, uint32_t max_parts,
							uint32_t * n_parts) {
	if (!n_parts || !part_offsets) return set_error(TM_ERR_INVALID, "NULL output argument");
	if (n && (!words || !perm)) return set_error(TM_ERR_INVALID, "NULL input/perm");
	if (maxp == 0) return set_error(TM_ERR_INVALID, "maxp must be > 0");
	*n_parts = 0;
	part_offsets[0] = 0;
	if (n == 0) return TM_OK;
	TM_CHECK(require_device());

	hipStream_t s;
	TM_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
	struct stream_guard {
		hipStream_t s;
		~stream_guard() { (void)hipStreamDestroy(s); }
	} sg{s};

	dev_buf d_words, d_rec[2], d_in, d_hist, d_freq, d_out, d_ord, d_nz;
	size_t c_in = 0, c_hist = 0, c_freq = 0, c_out = 0, c_nz = 0;
	TM_HIP(hipMalloc(&d_words.p, (size_t)n * 24));
	TM_HIP(hipMalloc(&d_rec[0].p, (size_t)n * 32));
	TM_HIP(hipMalloc(&d_rec[1].p, (size_t)n * 32));
	TM_HIP(hipMalloc(&d_ord.p, (size_t)n * 4));
	TM_HIP(hipMemcpyAsync(d_words.p, words, (size_t)n * 24, hipMemcpyHostToDevice, s));
	hipLaunchKernelGGL(k_pack, dim3((n + 255) / 256), dim3(256), 0, s, (const uint32_t *)d_words.p, n,
					   (uint32_t *)d_rec[0].p);
	int cur = 0;

	std::vector<seg_t> segs(1);
	std::memset(&segs[0], 0, sizeof(seg_t));
	segs[0].begin = 0;
	segs[0].end = n;
	segs[0].mode = n > maxp ? BALANCE : NONZERO;
	segs[0].bits = (uint64_t)n * 192;

	// Host arrays of a level, in one upload each; a buffer is filled again
	// only after the stream was waited for since its upload.
	std::vector<uint32_t> in0, in1, freq, hidx;
	std::vector<tile_t> tiles, all;
	auto push = [](std::vector<uint32_t> & v, const void * p, size_t words) {
		const size_t at = v.size();
		v.resize(at + words);
		if (words) std::memcpy(&v[at], p, words * 4);
		return at;
	};
	// bit counts of the segments `act`, by tiles of theirs
	std::vector<uint32_t> act, tb;
	auto histograms = [&]() -> int {
		tiles.clear();
		tb.assign(1, 0);
		for (uint32_t a = 0; a < act.size(); ++a) {
			const seg_t & g = segs[act[a]];
			for (uint32_t b = g.begin; b < g.end; b += TILE) tiles.push_back(tile_t{b, std::min(g.end, b + TILE), act[a], a});
			tb.push_back((uint32_t)tiles.size());
		}
		const uint32_t nt = (uint32_t)tiles.size(), na = (uint32_t)act.size();
		in0.clear();
		push(in0, tiles.data(), (size_t)nt * 4);
		TM_CHECK(ensure<uint32_t>(d_in, c_in, in0.size()));
		TM_CHECK(ensure<uint32_t>(d_hist, c_hist, (size_t)nt * 192));
		TM_CHECK(ensure<uint32_t>(d_freq, c_freq, (size_t)na * 192));
		TM_HIP(hipMemcpyAsync(d_in.p, in0.data(), in0.size() * 4, hipMemcpyHostToDevice, s));
		fill_u32((uint32_t *)d_freq.p, 0, (uint64_t)na * 192, s);
		if (nt)
			hipLaunchKernelGGL(k_tile_hist, dim3(nt), dim3(256), 0, s, (const uint32_t *)d_rec[cur].p,
							   (const tile_t *)d_in.p, (uint32_t *)d_hist.p, (uint32_t *)d_freq.p);
		TM_HIP(hipGetLastError());
		return TM_OK;
	};

	for (int level = 0;; ++level) {
		// segments to split by this level's kernels
		act.clear();
		for (uint32_t k = 0; k < segs.size(); ++k)
			if (segs[k].mode == BALANCE ||
				(segs[k].mode == NONZERO && (segs[k].end - segs[k].begin > NZ_MAX || segs[k].bits > NZ_BITS)))
				act.push_back(k);
		if (act.empty()) break;
		if (level > 100000) return set_error(TM_ERR_HIP, "partitioner did not converge");
		TM_CHECK(histograms());
		const uint32_t na = (uint32_t)act.size();
		freq.resize((size_t)na * 192);
		TM_HIP(hipMemcpyAsync(freq.data(), d_freq.p, freq.size() * 4, hipMemcpyDeviceToHost, s));
		TM_HIP(hipStreamSynchronize(s));

		// decisions; the segment list stays in order of position
		std::vector<int32_t> piv, tpiv, split_piv;
		std::vector<uint32_t> split_tb(1, 0), split_zeros;
		std::vector<seg_t> next;
		next.reserve(segs.size() + na);
		all.clear();
		hidx.clear();
		std::vector<std::pair<uint32_t, uint32_t>> split_ranges;
		uint32_t a = 0;
		for (uint32_t k = 0; k < segs.size(); ++k) {
			seg_t g = segs[k];
			if (a >= na || act[a] != k) {
				next.push_back(g);
				continue;
			}
			const uint32_t * f = &freq[(size_t)a * 192];
			const uint32_t size = g.end - g.begin;
			g.bits = 0;
			for (int b = 0; b < 192; ++b) g.bits += f[b];
			if (g.mode == NONZERO && size <= NZ_MAX && g.bits <= NZ_BITS) {   // now that its bits are known
				next.push_back(g);
				++a;
				continue;
			}
			int pv = NO_PIVOT;
			if (g.mode == NONZERO) {
				uint32_t mf = f[0];
				pv = 0;
				for (int b = 1; b < 192; ++b)
					if (f[b] > mf) { mf = f[b]; pv = b; }
				if (mf == size || mf == 0) pv = NO_PIVOT;
			} else {
				pv = balancing_pivot(g, f);
			}
			if (pv == NO_PIVOT) {
				seg_t d = g;
				d.mode = DONE;
				next.push_back(d);
				++a;
				continue;
			}
			seg_t z = g, o = g;
			z.end = g.begin + (size - f[pv]);
			o.begin = z.end;
			z.bits = g.bits - f[pv];   // the pivot's are the other side's
			for (seg_t * c : {&z, &o}) c->bits = std::min(c->bits, (uint64_t)(c->end - c->begin) * 192);
			if (g.mode == NONZERO) {
				o.mode = DONE;
			} else {
				z.used[pv >> 5] |= 1u << (pv & 31);
				o.used[pv >> 5] |= 1u << (pv & 31);
				o.mask_nonempty = 1;
				for (seg_t * c : {&z, &o}) {
					const uint32_t cs = c->end - c->begin;
					c->mode = cs > maxp ? BALANCE : (c->mask_nonempty ? DONE : NONZERO);
				}
			}
			next.push_back(z);
			next.push_back(o);
			for (uint32_t t = tb[a]; t < tb[a + 1]; ++t) {
				all.push_back(tiles[t]);
				tpiv.push_back(pv);
				hidx.push_back(t);   // its row of the histograms
			}
			split_tb.push_back((uint32_t)all.size());
			split_piv.push_back(pv);
			split_zeros.push_back(size - f[pv]);
			split_ranges.push_back({g.begin, g.end});
			++a;
		}
		const uint32_t n_split = (uint32_t)all.size(), nsplit = (uint32_t)split_piv.size();
		if (nsplit == 0) {   // nothing moves
			segs.swap(next);
			continue;
		}
		// copy tiles cover every position outside the split segments
		uint32_t pos = 0;
		split_ranges.push_back({n, n});
		for (const auto & r : split_ranges) {
			for (uint32_t b = pos; b < r.first; b += TILE * 4) {
				all.push_back(tile_t{b, std::min(r.first, b + TILE * 4), 0, 0});
				tpiv.push_back(NO_PIVOT);
			}
			pos = r.second;
		}
		const uint32_t nall = (uint32_t)all.size();
		in1.clear();
		push(in1, all.data(), (size_t)nall * 4);
		const size_t at_tpiv = push(in1, tpiv.data(), nall), at_hidx = push(in1, hidx.data(), n_split),
					 at_tb = push(in1, split_tb.data(), nsplit + 1), at_piv = push(in1, split_piv.data(), nsplit),
					 at_zeros = push(in1, split_zeros.data(), nsplit);
		TM_CHECK(ensure<uint32_t>(d_in, c_in, in1.size()));
		TM_CHECK(ensure<uint32_t>(d_out, c_out, 2 * (size_t)n_split));
		uint32_t * in = (uint32_t *)d_in.p, * zb = (uint32_t *)d_out.p, * ob = zb + n_split;
		TM_HIP(hipMemcpyAsync(in, in1.data(), in1.size() * 4, hipMemcpyHostToDevice, s));
		hipLaunchKernelGGL(k_tile_bases, dim3(nsplit), dim3(64), 0, s, (const uint32_t *)d_hist.p, in + at_hidx,
						   (const tile_t *)in, in + at_tb, (const int32_t *)(in + at_piv), in + at_zeros, zb, ob);
		hipLaunchKernelGGL(k_scatter, dim3(nall), dim3(256), 0, s, (const uint32_t *)d_rec[cur].p,
						   (uint32_t *)d_rec[cur ^ 1].p, (const tile_t *)in, (const int32_t *)(in + at_tpiv), zb, ob);
		TM_HIP(hipGetLastError());
		cur ^= 1;
		segs.swap(next);
	}

	// the NONZERO segments left, all their splits at once
	hipLaunchKernelGGL(k_identity, dim3((n + 255) / 256), dim3(256), 0, s, (uint32_t *)d_ord.p, n);
	act.clear();
	for (uint32_t k = 0; k < segs.size(); ++k)
		if (segs[k].mode == NONZERO) act.push_back(k);
	std::vector<uint32_t> ranges;   // first position of each partition
	std::vector<uint32_t> counts;
	const uint32_t nz = (uint32_t)act.size();
	if (nz) {
		TM_CHECK(histograms());
		TM_HIP(hipStreamSynchronize(s));   // in1 may still be uploading
		in1.clear();
		for (uint32_t a = 0; a < nz; ++a) {
			const nz_seg g{segs[act[a]].begin, segs[act[a]].end, a, 0};
			push(in1, &g, 4);
		}
		// segments, counts, rounds; the lists go where the other record
		// buffer (no longer needed) is: 8 words per position
		const size_t at_cnt = in1.size(), words_nz = at_cnt + (size_t)nz * (NZ_ROUNDS + 1);
		TM_CHECK(ensure<uint32_t>(d_nz, c_nz, words_nz));
		uint32_t * z = (uint32_t *)d_nz.p, * lists = (uint32_t *)d_rec[cur ^ 1].p;
		TM_HIP(hipMemcpyAsync(z, in1.data(), in1.size() * 4, hipMemcpyHostToDevice, s));
		hipLaunchKernelGGL(k_nonzero, dim3(nz), dim3(1024), 0, s, (const uint32_t *)d_rec[cur].p, (const nz_seg *)z,
						   (const uint32_t *)d_freq.p, lists, lists + n, (uint32_t *)d_ord.p, z + at_cnt,
						   z + at_cnt + (size_t)nz * NZ_ROUNDS);
		TM_HIP(hipGetLastError());
		counts.resize(words_nz - at_cnt);
		TM_HIP(hipMemcpyAsync(counts.data(), z + at_cnt, counts.size() * 4, hipMemcpyDeviceToHost, s));
		TM_HIP(hipStreamSynchronize(s));
	}

	// finished partitions in position order (segments never overlap and are
	// kept in order)
	for (uint32_t k = 0, a = 0; k < segs.size(); ++k) {
		ranges.push_back(segs[k].begin);
		if (a >= nz || act[a] != k) continue;
		const uint32_t * c = &counts[(size_t)a * NZ_ROUNDS];
		uint32_t at = segs[k].begin + c[0];
		for (uint32_t r = counts[(size_t)nz * NZ_ROUNDS + a]; r > 0; --r) {
			ranges.push_back(at);
			at += c[r];
		}
		++a;
	}
	const uint32_t np = (uint32_t)ranges.size();
	if (np > max_parts) {
		*n_parts = np;
		return set_error(TM_ERR_OVERFLOW, "%u partitions exceed max_parts %u", np, max_parts);
	}
	ranges.push_back(n);
	for (uint32_t p = 0; p <= np; ++p) part_offsets[p] = ranges[p];
	TM_CHECK(ensure<uint32_t>(d_out, c_out, (size_t)np * 7 + 1));
	uint32_t * d_rng = (uint32_t *)d_out.p, * d_mask = d_rng + np + 1;
	TM_HIP(hipMemcpyAsync(d_rng, ranges.data(), ((size_t)np + 1) * 4, hipMemcpyHostToDevice, s));
	hipLaunchKernelGGL(k_part_masks, dim3(np), dim3(1024), 0, s, (const uint32_t *)d_rec[cur].p,
					   (const uint32_t *)d_ord.p, d_rng, d_mask);
	uint32_t * d_perm = (uint32_t *)d_words.p;  // reuse: n x 6 words >= n
	hipLaunchKernelGGL(k_extract_perm, dim3((n + 255) / 256), dim3(256), 0, s, (const uint32_t *)d_rec[cur].p,
					   (const uint32_t *)d_ord.p, n, d_perm);
	TM_HIP(hipGetLastError());
	if (part_masks) TM_HIP(hipMemcpyAsync(part_masks, d_mask, (size_t)np * 24, hipMemcpyDeviceToHost, s));
	TM_HIP(hipMemcpyAsync(perm, d_perm, (size_t)n * 4, hipMemcpyDeviceToHost, s));
	TM_HIP(hipStreamSynchronize(s));
	*n_parts = np;
	return TM_OK;
}
