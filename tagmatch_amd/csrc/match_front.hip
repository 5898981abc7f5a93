// What a step does before the match: the queries of each partition are
// counted (reference front_end.cc:465-477 do_match, on the device), and each
// query's key row starts with the keys of the rich filters it contains.
//
// Exact: a filter contained in the query matches it, whatever the partition
// lookup.  A row that then holds every key needs no match at all, and its
// query is not listed.
#include "match_front.h"
#include "match_dev.h"
#include "match_mfma.h"

#include <algorithm>

using namespace tmx;

namespace {

constexpr uint32_t WAVES = 8;
constexpr uint32_t CHUNK = 2048;    // queries of a workgroup, at most
constexpr uint32_t PARTS = 2048;    // partitions counted at a time
constexpr uint32_t GROUP = 64;      // listed queries tested together
constexpr uint32_t MASKS = MAX_RICH / 32 + 1;   // words of a query's rich-filter mask, odd
constexpr uint32_t IDS = 512;       // rich filters of a query taken at a time
constexpr uint32_t DONE = 0x8000;   // marks a listed query whose row is full

// Sum over the lanes of the wave's 16-lane row up to this one.
__device__ inline uint32_t row_prefix(uint32_t x) {
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);   // row_shr:1
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
	x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
	return x;
}

// Words w .. w + 3 of the row that holds every key.
__device__ inline quad full_words(uint32_t w, uint32_t kw, uint32_t last_mask) {
	quad v = {~0u, ~0u, ~0u, ~0u};
#pragma unroll
	for (uint32_t k = 0; k < 4; ++k)
		if (w + k + 1 == kw) v[k] = last_mask;
	return v;
}

// A workgroup takes `chunk` queries.  First each wave its 64: partitions
// counted on the matrix cores (a column per partition, so that its count is
// a population count), one lane per query against the rich filters that hold
// every key.  The queries left go to a list; 64 of it at a time are tested
// against all rich filters, again on the matrix cores, and sixteen lanes per
// query OR the bitmaps of those it contains, eight in flight (with eight
// listed queries or fewer, the whole wave for one).
//
// Bound by latency: 1M queries that nearly all contain a filter of every key
// read 32 MB and write 256 MB (45 us at the copy rate) in 125 us, where a
// kernel for the rows and one for the counts, both a lane per query or
// partition, took 248; 100k queries that contain 20 of 349 rich filters each
// 128 (250), 1000 queries 15 (32), 64 queries 13 (15).  Counters meet in
// local memory first, and the list takes one global atomic per workgroup:
// atomics on one address take 12-24 ns each, one after another.  Rows as a
// second product (rich filters held x keys of each) came out the same (126
// us, 24 for 1000 queries) and need the bitmaps a second time, transposed.
__global__ void __launch_bounds__(WAVES * 64, 4)
k_front(front_args a) {
	__shared__ uint32_t s_cnt[PARTS];
	__shared__ uint16_t s_list[CHUNK];
	__shared__ uint32_t s_mask[GROUP * MASKS];     // rich filters of each listed query
	__shared__ uint16_t s_ids[WAVES][4][IDS];
	__shared__ unsigned long long s_hold[WAVES];   // few queries: those that contain a filter of every key
	__shared__ uint32_t s_n, s_left, s_base;
	const uint32_t tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
	const uint32_t wave = uniform(tid >> 6);
	const uint32_t rows[2] = {row_of(0, n), row_of(1, n)};   // of 64 queries or filters, in this lane
	const uint32_t base = blockIdx.x * a.chunk, nqc = min(a.chunk, a.nq - base);
	const uint32_t nsub = (nqc + 63) / 64;
	// fewer than one 64 per wave: the waves share each one's filters
	const bool split = nsub < WAVES;
	const uint32_t sub0 = split ? 0u : wave, sub_step = split ? 1u : WAVES;
	const uint32_t f0 = split ? wave : 0u, f_step = split ? WAVES : 1u;
	auto query_words = [&](uint32_t i, bool valid, uint32_t (&w)[3]) {
#pragma unroll
		for (int k = 0; k < 3; ++k) w[k] = valid ? ~a.q[(size_t)(base + i) * 8 + 2 * k + h] : ~0u;
	};
	if (tid == 0) s_n = s_left = 0;
	if (tid < WAVES) s_hold[tid] = 0;

	for (uint32_t p0 = 0; a.pcount && p0 < a.P; p0 += PARTS) {
		const uint32_t np = min(PARTS, a.P - p0), tiles = (np + 31) / 32;
		__syncthreads();
		for (uint32_t p = tid; p < np; p += WAVES * 64) s_cnt[p] = 0;
		__syncthreads();
		for (uint32_t sub = sub0; sub < nsub; sub += sub_step) {
			const uint32_t nv = min(64u, nqc - sub * 64);
			const uint32_t keep = (uint32_t)((nv < 64 ? (1ULL << nv) - 1ULL : ~0ULL) >> (32 * h));
			v8i qv[2][3];
#pragma unroll
			for (uint32_t mt = 0; mt < 2; ++mt) {
				uint32_t w[3];
				query_words(sub * 64 + rows[mt], rows[mt] < nv, w);
#pragma unroll
				for (int k = 0; k < 3; ++k) qv[mt][k] = spread_up(w[k]);
			}
			uint32_t m[3], m1[3];
			auto load_masks = [&](uint32_t t, uint32_t (&w)[3]) {
#pragma unroll
				for (int k = 0; k < 3; ++k) w[k] = a.part_info[(size_t)(p0 + min(t * 32 + n, np - 1)) * 8 + 2 * k + h];
			};
			load_masks(f0, m);
			for (uint32_t t = f0; t < tiles; t += f_step) {
				load_masks(t + f_step, m1);   // past the end: the last again
				const uint32_t p = t * 32 + n;
				v16f lo = start_lo(), hi = start_hi();
#pragma unroll
				for (int k = 0; k < 3; ++k) {
					const v8i pv = spread(m[k]);
					lo = mfma(qv[0][k], pv, lo);
					hi = mfma(qv[1][k], pv, hi);
					m[k] = m1[k];
				}
				const uint32_t c = (uint32_t)__popc(subset_mask(lo, hi) & keep);
				if (p < np && c) atomicAdd(&s_cnt[p], c);
			}
		}
		__syncthreads();
		for (uint32_t p = tid; p < np; p += WAVES * 64)
			if (s_cnt[p]) atomicAdd(&a.pcount[p0 + p], s_cnt[p]);
	}
	if (a.n_rich == 0) return;
	__syncthreads();

	// rich filters that hold every key: one contained is enough
	auto holds_full = [&](uint32_t i, bool valid) -> bool {
		uint4 x = make_uint4(0, 0, 0, 0);
		uint2 y = make_uint2(0, 0);
		if (valid) {
			const uint32_t * w = a.q + (size_t)(base + i) * 8;
			const quad v = *reinterpret_cast<const quad *>(w);
			x = make_uint4(v[0], v[1], v[2], v[3]);
			y = make_uint2(w[4], w[5]);
		}
		bool full = false;
		for (uint32_t f = f0 * 8; f < a.n_full; f += f_step * 8) {
#pragma unroll
			for (uint32_t k = 0; k < 8; ++k) {   // past the end: the last again
				const uint32_t * r = a.rich_words + (size_t)min(f + k, a.n_full - 1) * 8;
				const uint4 c = sld4(r);
				const uint2 d = sld2(r + 4);
				full |= ((c.x & ~x.x) | (c.y & ~x.y) | (c.z & ~x.z) | (c.w & ~x.w) | (d.x & ~y.x) | (d.y & ~y.y)) == 0;
			}
			if (__ballot(valid && !full) == 0) break;
		}
		return full;
	};
	if (split && a.n_full) {
		for (uint32_t sub = 0; sub < nsub; ++sub) {
			const uint32_t i = sub * 64 + lane;
			const uint64_t m = __ballot(holds_full(i, i < nqc));
			if (lane == 0 && m) atomicOr(&s_hold[sub], (unsigned long long)m);
		}
		__syncthreads();
	}
	const uint32_t g = lane >> 4, l = lane & 15;   // sixteen lanes per query
	for (uint32_t sub = wave; sub < nsub; sub += WAVES) {
		const uint32_t i = sub * 64 + lane;
		const bool valid = i < nqc;
		const bool full = split ? (s_hold[sub] >> lane) & 1 : holds_full(i, valid);
		const uint64_t fm = __ballot(valid && full), lm = __ballot(valid && !full);
		if (valid && full) a.qfull[base + i] = 2u;
		if (fm)
			for (uint32_t r = g; r < 64; r += 4)
				if ((fm >> r) & 1)
					for (uint32_t w = l * 4; w < a.kw; w += 64)
						store_words(a.gbm + (size_t)(base + sub * 64 + r) * a.kw, w, a.kw, full_words(w, a.kw, a.last_mask));
		if (lm == 0) continue;
		uint32_t at = 0;
		if (lane == 0) at = atomicAdd(&s_n, (uint32_t)__popcll(lm));
		at = uniform(at);
		if (valid && !full) s_list[at + mbcnt64(lm)] = (uint16_t)i;
	}
	__syncthreads();
	const uint32_t nl = uniform(s_n), fts = (a.n_rich + 63) / 64;

	for (uint32_t g0 = 0; g0 < nl; g0 += GROUP) {
		const uint32_t ng = min(GROUP, nl - g0), qts = ng > 32 ? 2u : 1u;
		{
			const uint32_t c = (wave % qts) * 32 + n, ft0 = wave / qts, step = WAVES / qts;
			v8i qv[3];
			uint32_t w[3], f[6], f1[6];
			query_words(c < ng ? s_list[g0 + c] : 0u, c < ng, w);
			auto load_filters = [&](uint32_t ft, uint32_t (&f)[6]) {   // past the end: the last again
				const uint32_t * r = a.rich_words + h;
#pragma unroll
				for (int k = 0; k < 6; ++k) f[k] = r[(size_t)min(ft * 64 + rows[k / 3], a.n_rich - 1) * 8 + k % 3 * 2];
			};
			load_filters(ft0, f);
#pragma unroll
			for (int k = 0; k < 3; ++k) qv[k] = spread_up(w[k]);
			for (uint32_t ft = ft0; ft < fts; ft += step) {
				load_filters(ft + step, f1);
				v16f lo = start_lo(), hi = start_hi();
#pragma unroll
				for (int k = 0; k < 3; ++k) {
					lo = mfma(spread(f[k]), qv[k], lo);
					hi = mfma(spread(f[3 + k]), qv[k], hi);
				}
#pragma unroll
				for (int k = 0; k < 6; ++k) f[k] = f1[k];
				const uint32_t nf = min(64u, a.n_rich - ft * 64);
				s_mask[c * MASKS + 2 * ft + h] = subset_mask(lo, hi) & (uint32_t)((nf < 64 ? (1ULL << nf) - 1ULL : ~0ULL) >> (32 * h));
			}
		}
		__syncthreads();
		// few queries: the wave's four teams of sixteen lanes share one
		const bool share = ng <= WAVES;
		for (uint32_t r = 0; r * 32 < ng; ++r) {
			const uint32_t c = share ? wave : r * 32 + g * WAVES + wave;
			const bool mine = c < ng;
			if (__ballot(mine) == 0) continue;
			const uint32_t i = mine ? s_list[g0 + c] : 0u;
			const uint32_t first = share ? g * 8 : 0u, step = share ? 32u : 8u;
			uint16_t * ids = s_ids[wave][g];
			bool miss = false;
			for (uint32_t wb = 0; wb < a.kw; wb += 64) {   // 64 words (2048 keys) per pass
				const uint32_t w = wb + l * 4;
				quad acc = {0, 0, 0, 0};
				for (uint32_t c0 = 0; c0 < 2 * fts; c0 += 16) {
					uint32_t m = mine && c0 + l < 2 * fts ? s_mask[c * MASKS + c0 + l] : 0u;
					uint32_t at = row_prefix((uint32_t)__popc(m));
					const uint32_t total = (uint32_t)__shfl((int)at, (int)(lane | 15), 64);
					at -= (uint32_t)__popc(m);
					const uint32_t f = (c0 + l) * 32;
					while (m) {
						const uint32_t bit = (uint32_t)__builtin_ctz(m);
						m &= m - 1;
						ids[at++] = (uint16_t)(f + bit);
					}
					wave_fence();
					if (w < a.kw)
						for (uint32_t k0 = first; k0 < total; k0 += step) {
							quad v[8];
#pragma unroll
							for (uint32_t k = 0; k < 8; ++k)   // past the end: the last again
								v[k] = load_words(a.rich_bm + (size_t)ids[min(k0 + k, total - 1)] * a.kw, w, a.kw);
#pragma unroll
							for (uint32_t k = 0; k < 8; ++k) acc |= v[k];
						}
					wave_fence();
				}
				if (share)
#pragma unroll
					for (uint32_t k = 0; k < 4; ++k) {
						acc[k] |= (uint32_t)__shfl_xor((int)acc[k], 16, 64);
						acc[k] |= (uint32_t)__shfl_xor((int)acc[k], 32, 64);
					}
				if (mine && w < a.kw) {
					if (!share || g == 0) store_words(a.gbm + (size_t)(base + i) * a.kw, w, a.kw, acc);
					const quad want = full_words(w, a.kw, a.last_mask);
#pragma unroll
					for (uint32_t k = 0; k < 4; ++k) miss |= w + k < a.kw && (want[k] & ~acc[k]) != 0;
				}
			}
			const bool full = ((__ballot(miss) >> (g * 16)) & 0xFFFFu) == 0;
			if (mine && l == 0 && (!share || g == 0)) {
				a.qfull[base + i] = full ? 2u : 0u;
				if (full) s_list[g0 + c] = (uint16_t)(i | DONE);
			}
		}
		__syncthreads();
	}
	if (!a.active || nl == 0) return;

	// one global atomic per workgroup: they serialize
	uint32_t at[CHUNK / (WAVES * 64)];
#pragma unroll
	for (uint32_t k = 0; k < CHUNK / (WAVES * 64); ++k) {
		const uint32_t x = k * WAVES * 64 + tid;
		const bool left = x < nl && !(s_list[x] & DONE);
		const uint64_t m = __ballot(left);
		uint32_t b = 0;
		if (lane == 0 && m) b = atomicAdd(&s_left, (uint32_t)__popcll(m));
		b = uniform(b);
		at[k] = left ? b + mbcnt64(m) : ~0u;
	}
	__syncthreads();
	if (tid == 0) s_base = s_left ? atomicAdd(a.n_active, s_left) : 0u;
	__syncthreads();
#pragma unroll
	for (uint32_t k = 0; k < CHUNK / (WAVES * 64); ++k) {
		if (at[k] == ~0u) continue;
		const uint32_t qi = base + s_list[k * WAVES * 64 + tid], to = s_base + at[k];
		a.active[to] = qi;
		const uint32_t * w = a.q + (size_t)qi * 8;
		const quad v = *reinterpret_cast<const quad *>(w);
		uint4 * d = reinterpret_cast<uint4 *>(a.qact + (size_t)to * 8);
		d[0] = make_uint4(v[0], v[1], v[2], v[3]);
		d[1] = make_uint4(w[4], w[5], 0u, 0u);
	}
}

} // namespace

namespace tmx {

// About two workgroups per CU (with three or four 100k queries take 126-134
// us instead of 128, 1M 129-146 instead of 125); at least eight queries each,
// a wave for the rows of each, so that small steps spread too: 64 queries
// take 13 us with eight per workgroup, 20 with 16 or 32.
void front_launch(front_args a, hipStream_t s) {
	if (a.nq == 0) return;
	const uint32_t per = (a.nq + 511) / 512;
	a.chunk = std::min(CHUNK, std::max(8u, (per + 7) & ~7u));
	hipLaunchKernelGGL(k_front, dim3((a.nq + a.chunk - 1) / a.chunk), dim3(WAVES * 64), 0, s, a);
}

} // namespace tmx
