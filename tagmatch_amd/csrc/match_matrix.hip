// The subset match on the matrix cores.
#include "match_matrix.h"
#include "match_dev.h"
#include "match_mfma.h"

#include <algorithm>

using namespace tmx;

namespace {

constexpr uint32_t LIST = 256;   // candidate queries of a block taken at a time
constexpr uint32_t LOG = 128;    // hits a wave stages
constexpr uint32_t AHEAD = 3;    // blocks whose words are loaded together (one tile of queries)
constexpr uint32_t PARTIAL = 0x8000;   // marks a listed block with fewer than 64 filters

// ORs key ids into a row: a word is read first, and written only where the
// bit is missing (rows hold most keys already; a stale read costs a
// redundant atomic, nothing else).
__device__ inline void or_key(uint32_t * row, uint32_t id) {
	const uint32_t bit = 1u << (id & 31);
	if ((row[id >> 5] & bit) == 0) atomicOr(&row[id >> 5], bit);
}

__device__ inline uint32_t inline_keys(uint64_t kv) {
	uint32_t n = 0;
#pragma unroll
	for (int x = 0; x < 4; ++x) n += ((kv >> (16 * x)) & 0xFFFFu) != KEY_NONE;
	return n;
}

// The match.  A workgroup takes an item: up to SUPER queries, their inverted
// words in local memory, and a segment's blocks of 64 filters.
//
//   Candidates: the blocks' AND masks (columns) against the queries (rows): a
//   bit per pair, 6 instructions of the matrix unit for 64 x 32 pairs, and
//   the blocks that have any listed.
//   Tests: a wave takes a listed block, spreads its filters (rows) once, and
//   tests them against its candidates (columns), 32 at a time: 6 matrix
//   instructions, a conversion and about 40 others for 2048 pairs.
//   Hits go to a log in local memory, which the wave empties 64 at a time.
//
// Bound by the vector unit, which spreads the operands, turns accumulators
// into masks and logs hits: where every match is enumerated (1M queries, 10M
// filters, 140 ms, 50 G matches/s) it is busy 79 % of the time and the matrix
// unit 40 %; with the full-row exit (0.95 ms) it is busy 57 %, and the waves
// wait for blocks and keys 55 % of theirs.  One query at a time against 64
// filters on the vector unit took 556 and 1.98 ms: each test read 24 bytes
// of local memory per lane, 12 of its cycles, and 7 instructions.  Of the 556
// ms' gain a part is key work left out: matches of rows that are complete
// before the match (97 % of them there) are counted and their keys not read;
// with them read the 140 ms are 335 (65k queries: 9.2 and 21.8).
//
// Two workgroups of eight waves per CU: 128 registers; with 96 (five waves a
// SIMD) the operands spill (a third slower).  A block's words are loaded
// before its candidates are listed, and the next 32 queries' words during the
// tests of the last (9.39 and 9.19 ms for 65k queries against all matches;
// loaded a whole block ahead, they went to scratch memory: 9.68).
template <int MODE>
__global__ void __launch_bounds__(MX_WAVES * 64, 4)
k_match_x(mx_args a) {
	constexpr int WAVES = MX_WAVES, NT = WAVES * 64;
	constexpr uint32_t SUPER = mx_super(MODE), MASK = mx_mask_words(MODE), VISITS = mx_visits(MODE);
	constexpr bool ROWS = MODE == MX_KEYS || MODE == MX_KEYS_LDS;
	__shared__ uint32_t s_rows[MODE == MX_KEYS_LDS ? MX_ROW_WORDS : 1];   // key rows, kw words each
	__shared__ uint32_t s_cnt[ROWS ? 1 : SUPER];    // values of each query so far
	__shared__ uint32_t s_q[6 * SUPER];             // inverted words, one plane per word
	__shared__ uint32_t s_full[SUPER / 32];         // queries whose rows hold every key
	__shared__ uint32_t s_mask[MASK];               // candidate masks
	__shared__ uint16_t s_vis[VISITS];              // blocks with candidates
	__shared__ uint32_t s_nvis, s_seen[VISITS / 32];
	__shared__ uint16_t s_list[WAVES][LIST];
	__shared__ uint32_t s_log[WAVES][LOG];
	__shared__ uint32_t s_item;
	__shared__ uint64_t s_stat[WAVES][4];
	const uint32_t tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
	const uint32_t wave = uniform(tid >> 6);
	const uint32_t frow[2] = {near_row(0, n), near_row(1, n)};   // a block's filters in this lane
	const uint32_t kw = a.f.kw;
	const uint32_t nq_all = a.nq_dev ? sld1(a.nq_dev) : a.nq;
	const uint32_t epoch = a.step_vals ? sld1(a.step_vals) : a.epoch;
	const uint32_t ovf_n = a.step_vals ? sld1(a.step_vals + 1) : a.f.ovf_n;
	mx_shape sh = {0, 0, 0, 0};
	if (!a.units) sh = mx_shape_of(MODE, kw, nq_all, a.nblk, a.resident, a.seg_fixed, a.seg_min);
	const uint32_t items = a.units ? sld1(a.uprefix + a.n_units) : sh.nsuper * sh.nseg;
	if (blockIdx.x == 0 && tid == 0) *a.n_items = items;
	const bool queued = items > gridDim.x;
	uint64_t l_hits = 0, w_visit = 0, w_test = 0, w_hev = 0;   // hits by lane, the rest by wave
	if (tid < VISITS / 32) s_seen[tid] = 0;

	for (uint32_t turn = 0;; ++turn) {
		uint32_t item;
		if (queued) {
			if (tid == 0) {
				uint32_t got = 0xFFFFFFFFu;
				for (uint32_t k = 0; k < MX_QUEUES; ++k) {
					const uint32_t x = (blockIdx.x + k) % MX_QUEUES;
					const uint32_t lo = (uint32_t)((uint64_t)items * x / MX_QUEUES);
					const uint32_t hi = (uint32_t)((uint64_t)items * (x + 1) / MX_QUEUES);
					if (a.qnext[x * MX_QPAD] >= hi - lo) continue;
					const unsigned long long i = atomicAdd(&a.qnext[x * MX_QPAD], 1ULL);
					if (i < hi - lo) { got = lo + (uint32_t)i; break; }
				}
				s_item = got;
			}
			__syncthreads();
			item = uniform(s_item);
			if (item == 0xFFFFFFFFu) break;
		} else {
			item = blockIdx.x;
			if (turn || item >= items) break;
		}
		// blocks of the item: tiles of 32, `apart` blocks from one to the next
		uint32_t q0, nqs, b0, apart, nloc, b_end, seg;
		bool sole = false;   // no other item adds to its queries' rows, which are empty
		if (a.units) {
			uint32_t lo = 0, hi = a.n_units;
			while (hi - lo > 1) {
				const uint32_t mid = (lo + hi) >> 1;
				if (sld1(a.uprefix + mid) <= item) lo = mid; else hi = mid;
			}
			const uint4 u0 = sld4(a.units + (size_t)lo * 8);       // part, first query, queries, supers
			const uint4 u1 = sld4(a.units + (size_t)lo * 8 + 4);   // segments, seg blocks, first, end block
			const uint32_t local = item - sld1(a.uprefix + lo);
			seg = local / u0.w;
			const uint32_t sup = local - seg * u0.w;
			q0 = u0.y + sup * a.unit_sq;
			nqs = min(a.unit_sq, u0.y + u0.z - q0);
			b0 = u1.z + seg * 32;
			apart = u1.x * 32;
			b_end = u1.w;
			sole = u1.x == 1;
		} else {
			seg = item / sh.nsuper;
			const uint32_t sup = item - seg * sh.nsuper;
			q0 = sup * sh.sq;
			nqs = min(sh.sq, nq_all - q0);
			b0 = seg * 32;
			apart = sh.nseg * 32;
			b_end = a.nblk;
		}
		nloc = b0 < b_end ? ((b_end - b0 + apart - 1) / apart) * 32 : 0u;
		auto block_of = [&](uint32_t i) -> uint32_t { return b0 + (i >> 5) * apart + (i & 31u); };
		// the item's queries, inverted; all ones (a subset of nothing but the
		// empty filter) up to a whole number of tiles
		if (MODE == MX_KEYS_LDS)
			for (uint32_t w = tid; w < nqs * kw; w += NT) s_rows[w] = 0;
		uint32_t * const hc = ROWS ? nullptr : a.hcnt + (size_t)seg * nq_all + q0;
		if (!ROWS)
			for (uint32_t t = tid; t < nqs; t += NT) s_cnt[t] = MODE == MX_WRITE || MODE == MX_WRITE_KEYS ? hc[t] : 0u;
		for (uint32_t t = tid; t < ((nqs + 63) & ~63u); t += NT) {
			uint4 x = make_uint4(0, 0, 0, 0);
			uint2 y = make_uint2(0, 0);
			bool full = false;
			if (t < nqs) {
				x = *reinterpret_cast<const uint4 *>(a.q + (size_t)(q0 + t) * 8);
				y = *reinterpret_cast<const uint2 *>(a.q + (size_t)(q0 + t) * 8 + 4);
				if (MODE == MX_KEYS && a.qfull) full = a.qfull[a.qmap ? a.qmap[q0 + t] : q0 + t] != 0u;
			}
			s_q[t] = ~x.x;
			s_q[SUPER + t] = ~x.y;
			s_q[2 * SUPER + t] = ~x.z;
			s_q[3 * SUPER + t] = ~x.w;
			s_q[4 * SUPER + t] = ~y.x;
			s_q[5 * SUPER + t] = ~y.y;
			const uint64_t fm = __ballot(full);
			if (n == 0) s_full[t >> 5] = (uint32_t)(fm >> (32 * h));
		}
		__syncthreads();

		uint32_t * log = s_log[wave];
		uint16_t * list = s_list[wave];
		uint32_t nlog = 0;
		// The staged hits (query, mask bit and block of each, 64 at a time): their
		// keys into the queries' rows, or their values counted or written.
		auto drain = [&]() {
			for (uint32_t base = 0; base < nlog; base += 64) {
				const bool mine = base + lane < nlog;
				const uint32_t e = mine ? log[base + lane] : 0u;
				const uint32_t qi = e & 0xFFFu, ql = q0 + qi;
				const uint32_t slot = block_of(e >> 18) * 64 + near_bit((e >> 12) & 31u, (e >> 17) & 1u);
				if (MODE == MX_WRITE) {
					if (mine) {
						const uint64_t at = a.off[ql] + atomicAdd(&s_cnt[qi], 1u);
						if (at < a.vcap) a.vals[at] = a.f.slot_fid[slot];
					}
					continue;
				}
				const uint32_t gq = mine && a.qmap ? a.qmap[ql] : ql;
				const uint32_t rq = MODE == MX_KEYS_LDS ? qi : gq;   // row
				uint64_t kv = ~0ULL;
				if (mine) kv = a.f.slot_keys[slot];
				uint32_t off = 0, cnt = 0;   // an overflow list
				if (MODE == MX_COUNT_KEYS) {
					if (mine)
						atomicAdd(&s_cnt[qi], (kv & 0xFFFFu) == KEY_NONE ? ovf_list(kv, a.f.ovf, ovf_n, off) : inline_keys(kv));
					continue;
				}
				uint64_t at0 = 0;            // MX_WRITE_KEYS: its first value
				if (MODE == MX_WRITE_KEYS) {
					const bool lst = mine && (kv & 0xFFFFu) == KEY_NONE;
					uint32_t c = 0;
					if (lst) c = cnt = ovf_list(kv, a.f.ovf, ovf_n, off);
					else if (mine) c = inline_keys(kv);
					if (mine) at0 = a.off[ql] + atomicAdd(&s_cnt[qi], c);
					if (mine && !lst)
						for (uint32_t x = 0; x < c; ++x) {
							const uint32_t id = (uint32_t)(kv >> (16 * x)) & 0xFFFFu;
							if (at0 + x < a.vcap) a.vals[at0 + x] = a.f.key_dict[id < a.f.n_keys ? id : 0u];
						}
					// long lists are left to k_write_lists: one wave would be
					// busy with its own for long after the others
					const uint64_t lb = __ballot(cnt >= MX_LONG_LIST);
					if (lb) {
						uint64_t r = 0;
						if (lane == 0) r = atomicAdd(a.n_lists, (unsigned long long)__popcll(lb));
						r = (uint64_t)__shfl((unsigned long long)r, 0) + mbcnt64(lb);
						if (cnt >= MX_LONG_LIST && r < a.lists_cap) {
							a.lists[r] = make_uint4((uint32_t)at0, (uint32_t)(at0 >> 32), off, cnt);
							cnt = 0;
						}
					}
				}
				uint32_t * row = MODE == MX_KEYS_LDS ? s_rows + qi * kw : a.gbm + (size_t)gq * kw;
				bool lst = false;
				uint32_t rich = 0;
				if (ROWS && mine) {
					if ((kv & 0xFFFFu) != KEY_NONE) {
						uint32_t id[4], w[4];
#pragma unroll
						for (int x = 0; x < 4; ++x) {
							id[x] = (uint32_t)(kv >> (16 * x)) & 0xFFFFu;
							if (id[x] == KEY_NONE) id[x] = id[0];
							w[x] = MODE == MX_KEYS_LDS ? 0u : row[id[x] >> 5];
						}
#pragma unroll
						for (int x = 0; x < 4; ++x)
							if (((w[x] >> (id[x] & 31)) & 1u) == 0 && (x == 0 || id[x] != id[0]))
								atomicOr(&row[id[x] >> 5], 1u << (id[x] & 31));
					} else {
						rich = (uint32_t)(kv >> 48);   // 1 + index of a rich filter, or 0
						if (rich > a.n_rich) rich = 0;
						lst = rich == 0;
					}
				}
				// rich filters: their key sets as bitmaps, unless the rows
				// hold them already
				uint64_t rm = !ROWS || a.rich_done ? 0ULL : __ballot(rich != 0);
				while (rm) {
					const uint32_t j = (uint32_t)__builtin_ctzll(rm);
					rm &= rm - 1;
					const uint32_t jr = (uint32_t)__builtin_amdgcn_readlane((int)rich, (int)j);
					const uint32_t jq = (uint32_t)__builtin_amdgcn_readlane((int)rq, (int)j);
					const uint32_t * src = a.rich_bm + (size_t)(jr - 1) * kw;
					uint32_t * jrow = MODE == MX_KEYS_LDS ? s_rows + jq * kw : a.gbm + (size_t)jq * kw;
					for (uint32_t w = lane; w < kw; w += 64) {
						const uint32_t miss = src[w] & ~jrow[w];
						if (miss) atomicOr(&jrow[w], miss);
					}
				}
				// overflow lists: their ids one after another over the lanes
				if (lst) cnt = ovf_list(kv, a.f.ovf, ovf_n, off);
				if (__ballot(cnt != 0) == 0) continue;
				uint32_t pre = wave_prefix(cnt);
				const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)pre, 63);
				pre -= cnt;
				for (uint32_t k0 = 0; k0 < total; k0 += 64) {
					const uint32_t k = k0 + lane;
					uint32_t e0 = 0;   // the last entry that starts at or before k
#pragma unroll
					for (uint32_t d = 32; d > 0; d >>= 1)
						if (__shfl(pre, (int)(e0 + d), 64) <= k) e0 += d;
					const uint32_t at = __shfl(off, (int)e0, 64) + 1 + k - __shfl(pre, (int)e0, 64);
					const uint32_t eq = __shfl(rq, (int)e0, 64);
					if (MODE == MX_WRITE_KEYS) {
						const uint64_t va = ((uint64_t)(uint32_t)__shfl((int)(at0 >> 32), (int)e0, 64) << 32 |
											 (uint32_t)__shfl((int)(uint32_t)at0, (int)e0, 64)) +
											(k - __shfl(pre, (int)e0, 64));
						if (k < total && va < a.vcap) {
							const uint32_t id = a.f.ovf[at];
							a.vals[va] = a.f.key_dict[id < a.f.n_keys ? id : 0u];
						}
					} else if (k < total) {
						const uint32_t id = a.f.ovf[at];
						if (id < a.f.n_keys) or_key((MODE == MX_KEYS_LDS ? s_rows : a.gbm) + (size_t)eq * kw, id);
					}
				}
			}
			nlog = 0;
			wave_fence();
		};

		const uint32_t np = (nqs + 63) / 64;   // pairs of 32-query tiles
		const uint32_t stride = 2 * np + 1;
		// the queries of this lane's half of 64 that the item has
		uint32_t tail = ~0u;
		if (n * 64 + h * 32 + 32 > nqs) tail = n * 64 + h * 32 < nqs ? (1u << (nqs & 31u)) - 1u : 0u;
		const uint32_t pass = min(VISITS, MASK / stride) & ~31u;
		for (uint32_t p0 = 0; p0 < nloc; p0 += pass) {
			const uint32_t nb = min(pass, nloc - p0);
			if (tid == 0) s_nvis = 0;
			__syncthreads();
			// Candidates: block masks (columns, 32 at a time) against every
			// query (rows, two tiles of 32 at a time).  Lane n holds a block's
			// column, half h of the rows.
			const uint32_t steps = ((nb + 31) / 32) * np;
			uint32_t st = steps * wave / WAVES;
			const uint32_t st_end = steps * (wave + 1) / WAVES;
			while (st < st_end) {
				const uint32_t bt = st / np;
				uint32_t t = st - bt * np;
				const uint32_t t1 = min(np, t + st_end - st);
				st += t1 - t;
				uint32_t nv = 0;
				v8i bm[3];
				{
					uint32_t w[3] = {~0u, ~0u, ~0u};
					const uint32_t b = bt * 32 + n;
					const uint32_t blk = block_of(p0 + b);
					if (b < nb && blk < b_end) {
						const uint32_t * bi = a.f.blk_info + (size_t)blk * 8;
#pragma unroll
						for (int k = 0; k < 3; ++k) w[k] = bi[2 * k + h];
						nv = bi[6];
					}
#pragma unroll
					for (int k = 0; k < 3; ++k) bm[k] = spread_up(w[k]);
				}
				uint32_t any = 0;
				uint32_t * mw = s_mask + (bt * 32 + n) * stride + h * np;
				for (; t < t1; ++t) {
					const uint32_t * sq = s_q + h * SUPER + t * 64;
					v16f lo = start_lo(), hi = start_hi();
#pragma unroll
					for (int k = 0; k < 3; ++k) {
						lo = mfma(spread(sq[2 * k * SUPER + row_of(0, n)]), bm[k], lo);
						hi = mfma(spread(sq[2 * k * SUPER + row_of(1, n)]), bm[k], hi);
					}
					const uint32_t m = nv ? subset_mask(lo, hi) : 0u;
					if (bt * 32 + n < nb) mw[t] = m;
					any |= m;
				}
				// blocks with candidates; a block whose pairs are split over
				// two waves is listed by the first that finds one
				uint64_t av = __ballot(any != 0);
				const uint32_t a32 = (uint32_t)av | (uint32_t)(av >> 32);
				if (a32) {
					uint32_t seen = 0;
					if (lane == 0) seen = atomicOr(&s_seen[bt], a32);
					const bool list_it = h == 0 && ((a32 & ~uniform(seen)) >> n & 1u);
					const uint64_t lb = __ballot(list_it);
					uint32_t at = 0;
					if (lane == 0 && lb) at = atomicAdd(&s_nvis, (uint32_t)__popcll(lb));
					at = uniform(at);
					if (list_it) s_vis[at + mbcnt64(lb)] = (uint16_t)(bt * 32 + n + (nv < 64 ? PARTIAL : 0u));
				}
			}
			__syncthreads();
			const uint32_t nvis = s_nvis;
			if (tid < VISITS / 32) s_seen[tid] = 0;   // for the next pass
			// the lanes of a block whose filters the step sees
			auto valid_lanes = [&](uint32_t vis, uint32_t b) -> uint64_t {
				uint64_t lm = ~0ULL;
				if (vis & PARTIAL) {
					const uint32_t bnv = sld1(a.f.blk_info + (size_t)b * 8 + 6);
					if (bnv < 64) lm = (1ULL << bnv) - 1ULL;
				}
				if (a.slot_epoch) lm &= __ballot(a.slot_epoch[(size_t)b * 64 + lane] <= epoch);
				return lm;
			};
			auto load_words = [&](uint32_t b, uint32_t (&fw)[3][2]) {
				const uint32_t * bw = a.f.blk_words + (size_t)b * BLOCK_WORDS + h * 64;
#pragma unroll
				for (int k = 0; k < 3; ++k)
#pragma unroll
					for (int mt = 0; mt < 2; ++mt) fw[k][mt] = bw[k * 128 + frow[mt]];
			};
			// filter operands; lanes without a filter: all ones, a subset of
			// no query but the full one
			auto operands = [&](const uint32_t (&fw)[3][2], uint64_t lm, v8i (&fa)[3][2]) {
#pragma unroll
				for (int mt = 0; mt < 2; ++mt) {
					const uint32_t dead = (lm >> frow[mt]) & 1 ? 0u : ~0u;
#pragma unroll
					for (int k = 0; k < 3; ++k) fa[k][mt] = spread_up(fw[k][mt] | dead);
				}
			};
			// hm: the filters of the item's block `at` that
			// query qi of this lane contains
			auto take_hits = [&](uint32_t hm, uint32_t qi, uint32_t at) {
				const uint64_t ev = __ballot(hm != 0);
				if (ev == 0) return;
				w_hev += (uint32_t)__popc((uint32_t)ev | (uint32_t)(ev >> 32));
				l_hits += (uint32_t)__popc(hm);
				if (MODE == MX_COUNT) {
					if (hm) atomicAdd(&s_cnt[qi], (uint32_t)__popc(hm));
					return;
				}
				// rows known to hold every key gain nothing
				if (MODE == MX_KEYS && a.qfull && ((s_full[qi >> 5] >> (qi & 31)) & 1u)) hm = 0;
				const uint32_t tag = qi | (at << 18) | (h << 17);
				uint64_t hb = __ballot(hm != 0);
				while (hb) {
					const uint32_t c = (uint32_t)__popcll(hb);
					if (nlog + c > LOG) drain();
					if (hm) {
						const uint32_t bit = (uint32_t)__builtin_ctz(hm);
						log[nlog + mbcnt64(hb)] = tag + (bit << 12);
						hm &= hm - 1;
					}
					nlog += c;
					hb = __ballot(hm != 0);
				}
				wave_fence();
			};
			if (nqs <= 32) {
				// One tile of queries: every listed block against all of it, its
				// operand kept in registers, the words of AHEAD blocks in flight.
				v8i qv[3];
#pragma unroll
				for (int k = 0; k < 3; ++k) qv[k] = spread(s_q[(2 * k + h) * SUPER + n]);
				for (uint32_t v0 = wave; v0 < nvis; v0 += AHEAD * WAVES) {
					uint32_t fw[AHEAD][3][2], vis[AHEAD];
#pragma unroll
					for (uint32_t g = 0; g < AHEAD; ++g) {
						// past the end: the first block again, not used
						vis[g] = uniform(s_vis[v0 + g * WAVES < nvis ? v0 + g * WAVES : v0]);
						load_words(block_of(p0 + (vis[g] & ~PARTIAL)), fw[g]);
					}
#pragma unroll
					for (uint32_t g = 0; g < AHEAD; ++g) {
						if (v0 + g * WAVES >= nvis) break;
						const uint32_t at = p0 + (vis[g] & ~PARTIAL);
						const uint64_t lm = valid_lanes(vis[g], block_of(at));
						v8i fa[3][2];
						operands(fw[g], lm, fa);
						w_test += nqs;
						w_visit += 1;
						v16f lo = start_lo(), hi = start_hi();
#pragma unroll
						for (int k = 0; k < 3; ++k) {
							lo = mfma(fa[k][0], qv[k], lo);
							hi = mfma(fa[k][1], qv[k], hi);
						}
						take_hits(n < nqs ? subset_mask(lo, hi) & near_mask(lm, h) : 0u, n, at);
					}
				}
			} else {
				// A block's filters (rows) against its candidates (columns),
				// 32 at a time.
				for (uint32_t v = wave; v < nvis; v += WAVES) {
					const uint32_t vis = uniform(s_vis[v]), bn = vis & ~PARTIAL, at = p0 + bn;
					uint32_t fw[3][2];
					load_words(block_of(at), fw);   // (on their way while the list is written)
					uint32_t m = n < np ? s_mask[bn * stride + h * np + n] : 0u;
					// candidates as a list: each lane writes those of its mask
					// behind the lanes before it, LIST at a time
					const uint32_t qb = n * 64 + h * 32;
					m &= tail;
					uint32_t pos = wave_prefix((uint32_t)__popc(m));
					uint32_t left = (uint32_t)__builtin_amdgcn_readlane((int)pos, 63);
					pos -= (uint32_t)__popc(m);
					w_test += left;
					w_visit += left != 0;
					auto write_list = [&]() {
						while (__ballot(m != 0 && pos < LIST)) {
							if (m != 0 && pos < LIST) {
								const uint32_t bit = (uint32_t)__builtin_ctz(m);
								m &= m - 1;
								list[pos++] = (uint16_t)(qb + bit);
							}
						}
					};
					write_list();
					const uint64_t lm = valid_lanes(vis, block_of(at));
					v8i fa[3][2];
					operands(fw, lm, fa);
					const uint32_t keep = near_mask(lm, h);
					while (left) {
						const uint32_t cnt = min(left, LIST);
						left -= cnt;
						pos -= LIST;   // only of lanes with more to list
						wave_fence();
						// the words of the next 32 are read meanwhile
						auto read_words = [&](uint32_t qi, uint32_t (&w)[3]) {
#pragma unroll
							for (int k = 0; k < 3; ++k) w[k] = s_q[(2 * k + h) * SUPER + qi];
						};
						uint32_t qi = list[n < cnt ? n : 0u], w[3];
						read_words(qi, w);
						for (uint32_t base = 0; base < cnt; base += 32) {
							const bool valid = base + n < cnt;
							const uint32_t qi1 = list[base + 32 + n < cnt ? base + 32 + n : base];
							uint32_t w1[3];
							read_words(qi1, w1);
							v16f lo = start_lo(), hi = start_hi();
#pragma unroll
							for (int k = 0; k < 3; ++k) {
								const v8i qv = spread(w[k]);
								lo = mfma(fa[k][0], qv, lo);
								hi = mfma(fa[k][1], qv, hi);
							}
							const uint32_t hm = subset_mask(lo, hi);
							take_hits(valid ? hm & keep : 0u, qi, at);
							qi = qi1;
#pragma unroll
							for (int k = 0; k < 3; ++k) w[k] = w1[k];
						}
						wave_fence();
						if (left) write_list();
					}
				}
			}
			__syncthreads();   // the masks' readers are done
		}
		if (nlog) drain();
		__syncthreads();
		if (MODE == MX_COUNT || MODE == MX_COUNT_KEYS) {
			for (uint32_t t = tid; t < nqs; t += NT) hc[t] = s_cnt[t];
			__syncthreads();
		}
		if (MODE == MX_KEYS_LDS) {
			// merged with what the rows hold: a wave per row, an atomic only
			// for words that gain bits
			for (uint32_t j = wave; j < nqs; j += WAVES) {
				uint32_t * dst = a.gbm + (size_t)(a.qmap ? sld1(a.qmap + q0 + j) : q0 + j) * kw;
				for (uint32_t w = lane; w < kw; w += 64) {
					const uint32_t v = s_rows[j * kw + w];
					if (sole && v) dst[w] = v;
					else if (v && (v & ~dst[w])) atomicOr(&dst[w], v);
				}
			}
			__syncthreads();
		}
	}
	// statistics: one record per workgroup, summed with the step's other
	// counts (thousands of waves adding to the same counters took 0.2 ms)
	for (int d = 32; d > 0; d >>= 1) l_hits += __shfl_xor(l_hits, d, 64);
	if (lane == 0) {
		s_stat[wave][0] = l_hits;
		s_stat[wave][1] = w_visit;
		s_stat[wave][2] = w_test;
		s_stat[wave][3] = w_hev;
	}
	__syncthreads();
	if (tid < 4) {
		uint64_t v = 0;
		for (int w = 0; w < WAVES; ++w) v += s_stat[w][tid];
		a.wg_stats[(size_t)blockIdx.x * 4 + tid] = v;
	}
}

} // namespace

namespace tmx {

namespace {

// 64 queries per workgroup, a share of the rows per wave.
__global__ void __launch_bounds__(1024)
k_prefix(uint32_t * __restrict__ hcnt, uint32_t rows, uint32_t nq, uint32_t * __restrict__ total) {
	__shared__ uint32_t s_sum[16][64];
	const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = blockIdx.x * 64 + lane;
	const uint32_t r0 = (uint32_t)((uint64_t)rows * w / 16), r1 = (uint32_t)((uint64_t)rows * (w + 1) / 16);
	uint32_t sum = 0;
	if (q < nq) {
#pragma unroll 8
		for (uint32_t r = r0; r < r1; ++r) sum += hcnt[(size_t)r * nq + q];
	}
	s_sum[w][lane] = sum;
	__syncthreads();
	uint32_t at = 0, all = 0;
	for (uint32_t k = 0; k < 16; ++k) {
		if (k < w) at += s_sum[k][lane];
		all += s_sum[k][lane];
	}
	if (q >= nq) return;
	if (w == 0) total[q] = all;
#pragma unroll 8
	for (uint32_t r = r0; r < r1; ++r) {
		const uint32_t v = hcnt[(size_t)r * nq + q];
		hcnt[(size_t)r * nq + q] = at;
		at += v;
	}
}

// The recorded lists, a wave for each in turn, eight ids per lane in flight.
__global__ void __launch_bounds__(256)
k_write_lists(const uint4 * __restrict__ lists, const unsigned long long * __restrict__ n_lists, uint64_t cap,
			  dev_fib_view f, uint32_t * __restrict__ vals, uint64_t vcap) {
	const uint32_t lane = threadIdx.x & 63;
	const uint64_t n = min((uint64_t)*n_lists, cap);
	for (uint64_t r = ((uint64_t)blockIdx.x * 256 + threadIdx.x) >> 6; r < n; r += (uint64_t)gridDim.x * 4) {
		const uint4 l = lists[r];
		const uint64_t at = (uint64_t)l.x | ((uint64_t)l.y << 32);
		for (uint32_t i0 = 0; i0 < l.w; i0 += 512) {
			uint32_t id[8];
#pragma unroll
			for (uint32_t k = 0; k < 8; ++k) {
				const uint32_t i = i0 + k * 64 + lane;
				id[k] = i < l.w ? f.ovf[l.z + 1 + i] : 0u;
			}
#pragma unroll
			for (uint32_t k = 0; k < 8; ++k) id[k] = f.key_dict[id[k] < f.n_keys ? id[k] : 0u];
#pragma unroll
			for (uint32_t k = 0; k < 8; ++k) {
				const uint32_t i = i0 + k * 64 + lane;
				if (i < l.w && at + i < vcap) vals[at + i] = id[k];
			}
		}
	}
}

using mx_fn = void (*)(mx_args);
mx_fn kernel_of(int mode) {
	switch (mode) {
	case MX_KEYS: return k_match_x<MX_KEYS>;
	case MX_KEYS_LDS: return k_match_x<MX_KEYS_LDS>;
	case MX_COUNT: return k_match_x<MX_COUNT>;
	case MX_COUNT_KEYS: return k_match_x<MX_COUNT_KEYS>;
	case MX_WRITE: return k_match_x<MX_WRITE>;
	default: return k_match_x<MX_WRITE_KEYS>;
	}
}

} // namespace

void mx_prefix(uint32_t * hcnt, uint32_t rows, uint32_t nq, uint32_t * total, hipStream_t s) {
	if (nq) hipLaunchKernelGGL(k_prefix, dim3((nq + 63) / 64), dim3(1024), 0, s, hcnt, rows, nq, total);
}

void mx_write_lists(const mx_args & a, hipStream_t s) {
	hipLaunchKernelGGL(k_write_lists, dim3(2048), dim3(256), 0, s, a.lists, a.n_lists, a.lists_cap, a.f, a.vals, a.vcap);
}

uint32_t mx_resident(int mode) {
	int n = 0;
	if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(kernel_of(mode)),
													MX_WAVES * 64, 0) !=
			hipSuccess || n < 1)
		n = 1;
	return std::min((uint32_t)(n * dev().num_cu), MX_MAX_GROUPS);
}

void mx_launch(const mx_args & a, int mode, uint32_t grid, hipStream_t s) {
	hipLaunchKernelGGL(kernel_of(mode), dim3(grid), dim3(MX_WAVES * 64), 0, s, a);
}

} // namespace tmx
