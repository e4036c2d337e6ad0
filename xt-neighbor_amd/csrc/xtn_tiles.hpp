// xtn_tiles.hpp -- the record path of one key-space chunk at distances 1 to 4:
// deletion variants generated once, ordered once, and grouped where they lie.
//
//   k_tiles / k_tiles1  a workgroup generates the deletion variants of a range of
//                sequences (a tile, at most TL_CAP records) and leaves them
//                in its slot of HBM ordered by bin, the top bin_bits of a
//                32-bit key; a record is four bytes, the rest of the key
//                above the sequence's index in the tile, since bin and tile
//                are given by where the record lies. The slot is written
//                front to back, so no workgroup claims space from another
//                and no store is scattered.
//   k_tile_cols  the tiles' bin starts, turned to one row per bin (a small input's
//                bins read the tiles' rows instead)
//   k_bins       a workgroup gathers a bin's runs from every tile into
//                registers and finds the records sharing a key: two bitmaps
//                in LDS leave those that may (about one in ten), a hash list
//                over these finds the pairs, and the pairs go out as
//                candidates
//
// Measured at 1M CDR3s, d = 2 (1.12e8 records): k_tiles 318 us (vector units
// busy 60% of the time, LDS 48%), k_tile_cols 25 us, k_bins 430 us (half of its
// wave cycles wait; vector and address units are busy 46% of the time, LDS
// 28%), against 465 + 427 + 298 us for the three kernels of the
// sub-range path; the candidates fall from 2.69M to 0.88M (tile_pair), which
// takes another 45 us off their sort. 10 000 CDR3s, d = 1 (160 003 records):
// tiles 9, bins 15 us.
// Per record this moves 4 bytes out and 4 back, against 8 out, 8 in, 8 out
// and 8 in for the sub-range path (k_gen<GEN_COARSE>, k_region_scatter,
// k_bucket), which stays for distances above 4, for fewer than 4096 records,
// for searches that ask for the separate pass, and for inputs with a group of
// more than TL_GROUP_MAX equal keys: such a run raises coarse_ovf and is redone
// there. No order of the rows outgrows a tile (plan_tiles); a bin over its
// slots has the tiles planned again with more bins first.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "xtn_kernels.hpp"
#include "xtn_plan.hpp"

namespace xtn {

constexpr uint32_t TL_NONE = 0xFFFFFFFFu;  // no record (a tile's last index is never used)
// coarse_ovf where the only bound outgrown is a bin's slots: the tiles are
// planned again with more bins
constexpr uint32_t TL_BIN_FULL = 2;
// equal keys before a record: a longer group is left to the run kernels, which
// spread its pairs over the chip (one string 1100 times among 300 000 rows, d =
// 1: 10.8 ms there)
constexpr int TL_GROUP_MAX = 1024;
// the same for the 18-group form without rounds: a longer group costs its
// workgroup 16 us or more (8 ns a pair), and the form with parts takes it
constexpr int TL_GROUP_LONG = 64;

constexpr int TL_MAX_D = 4;  // at 5 half of the records are listed and the bins go in parts: 2.4 ms against
                             // 2.0 for 9000 CDR3s on the sub-range path
constexpr int DEL_SETS4 = DEL_SETS3 + 3060;
__host__ __device__ constexpr int tl_sets(int d) {
	return d == 1 ? DEL_SETS1 : d == 2 ? DEL_SETS2 : d == 3 ? DEL_SETS3 : DEL_SETS4;
}

// The key of a variant is the exclusive or of one random word per slot and
// residue (tabulation hashing: Zobrist 1970, Carter and Wegman 1979). A
// deletion moves every later slot down one place, so with
// P_k[q] = xor over i < q of term(i - k, residue i) the variant of a string of
// length L with slots q1 < ... < qm deleted has the key
//   A_1[q1] ^ ... ^ A_m[qm] ^ P_m[L],   A_k[q] = P_(k-1)[q] ^ P_k[q + 1]
// and A_k[none] = P_(k-1)[L] ^ P_k[L] lets every set of at most d deletions
// read exactly d words: no multiplication, no mixing step.
struct TileTerms {
	uint32_t t[MAX_PREFIX][32];
};

constexpr TileTerms make_tile_terms() {
	TileTerms r{};
	uint64_t s = 0x243F6A8885A308D3ull;
	for (int p = 0; p < MAX_PREFIX; ++p)
		for (int c = 1; c < 32; ++c) {  // SplitMix64 (Steele, Lea, Flood 2014); an empty slot adds nothing
			s += 0x9E3779B97F4A7C15ull;
			uint64_t z = s;
			z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
			z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
			r.t[p][c] = (uint32_t)((z ^ (z >> 31)) >> 32);
		}
	return r;
}

__constant__ TileTerms c_tile_terms = make_tile_terms();

__device__ __forceinline__ uint32_t set_term(uint64_t hw) {  // the query set's word
	uint32_t x = (uint32_t)(hw >> PK_SET_SHIFT) & PK_SET_MASK;
	x = (x ^ (x >> 16)) * 0x85EBCA6Bu;
	x = (x ^ (x >> 13)) * 0xC2B2AE35u;
	return x ^ (x >> 16);
}

struct TileArgs {
	const uint64_t* pk;
	const uint64_t* voff;
	const uint32_t* first;   // first sequence of each tile, [ntiles] = n (k_pack_scan)
	uint32_t* out;           // 2^slot_bits slots per tile
	uint16_t* offs;          // a row of `pitch` per tile: the start of each bin, then the tile's total
	unsigned long long* ovf;
	int32_t pitch;
	int32_t bin_bits;        // 6..13
	int32_t lb;              // index bits of a record
	int32_t sets;            // the prefixes carry query sets
	int32_t repeats;         // repeated variants too (the search in static scratch, which counts them)
	uint32_t n;              // sequences
	int32_t slot_bits;       // a tile's slots, at most TL_CAP
};

// A record: key bits below the bin, the low bits of the variant's length, the
// index in the tile. Equal keys mean equal records above the index.
template <int D>
__device__ __forceinline__ uint32_t tile_record(uint32_t h, int bin_bits, uint32_t len, int lb, uint32_t idx) {
	constexpr uint32_t LM = (1u << tl_len_bits(D)) - 1u;
	return ((h << bin_bits) & ~(((LM + 1u) << lb) - 1u)) | ((len & LM) << lb) | idx;
}

// The deletion sets of at most 2, 3 and 4 positions, ordered by their largest
// position as c_del_tables is: positions ascending, five bits each from bit 0,
// NO_DEL above the real ones, the number of deletions from bit 25. In global
// memory: each workgroup copies its distance's to LDS once.
struct TileDelSets {
	uint32_t d2[DEL_SETS2], d3[DEL_SETS3], d4[DEL_SETS4];
};

constexpr uint32_t tile_del_entry(int m, int a, int b, int c, int d) {
	return (uint32_t)a | ((uint32_t)b << 5) | ((uint32_t)c << 10) | ((uint32_t)d << 15) | ((uint32_t)m << 25);
}

constexpr TileDelSets make_tile_del_sets() {
	TileDelSets t{};
	constexpr int N = NO_DEL;
	t.d2[0] = t.d3[0] = t.d4[0] = tile_del_entry(0, N, N, N, N);
	int q2 = 1, q3 = 1, q4 = 1;
	for (int m = 0; m < MAX_PREFIX; ++m) {
		t.d2[q2++] = t.d3[q3++] = t.d4[q4++] = tile_del_entry(1, m, N, N, N);
		for (int k = 0; k < m; ++k) {
			t.d2[q2++] = t.d3[q3++] = t.d4[q4++] = tile_del_entry(2, k, m, N, N);
			for (int j = 0; j < k; ++j) {
				t.d3[q3++] = t.d4[q4++] = tile_del_entry(3, j, k, m, N);
				for (int i = 0; i < j; ++i)
					t.d4[q4++] = tile_del_entry(4, i, j, k, m);
			}
		}
	}
	return t;
}

__device__ const TileDelSets g_tile_del_sets = make_tile_del_sets();

// the bins' counts (16 bits each, two to a word) turned into their starts,
// also written to the tile's row; returns the total
__device__ __forceinline__ uint32_t tile_starts(uint32_t* s_cnt, int nb, uint16_t* row, uint32_t* s_tmp) {
	const int t = threadIdx.x;
	uint16_t* const c16 = reinterpret_cast<uint16_t*>(s_cnt);
	const int per = nb > TL_NT ? nb / TL_NT : 1;
	const int b0 = t * per;
	uint32_t sum = 0;
	if (b0 < nb)
		for (int i = 0; i < per; ++i)
			sum += c16[b0 + i];
	uint32_t total;
	uint32_t run = block_excl_scan<TL_NT>(sum, s_tmp, &total);
	if (b0 < nb)
		for (int i = 0; i < per; ++i) {
			const uint32_t c = c16[b0 + i];
			c16[b0 + i] = (uint16_t)run;
			run += c;
		}
	__syncthreads();
	uint32_t* const row32 = reinterpret_cast<uint32_t*>(row);
	for (int i = t; i < nb / 2; i += TL_NT)
		row32[i] = s_cnt[i];
	if (t == 0)
		row[nb] = (uint16_t)total;
	return total;
}

// the ordered tile from LDS to its slot
__device__ __forceinline__ void tile_out(const uint32_t* s_rec, uint32_t* slot, uint32_t total) {
	const uint4* src = reinterpret_cast<const uint4*>(s_rec);
	uint4* dst = reinterpret_cast<uint4*>(slot);
	for (uint32_t i = threadIdx.x; i < (total + 3) / 4; i += TL_NT)
		dst[i] = src[i];
}

// a tile that cannot be held: an empty row, and the run is redone elsewhere
__device__ __forceinline__ void tile_refuse(const TileArgs& a, uint16_t* row, int nb, bool flag) {
	for (int i = threadIdx.x; i <= nb; i += TL_NT)
		row[i] = 0;
	if (flag && threadIdx.x == 0)
		atomicOr(a.ovf, 1ull);
}

// Distances 2 to 4. The deletion sets of a prefix come in the order of
// their largest position, a thread takes consecutive records,
// and the record's rank inside its bin comes from the same LDS atomic that
// counts it; the records stay in registers until the tables are dead and
// the ordered tile takes their LDS. At distance 4 the colex unranking this
// replaces took 1615 us for 1.05e8 variants (50 000 CDR3s).
template <int D>
__global__ __launch_bounds__(TL_NT, 4) void k_tiles(TileArgs a) {
	static_assert(D >= 2 && D <= TL_MAX_D, "distance 1 has a kernel of its own");
	constexpr int SEQS = tl_seqs(D);
	constexpr int W = MAX_PREFIX + 1;            // words of one A_k
	constexpr int ST = D * W + (D & 1 ? 0 : 1);  // odd: the threads of a wave build side by side without bank conflicts
	constexpr int NSETS = tl_sets(D);
	__shared__ union {
		uint32_t rec[TL_CAP];
		struct {
			uint32_t terms[MAX_PREFIX][32];
			uint32_t del[NSETS];
			uint32_t tab[SEQS * ST];
			uint32_t info[SEQS];      // run_mask, the length above it
			uint16_t start[SEQS + 2];  // the sequence's first record in the tile
		} s;
	} u;
	__shared__ uint32_t s_cnt[TL_BINS_MAX / 2];
	__shared__ uint32_t s_tmp[TL_NT / WAVE + 1];
	static_assert(sizeof(u) == sizeof(u.rec), "the tables fit the records' LDS");
	static_assert(SEQS < (1 << tl_idx_bits(D)), "the last index stays free");

	const int t = threadIdx.x;
	const int64_t tile = blockIdx.x;
	const int nb = 1 << a.bin_bits;
	uint16_t* const row = a.offs + tile * a.pitch;
	const uint32_t s0 = a.first[tile], s1 = a.first[tile + 1];
	const int cnt = (int)(s1 - s0);
	const int most = SEQS < (1 << a.lb) - 1 ? SEQS : (1 << a.lb) - 1;
	if (cnt <= 0 || cnt > most || s1 > a.n) {  // uniform (past n: a packing that gave up left the table undone)
		tile_refuse(a, row, nb, cnt > 0);  // (the tiling leaves a tile no more than its limit)
		return;
	}
	const uint64_t v0 = a.voff[s0];
	const uint32_t total = (uint32_t)(a.voff[s1] - v0);
	if (total > 1u << a.slot_bits) {  // uniform; the tiling rules it out
		tile_refuse(a, row, nb, true);
		return;
	}
	for (int i = t; i < nb / 2; i += TL_NT)
		s_cnt[i] = 0;
	for (int i = t; i < MAX_PREFIX * 32; i += TL_NT)
		(&u.s.terms[0][0])[i] = (&c_tile_terms.t[0][0])[i];
	const uint32_t* const del = D == 2 ? g_tile_del_sets.d2 : D == 3 ? g_tile_del_sets.d3 : g_tile_del_sets.d4;
	for (int i = t; i < NSETS; i += TL_NT)
		u.s.del[i] = del[i];
	__syncthreads();
	for (int i = t; i < cnt; i += TL_NT) {
		const uint64_t lo = a.pk[2 * (int64_t)(s0 + i)];
		const uint64_t hw = a.pk[2 * (int64_t)(s0 + i) + 1];
		u.s.start[i] = (uint16_t)(a.voff[s0 + i] - v0);
		const uint32_t hi26 = (uint32_t)hw & PK_SLOT_HI_MASK;
		uint32_t* const tab = &u.s.tab[i * ST];
		uint32_t pre[D + 1], a1[MAX_PREFIX];
#pragma unroll
		for (int k = 0; k <= D; ++k)
			pre[k] = 0;
#pragma unroll
		for (int q = 0; q < MAX_PREFIX; ++q) {
			const uint32_t c = slot_of(lo, hi26, q);
			uint32_t nxt[D + 1];
#pragma unroll
			for (int k = 0; k <= D; ++k)
				nxt[k] = q >= k ? pre[k] ^ u.s.terms[q - k][c] : 0u;
			a1[q] = pre[0] ^ nxt[1];
#pragma unroll
			for (int k = 2; k <= D; ++k)
				tab[(k - 1) * W + q] = pre[k - 1] ^ nxt[k];
#pragma unroll
			for (int k = 0; k <= D; ++k)
				pre[k] = nxt[k];
		}
		const uint32_t base = pre[D] ^ (a.sets ? set_term(hw) : 0u);
#pragma unroll
		for (int q = 0; q < MAX_PREFIX; ++q)
			tab[q] = a1[q] ^ base;
		tab[NO_DEL] = pre[0] ^ pre[1] ^ base;
#pragma unroll
		for (int k = 2; k <= D; ++k)
			tab[(k - 1) * W + NO_DEL] = pre[k - 1] ^ pre[k];
		u.s.info[i] = (a.repeats ? 0u : run_mask(lo, hw)) | ((uint32_t)(hw >> 56) << MAX_PREFIX);
	}
	if (t == 0)
		u.s.start[cnt] = (uint16_t)total;
	__syncthreads();

	uint32_t rec[TL_IT], at[TL_IT];  // at: bin, rank in it
	const int per = (int)((total + TL_NT - 1) / TL_NT);
	uint32_t r = (uint32_t)(t * per);
	int idx = 0;
	uint32_t k = 0, nv = 0, info = 0;
	if (r < total) {  // the sequence holding record r: the last one starting at or before it
		int lo = 0, hi = cnt - 1;
		while (lo < hi) {
			const int mid = (lo + hi + 1) >> 1;
			if (u.s.start[mid] <= r)
				lo = mid;
			else
				hi = mid - 1;
		}
		idx = lo;
		k = r - u.s.start[idx];
		nv = (uint32_t)u.s.start[idx + 1] - u.s.start[idx];
		info = u.s.info[idx];
	}
#pragma unroll
	for (int it = 0; it < TL_IT; ++it) {
		rec[it] = 0;
		at[it] = TL_NONE;
		if (it < per) {  // uniform
			if (r + it < total) {
				const uint32_t e = u.s.del[k];
				const uint32_t* tab = &u.s.tab[idx * ST];
				uint32_t h = 0, gone = 0;
#pragma unroll
				for (int j = 0; j < D; ++j) {
					const uint32_t q = (e >> (5 * j)) & 31u;
					h ^= tab[j * W + q];
					gone |= 1u << q;
				}
				// repeated variants left out as dup_deletion_set does (NO_DEL
				// lies on the first length bit: masked)
				if ((gone & info & ~(gone << 1) & ((1u << MAX_PREFIX) - 1u)) == 0u) {
					const uint32_t bin = h >> (32 - a.bin_bits);
					const int sh = (int)(bin & 1u) * 16;
					const uint32_t old = atomicAdd(&s_cnt[bin >> 1], 1u << sh);
					at[it] = (bin << 16) | ((old >> sh) & 0xFFFFu);
					rec[it] = tile_record<D>(h, a.bin_bits, (info >> MAX_PREFIX) - (e >> 25), a.lb, (uint32_t)idx);
				}
				if (++k == nv && idx + 1 < cnt) {
					++idx;
					k = 0;
					nv = (uint32_t)u.s.start[idx + 1] - u.s.start[idx];
					info = u.s.info[idx];
				}
			}
		}
	}
	__syncthreads();
	const uint32_t kept = tile_starts(s_cnt, nb, row, s_tmp);
	const uint16_t* const c16 = reinterpret_cast<const uint16_t*>(s_cnt);
#pragma unroll
	for (int it = 0; it < TL_IT; ++it)
		if (at[it] != TL_NONE)
			u.rec[c16[at[it] >> 16] + (at[it] & 0xFFFFu)] = rec[it];
	__syncthreads();
	tile_out(u.rec, a.out + (tile << a.slot_bits), kept);
}

// Distance 1: a thread takes whole sequences and steps the key from one
// deleted slot to the next (two terms change), once to count the bins and
// once more to place the records: no tables, and a tile of short strings
// holds as many sequences as its index bits name. Every variant is kept.
__global__ __launch_bounds__(TL_NT, 4) void k_tiles1(TileArgs a) {
	__shared__ uint32_t s_rec[TL_CAP];
	__shared__ uint32_t s_cnt[TL_BINS_MAX / 2];
	__shared__ uint32_t s_terms[MAX_PREFIX][32];
	__shared__ uint32_t s_tmp[TL_NT / WAVE + 1];
	const int t = threadIdx.x;
	const int64_t tile = blockIdx.x;
	const int nb = 1 << a.bin_bits;
	uint16_t* const row = a.offs + tile * a.pitch;
	const uint32_t s0 = a.first[tile], s1 = a.first[tile + 1];
	const int cnt = (int)(s1 - s0);
	if (cnt <= 0 || cnt > (1 << a.lb) - 1 || s1 > a.n) {  // uniform
		tile_refuse(a, row, nb, cnt > 0);
		return;
	}
	if (a.voff[s1] - a.voff[s0] > 1ull << a.slot_bits) {  // uniform; the tiling rules it out
		tile_refuse(a, row, nb, true);
		return;
	}
	for (int i = t; i < nb / 2; i += TL_NT)
		s_cnt[i] = 0;
	for (int i = t; i < MAX_PREFIX * 32; i += TL_NT)
		(&s_terms[0][0])[i] = (&c_tile_terms.t[0][0])[i];
	__syncthreads();
	auto variants = [&](auto&& put) {
		for (int i = t; i < cnt; i += TL_NT) {
			const uint64_t lo = a.pk[2 * (int64_t)(s0 + i)];
			const uint64_t hw = a.pk[2 * (int64_t)(s0 + i) + 1];
			const uint32_t hi26 = (uint32_t)hw & PK_SLOT_HI_MASK;
			const int L = (int)(hw >> 56);
			uint32_t c[MAX_PREFIX + 1];
			c[MAX_PREFIX] = 0;
			uint32_t full = a.sets ? set_term(hw) : 0u, h = full;
#pragma unroll
			for (int q = 0; q < MAX_PREFIX; ++q) {
				c[q] = slot_of(lo, hi26, q);
				full ^= s_terms[q][c[q]];
				if (q > 0)
					h ^= s_terms[q - 1][c[q]];
			}
			put(full, (uint32_t)L, (uint32_t)i);
#pragma unroll
			for (int q = 0; q < MAX_PREFIX; ++q)
				if (q < L) {
					put(h, (uint32_t)L - 1u, (uint32_t)i);
					h ^= s_terms[q][c[q]] ^ s_terms[q][c[q + 1]];
				}
		}
	};
	variants([&](uint32_t h, uint32_t, uint32_t) {
		const uint32_t bin = h >> (32 - a.bin_bits);
		atomicAdd(&s_cnt[bin >> 1], 1u << ((bin & 1u) * 16));
	});
	__syncthreads();
	const uint32_t total = tile_starts(s_cnt, nb, row, s_tmp);
	__syncthreads();  // the row is out before the starts become cursors
	variants([&](uint32_t h, uint32_t len, uint32_t idx) {
		const uint32_t bin = h >> (32 - a.bin_bits);
		const int sh = (int)(bin & 1u) * 16;
		const uint32_t pos = (atomicAdd(&s_cnt[bin >> 1], 1u << sh) >> sh) & 0xFFFFu;
		s_rec[pos] = tile_record<1>(h, a.bin_bits, len, a.lb, idx);
	});
	__syncthreads();
	tile_out(s_rec, a.out + (tile << a.slot_bits), total);
}

// The tiles' rows of bin starts to one row per bin, [nb + 1][cpitch], in
// blocks of 64 x 64; columns past the last tile read as 0. n_rec: the
// records of all tiles (the last bin row holds the tiles' totals).
__global__ __launch_bounds__(256) void k_tile_cols(const uint16_t* __restrict__ offs, int64_t ntiles, int nb, int pitch,
                                                   uint16_t* __restrict__ cols, int64_t cpitch,
                                                   unsigned long long* __restrict__ n_rec) {
	__shared__ uint32_t s_w[64][33];
	const int t = threadIdx.x;
	const int64_t tile0 = (int64_t)blockIdx.x * 64;
	const int bin0 = (int)blockIdx.y * 64;
	const uint32_t* const in = reinterpret_cast<const uint32_t*>(offs);
	for (int k = t; k < 64 * 32; k += 256) {
		const int r = k / 32, w = k % 32;
		s_w[r][w] = tile0 + r < ntiles ? in[((tile0 + r) * pitch + bin0) / 2 + w] : 0u;
	}
	__syncthreads();
	uint32_t* const out = reinterpret_cast<uint32_t*>(cols);
	for (int k = t; k < 64 * 32; k += 256) {
		const int b = k / 32, w = k % 32;  // bin0 + b, tiles tile0 + 2w and the next
		const uint32_t x = s_w[2 * w][b / 2], y = s_w[2 * w + 1][b / 2];
		const int sh = (b & 1) * 16;
		if (bin0 + b <= nb)
			out[((int64_t)(bin0 + b) * cpitch + tile0) / 2 + w] = ((x >> sh) & 0xFFFFu) | (((y >> sh) & 0xFFFFu) << 16);
	}
	if (bin0 <= nb && nb < bin0 + 64 && t < WAVE) {
		const int b = nb - bin0;
		unsigned long long c = (s_w[t][b / 2] >> ((b & 1) * 16)) & 0xFFFFu;
		for (int o = WAVE / 2; o > 0; o >>= 1)
			c += __shfl_xor(c, o);
		if (t == 0)
			atomicAdd(n_rec, c);
	}
}

// ------------------------------------------------------------- pairs --

struct BinArgs {
	const uint32_t* rec;     // the tiles
	const uint16_t* cols;    // k_tile_cols
	const uint32_t* first;
	const uint64_t* pk;
	int64_t ntiles, cpitch;
	const uint16_t* offs;    // the tiles' own rows, `pitch` apart (groups 3, which has no cols)
	int32_t pitch;
	int32_t slot_bits;       // a tile's
	int32_t nb;
	int32_t nt, groups;      // the instantiation: BIN_NT or BIN_WIDE_NT threads, 18, 9 or 3 groups each
	int32_t lb;              // index bits of a record
	int32_t len_bits;        // length bits above them
	int32_t key_low;         // lowest key bit of a record (above it the key's bits below the bin; zeros may lie
	                         // between it and the length bits)
	int32_t idb;
	int32_t distance;
	uint32_t id_lo, id_hi;   // only pairs whose smaller id lies in [id_lo, id_hi)
	uint64_t* pairs;
	int64_t pcap;
	RunCtrs* ctr;            // n_cand; n_records (groups 3); pairs_small: record pairs of equal key; n_big set when a bin lists more
	                         // records than fit, coarse_ovf when it outgrows another bound
};

// the residues present in a packed prefix, a bit per code
__device__ __forceinline__ uint32_t residue_set(uint64_t lo, uint32_t hi26) {
	uint32_t m = 0;
#pragma unroll
	for (int q = 0; q < MAX_PREFIX; ++q)
		m |= 1u << slot_of(lo, hi26, q);
	return m & ~1u;  // code 0: past the end
}

// Two sequences whose records share a key: whether they go out as a candidate
// pair. Each deletion takes at most one residue out of a string's set of
// residues, so sets further apart than the two sides' deletions show that
// only the keys met (bin and record together keep at most 32 bits of the key,
// about 11 keys for each record, so one record in 20 or so meets another by
// chance). Two prefixes within one edit of each other share a variant
// for every further deletion as well (about a dozen at distance 2, a hundred
// at 3): the pair goes out only from the variant with the fewest deletions, which
// both sides hold and whose length is known from the two strings.
__device__ __forceinline__ bool tile_pair(uint64_t la, uint64_t wa, uint64_t lb, uint64_t wb, uint32_t len,
                                          int len_bits, int distance) {  // (the two packed prefixes)
	const uint32_t ha = (uint32_t)wa & PK_SLOT_HI_MASK, hb = (uint32_t)wb & PK_SLOT_HI_MASK;
	const int La = (int)(wa >> 56), Lb = (int)(wb >> 56);
	const int lm = (1 << len_bits) - 1;
	const int ma = (La - (int)len) & lm, mb = (Lb - (int)len) & lm;  // deletions on each side, at most the distance
	if (ma > distance || mb > distance || La - ma != Lb - mb)
		return false;
	if (__popc(residue_set(la, ha) ^ residue_set(lb, hb)) > ma + mb)
		return false;
	if (La - Lb > 1 || Lb - La > 1)
		return true;
	// residues shared from the front and from the back
	const u128 x = (((u128)ha << 64) | la), y = (((u128)hb << 64) | lb);
	const u128 f = x ^ y;
	const int m = La < Lb ? La : Lb;
	int front = m, back = m;
	if (f != 0) {
		const uint64_t fh = (uint64_t)(f >> 64), fl = (uint64_t)f;
		const int top = fh ? 63 - __clzll(fh) + 64 : 63 - __clzll(fl);  // highest differing bit, 89 at most
		const int c = (89 - top) / 5;
		front = c < m ? c : m;
	}
	const u128 g = (x >> (5 * (MAX_PREFIX - La))) ^ (y >> (5 * (MAX_PREFIX - Lb)));
	if (g != 0) {
		const uint64_t gl = (uint64_t)g;
		const int low = gl ? __ffsll((unsigned long long)gl) - 1 : 63 + __ffsll((unsigned long long)(uint64_t)(g >> 64));
		const int c = low / 5;
		back = c < m ? c : m;
	}
	if (La == Lb) {
		if (f == 0)
			return ma == 0;
		return front + back < La - 1 || ma == 1;
	}
	return front + back < m || (La > Lb ? ma : mb) == 1;
}

__device__ __forceinline__ bool tile_pair(const uint64_t* __restrict__ pk, uint32_t ia, uint32_t ib, uint32_t len,
                                          int len_bits, int distance) {
	return tile_pair(pk[2 * (int64_t)ia], pk[2 * (int64_t)ia + 1], pk[2 * (int64_t)ib], pk[2 * (int64_t)ib + 1], len,
	                 len_bits, distance);
}

typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));

// Bins over resident workgroups. NT threads hold QPT groups of four records
// each.
//   1. the runs of the bin (k_tile_cols' row and the next one) are listed as
//      groups of up to four records, and every group is loaded into
//      registers: each record is read once
//   2. every record sets its bit in the first bitmap; one that finds it set
//      sets the bit of its key in the second
//   3. the records whose bit in the second is set are listed (any two of
//      equal key are among them)
//   4. these go on hash lists, each walks the ones before it, and equal keys
//      of two sequences are candidate pairs (tile_pair)
// PARTS: a bin that lists more than SVC records (an input with many
// duplicates or neighbours) goes through the steps once per part of its
// records by their top key bits; without it such a bin raises n_big and the
// host runs the instantiation that has it, which the common case would pay for
// in registers (8% of the kernel).
// QPT 18: bins of up to 36864 slots, an eighth of whose records may be
// listed; QPT 9 (distances 3 and 4, where a neighbouring pair shares hundreds
// of variants): half as many slots and a list for half of their records.
// QPT 3: bins of up to 6144 slots of a small input, where the time is latency:
// less to clear and fewer rounds, every record may be listed, and the runs
// come from the tiles' own rows, a tile per thread (a few hundred lines per
// bin instead of a transposing launch). 160 003 records (10 000 CDR3s, d = 1):
// 15 us, with 18 groups 21 beside 7 of k_tile_cols.
template <int NT, int QPT, bool PARTS>
__global__ __launch_bounds__(NT, 4) void k_bins(BinArgs a) {
	constexpr int X = NT / BIN_NT;  // the wide form: everything twice, one workgroup per CU
	constexpr bool FEW = QPT == 3;
	constexpr bool ROUNDS = PARTS || FEW;
	constexpr int B1 = FEW ? 16 : 17 + X, B2 = B1 - 2, HBITS = (QPT == 18 ? 11 : 10) + X;
	static_assert((X == 1 || X == 2) && (QPT == 18 || QPT == 9 || FEW), "bitmaps of 7 bits or more and a quarter of that per record");
	static_assert(!FEW || !PARTS, "every record fits the list");
	constexpr int QCAP = NT * QPT;
	constexpr int SVC = QPT == 18 ? (1 << B1) / 8 / 6 / 64 * 64 : FEW ? QCAP * 4 : 7168 * X;  // records listed in step 3
	constexpr int HEADS = 1 << HBITS;
	constexpr int PLC = QPT == 18 ? (QCAP * 4 - HEADS * 4 - SVC * 2) / 4 : 1024 * X;
	static_assert(PLC >= NT, "room for pairs beside the lists");
	__shared__ union {
		uint32_t bm1[(1 << B1) / 32];
		struct {
			uint32_t rec[SVC];
			uint16_t tile[SVC];  // at most TL_TILES_MAX
		} sv;
	} u1;
	__shared__ uint32_t s_bm2[(1 << B2) / 32];
	__shared__ union {
		uint32_t list[QCAP];  // (first record << 2) | records - 1, slots below TL_SLOTS_MAX
		struct {
			uint32_t head[HEADS];
			uint32_t pl[PLC];     // two listed records of equal key
			uint16_t next[SVC];
		} g;
	} u2;
	__shared__ uint32_t s_tmp[NT / WAVE + 1];
	__shared__ unsigned long long s_base;
	__shared__ uint32_t s_nsv, s_npl;
	__shared__ int s_stop;
	static_assert(sizeof(u1) + sizeof(u2) + sizeof(s_bm2) <= 79 * 1024 * X, "two workgroups per CU");
	const int t = threadIdx.x;
	const int lane = lane_id();
	const int G = (int)gridDim.x;
	// neighbouring bins, which share cache lines of every tile, run on one
	// XCD at a time
	const bool by_xcd = G % 8 == 0 && a.nb % 8 == 0;
	const int step = by_xcd ? G / 8 : G;
	const int b_end = by_xcd ? (int)(blockIdx.x % 8 + 1) * (a.nb / 8) : a.nb;
	const int b_beg = by_xcd ? (int)(blockIdx.x % 8) * (a.nb / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
	const int s1 = 32 - B1 > a.key_low ? 32 - B1 : a.key_low;
	const uint32_t lmask = (1u << a.lb) - 1u;

	int lp = 0, part = 0;  // PARTS: part of 2^lp; the next bin starts with as many
	bool fresh = true;
	for (int b = b_beg; b < b_end;) {  // uniform
		if (!PARTS || fresh) {
			for (int i = t; i < (1 << B1) / 128; i += NT)
				reinterpret_cast<uint4*>(u1.bm1)[i] = make_uint4(0u, 0u, 0u, 0u);
			for (int i = t; i < (1 << B2) / 128; i += NT)
				reinterpret_cast<uint4*>(s_bm2)[i] = make_uint4(0u, 0u, 0u, 0u);
		}
		if (t == 0)
			s_nsv = s_npl = 0;
		if (ROUNDS && t == 0)
			s_stop = 0;
		// 1. eight tiles per thread and round
		constexpr int TR = FEW ? 1 : 8;
		uint32_t nq = 0;
		const uint16_t* const r0 = FEW ? a.offs + b : a.cols + (int64_t)b * a.cpitch;
		if (FEW && b == 0) {
			uint32_t c = 0;
			for (int64_t tile = t; tile < a.ntiles; tile += NT)
				c += a.offs[tile * a.pitch + a.nb];
			uint32_t tot;
			block_excl_scan<NT>(c, s_tmp, &tot);
			if (t == 0)
				atomicAdd(&a.ctr->n_records, (unsigned long long)tot);
		}
		for (int64_t tb = 0; tb < a.ntiles; tb += NT * TR) {
			const int64_t tile0 = tb + t * TR;
			uint32_t st[TR], n[TR], q = 0;
			if constexpr (FEW) {
				const bool in = tile0 < a.ntiles;
				st[0] = in ? r0[tile0 * a.pitch] : 0u;
				n[0] = in ? r0[tile0 * a.pitch + 1] - st[0] : 0u;
				q = (n[0] + 3) / 4;
			} else {
				uint4 x = make_uint4(0u, 0u, 0u, 0u), y = x;
				if (tile0 < a.cpitch) {
					x = *reinterpret_cast<const uint4*>(r0 + tile0);
					y = *reinterpret_cast<const uint4*>(r0 + a.cpitch + tile0);
				}
				const uint32_t xs[4] = {x.x, x.y, x.z, x.w}, ys[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
				for (int j = 0; j < TR; ++j) {
					st[j] = (xs[j / 2] >> (16 * (j & 1))) & 0xFFFFu;
					n[j] = ((ys[j / 2] >> (16 * (j & 1))) & 0xFFFFu) - st[j];
					q += (n[j] + 3) / 4;
				}
			}
			uint32_t tot;
			uint32_t pos = nq + block_excl_scan<NT>(q, s_tmp, &tot);
#pragma unroll
			for (int j = 0; j < TR; ++j) {
				uint32_t at = ((uint32_t)(tile0 + j) << a.slot_bits) + st[j];
				for (uint32_t left = n[j]; left > 0;) {
					const uint32_t c = left < 4u ? left : 4u;
					if (pos < (uint32_t)QCAP)
						u2.list[pos] = (at << 2) | (c - 1u);
					++pos;
					at += 4;
					left -= c;
				}
			}
			nq += (uint32_t)__builtin_amdgcn_readfirstlane((int)tot);
		}
		if (nq > (uint32_t)QCAP) {  // uniform
			if (t == 0)
				atomicOr(&a.ctr->coarse_ovf, (unsigned long long)TL_BIN_FULL);
			__syncthreads();
			b += step;
			continue;
		}
		__syncthreads();
		uint32_t e[QPT];
		u32x4u v[QPT];
#pragma unroll
		for (int k = 0; k < QPT; ++k) {
			const uint32_t i = (uint32_t)(k * NT + t);
			e[k] = i < nq ? u2.list[i] : TL_NONE;
		}
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int k = 0; k < QPT; ++k) {  // up to three records past a run's end are read too
			const uint32_t off = e[k] != TL_NONE ? e[k] & ~3u : 0u;
			v[k] = *reinterpret_cast<const u32x4u*>(reinterpret_cast<const char*>(a.rec) + off);
		}
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int k = 0; k < QPT; ++k) {
			const uint32_t c = e[k] == TL_NONE ? 0u : (e[k] & 3u) + 1u;
			v[k].x = c > 0 ? v[k].x : TL_NONE;
			v[k].y = c > 1 ? v[k].y : TL_NONE;
			v[k].z = c > 2 ? v[k].z : TL_NONE;
			v[k].w = c > 3 ? v[k].w : TL_NONE;
		}
		// 2.
		if (!PARTS || fresh) {
#pragma unroll
			for (int k = 0; k < QPT; ++k)
#pragma unroll
				for (int j = 0; j < 4; ++j) {
					const uint32_t r = v[k][j];
					if (r != TL_NONE) {
						const uint32_t x = r >> s1;
						const uint32_t old = atomicOr(&u1.bm1[x >> 5], 1u << (x & 31u));
						if ((old >> (x & 31u)) & 1u) {
							const uint32_t y = (r >> a.key_low) & ((1u << B2) - 1u);
							atomicOr(&s_bm2[y >> 5], 1u << (y & 31u));
						}
					}
				}
			__syncthreads();
		}
		// 3. (computed anew from the records: what step 2 found would take as
		// many registers as the records themselves)
		uint32_t hit[(QPT * 4 + 31) / 32];
#pragma unroll
		for (int k = 0; k < (QPT * 4 + 31) / 32; ++k)
			hit[k] = 0;
		uint32_t found = 0;
#pragma unroll
		for (int k = 0; k < QPT; ++k)
			asm volatile("" : "+v"(v[k]));
#pragma unroll
		for (int k = 0; k < QPT; ++k) {
			if (k % 2 == 0 && k > 0)  // eight reads in flight
				asm volatile("" : "+v"(hit[(k * 4 - 1) / 32]), "+v"(found));
#pragma unroll
			for (int j = 0; j < 4; ++j) {
				const uint32_t r = v[k][j];
				const uint32_t y = (r >> a.key_low) & ((1u << B2) - 1u);
				uint32_t on = r != TL_NONE ? (s_bm2[y >> 5] >> (y & 31u)) & 1u : 0u;
				if constexpr (PARTS)
					on = (r >> 1) >> (31 - lp) == (uint32_t)part ? on : 0u;
				hit[(k * 4 + j) / 32] |= on << ((k * 4 + j) % 32);
				found += on;
			}
		}
		const uint32_t inc = wave_incl_scan(found);
		uint32_t wbase = 0;
		if (lane == WAVE - 1 && inc)
			wbase = atomicAdd(&s_nsv, inc);
		uint32_t pos = (uint32_t)__shfl((int)wbase, WAVE - 1, WAVE) + inc - found;
#pragma unroll
		for (int k = 0; k < QPT; ++k) {
			if (((hit[k * 4 / 32] >> (k * 4 % 32)) & 15u) == 0u)
				continue;
			const uint16_t tile = (uint16_t)(u2.list[k * NT + t] >> (a.slot_bits + 2));
#pragma unroll
			for (int j = 0; j < 4; ++j)
				if ((hit[(k * 4 + j) / 32] >> ((k * 4 + j) % 32)) & 1u) {
					if (pos < (uint32_t)SVC) {
						u1.sv.rec[pos] = v[k][j];
						u1.sv.tile[pos] = tile;
					}
					++pos;
				}
		}
		__syncthreads();
		const uint32_t nsv = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_nsv);
		if (nsv > (uint32_t)SVC) {  // uniform
			__syncthreads();
			fresh = false;
			part = 0;
			if (!PARTS || lp == 6) {
				if (t == 0)
					atomicOr(PARTS ? &a.ctr->coarse_ovf : &a.ctr->n_big, 1ull);
				b += step;
				fresh = true;
			} else {
				++lp;  // the bin again in more parts
			}
			continue;
		}
		// 4.
		for (int i = t; i < HEADS; i += NT)
			u2.g.head[i] = 0xFFFFu;
		__syncthreads();
		for (uint32_t i = t; i < nsv; i += NT)
			u2.g.next[i] = (uint16_t)atomicExch(&u2.g.head[(u1.sv.rec[i] >> a.key_low) & (HEADS - 1)], i);
		__syncthreads();
		// Every record walks its list; the pairs that it finds go to a list in
		// LDS, which all threads evaluate. Where that list is full,
		//   - ROUNDS: a thread takes its walk up again after the pairs listed so
		//     far, so that the many pairs of a long group are not left to the
		//     threads that meet them, one dependent load after the other;
		//   - else it evaluates the pair itself, as long as no group is longer
		//     than TL_GROUP_LONG (with rounds the kernel holds more registers than
		//     the gather leaves: 447 us against 430 at 1M CDR3s, d = 2).
		// Resident searches with rounds against without: 10 copies of each of
		// 30 000 rows, d = 2, 7.5 ms against 40; 3 copies of 100 000 2.1 against
		// 7.9; one string 300 times among 300 000 rows, d = 1, 1.2 against 1.7.
		if constexpr (ROUNDS) {
			int u = t;  // kept from the compiler, which would hold what it makes of it in registers that the gather needs
			asm volatile("" : "+v"(u));
			constexpr int EV = FEW ? 1 : QPT == 18 ? 5 : 2;
			uint32_t i = u, n = 0xFFFFu, same = 0;
			bool mid = false;  // the walk of record i stands at link n
			bool checked = false;
			for (;;) {
				for (; i < nsv; i += NT) {
					const uint32_t r = u1.sv.rec[i];
					if (!mid) {
						n = u2.g.next[i];
						same = 0;
					}
					mid = false;
					while (n != 0xFFFFu) {
						const uint32_t rn = u1.sv.rec[n];  // record and link read together
						const uint32_t nn = u2.g.next[n];
						const uint32_t m = n;
						n = nn;
						if ((r ^ rn) >> a.lb)
							continue;
						const uint32_t q = atomicAdd(&s_npl, 1u);
						if (q >= (uint32_t)PLC) {
							n = m;
							mid = true;
							break;
						}
						u2.g.pl[q] = (i << 16) | m;
						if (++same >= (uint32_t)TL_GROUP_MAX) {
							atomicOr(&a.ctr->coarse_ovf, 1ull);
							break;
						}
					}
					if (mid)
						break;
				}
				__syncthreads();
				const uint32_t listed = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_npl);
				const uint32_t npl = listed < (uint32_t)PLC ? listed : (uint32_t)PLC;
				if (u == 0)
					atomicAdd(&a.ctr->pairs_small, (unsigned long long)npl);
				for (uint32_t q0 = 0; q0 < npl; q0 += EV * NT) {  // uniform
					uint32_t lo[EV], hi[EV], ok = 0;
					u64x2 pl[EV], ph[EV];
					uint32_t len[EV];
#pragma unroll
					for (int k = 0; k < EV; ++k)
						if (q0 + k * NT + u < npl) {
							const uint32_t w = u2.g.pl[q0 + k * NT + u];
							const uint32_t rx = u1.sv.rec[w >> 16], ry = u1.sv.rec[w & 0xFFFFu];
							const uint32_t x = a.first[u1.sv.tile[w >> 16]] + (rx & lmask);
							const uint32_t y = a.first[u1.sv.tile[w & 0xFFFFu]] + (ry & lmask);
							lo[k] = x < y ? x : y;
							hi[k] = x < y ? y : x;
							len[k] = (rx >> a.lb) & ((1u << a.len_bits) - 1u);
							if (x != y && lo[k] >= a.id_lo && lo[k] < a.id_hi) {
								ok |= 1u << k;
								pl[k] = reinterpret_cast<const u64x2*>(a.pk)[lo[k]];
								ph[k] = reinterpret_cast<const u64x2*>(a.pk)[hi[k]];
							}
						}
#pragma unroll
					for (int k = 0; k < EV; ++k)
						if (((ok >> k) & 1u) &&
						    !tile_pair(pl[k].x, pl[k].y, ph[k].x, ph[k].y, len[k], a.len_bits, a.distance))
							ok &= ~(1u << k);
					unsigned long long slot = block_append<NT>(&a.ctr->n_cand, (uint32_t)__popc(ok), s_tmp, &s_base);
#pragma unroll
					for (int k = 0; k < EV; ++k)
						if ((ok >> k) & 1u) {
							if ((int64_t)slot < a.pcap)
								a.pairs[slot] = ((uint64_t)lo[k] << a.idb) | hi[k];
							++slot;
						}
				}
				if (listed <= (uint32_t)PLC) {  // every walk is at its end
					__syncthreads();
					break;
				}
				if (!checked) {  // once: a group too long for the rounds is found before they are spent on it
					checked = true;
					for (uint32_t j = u; j < nsv; j += NT) {
						const uint32_t r = u1.sv.rec[j];
						int equal = 0;
						for (uint32_t m = u2.g.next[j]; m != 0xFFFFu; m = u2.g.next[m])
							equal += (r ^ u1.sv.rec[m]) >> a.lb == 0u;
						if (equal >= TL_GROUP_MAX) {
							atomicOr(&a.ctr->coarse_ovf, 1ull);
							s_stop = 1;
						}
					}
				}
				if (u == 0) {  // (s_npl read by all before the append's barriers)
					s_npl = 0;
					if (__hip_atomic_load(&a.ctr->coarse_ovf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
						s_stop = 1;  // another bin gave the run up
				}
				__syncthreads();
				if (__builtin_amdgcn_readfirstlane(s_stop)) {  // the run is redone elsewhere
					__syncthreads();
					break;
				}
			}
		} else {
			auto candidate = [&](uint32_t i, uint32_t n, uint64_t* p) -> bool {
				const uint32_t ri = u1.sv.rec[i], rn = u1.sv.rec[n];
				const uint32_t x = a.first[u1.sv.tile[i]] + (ri & lmask), y = a.first[u1.sv.tile[n]] + (rn & lmask);
				if (x == y)
					return false;
				const uint32_t lo = x < y ? x : y, hi = x < y ? y : x;
				if (lo < a.id_lo || lo >= a.id_hi)
					return false;
				*p = ((uint64_t)lo << a.idb) | hi;
				return tile_pair(a.pk, lo, hi, (ri >> a.lb) & ((1u << a.len_bits) - 1u), a.len_bits,
				                 a.distance);
			};
			for (uint32_t i = t; i < nsv; i += NT) {
				const uint32_t r = u1.sv.rec[i];
				uint32_t same = 0;
				for (uint32_t n = u2.g.next[i]; n != 0xFFFFu;) {
					const uint32_t rn = u1.sv.rec[n];  // record and link read together
					const uint32_t nn = u2.g.next[n];
					const uint32_t m = n;
					n = nn;
					if ((r ^ rn) >> a.lb)
						continue;
					const uint32_t q = atomicAdd(&s_npl, 1u);
					if (q < (uint32_t)PLC) {
						u2.g.pl[q] = (i << 16) | m;
					} else {
						uint64_t p;
						if (candidate(i, m, &p)) {
							const unsigned long long slot = atomicAdd(&a.ctr->n_cand, 1ull);
							if ((int64_t)slot < a.pcap)
								a.pairs[slot] = p;
						}
					}
					if (++same >= (uint32_t)(QPT == 18 ? TL_GROUP_LONG : TL_GROUP_MAX)) {
						atomicOr(QPT == 18 ? &a.ctr->n_big : &a.ctr->coarse_ovf, 1ull);
						break;
					}
				}
			}
			__syncthreads();
			uint32_t npl = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_npl);
			if (t == 0)
				atomicAdd(&a.ctr->pairs_small, (unsigned long long)npl);
			npl = npl < (uint32_t)PLC ? npl : (uint32_t)PLC;
			for (uint32_t q0 = 0; q0 < npl; q0 += NT) {  // uniform
				bool ok = false;
				uint64_t p = 0;
				if (q0 + t < npl) {
					const uint32_t w = u2.g.pl[q0 + t];
					ok = candidate(w >> 16, w & 0xFFFFu, &p);
				}
				const unsigned long long slot = block_append<NT>(&a.ctr->n_cand, ok ? 1u : 0u, s_tmp, &s_base);
				if (ok && (int64_t)slot < a.pcap)
					a.pairs[slot] = p;
			}
			__syncthreads();
		}
		fresh = false;
		if (!PARTS || ++part == 1 << lp) {
			part = 0;
			fresh = true;
			b += step;
		}
	}
}

}  // namespace xtn
