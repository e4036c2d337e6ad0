// xtn_plan.hpp -- how a search's deletion records are cut into the tiles and
// bins of xtn_tiles.hpp: host arithmetic over the counts of the sequences'
// lengths, without the device.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace xtn {

constexpr int MAX_PREFIX = 18;  // xtn.h:8 MAX_COMPRESSED_LENGTH

constexpr int TL_NT = 1024;
constexpr int TL_CAP_BITS = 15;
constexpr int TL_CAP = 1 << TL_CAP_BITS;  // records of a tile, at most
constexpr int TL_IT = TL_CAP / TL_NT;     // records of a thread
constexpr int TL_BINS_MAX = 8192;
constexpr int64_t TL_TILES_MAX = 65535, TL_SLOTS_MAX = ((int64_t)1 << 30) - 1;

// sequences a tile may hold and the bits of an index in it, by distance: the
// tables of a tile's sequences share LDS with its records
constexpr int tl_seqs(int d) { return d == 1 ? 4095 : d == 2 ? 768 : d == 3 ? 480 : 127; }
constexpr int tl_idx_bits(int d) { return d == 1 ? 12 : d == 2 ? 10 : d == 3 ? 9 : 7; }
// bits of a variant's length kept in its record: enough to tell d + 1
// numbers of deletions apart
constexpr int tl_len_bits(int d) { return d <= 3 ? 2 : 3; }

// threads of a bin's workgroup, two workgroups per CU (one's loads and
// barriers under the other's work: 430 us against 476 at 1M CDR3s, d = 2, for
// one of 1024 threads over half as many bins); the wide form takes the records
// that the narrow one would need too many bins for
constexpr int BIN_NT = 512, BIN_WIDE_NT = 1024;

inline int bits_for(int64_t maxval) {
	int b = 1;
	while (b < 62 && (1ll << b) <= maxval)
		++b;
	return b;
}

// sum_{k <= min(d, L)} C(L, k) by distance and length
struct VariantCounts {
	uint32_t v[MAX_PREFIX + 1][MAX_PREFIX + 1] = {};
	constexpr VariantCounts() {
		for (int d = 0; d <= MAX_PREFIX; ++d)
			for (int L = 0; L <= MAX_PREFIX; ++L) {
				uint64_t c = 1, total = 1;
				for (int j = 1; j <= d && j <= L; ++j) {
					c = c * (uint64_t)(L - j + 1) / (uint64_t)j;
					total += c;
				}
				v[d][L] = (uint32_t)total;  // at most 2^18
			}
	}
};

// the variants of the 18-residue prefix of a len-residue sequence (the count
// k_pack computes on the device)
inline uint64_t host_variant_count(uint32_t len, int d) {
	static constexpr VariantCounts counts;
	return counts.v[d < MAX_PREFIX ? d : MAX_PREFIX][len < (uint32_t)MAX_PREFIX ? len : (uint32_t)MAX_PREFIX];
}

// sequences by the length of their prefix
struct LenCounts {
	int64_t c[MAX_PREFIX + 1] = {};
	// the sum of every sequence's records, each counted as `least` or more
	int64_t records(int d, int64_t least) const {
		int64_t sum = 0;
		for (int L = 0; L <= MAX_PREFIX; ++L)
			sum += c[L] * std::max<int64_t>((int64_t)host_variant_count((uint32_t)L, d), least);
		return sum;
	}
};

struct TilePlan {
	uint32_t tile = 0;   // weight between the starts of two tiles
	uint32_t least = 0;  // a sequence weighs its records, or this where it has fewer
	int64_t ntiles = 0;
	int slot_bits = 0;  // of a tile's slots
	int bin_bits = 0;
	int idx_bits = 0;
	int bin_nt = BIN_NT, bin_groups = 18;  // the bin kernel's instantiation
	int pitch() const { return ((1 << bin_bits) + 64 + 63) / 64 * 64; }
	// slots, with room for the 16-byte read at the end of the last run
	size_t rec_bytes() const { return sizeof(uint32_t) * ((size_t)(ntiles << slot_bits) + 4); }
	size_t offs_bytes() const { return sizeof(uint16_t) * (size_t)(ntiles * pitch()); }
	int64_t cpitch() const { return (ntiles + 63) / 64 * 64; }
	size_t cols_bytes() const {
		return bin_groups == 3 ? 0 : sizeof(uint16_t) * (size_t)(((1 << bin_bits) + 1) * cpitch());
	}
};

// The tiling of n sequences of these lengths. A tile holds the sequences
// starting in its stretch of `tile` weight. A sequence weighs its records, and
// `least` where it has fewer, so that no stretch holds more sequences than a
// tile's tables and indexes take, in whatever order the lengths come, nor more
// records than `tile` and one sequence's. Cut by records alone, short strings
// standing together (rows sorted by length) outgrew a tile here and there: 1
// of 3840 tiles for 1M CDR3s at d = 2, which cost the whole run the tiles, 1.69
// ms instead of 0.90. Ordinary lengths weigh 0 to 2 % more than their records.
// tight: how often a bin of these rows has outgrown its slots; each time the
// bins get a fifth more room than their mean needs, and not the few slots.
inline TilePlan plan_tiles(const LenCounts& len, int64_t n, int d, int n_cu, int tight = 0) {
	const int64_t vmax = (int64_t)host_variant_count(MAX_PREFIX, d), most = TL_CAP - vmax;
	const int64_t V = len.records(d, 0);
	const double avg = (double)V / (double)n;
	// half as many sequences as the tables hold, on average, for uneven lengths
	const int64_t cap =
	    std::min(most, std::max<int64_t>(2048, (int64_t)std::min(0.5 * tl_seqs(d) * avg, (double)TL_CAP)));
	TilePlan p;
	int64_t tile = cap, W = V, least = 0;
	for (int step = 0; step < 4; ++step) {
		// whole rounds of one workgroup per CU
		const int64_t rounds = (W + n_cu * cap - 1) / (n_cu * cap);
		tile = std::min(cap, std::max<int64_t>((W + n_cu * rounds - 1) / (n_cu * rounds), 2048));
		// index bits for twice the average tile's sequences (at distance 4 a
		// short string has a tenth or less of the average's variants, so that
		// the few sequences of a tile vary more)
		p.idx_bits =
		    d >= 4 ? tl_idx_bits(d) : std::min(bits_for((int64_t)(2.0 * (double)tile / avg) + 1), tl_idx_bits(d));
		const int64_t limit = std::min(tl_seqs(d), (1 << p.idx_bits) - 1);
		least = (tile + limit - 1) / limit;
		const int64_t w = len.records(d, least);
		if (w == W)
			break;
		W = w;
	}
	p.tile = (uint32_t)tile;
	p.least = (uint32_t)least;
	p.ntiles = (W + tile - 1) / tile;
	if (W > (int64_t)INT32_MAX)
		p.ntiles = 0;  // the packing sums weights in 31 bits
	if (!p.ntiles)
		return p;
	p.slot_bits = bits_for(tile + vmax - 1);
	// a listed record keeps its tile in 16 bits, a group of records its first
	// slot in 30 (k_bins)
	if (p.ntiles > TL_TILES_MAX || p.ntiles << p.slot_bits > TL_SLOTS_MAX) {
		p.ntiles = 0;
		return p;
	}
	// The fewest bins whose runs fit the bin kernel's registers (a run, the
	// records that one tile has for one bin, is Poisson and takes a group per
	// four of them), and enough of them that bin and record leave 11 keys per
	// record: two records meet by chance once in 20 or so. They fit with a margin
	// of 3.5 % and of six standard deviations over the tiles' runs: the spread is
	// what counts for bins of few slots (177 000 CDR3s, d = 1: mean 1474 of 1536
	// groups, deviation 19, the fullest of 512 bins 1535).
	const double key_bits = std::log2((double)V) + 3.5;
	const double tile_recs = (double)V / (double)p.ntiles;
	// a bin for every resident workgroup of the narrow form (two per CU)
	// while they keep 512 records or more
	const int min_bits = std::max(6, std::min(9, bits_for(V / 512) - 1));
	auto bins_for = [&](int nt, int groups) {
		for (int bits = min_bits; (1 << bits) <= TL_BINS_MAX; ++bits) {
			const double lambda = tile_recs / (1 << bits);
			double q = 0, q2 = 0, w = std::exp(-lambda);  // a run's groups, and their squares
			if (lambda > 200) {
				q = lambda / 4 + 0.375;
				q2 = q * q + lambda / 16 + 0.08;
			} else {
				for (int k = 1; k < 400; ++k) {
					w *= lambda / k;
					q += w * ((k + 3) / 4);
					q2 += w * ((k + 3) / 4) * ((k + 3) / 4);
					if (k > lambda && w < 1e-12)
						break;
				}
			}
			const double mean = q * (double)p.ntiles, spread = std::sqrt((q2 - q * q) * (double)p.ntiles);
			const double room = nt * groups * (1.0 - 0.2 * tight);
			if (std::max(mean / 0.965, mean + 6.0 * spread) <= room && bits + 32 - tl_len_bits(d) - p.idx_bits >= key_bits)
				return bits;
		}
		return 0;
	};
	// The form of few slots where the fewest bins suffice.
	if (!tight && bins_for(BIN_NT, 3) == min_bits) {
		p.bin_bits = min_bits;
		p.bin_groups = 3;
		return p;
	}
	// The narrow form first; where its bins would leave runs of fewer than six
	// records, the wide one over half as many (at 1.15M CDR3s, d = 2: columns
	// 29 us and bins 656 us against 51 and 660; at 50 000, d = 4, 24 and 599
	// against 44 and 629); at distances 3 and 4 then the wide one of 18 groups,
	// whose list still takes a fifth of the records.
	const struct {
		int nt, groups;
	} forms[] = {{BIN_NT, d <= 2 ? 18 : 9}, {BIN_WIDE_NT, d <= 2 ? 18 : 9}, {BIN_WIDE_NT, 18}};
	for (const auto& f : forms) {
		const int bits = bins_for(f.nt, f.groups);
		if (!bits || (p.bin_bits && bits >= p.bin_bits))
			continue;
		p.bin_bits = bits;
		p.bin_nt = f.nt;
		p.bin_groups = f.groups;
		if (tile_recs / (1 << bits) >= 6.0)
			break;
	}
	if (!p.bin_bits)
		p.ntiles = 0;  // more records than the bins take
	return p;
}

}  // namespace xtn
