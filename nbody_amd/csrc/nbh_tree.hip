// nbh_tree.hip -- Barnes-Hut heap kd-tree on the GPU: exact build, refit and
// traversal (gfx950).
//
// Layout (nbody/nbody_space_heap.cpp:13-37): n = 2^L bodies, heap indices
// 1..2n-1 (root 1, children 2i and 2i+1, leaves at [n, 2n)).
//
// Build = the reference's recursive median split (nbody_space_heap.cpp:136-191)
// done level by level for every segment at once:
//   1. three stable LSD radix sorts give the bodies in x, y and z order (keys:
//      order-preserving 64-bit images of the FP64 coordinates; equal
//      coordinates keep index order);
//   2. at level l every segment of S = n >> l consecutive list entries holds the
//      bodies of one node; along axis a = l % 3 the first S/2 entries of the
//      a-sorted list are exactly the count/2 smallest, i.e. std::nth_element's
//      left part.  Each body is tagged left/right, and the two other lists are
//      stably partitioned inside every segment (counts of the tiles before + scatter), so
//      every child segment again holds its bodies sorted along all three axes;
//   3. after L levels entry s of any list is the body of leaf n + s;
//   4. moments bottom-up with the operations of nbody_space_heap::update
//      (:119-134), in FP64 with contraction off: bit-identical node records.
// Traversal: a wave walks for consecutive leaves of the heap (spatially coherent):
// 32 in the FP64 parity walk (k_bh_walk64), 64 in the FP32 group walks, up to 128 on the
// Morton tree; nodes as 32-byte records {cm.xyz, crit_r2} plus mass, or packed with the
// second moments in 64 bytes.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "nbh_common.h"
#include "nbh_f64.h"
#include "nbh_mlp_dev.h"

namespace {

constexpr int kRoot = 1;               // NBODY_HEAP_ROOT_INDEX
constexpr int kSortThreads = 512;
constexpr int kSortItems = 8;
constexpr int kSortTile = kSortThreads * kSortItems;   // 4096 keys per work-group
constexpr int kSortOneThreads = 1024;                  // up to 4096 keys sorted by one work-group
constexpr int kSortOneItems = kSortTile / kSortOneThreads;
constexpr int kSortSets = 3;                           // lists sorted together
constexpr int kSortPasses = 8;
constexpr int kPartThreads = 256;
constexpr int kPartItems = 4;
constexpr int kPartTile = kPartThreads * kPartItems;   // 1024 entries per work-group
constexpr size_t kPartSum = 4096;                    // tiles of a segment that a tile sums itself, without a scan
constexpr int kScanThreads = 256;
constexpr int kScanParts = 1024;                     // chunks of one scan
constexpr int kScanOneThreads = 1024;
constexpr int kScanOneItems = 16;                    // scans of up to 16384 counts in one work-group
constexpr int kLocalSeg = 4096;                      // segments split in LDS, one work-group each
constexpr int kLocalThreads = 1024;
constexpr int kBoxParts = 2048;                      // partial boxes of the Morton tree's bounding box
constexpr int kRadixTiers = 6;                       // sizes 64 * 32^t of the Morton tree's subtrees, t = 0..5
constexpr int kMarkParts = 1024;                     // runs of group mark words that are counted together

}  // namespace

// Node record of the group walks: what a walk step reads for one node, in 64
// bytes, so that a sibling pair (2i, 2i + 1) is one 128-byte cache line.
struct __align__(64) nbh_walk_rec {
	double4 c;      // cm.x, cm.y, cm.z, crit_r2 (as xyzr)
	double  m;      // mass
	float   q[6];   // second central moments xx yy zz xy xz yz (0 on leaves), rounded to float
};
static_assert(sizeof(nbh_walk_rec) == 64, "walk record must be 64 bytes");

struct nbh_tree {
	nbh_ctx*  ctx = nullptr;
	size_t    n = 0;
	int       levels = 0;
	// per-axis sorted body lists and scratch
	uint32_t* list[3] = {nullptr, nullptr, nullptr};
	uint32_t* tmp = nullptr;
	uint8_t*  side = nullptr;
	uint64_t* keys = nullptr;      // [2][n] radix sort ping-pong
	uint32_t* vals = nullptr;      // [2][n]
	uint32_t* counts = nullptr;    // radix / partition block counts
	uint32_t* scan_part = nullptr; // [kScanParts] chunk sums of a scan
	// nodes, heap index 0..2n-1 (0 unused)
	double4*  xyzr = nullptr;      // cm.x, cm.y, cm.z, crit_r2
	double*   mass = nullptr;
	double*   bmin = nullptr;      // [2n*3]
	double*   bmax = nullptr;      // [2n*3]
	double*   quad = nullptr;      // [2n*6] second central moments (0 on leaves)
	nbh_walk_rec* wrec = nullptr;  // [2n] packed copy for the group walks
	int32_t*  body_n = nullptr;    // -1 on internal nodes
	unsigned long long* counters = nullptr;   // [5] interactions, visits, stack spills, far cells, near cells
	// two-level local walk (allocated on first use): per super-group node lists,
	// their lengths and the super-group expansions
	int       two_cap = 0;           // list capacity per super-group (0: kTwoCap)
	int*      two_lists = nullptr;
	int*      two_count = nullptr;
	float*    two_coef = nullptr;
	// the super-groups' far cells for the learned correction (allocated on first use)
	int*      far_list = nullptr;
	int*      far_count = nullptr;
	// Morton radix tree (nbh_tree_build_radix; allocated on its first build)
	int2*     child = nullptr;     // [n] children of internal ids 1..n-1
	int*      parent = nullptr;    // [2n] parent id of every non-root node
	uint8_t*  tier = nullptr;      // [n] tier of internal ids (k_radix_nodes)
	int*      tier_list = nullptr; // [n + kRadixTiers] roots of the tiers' subtrees, tier by tier
	int2*     gmark = nullptr;     // [n] group marks at their first sorted leaf (build scratch)
	int2*     smark = nullptr;     // [n] super-group marks
	int2*     wmark = nullptr;     // [n] walk group marks
	uint32_t* marks = nullptr;     // mark_words(n): bits of the three kinds of marks, counts, then the info counts
	int4*     grp = nullptr;       // [n] build groups (node, first leaf, leaves)
	int4*     wgrp = nullptr;      // [n] walk groups (node, first leaf, leaves, super-group)
	int2*     sup = nullptr;       // [n / kRadixWalk + 1] super-groups (node, first leaf)
	double*   box = nullptr;       // [6 * (kBoxParts + 1)] partial boxes, then the bounding box
	double4*  pk = nullptr;        // [n] position and mass of each body, packed for the sorted gather
	int       ngroups = 0;         // build groups, walk groups and super-groups of the last Morton build
	int       nwalk = 0;
	int       nsupers = 0;
	int       tier_count[kRadixTiers] = {};   // subtrees of each tier of the last Morton build
	hipEvent_t info_ready = nullptr;          // the counts of a Morton build are in pinned memory
	int       two_slots = 0;       // super-groups the two-level buffers hold
	bool      radix = false;       // the last build made the Morton tree
	bool      radix_lean = false;  // Morton node arrays only where the build reads them back
	double    ratio = 0.0;         // opening ratio of the last build / refit
	bool      built = false;
};

namespace {

// ---------------------------------------------------------------------------
// radix sort of (64-bit key, 32-bit value), stable, 8 bits per pass
// ---------------------------------------------------------------------------
__device__ inline uint64_t order_key(double v)
{
	v = v + 0.0;                                   // -0 -> +0: equal values compare equal
	uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
	return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

// The buffers of one list to be sorted: pass p reads (k, v)[p % 2] and writes the
// other half; the last pass writes the values to `out`.
struct sort_list {
	uint64_t* k[2];
	uint32_t* v[2];
	uint32_t* out;
};
struct sort_lists {
	sort_list l[kSortSets];
};

// Scratch of one list's sort, in 32-bit words: per tile and digit a 64-bit status
// word (step << 32 | count), the counts of every digit of every pass and the
// tickets handed out in every pass.
struct sort_scratch {
	unsigned long long* status;
	uint32_t* hist;
	uint32_t* ticket;
};

constexpr size_t sort_words(size_t tiles)
{
	return tiles * 256 * 2 + kSortPasses * 256 + kSortPasses;
}

__device__ inline sort_scratch sort_scratch_of(uint32_t* words, int set, size_t tiles)
{
	uint32_t* w = words + static_cast<size_t>(set) * sort_words(tiles);
	sort_scratch s;
	s.status = reinterpret_cast<unsigned long long*>(w);
	s.hist = w + tiles * 512;
	s.ticket = s.hist + kSortPasses * 256;
	return s;
}

// Keys and body numbers of the three coordinate lists (blockIdx.y), and their
// sorts' scratch cleared.
__global__ void __launch_bounds__(256)
k_make_keys(const double* __restrict__ y, sort_lists a, size_t n, uint32_t* __restrict__ scratch, size_t words)
{
	const double* coord = y + static_cast<size_t>(blockIdx.y) * n;
	uint64_t* keys = a.l[blockIdx.y].k[0];
	uint32_t* vals = a.l[blockIdx.y].v[0];
	const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
	const size_t first = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
	for(size_t i = first; i < n; i += stride)
	{
		keys[i] = order_key(coord[i]);
		vals[i] = static_cast<uint32_t>(i);
	}
	for(size_t i = first; i < words; i += stride) { scratch[blockIdx.y * words + i] = 0; }
}

// Counts of the digits of all passes, once over the keys (their multiset does not
// change from pass to pass).
__global__ void __launch_bounds__(kSortThreads)
k_sort_hist(sort_lists a, size_t n, int passes, uint32_t* __restrict__ scratch, size_t tiles)
{
	__shared__ uint32_t h[kSortPasses][256];
	const uint64_t* keys = a.l[blockIdx.y].k[0];
	for(int i = threadIdx.x; i < passes * 256; i += kSortThreads) { (&h[0][0])[i] = 0; }
	__syncthreads();
	const size_t stride = static_cast<size_t>(gridDim.x) * kSortThreads;
	for(size_t i = static_cast<size_t>(blockIdx.x) * kSortThreads + threadIdx.x; i < n; i += stride)
	{
		const uint64_t k = keys[i];
		for(int p = 0; p < passes; ++p) { atomicAdd(&h[p][(k >> (8 * p)) & 0xFF], 1u); }
	}
	__syncthreads();
	const sort_scratch s = sort_scratch_of(scratch, blockIdx.y, tiles);
	for(int i = threadIdx.x; i < passes * 256; i += kSortThreads)
	{
		const uint32_t c = (&h[0][0])[i];
		if(c != 0) { atomicAdd(&s.hist[i], c); }
	}
}

// Exclusive prefix sum over the first 256 work-items of a group (the others pass
// anything); ws: four words of LDS.
__device__ inline uint32_t scan256(uint32_t v, uint32_t* ws)
{
	const int lane = threadIdx.x & 63;
	const int wave = threadIdx.x >> 6;
	uint32_t x = v;
	for(int off = 1; off < 64; off <<= 1)
	{
		const uint32_t u = __shfl_up(x, off, 64);
		if(lane >= off) { x += u; }
	}
	if(lane == 63 && wave < 4) { ws[wave] = x; }
	__syncthreads();
	uint32_t ex = x - v;
	for(int w = 0; w < 4; ++w) { ex += w < wave ? ws[w] : 0; }
	__syncthreads();
	return ex;
}

// The lanes of the wave whose digit equals this one's.
__device__ inline uint64_t digit_peers(uint32_t d, bool ok)
{
	uint64_t peers = __ballot(ok);
#pragma unroll
	for(int bit = 0; bit < 8; ++bit)
	{
		const uint64_t bal = __ballot((d >> bit) & 1u);
		peers &= ((d >> bit) & 1u) ? bal : ~bal;
	}
	return peers;
}

// Ranks a tile's keys stably by digit, each wave its own run of keys with its own
// counters (no work-group synchronisation between rows): rank[] within the wave's
// keys of that digit.  counts[wave][256] end as the waves' digit counts.
template <int kItems>
__device__ inline void rank_tile(const uint64_t (&key)[kItems], const bool (&ok)[kItems], int shift,
                                 uint32_t* __restrict__ counts, uint32_t (&rank)[kItems])
{
	const int lane = threadIdx.x & 63;
	const uint64_t lt_mask = lane == 0 ? 0ull : ~0ull >> (64 - lane);
#pragma unroll
	for(int k = 0; k < kItems; ++k)
	{
		const uint32_t d = static_cast<uint32_t>((key[k] >> shift) & 0xFF);
		const uint64_t peers = digit_peers(d, ok[k]);
		const uint32_t before = ok[k] ? counts[d] : 0;
		rank[k] = before + static_cast<uint32_t>(__popcll(peers & lt_mask));
		__builtin_amdgcn_wave_barrier();
		if(ok[k] && (peers & lt_mask) == 0) { counts[d] = before + static_cast<uint32_t>(__popcll(peers)); }
		__builtin_amdgcn_wave_barrier();
	}
}

// Exclusive scan in place of `m` uint32 counts: chunk sums, a scan of the (at
// most kScanParts) chunk sums, then a scan of every chunk from its offset.
__global__ void __launch_bounds__(kScanThreads)
k_scan_reduce(const uint32_t* __restrict__ c, size_t m, size_t chunk, uint32_t* __restrict__ part)
{
	__shared__ uint32_t ws[kScanThreads / 64];
	const size_t b0 = static_cast<size_t>(blockIdx.x) * chunk;
	const size_t b1 = b0 + chunk < m ? b0 + chunk : m;
	uint32_t s = 0;
	for(size_t i = b0 + threadIdx.x; i < b1; i += kScanThreads) { s += c[i]; }
	for(int off = 32; off > 0; off >>= 1) { s += __shfl_down(s, off, 64); }
	if((threadIdx.x & 63) == 0) { ws[threadIdx.x >> 6] = s; }
	__syncthreads();
	if(threadIdx.x == 0)
	{
		uint32_t t = 0;
		for(int w = 0; w < kScanThreads / 64; ++w) { t += ws[w]; }
		part[blockIdx.x] = t;
	}
}

__global__ void __launch_bounds__(kScanParts)
k_scan_parts(uint32_t* __restrict__ part, int g)
{
	__shared__ uint32_t sh[kScanParts];
	const uint32_t v = static_cast<int>(threadIdx.x) < g ? part[threadIdx.x] : 0;
	sh[threadIdx.x] = v;
	__syncthreads();
	for(int off = 1; off < kScanParts; off <<= 1)
	{
		const uint32_t u = threadIdx.x >= static_cast<unsigned>(off) ? sh[threadIdx.x - off] : 0;
		__syncthreads();
		sh[threadIdx.x] += u;
		__syncthreads();
	}
	if(static_cast<int>(threadIdx.x) < g) { part[threadIdx.x] = sh[threadIdx.x] - v; }
}

__global__ void __launch_bounds__(kScanThreads)
k_scan_apply(uint32_t* __restrict__ c, size_t m, size_t chunk, const uint32_t* __restrict__ part)
{
	constexpr int kWaves = kScanThreads / 64;
	__shared__ uint32_t ws[kWaves];
	const int lane = threadIdx.x & 63;
	const int wave = threadIdx.x >> 6;
	uint32_t carry = part[blockIdx.x];
	const size_t b0 = static_cast<size_t>(blockIdx.x) * chunk;
	const size_t b1 = b0 + chunk < m ? b0 + chunk : m;
	for(size_t t0 = b0; t0 < b1; t0 += 4 * kScanThreads)
	{
		const size_t i0 = t0 + 4 * static_cast<size_t>(threadIdx.x);
		uint32_t v[4];
		for(int k = 0; k < 4; ++k) { v[k] = i0 + k < b1 ? c[i0 + k] : 0; }
		const uint32_t tsum = v[0] + v[1] + v[2] + v[3];
		uint32_t x = tsum;
		for(int off = 1; off < 64; off <<= 1)
		{
			const uint32_t u = __shfl_up(x, off, 64);
			if(lane >= off) { x += u; }
		}
		if(lane == 63) { ws[wave] = x; }
		__syncthreads();
		uint32_t wbase = 0, total = 0;
		for(int w = 0; w < kWaves; ++w)
		{
			wbase += w < wave ? ws[w] : 0;
			total += ws[w];
		}
		uint32_t run = carry + wbase + x - tsum;
		for(int k = 0; k < 4; ++k)
		{
			if(i0 + k < b1) { c[i0 + k] = run; }
			run += v[k];
		}
		carry += total;
		__syncthreads();
	}
}

// Exclusive scan in place of m <= kScanOneThreads * kScanOneItems counts by one
// work-group: each work-item scans a run of consecutive counts.
__global__ void __launch_bounds__(kScanOneThreads)
k_scan_one(uint32_t* __restrict__ c, int m)
{
	__shared__ uint32_t ws[kScanOneThreads / 64];
	const int lane = threadIdx.x & 63;
	const int wave = threadIdx.x >> 6;
	const int per = (m + kScanOneThreads - 1) / kScanOneThreads;
	const int i0 = static_cast<int>(threadIdx.x) * per;
	uint32_t v[kScanOneItems];
	uint32_t s = 0;
#pragma unroll
	for(int k = 0; k < kScanOneItems; ++k)
	{
		v[k] = k < per && i0 + k < m ? c[i0 + k] : 0;
		s += v[k];
	}
	uint32_t x = s;
	for(int off = 1; off < 64; off <<= 1)
	{
		const uint32_t u = __shfl_up(x, off, 64);
		if(lane >= off) { x += u; }
	}
	if(lane == 63) { ws[wave] = x; }
	__syncthreads();
	uint32_t run = x - s;
	for(int w = 0; w < wave; ++w) { run += ws[w]; }
#pragma unroll
	for(int k = 0; k < kScanOneItems; ++k)
	{
		if(k < per && i0 + k < m) { c[i0 + k] = run; }
		run += v[k];
	}
}

// One pass of the sort in one launch: a tile ranks its keys, publishes its digit
// counts, sums the counts of the tiles before it from their status words (the sums
// of a tile that has done so itself end the search) and writes its keys out, one
// contiguous run per digit.  Tiles are numbered by ticket, so every tile before one
// that waits has started; it publishes its counts before it waits for any other,
// so every wait ends.  A pass's words carry its number: those of the passes before
// read as not there yet.  Latency bound below some 2^19 keys: with a histogram, a
// scan and a scatter with a work-group barrier per row of keys for every pass, list
// by list, the heap build of 2^17 bodies took 1065 us (24 passes of 31 us), with this
// pass 366, and the Morton build of 2^22 bodies 1.96 ms, with this pass 1.70 (213 us
// and 1.15 ms with the rest of the builds as they are now).
__global__ void __launch_bounds__(kSortThreads)
k_sort_pass(sort_lists a, size_t n, int pass, int last, int keep_keys, uint32_t* __restrict__ scratch, size_t tiles)
{
	constexpr int kWaves = kSortThreads / 64;
	constexpr int kLook = 8;                // status words read at a time
	__shared__ uint64_t skey[kSortTile];
	__shared__ uint32_t sval[kSortTile];
	__shared__ uint32_t counts[kWaves][256];
	__shared__ uint32_t goff[256];          // output position of the tile's first key of a digit, minus its place in LDS
	__shared__ uint32_t loff[256];          // place of that key in LDS
	__shared__ uint32_t ws[4];
	__shared__ uint32_t my_tile;
	const sort_scratch s = sort_scratch_of(scratch, blockIdx.y, tiles);
	const sort_list& l = a.l[blockIdx.y];
	const uint64_t* kin = l.k[pass & 1];
	const uint32_t* vin = l.v[pass & 1];
	uint64_t* kout = l.k[(pass & 1) ^ 1];
	uint32_t* vout = last ? l.out : l.v[(pass & 1) ^ 1];
	const int shift = 8 * pass;
	if(threadIdx.x == 0) { my_tile = atomicAdd(&s.ticket[pass], 1u); }
	for(int i = threadIdx.x; i < kWaves * 256; i += kSortThreads) { (&counts[0][0])[i] = 0; }
	__syncthreads();
	const uint32_t tile = my_tile;
	const size_t base = static_cast<size_t>(tile) * kSortTile;
	const int tcount = n - base < static_cast<size_t>(kSortTile) ? static_cast<int>(n - base) : kSortTile;
	const int wave = threadIdx.x >> 6;
	const int first = wave * (64 * kSortItems) + (threadIdx.x & 63);
	uint64_t key[kSortItems];
	uint32_t val[kSortItems], rank[kSortItems];
	bool ok[kSortItems];
#pragma unroll
	for(int k = 0; k < kSortItems; ++k)
	{
		const int r = first + 64 * k;
		ok[k] = r < tcount;
		key[k] = ok[k] ? kin[base + r] : 0;
		val[k] = ok[k] ? vin[base + r] : 0;
	}
	rank_tile<kSortItems>(key, ok, shift, counts[wave], rank);
	__syncthreads();
	const bool digit = threadIdx.x < 256;
	uint32_t total = 0;
	if(digit)
	{
		for(int w = 0; w < kWaves; ++w)
		{
			const uint32_t c = counts[w][threadIdx.x];
			counts[w][threadIdx.x] = total;
			total += c;
		}
		const unsigned long long tag = tile == 0 ? 2 * pass + 2 : 2 * pass + 1;
		__hip_atomic_store(&s.status[static_cast<size_t>(tile) * 256 + threadIdx.x], tag << 32 | total,
		                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	const uint32_t place = scan256(total, ws);
	const uint32_t start = scan256(digit ? s.hist[pass * 256 + threadIdx.x] : 0, ws);
	if(digit) { loff[threadIdx.x] = place; }
	__syncthreads();
#pragma unroll
	for(int k = 0; k < kSortItems; ++k)
	{
		if(ok[k])
		{
			const uint32_t d = static_cast<uint32_t>((key[k] >> shift) & 0xFF);
			const uint32_t pos = loff[d] + counts[wave][d] + rank[k];
			skey[pos] = key[k];
			sval[pos] = val[k];
		}
	}
	if(digit)
	{
		uint32_t before = 0;
		const unsigned long long part = 2 * pass + 1, sum = 2 * pass + 2;
		long long t = static_cast<long long>(tile) - 1;
		while(t >= 0)
		{
			unsigned long long v[kLook];
#pragma unroll
			for(int k = 0; k < kLook; ++k)
			{
				v[k] = t - k >= 0 ? __hip_atomic_load(&s.status[static_cast<size_t>(t - k) * 256 + threadIdx.x],
				                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
				                  : sum << 32;
			}
			bool open = true;
			int used = 0;
#pragma unroll
			for(int k = 0; k < kLook; ++k)
			{
				const unsigned long long tag = v[k] >> 32;
				if(open && (tag == part || tag == sum))
				{
					before += static_cast<uint32_t>(v[k]);
					++used;
					open = tag == part;
					if(tag == sum) { t = -1; }
				}
				else
				{
					open = false;
				}
			}
			if(t >= 0) { t -= used; }
		}
		if(tile != 0)
		{
			__hip_atomic_store(&s.status[static_cast<size_t>(tile) * 256 + threadIdx.x], sum << 32 | (before + total),
			                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		}
		goff[threadIdx.x] = start + before - place;
	}
	__syncthreads();
	for(int i = threadIdx.x; i < tcount; i += kSortThreads)
	{
		const uint64_t k = skey[i];
		const uint32_t pos = goff[(k >> shift) & 0xFF] + static_cast<uint32_t>(i);
		if(keep_keys || !last) { kout[pos] = k; }
		vout[pos] = sval[i];
	}
}

// All passes over at most kSortTile keys by one work-group per list, in LDS.
__global__ void __launch_bounds__(kSortOneThreads)
k_sort_one(sort_lists a, int n, int passes, int keep_keys)
{
	constexpr int kWaves = kSortOneThreads / 64;
	__shared__ uint64_t skey[kSortTile];
	__shared__ uint32_t sval[kSortTile];
	__shared__ uint32_t counts[kWaves][256];
	__shared__ uint32_t loff[256];
	__shared__ uint32_t ws[4];
	const sort_list& l = a.l[blockIdx.y];
	const int wave = threadIdx.x >> 6;
	const int first = wave * (64 * kSortOneItems) + (threadIdx.x & 63);
	for(int i = threadIdx.x; i < n; i += kSortOneThreads)
	{
		skey[i] = l.k[0][i];
		sval[i] = l.v[0][i];
	}
	for(int pass = 0; pass < passes; ++pass)
	{
		const int shift = 8 * pass;
		for(int i = threadIdx.x; i < kWaves * 256; i += kSortOneThreads) { (&counts[0][0])[i] = 0; }
		__syncthreads();
		uint64_t key[kSortOneItems];
		uint32_t val[kSortOneItems], rank[kSortOneItems];
		bool ok[kSortOneItems];
#pragma unroll
		for(int k = 0; k < kSortOneItems; ++k)
		{
			const int r = first + 64 * k;
			ok[k] = r < n;
			key[k] = ok[k] ? skey[r] : 0;
			val[k] = ok[k] ? sval[r] : 0;
		}
		rank_tile<kSortOneItems>(key, ok, shift, counts[wave], rank);
		__syncthreads();
		uint32_t total = 0;
		if(threadIdx.x < 256)
		{
			for(int w = 0; w < kWaves; ++w)
			{
				const uint32_t c = counts[w][threadIdx.x];
				counts[w][threadIdx.x] = total;
				total += c;
			}
		}
		const uint32_t place = scan256(total, ws);
		if(threadIdx.x < 256) { loff[threadIdx.x] = place; }
		__syncthreads();
#pragma unroll
		for(int k = 0; k < kSortOneItems; ++k)
		{
			if(ok[k])
			{
				const uint32_t d = static_cast<uint32_t>((key[k] >> shift) & 0xFF);
				const uint32_t pos = loff[d] + counts[wave][d] + rank[k];
				skey[pos] = key[k];
				sval[pos] = val[k];
			}
		}
		__syncthreads();
	}
	for(int i = threadIdx.x; i < n; i += kSortOneThreads)
	{
		if(keep_keys) { l.k[passes & 1][i] = skey[i]; }
		l.out[i] = sval[i];
	}
}

// ---------------------------------------------------------------------------
// per-level split
// ---------------------------------------------------------------------------
// side[list_a[p]] = 1 for the upper half of p's segment
__global__ void __launch_bounds__(256)
k_mark_side(const uint32_t* __restrict__ list_a, uint8_t* __restrict__ side, size_t n, size_t seg)
{
	size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
	size_t half = seg >> 1;
	for(size_t p = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; p < n; p += stride)
	{
		side[list_a[p]] = (p & (seg - 1)) >= half ? 1 : 0;
	}
}

// The two lists that a level partitions: from in[] to out[].
struct part_lists {
	const uint32_t* in[2];
	uint32_t*       out[2];
};

// rights[list][b] = number of upper-half bodies in tile b of a list (blockIdx.y)
__global__ void __launch_bounds__(kPartThreads)
k_part_count(part_lists l, const uint8_t* __restrict__ side, uint32_t* __restrict__ rights)
{
	__shared__ uint32_t wsum[kPartThreads / 64];
	const uint4 body = reinterpret_cast<const uint4*>(l.in[blockIdx.y])[blockIdx.x * kPartThreads + threadIdx.x];
	uint32_t c = side[body.x] + side[body.y] + side[body.z] + side[body.w];
	for(int off = 32; off > 0; off >>= 1) { c += __shfl_down(c, off, 64); }
	if((threadIdx.x & 63) == 0) { wsum[threadIdx.x >> 6] = c; }
	__syncthreads();
	if(threadIdx.x == 0)
	{
		uint32_t t = 0;
		for(int w = 0; w < kPartThreads / 64; ++w) { t += wsum[w]; }
		rights[blockIdx.y * gridDim.x + blockIdx.x] = t;
	}
}

// Stable partition of every segment (at least a tile) of both lists into lower-half
// then upper-half bodies (flags in `side`).  The upper-half bodies of the segment's
// tiles before this one are summed here from `rights`, or, scanned != 0, `rights` is
// its exclusive scan.  The list of the next level's axis (next, -1: none) also sets
// that level's flags, side_next.  Latency bound at 2^18 bodies: a list and a step at a
// time (mark, then count, scan and scatter twice), the six levels above the LDS took
// 190 us there, now 70.
__global__ void __launch_bounds__(kPartThreads)
k_part_scatter(part_lists l, const uint8_t* __restrict__ side, size_t seg, const uint32_t* __restrict__ rights,
               int scanned, int next, uint8_t* __restrict__ side_next)
{
	constexpr int kWaves = kPartThreads / 64;
	__shared__ uint32_t wsum[kWaves], wbefore[kWaves];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const uint32_t* r = rights + blockIdx.y * gridDim.x;
	const uint32_t first = blockIdx.x & ~static_cast<uint32_t>(seg / kPartTile - 1);
	const uint4 b4 = reinterpret_cast<const uint4*>(l.in[blockIdx.y])[blockIdx.x * kPartThreads + threadIdx.x];
	const uint32_t body[kPartItems] = {b4.x, b4.y, b4.z, b4.w};
	uint32_t fl[kPartItems], c = 0, before = 0;
	for(int k = 0; k < kPartItems; ++k)
	{
		fl[k] = side[body[k]];
		c += fl[k];
	}
	if(scanned != 0)
	{
		before = threadIdx.x == 0 ? r[blockIdx.x] - r[first] : 0;
	}
	else
	{
		for(uint32_t i = first + threadIdx.x; i < blockIdx.x; i += kPartThreads) { before += r[i]; }
	}
	uint32_t x = c;
	for(int off = 1; off < 64; off <<= 1)
	{
		const uint32_t u = __shfl_up(x, off, 64);
		if(lane >= off) { x += u; }
		before += __shfl_xor(before, off, 64);
	}
	if(lane == 63)
	{
		wsum[wave] = x;
		wbefore[wave] = before;
	}
	__syncthreads();
	uint32_t ex = x - c;
	for(int w = 0; w < kWaves; ++w) { ex += wbefore[w] + (w < wave ? wsum[w] : 0); }
	uint32_t* out = l.out[blockIdx.y];
	const bool flags = static_cast<int>(blockIdx.y) == next;
	const size_t half = seg >> 1;
	const size_t p0 = static_cast<size_t>(blockIdx.x) * kPartTile + threadIdx.x * kPartItems;
	const size_t upper = (p0 & ~(seg - 1)) + half;
	for(int k = 0; k < kPartItems; ++k)
	{
		const size_t pos = fl[k] ? upper + ex : p0 + k - ex;
		out[pos] = body[k];
		if(flags) { side_next[body[k]] = (pos & (half - 1)) >= half >> 1 ? 1 : 0; }
		ex += fl[k];
	}
}

// Levels first_level .. levels-1 of the split (the steps of k_mark_side and
// k_part_scatter) for segments of seg0 <= kLocalSeg bodies, one work-group per
// segment, in LDS.  Bodies get local numbers (their position in list0's
// segment, through the global table g2l) so that the side flags live in LDS.
// Only the final order is written back, to list0: after the last level every
// segment holds one body and the three lists agree.  A work-item has kLocalItems
// positions of both lists that move, their counts in one word, and writes the next
// level's flags with the list that sets them: two barriers a level, 38 us at 2^18
// bodies, 87 with eleven.
constexpr int kLocalItems = kLocalSeg / kLocalThreads;
static_assert(kLocalItems == 4 && kLocalSeg < (1 << 16), "positions of a work-item in 8 bytes, two counts in a word");

__global__ void __launch_bounds__(kLocalThreads)
k_split_local(uint32_t* __restrict__ list0, const uint32_t* __restrict__ list1, const uint32_t* __restrict__ list2,
              uint32_t* __restrict__ g2l, int seg0, int first_level, int levels)
{
	__shared__ __align__(8) uint16_t ls[5][kLocalSeg];     // three lists and two to write
	__shared__ uint32_t l2g[kLocalSeg];
	__shared__ uint8_t side[2][kLocalSeg];
	__shared__ uint32_t ws[kLocalThreads / 64];
	const size_t base = static_cast<size_t>(blockIdx.x) * seg0;
	const int lane = threadIdx.x & 63;
	const int wave = threadIdx.x >> 6;
	for(int p = threadIdx.x; p < seg0; p += kLocalThreads)
	{
		const uint32_t b = list0[base + p];
		l2g[p] = b;
		ls[0][p] = static_cast<uint16_t>(p);
		g2l[b] = static_cast<uint32_t>(p);
	}
	__syncthreads();
	for(int p = threadIdx.x; p < seg0; p += kLocalThreads)
	{
		ls[1][p] = static_cast<uint16_t>(g2l[list1[base + p]]);
		ls[2][p] = static_cast<uint16_t>(g2l[list2[base + p]]);
	}
	__syncthreads();
	{
		const uint16_t* l = ls[first_level % 3];
		for(int p = threadIdx.x; p < seg0; p += kLocalThreads) { side[0][l[p]] = p >= seg0 >> 1 ? 1 : 0; }
	}
	__syncthreads();
	const int p0 = static_cast<int>(threadIdx.x) * kLocalItems;
	int cur0 = 0, cur1 = 1, cur2 = 2, free0 = 3, free1 = 4;   // rows of ls: the lists, the two to write
	for(int level = first_level; level < levels; ++level)
	{
		const int seg = seg0 >> (level - first_level);
		const int half = seg >> 1;
		const int a = level % 3;
		const uint8_t* now = side[(level - first_level) & 1];
		uint8_t* then = side[~(level - first_level) & 1];
		// the list of the next level's axis first
		const int from[2] = {a == 0 ? cur1 : a == 1 ? cur2 : cur0, a == 0 ? cur2 : a == 1 ? cur0 : cur1};
		const int to[2] = {free0, free1};
		uint16_t id[2][kLocalItems];
		uint32_t up[kLocalItems], c = 0;       // flags of the two lists, counts: 16 bits each
		for(int b = 0; b < 2; ++b)
		{
			const ushort4 v = *reinterpret_cast<const ushort4*>(&ls[from[b]][p0]);
			id[b][0] = v.x; id[b][1] = v.y; id[b][2] = v.z; id[b][3] = v.w;
		}
		for(int k = 0; k < kLocalItems; ++k)
		{
			const bool in = p0 + k < seg0;
			up[k] = in ? now[id[0][k]] | static_cast<uint32_t>(now[id[1][k]]) << 16 : 0;
			c += up[k];
		}
		uint32_t x = c;
		for(int off = 1; off < 64; off <<= 1)
		{
			const uint32_t u = __shfl_up(x, off, 64);
			if(lane >= off) { x += u; }
		}
		if(lane == 63) { ws[wave] = x; }
		__syncthreads();
		uint32_t ex = x - c;
		for(int w = 0; w < wave; ++w) { ex += ws[w]; }
		for(int k = 0; k < kLocalItems; ++k)
		{
			const int p = p0 + k;
			if(p < seg0)
			{
				const int start = p & ~(seg - 1);
				for(int b = 0; b < 2; ++b)
				{
					// upper-half bodies of the segment before p: half of every earlier
					// segment's bodies are
					const int before = static_cast<int>(b == 0 ? ex & 0xFFFF : ex >> 16) - (start >> 1);
					const bool u = ((b == 0 ? up[k] : up[k] >> 16) & 1) != 0;
					const int pos = u ? start + half + before : p - before;
					ls[to[b]][pos] = id[b][k];
					if(b == 0) { then[id[0][k]] = (pos & (half - 1)) >= half >> 1 ? 1 : 0; }
				}
			}
			ex += up[k];
		}
		__syncthreads();
		free0 = from[0];
		free1 = from[1];
		if(a == 0) { cur1 = to[0]; cur2 = to[1]; }
		else if(a == 1) { cur2 = to[0]; cur0 = to[1]; }
		else { cur0 = to[0]; cur1 = to[1]; }
	}
	for(int p = threadIdx.x; p < seg0; p += kLocalThreads) { list0[base + p] = l2g[ls[cur0][p]]; }
}

// ---------------------------------------------------------------------------
// moments (nbody/nbody_space_heap.cpp:119-134), FP64, contraction off
// ---------------------------------------------------------------------------
__device__ inline double min_ref(double a, double b) { return (b < a) ? b : a; }   // std::min
__device__ inline double max_ref(double a, double b) { return (a < b) ? b : a; }   // std::max

// Opening radius crit_r2 = (radius * ratio)^2 of a node with mass centre c and
// box lo, hi, in the heap's operation order.
__device__ inline double crit_radius(double cx, double cy, double cz, const double* lo, const double* hi,
                                     double ratio_sqr)
{
	double ex = hi[0] - lo[0], ey = hi[1] - lo[1], ez = hi[2] - lo[2];
	double gx = (hi[0] + lo[0]) / 2.0 - cx;
	double gy = (hi[1] + lo[1]) / 2.0 - cy;
	double gz = (hi[2] + lo[2]) / 2.0 - cz;
	double rad = sqrt(ex * ex + ey * ey + ez * ez) * 0.5 + sqrt(gx * gx + gy * gy + gz * gz);
	return (rad * rad) * ratio_sqr;
}

// A node's moments from its children's (mass centre cl / cr, masses ml / mr,
// boxes lol..hil / lor..hir): mass, mass centre, box and opening radius with the
// heap's operation order.
__device__ inline void combine_node(const double4& cl, double ml, const double* lol, const double* hil,
                                    const double4& cr, double mr, const double* lor, const double* hir,
                                    double ratio_sqr, double4& c, double& m, double* lo, double* hi)
{
	m = ml + mr;
	double cx = (cl.x * ml + cr.x * mr) / m;
	double cy = (cl.y * ml + cr.y * mr) / m;
	double cz = (cl.z * ml + cr.z * mr) / m;
	for(int d = 0; d < 3; ++d)
	{
		lo[d] = min_ref(lol[d], lor[d]);
		hi[d] = max_ref(hil[d], hir[d]);
	}
	c = make_double4(cx, cy, cz, crit_radius(cx, cy, cz, lo, hi, ratio_sqr));
}

// Second central moments Q = sum m (x - cm)(x - cm)^T of a node from its
// children (parallel-axis theorem); components xx yy zz xy xz yz.  Not part of
// the reference tree: input of the learned correction.
__device__ inline void combine_quad(const double4& c, const double4& cl, double ml, const double* ql,
                                    const double4& cr, double mr, const double* qr, double* q)
{
	for(int k = 0; k < 6; ++k) { q[k] = 0.0; }
	for(int side = 0; side < 2; ++side)
	{
		const double4 cc = side == 0 ? cl : cr;
		const double m = side == 0 ? ml : mr;
		const double* qc = side == 0 ? ql : qr;
		const double dx = cc.x - c.x, dy = cc.y - c.y, dz = cc.z - c.z;
		q[0] += qc[0] + m * dx * dx;
		q[1] += qc[1] + m * dy * dy;
		q[2] += qc[2] + m * dz * dz;
		q[3] += qc[3] + m * dx * dy;
		q[4] += qc[4] + m * dx * dz;
		q[5] += qc[5] + m * dy * dz;
	}
}

// Node idx with its walk record from its children l and r, each read once.
__device__ inline void join_nodes(size_t idx, size_t l, size_t r, double4* xyzr, double* nmass, double* bmin,
                                  double* bmax, double* quad, double ratio_sqr, nbh_walk_rec* wr)
{
	const double4 cl = xyzr[l], cr = xyzr[r];
	const double ml = nmass[l], mr = nmass[r];
	double lol[3], hil[3], lor[3], hir[3], ql[6], qr[6];
	for(int d = 0; d < 3; ++d)
	{
		lol[d] = bmin[3 * l + d];
		hil[d] = bmax[3 * l + d];
		lor[d] = bmin[3 * r + d];
		hir[d] = bmax[3 * r + d];
	}
	for(int k = 0; k < 6; ++k)
	{
		ql[k] = quad[6 * l + k];
		qr[k] = quad[6 * r + k];
	}
	nbh_walk_rec rec;
	double lo[3], hi[3], q[6];
	combine_node(cl, ml, lol, hil, cr, mr, lor, hir, ratio_sqr, rec.c, rec.m, lo, hi);
	combine_quad(rec.c, cl, ml, ql, cr, mr, qr, q);
	xyzr[idx] = rec.c;
	nmass[idx] = rec.m;
	for(int d = 0; d < 3; ++d)
	{
		bmin[3 * idx + d] = lo[d];
		bmax[3 * idx + d] = hi[d];
	}
	for(int k = 0; k < 6; ++k) { quad[6 * idx + k] = q[k]; }
	for(int k = 0; k < 6; ++k) { rec.q[k] = static_cast<float>(q[k]); }
	wr[idx] = rec;
}

// ---------------------------------------------------------------------------
// Morton radix tree (the fast path of the FP32 group walks; no counterpart in
// the reference, whose heap kd-tree stays the tree of the parity walks)
// ---------------------------------------------------------------------------
// Bodies sorted by 63-bit Morton codes (21 bits per axis over the bounding
// cube), ties broken by body index; internal nodes by the binary radix tree
// construction of Karras (2012, "Maximizing parallelism in the construction of
// BVHs, octrees, and k-d trees"): internal node i covers a key range with i at
// one end and splits it at the highest bit where its keys differ.  Node ids
// follow the heap's conventions where the walks rely on them: the root is id 1
// (internal node i is id i + 1), the body at sorted position j is leaf id n + j,
// and ids >= n are leaves.  Cells are bounded by the boxes of their bodies,
// with the heap's opening radius, so a cell of the Morton tree is compact where
// a count-balanced heap node of a centrally concentrated state spans from the
// core to the outskirts.

// Spread the low 21 bits of v to every third bit.
__device__ inline uint64_t morton_spread(uint64_t v)
{
	v &= 0x1fffffull;
	v = (v | (v << 32)) & 0x1f00000000ffffull;
	v = (v | (v << 16)) & 0x1f0000ff0000ffull;
	v = (v | (v << 8)) & 0x100f00f00f00f00full;
	v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
	v = (v | (v << 2)) & 0x1249249249249249ull;
	return v;
}

// Cell coordinate of x on a grid of 2^21 cells over [lo, lo + 2^21 / scale).
__device__ inline uint64_t morton_cell(double x, double lo, double scale)
{
	double c = floor((x - lo) * scale);
	c = c < 0.0 ? 0.0 : c;
	c = c > 2097151.0 ? 2097151.0 : c;
	return static_cast<uint64_t>(c);
}

// box[6] = bounding box lo.xyz hi.xyz of the bodies: scale = 2^21 / longest side
__global__ void __launch_bounds__(256)
k_morton_codes(const double* __restrict__ y, const double* __restrict__ mass, size_t n, const double* __restrict__ box,
               uint64_t* __restrict__ keys, uint32_t* __restrict__ vals, double4* __restrict__ pk,
               uint32_t* __restrict__ marks, size_t words, int* __restrict__ parent, uint32_t* __restrict__ counts,
               size_t count_words)
{
	const double side = fmax(fmax(box[3] - box[0], box[4] - box[1]), box[5] - box[2]);
	const double scale = side > 0.0 ? 2097152.0 / side : 0.0;
	const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
	for(size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
	{
		const double x = y[i], yy = y[n + i], z = y[2 * n + i];
		const uint64_t cx = morton_cell(x, box[0], scale);
		const uint64_t cy = morton_cell(yy, box[1], scale);
		const uint64_t cz = morton_cell(z, box[2], scale);
		keys[i] = (morton_spread(cx) << 2) | (morton_spread(cy) << 1) | morton_spread(cz);
		vals[i] = static_cast<uint32_t>(i);
		pk[i] = make_double4(x, yy, z, mass[i]);
	}
	// what the sort and the tree's kernels count and mark in, and the parents that no
	// node has
	for(size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count_words; i += stride) { counts[i] = 0; }
	for(size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < words; i += stride) { marks[i] = 0; }
	if(blockIdx.x == 0 && threadIdx.x < 2) { parent[threadIdx.x] = 0; }
}

// Bounding box partials of the positions, then the box (lo.xyz hi.xyz).
__global__ void __launch_bounds__(256)
k_box_partial(const double* __restrict__ y, size_t n, double* __restrict__ part)
{
	__shared__ double sh[6][256];
	double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
	const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
	for(size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
	{
		for(int d = 0; d < 3; ++d)
		{
			const double v = y[static_cast<size_t>(d) * n + i];
			lo[d] = fmin(lo[d], v);
			hi[d] = fmax(hi[d], v);
		}
	}
	for(int d = 0; d < 3; ++d) { sh[d][threadIdx.x] = lo[d]; sh[3 + d][threadIdx.x] = hi[d]; }
	__syncthreads();
	for(int w = 128; w > 0; w >>= 1)
	{
		if(static_cast<int>(threadIdx.x) < w)
		{
			for(int d = 0; d < 3; ++d)
			{
				sh[d][threadIdx.x] = fmin(sh[d][threadIdx.x], sh[d][threadIdx.x + w]);
				sh[3 + d][threadIdx.x] = fmax(sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + w]);
			}
		}
		__syncthreads();
	}
	if(threadIdx.x < 6) { part[6 * blockIdx.x + threadIdx.x] = sh[threadIdx.x][0]; }
}

// The partials are taken strided by 256 threads, then reduced in LDS (min and
// max are exact, so the order does not change the box).
__global__ void __launch_bounds__(256)
k_box_final(const double* __restrict__ part, int count, double* __restrict__ box)
{
	__shared__ double sh[6][256];
	double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
	for(int k = threadIdx.x; k < count; k += blockDim.x)
	{
		for(int d = 0; d < 3; ++d)
		{
			lo[d] = fmin(lo[d], part[6 * k + d]);
			hi[d] = fmax(hi[d], part[6 * k + 3 + d]);
		}
	}
	for(int d = 0; d < 3; ++d) { sh[d][threadIdx.x] = lo[d]; sh[3 + d][threadIdx.x] = hi[d]; }
	__syncthreads();
	for(int w = 128; w > 0; w >>= 1)
	{
		if(static_cast<int>(threadIdx.x) < w)
		{
			for(int d = 0; d < 3; ++d)
			{
				sh[d][threadIdx.x] = fmin(sh[d][threadIdx.x], sh[d][threadIdx.x + w]);
				sh[3 + d][threadIdx.x] = fmax(sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + w]);
			}
		}
		__syncthreads();
	}
	if(threadIdx.x < 6) { box[threadIdx.x] = sh[threadIdx.x][0]; }
}

// Length of the common prefix of sorted keys i and j (with the index as a
// tie-breaking suffix), -1 outside [0, n).
__device__ inline int radix_delta(const uint64_t* __restrict__ k, long long n, long long i, long long j)
{
	if(j < 0 || j >= n) { return -1; }
	const uint64_t a = k[i], b = k[j];
	if(a == b)
	{
		return 64 + __clzll(static_cast<unsigned long long>(i ^ j));
	}
	return __clzll(a ^ b);
}

// Groups of the Morton tree, all maximal subtrees: build groups of at most
// kRadixGroup leaves (one wave computes their nodes' moments), walk groups of at
// most kRadixWalk leaves (one wave walks for them, two bodies per lane), and
// super-groups of at most kRadixSuper leaves that hold more than one walk group
// (a walk group in no super-group walks in one level).  Their leaves are
// consecutive in Morton order and their boxes are node boxes, so they never
// straddle the core of the state the way a fixed run of the Morton order can.
constexpr int kRadixGroup = 64;
constexpr int kRadixWalk = 128;
constexpr int kRadixSuper = 2048;
constexpr int kRadixSuperMin = kRadixWalk + 1;   // at least two walk groups

// Scratch of a Morton build: a bit per sorted position and kind of mark (a mark sits
// at the first sorted position of its group's leaves), the marks counted by runs of
// `run` words, and the info counts: subtrees of each tier, then build groups,
// super-groups and walk groups.
enum MarkKind { kMarkBuild, kMarkSuper, kMarkWalk };

struct RadixMarks {
	uint32_t* bits;
	uint32_t* part;
	int*      info;
	size_t    words;      // of one kind
	int       run;        // log2 of the positions of a part
	__host__ __device__ int parts() const
	{
		return static_cast<int>(((words << 5) + (static_cast<size_t>(1) << run) - 1) >> run);
	}
};

constexpr int kInfoCounts = kRadixTiers + 3;

inline size_t mark_words(size_t n) { return 3 * ((n + 31) / 32) + 3 * kMarkParts + kInfoCounts; }

inline RadixMarks radix_marks(uint32_t* p, size_t n)
{
	RadixMarks m;
	m.words = (n + 31) / 32;
	m.bits = p;
	m.part = p + 3 * m.words;
	m.info = reinterpret_cast<int*>(m.part + 3 * kMarkParts);
	m.run = 11;           // one wave takes 64 words at a time
	while(m.parts() > kMarkParts) { ++m.run; }
	return m;
}

__device__ inline void put_mark(const RadixMarks& m, MarkKind kind, int2* __restrict__ mark, long long pos, int id,
                                long long cnt)
{
	mark[pos] = make_int2(id, static_cast<int>(cnt));
	atomicOr(&m.bits[kind * m.words + (pos >> 5)], 1u << (pos & 31));
}

// Subtrees of the Morton tree by size: a node of more than 64 * 32^(t - 1) and at
// most 64 * 32^t leaves has tier t (0: inside a build group).
__device__ inline int radix_tier(long long cnt)
{
	int t = 0;
	while(cnt > (static_cast<long long>(kRadixGroup) << (5 * t))) { ++t; }
	return t;
}

// First entry of tier t in the list of subtree roots: a tier-t subtree has more than
// 64 * 32^(t - 1) leaves.
__host__ __device__ inline size_t tier_offset(size_t n, int t)
{
	size_t off = 0;
	for(int k = 1; k < t; ++k) { off += n / (static_cast<size_t>(kRadixGroup) << (5 * (k - 1))) + 1; }
	return off;
}

// Internal node i of [0, n - 1): its key range, split and children (ids), the
// parent links of the children, its tier, the roots of the tiers' subtrees (in any
// order) and the marks of build groups, walk groups and super-groups: (node id, leaves).
__global__ void __launch_bounds__(256)
k_radix_nodes(const uint64_t* __restrict__ k, long long n, int2* __restrict__ child, int* __restrict__ parent,
              uint8_t* __restrict__ tier, int* __restrict__ tier_list, RadixMarks marks, int2* __restrict__ gmark,
              int2* __restrict__ smark, int2* __restrict__ wmark)
{
	const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
	for(long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n - 1; i += stride)
	{
		const int dir = radix_delta(k, n, i, i + 1) - radix_delta(k, n, i, i - 1) > 0 ? 1 : -1;
		const int dmin = radix_delta(k, n, i, i - dir);
		long long lmax = 2;
		while(radix_delta(k, n, i, i + lmax * dir) > dmin) { lmax <<= 1; }
		long long l = 0;
		for(long long t = lmax >> 1; t >= 1; t >>= 1)
		{
			if(radix_delta(k, n, i, i + (l + t) * dir) > dmin) { l += t; }
		}
		const long long j = i + l * dir;
		const int dnode = radix_delta(k, n, i, j);
		long long s = 0;
		for(long long t = (l + 1) >> 1;; t = (t + 1) >> 1)
		{
			if(s + t < l + 1 && radix_delta(k, n, i, i + (s + t) * dir) > dnode) { s += t; }
			if(t <= 1) { break; }
		}
		const long long gamma = i + s * dir + (dir < 0 ? -1 : 0);
		const long long lo = i < j ? i : j, hi = i < j ? j : i;
		const int left = lo == gamma ? static_cast<int>(n + gamma) : static_cast<int>(gamma + 1);
		const int right = hi == gamma + 1 ? static_cast<int>(n + gamma + 1) : static_cast<int>(gamma + 2);
		const int id = static_cast<int>(i + 1);
		child[id] = make_int2(left, right);
		parent[left] = id;
		parent[right] = id;
		const long long cnt = hi - lo + 1;
		tier[id] = static_cast<uint8_t>(radix_tier(cnt));
		if(cnt <= kRadixGroup && id != kRoot) { continue; }     // inside a build group
		const auto mark = [&](int node, long long pos, long long leaves, long long above, bool internal)
		{
			if(above > kRadixGroup && leaves <= kRadixGroup) { put_mark(marks, kMarkBuild, gmark, pos, node, leaves); }
			if(above > kRadixWalk && leaves <= kRadixWalk) { put_mark(marks, kMarkWalk, wmark, pos, node, leaves); }
			if(above > kRadixSuper && leaves <= kRadixSuper && leaves >= kRadixSuperMin)
			{
				put_mark(marks, kMarkSuper, smark, pos, node, leaves);
			}
			if(internal && leaves > kRadixGroup)
			{
				const int t = radix_tier(leaves);
				if(above > (static_cast<long long>(kRadixGroup) << (5 * t)))
				{
					tier_list[tier_offset(static_cast<size_t>(n), t) + atomicAdd(&marks.info[t], 1)] = node;
				}
			}
		};
		if(id == kRoot) { mark(id, lo, cnt, LLONG_MAX, true); }
		mark(left, lo, gamma - lo + 1, cnt, lo != gamma);
		mark(right, gamma + 1, hi - gamma, cnt, hi != gamma + 1);
	}
}

__global__ void __launch_bounds__(256)
k_fill_int(int* __restrict__ a, size_t count, int v)
{
	const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
	for(size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += stride) { a[i] = v; }
}

// Marks of each kind in each part, a wave per part.  (Counted by atomics where the
// marks are set, k_radix_nodes takes 193 us at 4M bodies against 152, and 22.6 at 100003
// against 18.)
__global__ void __launch_bounds__(256)
k_radix_count(RadixMarks m)
{
	const int lane = threadIdx.x & 63;
	const int part = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
	if(part >= m.parts()) { return; }
	const size_t per = (static_cast<size_t>(1) << m.run) >> 5, w0 = part * per;
	const size_t w1 = w0 + per < m.words ? w0 + per : m.words;
	for(int kind = 0; kind < 3; ++kind)
	{
		uint32_t v = 0;
		for(size_t w = w0 + lane; w < w1; w += 64) { v += __popc(m.bits[kind * m.words + w]); }
		for(int sh = 32; sh > 0; sh >>= 1) { v += __shfl_xor(v, sh, 64); }
		if(lane == 0) { m.part[kind * kMarkParts + part] = v; }
	}
}

// Build groups grp[g] and walk groups wgrp[w] = (node id, first sorted leaf,
// leaves, super-group or -1) and super-groups sup[s] = (node id, first sorted
// leaf), all in Morton order, and their counts; a wave per part of the marks, 64 words
// at a time, from the counts of the parts before it.  The super-group of a walk group
// is the last one marked at or before its first leaf, if its leaves reach it (both are
// subtrees); it lies at most kRadixSuper positions, 64 words, back.  Latency bound:
// with flags, three scans, a compaction, a search per walk group and cleared marks of
// 8 bytes per position this took 85 us in 17 launches at 100003 bodies and 240 us at
// 4M.
__global__ void __launch_bounds__(256)
k_radix_groups(RadixMarks m, const int2* __restrict__ gmark, const int2* __restrict__ smark,
               const int2* __restrict__ wmark, int4* __restrict__ grp, int2* __restrict__ sup,
               int4* __restrict__ wgrp)
{
	const int lane = threadIdx.x & 63;
	const int part = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, parts = m.parts();
	if(part >= parts) { return; }
	const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
	uint32_t base[3];
	for(int kind = 0; kind < 3; ++kind)
	{
		uint32_t v = 0;
		for(int i = lane; i < part; i += 64) { v += m.part[kind * kMarkParts + i]; }
		for(int sh = 32; sh > 0; sh >>= 1) { v += __shfl_xor(v, sh, 64); }
		base[kind] = v;
		if(part == parts - 1 && lane == 0)
		{
			m.info[kRadixTiers + kind] = static_cast<int>(v + m.part[kind * kMarkParts + part]);
		}
	}
	const size_t w0 = (static_cast<size_t>(part) << m.run) >> 5;
	const size_t w1 = w0 + ((static_cast<size_t>(1) << m.run) >> 5) < m.words
	                      ? w0 + ((static_cast<size_t>(1) << m.run) >> 5) : m.words;
	// position of the last super-group mark before the words at hand, -1: none in reach
	const auto last_of = [](uint32_t word, size_t first, uint64_t has)
	{
		const int src = 63 - __clzll(static_cast<long long>(has));
		const uint32_t v = __shfl(word, src & 63, 64);
		return has != 0 ? static_cast<int>((first + src) * 32 + 31 - __clz(static_cast<int>(v))) : -1;
	};
	int carry = -1;
	if(w0 >= 64)
	{
		const uint32_t sw = m.bits[kMarkSuper * m.words + w0 - 64 + lane];
		carry = last_of(sw, w0 - 64, __ballot(sw != 0));
	}
	for(size_t wb = w0; wb < w1; wb += 64)
	{
		const size_t w = wb + lane;
		uint32_t word[3], at[3];
		for(int kind = 0; kind < 3; ++kind)
		{
			word[kind] = w < w1 ? m.bits[kind * m.words + w] : 0;
			const uint32_t c = __popc(word[kind]);
			uint32_t x = c;
			for(int sh = 1; sh < 64; sh <<= 1)
			{
				const uint32_t u = __shfl_up(x, sh, 64);
				if(lane >= sh) { x += u; }
			}
			at[kind] = base[kind] + x - c;
			base[kind] += __shfl(x, 63, 64);
		}
		const uint64_t has = __ballot(word[kMarkSuper] != 0);
		const int before = last_of(word[kMarkSuper], wb, has & lt);
		const int last = (has & lt) != 0 ? before : carry;
		for(uint32_t b = word[kMarkBuild]; b != 0; b &= b - 1)
		{
			const int p = static_cast<int>(w * 32) + __builtin_ctz(b);
			const int2 g = gmark[p];
			grp[at[kMarkBuild]++] = make_int4(g.x, p, g.y, -1);
		}
		for(uint32_t b = word[kMarkWalk]; b != 0; b &= b - 1)
		{
			const int bit = __builtin_ctz(b), p = static_cast<int>(w * 32) + bit;
			const int2 g = wmark[p];
			const uint32_t mine = word[kMarkSuper] & (0xFFFFFFFFu >> (31 - bit));
			const int sp = mine != 0 ? static_cast<int>(w * 32) + 31 - __clz(static_cast<int>(mine)) : last;
			const bool in = sp >= 0 && sp + smark[sp < 0 ? 0 : sp].y > p;
			wgrp[at[kMarkWalk]++] = make_int4(g.x, p, g.y, in ? static_cast<int>(at[kMarkSuper] + __popc(mine)) - 1 : -1);
		}
		for(uint32_t b = word[kMarkSuper]; b != 0; b &= b - 1)
		{
			const int p = static_cast<int>(w * 32) + __builtin_ctz(b);
			sup[at[kMarkSuper]++] = make_int2(smark[p].x, p);
		}
		const int end = last_of(word[kMarkSuper], wb, has);
		if(has != 0) { carry = end; }
	}
}

// LDS written by some lanes of a wave is read by others after this.
__device__ inline void wave_sync()
{
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
}

// `v` of another lane of the same four (kCtrl: the source lane of each, 2 bits a lane).
template <int kCtrl>
__device__ inline double quad_lane(double v)
{
	const long long b = __double_as_longlong(v);
	const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(b), kCtrl, 0xF, 0xF, true);
	const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(b >> 32), kCtrl, 0xF, 0xF, true);
	return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}

// A node's moments from its children's by four lanes: lane d (at most 2) takes
// coordinate d of the mass centre and box, the diagonal second moment dd and one of
// xy, xz, yz (combine_node and combine_quad, in their order).
__device__ inline void join_part(const double (&cc)[2], const double (&mm)[2], const double (&lo2)[2],
                                 const double (&hi2)[2], const double (&qd)[2], const double (&qo)[2], double& c,
                                 double& m, double& lo, double& hi, double& qdd, double& qoo)
{
	m = mm[0] + mm[1];
	c = (cc[0] * mm[0] + cc[1] * mm[1]) / m;
	lo = min_ref(lo2[0], lo2[1]);
	hi = max_ref(hi2[0], hi2[1]);
	qdd = 0.0;
	qoo = 0.0;
	for(int side = 0; side < 2; ++side)
	{
		const double e = cc[side] - c;
		// the factors of xy, xz, yz: (x, x, y) and (y, z, z)
		const double ea = quad_lane<0xD0>(e), eb = quad_lane<0xE9>(e);
		qdd += qd[side] + mm[side] * e * e;
		qoo += qo[side] + mm[side] * ea * eb;
	}
}

// Leaves and internal nodes of each build group (a subtree of at most
// kRadixGroup leaves), one wave per group, with their walk records.  The
// group's leaves (kBuild: the body at sorted position s is
// order[s], read from its packed record; refit: the body numbers of the build,
// positions from y and the masses of the leaf records) and node moments are held
// in LDS: leaf first + j in slot j, internal id k in slot k - first - 1 (the
// internal ids of a subtree over the sorted leaves [a, b] are the ids [a + 1, b + 1]
// without the end that is not its root: each internal node's index is one end of
// its key range).  The internal nodes are listed breadth-first, then taken depth by
// depth from the deepest (combine_node and combine_quad on the LDS slots), four
// lanes a node: lane d has coordinate d, its diagonal second moment and one of the
// other three.  The opening radii, which no parent reads, follow for all nodes at
// once, and the nodes go out in id order.
// lean: every node's walk record is written (and each leaf's body number), the
// FP64 node arrays only for the group's root, which the levels above read, or
// for a group of one leaf.
// With a lane per node, radius and stores in the depth loop, it was bound by FP64
// issue there (some 40 nodes in 10 depths): 541 us at 4M bodies, now 363 (0.8 GB
// moved), latency of the depths and memory alike.
template <bool kBuild>
__global__ void __launch_bounds__(kRadixGroup)
k_radix_group_moments(const int4* __restrict__ grp, const int* __restrict__ groups, int n, const int2* __restrict__ child,
                      const uint32_t* __restrict__ order, const double4* __restrict__ pk, const double* __restrict__ y,
                      int32_t* __restrict__ body_n, double4* __restrict__ xyzr, double* __restrict__ nmass,
                      double* __restrict__ bmin, double* __restrict__ bmax, double* __restrict__ quad,
                      double ratio_sqr, nbh_walk_rec* __restrict__ wr, int lean)
{
	// LDS of doubles: leaf positions and masses; the internal slots' mass centres,
	// masses, boxes and second moments; the second moments of a leaf
	constexpr int kG = kRadixGroup;
	constexpr int kLC = 0, kLM = 3 * kG, kC = 4 * kG, kM = 7 * kG, kLo = 8 * kG, kHi = 11 * kG, kQ = 14 * kG,
	              kZero = 20 * kG;
	__shared__ double sh[20 * kG + 6];
	__shared__ int2 s_child[kG];
	__shared__ int q[kG];          // internal nodes, breadth-first (at most kRadixGroup - 1)
	__shared__ int start[kG + 1];  // first entry of each depth
	const int lane = threadIdx.x;
	if(lane < 6) { sh[kZero + lane] = 0.0; }
	const int count = *groups;
	for(int g = blockIdx.x; g < count; g += gridDim.x)
	{
		__syncthreads();
		const int4 gr = grp[g];
		const int root = gr.x, first = gr.y, cnt = gr.z;
		if(lane < cnt)
		{
			const size_t sidx = static_cast<size_t>(first) + lane;
			const size_t idx = static_cast<size_t>(n) + sidx;
			double x, yy, z, m;
			if constexpr(kBuild)
			{
				const uint32_t b = order[sidx];
				const double4 p = pk[b];
				x = p.x;
				yy = p.y;
				z = p.z;
				m = p.w;
				body_n[idx] = static_cast<int32_t>(b);
				if(!lean || root >= n) { nmass[idx] = m; }
			}
			else
			{
				// the mass from the leaf's walk record, which every build writes
				const size_t b = static_cast<uint32_t>(body_n[idx]);
				x = y[b];
				yy = y[n + b];
				z = y[2 * static_cast<size_t>(n) + b];
				m = wr[idx].m;
			}
			nbh_walk_rec r;
			r.c = make_double4(x, yy, z, 0.0);
			r.m = m;
			for(int k = 0; k < 6; ++k) { r.q[k] = 0.0f; }
			if(!lean || root >= n)
			{
				xyzr[idx] = r.c;
				bmin[3 * idx] = x; bmin[3 * idx + 1] = yy; bmin[3 * idx + 2] = z;
				bmax[3 * idx] = x; bmax[3 * idx + 1] = yy; bmax[3 * idx + 2] = z;
			}
			wr[idx] = r;
			sh[kLC + 3 * lane] = x;
			sh[kLC + 3 * lane + 1] = yy;
			sh[kLC + 3 * lane + 2] = z;
			sh[kLM + lane] = m;
			const int id = first + 1 + lane;
			s_child[lane] = id < n ? child[id] : make_int2(0, 0);
		}
		if(root >= n) { continue; }            // a group of one leaf
		const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
		if(lane == 0)
		{
			q[0] = root;
			start[0] = 0;
		}
		int head = 0, tail = 1, depth = 0;
		__syncthreads();
		while(head < tail)
		{
			const int width = tail - head;
			const bool act = lane < width;
			const int2 c = act ? s_child[q[head + lane] - first - 1] : make_int2(n, n);
			const bool li = c.x < n, ri = c.y < n;
			const uint64_t bl = __ballot(li), br = __ballot(ri);
			int pos = tail + __popcll(bl & lt) + __popcll(br & lt);
			if(li) { q[pos++] = c.x; }
			if(ri) { q[pos] = c.y; }
			head = tail;
			tail += __popcll(bl) + __popcll(br);
			++depth;
			if(lane == 0) { start[depth] = head; }
			__syncthreads();
		}
		// depth d holds q[start[d], start[d + 1]); start[depth] == tail.  A child is
		// leaf first + j (id n + first + j) or internal slot id - first - 1.
		const int part = lane & 3, dim = part < 3 ? part : 2;
		for(int d = depth - 1; d >= 0; --d)
		{
			const int end = start[d + 1];
			for(int i = start[d] + (lane >> 2); i < end; i += kG / 4)
			{
				const int k = q[i] - first - 1;
				const int2 ch = s_child[k];
				double cc[2], mm[2], lo2[2], hi2[2], qd[2], qo[2];
				for(int side = 0; side < 2; ++side)
				{
					const int cid = side == 0 ? ch.x : ch.y;
					const bool leaf = cid >= n;
					const int j = leaf ? cid - n - first : cid - first - 1;
					const int at = 3 * j + dim;
					const int qat = leaf ? kZero : kQ + 6 * j;
					cc[side] = sh[(leaf ? kLC : kC) + at];
					mm[side] = sh[(leaf ? kLM : kM) + j];
					lo2[side] = sh[(leaf ? kLC : kLo) + at];
					hi2[side] = sh[(leaf ? kLC : kHi) + at];
					qd[side] = sh[qat + dim];
					qo[side] = sh[qat + 3 + dim];
				}
				double c, m, lo, hi, qdd, qoo;
				join_part(cc, mm, lo2, hi2, qd, qo, c, m, lo, hi, qdd, qoo);
				if(part < 3)
				{
					sh[kC + 3 * k + part] = c;
					sh[kLo + 3 * k + part] = lo;
					sh[kHi + 3 * k + part] = hi;
					sh[kQ + 6 * k + part] = qdd;
					sh[kQ + 6 * k + 3 + part] = qoo;
				}
				else
				{
					sh[kM + k] = m;
				}
			}
			__syncthreads();
		}
		const int k = lane + (root == first + 1 ? 0 : 1);
		if(lane < cnt - 1)
		{
			const size_t gid = static_cast<size_t>(first) + 1 + k;
			const double* lo = sh + kLo + 3 * k;
			const double* hi = sh + kHi + 3 * k;
			const double cx = sh[kC + 3 * k], cy = sh[kC + 3 * k + 1], cz = sh[kC + 3 * k + 2];
			nbh_walk_rec rec;
			rec.c = make_double4(cx, cy, cz, crit_radius(cx, cy, cz, lo, hi, ratio_sqr));
			rec.m = sh[kM + k];
			for(int e = 0; e < 6; ++e) { rec.q[e] = static_cast<float>(sh[kQ + 6 * k + e]); }
			wr[gid] = rec;
			if(!lean || gid == static_cast<size_t>(root))
			{
				xyzr[gid] = rec.c;
				nmass[gid] = rec.m;
				for(int e = 0; e < 3; ++e)
				{
					bmin[3 * gid + e] = lo[e];
					bmax[3 * gid + e] = hi[e];
				}
				for(int e = 0; e < 6; ++e) { quad[6 * gid + e] = sh[kQ + 6 * k + e]; }
			}
		}
	}
}

// Moments of the nodes of one tier, a work-group per subtree of more than
// 64 * 32^(t - 1) and at most 64 * 32^t leaves: the nodes of the tier below its root are
// listed breadth-first (at most 31 in a depth, as each holds more than 1/32 of the
// leaves, and at most kTierDepth depths, as prefixes grow along a branch), then taken
// depth by depth from the deepest, like a build group.  The first kTierNodes of
// them and their children of lower tiers are held in LDS; any further ones, which
// only branches of bodies at ever closer distances bring about, go through the node
// arrays.  Latency bound (a read per depth down, divides per depth up); with a launch
// or a barrier per prefix length in place of a depth of one subtree, the nodes above
// the build groups took 88 us at 100003 bodies and 310 at 4M.
constexpr int kTierDepth = 96;
constexpr int kTierList = 31 * kTierDepth;
constexpr int kTierNodes = 80;
constexpr int kTierSlots = 2 * kTierNodes + 1;
__global__ void __launch_bounds__(256)
k_radix_tier(const int* __restrict__ roots, int t, int n, const int2* __restrict__ child,
             const uint8_t* __restrict__ tier, double4* xyzr, double* nmass, double* bmin, double* bmax, double* quad,
             double ratio_sqr, nbh_walk_rec* __restrict__ wr)
{
	// per slot: mass centre, mass, box, second moments
	constexpr int kC = 0, kM = 3, kLo = 4, kHi = 7, kQ = 10, kPer = 17;
	__shared__ double sh[kTierSlots * kPer];
	__shared__ int q[kTierList];
	__shared__ int start[kTierDepth + 1];
	__shared__ int2 ref[kTierNodes];       // children: ~slot or node id
	__shared__ int below[kTierNodes + 1];  // children of lower tiers
	__shared__ int2 kids[64];              // children of the depth at hand
	__shared__ int s_depth, s_below;
	const int tid = threadIdx.x;
	if(tid < 64)
	{
		const uint64_t lt = tid == 0 ? 0ull : (~0ull >> (64 - tid));
		if(tid == 0)
		{
			const int root = roots[blockIdx.x];
			q[0] = root;
			start[0] = 0;
			kids[0] = child[root];
		}
		int head = 0, tail = 1, depth = 0, nb = 0;
		wave_sync();
		while(head < tail)
		{
			const bool act = tid < tail - head;
			const int2 c = act ? kids[tid] : make_int2(n, n);
			bool in[2], out[2];
			int2 kk[2];
			for(int side = 0; side < 2; ++side)
			{
				const int id = side == 0 ? c.x : c.y;
				const int safe = id < n ? id : kRoot;
				kk[side] = child[safe];
				in[side] = act && id < n && tier[safe] == t;
				out[side] = act && !in[side] && head + tid < kTierNodes;
			}
			const uint64_t bl = __ballot(in[0]), br = __ballot(in[1]);
			const uint64_t ol = __ballot(out[0]), orr = __ballot(out[1]);
			int pos = tail + __popcll(bl & lt) + __popcll(br & lt);
			int bpos = nb + __popcll(ol & lt) + __popcll(orr & lt);
			int r[2];
			wave_sync();
			for(int side = 0; side < 2; ++side)
			{
				const int id = side == 0 ? c.x : c.y;
				r[side] = id;
				if(in[side])
				{
					if(pos < kTierNodes) { r[side] = ~pos; }
					q[pos] = id;
					kids[pos - tail] = kk[side];
					++pos;
				}
				else if(out[side])
				{
					r[side] = ~(kTierNodes + bpos);
					below[bpos++] = id;
				}
			}
			if(act && head + tid < kTierNodes) { ref[head + tid] = make_int2(r[0], r[1]); }
			head = tail;
			tail += __popcll(bl) + __popcll(br);
			nb += __popcll(ol) + __popcll(orr);
			++depth;
			if(tid == 0) { start[depth] = head; }
			wave_sync();
		}
		if(tid == 0)
		{
			s_depth = depth;
			s_below = nb;
		}
	}
	__syncthreads();
	const int depth = s_depth, nbelow = s_below, count = start[depth];
	const int part = tid & 3, dim = part < 3 ? part : 2;
	// one coordinate of a node's moments, from the node arrays
	const auto read = [&](int id, double& c, double& m, double& lo, double& hi, double& qd, double& qo)
	{
		const size_t i = static_cast<size_t>(id);
		c = reinterpret_cast<const double*>(xyzr)[4 * i + dim];
		m = nmass[i];
		lo = bmin[3 * i + dim];
		hi = bmax[3 * i + dim];
		qd = quad[6 * i + dim];
		qo = quad[6 * i + 3 + dim];
	};
	const auto put = [&](int slot, double c, double m, double lo, double hi, double qd, double qo)
	{
		double* p = sh + slot * kPer;
		if(part < 3)
		{
			p[kC + part] = c;
			p[kLo + part] = lo;
			p[kHi + part] = hi;
			p[kQ + part] = qd;
			p[kQ + 3 + part] = qo;
		}
		else
		{
			p[kM] = m;
		}
	};
	for(int i = tid >> 2; i < nbelow; i += 64)
	{
		double c, m, lo, hi, qd, qo;
		read(below[i], c, m, lo, hi, qd, qo);
		put(kTierNodes + i, c, m, lo, hi, qd, qo);
	}
	for(int d = depth - 1; d >= 0 && start[d + 1] > kTierNodes; --d)
	{
		const int lo = start[d] > kTierNodes ? start[d] : kTierNodes;
		const int i = lo + tid;
		if(i < start[d + 1])
		{
			const int2 c = child[q[i]];
			join_nodes(q[i], c.x, c.y, xyzr, nmass, bmin, bmax, quad, ratio_sqr, wr);
		}
		__syncthreads();
	}
	__syncthreads();
	for(int d = depth - 1; d >= 0; --d)
	{
		const int i = start[d] + (tid >> 2);
		const bool act = i < start[d + 1] && i < kTierNodes;
		double cc[2] = {}, mm[2] = {}, lo2[2] = {}, hi2[2] = {}, qd[2] = {}, qo[2] = {};
		if(act)
		{
			const int2 rr = ref[i];
			for(int side = 0; side < 2; ++side)
			{
				const int r = side == 0 ? rr.x : rr.y;
				if(r < 0)
				{
					const double* p = sh + ~r * kPer;
					cc[side] = p[kC + dim];
					mm[side] = p[kM];
					lo2[side] = p[kLo + dim];
					hi2[side] = p[kHi + dim];
					qd[side] = p[kQ + dim];
					qo[side] = p[kQ + 3 + dim];
				}
				else
				{
					read(r, cc[side], mm[side], lo2[side], hi2[side], qd[side], qo[side]);
				}
			}
			double c, m, lo, hi, qdd, qoo;
			join_part(cc, mm, lo2, hi2, qd, qo, c, m, lo, hi, qdd, qoo);
			put(i, c, m, lo, hi, qdd, qoo);
		}
		__syncthreads();
	}
	if(tid < count && tid < kTierNodes)
	{
		const double* p = sh + tid * kPer;
		const size_t id = static_cast<size_t>(q[tid]);
		nbh_walk_rec rec;
		rec.c = make_double4(p[kC], p[kC + 1], p[kC + 2],
		                     crit_radius(p[kC], p[kC + 1], p[kC + 2], p + kLo, p + kHi, ratio_sqr));
		rec.m = p[kM];
		for(int e = 0; e < 6; ++e) { rec.q[e] = static_cast<float>(p[kQ + e]); }
		wr[id] = rec;
		xyzr[id] = rec.c;
		nmass[id] = rec.m;
		for(int e = 0; e < 3; ++e)
		{
			bmin[3 * id + e] = p[kLo + e];
			bmax[3 * id + e] = p[kHi + e];
		}
		for(int e = 0; e < 6; ++e) { quad[6 * id + e] = p[kQ + e]; }
	}
}

// Moments and walk records of the heap's nodes above the `width` (a power of two, at
// most kHeapBase) ids from lo + blockIdx.x * width, a subtree whose root the work-group
// ends with.  kLeaf: the ids are leaves, set here too: the body at sorted position s is
// order[s], or with no order (refit) the leaf's body and mass of the last build.  The
// subtree is held in LDS, four lanes a node (join_part), and the nodes go out at the
// end, when their opening radii are known.  Bound by memory: with a launch for the
// leaves, one for each level and one for the records, which read all of it again,
// 100 us at 2^18 bodies and 285 at 2^20, now 55 and 153.
constexpr int kHeapBase = 256;

template <bool kLeaf>
__global__ void __launch_bounds__(kHeapBase)
k_heap_moments(size_t lo, int width, size_t n, const uint32_t* __restrict__ order, const double* __restrict__ y,
               const double* __restrict__ mass, double4* __restrict__ xyzr, double* __restrict__ nmass,
               double* __restrict__ bmin, double* __restrict__ bmax, double* __restrict__ quad,
               int32_t* __restrict__ body_n, double ratio_sqr, nbh_walk_rec* __restrict__ wr)
{
	// local ids as in a heap: root 1, the given nodes [width, 2 width).  Per node mass
	// centre, mass, box, second moments; leaves: position and mass
	constexpr int kC = 0, kM = 3, kLo = 4, kHi = 7, kQ = 10, kPer = 17, kLeafPer = 4;
	__shared__ double sh[kHeapBase * kPer];
	__shared__ double base[kHeapBase * (kLeaf ? kLeafPer : kPer)];
	const int tid = threadIdx.x;
	const int part = tid & 3, dim = part < 3 ? part : 2;
	const size_t first = lo + static_cast<size_t>(blockIdx.x) * width;
	if constexpr(kLeaf)
	{
		if(tid < width)
		{
			const size_t idx = first + tid;
			const uint32_t b = order != nullptr ? order[idx - n] : static_cast<uint32_t>(body_n[idx]);
			nbh_walk_rec r;
			r.c = make_double4(y[b], y[n + b], y[2 * n + b], 0.0);
			r.m = order != nullptr ? mass[b] : nmass[idx];
			for(int k = 0; k < 6; ++k) { r.q[k] = 0.0f; }
			if(order != nullptr)
			{
				body_n[idx] = static_cast<int32_t>(b);
				nmass[idx] = r.m;
			}
			xyzr[idx] = r.c;
			bmin[3 * idx] = r.c.x; bmin[3 * idx + 1] = r.c.y; bmin[3 * idx + 2] = r.c.z;
			bmax[3 * idx] = r.c.x; bmax[3 * idx + 1] = r.c.y; bmax[3 * idx + 2] = r.c.z;
			wr[idx] = r;
			double* p = base + kLeafPer * tid;
			p[0] = r.c.x;
			p[1] = r.c.y;
			p[2] = r.c.z;
			p[3] = r.m;
		}
	}
	else
	{
		for(int i = tid >> 2; i < width; i += kHeapBase / 4)
		{
			const size_t idx = first + i;
			double* p = base + kPer * i;
			if(part < 3)
			{
				p[kC + part] = reinterpret_cast<const double*>(xyzr)[4 * idx + part];
				p[kLo + part] = bmin[3 * idx + part];
				p[kHi + part] = bmax[3 * idx + part];
				p[kQ + part] = quad[6 * idx + part];
				p[kQ + 3 + part] = quad[6 * idx + 3 + part];
			}
			else
			{
				p[kM] = nmass[idx];
			}
		}
	}
	__syncthreads();
	for(int w = width >> 1; w >= 1; w >>= 1)
	{
		for(int i = w + (tid >> 2); i < 2 * w; i += kHeapBase / 4)
		{
			double cc[2], mm[2], lo2[2], hi2[2], qd[2], qo[2];
			for(int side = 0; side < 2; ++side)
			{
				const int ch = 2 * i + side;
				if(kLeaf && ch >= width)
				{
					const double* p = base + kLeafPer * (ch - width);
					cc[side] = lo2[side] = hi2[side] = p[dim];
					mm[side] = p[3];
					qd[side] = qo[side] = 0.0;
				}
				else
				{
					const double* p = ch >= width ? base + kPer * (ch - width) : sh + kPer * ch;
					cc[side] = p[kC + dim];
					mm[side] = p[kM];
					lo2[side] = p[kLo + dim];
					hi2[side] = p[kHi + dim];
					qd[side] = p[kQ + dim];
					qo[side] = p[kQ + 3 + dim];
				}
			}
			double c, m, l, h, qdd, qoo;
			join_part(cc, mm, lo2, hi2, qd, qo, c, m, l, h, qdd, qoo);
			double* p = sh + kPer * i;
			if(part < 3)
			{
				p[kC + part] = c;
				p[kLo + part] = l;
				p[kHi + part] = h;
				p[kQ + part] = qdd;
				p[kQ + 3 + part] = qoo;
			}
			else
			{
				p[kM] = m;
			}
		}
		__syncthreads();
	}
	if(tid >= 1 && tid < width)
	{
		const int d = 31 - __clz(tid);
		const size_t idx = ((first / width) << d) + (tid - (1 << d));
		const double* p = sh + kPer * tid;
		nbh_walk_rec rec;
		rec.c = make_double4(p[kC], p[kC + 1], p[kC + 2],
		                     crit_radius(p[kC], p[kC + 1], p[kC + 2], p + kLo, p + kHi, ratio_sqr));
		rec.m = p[kM];
		for(int e = 0; e < 6; ++e) { rec.q[e] = static_cast<float>(p[kQ + e]); }
		wr[idx] = rec;
		xyzr[idx] = rec.c;
		nmass[idx] = rec.m;
		for(int e = 0; e < 3; ++e)
		{
			bmin[3 * idx + e] = p[kLo + e];
			bmax[3 * idx + e] = p[kHi + e];
		}
		for(int e = 0; e < 6; ++e) { quad[6 * idx + e] = p[kQ + e]; }
	}
}

// ---------------------------------------------------------------------------
// traversal
// ---------------------------------------------------------------------------
// heap index algebra (nbody/nbody_space_heap_func_priv.h:4-72)
__device__ inline int next_down(int idx)
{
	idx = idx >> __builtin_ctz(~static_cast<unsigned>(idx));
	return idx + 1;
}

__device__ inline int next_up(int idx, int tree_size)
{
	int left = idx << 1;
	return left < tree_size ? left : next_down(idx);
}

// Counters are cleared by a kernel rather than a memset node, so a captured
// sequence of calls replays correctly.
__global__ void k_zero_counters(unsigned long long* counters)
{
	if(threadIdx.x < 5) { counters[threadIdx.x] = 0; }
}

__device__ inline void count_add(unsigned long long* counters, unsigned long long inter, unsigned long long vis)
{
	for(int off = 32; off > 0; off >>= 1)
	{
		inter += __shfl_down(inter, off, 64);
		vis += __shfl_down(vis, off, 64);
	}
	if((threadIdx.x & 63) == 0)
	{
		atomicAdd(&counters[0], inter);
		atomicAdd(&counters[1], vis);
	}
}

// FP64 monopole term of nbody_data::force: u = (v1 - cm) * (-(m1 M) / r^3)
__device__ inline void term64(double x1, double y1, double z1, double gm1, const double4& nd, double M, double& ux,
                              double& uy, double& uz)
{
	double dx = x1 - nd.x;
	double dy = y1 - nd.y;
	double dz = z1 - nd.z;
	double r2 = dx * dx + dy * dy + dz * dz;
	if(r2 < 1e-8) { r2 = 1e-8; }
	double coeff = (gm1 * M) / (r2 * sqrt(r2));
	ux = dx * coeff;
	uy = dy * coeff;
	uz = dz * coeff;
}

__device__ inline void write_f(const double* __restrict__ y, const double* __restrict__ mass, double* __restrict__ f,
                               size_t n, int b, double tx, double ty, double tz)
{
	double m1 = mass[b];
	f[b] = y[3 * n + b];
	f[n + b] = y[4 * n + b];
	f[2 * n + b] = y[5 * n + b];
	f[3 * n + b] = tx / m1;
	f[4 * n + b] = ty / m1;
	f[5 * n + b] = tz / m1;
}

// The FP64 walks: nbody_space_heap::traverse (nbody_space_heap.cpp:64-97) and
// nbody_space_heap_stackless::traverse (nbody_space_heap_stackless.cpp:3-26) visit
// a body's nodes in the same order (left subtree first) and add the accepted ones
// in that order, so one kernel serves both layouts bit for bit.
//
// One wave walks for 32 neighbouring leaves at once: it visits every node that any
// of its bodies visits (13% more nodes than one body alone at 2^17 bodies, ratio
// 2), and a 32-bit mask says whose node it is.  What is left of the walk is a stack
// of elements (node, bodies that take it, bodies that open it) in walk order, the
// next one on top.  A step moves the elements at the top that nobody opens to a
// list, then opens up to kWalkOpen nodes at once and puts what each leaves --
// itself for its takers, its children -- in its place, in order.  One lane per
// child decides from the bodies' box whether all of them or none pass its test
// (four children in five); the others are tested body by body, two at a time (one
// per half of the wave), four tests interleaved.  64
// listed nodes at a time are evaluated: the halves take eight consecutive entries
// each, two terms in flight (with four waves per SIMD that covers the 16 clocks of
// a dependent FP64 operation), and then add them in list order, one half after the other; a body whose
// mask bit is clear adds a zero.
//
// A body per lane, each on its own way through the tree, spent its time on gathers,
// divergent branches and the general quotient and root: 252 us at 1024 bodies, 1.56
// ms at 16384, 3.8 at 65536, 7.6 at 2^17 and 313 at 2^20 (ratio 2) against 90 us,
// 0.44, 1.49, 3.9 and 72 ms.  At 2^17 bodies a SIMD then issues 0.155 VALU
// instructions a clock (0.22 is the most for FP64), some 60% of them the terms'.
// Without the box test it took 5.0 ms; four terms in flight at two or three waves per
// SIMD 4.1 and 4.8 (spills), four entries per half 4.0.
constexpr int kWalkTgt = 32;
constexpr int kWalkEntries = 64;
constexpr int kWalkPer = 8;
constexpr int kWalkIlp = 2;
constexpr int kWalkOpen = 32;
// Stack elements.  Opening one node at a time leaves at most three elements per
// level (31 levels at most): that many stay in reserve, and what is above them
// limits how many nodes open together.
constexpr int kWalkStack64 = 400;   // with the list, 9.4 KB of LDS: 16 waves per CU
constexpr int kWalkReserve = 3 * 33;

// The value of lane l mod 32 (upper: l mod 32 + 32) in every lane.
template <bool kUpper>
__device__ inline double half_wave(double v)
{
	const unsigned lo = static_cast<unsigned>(__double2loint(v));
	const unsigned hi = static_cast<unsigned>(__double2hiint(v));
	const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
	const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
	return __hiloint2double(static_cast<int>(h[kUpper ? 1 : 0]), static_cast<int>(l[kUpper ? 1 : 0]));
}

struct walk64_lds {
	double4 rec[kWalkEntries];      // x, y, z, mass of the listed nodes, or records of undecided children
	unsigned mask[kWalkEntries];
	int list_node[2 * kWalkEntries];
	unsigned list_mask[2 * kWalkEntries];
	int node[kWalkStack64];
	unsigned take[kWalkStack64];
	unsigned open[kWalkStack64];
	int open_node[kWalkOpen];
	unsigned open_mask[kWalkOpen];
	unsigned passed[2 * kWalkOpen + 8];     // bodies whose test an undecided child passes
	uint2 child[2 * kWalkOpen];             // bodies that take / open a child
};

// The terms of entries e0 .. e0 + 2 kWalkPer - 1 of the list, added in order to the
// sums that half kFrom of the wave holds; the other half holds them afterwards.
template <bool kFrom>
__device__ inline void walk64_chunk(const walk64_lds& w, int e0, int lane, const double4& me, double gm8, double& tx,
                                    double& ty, double& tz)
{
	const int t = lane & (kWalkTgt - 1);
	const int own = e0 + ((lane >= kWalkTgt) != kFrom ? kWalkPer : 0);
	double ux[kWalkPer], uy[kWalkPer], uz[kWalkPer];
#pragma unroll
	for(int p = 0; p < kWalkPer; p += kWalkIlp)
	{
		double r2[kWalkIlp], s[kWalkIlp], q[kWalkIlp];
		bool mine[kWalkIlp];
#pragma unroll
		for(int k = 0; k < kWalkIlp; ++k)
		{
			const double4 nd = w.rec[own + p + k];
			mine[k] = (w.mask[own + p + k] >> t) & 1u;
			ux[p + k] = me.x - nd.x;
			uy[p + k] = me.y - nd.y;
			uz[p + k] = me.z - nd.z;
			s[k] = gm8 * nd.w;
		}
#pragma unroll
		for(int k = 0; k < kWalkIlp; ++k) { r2[k] = ux[p + k] * ux[p + k]; }
#pragma unroll
		for(int k = 0; k < kWalkIlp; ++k) { q[k] = uy[p + k] * uy[p + k]; }
#pragma unroll
		for(int k = 0; k < kWalkIlp; ++k) { r2[k] = r2[k] + q[k]; }
#pragma unroll
		for(int k = 0; k < kWalkIlp; ++k) { q[k] = uz[p + k] * uz[p + k]; }
#pragma unroll
		for(int k = 0; k < kWalkIlp; ++k) { r2[k] = r2[k] + q[k]; }
#pragma unroll
		for(int k = 0; k < kWalkIlp; ++k) { r2[k] = fmax(r2[k], 1e-8); }    // finite here: the same as term64's branch
		pair_quot_rn<kWalkIlp>(s, r2, q);
#pragma unroll
		for(int k = 0; k < kWalkIlp; ++k)
		{
			// a sum that starts at +0 is never -0, so adding a zero of either sign keeps it
			q[k] = mine[k] ? q[k] : 0.0;
			ux[p + k] = ux[p + k] * q[k];
			uy[p + k] = uy[p + k] * q[k];
			uz[p + k] = uz[p + k] * q[k];
		}
	}
#pragma unroll
	for(int h = 0; h < 2; ++h)
	{
		if(h == 1)
		{
			tx = half_wave<kFrom>(tx);
			ty = half_wave<kFrom>(ty);
			tz = half_wave<kFrom>(tz);
		}
#pragma unroll
		for(int p = 0; p < kWalkPer; ++p)
		{
			tx += ux[p];
			ty += uy[p];
			tz += uz[p];
		}
	}
}

__global__ void __launch_bounds__(64, 4)
k_bh_walk64(const double4* __restrict__ xyzr, const double* __restrict__ nmass, const int32_t* __restrict__ body_n,
            const double* __restrict__ y, const double* __restrict__ mass, double* __restrict__ f, int n,
            unsigned long long* __restrict__ counters)
{
	__shared__ walk64_lds w;
	const int lane = threadIdx.x;
	const int t = lane & (kWalkTgt - 1);
	const int upper = lane / kWalkTgt;
	// neighbouring groups on one XCD (work-groups go round robin over eight), so
	// that its L2 serves the nodes they share
	const unsigned groups = gridDim.x;
	const unsigned group = groups % 8 == 0 ? (blockIdx.x % 8) * (groups / 8) + blockIdx.x / 8 : blockIdx.x;
	const int first = static_cast<int>(group) * kWalkTgt;
	const bool active = first + t < n;
	const int tn = n + (active ? first + t : first);
	const double4 me = xyzr[tn];
	const double gm1 = -1.0 * nmass[tn];
	const double gm8 = 8.0 * gm1;
	const bool all_safe =
	    __ballot(!(coord_in_range(me.x) && coord_in_range(me.y) && coord_in_range(me.z) && mass_in_range(gm1))) == 0;
	// box of the bodies (lanes without one repeat the first); it says nothing of a body
	// that is not a number or infinite, whose offset from a node may be no number
	const bool box_holds = __ballot(!(isfinite(me.x) && isfinite(me.y) && isfinite(me.z))) == 0;
	double3 lo = make_double3(me.x, me.y, me.z), hi = lo;
	for(int off = 16; off > 0; off >>= 1)
	{
		lo.x = fmin(lo.x, __shfl_xor(lo.x, off, 64));
		lo.y = fmin(lo.y, __shfl_xor(lo.y, off, 64));
		lo.z = fmin(lo.z, __shfl_xor(lo.z, off, 64));
		hi.x = fmax(hi.x, __shfl_xor(hi.x, off, 64));
		hi.y = fmax(hi.y, __shfl_xor(hi.y, off, 64));
		hi.z = fmax(hi.z, __shfl_xor(hi.z, off, 64));
	}
	double tx = 0.0, ty = 0.0, tz = 0.0;
	unsigned long long inter = 0, vis = 0;      // per lane
	int count = 0, sp = 0;
	const unsigned long long lt_mask = lane == 0 ? 0ull : ~0ull >> (64 - lane);
	auto below = [&](unsigned long long b) { return __popcll(b & lt_mask); };
	auto passes = [&](const double4& nd) {
		const double dx = me.x - nd.x;
		const double dy = me.y - nd.y;
		const double dz = me.z - nd.z;
		return __ballot(dx * dx + dy * dy + dz * dz > nd.w);
	};
	// the first `e` <= 64 listed nodes; the list keeps the others
	auto evaluate = [&](int e) {
		__builtin_amdgcn_wave_barrier();
		const int node = lane < e ? w.list_node[lane] : kRoot;
		const unsigned mask = lane < e ? w.list_mask[lane] : 0u;
		const double4 c = xyzr[node];
		const double m = nmass[node];
		const bool ok = coord_in_range(c.x) && coord_in_range(c.y) && coord_in_range(c.z) && mass_in_range(m);
		const bool fast = __ballot(!ok) == 0 && all_safe;
		w.rec[lane] = make_double4(c.x, c.y, c.z, m);
		w.mask[lane] = mask;
		if(kWalkEntries + lane < count)
		{
			w.list_node[lane] = w.list_node[kWalkEntries + lane];
			w.list_mask[lane] = w.list_mask[kWalkEntries + lane];
		}
		__builtin_amdgcn_wave_barrier();
		if(fast)
		{
			for(int k = 0; k < e; k += 4 * kWalkPer)
			{
				walk64_chunk<false>(w, k, lane, me, gm8, tx, ty, tz);
				walk64_chunk<true>(w, k + 2 * kWalkPer, lane, me, gm8, tx, ty, tz);
			}
		}
		else
		{
			// the general sequences, one entry at a time
#pragma unroll 1
			for(int k = 0; k < e; ++k)
			{
				if((w.mask[k] >> t) & 1u)
				{
					const double4 nd = w.rec[k];
					double ux, uy, uz;
					term64(me.x, me.y, me.z, gm1, nd, nd.w, ux, uy, uz);
					tx += ux;
					ty += uy;
					tz += uz;
				}
			}
		}
		__builtin_amdgcn_wave_barrier();
		count -= e;
	};

	{
		const unsigned all = static_cast<unsigned>(__ballot(active));
		const unsigned take = static_cast<unsigned>(passes(xyzr[kRoot])) & all;
		if(lane == 0)
		{
			w.node[0] = kRoot;
			w.take[0] = take;
			w.open[0] = kRoot < n ? all & ~take : 0u;
			vis = __popc(all);
			inter = __popc(take);
		}
		sp = 1;
	}
	for(;;)
	{
		if(count >= kWalkEntries || sp == 0)
		{
			if(count == 0) { break; }
			evaluate(count < kWalkEntries ? count : kWalkEntries);
			continue;
		}
		__builtin_amdgcn_wave_barrier();
		// the top of the stack in walk order, lane 0 first
		const bool have = lane < sp;
		const int at = have ? sp - 1 - lane : 0;
		const int node = w.node[at];
		const unsigned take = w.take[at];
		const bool opened = have && w.open[at] != 0;
		const unsigned long long opens = __ballot(opened);
		const int seen = sp < 64 ? sp : 64;
		// elements before the first opened one go to the list
		const int lead = opens == 0 ? seen : __builtin_ctzll(opens);
		if(lane < lead)
		{
			w.list_node[count + lane] = node;
			w.list_mask[count + lane] = take;
		}
		count += lead;
		if(opens != 0)
		{
			int most = (kWalkStack64 - kWalkReserve - sp) / 2;
			most = most > kWalkOpen ? kWalkOpen : most < 1 ? 1 : most;
			const int rank = below(opens);
			const bool mine = opened && rank < most;
			const int total = __popcll(opens);
			const int used = total < most ? total : most;
			// the window ends before the first opened element that is left for later
			const unsigned long long later = __ballot(opened && rank >= most);
			const int window = later == 0 ? seen : __builtin_ctzll(later);
			if(mine)
			{
				w.open_node[rank] = node;
				w.open_mask[rank] = w.open[at];
			}
			__builtin_amdgcn_wave_barrier();
			const bool born = lane < 2 * used;
			const int child = born ? 2 * w.open_node[lane >> 1] + (lane & 1) : kRoot;
			const unsigned parents = born ? w.open_mask[lane >> 1] : 0u;
			const double4 c = xyzr[child];
			// the nearest and the farthest point of the bodies' box, against the test
			// d2 > crit: rounding moves either side by less than 1e-14 of it, and 1e-300
			// stands above what underflow can take
			double near2 = 0.0, far2 = 0.0;
			{
				const double ax = lo.x - c.x, bx = c.x - hi.x;
				const double ay = lo.y - c.y, by = c.y - hi.y;
				const double az = lo.z - c.z, bz = c.z - hi.z;
				const double ex = fmax(fmax(ax, bx), 0.0), ey = fmax(fmax(ay, by), 0.0), ez = fmax(fmax(az, bz), 0.0);
				const double fx = fmax(fabs(ax), fabs(bx)), fy = fmax(fabs(ay), fabs(by)), fz = fmax(fabs(az), fabs(bz));
				near2 = fma(ez, ez, fma(ey, ey, ex * ex));
				far2 = fma(fz, fz, fma(fy, fy, fx * fx));
			}
			const bool all_pass = box_holds && far2 == far2 && fma(near2, 1.0 - 1e-12, -1e-300) > c.w;
			const bool none_pass = box_holds && fma(far2, 1.0 + 1e-12, 1e-300) < c.w;
			const bool undecided = born && !all_pass && !none_pass;
			const unsigned long long und = __ballot(undecided);
			unsigned pass = all_pass ? ~0u : 0u;
			if(und != 0)
			{
				const int place = below(und);
				const int tests = (__popcll(und) + 1) / 2;      // two children each
				if(undecided) { w.rec[place] = c; }
				__builtin_amdgcn_wave_barrier();
				for(int p0 = 0; p0 < tests; p0 += 4)
				{
					double r[4], d[4], dy[4], dz[4];
#pragma unroll
					for(int k = 0; k < 4; ++k)
					{
						// records beyond the undecided ones are old ones; their results are not read
						const double4 nd = w.rec[(2 * (p0 + k) + upper) & (kWalkEntries - 1)];
						r[k] = nd.w;
						d[k] = me.x - nd.x;
						dy[k] = me.y - nd.y;
						dz[k] = me.z - nd.z;
					}
#pragma unroll
					for(int k = 0; k < 4; ++k) { d[k] = d[k] * d[k]; }
#pragma unroll
					for(int k = 0; k < 4; ++k) { dy[k] = dy[k] * dy[k]; }
#pragma unroll
					for(int k = 0; k < 4; ++k) { d[k] = d[k] + dy[k]; }
#pragma unroll
					for(int k = 0; k < 4; ++k) { dz[k] = dz[k] * dz[k]; }
#pragma unroll
					for(int k = 0; k < 4; ++k) { d[k] = d[k] + dz[k]; }
					unsigned long long b[4];
#pragma unroll
					for(int k = 0; k < 4; ++k) { b[k] = __ballot(d[k] > r[k]); }
					if(lane < 8)
					{
						const unsigned long long m = (lane & 4) ? ((lane & 2) ? b[3] : b[2]) : ((lane & 2) ? b[1] : b[0]);
						w.passed[2 * p0 + lane] = static_cast<unsigned>(lane & 1 ? m >> 32 : m);
					}
				}
				__builtin_amdgcn_wave_barrier();
				if(undecided) { pass = w.passed[place]; }
			}
			if(born)
			{
				const unsigned taken = pass & parents;
				w.child[lane] = make_uint2(taken, child < n ? parents & ~taken : 0u);
				vis += __popc(parents);
				inter += __popc(taken);
			}
			__builtin_amdgcn_wave_barrier();
			// what every element of the window leaves
			const bool stays = have && lane >= lead && lane < window && !opened;
			uint2 l = make_uint2(0u, 0u), r = make_uint2(0u, 0u);
			if(mine)
			{
				l = w.child[2 * rank];
				r = w.child[2 * rank + 1];
			}
			const bool self = stays || (mine && take != 0);
			const bool left = (l.x | l.y) != 0;
			const bool right = (r.x | r.y) != 0;
			const unsigned long long bs = __ballot(self), bl = __ballot(left), br = __ballot(right);
			int pos = sp - window + __popcll(bs) + __popcll(bl) + __popcll(br);
			sp = pos;
			pos -= 1 + below(bs) + below(bl) + below(br);
			__builtin_amdgcn_wave_barrier();
			if(self)
			{
				w.node[pos] = node;
				w.take[pos] = take;
				w.open[pos] = 0;
				--pos;
			}
			if(left)
			{
				w.node[pos] = 2 * node;
				w.take[pos] = l.x;
				w.open[pos] = l.y;
				--pos;
			}
			if(right)
			{
				w.node[pos] = 2 * node + 1;
				w.take[pos] = r.x;
				w.open[pos] = r.y;
			}
		}
		else
		{
			sp -= lead;
		}
	}
	// the last chunk leaves the sums in the lower half
	if(active && upper == 0) { write_f(y, mass, f, n, body_n[tn], tx, ty, tz); }
	count_add(counters, inter, vis);
}

// FP32 interaction math: FP64 offsets to the node centre are rounded to FP32,
// the opening test and the monopole term run in FP32 with v_rsq_f32; sums in
// FP32 with a Kahan carry.
__global__ void __launch_bounds__(256)
k_bh_stackless32(const double4* __restrict__ xyzr, const double* __restrict__ nmass,
                 const int32_t* __restrict__ body_n, const double* __restrict__ y, const double* __restrict__ mass,
                 double* __restrict__ f, int n, unsigned long long* __restrict__ counters)
{
	const int t = blockIdx.x * blockDim.x + threadIdx.x;
	const int tree_size = 2 * n;
	unsigned long long inter = 0, vis = 0;
	if(t < n)
	{
		const int tn = n + t;
		const double4 me = xyzr[tn];
		float ax = 0.0f, ay = 0.0f, az = 0.0f, cx = 0.0f, cy = 0.0f, cz = 0.0f;
		int curr = kRoot;
		do
		{
			const double4 nd = xyzr[curr];
			const float dx = static_cast<float>(nd.x - me.x);
			const float dy = static_cast<float>(nd.y - me.y);
			const float dz = static_cast<float>(nd.z - me.z);
			const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
			++vis;
			if(d2 > static_cast<float>(nd.w))
			{
				const float r2 = fmaxf(d2, 1e-8f);
				const float ri = __builtin_amdgcn_rsqf(r2);
				const float w = (static_cast<float>(nmass[curr]) * ri) * (ri * ri);
				float v = dx * w - cx; float s = ax + v; cx = (s - ax) - v; ax = s;
				v = dy * w - cy; s = ay + v; cy = (s - ay) - v; ay = s;
				v = dz * w - cz; s = az + v; cz = (s - az) - v; az = s;
				++inter;
				curr = next_down(curr);
			}
			else
			{
				curr = next_up(curr, tree_size);
			}
		}
		while(curr != kRoot);
		const int b = body_n[tn];
		f[b] = y[3 * n + b];
		f[n + b] = y[4 * n + b];
		f[2 * n + b] = y[5 * n + b];
		f[3 * n + b] = static_cast<double>(ax) - static_cast<double>(cx);
		f[4 * n + b] = static_cast<double>(ay) - static_cast<double>(cy);
		f[5 * n + b] = static_cast<double>(az) - static_cast<double>(cz);
	}
	count_add(counters, inter, vis);
}

// ---------------------------------------------------------------------------
// group walk: one wave per subtree of 64 leaves
// ---------------------------------------------------------------------------
// The 64 targets of a wave are the leaves of one heap node g, whose tight box
// bounds them all.  The wave walks the tree once for the whole group, 64 nodes
// per step from an LDS stack: a leaf is always taken as a body; an internal node
// is taken as a monopole when the distance from the group box to its mass
// centre exceeds its opening radius (then every target of the group accepts it
// too, so the cell set refines each target's own walk); otherwise its children
// are pushed.  Accepted entries are buffered in LDS as FP32 offsets from the
// box centre and swept by all 64 lanes, the same pair arithmetic as the direct
// FP32 kernel.  No node is dropped: a child push that would overflow the stack
// takes the node as a monopole instead (counted in counters[2]).
constexpr int kGroup = 64;
constexpr int kWalkStack = 1024;   // entries of sibling pairs; (levels + 2) * 32 suffice
constexpr int kWalkBuf = 128;

// Group handled by this work-group.  Work-groups are dispatched round-robin
// over the 8 XCDs, each with its own L2; consecutive groups are spatial
// neighbours that read mostly the same tree nodes, so the ids are permuted to
// give each XCD one contiguous run of groups (when their count divides by 8).
constexpr int kXcds = 8;

__device__ inline int xcd_group(int block, int nblocks)
{
	if(nblocks % kXcds != 0) { return block; }
	return (block % kXcds) * (nblocks / kXcds) + block / kXcds;
}


// Half the diagonal of a box.
__device__ inline double half_diagonal(double x0, double y0, double z0, double x1, double y1, double z1)
{
	const double ex = x1 - x0, ey = y1 - y0, ez = z1 - z0;
	return 0.5 * sqrt(ex * ex + ey * ey + ez * ez);
}

// The walk stack holds sibling pairs: an even entry e stands for the nodes e and
// e + 1, the odd entry kRoot for the root alone.  A step pops up to 32 entries,
// one node per lane (lane 2i takes the left node of entry i, lane 2i + 1 the
// right one); every node the step opens pushes one entry, its two children.
// Popped in this order, the stack never holds more than (levels + 2) * 32
// entries.  In the Morton tree (kRadix) an entry encodes the children of the
// opened node (radix_kids), so that popping reads no memory, and 0 stands for
// the root alone.
template <bool kRadix = false>
__device__ inline int walk_pop(const int* stack, int& sp, int lane, bool& valid, int n = 0)
{
	const int cnt = sp < kGroup / 2 ? sp : kGroup / 2;
	const int i = lane >> 1;
	int node = kRoot;
	valid = false;
	if(i < cnt)
	{
		const int e = stack[sp - cnt + i];
		if constexpr(kRadix)
		{
			if(e == 0)
			{
				valid = (lane & 1) == 0;
			}
			else
			{
				// g = split + 1; bit 30: the left child is leaf n + g - 1 (else
				// internal id g), bit 31: the right child is leaf n + g (else g + 1)
				const unsigned u = static_cast<unsigned>(e);
				const int g = static_cast<int>(u & 0x3fffffffu);
				node = (lane & 1) ? ((u >> 31) ? n + g : g + 1) : (((u >> 30) & 1u) ? n + g - 1 : g);
				valid = true;
			}
		}
		else
		{
			node = e == kRoot ? kRoot : e + (lane & 1);
			valid = e != kRoot || (lane & 1) == 0;
		}
	}
	sp -= cnt;
	return node;
}

// Stack entry of an opened node (in the Morton tree: from its children kids,
// which are leaf n + s / internal id s + 1 and leaf n + s + 1 / internal id s + 2
// for the split s), and the entry the walk starts from.
template <bool kRadix>
__device__ inline int walk_entry(int node, int2 kids = make_int2(0, 0), int n = 0)
{
	if constexpr(kRadix)
	{
		const unsigned g = static_cast<unsigned>(kids.x < n ? kids.x : kids.x - n + 1);
		return static_cast<int>(g | (kids.x >= n ? 1u << 30 : 0u) | (kids.y >= n ? 1u << 31 : 0u));
	}
	return 2 * node;
}
template <bool kRadix>
__device__ inline int walk_start() { return kRadix ? 0 : kRoot; }

// The group walks sweep in scaled units: offsets x' = 1e4 x, masses m' = 1e8 m
// and second moments Q' = 1e16 Q (mass x length^2), each formed in FP64 and
// rounded once.  r'^2 >= 1 is then the reference's clamp r^2 >= 1e-8
// (nbody/nbody_data.cpp:35-44), which the [0, 1] output clamp of v_rsq_f32
// applies at no cost: q = min(1/r', 1) = 1e-4 / sqrt(max(r^2, 1e-8)), and the
// monopole term m' x' q^3 and the quadrupole term below come out in unscaled
// acceleration units.
constexpr double kSweepLen = 1e4;
constexpr double kSweepMass = 1e8;
constexpr double kSweepQuad = 1e16;

__device__ inline float rsq_clamped(float r2)
{
	return __builtin_amdgcn_fmed3f(__builtin_amdgcn_rsqf(r2), 0.0f, 1.0f);   // folds into v_rsq_f32 clamp
}

// Sweep entry (scaled offset from the group centre, scaled mass) of a node.
__device__ inline float4 sweep_entry(const double4& rec, double m, double ccx, double ccy, double ccz)
{
	return make_float4(static_cast<float>((rec.x - ccx) * kSweepLen), static_cast<float>((rec.y - ccy) * kSweepLen),
	                   static_cast<float>((rec.z - ccz) * kSweepLen), static_cast<float>(m * kSweepMass));
}

// Pop the next chunk of the walk stack (walk_pop) and request its node records;
// returns the number of stack entries taken.
// In the Morton tree the children of internal nodes are requested with the
// records (kids), for the stack entries of the nodes the step opens; kQ: the
// second moments too (q), from the same 64-byte record.
template <bool kRadix = false, bool kQ = false>
__device__ inline int walk_fetch(const int* stack, int& sp, int lane, const nbh_walk_rec* __restrict__ wr, int& node,
                                 bool& valid, double4& rec, double& m, int2& kids, const int2* __restrict__ child = nullptr,
                                 int n = 0, float* q = nullptr)
{
	const int cnt = sp < kGroup / 2 ? sp : kGroup / 2;
	node = walk_pop<kRadix>(stack, sp, lane, valid, n);
	rec = make_double4(0.0, 0.0, 0.0, 0.0);
	m = 0.0;
	kids = make_int2(0, 0);
	if constexpr(kQ)
	{
		for(int k = 0; k < 6; ++k) { q[k] = 0.0f; }
	}
	if(valid)
	{
		rec = wr[node].c;
		m = wr[node].m;
		if constexpr(kQ)
		{
			for(int k = 0; k < 6; ++k) { q[k] = wr[node].q[k]; }
		}
		if(kRadix && node < n) { kids = child[node]; }
	}
	return cnt;
}

__device__ inline void sweep32(const float4* __restrict__ buf, int count, float tx, float ty, float tz,
                               float& ax, float& ay, float& az, float& cx, float& cy, float& cz)
{
	float px = 0.0f, py = 0.0f, pz = 0.0f;
#pragma unroll 4
	for(int j = 0; j < count; ++j)
	{
		const float4 s = buf[j];
		const float dx = s.x - tx;
		const float dy = s.y - ty;
		const float dz = s.z - tz;
		const float ri = rsq_clamped(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
		const float w = (s.w * ri) * (ri * ri);
		px = fmaf(dx, w, px);
		py = fmaf(dy, w, py);
		pz = fmaf(dz, w, pz);
	}
	float v = px - cx; float t = ax + v; cx = (t - ax) - v; ax = t;
	v = py - cy; t = ay + v; cy = (t - ay) - v; ay = t;
	v = pz - cz; t = az + v; cz = (t - az) - v; az = t;
}

// sweep32 for kT bodies of one lane at once: each buffer entry is read once
// for all of them, and their independent chains interleave.  Every body's sums
// take the same operations in the same order as sweep32's.
template <int kT>
__device__ inline void sweep32_n(const float4* __restrict__ buf, int count, const float* tx, const float* ty,
                                 const float* tz, float* ax, float* ay, float* az, float* cx, float* cy, float* cz)
{
	float px[kT], py[kT], pz[kT];
#pragma unroll
	for(int t = 0; t < kT; ++t) { px[t] = py[t] = pz[t] = 0.0f; }
	// four chains in flight (one body per lane: 2^18 bodies, monopole, 1.85 ms
	// against 1.94 with two)
#pragma unroll kT == 1 ? 4 : 2
	for(int j = 0; j < count; ++j)
	{
		const float4 s = buf[j];
#pragma unroll
		for(int t = 0; t < kT; ++t)
		{
			const float dx = s.x - tx[t];
			const float dy = s.y - ty[t];
			const float dz = s.z - tz[t];
			const float ri = rsq_clamped(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
			const float w = (s.w * ri) * (ri * ri);
			px[t] = fmaf(dx, w, px[t]);
			py[t] = fmaf(dy, w, py[t]);
			pz[t] = fmaf(dz, w, pz[t]);
		}
	}
#pragma unroll
	for(int t = 0; t < kT; ++t)
	{
		float v = px[t] - cx[t]; float u = ax[t] + v; cx[t] = (u - ax[t]) - v; ax[t] = u;
		v = py[t] - cy[t]; u = ay[t] + v; cy[t] = (u - ay[t]) - v; ay[t] = u;
		v = pz[t] - cz[t]; u = az[t] + v; cz[t] = (u - az[t]) - v; az[t] = u;
	}
}

// Cells waiting for the monopole + quadrupole sweep, 40 bytes each in LDS:
// e0 = (mass-centre offset from the group centre, M), e1 = 2.5 x (Q'xx Q'yy
// Q'zz Q'xy), e2 = 2.5 x (Q'xz Q'yz), with Q' = 3 Q - tr(Q) I the traceless
// second moment about the mass centre (all scaled as the sweeps are).
template <int kN>
struct quad_lds {
	float4 e0[kN];
	float4 e1[kN];
	float2 e2[kN];
};

// Monopole + quadrupole field of the cells in qb at the lane's body; with
// r = cm - x, d = |r|, u = 1/d:
//   a = M r / d^3 + (2.5 (r.Q'.r) / d^2 r - Q' r) / d^5
//     = (M + s u^4) u^3 r - 0.4 u^5 (2.5 Q' r),   s = r.(2.5 Q').r,
// all in the scaled units of sweep32 (Q' times kSweepQuad).  Kahan per sweep.
template <int kN>
__device__ inline void sweep_mq(const quad_lds<kN>& qb, int count, float tx, float ty, float tz, float& ax, float& ay,
                                float& az, float& cx, float& cy, float& cz)
{
	float px = 0.0f, py = 0.0f, pz = 0.0f;
	for(int j = 0; j < count; ++j)
	{
		const float4 e0 = qb.e0[j], e1 = qb.e1[j];
		const float2 e2 = qb.e2[j];
		const float rx = e0.x - tx, ry = e0.y - ty, rz = e0.z - tz;
		const float u = rsq_clamped(fmaf(rz, rz, fmaf(ry, ry, rx * rx)));
		const float u2 = u * u;
		const float u3 = u2 * u;
		const float u4 = u2 * u2;
		const float Qx = fmaf(e1.x, rx, fmaf(e1.w, ry, e2.x * rz));
		const float Qy = fmaf(e1.w, rx, fmaf(e1.y, ry, e2.y * rz));
		const float Qz = fmaf(e2.x, rx, fmaf(e2.y, ry, e1.z * rz));
		const float s = fmaf(rx, Qx, fmaf(ry, Qy, rz * Qz));
		const float k = fmaf(s, u4, e0.w) * u3;
		const float g = -0.4f * (u4 * u);
		px = fmaf(rx, k, fmaf(Qx, g, px));
		py = fmaf(ry, k, fmaf(Qy, g, py));
		pz = fmaf(rz, k, fmaf(Qz, g, pz));
	}
	float v = px - cx; float t = ax + v; cx = (t - ax) - v; ax = t;
	v = py - cy; t = ay + v; cy = (t - ay) - v; ay = t;
	v = pz - cz; t = az + v; cz = (t - az) - v; az = t;
}

// sweep_mq for kT bodies of one lane at once (as sweep32_n: one read of each
// cell, the same operations per body as sweep_mq).
template <int kT, int kN>
__device__ inline void sweep_mq_n(const quad_lds<kN>& qb, int count, const float* tx, const float* ty, const float* tz,
                                  float* ax, float* ay, float* az, float* cx, float* cy, float* cz)
{
	float px[kT], py[kT], pz[kT];
#pragma unroll
	for(int t = 0; t < kT; ++t) { px[t] = py[t] = pz[t] = 0.0f; }
	for(int j = 0; j < count; ++j)
	{
		const float4 e0 = qb.e0[j], e1 = qb.e1[j];
		const float2 e2 = qb.e2[j];
#pragma unroll
		for(int t = 0; t < kT; ++t)
		{
			const float rx = e0.x - tx[t], ry = e0.y - ty[t], rz = e0.z - tz[t];
			const float u = rsq_clamped(fmaf(rz, rz, fmaf(ry, ry, rx * rx)));
			const float u2 = u * u;
			const float u3 = u2 * u;
			const float u4 = u2 * u2;
			const float Qx = fmaf(e1.x, rx, fmaf(e1.w, ry, e2.x * rz));
			const float Qy = fmaf(e1.w, rx, fmaf(e1.y, ry, e2.y * rz));
			const float Qz = fmaf(e2.x, rx, fmaf(e2.y, ry, e1.z * rz));
			const float s = fmaf(rx, Qx, fmaf(ry, Qy, rz * Qz));
			const float k = fmaf(s, u4, e0.w) * u3;
			const float g = -0.4f * (u4 * u);
			px[t] = fmaf(rx, k, fmaf(Qx, g, px[t]));
			py[t] = fmaf(ry, k, fmaf(Qy, g, py[t]));
			pz[t] = fmaf(rz, k, fmaf(Qz, g, pz[t]));
		}
	}
#pragma unroll
	for(int t = 0; t < kT; ++t)
	{
		float v = px[t] - cx[t]; float w = ax[t] + v; cx[t] = (w - ax[t]) - v; ax[t] = w;
		v = py[t] - cy[t]; w = ay[t] + v; cy[t] = (w - ay[t]) - v; ay[t] = w;
		v = pz[t] - cz[t]; w = az[t] + v; cz[t] = (w - az[t]) - v; az[t] = w;
	}
}

// Cells waiting for the monopole + quadrupole sweep; a sweep runs before a
// step whenever more than kQuadBuf - 64 wait.
constexpr int kQuadBuf = 88;

// Entry of a node (scaled mass-centre offset and mass in ent, second moments Q)
// at slot `slot` of qb, with the 2.5 x Q' that sweep_mq expects.
template <int kN>
__device__ inline void put_quad(quad_lds<kN>& qb, int slot, const float4& ent, const float* __restrict__ Q)
{
	const float q0 = Q[0], q1 = Q[1], q2 = Q[2], q3 = Q[3], q4 = Q[4], q5 = Q[5];
	const float tr = q0 + q1 + q2;
	const float k = static_cast<float>(2.5 * kSweepQuad);
	qb.e0[slot] = ent;
	qb.e1[slot] = make_float4((3.0f * q0 - tr) * k, (3.0f * q1 - tr) * k, (3.0f * q2 - tr) * k, 3.0f * q3 * k);
	qb.e2[slot] = make_float2(3.0f * q4 * k, 3.0f * q5 * k);
}

// Quadrupole field at the group centre of a cell whose mass centre sits at r
// from it, and its Jacobian, added to acc[9] (field, then J as xx yy zz xy xz
// yz).  With Q' = 3 Q - tr(Q) I, s = r.Q'.r and d = |r|:
//   g = (2.5 s / d^2 r - Q' r) / d^5,
//   G = dg/dr = (5 (r (Q'r)' + (Q'r) r') + 2.5 s I) / d^7 - 17.5 s r r' / d^9 - Q' / d^5,
// and since r = cm - x, the field at centre + delta is g - G delta: J = -G.
__device__ inline void quad_expansion(float rx, float ry, float rz, float qxx, float qyy, float qzz, float qxy,
                                      float qxz, float qyz, float* acc)
{
	const float Qx = fmaf(qxx, rx, fmaf(qxy, ry, qxz * rz));
	const float Qy = fmaf(qxy, rx, fmaf(qyy, ry, qyz * rz));
	const float Qz = fmaf(qxz, rx, fmaf(qyz, ry, qzz * rz));
	const float sq = fmaf(rx, Qx, fmaf(ry, Qy, rz * Qz));
	const float ri = __builtin_amdgcn_rsqf(fmaf(rz, rz, fmaf(ry, ry, rx * rx)));
	const float ri2 = ri * ri;
	const float ri5 = (ri2 * ri2) * ri;
	const float ri7 = ri5 * ri2;
	const float c = 2.5f * sq * ri7;
	acc[0] += fmaf(c, rx, -Qx * ri5);
	acc[1] += fmaf(c, ry, -Qy * ri5);
	acc[2] += fmaf(c, rz, -Qz * ri5);
	const float a = 5.0f * ri7;
	const float e = 17.5f * sq * (ri7 * ri2);
	acc[3] -= a * (2.0f * rx * Qx) + c - e * rx * rx - qxx * ri5;
	acc[4] -= a * (2.0f * ry * Qy) + c - e * ry * ry - qyy * ri5;
	acc[5] -= a * (2.0f * rz * Qz) + c - e * rz * rz - qzz * ri5;
	acc[6] -= a * (rx * Qy + ry * Qx) - e * rx * ry - qxy * ri5;
	acc[7] -= a * (rx * Qz + rz * Qx) - e * rx * rz - qxz * ri5;
	acc[8] -= a * (ry * Qz + rz * Qy) - e * ry * rz - qyz * ri5;
}

// Monopole field of a cell of mass M whose mass centre sits at r from the group
// centre, expanded about the centre to third order, added to acc[34]: field
// acc[0..2], Jacobian acc[3..8] (xx yy zz xy xz yz, as quad_expansion), the sum
// T = M r r r / d^7 in acc[9..18] (xxx xxy xxz xyy xyz xzz yyy yyz yzz zzz) and
// W = M r r r r / d^9 in acc[19..33] (xxxx xxxy xxxz xxyy xxyz xxzz xyyy xyyz
// xyzz xzzz yyyy yyyz yyzz yzzz zzzz).  With f(r) = M r / d^3, the field at
// centre + delta is f(r - delta):
//   a(delta) = f - D1 delta + 1/2 D2[delta^2] - 1/6 D3[delta^3] + O(|delta|^4),
//   D1 = M (I / d^3 - 3 r r' / d^5)            (J = -D1),
//   1/2 D2[delta^2] = -3 (V.delta) delta - 1.5 |delta|^2 V + 7.5 T[delta^2],
//   -1/6 D3[delta^3] = 1.5 s |delta|^2 delta - 7.5 (delta.A.delta) delta
//                      - 7.5 |delta|^2 A delta + 17.5 W[delta^3],
// where V = sum M r / d^5 = T_ikk, A = sum M r r' / d^7 = W_ijkk and
// s = sum M / d^5 = A_kk, so only T and W are accumulated (local_terms
// evaluates the last two lines per body).
__device__ inline void local_expansion(float rx, float ry, float rz, float M, float* acc)
{
	const float u = __builtin_amdgcn_rsqf(fmaf(rz, rz, fmaf(ry, ry, rx * rx)));
	const float u2 = u * u;
	const float w3 = (M * u) * u2;
	const float w5 = w3 * u2;
	const float w7 = w5 * u2;
	acc[0] = fmaf(w3, rx, acc[0]);
	acc[1] = fmaf(w3, ry, acc[1]);
	acc[2] = fmaf(w3, rz, acc[2]);
	const float t5 = 3.0f * w5;
	const float tx = t5 * rx, ty = t5 * ry;
	acc[3] += fmaf(tx, rx, -w3);
	acc[4] += fmaf(ty, ry, -w3);
	acc[5] += fmaf(t5 * rz, rz, -w3);
	acc[6] = fmaf(tx, ry, acc[6]);
	acc[7] = fmaf(tx, rz, acc[7]);
	acc[8] = fmaf(ty, rz, acc[8]);
	const float px = w7 * rx, py = w7 * ry, pz = w7 * rz;
	const float xx = rx * rx, yy = ry * ry, zz = rz * rz;
	acc[9] = fmaf(px, xx, acc[9]);
	acc[10] = fmaf(px * rx, ry, acc[10]);
	acc[11] = fmaf(px * rx, rz, acc[11]);
	acc[12] = fmaf(px, yy, acc[12]);
	acc[13] = fmaf(px * ry, rz, acc[13]);
	acc[14] = fmaf(px, zz, acc[14]);
	acc[15] = fmaf(py, yy, acc[15]);
	acc[16] = fmaf(py * ry, rz, acc[16]);
	acc[17] = fmaf(py, zz, acc[17]);
	acc[18] = fmaf(pz, zz, acc[18]);
	const float w9 = w7 * u2;
	const float a = w9 * xx, b = w9 * yy, c = w9 * zz;
	const float xy = rx * ry, xz = rx * rz, yz = ry * rz;
	acc[19] = fmaf(a, xx, acc[19]);
	acc[20] = fmaf(a, xy, acc[20]);
	acc[21] = fmaf(a, xz, acc[21]);
	acc[22] = fmaf(a, yy, acc[22]);
	acc[23] = fmaf(a, yz, acc[23]);
	acc[24] = fmaf(a, zz, acc[24]);
	acc[25] = fmaf(b, xy, acc[25]);
	acc[26] = fmaf(b, xz, acc[26]);
	acc[27] = fmaf(c, xy, acc[27]);
	acc[28] = fmaf(c, xz, acc[28]);
	acc[29] = fmaf(b, yy, acc[29]);
	acc[30] = fmaf(b, yz, acc[30]);
	acc[31] = fmaf(b, zz, acc[31]);
	acc[32] = fmaf(c, yz, acc[32]);
	acc[33] = fmaf(c, zz, acc[33]);
}

// Second- and third-order terms of the local expansion (T = acc[9..18] and
// W = acc[19..33] of local_expansion, summed over the cells) at offset
// (dx, dy, dz) from the group centre.
__device__ inline void local_terms(const float* T, float dx, float dy, float dz, float& ox, float& oy, float& oz)
{
	const float vx = T[0] + T[3] + T[5], vy = T[1] + T[6] + T[8], vz = T[2] + T[7] + T[9];
	const float xx = dx * dx, yy = dy * dy, zz = dz * dz;
	const float xy2 = 2.0f * dx * dy, xz2 = 2.0f * dx * dz, yz2 = 2.0f * dy * dz;
	const float tdx = T[0] * xx + T[3] * yy + T[5] * zz + T[1] * xy2 + T[2] * xz2 + T[4] * yz2;
	const float tdy = T[1] * xx + T[6] * yy + T[8] * zz + T[3] * xy2 + T[4] * xz2 + T[7] * yz2;
	const float tdz = T[2] * xx + T[7] * yy + T[9] * zz + T[4] * xy2 + T[5] * xz2 + T[8] * yz2;
	const float vd = vx * dx + vy * dy + vz * dz;
	const float dd = xx + yy + zz;
	ox = -3.0f * vd * dx - 1.5f * dd * vx + 7.5f * tdx;
	oy = -3.0f * vd * dy - 1.5f * dd * vy + 7.5f * tdy;
	oz = -3.0f * vd * dz - 1.5f * dd * vz + 7.5f * tdz;
	const float* W = T + 10;
	// monomials of delta^3 times their multiplicities
	const float m0 = xx * dx, m1 = 3.0f * xx * dy, m2 = 3.0f * xx * dz, m3 = 3.0f * dx * yy, m4 = 3.0f * xy2 * dz;
	const float m5 = 3.0f * dx * zz, m6 = yy * dy, m7 = 3.0f * yy * dz, m8 = 3.0f * dy * zz, m9 = zz * dz;
	const float wx = W[0] * m0 + W[1] * m1 + W[2] * m2 + W[3] * m3 + W[4] * m4 + W[5] * m5 + W[6] * m6 + W[7] * m7 +
	                 W[8] * m8 + W[9] * m9;
	const float wy = W[1] * m0 + W[3] * m1 + W[4] * m2 + W[6] * m3 + W[7] * m4 + W[8] * m5 + W[10] * m6 +
	                 W[11] * m7 + W[12] * m8 + W[13] * m9;
	const float wz = W[2] * m0 + W[4] * m1 + W[5] * m2 + W[7] * m3 + W[8] * m4 + W[9] * m5 + W[11] * m6 +
	                 W[12] * m7 + W[13] * m8 + W[14] * m9;
	const float axx = W[0] + W[3] + W[5], ayy = W[3] + W[10] + W[12], azz = W[5] + W[12] + W[14];
	const float axy = W[1] + W[6] + W[8], axz = W[2] + W[7] + W[9], ayz = W[4] + W[11] + W[13];
	const float adx = axx * dx + axy * dy + axz * dz;
	const float ady = axy * dx + ayy * dy + ayz * dz;
	const float adz = axz * dx + ayz * dy + azz * dz;
	const float dad = dx * adx + dy * ady + dz * adz;
	const float s5 = 1.5f * (axx + ayy + azz) * dd - 7.5f * dad;
	ox += s5 * dx - 7.5f * dd * adx + 17.5f * wx;
	oy += s5 * dy - 7.5f * dd * ady + 17.5f * wy;
	oz += s5 * dz - 7.5f * dd * adz + 17.5f * wz;
}

// Far cells wait in an LDS ring of kFarRing node numbers and are expanded 64 at
// a time, one per lane, so the expansion runs on full waves; the expansion
// reads the node's mass centre, mass and second moments from its record again
// (one cache line the walk step has just read).  A walk step adds at most 64
// entries and a batch is taken as soon as 64 wait, so at most 127 are ever
// pending.
constexpr int kFarRing = 128;

// Expand `count` (<= 64) ring entries from `head`, one per lane, about the
// centre (ccx, ccy, ccz): offsets of the mass centres from it, unscaled.
template <bool kLocal>
__device__ inline void far_batch(const int* fn, const nbh_walk_rec* __restrict__ wr, int head, int count, int lane,
                                 double ccx, double ccy, double ccz, float* acc)
{
	if(lane < count)
	{
		const int s = (head + lane) & (kFarRing - 1);
		const nbh_walk_rec* r = wr + fn[s];
		const double4 c = r->c;
		const float4 e = make_float4(static_cast<float>(c.x - ccx), static_cast<float>(c.y - ccy),
		                             static_cast<float>(c.z - ccz), static_cast<float>(r->m));
		const float* Q = r->q;
		const float q0 = Q[0], q1 = Q[1], q2 = Q[2], q3 = Q[3], q4 = Q[4], q5 = Q[5];
		const float tr = q0 + q1 + q2;
		quad_expansion(e.x, e.y, e.z, 3.0f * q0 - tr, 3.0f * q1 - tr, 3.0f * q2 - tr, 3.0f * q3, 3.0f * q4, 3.0f * q5,
		               acc);
		if constexpr(kLocal) { local_expansion(e.x, e.y, e.z, e.w, acc); }
	}
}

// Two-level local walk.  A super-group is the heap node of 2^kSuperShift
// consecutive groups (1024 bodies).  One wave walks the tree once for the
// super-group's box: a node it accepts is accepted by every group inside that
// box too (the distance from a smaller box inside is no shorter), so accepted
// cells at least near_k half-diagonals of the super box from its centre go into
// one local expansion about that centre (far_batch, third order).  Every other
// accepted node, and every rejected node whose bodies all lie within that
// distance, goes into a list instead of being opened; other rejected nodes are
// opened.  Each group then walks from the listed nodes instead of the
// root, with its own acceptance test (so near its box the cells are those of
// its own walk), sweeping and expanding about its own centre as the one-level
// walk does; each body adds both expansions.  A list longer than `cap`, or a
// stack spill in the super walk, makes the groups of that super-group walk from
// the root instead.  The super-group's near distance is max(near_k,
// kSuperNearMin) half-diagonals of its box: rejected nodes are then listed
// higher up the tree, for each group to open with its own test.  Measured at
// 2^22 Plummer bodies, theta 0.65, near_k 4: walk 52.7 -> 51.8 ms, RMS 1.0e-3 ->
// 9.9e-4; at theta 0.6, near_k 3 no list overflows where near_k alone had some.
constexpr int kSuperShift = 4;
constexpr float kSuperNearMin = 5.0f;

// The tree a group walk runs on.  Heap (child == nullptr): children of node k
// are 2k and 2k + 1, and the walk groups and super-groups are the heap nodes
// of 64 and 1024 bodies.  Morton tree: the children of internal id k are
// child[k]; group g is grp[g] = (node id, first sorted leaf, leaves (<= kRadixWalk),
// super-group or -1) and super-group s is sup[s] = (node id, first leaf).  In
// both, a group's or super-group's box is its node's box.
struct WalkTree {
	const int2* child = nullptr;
	const int4* grp = nullptr;
	const int2* sup = nullptr;
	int         ngroups = 0;
	int         nsupers = 0;
};

struct TwoLevel {
	int*   lists = nullptr;   // [super][cap] listed nodes
	int*   count = nullptr;   // [super] list length (> cap: overflowed)
	float* coef = nullptr;    // [super][34] expansion about the super box centre (local_expansion layout)
	int    cap = 0;
	// optional: the super-group's far cells, for the learned correction
	int*   far_list = nullptr;   // [super][far_cap] far nodes, in walk order
	int*   far_count = nullptr;  // [super] far cells found (> far_cap: the rest are not listed)
	int    far_cap = 0;
};

// Next 64 listed nodes from position pos and their records; `entry` holds this
// lane's list entry, read one list step ahead, and takes that of the next step.
template <bool kRadix = false, bool kQ = false>
__device__ inline void list_fetch(const int* __restrict__ list, int pos, int count, int lane,
                                  const nbh_walk_rec* __restrict__ wr, int& entry, int& node, bool& valid,
                                  double4& rec, double& m, int2& kids, const int2* __restrict__ child = nullptr,
                                  int n = 0, float* q = nullptr)
{
	const int i = pos + lane;
	valid = i < count;
	node = valid ? entry : kRoot;
	rec = make_double4(0.0, 0.0, 0.0, 0.0);
	m = 0.0;
	kids = make_int2(0, 0);
	if constexpr(kQ)
	{
		for(int k = 0; k < 6; ++k) { q[k] = 0.0f; }
	}
	if(valid)
	{
		rec = wr[node].c;
		m = wr[node].m;
		if constexpr(kQ)
		{
			for(int k = 0; k < 6; ++k) { q[k] = wr[node].q[k]; }
		}
		if(kRadix && node < n) { kids = child[node]; }
	}
	entry = i + kGroup < count ? list[i + kGroup] : kRoot;
}

// kQuad: internal cells taken as monopoles also contribute their quadrupole
// term (second central moments `quad`).  A cell whose mass centre lies within
// `near` of the group centre gets it per body (fused monopole + quadrupole
// sweep); a farther one gets the monopole per body and its quadrupole field
// expanded to first order about the group centre, once per group.
// kLocal (with kQuad): a far cell's monopole field is expanded too, to third
// order (local_expansion), instead of being swept per body.  kTwo (with kLocal):
// the group takes its super-group's list instead of walking (TwoLevel).
template <bool kQuad, bool kLocal, bool kTwo, bool kRadix>
__device__ inline void group_walk_one(int gi, int* __restrict__ stack, float4* __restrict__ buf,
                                      quad_lds<kQuad ? kQuadBuf : 1>& qbuf, int* __restrict__ farn,
                                      const nbh_walk_rec* __restrict__ wr, const double* __restrict__ bmin,
                                      const double* __restrict__ bmax, const int32_t* __restrict__ body_n,
                                      const double* __restrict__ y, double* __restrict__ f, int n, float near_k,
                                      unsigned long long* __restrict__ counters, const TwoLevel& two,
                                      const WalkTree& tree)
{
	const int lane = threadIdx.x;
	// the group's node, first leaf, size and super-group
	int gnode = n / kGroup + gi, gfirst = gi * kGroup, gcount = kGroup, gsuper = gi >> kSuperShift;
	if constexpr(kRadix)
	{
		const int4 gr = tree.grp[gi];
		gnode = gr.x;
		gfirst = gr.y;
		gcount = gr.z;
		gsuper = gr.w;
	}
	const double* glo = bmin + 3 * static_cast<size_t>(gnode);
	const double* ghi = bmax + 3 * static_cast<size_t>(gnode);
	const double gx0 = glo[0], gy0 = glo[1], gz0 = glo[2];
	const double gx1 = ghi[0], gy1 = ghi[1], gz1 = ghi[2];
	const double ccx = 0.5 * (gx0 + gx1), ccy = 0.5 * (gy0 + gy1), ccz = 0.5 * (gz0 + gz1);
	// this lane's bodies: leaf lane of the group, and leaf lane + 64 in the Morton
	// tree's walk groups of up to 128 bodies (kT = 2); lanes beyond a smaller
	// group's size repeat its first body and write nothing
	constexpr int kT = kRadix ? 2 : 1;
	bool body_lane[kT];
	int tn[kT];
	float tx[kT], ty[kT], tz[kT];                   // scaled offsets from the group centre, for the sweeps
	float ax[kT], ay[kT], az[kT], cx[kT], cy[kT], cz[kT];
#pragma unroll
	for(int t = 0; t < kT; ++t)
	{
		const int j = lane + kGroup * t;
		body_lane[t] = j < gcount;
		tn[t] = n + gfirst + (body_lane[t] ? j : 0);
		const double4 me = wr[tn[t]].c;
		tx[t] = static_cast<float>((me.x - ccx) * kSweepLen);
		ty[t] = static_cast<float>((me.y - ccy) * kSweepLen);
		tz[t] = static_cast<float>((me.z - ccz) * kSweepLen);
		ax[t] = ay[t] = az[t] = cx[t] = cy[t] = cz[t] = 0.0f;
	}
	const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
	unsigned vis = 0, taken = 0, spill = 0, nfar = 0, nnear = 0;
	constexpr int kAcc = kLocal ? 34 : 9;
	float acc[kAcc];
	for(int k = 0; k < kAcc; ++k) { acc[k] = 0.0f; }
	const float near_d = static_cast<float>(static_cast<double>(near_k) * kSweepLen *
	                                        half_diagonal(gx0, gy0, gz0, gx1, gy1, gz1));   // scaled

	int si = 0, lcnt = 0, lpos = 0;
	bool use_list = false;
	if constexpr(kTwo)
	{
		si = gsuper;
		use_list = si >= 0 && two.count[si] <= two.cap;
		lcnt = use_list ? two.count[si] : 0;
	}
	const int* list = kTwo ? two.lists + static_cast<size_t>(si) * two.cap : nullptr;
	int lentry = kTwo && lane < lcnt ? list[lane] : kRoot;   // list entry of the next list step
	int sp = use_list ? 0 : 1;
	int nbuf = 0;
	int nq = 0;
	int fhead = 0, ftail = 0;     // far-cell ring: entries [fhead, ftail) pending
	if(lane == 0) { stack[0] = walk_start<kRadix>(); }
	__syncthreads();
	while(sp > 0 || lpos < lcnt)
	{
		bool valid;
		int node;
		double4 rec;
		double m;
		int2 kids;
		float nq6[kQuad ? 6 : 1];     // second moments, read with the record
		// issue this step's node loads, then sweep the buffers the previous steps
		// filled while they are in flight; listed nodes are taken when the stack
		// below them is done
		if(sp == 0)
		{
			list_fetch<kRadix, kQuad>(list, lpos, lcnt, lane, wr, lentry, node, valid, rec, m, kids, tree.child, n,
			                          nq6);
			lpos += kGroup;
		}
		else
		{
			walk_fetch<kRadix, kQuad>(stack, sp, lane, wr, node, valid, rec, m, kids, tree.child, n, nq6);
		}
		if(nbuf > kWalkBuf - kGroup)
		{
			sweep32_n<kT>(buf, nbuf, tx, ty, tz, ax, ay, az, cx, cy, cz);
			nbuf = 0;
		}
		if constexpr(kQuad)
		{
			if(nq > kQuadBuf - kGroup)
			{
				sweep_mq_n<kT>(qbuf, nq, tx, ty, tz, ax, ay, az, cx, cy, cz);
				nq = 0;
			}
			if(ftail - fhead >= kGroup)
			{
				far_batch<kLocal>(farn, wr, fhead, kGroup, lane, ccx, ccy, ccz, acc);
				fhead += kGroup;
			}
		}
		__syncthreads();
		bool accept = false, open = false, cell = false;
		float4 ent = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		if(valid)
		{
			ent = sweep_entry(rec, m, ccx, ccy, ccz);
			if(node >= n)
			{
				accept = true;
			}
			else
			{
				// distance from the group box to the node's mass centre
				const double ex = fmax(fmax(gx0 - rec.x, rec.x - gx1), 0.0);
				const double ey = fmax(fmax(gy0 - rec.y, rec.y - gy1), 0.0);
				const double ez = fmax(fmax(gz0 - rec.z, rec.z - gz1), 0.0);
				accept = ex * ex + ey * ey + ez * ez > rec.w;
				open = !accept;
				cell = kQuad && accept;     // taken internal cell (stack spills stay monopoles)
			}
		}
		const uint64_t bopen = __ballot(open);
		const int nopen = __popcll(bopen);
		if(sp + nopen > kWalkStack)
		{
			// no room for the children: take these nodes as monopoles
			spill += open ? 1 : 0;
			accept = accept || open;
			open = false;
		}
		const uint64_t bacc = __ballot(accept);
		const uint64_t bopen2 = __ballot(open);
		if constexpr(kQuad)
		{
			// near taken internal cells: monopole + quadrupole sweep; the rest:
			// monopole sweep, far cells adding their expansion
			const bool far = cell && !(ent.x * ent.x + ent.y * ent.y + ent.z * ent.z < near_d * near_d);
			const bool nearc = cell && !far;
			const uint64_t bnear = __ballot(nearc);
			const uint64_t bfar = __ballot(far);
			const uint64_t bmono = kLocal ? bacc & ~bnear & ~bfar : bacc & ~bnear;
			if(nearc) { put_quad(qbuf, nq + __popcll(bnear & lt), ent, nq6); }
			else if(accept && !(kLocal && far)) { buf[nbuf + __popcll(bmono & lt)] = ent; }
			if(far)
			{
				farn[(ftail + __popcll(bfar & lt)) & (kFarRing - 1)] = node;
			}
			ftail += __popcll(bfar);
			nq += __popcll(bnear);
			nbuf += __popcll(bmono);
			nfar += far ? 1 : 0;
			nnear += nearc ? 1 : 0;
		}
		else
		{
			if(accept) { buf[nbuf + __popcll(bacc & lt)] = ent; }
			nbuf += __popcll(bacc);
		}
		if(open) { stack[sp + __popcll(bopen2 & lt)] = walk_entry<kRadix>(node, kids, n); }
		sp += __popcll(bopen2);
		vis += valid ? 1 : 0;
		taken += accept ? 1 : 0;
		__syncthreads();
	}
	if(nbuf > 0)
	{
		sweep32_n<kT>(buf, nbuf, tx, ty, tz, ax, ay, az, cx, cy, cz);
	}
	float kx[kT], ky[kT], kz[kT];
	for(int t = 0; t < kT; ++t) { kx[t] = ky[t] = kz[t] = 0.0f; }
	if constexpr(kQuad)
	{
		if(nq > 0) { sweep_mq_n<kT>(qbuf, nq, tx, ty, tz, ax, ay, az, cx, cy, cz); }
		for(; fhead < ftail; fhead += kGroup)
		{
			far_batch<kLocal>(farn, wr, fhead, ftail - fhead < kGroup ? ftail - fhead : kGroup, lane, ccx, ccy, ccz,
			                  acc);
		}
		for(int sh = 1; sh < 64; sh <<= 1)
		{
			for(int k = 0; k < kAcc; ++k) { acc[k] += __shfl_xor(acc[k], sh, 64); }
		}
#pragma unroll
		for(int t = 0; t < kT; ++t)
		{
			const double4 me = wr[tn[t]].c;
			const float ux = static_cast<float>(me.x - ccx);   // unscaled offset for the expansion
			const float uy = static_cast<float>(me.y - ccy);
			const float uz = static_cast<float>(me.z - ccz);
			kx[t] = acc[0] + acc[3] * ux + acc[6] * uy + acc[7] * uz;
			ky[t] = acc[1] + acc[6] * ux + acc[4] * uy + acc[8] * uz;
			kz[t] = acc[2] + acc[7] * ux + acc[8] * uy + acc[5] * uz;
			if constexpr(kLocal)
			{
				float sx, sy, sz;
				local_terms(acc + 9, ux, uy, uz, sx, sy, sz);
				kx[t] += sx;
				ky[t] += sy;
				kz[t] += sz;
			}
		}
		if constexpr(kTwo)
		{
			if(use_list)
			{
				// the super-group's expansion about its own box centre
				const size_t sg = kRadix ? static_cast<size_t>(tree.sup[si].x)
				                         : (static_cast<size_t>(n) >> (6 + kSuperShift)) + si;
				const double* slo = bmin + 3 * sg;
				const double* shi = bmax + 3 * sg;
				const double scx = 0.5 * (slo[0] + shi[0]);
				const double scy = 0.5 * (slo[1] + shi[1]);
				const double scz = 0.5 * (slo[2] + shi[2]);
				const float* c = two.coef + 34 * static_cast<size_t>(si);
				float e[34];
				for(int k = 0; k < 34; ++k) { e[k] = c[k]; }
#pragma unroll
				for(int t = 0; t < kT; ++t)
				{
					const double4 me = wr[tn[t]].c;
					const float vx = static_cast<float>(me.x - scx), vy = static_cast<float>(me.y - scy);
					const float vz = static_cast<float>(me.z - scz);
					float sx, sy, sz;
					local_terms(e + 9, vx, vy, vz, sx, sy, sz);
					kx[t] += e[0] + e[3] * vx + e[6] * vy + e[7] * vz + sx;
					ky[t] += e[1] + e[6] * vx + e[4] * vy + e[8] * vz + sy;
					kz[t] += e[2] + e[7] * vx + e[8] * vy + e[5] * vz + sz;
				}
			}
		}
	}
#pragma unroll
	for(int t = 0; t < kT; ++t)
	{
		if(body_lane[t])
		{
			const int b = body_n[tn[t]];
			f[b] = y[3 * n + b];
			f[n + b] = y[4 * n + b];
			f[2 * n + b] = y[5 * n + b];
			f[3 * n + b] = static_cast<double>(ax[t]) - static_cast<double>(cx[t]) + static_cast<double>(kx[t]);
			f[4 * n + b] = static_cast<double>(ay[t]) - static_cast<double>(cy[t]) + static_cast<double>(ky[t]);
			f[5 * n + b] = static_cast<double>(az[t]) - static_cast<double>(cz[t]) + static_cast<double>(kz[t]);
		}
	}
	// counters: [0] pair interactions (entries x the group's bodies), [1] node
	// visits, [2] spills
	for(int off = 32; off > 0; off >>= 1)
	{
		vis += __shfl_down(vis, off, 64);
		taken += __shfl_down(taken, off, 64);
		spill += __shfl_down(spill, off, 64);
		nfar += __shfl_down(nfar, off, 64);
		nnear += __shfl_down(nnear, off, 64);
	}
	if(lane == 0)
	{
		atomicAdd(&counters[0], static_cast<unsigned long long>(taken) * gcount);
		atomicAdd(&counters[1], static_cast<unsigned long long>(vis));
		if(spill) { atomicAdd(&counters[2], static_cast<unsigned long long>(spill)); }
		if(nfar) { atomicAdd(&counters[3], static_cast<unsigned long long>(nfar)); }
		if(nnear) { atomicAdd(&counters[4], static_cast<unsigned long long>(nnear)); }
	}
}

// The group walk kernel, one work-group per group: the heap's groups in
// XCD-contiguous order, the Morton tree's in runs of 128 per XCD (at 4M Plummer
// bodies 2.66 ms against 2.80 in launch order, 2.72 in runs of 32: neighbours share
// their super-group's list and nodes in one L2; persistent work-groups that take
// groups from counters, per XCD or in one queue, ran 9-19% slower; two waves that
// share a group's list gain 17% at 16384-50000 bodies and lose from 100003 on).
constexpr int kXcdRun = 128;

__device__ inline int xcd_run_group(int block, int nblocks)
{
	const int whole = nblocks / (kXcds * kXcdRun) * (kXcds * kXcdRun);
	if(block >= whole) { return block; }
	const int i = block / kXcds;
	return (i / kXcdRun * kXcds + block % kXcds) * kXcdRun + i % kXcdRun;
}

template <bool kQuad, bool kLocal = false, bool kTwo = false, bool kRadix = false>
__global__ void __launch_bounds__(kGroup)
k_bh_group32(const nbh_walk_rec* __restrict__ wr, const double* __restrict__ bmin, const double* __restrict__ bmax,
             const int32_t* __restrict__ body_n, const double* __restrict__ y, double* __restrict__ f, int n,
             float near_k, unsigned long long* __restrict__ counters, TwoLevel two = TwoLevel(),
             WalkTree tree = WalkTree())
{
	__shared__ int stack[kWalkStack];
	__shared__ float4 buf[kWalkBuf];
	__shared__ quad_lds<kQuad ? kQuadBuf : 1> qbuf;
	__shared__ int farn[kQuad ? kFarRing : 1];
	const int gi = kRadix ? xcd_run_group(blockIdx.x, gridDim.x) : xcd_group(blockIdx.x, gridDim.x);
	group_walk_one<kQuad, kLocal, kTwo, kRadix>(gi, stack, buf, qbuf, farn, wr, bmin, bmax, body_n, y, f, n, near_k,
	                                             counters, two, tree);
}

// Super-group walk of the two-level local walk (TwoLevel): the group walk's
// loop with the super box, far cells into the super expansion, every other
// accepted node into the list.
template <bool kRadix = false>
__global__ void __launch_bounds__(kGroup)
k_bh_super(const nbh_walk_rec* __restrict__ wr, const double* __restrict__ bmin, const double* __restrict__ bmax,
           int n, float near_k, double inv_ratio, TwoLevel two, unsigned long long* __restrict__ counters,
           int stack_limit, WalkTree tree = WalkTree())
{
	__shared__ int stack[kWalkStack];
	__shared__ int farn[kFarRing];
	const int lane = threadIdx.x;
	const int si = kRadix ? static_cast<int>(blockIdx.x) : xcd_group(blockIdx.x, gridDim.x);
	// node of the super-group
	const size_t sg = kRadix ? static_cast<size_t>(tree.sup[si].x) : (static_cast<size_t>(n) >> (6 + kSuperShift)) + si;
	const double* glo = bmin + 3 * sg;
	const double* ghi = bmax + 3 * sg;
	const double gx0 = glo[0], gy0 = glo[1], gz0 = glo[2];
	const double gx1 = ghi[0], gy1 = ghi[1], gz1 = ghi[2];
	const double ccx = 0.5 * (gx0 + gx1), ccy = 0.5 * (gy0 + gy1), ccz = 0.5 * (gz0 + gz1);
	const double super_hd64 = half_diagonal(gx0, gy0, gz0, gx1, gy1, gz1);
	const float near_d = static_cast<float>(static_cast<double>(near_k) * super_hd64);
	const float super_hd = static_cast<float>(super_hd64);
	const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
	int* list = two.lists + static_cast<size_t>(si) * two.cap;
	float acc[34];
	for(int k = 0; k < 34; ++k) { acc[k] = 0.0f; }
	unsigned long long vis = 0, nfar = 0;
	int lcount = 0;
	int nfar_listed = 0;
	bool overflow = false;
	int sp = 1;
	int fhead = 0, ftail = 0;
	if(lane == 0) { stack[0] = walk_start<kRadix>(); }
	__syncthreads();
	while(sp > 0)
	{
		bool valid;
		int node;
		double4 rec;
		double m;
		int2 kids;
		walk_fetch<kRadix>(stack, sp, lane, wr, node, valid, rec, m, kids, tree.child, n);
		if(ftail - fhead >= kGroup)
		{
			far_batch<true>(farn, wr, fhead, kGroup, lane, ccx, ccy, ccz, acc);
			fhead += kGroup;
		}
		__syncthreads();
		bool accept = false, open = false, far = false;
		float ux = 0.0f, uy = 0.0f, uz = 0.0f;
		if(valid)
		{
			ux = static_cast<float>(rec.x - ccx);
			uy = static_cast<float>(rec.y - ccy);
			uz = static_cast<float>(rec.z - ccz);
			if(node >= n)
			{
				accept = true;
			}
			else
			{
				const double ex = fmax(fmax(gx0 - rec.x, rec.x - gx1), 0.0);
				const double ey = fmax(fmax(gy0 - rec.y, rec.y - gy1), 0.0);
				const double ez = fmax(fmax(gz0 - rec.z, rec.z - gz1), 0.0);
				accept = ex * ex + ey * ey + ez * ez > rec.w;
				const float du = sqrtf(ux * ux + uy * uy + uz * uz);
				far = accept && !(du < near_d);
				// a rejected node whose bodies all lie within near_d of the centre
				// (ball of the cell radius sqrt(crit_r2) / ratio about its mass
				// centre) is left to the groups; others are opened here
				// (in the Morton tree also one wider than half the super box: it is
				// opened here once rather than by every walk group, which lowers the
				// error at the same cost)
				const float rad = static_cast<float>(sqrt(rec.w) * inv_ratio);
				open = !accept && (!(du + rad < near_d) || (kRadix && rad > 0.5f * super_hd));
			}
		}
		const bool tolist = valid && !far && !open;
		if(sp + __popcll(__ballot(open)) > stack_limit)
		{
			overflow = true;           // the groups of this super-group will walk for themselves
			open = false;
		}
		const uint64_t bopen = __ballot(open);
		const uint64_t bfar = __ballot(far);
		const uint64_t blist = __ballot(tolist);
		if(far)
		{
			farn[(ftail + __popcll(bfar & lt)) & (kFarRing - 1)] = node;
			if(two.far_list != nullptr)
			{
				const int fslot = nfar_listed + __popcll(bfar & lt);
				if(fslot < two.far_cap) { two.far_list[static_cast<size_t>(si) * two.far_cap + fslot] = node; }
			}
		}
		nfar_listed += __popcll(bfar);
		if(tolist)
		{
			const int slot = lcount + __popcll(blist & lt);
			if(slot < two.cap) { list[slot] = node; }
		}
		if(open) { stack[sp + __popcll(bopen & lt)] = walk_entry<kRadix>(node, kids, n); }
		ftail += __popcll(bfar);
		lcount += __popcll(blist);
		sp += __popcll(bopen);
		vis += valid ? 1 : 0;
		nfar += far ? 1 : 0;
		__syncthreads();
	}
	for(; fhead < ftail; fhead += kGroup)
	{
		far_batch<true>(farn, wr, fhead, ftail - fhead < kGroup ? ftail - fhead : kGroup, lane, ccx, ccy, ccz, acc);
	}
	for(int sh = 1; sh < 64; sh <<= 1)
	{
		for(int k = 0; k < 34; ++k) { acc[k] += __shfl_xor(acc[k], sh, 64); }
	}
	overflow = __ballot(overflow) != 0;
	if(lane == 0)
	{
		float* c = two.coef + 34 * static_cast<size_t>(si);
		for(int k = 0; k < 34; ++k) { c[k] = acc[k]; }
		two.count[si] = overflow || lcount > two.cap ? two.cap + 1 : lcount;
		if(two.far_count != nullptr) { two.far_count[si] = nfar_listed; }
	}
	for(int off = 32; off > 0; off >>= 1)
	{
		vis += __shfl_down(vis, off, 64);
		nfar += __shfl_down(nfar, off, 64);
	}
	if(lane == 0)
	{
		atomicAdd(&counters[1], vis);
		if(nfar) { atomicAdd(&counters[3], nfar); }
		if(overflow || lcount > two.cap) { atomicAdd(&counters[2], 1ull); }
	}
}

// ---------------------------------------------------------------------------
// learned correction: samples, and the group walk with the network
// ---------------------------------------------------------------------------
// Internal cells the group walk takes as monopoles are split by the distance
// dc from the group's box centre to their mass centre, in units of the box's
// half-diagonal h:
//   near (dc < near_k h): the cell's second moments are applied to every body
//        of the group (quadrupole term), since its field varies too much over
//        the group for one expansion about the centre;
//   far  (otherwise), with bounding radius r > rho_min dc: the network predicts
//        the cell's residual field at the centre and its Jacobian.
enum { kCellNone = 0, kCellNear = 1, kCellFar = 2 };

__device__ inline double cell_radius(const double* lo, const double* hi, double cx, double cy, double cz)
{
	const double ex = hi[0] - lo[0], ey = hi[1] - lo[1], ez = hi[2] - lo[2];
	const double gx = 0.5 * (hi[0] + lo[0]) - cx, gy = 0.5 * (hi[1] + lo[1]) - cy, gz = 0.5 * (hi[2] + lo[2]) - cz;
	return 0.5 * sqrt(ex * ex + ey * ey + ez * ez) + sqrt(gx * gx + gy * gy + gz * gz);
}

__device__ inline int classify_cell(const double* lo, const double* hi, const double4& rec, double ccx, double ccy,
                                    double ccz, double half_diag, float near_k, float rho_min, double* dc_out)
{
	const double dx = rec.x - ccx, dy = rec.y - ccy, dz = rec.z - ccz;
	const double dc = sqrt(dx * dx + dy * dy + dz * dz);
	*dc_out = dc;
	if(dc < static_cast<double>(near_k) * half_diag) { return kCellNear; }
	const double r = cell_radius(lo, hi, rec.x, rec.y, rec.z);
	return r > static_cast<double>(rho_min) * dc ? kCellFar : kCellNone;
}

// Group walk without forces: emit (group ordinal, node) for every far cell.
__global__ void __launch_bounds__(kGroup)
k_band_collect(const double4* __restrict__ xyzr, const double* __restrict__ bmin, const double* __restrict__ bmax,
               int n, const uint32_t* __restrict__ groups, float rho_min, float near_k, uint32_t* __restrict__ pairs,
               unsigned long long capacity, unsigned long long* __restrict__ counter)
{
	__shared__ int stack[kWalkStack];
	const int lane = threadIdx.x;
	const uint32_t go = groups[blockIdx.x];
	const int g = n / kGroup + static_cast<int>(go);
	const double gx0 = bmin[3 * g], gy0 = bmin[3 * g + 1], gz0 = bmin[3 * g + 2];
	const double gx1 = bmax[3 * g], gy1 = bmax[3 * g + 1], gz1 = bmax[3 * g + 2];
	const double ccx = 0.5 * (gx0 + gx1), ccy = 0.5 * (gy0 + gy1), ccz = 0.5 * (gz0 + gz1);
	const double hd = half_diagonal(gx0, gy0, gz0, gx1, gy1, gz1);
	const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
	int sp = 1;
	if(lane == 0) { stack[0] = kRoot; }
	__syncthreads();
	while(sp > 0)
	{
		bool valid;
		const int node = walk_pop(stack, sp, lane, valid);
		__syncthreads();
		bool open = false, band = false;
		if(valid && node < n)
		{
			const double4 rec = xyzr[node];
			const double ex = fmax(fmax(gx0 - rec.x, rec.x - gx1), 0.0);
			const double ey = fmax(fmax(gy0 - rec.y, rec.y - gy1), 0.0);
			const double ez = fmax(fmax(gz0 - rec.z, rec.z - gz1), 0.0);
			open = !(ex * ex + ey * ey + ez * ez > rec.w);
			if(!open)
			{
				double dc;
				band = classify_cell(bmin + 3 * node, bmax + 3 * node, rec, ccx, ccy, ccz, hd, near_k, rho_min, &dc) ==
				       kCellFar;
			}
		}
		const int nopen = __popcll(__ballot(open));
		if(sp + nopen > kWalkStack) { open = false; }
		const uint64_t bopen = __ballot(open);
		if(open) { stack[sp + __popcll(bopen & lt)] = 2 * node; }
		sp += __popcll(bopen);
		const uint64_t bband = __ballot(band);
		const int nband = __popcll(bband);
		if(nband > 0)
		{
			unsigned long long base = 0;
			if(lane == 0) { base = atomicAdd(counter, static_cast<unsigned long long>(nband)); }
			base = __shfl(base, 0, 64);
			const unsigned long long slot = base + __popcll(bband & lt);
			if(band && slot < capacity)
			{
				pairs[2 * slot] = go;
				pairs[2 * slot + 1] = static_cast<uint32_t>(node);
			}
		}
		__syncthreads();
	}
}

// Quadrupole term of a cell's field at p and its Jacobian, FP64: Q the second
// central moments (xx yy zz xy xz yz) about the mass centre cm; with
// r = cm - p, d = |r|, Q' = 3 Q - tr(Q) I and s = r.Q'.r,
//   g = (2.5 s / d^2 r - Q' r) / d^5,
//   J = dg/dp = -(5 (r (Q'r)' + (Q'r) r') + 2.5 s I) / d^7 + 17.5 s r r' / d^9 + Q' / d^5
// (the terms quad_expansion evaluates in FP32); out[9] = g (3), J (6).
__device__ inline void quad_field64(double rx, double ry, double rz, const double* Q, double* out)
{
	const double tr = Q[0] + Q[1] + Q[2];
	const double qxx = 3.0 * Q[0] - tr, qyy = 3.0 * Q[1] - tr, qzz = 3.0 * Q[2] - tr;
	const double qxy = 3.0 * Q[3], qxz = 3.0 * Q[4], qyz = 3.0 * Q[5];
	const double Qx = qxx * rx + qxy * ry + qxz * rz;
	const double Qy = qxy * rx + qyy * ry + qyz * rz;
	const double Qz = qxz * rx + qyz * ry + qzz * rz;
	const double sq = rx * Qx + ry * Qy + rz * Qz;
	const double d2 = rx * rx + ry * ry + rz * rz;
	const double d = sqrt(d2);
	const double i5 = 1.0 / (d2 * d2 * d);
	const double i7 = i5 / d2;
	const double c = 2.5 * sq * i7;
	out[0] = c * rx - Qx * i5;
	out[1] = c * ry - Qy * i5;
	out[2] = c * rz - Qz * i5;
	const double a = 5.0 * i7;
	const double e = 17.5 * sq * i7 / d2;
	out[3] = -(a * (2.0 * rx * Qx) + c - e * rx * rx - qxx * i5);
	out[4] = -(a * (2.0 * ry * Qy) + c - e * ry * ry - qyy * i5);
	out[5] = -(a * (2.0 * rz * Qz) + c - e * rz * rz - qzz * i5);
	out[6] = -(a * (rx * Qy + ry * Qx) - e * rx * ry - qxy * i5);
	out[7] = -(a * (rx * Qz + rz * Qx) - e * rx * rz - qxz * i5);
	out[8] = -(a * (ry * Qz + rz * Qy) - e * ry * rz - qyz * i5);
}

// One wave per sample (centre node centre_base + pairs[2s], cell pairs[2s+1]):
// the exact FP64 field of the cell's bodies at the centre node's box centre p
// and its Jacobian, minus those of the monopole (order 1) or of the monopole
// and the quadrupole term (order 2), written as features x[16], basis b[16] and
// target t[9] = [R / w, kJac J d / w] (J as xx yy zz xy xz yz), where w is the
// scale of cell_features (M rho^2 / d^2) times rho^(order - 1).
__global__ void __launch_bounds__(64)
k_band_residual(const double4* __restrict__ xyzr, const double* __restrict__ nmass, const double* __restrict__ bmin,
                const double* __restrict__ bmax, const double* __restrict__ quad, int n, int levels, int centre_base,
                int order, const uint32_t* __restrict__ pairs, size_t count, float* __restrict__ x,
                float* __restrict__ bs, float* __restrict__ t)
{
	const int lane = threadIdx.x;
	for(size_t s = blockIdx.x; s < count; s += gridDim.x)
	{
		const int g = centre_base + static_cast<int>(pairs[2 * s]);
		const int c = static_cast<int>(pairs[2 * s + 1]);
		const double px = 0.5 * (bmin[3 * g] + bmax[3 * g]);
		const double py = 0.5 * (bmin[3 * g + 1] + bmax[3 * g + 1]);
		const double pz = 0.5 * (bmin[3 * g + 2] + bmax[3 * g + 2]);
		const int depth = 31 - __builtin_clz(static_cast<unsigned>(c));
		const int span = levels - depth;
		const int leaf0 = c << span, leaf1 = (c + 1) << span;
		double a[9];
		for(int k = 0; k < 9; ++k) { a[k] = 0.0; }
		for(int leaf = leaf0 + lane; leaf < leaf1; leaf += 64)
		{
			const double4 b = xyzr[leaf];
			const double dx = b.x - px, dy = b.y - py, dz = b.z - pz;
			double r2 = dx * dx + dy * dy + dz * dz;
			if(r2 < 1e-8) { r2 = 1e-8; }
			const double w = nmass[leaf] / (r2 * sqrt(r2));
			const double w5 = 3.0 * w / r2;
			a[0] += dx * w;
			a[1] += dy * w;
			a[2] += dz * w;
			a[3] += w5 * dx * dx - w;
			a[4] += w5 * dy * dy - w;
			a[5] += w5 * dz * dz - w;
			a[6] += w5 * dx * dy;
			a[7] += w5 * dx * dz;
			a[8] += w5 * dy * dz;
		}
		for(int off = 32; off > 0; off >>= 1)
		{
			for(int k = 0; k < 9; ++k) { a[k] += __shfl_down(a[k], off, 64); }
		}
		if(lane == 0)
		{
			const double4 rec = xyzr[c];
			const double M = nmass[c];
			const double dx = rec.x - px, dy = rec.y - py, dz = rec.z - pz;
			const double d2 = dx * dx + dy * dy + dz * dz;
			const double d = sqrt(d2);
			const double w = M / (d2 * d);
			const double w5 = 3.0 * w / d2;
			a[0] -= dx * w;
			a[1] -= dy * w;
			a[2] -= dz * w;
			a[3] -= w5 * dx * dx - w;
			a[4] -= w5 * dy * dy - w;
			a[5] -= w5 * dz * dz - w;
			a[6] -= w5 * dx * dy;
			a[7] -= w5 * dx * dz;
			a[8] -= w5 * dy * dz;
			if(order >= 2)
			{
				double q[9];
				quad_field64(dx, dy, dz, quad + 6 * c, q);
				for(int k = 0; k < 9; ++k) { a[k] -= q[k]; }
			}
			float f[nbh_net::kIn];
			float bv[nbh_net::kBasis];
			double scale = nbh_net::cell_features(px, py, pz, rec.x, rec.y, rec.z, M, bmin + 3 * c, bmax + 3 * c,
			                                      quad + 6 * c, f, bv);
			if(order >= 2) { scale *= static_cast<double>(f[0]); }    // f[0] = rho
			for(int k = 0; k < nbh_net::kIn; ++k) { x[s * nbh_net::kIn + k] = f[k]; }
			for(int k = 0; k < nbh_net::kBasis; ++k) { bs[s * nbh_net::kBasis + k] = bv[k]; }
			for(int k = 0; k < 3; ++k) { t[s * nbh_net::kOut + k] = static_cast<float>(a[k] / scale); }
			for(int k = 3; k < 9; ++k) { t[s * nbh_net::kOut + k] = static_cast<float>(a[k] * nbh_net::kJac * d / scale); }
		}
	}
}

// Learned correction of the two-level walk's shared far field: one wave per
// super-group evaluates the network on the super-group's far cells (listed by
// k_bh_super), 16 at a time on the matrix cores, and adds the predicted
// remainder after the monopole and quadrupole terms -- field R and Jacobian J
// at the super box centre, R / w = c0 uh + c1 w + c2 o and kJac J d / w =
// (basis of nbh_mlp_dev.h), w = M rho^3 / d^2 -- to the super-group's
// expansion coefficients (field and Jacobian slots), which every body of the
// super-group applies.  Features are formed in FP64 and rounded once.
__global__ void __launch_bounds__(64)
k_super_net(const double4* __restrict__ xyzr, const double* __restrict__ nmass, const double* __restrict__ bmin,
            const double* __restrict__ bmax, const double* __restrict__ quad, int n, TwoLevel two,
            const uint2* __restrict__ frags, const float* __restrict__ mlp_p)
{
	__shared__ __align__(16) uint16_t tf[16 * nbh_net::kIn];
	__shared__ float tb[16 * nbh_net::kBasis];
	__shared__ float tw[2 * 16];
	__shared__ __align__(16) uint16_t mlds[2 * 16 * nbh_net::kHid];
	const int lane = threadIdx.x;
	const int col = lane & 15;
	const int si = blockIdx.x;
	const int sg = (n >> (6 + kSuperShift)) + si;
	const double px = 0.5 * (bmin[3 * sg] + bmax[3 * sg]);
	const double py = 0.5 * (bmin[3 * sg + 1] + bmax[3 * sg + 1]);
	const double pz = 0.5 * (bmin[3 * sg + 2] + bmax[3 * sg + 2]);
	const int rows = min(two.far_count[si], two.far_cap);
	const int* list = two.far_list + static_cast<size_t>(si) * two.far_cap;
	float acc[nbh_net::kOut];
	for(int k = 0; k < nbh_net::kOut; ++k) { acc[k] = 0.0f; }
	for(int base = 0; base < rows; base += 16)
	{
		if(lane < 16)
		{
			const int r = base + lane;
			float f[nbh_net::kIn];
			float bv[nbh_net::kBasis];
			float w0 = 0.0f, w1 = 0.0f;
			if(r < rows)
			{
				const int c = list[r];
				const double4 rec = xyzr[c];
				const double scale = nbh_net::cell_features(px, py, pz, rec.x, rec.y, rec.z, nmass[c], bmin + 3 * c,
				                                            bmax + 3 * c, quad + 6 * c, f, bv) *
				                     static_cast<double>(f[0]);
				const double dx = rec.x - px, dy = rec.y - py, dz = rec.z - pz;
				const double d = sqrt(dx * dx + dy * dy + dz * dz);
				w0 = static_cast<float>(scale);
				w1 = static_cast<float>(scale / (nbh_net::kJac * d));
			}
			else
			{
				for(int k = 0; k < nbh_net::kIn; ++k) { f[k] = 0.0f; }
				for(int k = 0; k < nbh_net::kBasis; ++k) { bv[k] = 0.0f; }
			}
			for(int k = 0; k < nbh_net::kIn; ++k) { tf[lane * nbh_net::kIn + k] = nbh_net::to_bf16(f[k]); }
			for(int k = 0; k < nbh_net::kBasis; ++k) { tb[lane * nbh_net::kBasis + k] = bv[k]; }
			tw[2 * lane] = w0;
			tw[2 * lane + 1] = w1;
		}
		__syncthreads();
		const nbh_net::bf16x4 xa = nbh_net::lds_afrag(tf, nbh_net::kIn, 0, lane);
		const nbh_net::f32x4 o = nbh_net::forward_tile(xa, frags, mlp_p, mlds, lane, nullptr, nullptr);
		for(int e = 0; e < 4; ++e)
		{
			const int row = 4 * (lane >> 4) + e;
			float v[nbh_net::kOut];
			nbh_net::basis_col(tb + row * nbh_net::kBasis, col, v);
			const float c0 = o[e] * tw[2 * row], c1 = o[e] * tw[2 * row + 1];
			for(int k = 0; k < 3; ++k) { acc[k] = fmaf(c0, v[k], acc[k]); }
			for(int k = 3; k < nbh_net::kOut; ++k) { acc[k] = fmaf(c1, v[k], acc[k]); }
		}
		__syncthreads();
	}
	for(int sh = 1; sh < 64; sh <<= 1)
	{
		for(int k = 0; k < nbh_net::kOut; ++k) { acc[k] += __shfl_xor(acc[k], sh, 64); }
	}
	if(lane == 0)
	{
		float* c = two.coef + 34 * static_cast<size_t>(si);
		for(int k = 0; k < nbh_net::kOut; ++k) { c[k] += acc[k]; }
	}
}

// Training pairs (super-group ordinal, far cell) of the super-groups sel[g]:
// block g copies the far list of super-group sel[g] to pairs[off[g] ...].
__global__ void __launch_bounds__(64)
k_super_pairs(TwoLevel two, const uint32_t* __restrict__ sel, const unsigned long long* __restrict__ off,
              uint32_t* __restrict__ pairs, unsigned long long capacity)
{
	const uint32_t si = sel[blockIdx.x];
	const int rows = min(two.far_count[si], two.far_cap);
	const int* list = two.far_list + static_cast<size_t>(si) * two.far_cap;
	for(int r = threadIdx.x; r < rows; r += blockDim.x)
	{
		const unsigned long long slot = off[blockIdx.x] + static_cast<unsigned long long>(r);
		if(slot < capacity)
		{
			pairs[2 * slot] = si;
			pairs[2 * slot + 1] = static_cast<uint32_t>(list[r]);
		}
	}
}

constexpr int kBand = 80;        // far-cell rows waiting for the network (< 16 + 64)
// k_bh_group32 plus the correction.  Near cells enter the monopole +
// quadrupole sweep, every other taken node the monopole sweep; far cells are
// fed to the network in tiles of 16, and the predicted residual field of each,
// expanded to first order about the group centre, is summed over the group's
// far cells into C (3) and J (6), the correction of a body at offset delta from
// the centre being C + J delta.
__global__ void __launch_bounds__(kGroup)
k_bh_group32_mlp(const nbh_walk_rec* __restrict__ wr, const double* __restrict__ bmin,
                 const double* __restrict__ bmax, const int32_t* __restrict__ body_n,
                 const double* __restrict__ y, double* __restrict__ f, int n, const uint2* __restrict__ frags,
                 const float* __restrict__ mlp_p, float rho_min, float near_k,
                 unsigned long long* __restrict__ counters)
{
	__shared__ int stack[kWalkStack];
	__shared__ float4 buf[kWalkBuf];
	__shared__ quad_lds<kQuadBuf> qbuf;
	__shared__ __align__(16) uint16_t bandf[kBand * nbh_net::kIn];
	__shared__ float bandw[2 * kBand];      // per far row: scale, scale / (kJac d)
	__shared__ float bandb[kBand * nbh_net::kBasis];
	__shared__ __align__(16) uint16_t mlds[2 * 16 * nbh_net::kHid];
	const int lane = threadIdx.x;
	const int col = lane & 15;
	const int gi = xcd_group(blockIdx.x, gridDim.x);
	const int g = n / kGroup + gi;
	const double gx0 = bmin[3 * g], gy0 = bmin[3 * g + 1], gz0 = bmin[3 * g + 2];
	const double gx1 = bmax[3 * g], gy1 = bmax[3 * g + 1], gz1 = bmax[3 * g + 2];
	const double ccx = 0.5 * (gx0 + gx1), ccy = 0.5 * (gy0 + gy1), ccz = 0.5 * (gz0 + gz1);
	const double hd = half_diagonal(gx0, gy0, gz0, gx1, gy1, gz1);
	const int tn = n + gi * kGroup + lane;
	const double4 me = wr[tn].c;
	const float tx = static_cast<float>((me.x - ccx) * kSweepLen);   // scaled, for the sweeps
	const float ty = static_cast<float>((me.y - ccy) * kSweepLen);
	const float tz = static_cast<float>((me.z - ccz) * kSweepLen);
	float ax = 0.0f, ay = 0.0f, az = 0.0f, cx = 0.0f, cy = 0.0f, cz = 0.0f;
	float acc[nbh_net::kOut];               // this lane's share of the far-cell correction (R, J)
	for(int k = 0; k < nbh_net::kOut; ++k) { acc[k] = 0.0f; }
	const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
	unsigned long long vis = 0, taken = 0, spill = 0, corrected = 0, nearq = 0;

	// Evaluate full tiles of 16 far rows (and, with flush, the zero-padded
	// remainder); rows not consumed move to the front.
	auto run_tiles = [&](int& nb, bool flush) {
		while(nb >= 16 || (flush && nb > 0))
		{
			if(nb < 16)
			{
				for(int r = nb + (lane >> 4); r < 16; r += 4)
				{
					bandf[r * nbh_net::kIn + col] = 0;
					bandb[r * nbh_net::kBasis + col] = 0.0f;
					if(col < 2) { bandw[2 * r + col] = 0.0f; }
				}
				__syncthreads();
			}
			const nbh_net::bf16x4 xa = nbh_net::lds_afrag(bandf, nbh_net::kIn, 0, lane);
			const nbh_net::f32x4 o = nbh_net::forward_tile(xa, frags, mlp_p, mlds, lane, nullptr, nullptr);
			for(int e = 0; e < 4; ++e)
			{
				const int row = 4 * (lane >> 4) + e;
				float v[nbh_net::kOut];
				nbh_net::basis_col(bandb + row * nbh_net::kBasis, col, v);
				const float c0 = o[e] * bandw[2 * row], c1 = o[e] * bandw[2 * row + 1];
				for(int k = 0; k < 3; ++k) { acc[k] = fmaf(c0, v[k], acc[k]); }
				for(int k = 3; k < nbh_net::kOut; ++k) { acc[k] = fmaf(c1, v[k], acc[k]); }
			}
			const int rest = nb > 16 ? nb - 16 : 0;
			__syncthreads();
			for(int r = lane >> 4; r < rest; r += 4)
			{
				bandf[r * nbh_net::kIn + col] = bandf[(r + 16) * nbh_net::kIn + col];
				bandb[r * nbh_net::kBasis + col] = bandb[(r + 16) * nbh_net::kBasis + col];
				if(col < 2) { bandw[2 * r + col] = bandw[2 * (r + 16) + col]; }
			}
			__syncthreads();
			nb = rest;
		}
	};

	int sp = 1;
	int nbuf = 0;
	int nband = 0;
	int nq = 0;
	if(lane == 0) { stack[0] = kRoot; }
	__syncthreads();
	while(sp > 0)
	{
		bool valid;
		int node;
		double4 rec;
		double m;
		// node loads first, then the pending sweeps (same order as k_bh_group32)
		int2 kids;
		walk_fetch(stack, sp, lane, wr, node, valid, rec, m, kids);
		if(nbuf > kWalkBuf - kGroup)
		{
			sweep32(buf, nbuf, tx, ty, tz, ax, ay, az, cx, cy, cz);
			nbuf = 0;
		}
		if(nq > kQuadBuf - kGroup)
		{
			sweep_mq(qbuf, nq, tx, ty, tz, ax, ay, az, cx, cy, cz);
			nq = 0;
		}
		__syncthreads();
		bool accept = false, open = false;
		int cls = kCellNone;
		float4 ent = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		double dc = 0.0;
		if(valid)
		{
			ent = sweep_entry(rec, m, ccx, ccy, ccz);
			if(node >= n)
			{
				accept = true;
			}
			else
			{
				const double ex = fmax(fmax(gx0 - rec.x, rec.x - gx1), 0.0);
				const double ey = fmax(fmax(gy0 - rec.y, rec.y - gy1), 0.0);
				const double ez = fmax(fmax(gz0 - rec.z, rec.z - gz1), 0.0);
				accept = ex * ex + ey * ey + ez * ez > rec.w;
				open = !accept;
				if(accept)
				{
					cls = classify_cell(bmin + 3 * node, bmax + 3 * node, rec, ccx, ccy, ccz, hd, near_k, rho_min, &dc);
				}
			}
		}
		const int nopen = __popcll(__ballot(open));
		if(sp + nopen > kWalkStack)
		{
			spill += open ? 1 : 0;
			accept = accept || open;
			open = false;
		}
		const bool band = cls == kCellFar;
		const bool isnear = cls == kCellNear;
		const uint64_t bacc = __ballot(accept);
		const uint64_t bopen = __ballot(open);
		const uint64_t bband = __ballot(band);
		const uint64_t bnear = __ballot(isnear);
		const uint64_t bmono = bacc & ~bnear;     // near cells go to the monopole + quadrupole sweep
		if(accept && !isnear) { buf[nbuf + __popcll(bmono & lt)] = ent; }
		if(open) { stack[sp + __popcll(bopen & lt)] = 2 * node; }
		if(band)
		{
			const int slot = nband + __popcll(bband & lt);
			float fe[nbh_net::kIn];
			float be[nbh_net::kBasis];
			const float scale = nbh_net::cell_features_fast(
			    static_cast<float>(rec.x - ccx), static_cast<float>(rec.y - ccy), static_cast<float>(rec.z - ccz),
			    rec.x, rec.y, rec.z, m, bmin + 3 * node, bmax + 3 * node, wr[node].q, fe, be);
			for(int k = 0; k < nbh_net::kBasis; ++k) { bandb[slot * nbh_net::kBasis + k] = be[k]; }
			bandw[2 * slot] = scale;
			bandw[2 * slot + 1] = scale / (static_cast<float>(nbh_net::kJac) * static_cast<float>(dc));
			for(int k = 0; k < nbh_net::kIn; ++k) { bandf[slot * nbh_net::kIn + k] = nbh_net::to_bf16(fe[k]); }
		}
		if(isnear)
		{
			put_quad(qbuf, nq + __popcll(bnear & lt), ent, wr[node].q);
		}
		nbuf += __popcll(bmono);
		sp += __popcll(bopen);
		nband += __popcll(bband);
		nq += __popcll(bnear);
		corrected += band ? 1 : 0;
		nearq += isnear ? 1 : 0;
		vis += valid ? 1 : 0;
		taken += accept ? 1 : 0;
		__syncthreads();
		if(nband >= 16) { run_tiles(nband, false); }
	}
	if(nbuf > 0)
	{
		sweep32(buf, nbuf, tx, ty, tz, ax, ay, az, cx, cy, cz);
	}
	if(nq > 0)
	{
		sweep_mq(qbuf, nq, tx, ty, tz, ax, ay, az, cx, cy, cz);
	}
	__syncthreads();
	run_tiles(nband, true);
	for(int sh = 1; sh < 64; sh <<= 1)
	{
		for(int k = 0; k < nbh_net::kOut; ++k) { acc[k] += __shfl_xor(acc[k], sh, 64); }
	}
	const float* S = acc;
	const float ux = static_cast<float>(me.x - ccx);   // unscaled offset for the correction
	const float uy = static_cast<float>(me.y - ccy);
	const float uz = static_cast<float>(me.z - ccz);
	const float kx = S[0] + S[3] * ux + S[6] * uy + S[7] * uz;
	const float ky = S[1] + S[6] * ux + S[4] * uy + S[8] * uz;
	const float kz = S[2] + S[7] * ux + S[8] * uy + S[5] * uz;
	const int b = body_n[tn];
	f[b] = y[3 * n + b];
	f[n + b] = y[4 * n + b];
	f[2 * n + b] = y[5 * n + b];
	f[3 * n + b] = static_cast<double>(ax) - static_cast<double>(cx) + static_cast<double>(kx);
	f[4 * n + b] = static_cast<double>(ay) - static_cast<double>(cy) + static_cast<double>(ky);
	f[5 * n + b] = static_cast<double>(az) - static_cast<double>(cz) + static_cast<double>(kz);
	for(int off = 32; off > 0; off >>= 1)
	{
		vis += __shfl_down(vis, off, 64);
		taken += __shfl_down(taken, off, 64);
		spill += __shfl_down(spill, off, 64);
		corrected += __shfl_down(corrected, off, 64);
		nearq += __shfl_down(nearq, off, 64);
	}
	if(lane == 0)
	{
		atomicAdd(&counters[0], taken * kGroup);
		atomicAdd(&counters[1], vis);
		if(spill) { atomicAdd(&counters[2], spill); }
		atomicAdd(&counters[3], corrected);
		atomicAdd(&counters[4], nearq);
	}
}

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------
nbh_status scan_exclusive(nbh_ctx* ctx, uint32_t* c, size_t m, uint32_t* scan_part)
{
	if(m <= static_cast<size_t>(kScanOneThreads) * kScanOneItems)
	{
		hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(kScanOneThreads), 0, ctx->stream, c, static_cast<int>(m));
		NBH_LAUNCHED();
		return NBH_OK;
	}
	size_t chunk = (m + kScanParts - 1) / kScanParts;
	chunk = (chunk + 4 * kScanThreads - 1) / (4 * kScanThreads) * (4 * kScanThreads);
	const unsigned g = static_cast<unsigned>((m + chunk - 1) / chunk);
	hipLaunchKernelGGL(k_scan_reduce, dim3(g), dim3(kScanThreads), 0, ctx->stream, c, m, chunk, scan_part);
	NBH_LAUNCHED();
	hipLaunchKernelGGL(k_scan_parts, dim3(1), dim3(kScanParts), 0, ctx->stream, scan_part, static_cast<int>(g));
	NBH_LAUNCHED();
	hipLaunchKernelGGL(k_scan_apply, dim3(g), dim3(kScanThreads), 0, ctx->stream, c, m, chunk, scan_part);
	NBH_LAUNCHED();
	return NBH_OK;
}

// Sorts `sets` lists whose keys, values and cleared scratch (sort_words each) are
// in place.
nbh_status sort_run(nbh_ctx* ctx, const sort_lists& a, int sets, size_t n, int passes, bool keep_keys,
                    uint32_t* scratch)
{
	const unsigned ys = static_cast<unsigned>(sets);
	if(n <= static_cast<size_t>(kSortTile))
	{
		hipLaunchKernelGGL(k_sort_one, dim3(1, ys), dim3(kSortOneThreads), 0, ctx->stream, a, static_cast<int>(n),
		                   passes, keep_keys ? 1 : 0);
		NBH_LAUNCHED();
		return NBH_OK;
	}
	const size_t tiles = (n + kSortTile - 1) / kSortTile;
	hipLaunchKernelGGL(k_sort_hist, dim3(static_cast<unsigned>(std::min<size_t>(tiles, 512)), ys), dim3(kSortThreads),
	                   0, ctx->stream, a, n, passes, scratch, tiles);
	NBH_LAUNCHED();
	for(int p = 0; p < passes; ++p)
	{
		hipLaunchKernelGGL(k_sort_pass, dim3(static_cast<unsigned>(tiles), ys), dim3(kSortThreads), 0, ctx->stream, a, n,
		                   p, p + 1 == passes ? 1 : 0, keep_keys ? 1 : 0, scratch, tiles);
		NBH_LAUNCHED();
	}
	return NBH_OK;
}

// The bodies in x, y and z order: t->list[0..2].  The three sorts run together;
// their keys and values take the walk records' space, which the build writes
// after them (record 0, which no build writes, stays).
nbh_status sort_axes(nbh_ctx* ctx, nbh_tree* t, const double* y)
{
	const size_t n = t->n;
	if(n == 1)
	{
		for(int a = 0; a < 3; ++a)
		{
			hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, ctx->stream, reinterpret_cast<int*>(t->list[a]),
			                   static_cast<size_t>(1), 0);
			NBH_LAUNCHED();
		}
		return NBH_OK;
	}
	static_assert(sizeof(nbh_walk_rec) * 3 >= 3 * 2 * 2 * (sizeof(uint64_t) + sizeof(uint32_t)), "n = 2 fits");
	sort_lists a;
	uint64_t* keys = reinterpret_cast<uint64_t*>(t->wrec + 1);
	uint32_t* vals = reinterpret_cast<uint32_t*>(keys + 6 * n);
	for(int d = 0; d < 3; ++d)
	{
		for(int h = 0; h < 2; ++h)
		{
			a.l[d].k[h] = keys + (2 * d + h) * n;
			a.l[d].v[h] = vals + (2 * d + h) * n;
		}
		a.l[d].out = t->list[d];
	}
	const size_t words = sort_words((n + kSortTile - 1) / kSortTile);
	hipLaunchKernelGGL(k_make_keys, dim3(nbh::grid_for(ctx, n, 256), 3), dim3(256), 0, ctx->stream, y, a, n, t->counts,
	                   words);
	NBH_LAUNCHED();
	return sort_run(ctx, a, 3, n, 8, false, t->counts);
}

nbh_status moments(nbh_ctx* ctx, nbh_tree* t, const double* y, const double* mass, const uint32_t* order, double ratio)
{
	t->ratio = ratio;
	const size_t n = t->n;
	size_t lo = n;
	do
	{
		const size_t width = std::min<size_t>(lo, kHeapBase);
		const auto kernel = lo == n ? k_heap_moments<true> : k_heap_moments<false>;
		hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(lo / width)), dim3(kHeapBase), 0, ctx->stream, lo,
		                   static_cast<int>(width), n, order, y, mass, t->xyzr, t->mass, t->bmin, t->bmax, t->quad,
		                   t->body_n, ratio * ratio, t->wrec);
		NBH_LAUNCHED();
		lo /= width;
	} while(lo > 1);
	return NBH_OK;
}

}  // namespace

namespace nbh {

size_t sort_counts_size(size_t n) { return sort_words((n + kSortTile - 1) / kSortTile); }

nbh_status sort_pairs(nbh_ctx* ctx, uint64_t* k0, uint32_t* v0, uint64_t* k1, uint32_t* v1, size_t n, int bits,
                      uint32_t* counts, uint32_t** sorted_vals)
{
	const int passes = (bits + 7) / 8;
	uint32_t* out = passes % 2 == 0 ? v0 : v1;
	sort_lists a = {};
	a.l[0] = {{k0, k1}, {v0, v1}, out};
	NBH_TRY(sort_run(ctx, a, 1, n, passes, true, counts));
	*sorted_vals = out;
	return NBH_OK;
}

}  // namespace nbh

extern "C" {

// The buffers a tree allocates at creation, with their sizes in bytes.
constexpr int kTreeBuffers = 17;
static void tree_buffers(nbh_tree* t, void** ptrs[kTreeBuffers], size_t sizes[kTreeBuffers])
{
	const size_t n = t->n;
	const size_t ncounts = std::max(kSortSets * sort_words((n + kSortTile - 1) / kSortTile),
	                                2 * ((n + kPartTile - 1) / kPartTile)) + 1;
	int k = 0;
	auto add = [&](void* p, size_t bytes) {
		ptrs[k] = static_cast<void**>(p);
		sizes[k] = bytes;
		++k;
	};
	for(int a = 0; a < 3; ++a) { add(&t->list[a], n * sizeof(uint32_t)); }
	add(&t->tmp, n * sizeof(uint32_t));
	add(&t->side, n);
	add(&t->keys, 2 * n * sizeof(uint64_t));
	add(&t->vals, 2 * n * sizeof(uint32_t));
	add(&t->counts, ncounts * sizeof(uint32_t));
	add(&t->scan_part, kScanParts * sizeof(uint32_t));
	add(&t->xyzr, 2 * n * sizeof(double4));
	add(&t->mass, 2 * n * sizeof(double));
	add(&t->bmin, 2 * n * 3 * sizeof(double));
	add(&t->bmax, 2 * n * 3 * sizeof(double));
	add(&t->quad, 2 * n * 6 * sizeof(double));
	add(&t->wrec, 2 * n * sizeof(nbh_walk_rec));
	add(&t->body_n, 2 * n * sizeof(int32_t));
	add(&t->counters, 5 * sizeof(unsigned long long));
}

static size_t tree_base_bytes(size_t n)
{
	nbh_tree probe;
	probe.n = n;
	void** ptrs[kTreeBuffers];
	size_t sizes[kTreeBuffers];
	tree_buffers(&probe, ptrs, sizes);
	size_t total = 0;
	for(size_t b : sizes) { total += b; }
	return total;
}

nbh_status nbh_tree_create(nbh_ctx* ctx, size_t n, nbh_tree** out)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(out != nullptr, "null output pointer");
	*out = nullptr;
	NBH_CHECK(n >= 1, "empty tree");
	NBH_CHECK(n <= (static_cast<size_t>(1) << 28), "body count %zu too large", n);
	nbh_tree* t = new nbh_tree();
	t->ctx = ctx;
	t->n = n;
	while((static_cast<size_t>(1) << t->levels) < n) { ++t->levels; }
	void** ptrs[kTreeBuffers];
	size_t sizes[kTreeBuffers];
	tree_buffers(t, ptrs, sizes);
	hipError_t e = hipSuccess;
	for(int k = 0; k < kTreeBuffers && e == hipSuccess; ++k)
	{
		e = hipMalloc(ptrs[k], sizes[k]);
	}
	if(e == hipSuccess) { e = hipMemsetAsync(t->xyzr, 0, 2 * n * sizeof(double4), ctx->stream); }
	if(e == hipSuccess) { e = hipMemsetAsync(t->mass, 0, 2 * n * sizeof(double), ctx->stream); }
	// box 0, which no node has and nbh_tree_get returns with the others
	if(e == hipSuccess) { e = hipMemsetAsync(t->bmin, 0, 3 * sizeof(double), ctx->stream); }
	if(e == hipSuccess) { e = hipMemsetAsync(t->bmax, 0, 3 * sizeof(double), ctx->stream); }
	if(e == hipSuccess) { e = hipMemsetAsync(t->quad, 0, 2 * n * 6 * sizeof(double), ctx->stream); }
	if(e == hipSuccess) { e = hipMemsetAsync(t->wrec, 0, 2 * n * sizeof(nbh_walk_rec), ctx->stream); }
	if(e == hipSuccess) { e = hipMemsetAsync(t->body_n, 0xff, 2 * n * sizeof(int32_t), ctx->stream); }
	if(e == hipSuccess) { e = hipMemsetAsync(t->counters, 0, 5 * sizeof(unsigned long long), ctx->stream); }
	if(e == hipSuccess) { e = hipStreamSynchronize(ctx->stream); }
	if(e != hipSuccess)
	{
		nbh_tree_destroy(t);
		return nbh::hip_fail(e, "tree allocation", __FILE__, __LINE__);
	}
	*out = t;
	return NBH_OK;
}

// The Morton tree's buffers, all together or none.
static nbh_status radix_alloc(nbh_tree* t)
{
	if(t->child != nullptr)
	{
		return NBH_OK;
	}
	const size_t n = t->n;
	constexpr int kBufs = 13;
	void* p[kBufs] = {};
	const size_t sizes[kBufs] = { n * sizeof(int2), 2 * n * sizeof(int), n * sizeof(uint8_t),
	                              (n + kRadixTiers) * sizeof(int), n * sizeof(int2), n * sizeof(int2),
	                              mark_words(n) * sizeof(uint32_t), n * sizeof(int4),
	                              (n / kRadixWalk + 1) * sizeof(int2), 6 * (kBoxParts + 1) * sizeof(double),
	                              n * sizeof(double4), n * sizeof(int2), n * sizeof(int4) };
	hipError_t e = hipSuccess;
	for(int k = 0; k < kBufs && e == hipSuccess; ++k)
	{
		e = hipMalloc(&p[k], sizes[k]);
	}
	if(e == hipSuccess && t->info_ready == nullptr)
	{
		e = hipEventCreateWithFlags(&t->info_ready, hipEventDisableTiming);
	}
	if(e != hipSuccess)
	{
		for(void* q : p)
		{
			if(q != nullptr) { (void)hipFree(q); }
		}
		return nbh::hip_fail(e, "Morton tree allocation", __FILE__, __LINE__);
	}
	t->child = static_cast<int2*>(p[0]);
	t->parent = static_cast<int*>(p[1]);
	t->tier = static_cast<uint8_t*>(p[2]);
	t->tier_list = static_cast<int*>(p[3]);
	t->gmark = static_cast<int2*>(p[4]);
	t->smark = static_cast<int2*>(p[5]);
	t->marks = static_cast<uint32_t*>(p[6]);
	t->grp = static_cast<int4*>(p[7]);
	t->sup = static_cast<int2*>(p[8]);
	t->box = static_cast<double*>(p[9]);
	t->pk = static_cast<double4*>(p[10]);
	t->wmark = static_cast<int2*>(p[11]);
	t->wgrp = static_cast<int4*>(p[12]);
	return NBH_OK;
}

// Leaves, moments and walk records of the Morton tree's build groups, one wave per
// group (any number of work-groups will do).  build: leaves from `order` (sorted body
// numbers) and the packed bodies, else from the body numbers of the last build and
// the positions y.
static nbh_status radix_groups(nbh_ctx* ctx, nbh_tree* t, const double* y, const uint32_t* order, bool build,
                               size_t blocks)
{
	const auto kernel = build ? k_radix_group_moments<true> : k_radix_group_moments<false>;
	hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(kRadixGroup), 0, ctx->stream, t->grp,
	                   radix_marks(t->marks, t->n).info + kRadixTiers + kMarkBuild, static_cast<int>(t->n), t->child,
	                   order, t->pk, y, t->body_n, t->xyzr, t->mass, t->bmin, t->bmax, t->quad, t->ratio * t->ratio,
	                   t->wrec, t->radix_lean ? 1 : 0);
	NBH_LAUNCHED();
	return NBH_OK;
}

// The nodes above the build groups, tier by tier up to the root.
static nbh_status radix_tiers(nbh_ctx* ctx, nbh_tree* t)
{
	for(int k = 1; k < kRadixTiers; ++k)
	{
		if(t->tier_count[k] == 0) { continue; }
		hipLaunchKernelGGL(k_radix_tier, dim3(static_cast<unsigned>(t->tier_count[k])), dim3(256), 0, ctx->stream,
		                   t->tier_list + tier_offset(t->n, k), k, static_cast<int>(t->n), t->child, t->tier, t->xyzr,
		                   t->mass, t->bmin, t->bmax, t->quad, t->ratio * t->ratio, t->wrec);
		NBH_LAUNCHED();
	}
	return NBH_OK;
}

nbh_status nbh_tree_build_radix(nbh_ctx* ctx, nbh_tree* t, const double* y, const double* mass, double ratio)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(y != nullptr && mass != nullptr, "null buffer");
	NBH_CHECK(t->n >= 2, "the Morton tree needs at least 2 bodies");
	NBH_TRY(radix_alloc(t));
	nbh::scoped_timer timer(ctx, "tree_build");
	const size_t n = t->n;
	t->built = false;
	const unsigned parts = std::min<unsigned>(kBoxParts, nbh::grid_for(ctx, n, 256));
	hipLaunchKernelGGL(k_box_partial, dim3(parts), dim3(256), 0, ctx->stream, y, n, t->box + 6);
	NBH_LAUNCHED();
	hipLaunchKernelGGL(k_box_final, dim3(1), dim3(256), 0, ctx->stream, t->box + 6, static_cast<int>(parts), t->box);
	NBH_LAUNCHED();
	hipLaunchKernelGGL(k_morton_codes, dim3(nbh::grid_for(ctx, n, 256)), dim3(256), 0, ctx->stream, y, mass, n,
	                   t->box, t->keys, t->vals, t->pk, t->marks, mark_words(n), t->parent, t->counts,
	                   nbh::sort_counts_size(n));
	NBH_LAUNCHED();
	uint32_t* order = nullptr;
	// 63-bit keys: 8 passes, so the sorted keys end where they started
	NBH_TRY(nbh::sort_pairs(ctx, t->keys, t->vals, t->keys + n, t->vals + n, n, 63, t->counts, &order));
	const RadixMarks marks = radix_marks(t->marks, n);
	hipLaunchKernelGGL(k_radix_nodes, dim3(nbh::grid_for(ctx, n, 256)), dim3(256), 0, ctx->stream, t->keys,
	                   static_cast<long long>(n), t->child, t->parent, t->tier, t->tier_list, marks, t->gmark,
	                   t->smark, t->wmark);
	NBH_LAUNCHED();
	const unsigned mark_grid = static_cast<unsigned>((marks.parts() + 3) / 4);
	hipLaunchKernelGGL(k_radix_count, dim3(mark_grid), dim3(256), 0, ctx->stream, marks);
	NBH_LAUNCHED();
	hipLaunchKernelGGL(k_radix_groups, dim3(mark_grid), dim3(256), 0, ctx->stream,
	                   marks, t->gmark, t->smark, t->wmark, t->grp, t->sup, t->wgrp);
	NBH_LAUNCHED();
	// the counts drive the launches that follow the build groups' moments, which run
	// while they travel (a group holds some 40 leaves)
	constexpr size_t kInfoBytes = kInfoCounts * sizeof(int);
	NBH_TRY(nbh::pinned(ctx, kInfoBytes));
	const int* host_info = reinterpret_cast<const int*>(ctx->pinned);
	NBH_HIP(hipMemcpyAsync(ctx->pinned, marks.info, kInfoBytes, hipMemcpyDeviceToHost, ctx->stream));
	hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
	NBH_HIP(hipStreamIsCapturing(ctx->stream, &capture));
	if(capture != hipStreamCaptureStatusNone)
	{
		NBH_HIP(hipStreamSynchronize(ctx->stream));      // not in a capture: the host needs the counts
	}
	NBH_HIP(hipEventRecord(t->info_ready, ctx->stream));
	t->ratio = ratio;
	NBH_TRY(radix_groups(ctx, t, y, order, true, n / 32 + 1));
	NBH_HIP(hipEventSynchronize(t->info_ready));
	for(int k = 0; k < kRadixTiers; ++k)
	{
		t->tier_count[k] = host_info[k];
		NBH_CHECK(k == 0 || (t->tier_count[k] >= 0 && tier_offset(n, k) + t->tier_count[k] <= tier_offset(n, k + 1)),
		          "bad count %d of tier %d", t->tier_count[k], k);
	}
	t->ngroups = host_info[kRadixTiers + kMarkBuild];
	t->nsupers = host_info[kRadixTiers + kMarkSuper];
	t->nwalk = host_info[kRadixTiers + kMarkWalk];
	NBH_CHECK(t->ngroups >= 1 && static_cast<size_t>(t->ngroups) <= n, "bad group count %d", t->ngroups);
	NBH_CHECK(t->nwalk >= 1 && t->nwalk <= t->ngroups, "bad walk group count %d", t->nwalk);
	NBH_CHECK(t->nsupers >= 0 && static_cast<size_t>(t->nsupers) <= n / kRadixWalk + 1,
	          "bad super-group count %d", t->nsupers);
	NBH_TRY(radix_tiers(ctx, t));
	t->radix = true;
	t->built = true;
	return NBH_OK;
}

nbh_status nbh_tree_get_children(nbh_ctx* ctx, const nbh_tree* t, int32_t* child, int32_t* parent)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(t->built && t->radix, "no Morton tree has been built");
	if(child != nullptr)
	{
		NBH_HIP(hipMemcpyAsync(child, t->child, t->n * sizeof(int2), hipMemcpyDeviceToHost, ctx->stream));
	}
	if(parent != nullptr)
	{
		NBH_HIP(hipMemcpyAsync(parent, t->parent, 2 * t->n * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
	}
	NBH_HIP(hipStreamSynchronize(ctx->stream));
	return NBH_OK;
}

nbh_status nbh_tree_destroy(nbh_tree* t)
{
	if(t == nullptr)
	{
		return NBH_OK;
	}
	if(t->ctx != nullptr)
	{
		(void)hipSetDevice(t->ctx->device);
		(void)hipStreamSynchronize(t->ctx->stream);
	}
	void* ptrs[] = { t->list[0], t->list[1], t->list[2], t->tmp, t->side, t->keys, t->vals, t->counts, t->scan_part,
	                 t->xyzr, t->mass, t->bmin, t->bmax, t->quad, t->wrec, t->body_n, t->counters,
	                 t->two_lists, t->two_count, t->two_coef, t->far_list, t->far_count,
	                 t->child, t->parent, t->tier, t->tier_list, t->gmark, t->smark, t->marks,
	                 t->grp, t->sup, t->box, t->pk, t->wmark, t->wgrp };
	for(void* p : ptrs)
	{
		if(p != nullptr) { (void)hipFree(p); }
	}
	if(t->info_ready != nullptr) { (void)hipEventDestroy(t->info_ready); }
	delete t;
	return NBH_OK;
}

nbh_status nbh_tree_build(nbh_ctx* ctx, nbh_tree* t, const double* y, const double* mass, double ratio)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(y != nullptr && mass != nullptr, "null buffer");
	NBH_CHECK((t->n & (t->n - 1)) == 0, "body count %zu is not a power of two (the heap tree needs 2^k leaves)", t->n);
	nbh::scoped_timer timer(ctx, "tree_build");
	const size_t n = t->n;
	t->radix = false;
	NBH_TRY(sort_axes(ctx, t, y));
	const unsigned ntiles = static_cast<unsigned>((n + kPartTile - 1) / kPartTile);
	// the last levels (segments of at most kLocalSeg bodies) run in LDS
	const int local_levels = std::min(t->levels, 12);
	static_assert(kLocalSeg == 1 << 12 && kLocalSeg >= kPartTile, "kLocalSeg is 2^12, whole tiles");
	const int global_levels = t->levels - local_levels;
	// lists to write and the next level's flags: what the sort no longer needs
	uint32_t* cur[3] = {t->list[0], t->list[1], t->list[2]};
	uint32_t* spare[2] = {t->tmp, reinterpret_cast<uint32_t*>(t->keys)};
	uint8_t*  side[2] = {t->side, reinterpret_cast<uint8_t*>(t->vals)};
	if(global_levels > 0)
	{
		hipLaunchKernelGGL(k_mark_side, dim3(nbh::grid_for(ctx, n, 256)), dim3(256), 0, ctx->stream, cur[0], side[0], n,
		                   n);
		NBH_LAUNCHED();
	}
	for(int level = 0; level < global_levels; ++level)
	{
		const size_t seg = n >> level;
		const int b0 = (level + 1) % 3, b1 = (level + 2) % 3;
		const part_lists lists = {{cur[b0], cur[b1]}, {spare[0], spare[1]}};
		hipLaunchKernelGGL(k_part_count, dim3(ntiles, 2), dim3(kPartThreads), 0, ctx->stream, lists, side[level & 1],
		                   t->counts);
		NBH_LAUNCHED();
		const int scanned = seg / kPartTile > kPartSum ? 1 : 0;
		if(scanned != 0) { NBH_TRY(scan_exclusive(ctx, t->counts, 2 * static_cast<size_t>(ntiles), t->scan_part)); }
		hipLaunchKernelGGL(k_part_scatter, dim3(ntiles, 2), dim3(kPartThreads), 0, ctx->stream, lists, side[level & 1],
		                   seg, t->counts, scanned, level + 1 < global_levels ? 0 : -1, side[~level & 1]);
		NBH_LAUNCHED();
		std::swap(cur[b0], spare[0]);
		std::swap(cur[b1], spare[1]);
	}
	if(local_levels > 0)
	{
		const size_t seg0 = n >> global_levels;
		hipLaunchKernelGGL(k_split_local, dim3(static_cast<unsigned>(n / seg0)), dim3(kLocalThreads), 0, ctx->stream,
		                   cur[0], cur[1], cur[2], spare[0], static_cast<int>(seg0), global_levels, t->levels);
		NBH_LAUNCHED();
	}
	NBH_TRY(moments(ctx, t, y, mass, cur[0], ratio));
	t->built = true;
	return NBH_OK;
}

nbh_status nbh_tree_set_radix_lean(nbh_ctx* ctx, nbh_tree* t, int lean)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	t->radix_lean = lean != 0;
	return NBH_OK;
}

nbh_status nbh_tree_refit(nbh_ctx* ctx, nbh_tree* t, const double* y, double ratio)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(t->built, "tree has not been built");
	NBH_CHECK(y != nullptr, "null buffer");
	nbh::scoped_timer timer(ctx, "tree_refit");
	if(t->radix)
	{
		t->ratio = ratio;
		NBH_TRY(radix_groups(ctx, t, y, nullptr, false, static_cast<size_t>(t->ngroups)));
		return radix_tiers(ctx, t);
	}
	return moments(ctx, t, y, nullptr, nullptr, ratio);
}

nbh_status nbh_bh_fcompute(nbh_ctx* ctx, const nbh_tree* t, const double* y, const double* mass, double* f,
                           nbh_tree_layout layout, nbh_precision precision)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(t->built, "tree has not been built");
	NBH_CHECK(!t->radix, "this walk runs on the heap tree only (the last build made the Morton tree)");
	NBH_CHECK(y != nullptr && mass != nullptr && f != nullptr && y != f, "bad buffers");
	NBH_CHECK(layout == NBH_LAYOUT_HEAP || layout == NBH_LAYOUT_HEAP_STACKLESS, "unknown layout %d",
	          static_cast<int>(layout));
	NBH_CHECK(precision == NBH_FP64 || precision == NBH_FP32, "unknown precision %d", static_cast<int>(precision));
	const int n = static_cast<int>(t->n);
	hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, ctx->stream, t->counters);
	NBH_LAUNCHED();
	nbh::scoped_timer timer(ctx, "bh_traverse");
	dim3 grid((n + 255) / 256);
	if(precision == NBH_FP32)
	{
		hipLaunchKernelGGL(k_bh_stackless32, grid, dim3(256), 0, ctx->stream, t->xyzr, t->mass, t->body_n, y, mass,
		                   f, n, t->counters);
	}
	else
	{
		hipLaunchKernelGGL(k_bh_walk64, dim3((n + kWalkTgt - 1) / kWalkTgt), dim3(64), 0, ctx->stream, t->xyzr, t->mass,
		                   t->body_n, y, mass, f, n, t->counters);
	}
	NBH_LAUNCHED();
	return NBH_OK;
}

enum GroupMode { kGroupMonopole, kGroupQuad, kGroupLocal };

static WalkTree walk_tree(const nbh_tree* t)
{
	WalkTree wt;
	if(t->radix)
	{
		wt.child = t->child;
		wt.grp = t->wgrp;
		wt.sup = t->sup;
		wt.ngroups = t->nwalk;
		wt.nsupers = t->nsupers;
	}
	return wt;
}

static nbh_status group_walk(nbh_ctx* ctx, const nbh_tree* t, const double* y, double* f, GroupMode mode,
                             float near_k)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(t->built, "tree has not been built");
	NBH_CHECK(y != nullptr && f != nullptr && y != f, "bad buffers");
	NBH_CHECK(t->radix || t->n >= static_cast<size_t>(kGroup), "group walk needs at least %d bodies", kGroup);
	NBH_CHECK(t->radix || (t->levels + 2) * (kGroup / 2) <= kWalkStack, "tree too deep for the walk stack");
	const int n = static_cast<int>(t->n);
	hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, ctx->stream, t->counters);
	NBH_LAUNCHED();
	nbh::scoped_timer timer(ctx, "bh_traverse");
	if(t->radix)
	{
		// the Morton tree's depth is not bounded by log2(n): a step whose children
		// would not fit on the stack takes the nodes as monopoles (counters[2])
		const WalkTree wt = walk_tree(t);
		if(mode == kGroupQuad)
		{
			const unsigned grid = static_cast<unsigned>(t->nwalk);
			hipLaunchKernelGGL((k_bh_group32<true, false, false, true>), dim3(grid), dim3(kGroup), 0,
			                   ctx->stream, t->wrec, t->bmin, t->bmax, t->body_n, y, f, n, near_k, t->counters,
			                   TwoLevel(), wt);
		}
		else if(mode == kGroupLocal)
		{
			const unsigned grid = static_cast<unsigned>(t->nwalk);
			hipLaunchKernelGGL((k_bh_group32<true, true, false, true>), dim3(grid), dim3(kGroup), 0,
			                   ctx->stream, t->wrec, t->bmin, t->bmax, t->body_n, y, f, n, near_k, t->counters,
			                   TwoLevel(), wt);
		}
		else
		{
			const unsigned grid = static_cast<unsigned>(t->nwalk);
			hipLaunchKernelGGL((k_bh_group32<false, false, false, true>), dim3(grid), dim3(kGroup), 0,
			                   ctx->stream, t->wrec, t->bmin, t->bmax, t->body_n, y, f, n, 0.0f, t->counters,
			                   TwoLevel(), wt);
		}
		NBH_LAUNCHED();
		return NBH_OK;
	}
	if(mode == kGroupQuad)
	{
		const unsigned grid = static_cast<unsigned>(n / kGroup);
		hipLaunchKernelGGL((k_bh_group32<true>), dim3(grid), dim3(kGroup), 0, ctx->stream, t->wrec, t->bmin,
		                   t->bmax, t->body_n, y, f, n, near_k, t->counters);
	}
	else if(mode == kGroupLocal)
	{
		const unsigned grid = static_cast<unsigned>(n / kGroup);
		hipLaunchKernelGGL((k_bh_group32<true, true>), dim3(grid), dim3(kGroup), 0, ctx->stream, t->wrec,
		                   t->bmin, t->bmax, t->body_n, y, f, n, near_k, t->counters);
	}
	else
	{
		const unsigned grid = static_cast<unsigned>(n / kGroup);
		hipLaunchKernelGGL((k_bh_group32<false>), dim3(grid), dim3(kGroup), 0, ctx->stream, t->wrec, t->bmin,
		                   t->bmax, t->body_n, y, f, n, 0.0f, t->counters);
	}
	NBH_LAUNCHED();
	return NBH_OK;
}

nbh_status nbh_bh_fcompute_group(nbh_ctx* ctx, const nbh_tree* t, const double* y, double* f)
{
	return group_walk(ctx, t, y, f, kGroupMonopole, 0.0f);
}

nbh_status nbh_bh_fcompute_group_quad(nbh_ctx* ctx, const nbh_tree* t, const double* y, double* f, float near_k)
{
	NBH_CHECK(near_k >= 0.0f, "near_k must be >= 0");
	return group_walk(ctx, t, y, f, kGroupQuad, near_k);
}

nbh_status nbh_bh_fcompute_group_local(nbh_ctx* ctx, const nbh_tree* t, const double* y, double* f, float near_k)
{
	NBH_CHECK(near_k >= 1.0f, "near_k must be >= 1 (the expansion needs the cell outside the group)");
	return group_walk(ctx, t, y, f, kGroupLocal, near_k);
}

// List capacity per super-group of the two-level walk (4 bytes per entry).
constexpr int kTwoCap = 32768;

// Bytes of the two-level walk's buffers: per super-group a list of `cap` node
// indices, its length and the 34 coefficients of its expansion.
static size_t two_bytes(size_t supers, int cap)
{
	return supers * (static_cast<size_t>(cap) * sizeof(int) + sizeof(int) + 34 * sizeof(float));
}

// Super-groups of the tree's last build: 1024-body heap nodes, or the Morton
// tree's maximal subtrees of 129 to 2048 bodies.
static size_t super_count(const nbh_tree* t)
{
	return t->radix ? static_cast<size_t>(t->nsupers) : t->n >> (6 + kSuperShift);
}

// Frees the two-level walk's buffers.  Every pointer is null afterwards, also
// when a hipFree fails (the first failure is reported).
static nbh_status two_free(nbh_ctx* ctx, nbh_tree* t)
{
	if(t->two_lists == nullptr && t->two_count == nullptr && t->two_coef == nullptr)
	{
		return NBH_OK;
	}
	hipError_t e = hipStreamSynchronize(ctx->stream);
	void* ptrs[3] = { t->two_lists, t->two_count, t->two_coef };
	t->two_lists = nullptr;
	t->two_count = nullptr;
	t->two_coef = nullptr;
	t->two_slots = 0;
	for(void* p : ptrs)
	{
		if(p != nullptr)
		{
			hipError_t ef = hipFree(p);
			if(e == hipSuccess) { e = ef; }
		}
	}
	if(e != hipSuccess)
	{
		return nbh::hip_fail(e, "freeing the two-level walk lists", __FILE__, __LINE__);
	}
	return NBH_OK;
}

// Allocates the two-level walk's buffers all together or not at all: on any
// failure the ones already allocated are freed and every pointer stays null,
// so a later call allocates afresh instead of launching with a missing buffer.
// NBH_TEST_FAIL_ALLOC=k (k = 1, 2, 3) in the environment makes the k-th of the
// three allocations fail as out of memory (a test hook for this path).
static nbh_status two_alloc(nbh_ctx* ctx, nbh_tree* t, int cap, size_t supers)
{
	NBH_TRY(two_free(ctx, t));
	const size_t sizes[3] = { supers * static_cast<size_t>(cap) * sizeof(int), supers * sizeof(int),
	                          supers * 34 * sizeof(float) };
	int fail_at = 0;
	if(const char* env = getenv("NBH_TEST_FAIL_ALLOC"))
	{
		fail_at = atoi(env);
	}
	void* p[3] = { nullptr, nullptr, nullptr };
	hipError_t e = hipSuccess;
	for(int k = 0; k < 3 && e == hipSuccess; ++k)
	{
		e = (k + 1 == fail_at) ? hipErrorOutOfMemory : hipMalloc(&p[k], sizes[k]);
	}
	if(e != hipSuccess)
	{
		for(void* q : p)
		{
			if(q != nullptr) { (void)hipFree(q); }
		}
		return nbh::hip_fail(e, "two-level walk list allocation", __FILE__, __LINE__);
	}
	t->two_lists = static_cast<int*>(p[0]);
	t->two_count = static_cast<int*>(p[1]);
	t->two_coef = static_cast<float*>(p[2]);
	t->two_slots = static_cast<int>(supers);
	return NBH_OK;
}

// Far cells listed per super-group for the learned correction (4 bytes each);
// cells beyond the cap are left to the plain expansion.
constexpr int kFarCap = 8192;

// The super-groups' far-cell lists, all or nothing (as two_alloc).
static nbh_status far_alloc(nbh_ctx* ctx, nbh_tree* t)
{
	if(t->far_list != nullptr && t->far_count != nullptr)
	{
		return NBH_OK;
	}
	const size_t supers = t->n >> (6 + kSuperShift);
	void* a = nullptr;
	void* b = nullptr;
	hipError_t e = hipMalloc(&a, supers * static_cast<size_t>(kFarCap) * sizeof(int));
	if(e == hipSuccess) { e = hipMalloc(&b, supers * sizeof(int)); }
	if(e != hipSuccess)
	{
		if(a != nullptr) { (void)hipFree(a); }
		if(b != nullptr) { (void)hipFree(b); }
		return nbh::hip_fail(e, "far-cell list allocation", __FILE__, __LINE__);
	}
	(void)ctx;
	if(t->far_list != nullptr) { (void)hipFree(t->far_list); }
	if(t->far_count != nullptr) { (void)hipFree(t->far_count); }
	t->far_list = static_cast<int*>(a);
	t->far_count = static_cast<int*>(b);
	return NBH_OK;
}

// Super-group walk (k_bh_super) with the lists of t; with far lists when
// want_far.  Allocates the lists when they are missing.
static nbh_status super_walk(nbh_ctx* ctx, nbh_tree* t, float near_k, bool want_far, TwoLevel* two)
{
	const size_t supers = super_count(t);
	const int cap = t->two_cap > 0 ? t->two_cap : kTwoCap;
	if(t->two_lists == nullptr || t->two_count == nullptr || t->two_coef == nullptr ||
	   static_cast<size_t>(t->two_slots) < supers)
	{
		NBH_TRY(two_alloc(ctx, t, cap, supers));
	}
	if(want_far)
	{
		NBH_TRY(far_alloc(ctx, t));
	}
	two->lists = t->two_lists;
	two->count = t->two_count;
	two->coef = t->two_coef;
	two->cap = cap;
	two->far_list = want_far ? t->far_list : nullptr;
	two->far_count = want_far ? t->far_count : nullptr;
	two->far_cap = want_far ? kFarCap : 0;
	const int n = static_cast<int>(t->n);
	const float super_near = fmaxf(near_k, kSuperNearMin);
	// NBH_TEST_SUPER_STACK=k (64 <= k <= the stack size) in the environment lets
	// the super-group walk use only k stack entries, so that its overflow path
	// (the groups of a super-group that ran out walk from the root) can be tested
	int stack_limit = kWalkStack;
	if(const char* env = getenv("NBH_TEST_SUPER_STACK"))
	{
		const int k = atoi(env);
		if(k >= kGroup && k <= kWalkStack) { stack_limit = k; }
	}
	if(t->radix)
	{
		hipLaunchKernelGGL(k_bh_super<true>, dim3(static_cast<unsigned>(supers)), dim3(kGroup), 0, ctx->stream,
		                   t->wrec, t->bmin, t->bmax, n, super_near, 1.0 / t->ratio, *two, t->counters, stack_limit,
		                   walk_tree(t));
	}
	else
	{
		hipLaunchKernelGGL(k_bh_super<false>, dim3(static_cast<unsigned>(supers)), dim3(kGroup), 0, ctx->stream,
		                   t->wrec, t->bmin, t->bmax, n, super_near, 1.0 / t->ratio, *two, t->counters, stack_limit,
		                   WalkTree());
	}
	NBH_LAUNCHED();
	return NBH_OK;
}

// Two-level local walk, with the network's correction of the super-groups'
// far fields when net is not null.
static nbh_status two_level(nbh_ctx* ctx, nbh_tree* t, const nbh_mlp* net, const double* y, double* f, float near_k)
{
	NBH_CHECK(near_k >= 1.0f, "near_k must be >= 1 (the expansion needs the cell outside the group)");
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(net == nullptr || nbh::mlp_ctx(net) == ctx, "network does not belong to this context");
	const size_t supers = super_count(t);
	if(supers < 1)
	{
		NBH_CHECK(net == nullptr, "the learned two-level walk needs at least %d bodies", kGroup << kSuperShift);
		return group_walk(ctx, t, y, f, kGroupLocal, near_k);
	}
	NBH_CHECK(t->built, "tree has not been built");
	NBH_CHECK(y != nullptr && f != nullptr && y != f, "bad buffers");
	NBH_CHECK(t->radix || (t->levels + 2) * (kGroup / 2) <= kWalkStack, "tree too deep for the walk stack");
	NBH_CHECK(net == nullptr || !t->radix, "the learned two-level walk runs on the heap tree only");
	const int n = static_cast<int>(t->n);
	hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, ctx->stream, t->counters);
	NBH_LAUNCHED();
	nbh::scoped_timer timer(ctx, "bh_traverse");
	TwoLevel two;
	NBH_TRY(super_walk(ctx, t, near_k, net != nullptr, &two));
	if(net != nullptr)
	{
		hipLaunchKernelGGL(k_super_net, dim3(static_cast<unsigned>(supers)), dim3(64), 0, ctx->stream, t->xyzr,
		                   t->mass, t->bmin, t->bmax, t->quad, n, two, nbh::mlp_frags(net), nbh::mlp_params(net));
		NBH_LAUNCHED();
	}
	{
		// the group walks alone, inside bh_traverse
		nbh::scoped_timer group_timer(ctx, "bh_group_walk");
		if(t->radix)
		{
			const unsigned grid = static_cast<unsigned>(t->nwalk);
			hipLaunchKernelGGL((k_bh_group32<true, true, true, true>), dim3(grid), dim3(kGroup), 0,
			                   ctx->stream, t->wrec, t->bmin, t->bmax, t->body_n, y, f, n, near_k, t->counters, two,
			                   walk_tree(t));
		}
		else
		{
			const unsigned grid = static_cast<unsigned>(n / kGroup);
			hipLaunchKernelGGL((k_bh_group32<true, true, true>), dim3(grid), dim3(kGroup), 0, ctx->stream,
			                   t->wrec, t->bmin, t->bmax, t->body_n, y, f, n, near_k, t->counters, two);
		}
		NBH_LAUNCHED();
	}
	return NBH_OK;
}

nbh_status nbh_bh_fcompute_group_local2(nbh_ctx* ctx, nbh_tree* t, const double* y, double* f, float near_k)
{
	return two_level(ctx, t, nullptr, y, f, near_k);
}

nbh_status nbh_bh_fcompute_group_local2_mlp(nbh_ctx* ctx, nbh_tree* t, const nbh_mlp* net, const double* y,
                                            double* f, float near_k)
{
	NBH_CHECK(net != nullptr, "null network");
	return two_level(ctx, t, net, y, f, near_k);
}

nbh_status nbh_bh_super_samples(nbh_ctx* ctx, nbh_tree* t, float near_k, const uint32_t* supers, size_t n_supers,
                                float* x, float* basis, float* target, uint32_t* cells, size_t capacity,
                                size_t* count)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(t->built, "tree has not been built");
	NBH_CHECK(!t->radix, "this walk runs on the heap tree only (the last build made the Morton tree)");
	NBH_CHECK(near_k >= 1.0f, "near_k must be >= 1");
	NBH_CHECK(supers != nullptr && count != nullptr, "null argument");
	const size_t nsup = t->n >> (6 + kSuperShift);
	NBH_CHECK(nsup >= 1, "no super-group: at least %d bodies are needed", kGroup << kSuperShift);
	NBH_CHECK(n_supers > 0 && n_supers <= nsup, "bad super-group count %zu", n_supers);
	NBH_CHECK(capacity == 0 || (x != nullptr && basis != nullptr && target != nullptr), "null sample buffer");
	NBH_CHECK(capacity <= (static_cast<size_t>(1) << 31), "capacity %zu too large", capacity);
	NBH_CHECK((t->levels + 2) * (kGroup / 2) <= kWalkStack, "tree too deep for the walk stack");
	for(size_t i = 0; i < n_supers; ++i)
	{
		NBH_CHECK(supers[i] < nsup, "super-group %u out of range (%zu)", supers[i], nsup);
	}
	*count = 0;
	hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, ctx->stream, t->counters);
	NBH_LAUNCHED();
	TwoLevel two;
	NBH_TRY(super_walk(ctx, t, near_k, true, &two));
	std::vector<int> far_count(nsup);
	NBH_HIP(hipMemcpyAsync(far_count.data(), t->far_count, nsup * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
	NBH_HIP(hipStreamSynchronize(ctx->stream));
	std::vector<unsigned long long> off(n_supers);
	unsigned long long total = 0;
	for(size_t i = 0; i < n_supers; ++i)
	{
		off[i] = total;
		total += static_cast<unsigned long long>(std::min(far_count[supers[i]], kFarCap));
	}
	*count = static_cast<size_t>(total);
	const size_t m = std::min(static_cast<size_t>(total), capacity);
	if(m == 0)
	{
		return NBH_OK;
	}
	// scratch: selected super-groups, their offsets, then the pairs
	const size_t off_off = (n_supers * sizeof(uint32_t) + 255) / 256 * 256;
	const size_t off_pairs = off_off + (n_supers * sizeof(unsigned long long) + 255) / 256 * 256;
	void* sp = nullptr;
	NBH_TRY(nbh::scratch(ctx, off_pairs + m * 2 * sizeof(uint32_t), &sp));
	char* base = static_cast<char*>(sp);
	uint32_t* dsel = reinterpret_cast<uint32_t*>(base);
	unsigned long long* doff = reinterpret_cast<unsigned long long*>(base + off_off);
	uint32_t* pairs = reinterpret_cast<uint32_t*>(base + off_pairs);
	NBH_HIP(hipMemcpyAsync(dsel, supers, n_supers * sizeof(uint32_t), hipMemcpyHostToDevice, ctx->stream));
	NBH_HIP(hipMemcpyAsync(doff, off.data(), n_supers * sizeof(unsigned long long), hipMemcpyHostToDevice,
	                       ctx->stream));
	hipLaunchKernelGGL(k_super_pairs, dim3(static_cast<unsigned>(n_supers)), dim3(64), 0, ctx->stream, two, dsel, doff,
	                   pairs, static_cast<unsigned long long>(m));
	NBH_LAUNCHED();
	const int n = static_cast<int>(t->n);
	hipLaunchKernelGGL(k_band_residual, dim3(nbh::grid_for(ctx, m, 1)), dim3(64), 0, ctx->stream, t->xyzr, t->mass,
	                   t->bmin, t->bmax, t->quad, n, t->levels, n >> (6 + kSuperShift), 2, pairs, m, x, basis,
	                   target);
	NBH_LAUNCHED();
	if(cells != nullptr)
	{
		NBH_HIP(hipMemcpyAsync(cells, pairs, m * 2 * sizeof(uint32_t), hipMemcpyDeviceToDevice, ctx->stream));
	}
	NBH_HIP(hipStreamSynchronize(ctx->stream));
	return NBH_OK;
}

nbh_status nbh_tree_set_list_cap(nbh_ctx* ctx, nbh_tree* t, int cap)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(cap >= 64 && cap <= (1 << 24), "list capacity %d: must be in [64, 2^24]", cap);
	NBH_TRY(two_free(ctx, t));
	t->two_cap = cap;
	const size_t supers = t->built && t->radix ? super_count(t) : t->n >> (6 + kSuperShift);
	if(supers < 1)
	{
		return NBH_OK;   // no super-group: the walk runs in one level and needs no lists
	}
	return two_alloc(ctx, t, cap, supers);
}

nbh_status nbh_tree_bytes(nbh_ctx* ctx, const nbh_tree* t, size_t* bytes)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(bytes != nullptr, "null output");
	*bytes = tree_base_bytes(t->n) +
	         (t->two_lists != nullptr ? two_bytes(t->two_slots, t->two_cap > 0 ? t->two_cap : kTwoCap) : 0) +
	         (t->far_list != nullptr ? (t->n >> (6 + kSuperShift)) * (static_cast<size_t>(kFarCap) + 1) * sizeof(int) : 0);
	return NBH_OK;
}

nbh_status nbh_bh_band_samples(nbh_ctx* ctx, const nbh_tree* t, const uint32_t* groups, size_t n_groups,
                               float rho_min, float near_k, float* x, float* basis, float* target,
                               uint32_t* cells, size_t capacity, size_t* count)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(t->built, "tree has not been built");
	NBH_CHECK(!t->radix, "this walk runs on the heap tree only (the last build made the Morton tree)");
	NBH_CHECK(t->n >= static_cast<size_t>(kGroup), "group walk needs at least %d bodies", kGroup);
	NBH_CHECK((t->levels + 2) * (kGroup / 2) <= kWalkStack, "tree too deep for the walk stack");
	NBH_CHECK(groups != nullptr && count != nullptr, "null argument");
	NBH_CHECK(n_groups > 0 && n_groups <= (static_cast<size_t>(1) << 30), "bad group count %zu", n_groups);
	NBH_CHECK(capacity == 0 || (x != nullptr && basis != nullptr && target != nullptr), "null sample buffer");
	NBH_CHECK(capacity <= (static_cast<size_t>(1) << 31), "capacity %zu too large", capacity);
	NBH_CHECK(rho_min >= 0.0f && near_k >= 0.0f, "rho_min and near_k must be >= 0");
	const size_t ngroups_tree = t->n / kGroup;
	for(size_t i = 0; i < n_groups; ++i)
	{
		NBH_CHECK(groups[i] < ngroups_tree, "group %u out of range (%zu groups)", groups[i], ngroups_tree);
	}
	*count = 0;
	// scratch: [0, 256) counter, then the group list, then the (group, cell) pairs
	const size_t off_groups = 256;
	const size_t off_pairs = (off_groups + n_groups * sizeof(uint32_t) + 255) / 256 * 256;
	void* sp = nullptr;
	NBH_TRY(nbh::scratch(ctx, off_pairs + capacity * 2 * sizeof(uint32_t), &sp));
	char* base = static_cast<char*>(sp);
	unsigned long long* counter = reinterpret_cast<unsigned long long*>(base);
	uint32_t* dgroups = reinterpret_cast<uint32_t*>(base + off_groups);
	uint32_t* pairs = reinterpret_cast<uint32_t*>(base + off_pairs);
	NBH_HIP(hipMemcpyAsync(dgroups, groups, n_groups * sizeof(uint32_t), hipMemcpyHostToDevice, ctx->stream));
	hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, ctx->stream, counter);
	NBH_LAUNCHED();
	const int n = static_cast<int>(t->n);
	hipLaunchKernelGGL(k_band_collect, dim3(static_cast<unsigned>(n_groups)), dim3(kGroup), 0, ctx->stream, t->xyzr,
	                   t->bmin, t->bmax, n, dgroups, rho_min, near_k, pairs, static_cast<unsigned long long>(capacity),
	                   counter);
	NBH_LAUNCHED();
	unsigned long long found = 0;
	NBH_HIP(hipMemcpyAsync(&found, counter, sizeof(found), hipMemcpyDeviceToHost, ctx->stream));
	NBH_HIP(hipStreamSynchronize(ctx->stream));
	*count = static_cast<size_t>(found);
	const size_t m = std::min(static_cast<size_t>(found), capacity);
	if(m > 0)
	{
		hipLaunchKernelGGL(k_band_residual, dim3(nbh::grid_for(ctx, m, 1)), dim3(64), 0, ctx->stream, t->xyzr,
		                   t->mass, t->bmin, t->bmax, t->quad, n, t->levels, n / kGroup, 1, pairs, m, x, basis,
		                   target);
		NBH_LAUNCHED();
		if(cells != nullptr)
		{
			NBH_HIP(hipMemcpyAsync(cells, pairs, m * 2 * sizeof(uint32_t), hipMemcpyDeviceToDevice, ctx->stream));
		}
		NBH_HIP(hipStreamSynchronize(ctx->stream));
	}
	return NBH_OK;
}

nbh_status nbh_bh_fcompute_group_mlp(nbh_ctx* ctx, const nbh_tree* t, const nbh_mlp* net, const double* y,
                                     double* f, float rho_min, float near_k)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(net != nullptr && nbh::mlp_ctx(net) == ctx, "network does not belong to this context");
	NBH_CHECK(t->built, "tree has not been built");
	NBH_CHECK(!t->radix, "this walk runs on the heap tree only (the last build made the Morton tree)");
	NBH_CHECK(y != nullptr && f != nullptr && y != f, "bad buffers");
	NBH_CHECK(t->n >= static_cast<size_t>(kGroup), "group walk needs at least %d bodies", kGroup);
	NBH_CHECK((t->levels + 2) * (kGroup / 2) <= kWalkStack, "tree too deep for the walk stack");
	NBH_CHECK(rho_min >= 0.0f && near_k >= 0.0f, "rho_min and near_k must be >= 0");
	const int n = static_cast<int>(t->n);
	hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, ctx->stream, t->counters);
	NBH_LAUNCHED();
	nbh::scoped_timer timer(ctx, "bh_traverse");
	hipLaunchKernelGGL(k_bh_group32_mlp, dim3(n / kGroup), dim3(kGroup), 0, ctx->stream, t->wrec, t->bmin, t->bmax,
	                   t->body_n, y, f, n, nbh::mlp_frags(net), nbh::mlp_params(net), rho_min, near_k, t->counters);
	NBH_LAUNCHED();
	return NBH_OK;
}

nbh_status nbh_bh_walk_counters(nbh_ctx* ctx, const nbh_tree* t, uint64_t out[5])
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	NBH_CHECK(out != nullptr, "null output");
	unsigned long long c[5] = {0, 0, 0, 0, 0};
	NBH_HIP(hipMemcpyAsync(c, t->counters, sizeof(c), hipMemcpyDeviceToHost, ctx->stream));
	NBH_HIP(hipStreamSynchronize(ctx->stream));
	for(int k = 0; k < 5; ++k) { out[k] = c[k]; }
	return NBH_OK;
}

nbh_status nbh_tree_get(nbh_ctx* ctx, const nbh_tree* t, int32_t* body_n, double* cm, double* mass,
                        double* crit_r2, double* bmin, double* bmax)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	const size_t s = 2 * t->n;
	NBH_HIP(hipStreamSynchronize(ctx->stream));
	if(body_n != nullptr) { NBH_HIP(hipMemcpy(body_n, t->body_n, s * sizeof(int32_t), hipMemcpyDeviceToHost)); }
	if(mass != nullptr) { NBH_HIP(hipMemcpy(mass, t->mass, s * sizeof(double), hipMemcpyDeviceToHost)); }
	if(bmin != nullptr) { NBH_HIP(hipMemcpy(bmin, t->bmin, 3 * s * sizeof(double), hipMemcpyDeviceToHost)); }
	if(bmax != nullptr) { NBH_HIP(hipMemcpy(bmax, t->bmax, 3 * s * sizeof(double), hipMemcpyDeviceToHost)); }
	if(cm != nullptr || crit_r2 != nullptr)
	{
		std::vector<double> rec(4 * s);
		NBH_HIP(hipMemcpy(rec.data(), t->xyzr, s * sizeof(double4), hipMemcpyDeviceToHost));
		for(size_t i = 0; i < s; ++i)
		{
			if(cm != nullptr)
			{
				cm[3 * i] = rec[4 * i];
				cm[3 * i + 1] = rec[4 * i + 1];
				cm[3 * i + 2] = rec[4 * i + 2];
			}
			if(crit_r2 != nullptr) { crit_r2[i] = rec[4 * i + 3]; }
		}
	}
	return NBH_OK;
}

nbh_status nbh_bh_counters(nbh_ctx* ctx, const nbh_tree* t, uint64_t* interactions, uint64_t* visits)
{
	NBH_TRY(nbh::enter(ctx));
	NBH_CHECK(t != nullptr && t->ctx == ctx, "tree does not belong to this context");
	unsigned long long c[3] = {0, 0, 0};
	NBH_HIP(hipMemcpyAsync(c, t->counters, sizeof(c), hipMemcpyDeviceToHost, ctx->stream));
	NBH_HIP(hipStreamSynchronize(ctx->stream));
	if(interactions != nullptr) { *interactions = c[0]; }
	if(visits != nullptr) { *visits = c[1]; }
	return NBH_OK;
}

}  // extern "C"
