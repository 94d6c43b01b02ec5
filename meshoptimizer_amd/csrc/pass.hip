// Per-pass kernels of the edge-collapse simplifier (src/simplifier.cpp:2493-2541):
// welded adjacency, pick, rank, sort, the priority-round greedy commit with its prefix-scan
// stop, quadric update, edge-loop remap and index compaction.
#include "kernels.h"
#include "prims.h"
#include "quadric.h"

#include <algorithm>

namespace mhip
{

static constexpr int kThreads = 256;

static inline unsigned int grid_for(size_t n)
{
	return div_up(n ? n : 1, kThreads);
}

// kCanCollapse / kHasOpposite, src/simplifier.cpp:312-331
__constant__ uint8_t c_can_collapse[5][5] = {
    {1, 1, 1, 1, 1},
    {0, 1, 0, 0, 1},
    {0, 0, 1, 0, 1},
    {0, 0, 0, 1, 1},
    {0, 0, 0, 0, 0},
};

__constant__ uint8_t c_has_opposite[5][5] = {
    {1, 1, 1, 1, 1},
    {1, 0, 1, 0, 0},
    {1, 1, 1, 0, 1},
    {1, 0, 0, 0, 0},
    {1, 0, 1, 0, 0},
};

// ------------------------------------------------------------------------------------------
// welded corner CSR of the current index buffer (src/simplifier.cpp:52-109), from scratch: for the
// vertex solve, over the result, and after a pass that split a class.  Segment order is free: every consumer is a count or an any().
// One atomic pass counts the corners per class and hands each corner its slot in the class's
// segment; after the scan the fill places the corners without atomics.

__global__ void k_adj_count(const uint32_t* ib, size_t corners, const uint32_t* remap, uint32_t* counts, uint32_t* slot)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (j < corners)
		slot[j] = atomicAdd(&counts[remap[ib[j]]], 1u);
}

__global__ void k_adj_fill(const uint32_t* ib, size_t tris, const uint32_t* remap, const uint32_t* off, const uint32_t* slot, uint2* adj)
{
	size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= tris)
		return;
	uint32_t a = remap[ib[t * 3 + 0]], b = remap[ib[t * 3 + 1]], c = remap[ib[t * 3 + 2]];
	adj[off[a] + slot[t * 3 + 0]] = make_uint2(b, c);
	adj[off[b] + slot[t * 3 + 1]] = make_uint2(c, a);
	adj[off[c] + slot[t * 3 + 2]] = make_uint2(a, b);
}

__global__ void k_adj_ranges(const uint32_t* off, size_t n, uint2* range)
{
	size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (v < n)
		range[v] = make_uint2(off[v], off[v + 1]);
}

// the corner slots go to the space of the source lists, which a pass makes for itself
void launch_adjacency(hipStream_t s, Mesh& m, size_t tri_count)
{
	size_t n = m.vertex_count;
	fill_u32(s, m.adj_off, 0, n + 1);
	if (tri_count)
		k_adj_count<<<grid_for(tri_count * 3), kThreads, 0, s>>>(m.ib[m.ib_cur], tri_count * 3, m.remap, m.adj_off, m.src_rank);
	scan_exclusive(s, m.adj_off, m.adj_off, n, nullptr, m.adj_off + n, m.temp);
	if (tri_count)
		k_adj_fill<<<grid_for(tri_count), kThreads, 0, s>>>(m.ib[m.ib_cur], tri_count, m.remap, m.adj_off, m.src_rank, m.adj[m.adj_cur]);
}

void launch_adjacency_ranges(hipStream_t s, Mesh& m, size_t tri_count)
{
	launch_adjacency(s, m, tri_count);
	k_adj_ranges<<<grid_for(m.vertex_count), kThreads, 0, s>>>(m.adj_off, m.vertex_count, m.adj_range[m.adj_cur]);
}

// ------------------------------------------------------------------------------------------
// Blocked compaction: a count kernel leaves one sum per tile, and the workgroup that writes a tile
// adds the sums before its own and scans its items; no per-item counts or offsets go through
// memory and no scan kernels run in between.  At most kMaxTiles tiles, so that the sums before a
// tile stay a few reads per thread.

constexpr size_t kMaxTiles = 1024;

static inline uint32_t tile_items(size_t n)
{
	return div_up(n ? n : 1, (size_t)kThreads * kMaxTiles);
}

size_t compaction_tiles(size_t n)
{
	return std::min((size_t)div_up(n ? n : 1, kThreads), kMaxTiles);
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v)
{
#pragma unroll
	for (int o = 32; o > 0; o >>= 1)
		v += __shfl_xor(v, o, 64);
	return v;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
#pragma unroll
	for (int o = 32; o > 0; o >>= 1)
	{
		const uint32_t t = __shfl_xor(v, o, 64);
		v = t > v ? t : v;
	}
	return v;
}

// sums over the workgroup, in every thread; red: one word per wavefront and value
__device__ __forceinline__ uint2 block_sum2(uint2 v, uint2* red)
{
	const uint32_t x = wave_sum(v.x), y = wave_sum(v.y);
	if (__lane_id() == 0)
		red[threadIdx.x >> 6] = make_uint2(x, y);
	__syncthreads();
	uint2 t = make_uint2(0, 0);
#pragma unroll
	for (int w = 0; w < kThreads / 64; ++w)
	{
		t.x += red[w].x;
		t.y += red[w].y;
	}
	__syncthreads();
	return t;
}

__device__ __forceinline__ uint2 sums_before(const uint2* sums, uint32_t tile, uint2* red)
{
	uint2 v = make_uint2(0, 0);
	for (uint32_t b = threadIdx.x; b < tile; b += kThreads)
	{
		v.x += sums[b].x;
		v.y += sums[b].y;
	}
	return block_sum2(v, red);
}

// exclusive scan of one word per thread across the workgroup
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* red, uint32_t& total)
{
	uint32_t x = v;
	const int lane = __lane_id(), wave = threadIdx.x >> 6;
#pragma unroll
	for (int o = 1; o < 64; o <<= 1)
	{
		const uint32_t t = __shfl_up(x, o, 64);
		x += lane >= o ? t : 0u;
	}
	if (lane == 63)
		red[wave] = x;
	__syncthreads();
	uint32_t before = 0, all = 0;
#pragma unroll
	for (int w = 0; w < kThreads / 64; ++w)
	{
		before += w < wave ? red[w] : 0u;
		all += red[w];
	}
	__syncthreads();
	total = all;
	return before + x - v;
}

// ------------------------------------------------------------------------------------------
// remapIndexBuffer (src/simplifier.cpp:1811-1843) and the next pass's pickEdgeCollapses
// (1310-1372) in one sweep of two kernels: each triangle is taken through collapse_remap and kept
// when its primaries stay distinct, in order, and a kept triangle's candidates are listed in edge
// order.  kCompact false: the triangles as they are, candidates only (the first pass, and the
// triangles that Prune left).

struct TriArgs
{
	const uint32_t* in;
	uint32_t* out;
	const uint32_t* live; // device word bounding the triangle count (null: the host's)
	const uint32_t* cremap;
	const uint32_t* remap;
	const uint8_t* kind;
	const uint32_t* loop;
	const uint32_t* loopback;
	uint2* sums; // (kept triangles, candidates) per tile
	uint2* c_v;
	float* c_err;
	CallScalars* sc;
	uint32_t tris;
	uint32_t items;
};

__device__ __forceinline__ uint32_t live_tris(const TriArgs& a)
{
	if (!a.live)
		return a.tris;
	const uint32_t n = *a.live;
	return n < a.tris ? n : a.tris;
}

template <bool kCompact>
__device__ __forceinline__ bool load_triangle(const TriArgs& a, uint32_t t, uint32_t v[3], uint32_t r[3])
{
#pragma unroll
	for (int q = 0; q < 3; ++q)
	{
		const uint32_t i = a.in[(size_t)t * 3 + q];
		v[q] = kCompact ? a.cremap[i] : i;
	}
#pragma unroll
	for (int q = 0; q < 3; ++q)
		r[q] = a.remap[v[q]];
	return !kCompact || (r[0] != r[1] && r[0] != r[2] && r[1] != r[2]);
}

// the candidates of one triangle, pickEdgeCollapses (src/simplifier.cpp:1310-1372), in edge order
__device__ __forceinline__ uint32_t pick_triangle(const TriArgs& a, const uint32_t v[3], const uint32_t r[3], uint32_t v0[3], uint32_t v1[3], bool bidi[3])
{
	const uint8_t kd[3] = {a.kind[v[0]], a.kind[v[1]], a.kind[v[2]]};
	uint32_t count = 0;
#pragma unroll
	for (int e = 0; e < 3; ++e)
	{
		const int f = e == 2 ? 0 : e + 1;
		const uint32_t i0 = v[e], i1 = v[f];
		if (r[e] == r[f])
			continue;
		const uint8_t k0 = kd[e], k1 = kd[f];
		const uint8_t c01 = c_can_collapse[k0][k1], c10 = c_can_collapse[k1][k0];
		if (!(c01 | c10))
			continue;
		if (c_has_opposite[k0][k1] && r[f] > r[e])
			continue;
		if ((k0 == kBorder || k0 == kSeam) && k1 != kManifold && a.loop[i0] != i1)
			continue;
		if ((k1 == kBorder || k1 == kSeam) && k0 != kManifold && a.loopback[i1] != i0)
			continue;
		const bool both = c01 & c10, fwd = both || c01;
		// at a compile-time place, so that the arrays stay in registers
#pragma unroll
		for (uint32_t q = 0; q < 3; ++q)
			if (q == count)
			{
				v0[q] = fwd ? i0 : i1;
				v1[q] = fwd ? i1 : i0;
				bidi[q] = both;
			}
		count++;
	}
	return count;
}

template <bool kCompact>
__global__ void __launch_bounds__(kThreads) k_tri_count(TriArgs a)
{
	__shared__ uint2 red[kThreads / 64];
	if (kCompact && a.sc->extend)
		return;
	const uint32_t tris = live_tris(a), base = blockIdx.x * kThreads * a.items;
	uint2 n = make_uint2(0, 0);
	for (uint32_t j = 0; j < a.items; ++j)
	{
		const uint32_t t = base + j * kThreads + threadIdx.x;
		if (t >= tris)
			break;
		uint32_t v[3], r[3], v0[3], v1[3];
		bool bd[3];
		if (load_triangle<kCompact>(a, t, v, r))
		{
			n.x++;
			n.y += pick_triangle(a, v, r, v0, v1, bd);
		}
	}
	n = block_sum2(n, red);
	if (threadIdx.x == 0)
	{
		a.sums[blockIdx.x] = n;
		if (blockIdx.x == 0)
			a.sc->candidates = 0;
	}
}

// Candidates are taken while `written + 3 <= capacity` (src/simplifier.cpp:1318-1320): the taken
// triangles form a prefix.
template <bool kCompact>
__global__ void __launch_bounds__(kThreads) k_tri_write(TriArgs a)
{
	__shared__ uint2 red2[kThreads / 64];
	__shared__ uint32_t red[kThreads / 64];
	if (kCompact && a.sc->extend)
		return;
	const uint32_t tris = live_tris(a), base = blockIdx.x * kThreads * a.items;
	const uint64_t capacity = a.sc->pick_capacity;
	uint2 at = sums_before(a.sums, blockIdx.x, red2);
	for (uint32_t j = 0; j < a.items; ++j)
	{
		const uint32_t t = base + j * kThreads + threadIdx.x;
		uint32_t v[3], r[3], v0[3], v1[3];
		bool bd[3];
		const bool keep = t < tris && load_triangle<kCompact>(a, t, v, r);
		const uint32_t count = keep ? pick_triangle(a, v, r, v0, v1, bd) : 0;
		uint32_t total;
		const uint32_t ex = block_scan((keep ? 0x10000u : 0u) + count, red, total);
		if (keep)
		{
			if (kCompact)
			{
				uint32_t* out = a.out + (size_t)(at.x + (ex >> 16)) * 3;
				out[0] = v[0];
				out[1] = v[1];
				out[2] = v[2];
			}
			const uint32_t c = at.y + (ex & 0xffffu);
			if ((uint64_t)c + 3 <= capacity)
			{
#pragma unroll
				for (uint32_t q = 0; q < 3; ++q)
					if (q < count)
					{
						a.c_v[c + q] = make_uint2(v0[q], v1[q]);
						a.c_err[c + q] = __uint_as_float(bd[q] ? 1u : 0u); // the two-way flag until ranked
					}
				// the taken triangle after which the next does not fit ends the list
				if ((uint64_t)c + count + 3 > capacity)
					a.sc->candidates = c + count;
			}
		}
		at.x += total >> 16;
		at.y += total & 0xffffu;
	}
	if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0)
	{
		if (kCompact)
			a.sc->next_triangles = at.x;
		if ((uint64_t)at.y + 3 <= capacity)
			a.sc->candidates = at.y;
	}
}

static TriArgs tri_args(Mesh& m, size_t tri_count, const uint32_t* live, int loop_set)
{
	TriArgs a;
	a.in = m.ib[m.ib_cur];
	a.out = m.ib[m.ib_cur ^ 1];
	a.live = live;
	a.cremap = m.cremap;
	a.remap = m.remap;
	a.kind = m.kind;
	a.loop = m.loop[loop_set];
	a.loopback = m.loopback[loop_set];
	a.sums = m.tri_sums;
	a.c_v = m.c_v;
	a.c_err = m.c_err;
	a.sc = m.sc;
	a.tris = (uint32_t)tri_count;
	a.items = tile_items(tri_count);
	return a;
}

void launch_pick(hipStream_t s, Mesh& m, size_t tri_count, const uint32_t* live)
{
	const TriArgs a = tri_args(m, tri_count, live, m.loop_cur);
	const unsigned int tiles = div_up(tri_count ? tri_count : 1, (size_t)kThreads * a.items);
	k_tri_count<false><<<tiles, kThreads, 0, s>>>(a);
	k_tri_write<false><<<tiles, kThreads, 0, s>>>(a);
}

// ------------------------------------------------------------------------------------------
// rankEdgeCollapses, src/simplifier.cpp:1374-1450, and sortEdgeCollapses, 1452-1496

__device__ __forceinline__ uint32_t complex_target(uint32_t v, uint32_t target, const uint32_t* remap, const uint32_t* loop, const uint32_t* loopback)
{
	// getComplexTarget, src/simplifier.cpp:1278-1290
	uint32_t r = remap[target];
	uint32_t l = loop[v];
	if (l != kNone && remap[l] == r)
		return l;
	uint32_t lb = loopback[v];
	if (lb != kNone && remap[lb] == r)
		return lb;
	return target;
}

struct RankArgs
{
	const float4* pos;
	const float* va;
	const Quad* vq;
	const Quad* aq;
	const Grad* ag;
	int attr_count;
	const uint32_t* remap;
	const uint32_t* wedge;
	const uint8_t* kind;
	const uint32_t* loop;
	const uint32_t* loopback;
};

__device__ __forceinline__ float attr_error(const RankArgs& a, uint32_t v, uint32_t t)
{
	const int A = a.attr_count;
	return quad_error_attr(load_quad(a.aq, v), a.ag + (size_t)v * A, A, load_pos(a.pos, t), a.va + (size_t)t * A);
}

// the error of candidate i0 -> i1, and of i1 -> i0 when the edge collapses both ways (else FLT_MAX)
__device__ __forceinline__ float2 rank_errors(const RankArgs& a, uint32_t i0, uint32_t i1, bool bidi)
{
	float ei = quad_error(load_quad(a.vq, a.remap[i0]), load_pos(a.pos, i1));
	float ej = bidi ? quad_error(load_quad(a.vq, a.remap[i1]), load_pos(a.pos, i0)) : FLT_MAX;

	if (a.attr_count)
	{
		ei += attr_error(a, i0, i1);
		ej += bidi ? attr_error(a, i1, i0) : 0;

		uint8_t k0 = a.kind[i0];
		if (k0 == kSeam)
		{
			uint32_t s0 = a.wedge[i0];
			uint32_t s1 = a.loop[i0] == i1 ? a.loopback[s0] : a.loop[s0];
			s1 = (s1 != kNone) ? s1 : a.wedge[i1];

			ei += attr_error(a, s0, s1);
			ej += bidi ? attr_error(a, s1, s0) : 0;
		}
		else
		{
			if (k0 == kComplex)
				for (uint32_t v = a.wedge[i0]; v != i0; v = a.wedge[v])
					ei += attr_error(a, v, complex_target(v, i1, a.remap, a.loop, a.loopback));

			if (a.kind[i1] == kComplex && bidi)
				for (uint32_t v = a.wedge[i1]; v != i1; v = a.wedge[v])
					ej += attr_error(a, v, complex_target(v, i0, a.remap, a.loop, a.loopback));
		}
	}
	return make_float2(ei, ej);
}

// The sort by the 12-bit key is one stable counting pass over the key's 2560 values: the rank kernel
// counts each tile of candidates in LDS, the scan of the (value, tile) counts gives every tile its
// place in every value's run, and the scatter writes the ranked copies there directly.  Its
// wavefronts own consecutive parts of the tile with a count of their own per value, so nothing
// waits between 64 candidates and the next.  Icosphere L8's first pass, 2 M candidates: 93 us after
// the rank, where two 8-bit digits with their scans and a gather of the ranked copies took 150 in
// nine launches.
constexpr int kKeyValues = 2560;
constexpr int kRankThreads = 1024;
constexpr int kScatterThreads = 512;
constexpr int kScatterWaves = kScatterThreads / 64;

// tiles large enough that the counts stay well below the candidates, small enough to fill the chip
static uint32_t rank_tile(size_t cand_count)
{
	return cand_count <= 65536 ? 1024u : (cand_count <= 524288 ? 2048u : (cand_count <= 2097152 ? 4096u : 8192u));
}

// words of the counts for up to cand_count candidates (the largest of the steps of rank_tile below)
size_t rank_sort_words(size_t cand_count)
{
	size_t tiles = div_up(cand_count ? cand_count : 1, rank_tile(cand_count));
	for (size_t step : {(size_t)65536, (size_t)524288, (size_t)2097152})
		if (cand_count > step)
			tiles = std::max(tiles, (size_t)div_up(step, rank_tile(step)));
	return tiles * kKeyValues;
}

// one candidate's error and orientation
__device__ __forceinline__ float rank_one(const RankArgs& a, uint2* c_v, float* c_err, uint32_t c)
{
	const uint2 v = c_v[c];
	const bool bidi = __float_as_uint(c_err[c]) != 0;
	const float2 e = rank_errors(a, v.x, v.y, bidi);
	const bool rev = bidi & (e.y < e.x);
	const float err = e.y < e.x ? e.y : e.x;
	if (rev)
		c_v[c] = make_uint2(v.y, v.x);
	c_err[c] = err;
	return err;
}

// the commit state of the pass (collapse_remap, locks, list counters), set up beside the ranking
struct CommitInit
{
	uint32_t* cremap;
	uint32_t* lock_rank;
	uint32_t vertices;
	CallScalars* sc;
};

__device__ __forceinline__ void commit_init(const CommitInit& i)
{
	if (blockIdx.x == 0 && threadIdx.x < kListSegments)
	{
		CallScalars* sc = i.sc;
		sc->list_count[0][threadIdx.x] = 0;
		sc->list_count[1][threadIdx.x] = 0;
		sc->list_count[2][threadIdx.x] = 0;
		sc->window_count[threadIdx.x] = 0;
		if (threadIdx.x == 0)
		{
			sc->tail_rounds = 0;
			sc->round = 0;
		}
	}
	for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < i.vertices; v += gridDim.x * blockDim.x)
	{
		i.cremap[v] = v;
		i.lock_rank[v] = kNone;
	}
}

// Short lists: ranking and counting in one launch, a thread per candidate of the tile.  Longer ones
// rank with a thread per candidate in small workgroups first (the gathers want the whole chip in
// flight: 3.1 M candidates with attributes took 300 us from 383 workgroups of 1024 threads, 190 so).
template <bool kRank>
__global__ void __launch_bounds__(kRankThreads) k_rank_count(RankArgs a, CommitInit init, uint32_t count, uint32_t tile, uint2* c_v, float* c_err,
                                                             uint32_t* counts)
{
	__shared__ uint32_t hist[kKeyValues];
	for (uint32_t d = threadIdx.x; d < kKeyValues; d += kRankThreads)
		hist[d] = 0;
	if (kRank)
		commit_init(init);
	__syncthreads();
	const uint32_t begin = blockIdx.x * tile, end = count - begin < tile ? count : begin + tile;
	for (uint32_t c = begin + threadIdx.x; c < end; c += kRankThreads)
		atomicAdd(&hist[collapse_sort_key(kRank ? rank_one(a, c_v, c_err, c) : c_err[c])], 1u);
	__syncthreads();
	for (uint32_t d = threadIdx.x; d < kKeyValues; d += kRankThreads)
		counts[(size_t)d * gridDim.x + blockIdx.x] = hist[d];
}

__global__ void __launch_bounds__(kThreads) k_rank(RankArgs a, CommitInit init, uint32_t count, uint2* c_v, float* c_err)
{
	commit_init(init);
	const uint32_t c = blockIdx.x * kThreads + threadIdx.x;
	if (c < count)
		rank_one(a, c_v, c_err, c);
}

// list segment of a source class (see RoundState)
__device__ __forceinline__ uint32_t list_segment(uint64_t seg_mul, uint32_t c)
{
	return (uint32_t)(((uint64_t)c * seg_mul) >> 32);
}

__global__ void __launch_bounds__(kScatterThreads) k_rank_scatter(const uint2* c_v, const float* c_err, const uint32_t* remap, uint32_t count, uint32_t tile,
                                                                  const uint32_t* places, uint2* r_v, uint2* r_class, float* r_err, uint8_t* status,
                                                                  uint32_t window, uint64_t seg_mul, CallScalars* sc)
{
	__shared__ uint32_t before[kScatterWaves][kKeyValues / 2]; // two 16-bit counts a word
	__shared__ uint32_t place[kKeyValues];
	__shared__ uint32_t seg[kListSegments];
	const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6;
	for (uint32_t d = threadIdx.x; d < kScatterWaves * kKeyValues / 2; d += kScatterThreads)
		(&before[0][0])[d] = 0;
	for (uint32_t d = threadIdx.x; d < kKeyValues; d += kScatterThreads)
		place[d] = places[(size_t)d * gridDim.x + blockIdx.x];
	if (threadIdx.x < kListSegments)
		seg[threadIdx.x] = 0;
	__syncthreads();
	const uint32_t part = tile / kScatterWaves, first = blockIdx.x * tile + wave * part;
	const uint32_t end = first < count ? (count - first < part ? count : first + part) : first;
	uint32_t* mine = before[wave];
	for (uint32_t c = first + lane; c < end; c += 64)
	{
		const uint32_t key = collapse_sort_key(c_err[c]);
		atomicAdd(&mine[key >> 1], key & 1 ? 0x10000u : 1u);
	}
	__syncthreads();
	// each wavefront's counts become the sums of those before it
	for (uint32_t d = threadIdx.x; d < kKeyValues / 2; d += kScatterThreads)
	{
		uint32_t run = 0;
#pragma unroll
		for (int w = 0; w < kScatterWaves; ++w)
		{
			const uint32_t n = before[w][d];
			before[w][d] = run;
			run += n;
		}
	}
	__syncthreads();
	uint32_t in_segment = 0; // lane q: this wavefront's ranks in the window and segment q
	for (uint32_t c0 = first; c0 < end; c0 += 64)
	{
		const uint32_t c = c0 + lane;
		const bool valid = c < end;
		const float err = valid ? c_err[c] : 0.f;
		const uint2 v = valid ? c_v[c] : make_uint2(0, 0);
		const uint32_t key = collapse_sort_key(err), shift = key & 1 ? 16u : 0u;
		const uint2 cls = valid ? make_uint2(remap[v.x], remap[v.y]) : make_uint2(0, 0);
		uint64_t peers = __ballot(valid);
#pragma unroll
		for (int b = 0; b < 12; ++b)
		{
			const uint64_t set = __ballot((key >> b) & 1u);
			peers &= ((key >> b) & 1u) ? set : ~set;
		}
		const uint32_t ahead = (uint32_t)__popcll(peers & ((1ull << lane) - 1ull));
		const uint32_t rank = place[key] + ((mine[key >> 1] >> shift) & 0xffffu) + ahead;
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
		if (valid && ahead == 0)
			atomicAdd(&mine[key >> 1], (uint32_t)__popcll(peers) << shift);
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
		if (valid)
		{
			r_v[rank] = v;
			r_class[rank] = cls;
			r_err[rank] = err;
			status[c] = kUndecided;
		}
		const uint32_t q = valid && rank < window ? list_segment(seg_mul, cls.x) : kNone;
#pragma unroll
		for (uint32_t k = 0; k < kListSegments; ++k)
		{
			const uint64_t m = __ballot(q == k);
			in_segment += lane == k ? (uint32_t)__popcll(m) : 0u;
		}
	}
	if (lane < kListSegments && in_segment)
		atomicAdd(&seg[lane], in_segment);
	__syncthreads();
	if (threadIdx.x < kListSegments && seg[threadIdx.x])
		atomicAdd(&sc->window_count[threadIdx.x], seg[threadIdx.x]);
}

static uint64_t segment_mul(const Mesh& m)
{
	return m.vertex_count ? ((uint64_t)kListSegments << 32) / m.vertex_count : 0;
}

void launch_rank_sort(hipStream_t s, Mesh& m, size_t cand_count, size_t window)
{
	RankArgs a;
	a.pos = m.pos;
	a.va = m.va;
	a.vq = m.vq;
	a.aq = m.aq;
	a.ag = m.ag;
	a.attr_count = (int)m.attr_count;
	a.remap = m.remap;
	a.wedge = m.wedge;
	a.kind = m.kind;
	a.loop = m.loop[m.loop_cur];
	a.loopback = m.loopback[m.loop_cur];
	const uint32_t tile = rank_tile(cand_count), n = (uint32_t)cand_count;
	const unsigned int tiles = div_up(cand_count, tile);
	const CommitInit init{m.cremap, m.lock_rank, m.vertex_count, m.sc};
	if (tile == kRankThreads)
		k_rank_count<true><<<tiles, kRankThreads, 0, s>>>(a, init, n, tile, m.c_v, m.c_err, m.rank_counts);
	else
	{
		k_rank<<<grid_for(cand_count), kThreads, 0, s>>>(a, init, n, m.c_v, m.c_err);
		k_rank_count<false><<<tiles, kRankThreads, 0, s>>>(a, init, n, tile, m.c_v, m.c_err, m.rank_counts);
	}
	scan_exclusive(s, m.rank_counts, m.rank_counts, (size_t)kKeyValues * tiles, nullptr, nullptr, m.temp);
	k_rank_scatter<<<tiles, kScatterThreads, 0, s>>>(m.c_v, m.c_err, m.remap, n, tile, m.rank_counts, m.r_v, m.r_class, m.r_err, m.status,
	                                                (uint32_t)window, segment_mul(m), m.sc);
}

// ------------------------------------------------------------------------------------------
// performEdgeCollapses (src/simplifier.cpp:1498-1636) as priority rounds.
//
// Rank k's decision depends only on lower ranks j that share an endpoint class (the lock
// test) or whose source class is a welded neighbour of k's source class (the flip test reads
// collapse_remap only there; only sources are written, and the neighbour relation is
// symmetric).  Round e: an undecided rank whose endpoints are locked is skipped (a lock can
// only come from a lower commit); one that was the minimum published at both endpoints in
// round e-1 and is below every source-role entry of e-1 in its neighbourhood decides now
// (flip-rejected or committed); the rest publish their rank for round e as 64-bit minima
// tagged with ~e in the high word, into the buffer of parity e, and stay on the work list.  A
// class keeps one minimum per role (source, target), so a rank publishes with two atomics, and
// the minimum over both roles is the smaller of the pair.
// Ranks that decide in one round never touch each other's state.

enum : uint8_t
{
	kFlipPass = 4,        // flip test passes, now and for good; commits once lowest at its endpoints
	kFlipFail = 5,        // flip test fails for good; resolved as skipped or rejected at the end
	kCommittedBorder = 6, // committed, the source a border vertex (one triangle, not two)
};

__device__ __forceinline__ bool is_commit(uint8_t st)
{
	return st == kCommitted || st == kCommittedBorder;
}

__device__ __forceinline__ uint64_t round_key(uint32_t epoch, uint32_t k)
{
	return ((uint64_t)(~epoch) << 32) | k;
}

// commit writes of one collapse, src/simplifier.cpp:1573-1611; returns the status that records it
__device__ __forceinline__ uint8_t commit_collapse(uint32_t* cremap, uint32_t i0, uint32_t i1, const uint8_t* kind, const uint32_t* wedge,
                                                const uint32_t* remap, const uint32_t* loop, const uint32_t* loopback)
{
	uint8_t k = kind[i0];
	if (k == kComplex)
	{
		uint32_t v = i0;
		do
		{
			cremap[v] = complex_target(v, i1, remap, loop, loopback);
			v = wedge[v];
		} while (v != i0);
	}
	else if (k == kSeam)
	{
		uint32_t s0 = wedge[i0];
		uint32_t s1 = loop[i0] == i1 ? loopback[s0] : loop[s0];
		s1 = (s1 != kNone) ? s1 : wedge[i1];
		cremap[i0] = i1;
		cremap[s0] = s1;
	}
	else
		cremap[i0] = i1;
	return k == kBorder ? kCommittedBorder : kCommitted;
}

struct RoundState
{
	const uint2* r_v;
	const uint2* adj_range; // a class's entries of adj: (begin, end)
	const uint2* adj;
	const float4* pos;
	const uint8_t* kind;
	const uint32_t* wedge;
	const uint32_t* remap;
	const uint32_t* loop;
	const uint32_t* loopback;
	const uint32_t* src_off;  // candidate ranks grouped by source class
	const uint32_t* src_rank;
	const uint32_t* src_val;  // what each such candidate's commit writes at the class primary
	uint32_t* cremap;
	uint32_t* lock_rank;      // rank of the commit that locked a class (kNone: unlocked)
	uint8_t* status;
	uint64_t* pend[2];        // per class, the minimum rank published in a round (tagged with ~round)
	                          // over ranks whose source is the class (entry 2c) and over ranks
	                          // whose target is the class (entry 2c + 1); the minimum over both
	                          // roles is the smaller of the two
	uint4* list[2];           // work-list entries: (rank, source class, target class, 0)
	CallScalars* sc;
	uint64_t seg_mul;         // list segment of class c: (c * seg_mul) >> 32, below kListSegments.
	                          // Classes are numbered close to their neighbours in most meshes (grids,
	                          // subdivided and locality-optimised meshes), so a segment's ranks touch
	                          // mostly one range of the class arrays
};

// the value rank r's commit writes into collapse_remap[p], p the primary of its source class
// (src/simplifier.cpp:1573-1605)
__device__ __forceinline__ uint32_t commit_value_at(const RoundState& a, uint32_t r, uint32_t p)
{
	const uint32_t i0 = a.r_v[r].x, i1 = a.r_v[r].y;
	uint8_t kd = a.kind[i0];
	if (kd == kComplex)
		return complex_target(p, i1, a.remap, a.loop, a.loopback);
	if (kd == kSeam)
	{
		uint32_t s0 = a.wedge[i0];
		uint32_t s1 = a.loop[i0] == i1 ? a.loopback[s0] : a.loop[s0];
		s1 = (s1 != kNone) ? s1 : a.wedge[i1];
		uint32_t v = p;
		if (i0 == p)
			v = i1;
		if (s0 == p)
			v = s1;
		return v;
	}
	return i1;
}

// flip test (src/simplifier.cpp:1200-1232) of rank k over every way the lower candidates still in
// play could move its neighbours: 0 undetermined, 1 passes in all, 2 fails in all.  The test
// reads collapse_remap at the corners of the triangles around k's source; a corner whose class
// published a lower source-role rank in the previous round may still move (every pending rank
// publishes every round), every other corner keeps the value k sees now.  A moving corner's
// alternatives are the value seen and the values its lower candidates' commits write, taken from
// the per-source candidate lists; a candidate counts unless it is known never to commit (skipped,
// flip-failed, rejected), so the set is never smaller than the true one, whatever stores of the
// same round the test sees.  An outcome that holds in every combination is final; a triangle
// without a moving corner decides alone.  Limited to kMaxAlternatives per corner; beyond that the
// rank waits.
//
// The test is a chain of dependent gathers.  The deep test has kDeepLanes lanes for a rank, one for
// each adjacency entry, so that the entries' chains run side by side: its rounds have few ranks
// (tens of thousands falling to hundreds) and are bound by the length of the chain.  One thread
// going through the entries one after the other took 42 us a round on the 998 x 998 grid
// whatever the list's length; the lanes take 42 at 50 thousand ranks, 25 at 15 thousand and 12 below
// 4 thousand, and the call went from 17.3 to 10.9 ms.  The cheap test, whose first rounds have
// hundreds of thousands of ranks, keeps a thread for a rank and reads the adjacency
// kCheapFlipChunk entries at a time, the gathers of each level issued before any is used.

constexpr int kDeepLanes = 8;
constexpr int kCheapFlipChunk = 4;
constexpr int kCheapWaves = 5;     // waves per SIMD the cheap round kernel is built for
constexpr int kSrcChunk = 8;       // ranks of a source list read at a time
constexpr int kMaxAlternatives = 2; // per corner: its current value and one possible move

// collapse_remap of a class as rank k sees it: a move committed by a higher rank (possible once flip
// tests are decided early) reads as "not moved"
__device__ __forceinline__ uint32_t seen_by(uint32_t k, uint32_t cls, uint32_t moved, uint32_t lock_rank)
{
	return moved != cls && lock_rank > k ? cls : moved;
}

// one adjacency entry with moving corners (pend2: bit h set when corner h moves; tb, te: the corners'
// source lists): 0 mixed or too many alternatives, 1 passes in all combinations, 2 fails in all
__device__ int flip_entry_pending(const RoundState& a, uint32_t k, const uint32_t nb[2], const uint32_t seen[2], uint32_t pend2, uint32_t tb[2],
                                  uint32_t te[2], const V3& v0, const V3& v1, uint32_t i1)
{
	uint32_t alt[2][kMaxAlternatives];
	int na[2] = {1, 1};
	alt[0][0] = seen[0];
	alt[1][0] = seen[1];
#pragma unroll
	for (int q = 0; q < 2; ++q)
		te[q] = (pend2 >> q) & 1u ? te[q] : tb[q];
	bool more = true;
	for (uint32_t step = 0; more; step += kSrcChunk)
	{
		more = false;
		uint32_t r[2][kSrcChunk], val[2][kSrcChunk];
#pragma unroll
		for (int q = 0; q < 2; ++q)
#pragma unroll
			for (int u = 0; u < kSrcChunk; ++u)
			{
				const uint32_t t = tb[q] + step + u;
				const bool in = t < te[q];
				r[q][u] = in ? a.src_rank[t] : kNone;
				val[q][u] = in ? a.src_val[t] : 0;
			}
		uint8_t st[2][kSrcChunk];
#pragma unroll
		for (int q = 0; q < 2; ++q)
#pragma unroll
			for (int u = 0; u < kSrcChunk; ++u)
				st[q][u] = r[q][u] < k ? a.status[r[q][u]] : (uint8_t)kSkipped;
#pragma unroll
		for (int q = 0; q < 2; ++q)
		{
#pragma unroll
			for (int u = 0; u < kSrcChunk; ++u)
			{
				if (st[q][u] == kSkipped || st[q][u] == kRejected || st[q][u] == kFlipFail || val[q][u] == alt[q][0])
					continue;
				if (na[q] == kMaxAlternatives)
					return 0;
				alt[q][na[q]++] = val[q][u];
			}
			more |= tb[q] + step + kSrcChunk < te[q];
		}
	}
	bool any_flip = false, any_ok = false;
	for (int x = 0; x < na[0]; ++x)
		for (int y = 0; y < na[1]; ++y)
		{
			if (nb[0] == nb[1] && x != y)
				continue; // one vertex moves one way only
			uint32_t va = alt[0][x], vb = alt[1][y];
			if (va == i1 || vb == i1 || va == vb)
				any_ok = true;
			else if (triangle_flips(load_pos(a.pos, va), load_pos(a.pos, vb), v0, v1))
				any_flip = true;
			else
				any_ok = true;
		}
	return any_flip ? (any_ok ? 0 : 2) : 1;
}

// begin/end: rank k's source's adjacency range; v0, v1: the positions of its source and target.
// The cheap test: a rank with a moving corner waits (in the first rounds of a window most corners
// move), unless a triangle without one fails
__device__ __forceinline__ int flip_outcome_cheap(const RoundState& a, uint32_t i1, uint32_t k, uint32_t epoch, uint32_t begin, uint32_t end, const V3& v0,
                                                  const V3& v1)
{
	constexpr int kChunk = kCheapFlipChunk;
	const uint64_t* prev_pend = a.pend[(epoch - 1) & 1];
	const uint32_t prev_tag = ~(epoch - 1);
	bool all_pass = true;
	for (uint32_t p0 = begin; p0 < end; p0 += kChunk)
	{
		const uint32_t n = end - p0 < (uint32_t)kChunk ? end - p0 : (uint32_t)kChunk;
		uint32_t nb[2 * kChunk];
#pragma unroll
		for (int j = 0; j < kChunk; ++j)
		{
			const uint2 e = (uint32_t)j < n ? a.adj[p0 + j] : make_uint2(i1, i1);
			nb[2 * j] = e.x;
			nb[2 * j + 1] = e.y;
		}
		uint32_t cm[2 * kChunk], lr[2 * kChunk];
		uint64_t ps[2 * kChunk];
#pragma unroll
		for (int q = 0; q < 2 * kChunk; ++q)
		{
			cm[q] = a.cremap[nb[q]];
			lr[q] = a.lock_rank[nb[q]];
			ps[q] = prev_pend[2 * nb[q]];
		}
		uint32_t seen[2 * kChunk];
		uint32_t pend_mask = 0;
#pragma unroll
		for (int q = 0; q < 2 * kChunk; ++q)
		{
			seen[q] = seen_by(k, nb[q], cm[q], lr[q]);
			const bool moving = (uint32_t)(q / 2) < n && (uint32_t)(ps[q] >> 32) == prev_tag && (uint32_t)ps[q] < k;
			pend_mask |= moving ? 1u << q : 0u;
		}
		// entries without a moving corner have one scenario: the positions they need, all at once
		V3 pa[kChunk], pb[kChunk];
		uint32_t test_mask = 0;
#pragma unroll
		for (int j = 0; j < kChunk; ++j)
		{
			const uint32_t va = seen[2 * j], vb = seen[2 * j + 1];
			const bool single = (uint32_t)j < n && !((pend_mask >> (2 * j)) & 3u);
			const bool test = single && !(va == i1 || vb == i1 || va == vb);
			test_mask |= test ? 1u << j : 0u;
			pa[j] = test ? load_pos(a.pos, va) : V3{0.f, 0.f, 0.f};
			pb[j] = test ? load_pos(a.pos, vb) : V3{0.f, 0.f, 0.f};
		}
#pragma unroll
		for (int j = 0; j < kChunk; ++j)
			if (((test_mask >> j) & 1u) && triangle_flips(pa[j], pb[j], v0, v1))
				return 2;
		all_pass &= pend_mask == 0;
	}
	return all_pass ? 1 : 0;
}

// whether any lane of this lane's kDeepLanes has the bit set in a wavefront's mask
__device__ __forceinline__ bool any_of_group(uint64_t mask)
{
	return (mask >> (__lane_id() & ~(kDeepLanes - 1)) & ((1u << kDeepLanes) - 1)) != 0;
}

// the deep test, called by the rank's kDeepLanes lanes together: each takes an entry and every
// combination of its moving corners' alternatives.  What an entry may need is gathered with its
// state: the unmoved corners' positions and the bounds of their source lists
__device__ __forceinline__ int flip_outcome_deep(const RoundState& a, uint32_t i1, uint32_t k, uint32_t epoch, uint32_t begin, uint32_t end, const V3& v0,
                                                 const V3& v1)
{
	const uint64_t* prev_pend = a.pend[(epoch - 1) & 1];
	const uint32_t prev_tag = ~(epoch - 1);
	bool all_pass = true;
	for (uint32_t p0 = begin; p0 < end; p0 += kDeepLanes)
	{
		const uint32_t p = p0 + (__lane_id() & (kDeepLanes - 1));
		int outcome = 1;
		if (p < end)
		{
			const uint2 e = a.adj[p];
			const uint32_t nb[2] = {e.x, e.y};
			uint32_t cm[2], lr[2], tb[2], te[2], seen[2], pend2 = 0;
			uint64_t ps[2];
			V3 at[2];
#pragma unroll
			for (int q = 0; q < 2; ++q)
			{
				cm[q] = a.cremap[nb[q]];
				lr[q] = a.lock_rank[nb[q]];
				ps[q] = prev_pend[2 * (size_t)nb[q]];
				at[q] = load_pos(a.pos, nb[q]);
				tb[q] = a.src_off[nb[q]];
				te[q] = a.src_off[nb[q] + 1];
			}
#pragma unroll
			for (int q = 0; q < 2; ++q)
			{
				seen[q] = seen_by(k, nb[q], cm[q], lr[q]);
				pend2 |= (uint32_t)(ps[q] >> 32) == prev_tag && (uint32_t)ps[q] < k ? 1u << q : 0u;
			}
			if (pend2)
				outcome = flip_entry_pending(a, k, nb, seen, pend2, tb, te, v0, v1, i1);
			else if (seen[0] != i1 && seen[1] != i1 && seen[0] != seen[1])
			{
#pragma unroll
				for (int q = 0; q < 2; ++q)
					if (seen[q] != nb[q])
						at[q] = load_pos(a.pos, seen[q]);
				outcome = triangle_flips(at[0], at[1], v0, v1) ? 2 : 1;
			}
		}
		if (any_of_group(__ballot(outcome == 2)))
			return 2;
		all_pass &= !any_of_group(__ballot(outcome == 0));
	}
	return all_pass ? 1 : 0;
}

// round `epoch`, one rank.  A rank at a locked endpoint is skipped.  A rank that was the lowest
// published at one of its endpoints in the previous round gets its flip test; one that was the
// lowest at both and whose flip test has passed commits now (the commit phase of the previous
// round: no lower rank is left at its endpoints, and ranks committing in one round share no
// endpoint and no neighbourhood in which one of them is still pending for the other, so they
// never touch each other's state).  The rest publish their rank at both endpoint classes and
// stay on the list (true).  Every gather the decision may need is issued before the first is
// used.
//
// Commits run concurrently with the other ranks' tests of the same round.  A rank's flip test
// only trusts corners without a lower source published in the previous round, and every rank
// that commits in this round published its source then, so no test reads a move still in
// flight.  A lock written in this round may be missed by a rank sharing that endpoint: that rank
// publishes once more and is skipped in the next round, before it can commit.
//
// kDeep: the whole wavefront calls, and its ranks that need the test get it eight at a time.
template <bool kDeep>
__device__ __forceinline__ bool round_x(const RoundState& a, uint4 w, bool valid, uint32_t epoch)
{
	const uint32_t k = w.x, r0 = w.y, r1 = w.z;
	const ulonglong2* prev = reinterpret_cast<const ulonglong2*>(a.pend[(epoch - 1) & 1]);
	if (!kDeep && !valid)
		return false;
	// (a lane without a rank reads the entries of rank and class 0)
	const uint8_t st = a.status[k];
	const uint32_t l0 = a.lock_rank[r0], l1 = a.lock_rank[r1];
	const ulonglong2 q0 = prev[r0], q1 = prev[r1];
	const uint64_t p0 = q0.x < q0.y ? q0.x : q0.y, p1 = q1.x < q1.y ? q1.x : q1.y;
	const uint2 range = a.adj_range[r0];
	const V3 v0 = load_pos(a.pos, r0), v1 = load_pos(a.pos, r1);
	bool live = valid && (st == kUndecided || st == kFlipPass);
	if (!kDeep && !live)
		return false;
	if (live && (l0 != kNone || l1 != kNone))
	{
		a.status[k] = kSkipped;
		live = false;
	}
	if (!kDeep && !live)
		return false;
	// the flip test is only worth evaluating for a rank that was the lowest published at one of
	// its endpoints in the previous round (others cannot commit yet)
	const uint64_t was = round_key(epoch - 1, k);
	const bool low0 = p0 == was, low1 = p1 == was;
	const bool test = live && st == kUndecided && (low0 || low1);
	int o = 0;
	if (kDeep)
	{
		const uint32_t lane = __lane_id();
		const uint64_t below = (1ull << lane) - 1ull;
		for (uint64_t todo = __ballot(test); todo;)
		{
			// the next eight of them, one to each kDeepLanes lanes
			uint64_t left = todo, mine = 0;
#pragma unroll
			for (uint32_t g = 0; g < 64 / kDeepLanes; ++g)
			{
				mine = lane / kDeepLanes == g ? left : mine;
				left &= left - 1;
			}
			const int src = mine ? __ffsll((long long)mine) - 1 : 0;
			const uint32_t tk = __shfl(k, src, 64), t1 = __shfl(r1, src, 64), begin = __shfl(range.x, src, 64), end = __shfl(range.y, src, 64);
			const V3 t_v0 = {__shfl(v0.x, src, 64), __shfl(v0.y, src, 64), __shfl(v0.z, src, 64)};
			const V3 t_v1 = {__shfl(v1.x, src, 64), __shfl(v1.y, src, 64), __shfl(v1.z, src, 64)};
			const int outcome = mine ? flip_outcome_deep(a, t1, tk, epoch, begin, end, t_v0, t_v1) : 0;
			const uint32_t place = (uint32_t)__popcll(todo & below);
			const int got = __shfl(outcome, (int)(place * kDeepLanes) & 63, 64);
			if ((todo >> lane & 1) && place < 64 / kDeepLanes)
				o = got;
			todo = left;
		}
	}
	else if (test)
		o = flip_outcome_cheap(a, r1, k, epoch, range.x, range.y, v0, v1);
	if (!live)
		return false;
	if (o == 2)
	{
		a.status[k] = kFlipFail;
		return false;
	}
	const uint8_t now = o == 1 ? (uint8_t)kFlipPass : st;
	if (now == kFlipPass && low0 && low1)
	{
		const uint2 v = a.r_v[k];
		a.status[k] = commit_collapse(a.cremap, v.x, v.y, a.kind, a.wedge, a.remap, a.loop, a.loopback);
		a.lock_rank[r0] = k;
		a.lock_rank[r1] = k;
		return false;
	}
	if (now != st)
		a.status[k] = now;
	// two atomics: the source-role minimum at r0 and the target-role one at r1
	uint64_t key = round_key(epoch, k);
	unsigned long long* wr = (unsigned long long*)a.pend[epoch & 1];
	atomicMin(&wr[2 * (size_t)r0], (unsigned long long)key);
	atomicMin(&wr[2 * (size_t)r1 + 1], (unsigned long long)key);
	return true;
}

__device__ __forceinline__ void append_wave(bool keep, uint4 w, uint4* out_list, uint32_t* out_count)
{
	const int lane = __lane_id();
	uint64_t mask = __ballot(keep);
	if (mask)
	{
		uint32_t slot0 = 0;
		int leader = __ffsll((long long)mask) - 1;
		if (lane == leader)
			slot0 = atomicAdd(out_count, (uint32_t)__popcll(mask));
		slot0 = __shfl(slot0, leader, 64);
		if (keep)
			out_list[slot0 + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = w;
	}
}

// wavefronts of the deep round kernel that one XCD's 32 CUs hold at once (4 to each SIMD)
constexpr uint32_t kDeepSegmentWaves = 32 * 4 * 4;

// ranks a wavefront takes of n in a deep round: as few as `waves` of them get through at once
__device__ __forceinline__ uint32_t deep_ranks(uint32_t n, uint32_t waves)
{
	uint32_t ranks = 64 / kDeepLanes;
	while (ranks < 64 && n > ranks * waves)
		ranks *= 2;
	return ranks;
}

// head round.  Round r reads list (r & 1) / counters (r % 3), appends the survivors to list
// ((r + 1) & 1) / counters ((r + 1) % 3) and clears counters ((r + 2) % 3).  A rank stays in its
// segment, at the segment's offset in both lists.  Workgroups are dealt to the XCDs in turn, so
// workgroup i works on segment i mod kListSegments: each XCD's L2 then holds the class state of
// one segment's ranks rather than of all of them.  The grid is a multiple of kListSegments; one
// rank per thread when it is large enough, and the grid-stride loop covers any segment length.
// kDeep: this round examines the alternatives of moving corners (the window's per-source lists
// are built); a wavefront takes as few ranks as keep the list within the wavefronts that are
// resident at once, so that few of its ranks' tests come one after the other.  Two kernels rather
// than a flag, so that the cheap rounds are not held to the deep test's register count.
template <bool kDeep>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kDeep ? 4 : kCheapWaves))) k_round_x(RoundState a, uint32_t head_index, uint32_t rel)
{
	CallScalars* sc = a.sc;
	// rounds are numbered from a base on the device (the tail leaves it past its last round), so
	// rounds can follow a tail without a read-back; `rel` counts
	// the head rounds launched since the base was set
	const uint32_t round = sc->round + rel, epoch = sc->epoch + 1 + rel;
	const uint32_t seg = blockIdx.x % kListSegments;
	const uint32_t n = sc->list_count[round % 3][seg];
	const uint32_t off = sc->list_off[seg];
	if (blockIdx.x == 0)
	{
		if (threadIdx.x < kListSegments)
			sc->list_count[(round + 2) % 3][threadIdx.x] = 0;
		if (threadIdx.x == 0)
		{
			uint32_t total = 0;
			for (int q = 0; q < kListSegments; ++q)
				total += sc->list_count[round % 3][q];
			if (head_index < kHeadSizeSlots)
				sc->head_sizes[head_index] = total;
			sc->x_visits += total;
			sc->x_launches += 1;
		}
	}
	const uint4* in_list = a.list[round & 1] + off;
	uint4* out_list = a.list[(round + 1) & 1] + off;
	uint32_t* out_count = &sc->list_count[(round + 1) % 3][seg];
	const uint32_t lane = threadIdx.x & 63;
	const uint32_t waves = gridDim.x / kListSegments * (kThreads / 64);
	const uint32_t ranks = kDeep ? deep_ranks(n, kDeepSegmentWaves < waves ? kDeepSegmentWaves : waves) : 64;
	for (uint32_t base = (blockIdx.x / kListSegments * (kThreads / 64) + threadIdx.x / 64) * ranks; base < n; base += waves * ranks)
	{
		const uint32_t idx = base + lane;
		const bool valid = lane < ranks && idx < n;
		const uint4 w = valid ? in_list[idx] : make_uint4(0, 0, 0, 0);
		const bool keep = round_x<kDeep>(a, w, valid, epoch);
		append_wave(keep, w, out_list, out_count);
	}
}

constexpr int kTailThreads = 1024;

// tail: one workgroup runs the remaining rounds back to back (phases separated by barriers)
// until the list is empty.  The lowest undecided rank decides in every round, so a list of n
// ranks empties within n + 1 rounds; max_rounds bounds the loop regardless.  The first round
// reads the segments of the list; the survivors are appended as one list from offset 0 (segment
// 0, the others empty), which the later rounds read.
__global__ void __launch_bounds__(kTailThreads) k_round_tail(RoundState a, uint32_t rel, uint32_t max_rounds, bool deep)
{
	__shared__ uint32_t s_n, s_out;
	__shared__ uint32_t s_pre[kListSegments + 1], s_off[kListSegments];
	CallScalars* sc = a.sc;
	const uint32_t round0 = sc->round + rel, epoch0 = sc->epoch + 1 + rel;
	__syncthreads(); // every thread has read the base before thread 0 moves it below
	if (threadIdx.x == 0)
	{
		uint32_t total = 0;
		for (int q = 0; q < kListSegments; ++q)
		{
			s_pre[q] = total;
			s_off[q] = sc->list_off[q];
			total += sc->list_count[round0 % 3][q];
		}
		s_pre[kListSegments] = total;
		s_n = total;
		s_out = 0;
	}
	__syncthreads();

	uint32_t round = round0, epoch = epoch0, done = 0;
	for (;;)
	{
		uint32_t n = s_n;
		if (n == 0 || done >= max_rounds)
			break;
		const uint4* in_list = a.list[round & 1];
		uint4* out_list = a.list[(round + 1) & 1];
		const uint32_t lane = threadIdx.x & 63;
		const uint32_t ranks = deep ? deep_ranks(n, kTailThreads / 64) : 64;
		for (uint32_t base = threadIdx.x / 64 * ranks; base < n; base += kTailThreads / 64 * ranks)
		{
			const uint32_t idx = base + lane;
			const bool valid = lane < ranks && idx < n;
			uint4 w = make_uint4(0, 0, 0, 0);
			if (valid)
			{
				int q = 0;
				while (idx >= s_pre[q + 1]) // stops below kListSegments: idx < s_pre[kListSegments] = n
					++q;
				w = in_list[s_off[q] + (idx - s_pre[q])];
			}
			const bool keep = deep ? round_x<true>(a, w, valid, epoch) : round_x<false>(a, w, valid, epoch);
			append_wave(keep, w, out_list, &s_out);
		}
		__syncthreads();
		if (threadIdx.x == 0)
		{
			s_n = s_out;
			s_out = 0;
			s_pre[0] = 0;
			for (int q = 1; q <= kListSegments; ++q)
				s_pre[q] = s_n;
			for (int q = 0; q < kListSegments; ++q)
				s_off[q] = 0;
		}
		round++;
		epoch++;
		done++;
		__syncthreads();
	}

	if (threadIdx.x == 0)
	{
		for (int q = 0; q < kListSegments; ++q)
		{
			sc->list_count[round % 3][q] = q == 0 ? s_n : 0u;
			sc->list_count[(round + 1) % 3][q] = 0;
			sc->list_count[(round + 2) % 3][q] = 0;
			sc->list_off[q] = 0;
			sc->window_count[q] = 0; // the next window open counts from zero
		}
		sc->tail_rounds += done;
		sc->round = round;
		sc->epoch = epoch - 1;
		if (s_n)
			sc->work[3] = 1; // round guard hit: the host reports an error
	}
}

// candidate ranks grouped by source class (order inside a group is irrelevant): one atomic pass
// counts the ranks per source class and hands each its slot in the class's group; after the scan
// the fill places the ranks without atomics
__global__ void k_src_count(const uint2* r_class, size_t count, uint32_t* counts, uint32_t* slot)
{
	size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (k < count)
		slot[k] = atomicAdd(&counts[r_class[k].x], 1u);
}

__global__ void k_src_fill(RoundState a, const uint2* r_class, size_t count, const uint32_t* slot, uint32_t* src_rank, uint32_t* src_val)
{
	size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= count)
		return;
	uint32_t r0 = r_class[k].x;
	uint32_t at = a.src_off[r0] + slot[k];
	src_rank[at] = (uint32_t)k;
	src_val[at] = commit_value_at(a, (uint32_t)k, r0);
}

static RoundState round_state(Mesh& m)
{
	RoundState a;
	a.r_v = m.r_v;
	a.adj_range = m.adj_range[m.adj_cur];
	a.adj = m.adj[m.adj_cur];
	a.pos = m.pos;
	a.kind = m.kind;
	a.wedge = m.wedge;
	a.remap = m.remap;
	a.loop = m.loop[m.loop_cur];
	a.loopback = m.loopback[m.loop_cur];
	a.src_off = m.src_off;
	a.src_rank = m.src_rank;
	a.src_val = m.src_val;
	a.cremap = m.cremap;
	a.lock_rank = m.lock_rank;
	a.status = m.status;
	for (int b = 0; b < 2; ++b)
	{
		a.pend[b] = m.pend[b];
		a.list[b] = m.list[b];
	}
	a.sc = m.sc;
	a.seg_mul = segment_mul(m);
	return a;
}

// the per-source candidate lists deep rounds read, of the ranks below cand_count: a test looks at
// ranks lower than its own, so the window's end is enough (they depend on the ranks alone, so they
// may also be built between the rounds of a window)
void launch_source_lists(hipStream_t s, Mesh& m, size_t cand_count)
{
	size_t n = m.vertex_count;
	fill_u32(s, m.src_off, 0, n + 1);
	// the rank slots go to the candidates' errors: the ranked copies are made, the next pass's
	// candidates are not
	uint32_t* slot = reinterpret_cast<uint32_t*>(m.c_err);
	if (cand_count)
		k_src_count<<<grid_for(cand_count), kThreads, 0, s>>>(m.r_class, cand_count, m.src_off, slot);
	scan_exclusive(s, m.src_off, m.src_off, n, nullptr, m.src_off + n, m.temp);
	if (cand_count)
		k_src_fill<<<grid_for(cand_count), kThreads, 0, s>>>(round_state(m), m.r_class, cand_count, slot, m.src_rank, m.src_val);
}

// Ranks [lo, hi) become a work list, in segments by source class, and publish: the first round of a
// window, in which no rank can do anything else.  sc->window_count holds the ranks per segment (the
// scatter's counts; k_window_count's for the rest of a list); a workgroup takes its places with
// one atomic per segment.  77 us for the 885 k ranks of icosphere L8's first window,
// where a count and a placement of 256 ranks per workgroup, with LDS atomics on eight words, and
// the publishing round took 268.
constexpr int kOpenItems = 4;

__device__ __forceinline__ uint32_t segment_of(const RoundState& a, uint32_t k, uint32_t hi, const uint2* r_class, uint2& cls)
{
	cls = k < hi ? r_class[k] : make_uint2(0, 0);
	return k < hi ? list_segment(a.seg_mul, cls.x) : kNone;
}

template <int kOpenThreads>
__global__ void __launch_bounds__(kOpenThreads) k_window_count(RoundState a, uint32_t lo, uint32_t hi, const uint2* r_class)
{
	__shared__ uint32_t seg[kListSegments];
	if (threadIdx.x < kListSegments)
		seg[threadIdx.x] = 0;
	__syncthreads();
	const uint32_t lane = __lane_id();
	uint32_t n = 0;
	for (int j = 0; j < kOpenItems; ++j)
	{
		uint2 cls;
		const uint32_t q = segment_of(a, lo + (blockIdx.x * kOpenItems + j) * kOpenThreads + threadIdx.x, hi, r_class, cls);
#pragma unroll
		for (uint32_t k = 0; k < kListSegments; ++k)
		{
			const uint64_t m = __ballot(q == k);
			n += lane == k ? (uint32_t)__popcll(m) : 0u;
		}
	}
	if (lane < kListSegments && n)
		atomicAdd(&seg[lane], n);
	__syncthreads();
	if (threadIdx.x < kListSegments && seg[threadIdx.x])
		atomicAdd(&a.sc->window_count[threadIdx.x], seg[threadIdx.x]);
}

template <int kOpenThreads>
__global__ void __launch_bounds__(kOpenThreads) k_window_open(RoundState a, uint32_t lo, uint32_t hi, const uint2* r_class)
{
	__shared__ uint32_t count[kOpenThreads / 64][kListSegments], start[kListSegments];
	CallScalars* sc = a.sc;
	const uint32_t round = sc->round, epoch = sc->epoch + 1;
	const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6;
	const uint64_t below = (1ull << lane) - 1ull;
	uint2 cls[kOpenItems];
	uint32_t seg[kOpenItems], at[kOpenItems];
	uint32_t n = 0; // lane q: this wavefront's ranks of segment q so far
#pragma unroll
	for (int j = 0; j < kOpenItems; ++j)
	{
		seg[j] = segment_of(a, lo + (blockIdx.x * kOpenItems + j) * kOpenThreads + threadIdx.x, hi, r_class, cls[j]);
		at[j] = __shfl(n, (int)(seg[j] & (kListSegments - 1)), 64);
#pragma unroll
		for (uint32_t k = 0; k < kListSegments; ++k)
		{
			const uint64_t m = __ballot(seg[j] == k);
			at[j] += seg[j] == k ? (uint32_t)__popcll(m & below) : 0u;
			n += lane == k ? (uint32_t)__popcll(m) : 0u;
		}
	}
	if (lane < kListSegments)
		count[wave][lane] = n;
	__syncthreads();
	if (threadIdx.x < kListSegments)
	{
		uint32_t off = 0, total = 0;
		for (uint32_t q = 0; q < threadIdx.x; ++q)
			off += sc->window_count[q];
		for (int w = 0; w < kOpenThreads / 64; ++w)
		{
			const uint32_t c = count[w][threadIdx.x];
			count[w][threadIdx.x] = total;
			total += c;
		}
		start[threadIdx.x] = off + (total ? atomicAdd(&sc->list_count[(round + 1) % 3][threadIdx.x], total) : 0u);
		if (blockIdx.x == 0)
			sc->list_off[threadIdx.x] = off;
	}
	__syncthreads();
	uint4* list = a.list[(round + 1) & 1];
	unsigned long long* wr = (unsigned long long*)a.pend[epoch & 1];
#pragma unroll
	for (int j = 0; j < kOpenItems; ++j)
	{
		const uint32_t k = lo + (blockIdx.x * kOpenItems + j) * kOpenThreads + threadIdx.x;
		if (k >= hi)
			continue;
		list[start[seg[j]] + count[wave][seg[j]] + at[j]] = make_uint4(k, cls[j].x, cls[j].y, 0);
		const uint64_t key = round_key(epoch, k);
		atomicMin(&wr[2 * (size_t)cls[j].x], (unsigned long long)key);
		atomicMin(&wr[2 * (size_t)cls[j].y + 1], (unsigned long long)key);
	}
}

template <int kOpenThreads>
static void window_open(hipStream_t s, Mesh& m, size_t lo, size_t hi, bool counted)
{
	const unsigned int grid = div_up(hi > lo ? hi - lo : 1, (size_t)kOpenThreads * kOpenItems);
	const RoundState a = round_state(m);
	if (!counted)
		k_window_count<kOpenThreads><<<grid, kOpenThreads, 0, s>>>(a, (uint32_t)lo, (uint32_t)hi, m.r_class);
	k_window_open<kOpenThreads><<<grid, kOpenThreads, 0, s>>>(a, (uint32_t)lo, (uint32_t)hi, m.r_class);
}

// `counted`: the segments' counts are there already (launch_rank_sort's window).  Few ranks go to
// small workgroups, so that the list is spread over the chip (60 k ranks in sixteen workgroups of
// 1024 threads took 20 us); many go to large ones, for fewer atomics on the eight counters
void launch_window_open(hipStream_t s, Mesh& m, size_t lo, size_t hi, bool counted)
{
	if (hi - lo <= 65536)
		window_open<64>(s, m, lo, hi, counted);
	else if (hi - lo <= 262144)
		window_open<256>(s, m, lo, hi, counted);
	else
		window_open<1024>(s, m, lo, hi, counted);
}

// list_estimate sizes the grid (one rank per thread); the kernels stay correct for any length
void launch_round(hipStream_t s, Mesh& m, size_t list_estimate, int head_index, int rel, bool deep)
{
	// a multiple of kListSegments workgroups, at least one per segment
	unsigned int blocks = grid_for(list_estimate);
	blocks = (blocks + kListSegments - 1) / kListSegments * kListSegments;
	blocks = blocks < kListSegments ? kListSegments : (blocks > 8192 ? 8192 : blocks);
	RoundState a = round_state(m);
	KernelTimer* t = m.timer;
	bool timed = t && t->count < t->capacity;
	if (timed)
		HIP_CHECK(hipEventRecord(t->begin[t->count], s));
	if (deep)
		k_round_x<true><<<blocks, kThreads, 0, s>>>(a, (uint32_t)head_index, (uint32_t)rel);
	else
		k_round_x<false><<<blocks, kThreads, 0, s>>>(a, (uint32_t)head_index, (uint32_t)rel);
	if (timed)
		HIP_CHECK(hipEventRecord(t->end[t->count++], s));
}

void launch_round_tail(hipStream_t s, Mesh& m, int rel, uint32_t max_rounds, bool deep)
{
	k_round_tail<<<1, kTailThreads, 0, s>>>(round_state(m), (uint32_t)rel, max_rounds, deep);
}

// ------------------------------------------------------------------------------------------
// stop scan: the first rank where the sequential loop breaks (src/simplifier.cpp:1517-1539)
//   S1 err > error_limit
//   S2 tri_collapses >= goal
//   S3 err > 1.5 * err[goal/2 + rejects] && err > result_error && tri_collapses > goal/6
// with tri_collapses, rejects and result_error the exclusive prefix sums / max of the decided
// ranks.  Two kernels over tiles of ranks, each thread owning consecutive ones: the first settles
// the failed flip tests and adds up its tile; in the second each workgroup adds the tiles before
// its own, tests its ranks and leaves a record, and the workgroup that finishes last takes the
// first record with a break.  14 us a pass at 200 k candidates, where settling, tile scan, totals and
// finish as kernels of their own, with one block scan per 256 ranks, took 61.

struct StopAgg
{
	uint32_t commit; // committed | border << 16
	uint32_t other;  // rejected | skipped << 16
	uint32_t err;    // bits of the largest committed error; a NaN stays out (its `<` test fails)
};

constexpr int kStopWords = 5; // of a tile: committed, border, rejected, skipped, largest error

__device__ __forceinline__ void stop_add(StopAgg& a, uint8_t st, float err)
{
	a.commit += is_commit(st) ? (st == kCommittedBorder ? 0x10001u : 1u) : 0u;
	a.other += st == kRejected ? 1u : (st == kSkipped ? 0x10000u : 0u);
	const uint32_t e = is_commit(st) && err == err ? __float_as_uint(err) : 0u;
	a.err = e > a.err ? e : a.err;
}

// a failed flip test is a rejection unless a lower commit locked an endpoint first
__device__ __forceinline__ uint8_t settle(uint8_t st, uint32_t k, const uint2* r_class, const uint32_t* lock_rank)
{
	if (st != kFlipFail)
		return st;
	const uint32_t l0 = lock_rank[r_class[k].x], l1 = lock_rank[r_class[k].y];
	return ((l0 != kNone && l0 < k) || (l1 != kNone && l1 < k)) ? kSkipped : kRejected;
}

// thread t owns ranks [base, base + kItems): the status bytes of a full run as words
template <int kItems>
__device__ __forceinline__ void load_status(const uint8_t* status, uint32_t base, uint32_t count, uint8_t st[kItems])
{
	if (base + kItems <= count)
	{
#pragma unroll
		for (int q = 0; q < kItems / 4; ++q)
		{
			const uint32_t w = reinterpret_cast<const uint32_t*>(status + base)[q];
#pragma unroll
			for (int b = 0; b < 4; ++b)
				st[4 * q + b] = (uint8_t)(w >> (8 * b));
		}
	}
	else
	{
#pragma unroll
		for (int q = 0; q < kItems; ++q)
			st[q] = base + q < count ? status[base + q] : (uint8_t)kUndecided;
	}
}

template <int kItems>
__global__ void __launch_bounds__(kThreads) k_stop_reduce(uint8_t* status, const float* r_err, const uint2* r_class,
                                                          const uint32_t* lock_rank, uint32_t count, uint32_t* tiles)
{
	__shared__ uint32_t red[kStopWords][kThreads / 64];
	const uint32_t base = (blockIdx.x * kThreads + threadIdx.x) * kItems;
	uint8_t st[kItems];
	load_status<kItems>(status, base, count, st);
	StopAgg acc{0, 0, 0};
#pragma unroll
	for (int q = 0; q < kItems; ++q)
		if (base + q < count)
		{
			const uint8_t now = settle(st[q], base + q, r_class, lock_rank);
			if (now != st[q])
				status[base + q] = now;
			stop_add(acc, now, r_err[base + q]);
		}
	const uint32_t v[kStopWords] = {acc.commit & 0xffffu, acc.commit >> 16, acc.other & 0xffffu, acc.other >> 16, acc.err};
	const int wave = threadIdx.x >> 6;
#pragma unroll
	for (int q = 0; q < kStopWords; ++q)
	{
		const uint32_t x = q < 4 ? wave_sum(v[q]) : wave_max(v[q]);
		if (__lane_id() == 0)
			red[q][wave] = x;
	}
	__syncthreads();
	if (threadIdx.x < kStopWords)
	{
		uint32_t x = 0;
		for (int w = 0; w < kThreads / 64; ++w)
		{
			const uint32_t t = red[threadIdx.x][w];
			x = threadIdx.x < 4 ? x + t : (t > x ? t : x);
		}
		tiles[(size_t)blockIdx.x * kStopWords + threadIdx.x] = x;
	}
}

// words of a tile's record: the first stopping rank (kNone: none), then the totals below it (below
// the tile's end when there is none) and the reason
enum
{
	kRecRank,
	kRecCommitted,
	kRecBorder,
	kRecRejected,
	kRecSkipped,
	kRecError,
	kRecReason,
	kRecWords
};

template <int kItems>
__global__ void __launch_bounds__(kThreads) k_stop_find(const uint8_t* status, const float* r_err, uint32_t count, uint32_t cand_count, const uint32_t* tiles,
                                                        uint32_t* records, uint32_t goal, float error_limit, CallScalars* sc)
{
	__shared__ uint32_t red[kStopWords][kThreads / 64];
	__shared__ uint32_t before[kStopWords];
	__shared__ uint32_t s_first, s_last;
	const int wave = threadIdx.x >> 6, lane = __lane_id();
	// the tiles before this one
	{
		uint32_t v[kStopWords] = {0, 0, 0, 0, 0};
		for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kThreads)
		{
#pragma unroll
			for (int q = 0; q < kStopWords; ++q)
			{
				const uint32_t t = tiles[(size_t)b * kStopWords + q];
				v[q] = q < 4 ? v[q] + t : (t > v[q] ? t : v[q]);
			}
		}
#pragma unroll
		for (int q = 0; q < kStopWords; ++q)
		{
			const uint32_t x = q < 4 ? wave_sum(v[q]) : wave_max(v[q]);
			if (lane == 0)
				red[q][wave] = x;
		}
		if (threadIdx.x == 0)
			s_first = kNone;
		__syncthreads();
		if (threadIdx.x < kStopWords)
		{
			uint32_t x = threadIdx.x < 4 ? 0u : __float_as_uint(sc->result_error);
			for (int w = 0; w < kThreads / 64; ++w)
			{
				const uint32_t t = red[threadIdx.x][w];
				x = threadIdx.x < 4 ? x + t : (t > x ? t : x);
			}
			before[threadIdx.x] = x;
		}
		__syncthreads();
	}
	// the ranks before this thread's inside the tile
	const uint32_t base = (blockIdx.x * kThreads + threadIdx.x) * kItems;
	uint8_t st[kItems];
	float err[kItems];
	load_status<kItems>(status, base, count, st);
	StopAgg own{0, 0, 0};
#pragma unroll
	for (int q = 0; q < kItems; ++q)
	{
		err[q] = base + q < count ? r_err[base + q] : 0.f;
		if (base + q < count)
			stop_add(own, st[q], err[q]);
	}
	StopAgg in = own;
#pragma unroll
	for (int o = 1; o < 64; o <<= 1)
	{
		const uint32_t c = __shfl_up(in.commit, o, 64), r = __shfl_up(in.other, o, 64), e = __shfl_up(in.err, o, 64);
		if (lane >= o)
		{
			in.commit += c;
			in.other += r;
			in.err = e > in.err ? e : in.err;
		}
	}
	if (lane == 63)
	{
		red[0][wave] = in.commit;
		red[1][wave] = in.other;
		red[2][wave] = in.err;
	}
	__syncthreads();
	uint32_t up = __shfl_up(in.err, 1, 64);
	up = lane ? up : 0u;
	uint32_t wc = 0, wo = 0, we = 0;
#pragma unroll
	for (int w = 0; w < kThreads / 64; ++w)
		if (w < wave)
		{
			wc += red[0][w];
			wo += red[1][w];
			we = red[2][w] > we ? red[2][w] : we;
		}
	const uint32_t xc = wc + in.commit - own.commit, xo = wo + in.other - own.other;
	uint32_t committed = before[0] + (xc & 0xffffu), border = before[1] + (xc >> 16);
	uint32_t rejected = before[2] + (xo & 0xffffu), skipped = before[3] + (xo >> 16);
	uint32_t best = before[4];
	best = we > best ? we : best;
	best = up > best ? up : best;

	const uint32_t half = goal / 2, sixth = goal / 6;
	uint32_t reason = 0, at = kNone;
#pragma unroll
	for (int q = 0; q < kItems; ++q)
	{
		const uint32_t k = base + q;
		if (k >= count || reason)
			continue;
		const uint32_t tri = 2 * committed - border;
		if (err[q] > error_limit)
			reason = 1;
		else if (tri >= goal)
			reason = 2;
		else if (tri > sixth && err[q] > __uint_as_float(best))
		{
			const size_t eg = (size_t)half + rejected;
			const float error_goal = eg < cand_count ? 1.5f * r_err[eg] : FLT_MAX;
			reason = err[q] > error_goal ? 3u : 0u;
		}
		if (reason)
		{
			at = k;
			continue;
		}
		committed += is_commit(st[q]);
		border += st[q] == kCommittedBorder;
		rejected += st[q] == kRejected;
		skipped += st[q] == kSkipped;
		const uint32_t e = is_commit(st[q]) && err[q] == err[q] ? __float_as_uint(err[q]) : 0u;
		best = e > best ? e : best;
	}
	// ranks grow with the thread: the first stopping thread holds the tile's first stop; without one
	// the last thread's totals are the tile's end
	const uint64_t stops = __ballot(reason != 0);
	if (stops && lane == __builtin_ctzll(stops))
		atomicMin(&s_first, threadIdx.x);
	__syncthreads();
	const uint32_t owner = s_first != kNone ? s_first : kThreads - 1;
	if (threadIdx.x == owner)
	{
		uint32_t* rec = records + (size_t)blockIdx.x * kRecWords;
		const uint32_t w[kRecWords] = {at, committed, border, rejected, skipped, best, reason};
#pragma unroll
		for (int q = 0; q < kRecWords; ++q)
			(void)__hip_atomic_exchange(&rec[q], w[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		wait_for_memory();
		s_last = atomicAdd(&sc->stop_done, 1u) + 1 == gridDim.x;
	}
	__syncthreads();
	if (!s_last || threadIdx.x >= 64)
		return;
	if (threadIdx.x == 0)
		sc->split = 0;
	// the first record with a break, else the last tile's: one wavefront
	uint32_t hit = gridDim.x - 1;
	for (uint32_t b0 = 0; b0 < gridDim.x; b0 += 64)
	{
		const uint32_t b = b0 + lane;
		const bool found = b < gridDim.x && __hip_atomic_load(&records[(size_t)b * kRecWords + kRecRank], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != kNone;
		const uint64_t m = __ballot(found);
		if (m)
		{
			hit = b0 + (uint32_t)__builtin_ctzll(m);
			break;
		}
	}
	if (lane)
		return;
	uint32_t w[kRecWords];
	for (int q = 0; q < kRecWords; ++q)
		w[q] = __hip_atomic_load(&records[(size_t)hit * kRecWords + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	const bool more = w[kRecRank] == kNone && count < cand_count; // no break in the window: the host decides the rest
	sc->stop_done = 0;
	sc->extend = more;
	sc->stop = w[kRecRank] == kNone ? count : w[kRecRank];
	sc->stop_reason = w[kRecReason];
	sc->committed = w[kRecCommitted];
	sc->rejected = w[kRecRejected];
	sc->skipped = w[kRecSkipped];
	if (!more)
	{
		sc->result_error = __uint_as_float(w[kRecError]);
	}
}

// repeatable: reads the decisions of ranks [0, window) and writes only the stop rank (window if no
// rank in it breaks the loop), the totals below it and, unless the list goes on past a window
// without a break (sc->extend), the pass's result error
void launch_stop_scan(hipStream_t s, Mesh& m, size_t window, size_t cand_count, uint32_t goal, float error_limit)
{
	const uint32_t n = (uint32_t)window, c = (uint32_t)cand_count;
	// four ranks a thread until the tiles would be many (each workgroup reads those before it)
	const bool wide = window > (size_t)1024 * 1024;
	const unsigned int tiles = div_up(window, (size_t)kThreads * (wide ? 16 : 4));
	uint32_t* records = m.stop_tile + (size_t)kStopWords * tiles;
	if (wide)
	{
		k_stop_reduce<16><<<tiles, kThreads, 0, s>>>(m.status, m.r_err, m.r_class, m.lock_rank, n, m.stop_tile);
		k_stop_find<16><<<tiles, kThreads, 0, s>>>(m.status, m.r_err, n, c, m.stop_tile, records, goal, error_limit, m.sc);
	}
	else
	{
		k_stop_reduce<4><<<tiles, kThreads, 0, s>>>(m.status, m.r_err, m.r_class, m.lock_rank, n, m.stop_tile);
		k_stop_find<4><<<tiles, kThreads, 0, s>>>(m.status, m.r_err, n, c, m.stop_tile, records, goal, error_limit, m.sc);
	}
}

size_t stop_scan_words(size_t cand_count)
{
	// up to 1024 tiles of four ranks a thread, then tiles of sixteen
	const size_t short_tiles = std::min((size_t)div_up(cand_count, kThreads * 4), (size_t)1024);
	return (kStopWords + kRecWords) * std::max(short_tiles, (size_t)div_up(cand_count, kThreads * 16));
}

// ------------------------------------------------------------------------------------------
// updateQuadrics (src/simplifier.cpp:1638-1673), one thread per commit below the stop.
// The target class receives exactly one positional add (its primary is locked); attribute
// quadrics move wedge by wedge in ascending wedge order, as the reference's vertex loop does.

__device__ __forceinline__ uint32_t next_wedge_above(const uint32_t* wedge, uint32_t r, uint32_t after)
{
	// smallest member of r's ring greater than `after` (kNone if none)
	uint32_t best = kNone;
	uint32_t v = r;
	do
	{
		if (v > after && v < best)
			best = v;
		v = wedge[v];
	} while (v != r);
	return best;
}

// one committed collapse of k_update_quadrics; returns the bits of its non-NaN positional error
// (non-negative floats order like their bits), 0 without attributes
__device__ __forceinline__ uint32_t update_one(size_t k, const uint2* r_class, const uint32_t* cremap, const uint32_t* wedge,
                                               const float4* pos, int attr_count, Quad* vq, Grad* vg, Quad* aq, Grad* ag)
{
	const uint32_t r0 = r_class[k].x, r1 = r_class[k].y;

	Quad Q0 = load_quad(vq, r0);
	Quad Q1 = load_quad(vq, r1);
	quad_add(Q1, Q0);
	store_quad(vq, r1, Q1);
	if (vg)
	{
		// the class is a target of one collapse per pass at most: no other update of vg[r1]
		Grad G1 = vg[r1];
		grad_add(G1, vg[r0]);
		vg[r1] = G1;
	}

	if (attr_count)
	{
		const int A = attr_count;
		// r0 is the lowest index of its class, so ascending order starts there
		for (uint32_t v = r0; v != kNone; v = next_wedge_above(wedge, r0, v))
		{
			uint32_t t = cremap[v];
			if (t == v)
				continue;
			Quad Qt = load_quad(aq, t);
			quad_add(Qt, load_quad(aq, v));
			store_quad(aq, t, Qt);
			// four gradients at a time, all loads before the stores (which the compiler must take
			// to alias them)
			for (int a0 = 0; a0 < A; a0 += 4)
			{
				Grad to[4], from[4];
#pragma unroll
				for (int q = 0; q < 4; ++q)
				{
					const int a = a0 + q < A ? a0 + q : A - 1;
					to[q] = ag[(size_t)t * A + a];
					from[q] = ag[(size_t)v * A + a];
				}
#pragma unroll
				for (int q = 0; q < 4; ++q)
					if (a0 + q < A)
					{
						grad_add(to[q], from[q]);
						ag[(size_t)t * A + a0 + q] = to[q];
					}
			}
		}

		float derr = quad_error(Q0, load_pos(pos, r1));
		if (derr == derr)
			return __float_as_uint(derr);
	}
	return 0;
}

// After the stop is known, one launch over two ranges of workgroups that never touch each other's
// state: the ranks (updateQuadrics), and the vertices, each of which
//   - takes back a move at or past the stop (a commit wrote only its source class's wedges).  Other
//     vertices read collapse_remap through settled_remap, which gives the same before and after;
//   - remaps its edge loops (remapEdgeLoops, src/simplifier.cpp:1845-1864): collapse_remap is
//     idempotent within a pass (targets are locked, never sources), so reading loop[l] before or
//     after its own update gives the same result and the in-place loop becomes a double-buffered map;
//   - as a primary, leaves its class's new id and adds the room its adjacency may need to its tile,
//     and checks that a class that moves goes to its commit's target; as a secondary, checks that it
//     goes where its primary does.  Both hold while a seam class's two loops name neighbours of one
//     class, as the classification asks; no mesh is known where they stop to.
struct ApplyArgs
{
	const uint8_t* status;
	const uint2* r_class;
	uint32_t* cremap;
	const uint32_t* lock_rank;
	const uint32_t* remap;
	const uint32_t* wedge;
	const float4* pos;
	Quad* vq;
	Grad* vg;
	Quad* aq;
	Grad* ag;
	const uint32_t* loop_in;
	const uint32_t* back_in;
	uint32_t* loop_out;
	uint32_t* back_out;
	const uint2* range_in;
	const uint2* adj_in;
	uint2* range_out;
	uint2* adj_out;
	uint32_t* new_class;
	uint2* sums;
	CallScalars* sc;
	int attr_count;
	uint32_t rank_blocks;
	uint32_t vertices;
	uint32_t items;
};

__device__ __forceinline__ uint32_t settled_remap(const ApplyArgs& a, uint32_t v, uint32_t stop)
{
	const uint32_t c = a.cremap[v];
	return c != v && a.lock_rank[a.remap[v]] >= stop ? v : c;
}

__device__ __forceinline__ uint32_t remap_loop(const ApplyArgs& a, const uint32_t* in, uint32_t i, uint32_t stop)
{
	const uint32_t l = in[i];
	if (l == kNone)
		return kNone;
	const uint32_t r = settled_remap(a, l, stop);
	if (i != r)
		return r;
	const uint32_t ll = in[l];
	return ll != kNone ? settled_remap(a, ll, stop) : kNone;
}

// the old adjacency lists a class's new one is made of: its own, and that of the class collapsed
// into it this pass; none once it is collapsed itself (one commit at most touches a class)
struct ClassLists
{
	uint2 own, other;
	uint32_t target; // the class it is collapsed into (kNone: none)
	__device__ __forceinline__ uint32_t room() const
	{
		return (own.y - own.x) + (other.y - other.x);
	}
};

__device__ __forceinline__ ClassLists class_lists(const ApplyArgs& a, uint32_t v, uint32_t stop)
{
	ClassLists l;
	l.own = a.range_in[v];
	l.other = make_uint2(0, 0);
	l.target = kNone;
	const uint32_t k = a.lock_rank[v];
	if (k < stop)
	{
		const uint2 c = a.r_class[k];
		if (c.x == v)
		{
			l.own = make_uint2(0, 0);
			l.target = c.y;
		}
		else
			l.other = a.range_in[c.x];
	}
	return l;
}

__global__ void __launch_bounds__(kThreads) k_apply(ApplyArgs a)
{
	__shared__ uint2 red[kThreads / 64];
	if (a.sc->extend)
		return;
	const uint32_t stop = a.sc->stop;
	if (blockIdx.x < a.rank_blocks)
	{
		const uint32_t k = blockIdx.x * kThreads + threadIdx.x;
		// the largest positional error of the pass's commits (attribute path): one atomic per
		// wavefront, so every lane stays to the reduction
		uint32_t err_bits = 0;
		if (k < stop && is_commit(a.status[k]))
			err_bits = update_one(k, a.r_class, a.cremap, a.wedge, a.pos, a.attr_count, a.vq, a.vg, a.aq, a.ag);
		if (a.attr_count)
		{
			err_bits = wave_max(err_bits);
			if (__lane_id() == 0 && err_bits)
				atomicMax(&a.sc->vertex_error_bits, err_bits);
		}
		return;
	}
	const uint32_t tile = blockIdx.x - a.rank_blocks;
	uint2 room = make_uint2(0, 0);
	for (uint32_t j = 0; j < a.items; ++j)
	{
		const uint32_t v = (tile * a.items + j) * kThreads + threadIdx.x;
		if (v >= a.vertices)
			break;
		const uint32_t c = settled_remap(a, v, stop);
		if (c != a.cremap[v])
			a.cremap[v] = c;
		a.loop_out[v] = remap_loop(a, a.loop_in, v, stop);
		a.back_out[v] = remap_loop(a, a.back_in, v, stop);
		const uint32_t r = a.remap[v];
		if (r == v)
		{
			const uint32_t to = a.remap[c];
			const ClassLists l = class_lists(a, v, stop);
			a.new_class[v] = to;
			room.x += l.room();
			if (l.target != kNone && l.target != to)
				a.sc->split = 1; // its list would go to another class than its vertices
		}
		else if (a.remap[c] != a.remap[settled_remap(a, r, stop)])
			a.sc->split = 1; // this wedge went elsewhere than its primary: the lists by class do not hold
	}
	room = block_sum2(room, red);
	if (threadIdx.x == 0)
		a.sums[tile] = room;
}

// The next pass's welded adjacency from this one's: a class's list is its old one and that of the
// class collapsed into it, every entry through the classes' new ids, without the triangles that
// have fallen together (the rule of the index remap).  The lists lie at the sum of the rooms before
// them, so nothing is counted first and nothing is placed by atomics.  Lists of more than
// kLongList entries are walked by the whole wavefront.  Icosphere L8, after its first pass (919 k
// triangles left): 48 us, where counting by atomics, scan and fill took 176.
constexpr uint32_t kLongList = 64;

__device__ __forceinline__ bool entry_stays(uint32_t v, uint32_t x, uint32_t y)
{
	return x != y && x != v && y != v;
}

__global__ void __launch_bounds__(kThreads) k_adj_walk(ApplyArgs a)
{
	__shared__ uint2 red2[kThreads / 64];
	__shared__ uint32_t red[kThreads / 64];
	if (a.sc->extend)
		return;
	const uint32_t stop = a.sc->stop;
	uint32_t at = sums_before(a.sums, blockIdx.x, red2).x;
	const uint32_t lane = __lane_id();
	for (uint32_t j = 0; j < a.items; ++j)
	{
		const uint32_t v = (blockIdx.x * a.items + j) * kThreads + threadIdx.x;
		ClassLists l{make_uint2(0, 0), make_uint2(0, 0), kNone};
		if (v < a.vertices && a.remap[v] == v)
			l = class_lists(a, v, stop);
		const uint32_t room = l.room();
		uint32_t total;
		const uint32_t begin = at + block_scan(room, red, total);
		uint32_t end = begin;
		const bool longer = room > kLongList;
		if (!longer)
		{
			for (int part = 0; part < 2; ++part)
			{
				const uint2 r = part ? l.other : l.own;
				for (uint32_t p0 = r.x; p0 < r.y; p0 += 4)
				{
					uint2 e[4];
#pragma unroll
					for (int q = 0; q < 4; ++q)
						e[q] = p0 + q < r.y ? a.adj_in[p0 + q] : make_uint2(v, v);
					uint32_t x[4], y[4];
#pragma unroll
					for (int q = 0; q < 4; ++q)
					{
						x[q] = a.new_class[e[q].x];
						y[q] = a.new_class[e[q].y];
					}
#pragma unroll
					for (int q = 0; q < 4; ++q)
						if (p0 + q < r.y && entry_stays(v, x[q], y[q]))
							a.adj_out[end++] = make_uint2(x[q], y[q]);
				}
			}
		}
		for (uint64_t left = __ballot(longer); left; left &= left - 1)
		{
			const int from = __builtin_ctzll(left);
			const uint32_t w = __shfl(v, from, 64);
			uint32_t to = __shfl(begin, from, 64);
			for (int part = 0; part < 2; ++part)
			{
				const uint2 r = part ? l.other : l.own;
				const uint32_t rb = __shfl(r.x, from, 64), re = __shfl(r.y, from, 64);
				for (uint32_t p0 = rb; p0 < re; p0 += 64)
				{
					uint32_t x = w, y = w;
					if (p0 + lane < re)
					{
						const uint2 e = a.adj_in[p0 + lane];
						x = a.new_class[e.x];
						y = a.new_class[e.y];
					}
					const bool stays = entry_stays(w, x, y);
					const uint64_t m = __ballot(stays);
					if (stays)
						a.adj_out[to + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = make_uint2(x, y);
					to += (uint32_t)__popcll(m);
				}
			}
			if ((int)lane == from)
				end = to;
		}
		if (v < a.vertices)
			a.range_out[v] = make_uint2(begin, end);
		at += total;
	}
}

// the other set of index, loop and adjacency buffers is written; the caller makes it current once
// the read-back says that the pass committed something
void launch_apply(hipStream_t s, Mesh& m, size_t window, size_t tri_count)
{
	ApplyArgs a;
	a.status = m.status;
	a.r_class = m.r_class;
	a.cremap = m.cremap;
	a.lock_rank = m.lock_rank;
	a.remap = m.remap;
	a.wedge = m.wedge;
	a.pos = m.pos;
	a.vq = m.vq;
	a.vg = m.vg;
	a.aq = m.aq;
	a.ag = m.ag;
	a.loop_in = m.loop[m.loop_cur];
	a.back_in = m.loopback[m.loop_cur];
	a.loop_out = m.loop[m.loop_cur ^ 1];
	a.back_out = m.loopback[m.loop_cur ^ 1];
	a.range_in = m.adj_range[m.adj_cur];
	a.adj_in = m.adj[m.adj_cur];
	a.range_out = m.adj_range[m.adj_cur ^ 1];
	a.adj_out = m.adj[m.adj_cur ^ 1];
	a.new_class = m.new_class;
	a.sums = m.vertex_sums;
	a.sc = m.sc;
	a.attr_count = (int)m.attr_count;
	a.rank_blocks = grid_for(window);
	a.vertices = m.vertex_count;
	a.items = tile_items(m.vertex_count);
	const unsigned int tiles = div_up(m.vertex_count, (size_t)kThreads * a.items);
	k_apply<<<a.rank_blocks + tiles, kThreads, 0, s>>>(a);
	const TriArgs t = tri_args(m, tri_count, nullptr, m.loop_cur ^ 1);
	const unsigned int tri_tiles = div_up(tri_count, (size_t)kThreads * t.items);
	k_tri_count<true><<<tri_tiles, kThreads, 0, s>>>(t);
	k_tri_write<true><<<tri_tiles, kThreads, 0, s>>>(t);
	k_adj_walk<<<tiles, kThreads, 0, s>>>(a);
}

// ------------------------------------------------------------------------------------------
// finalisation (src/simplifier.cpp:2601-2619)

__global__ void k_debug_bits(uint32_t* ib, size_t tris, const uint8_t* kind, const uint32_t* loop, const uint32_t* loopback)
{
	size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= tris)
		return;
	uint32_t a = ib[t * 3 + 0], b = ib[t * 3 + 1], c = ib[t * 3 + 2];
	ib[t * 3 + 0] = a | ((uint32_t)kind[a] << 28) | ((uint32_t)(loop[a] == b || loopback[b] == a) << 31);
	ib[t * 3 + 1] = b | ((uint32_t)kind[b] << 28) | ((uint32_t)(loop[b] == c || loopback[c] == b) << 31);
	ib[t * 3 + 2] = c | ((uint32_t)kind[c] << 28) | ((uint32_t)(loop[c] == a || loopback[a] == c) << 31);
}

void launch_debug_bits(hipStream_t s, Mesh& m, size_t index_count)
{
	size_t tris = index_count / 3;
	if (tris)
		k_debug_bits<<<grid_for(tris), kThreads, 0, s>>>(m.ib[m.ib_cur], tris, m.kind, m.loop[m.loop_cur], m.loopback[m.loop_cur]);
}

__global__ void k_sparse_backmap(uint32_t* ib, size_t n, const uint32_t* sparse_remap)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		ib[i] = sparse_remap[ib[i]];
}

void launch_sparse_backmap(hipStream_t s, uint32_t* ib, size_t index_count, const uint32_t* sparse_remap)
{
	if (index_count)
		k_sparse_backmap<<<grid_for(index_count), kThreads, 0, s>>>(ib, index_count, sparse_remap);
}

} // namespace mhip
