// meshopt_simplifySloppy kernels (src/simplifier.cpp:2087-2334, 2647-2778).  Every step that the
// reference runs in input order is made order-independent: cells are numbered by the first
// vertex of each id (a minimum per id, then a scan), cell quadrics are summed per cell in the
// reference's (triangle, corner) order after a stable sort, the chosen vertex is a 64-bit
// minimum of (error bits, index), and a duplicate triangle keeps its first occurrence (a minimum
// per canonical triple, then an ordered compaction).  No float atomics.
#include "prims.h"
#include "quadric.h"
#include "sloppy.h"

#include <algorithm>

namespace mhip
{

static constexpr int kThreads = 256;
// entries per cell from which a wavefront sums a cell instead of 16 lanes (1.3 million triangles, the
// call: 547 us against 569 at 60 entries a cell, 773 against 748 at 20, 1023 against 953 at 12)
static constexpr size_t kLongCell = 48;

static inline unsigned int grid_for(size_t n, unsigned int cap = 65535)
{
	unsigned int g = div_up(n ? n : 1, kThreads);
	return g > cap ? cap : g;
}

// float to int as the reference's x86 build converts it (cvttss2si): truncation toward zero, and
// the "integer indefinite" 0x80000000 for NaN and for values outside the int range.  The GPU's
// own conversion gives 0 for NaN and saturates, so a NaN position (the rescale leaves NaN
// coordinates NaN) would fall into a different cell than on the CPU.
__device__ __forceinline__ int cvt_trunc_x86(float f)
{
	return (f >= -2147483648.f && f < 2147483648.f) ? (int)f : (int)0x80000000u;
}

// computeVertexIds (src/simplifier.cpp:2087-2105): round-half-up cell coordinates of the
// rescaled position, 10 bits per axis; a vertex locked by vertex_lock gets an id of its own
__device__ __forceinline__ uint32_t sloppy_id(float4 p, bool locked, uint32_t v, float cell_scale)
{
	if (locked)
		return (1u << 30) | v;
	const int xi = cvt_trunc_x86(p.x * cell_scale + 0.5f);
	const int yi = cvt_trunc_x86(p.y * cell_scale + 0.5f);
	const int zi = cvt_trunc_x86(p.z * cell_scale + 0.5f);
	return ((uint32_t)xi << 20) | ((uint32_t)yi << 10) | (uint32_t)zi;
}

__device__ __forceinline__ uint32_t mix32(uint32_t h)
{
	h ^= h >> 16;
	h *= 0x7feb352du;
	h ^= h >> 15;
	h *= 0x846ca68bu;
	h ^= h >> 16;
	return h;
}

__global__ void k_sloppy_ids(const float4* pos, const uint8_t* lock, uint32_t n, float cell_scale, uint32_t* ids)
{
	for (uint32_t v = blockIdx.x * kThreads + threadIdx.x; v < n; v += gridDim.x * kThreads)
		ids[v] = sloppy_id(pos[v], lock && (lock[v] & kVertexLock), v, cell_scale);
}

// countTriangles (src/simplifier.cpp:2107-2121) at one or two grid sizes.  The search is a chain of
// counts, each a launch and a wait of the host: the first two grid sizes are known together and are
// counted in one launch, and the workgroup that ends last writes the sums to host memory (no
// clearing, no copy).  A thread has the indices of kCountItems triangles in flight, then their
// positions.  1.3 million triangles over 655 thousand vertices: 29 us a count against 33, 31 for two,
// and two launches less for each.  What bounds it is the number of lines asked of the L2s: ids formed
// beforehand, a quarter of the bytes, took as long (5.6 and 22.6 us).
constexpr int kCountThreads = 512;
constexpr int kCountItems = 3;
constexpr unsigned int kCountGroups = 512;

template <int kGrids>
__global__ void __launch_bounds__(kCountThreads) k_sloppy_count(const uint32_t* idx, uint32_t tris, const float4* pos, const uint8_t* lock,
                                                                float cell_scale0, float cell_scale1, unsigned long long* parts, uint32_t* done,
                                                                uint32_t* host_counts)
{
	__shared__ unsigned long long part[kCountThreads / 64];
	__shared__ uint32_t last;
	const float cell_scale[2] = {cell_scale0, cell_scale1};
	// low half: triangles at the first grid size, high half: at the second
	unsigned long long local = 0;
	const size_t step = gridDim.x * kCountThreads;
	for (size_t t0 = blockIdx.x * kCountThreads + threadIdx.x; t0 < tris; t0 += step * kCountItems)
	{
		uint32_t v[kCountItems][3];
#pragma unroll
		for (int q = 0; q < kCountItems; ++q)
		{
			const size_t t = t0 + step * q < tris ? t0 + step * q : t0;
#pragma unroll
			for (int k = 0; k < 3; ++k)
				v[q][k] = idx[3 * t + k];
		}
		float4 p[kCountItems][3];
#pragma unroll
		for (int q = 0; q < kCountItems; ++q)
#pragma unroll
			for (int k = 0; k < 3; ++k)
				p[q][k] = pos[v[q][k]];
		uint32_t id[kGrids][kCountItems][3];
#pragma unroll
		for (int q = 0; q < kCountItems; ++q)
#pragma unroll
			for (int k = 0; k < 3; ++k)
			{
				const bool locked = lock && (lock[v[q][k]] & kVertexLock);
#pragma unroll
				for (int g = 0; g < kGrids; ++g)
					id[g][q][k] = sloppy_id(p[q][k], locked, v[q][k], cell_scale[g]);
			}
#pragma unroll
		for (int q = 0; q < kCountItems; ++q)
		{
			const bool live = t0 + step * q < tris;
#pragma unroll
			for (int g = 0; g < kGrids; ++g)
			{
				const uint32_t a = id[g][q][0], b = id[g][q][1], c = id[g][q][2];
				local += (unsigned long long)(live & (a != b) & (a != c) & (b != c)) << (32 * g);
			}
		}
	}
	for (int o = 32; o > 0; o >>= 1)
		local += __shfl_xor(local, o, 64);
	if (__lane_id() == 0)
		part[threadIdx.x >> 6] = local;
	__syncthreads();
	if (threadIdx.x == 0)
	{
		unsigned long long sum = 0;
		for (int w = 0; w < kCountThreads / 64; ++w)
			sum += part[w];
		atomicExch(&parts[blockIdx.x], sum);
		wait_for_memory();
		last = atomicAdd(done, 1u) + 1 == gridDim.x;
	}
	__syncthreads();
	if (!last)
		return;
	// at most kCountGroups = kCountThreads parts; an atomic reads what other XCDs wrote
	unsigned long long sum = threadIdx.x < gridDim.x ? atomicAdd(&parts[threadIdx.x], 0ull) : 0ull;
	for (int o = 32; o > 0; o >>= 1)
		sum += __shfl_xor(sum, o, 64);
	if (__lane_id() == 0)
		part[threadIdx.x >> 6] = sum;
	__syncthreads();
	if (threadIdx.x == 0)
	{
		sum = 0;
		for (int w = 0; w < kCountThreads / 64; ++w)
			sum += part[w];
		host_counts[0] = (uint32_t)sum;
		host_counts[1] = (uint32_t)(sum >> 32);
		atomicExch(done, 0u);
	}
}

// fillVertexCells (src/simplifier.cpp:2123-2146), step 1: the table slot of an id ends holding
// the lowest vertex with that id (a slot only ever holds vertices of one id).  Of neighbouring lanes
// with one id only the first, the lowest, goes to the table; a slot is read before it is written,
// since atomics on one address come one after the other (55 us for 655 thousand vertices in 20
// thousand cells without either, 22 with both).
__global__ void k_vtable_insert(const uint32_t* ids, uint32_t n, uint32_t* table, uint32_t mask)
{
	for (uint32_t v = blockIdx.x * kThreads + threadIdx.x; v < n; v += gridDim.x * kThreads)
	{
		const uint32_t id = ids[v];
		const uint32_t left = __shfl_up(id, 1, 64);
		if (__lane_id() && left == id)
			continue;
		uint32_t slot = mix32(id) & mask;
		for (uint32_t probe = 0; probe <= mask; ++probe)
		{
			uint32_t old = __hip_atomic_load(&table[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			if (old == kNone)
			{
				old = atomicCAS(&table[slot], kNone, v);
				if (old == kNone)
					break;
			}
			if (ids[old] == id)
			{
				if (v < old)
					atomicMin(&table[slot], v);
				break;
			}
			slot = (slot + 1) & mask;
		}
	}
}

// step 2: each vertex's representative (the first vertex of its id) and the representative flags
__global__ void k_vtable_rep(const uint32_t* ids, uint32_t n, const uint32_t* table, uint32_t mask, uint32_t* rep, uint32_t* flag)
{
	for (uint32_t v = blockIdx.x * kThreads + threadIdx.x; v < n; v += gridDim.x * kThreads)
	{
		const uint32_t id = ids[v];
		uint32_t slot = mix32(id) & mask, r = v;
		for (uint32_t probe = 0; probe <= mask; ++probe)
		{
			const uint32_t e = table[slot];
			if (e == kNone)
				break;
			if (ids[e] == id)
			{
				r = e;
				break;
			}
			slot = (slot + 1) & mask;
		}
		rep[v] = r;
		flag[v] = r == v ? 1u : 0u;
	}
}

// step 3: cell numbers are the ranks of the representatives in vertex order
__global__ void k_cells(const uint32_t* rep, const uint32_t* scan, uint32_t n, uint32_t* cells, uint32_t* cell_first)
{
	for (uint32_t v = blockIdx.x * kThreads + threadIdx.x; v < n; v += gridDim.x * kThreads)
	{
		const uint32_t c = scan[rep[v]];
		cells[v] = c;
		if (rep[v] == v)
			cell_first[c] = v;
	}
}

// fillCellQuadrics (src/simplifier.cpp:2169-2199), step 1: the key of entry 3t + k is the cell of
// the corner that adds triangle t's quadric to it (only corner 0 when the triangle lies in one
// cell); other entries get the key cell_count and sort to the end.  A bit per triangle says that it
// lies in one cell
__global__ void k_cell_entries(const uint32_t* idx, uint32_t tris, const uint32_t* cells, uint32_t cell_count, uint32_t* keys, uint64_t* single_bits)
{
	for (uint32_t t = blockIdx.x * kThreads + threadIdx.x; t < tris; t += gridDim.x * kThreads)
	{
		const uint32_t c0 = cells[idx[3 * t + 0]], c1 = cells[idx[3 * t + 1]], c2 = cells[idx[3 * t + 2]];
		const bool single = c0 == c1 && c0 == c2;
		const uint64_t bits = __ballot(single);
		if (__lane_id() == 0)
			single_bits[t >> 6] = bits;
		keys[3 * t + 0] = c0;
		keys[3 * t + 1] = single ? cell_count : c1;
		keys[3 * t + 2] = single ? cell_count : c2;
	}
}

// step 2: the start of each cell's run in the sorted keys (lower bound), off[cell_count] = the
// number of entries that add to a cell
__global__ void k_cell_runs(const uint32_t* keys, uint32_t n, uint32_t cell_count, uint32_t* off)
{
	for (uint32_t c = blockIdx.x * kThreads + threadIdx.x; c <= cell_count; c += gridDim.x * kThreads)
	{
		uint32_t lo = 0, hi = n;
		while (lo < hi)
		{
			const uint32_t mid = lo + (hi - lo) / 2;
			if (keys[mid] < c)
				lo = mid + 1;
			else
				hi = mid;
		}
		off[c] = lo;
	}
}

// step 3: each cell sums its entries' face quadrics from zero in entry order (the stable sort kept
// the reference's (triangle, corner) order; a triangle with corners in two or three cells adds the
// same weight-1 quadric to each, one inside a single cell adds weight 3).  kLanes lanes have a cell:
// each forms the quadric of one entry, then the first 12 add up one component each, one entry after
// the other as the order asks.  The quadrics of all triangles in memory, gathered by one lane per
// cell, took 105 us for 1.3 million triangles in 20 thousand cells against 49.
template <int kLanes>
__global__ void __launch_bounds__(kThreads) k_cell_quadrics(const uint32_t* vals, const uint32_t* off, uint32_t cell_count, const uint32_t* idx,
                                                            const uint64_t* single_bits, const float4* pos, Quad* cq)
{
	constexpr uint32_t kCells = kThreads / kLanes;
	__shared__ Quad face[kThreads];
	const uint32_t lane = threadIdx.x % kLanes;
	Quad* mine = face + (threadIdx.x - lane);
	for (uint32_t c = blockIdx.x * kCells + threadIdx.x / kLanes; c < cell_count; c += gridDim.x * kCells)
	{
		const uint32_t end = off[c + 1];
		float sum = 0.f;
		for (uint32_t p0 = off[c]; p0 < end; p0 += kLanes)
		{
			const uint32_t n = end - p0 < (uint32_t)kLanes ? end - p0 : (uint32_t)kLanes;
			if (lane < n)
			{
				const uint32_t t = vals[p0 + lane] / 3;
				const uint32_t i0 = idx[3 * t + 0], i1 = idx[3 * t + 1], i2 = idx[3 * t + 2];
				const bool single = single_bits[t >> 6] >> (t & 63) & 1;
				Quad F;
				quad_from_triangle(F, load_pos(pos, i0), load_pos(pos, i1), load_pos(pos, i2), single ? 3.f : 1.f);
				store_quad(mine, lane, F);
			}
			wave_fence();
			if (lane < sizeof(Quad) / sizeof(float))
			{
				const float* f = reinterpret_cast<const float*>(mine) + lane;
				if (n == (uint32_t)kLanes)
				{
#pragma unroll
					for (int u = 0; u < kLanes; ++u)
						sum += f[u * (sizeof(Quad) / sizeof(float))];
				}
				else
					for (uint32_t u = 0; u < n; ++u)
						sum += f[u * (sizeof(Quad) / sizeof(float))];
			}
			wave_fence();
		}
		if (lane < sizeof(Quad) / sizeof(float))
			reinterpret_cast<float*>(cq + c)[lane] = sum;
	}
}

// fillCellRemap (src/simplifier.cpp:2237-2254), step 1: the smallest (error, vertex) per cell
// over vertices with a non-NaN error (errors are non-negative, so their bits order like them).
// Neighbouring lanes of one cell take their minimum first, and a minimum that is no smaller than
// what the cell has leaves it alone: atomics on one address come one after the other.
__global__ void k_cell_best(const uint32_t* cells, const Quad* cq, const float4* pos, uint32_t n, unsigned long long* best)
{
	for (uint32_t v = blockIdx.x * kThreads + threadIdx.x; v < n; v += gridDim.x * kThreads)
	{
		const uint32_t c = cells[v];
		const float e = quad_error(load_quad(cq, c), load_pos(pos, v));
		unsigned long long key = e == e ? ((unsigned long long)__float_as_uint(e) << 32) | v : ~0ull;
		const uint32_t lane = __lane_id();
		const uint64_t active = __ballot(true);
#pragma unroll
		for (int o = 1; o < 64; o <<= 1)
		{
			const unsigned long long k = __shfl_down(key, o, 64);
			const uint32_t kc = __shfl_down(c, o, 64);
			const bool there = lane + o < 64 && (active >> (lane + o) & 1);
			key = there && kc == c && k < key ? k : key;
		}
		const uint32_t left = __shfl_up(c, 1, 64);
		if ((lane && left == c) || key == ~0ull)
			continue;
		if (key < __hip_atomic_load(&best[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
			atomicMin(&best[c], key);
	}
}

// step 2: the sequential scan keeps the cell's first vertex when its error is NaN (no comparison
// with NaN replaces it), else the first vertex of smallest error; the result error is the
// largest non-NaN cell error
__global__ void k_cell_final(const unsigned long long* best, const uint32_t* cell_first, const Quad* cq, const float4* pos, uint32_t cell_count,
                             uint32_t* cell_remap, uint32_t* error_bits)
{
	uint32_t largest = 0;
	for (uint32_t c = blockIdx.x * kThreads + threadIdx.x; c < cell_count; c += gridDim.x * kThreads)
	{
		const uint32_t first = cell_first[c];
		const float e0 = quad_error(load_quad(cq, c), load_pos(pos, first));
		if (e0 != e0)
		{
			cell_remap[c] = first;
			continue;
		}
		const unsigned long long b = best[c];
		cell_remap[c] = (uint32_t)b;
		const uint32_t bits = (uint32_t)(b >> 32);
		largest = bits > largest ? bits : largest;
	}
	for (int o = 32; o > 0; o >>= 1)
	{
		const uint32_t other = __shfl_xor(largest, o, 64);
		largest = other > largest ? other : largest;
	}
	if (__lane_id() == 0 && largest)
		atomicMax(error_bits, largest);
}

// filterTriangles (src/simplifier.cpp:2282-2325), step 1: the canonical triple of each triangle
// over three distinct cells (cell vertices, rotated so the smallest leads)
__global__ void k_tri_canon(const uint32_t* idx, uint32_t tris, const uint32_t* cells, const uint32_t* cell_remap, uint4* tri)
{
	for (uint32_t t = blockIdx.x * kThreads + threadIdx.x; t < tris; t += gridDim.x * kThreads)
	{
		const uint32_t c0 = cells[idx[3 * t + 0]], c1 = cells[idx[3 * t + 1]], c2 = cells[idx[3 * t + 2]];
		uint4 r = make_uint4(0, 0, 0, 0);
		if (c0 != c1 && c0 != c2 && c1 != c2)
		{
			uint32_t a = cell_remap[c0], b = cell_remap[c1], c = cell_remap[c2];
			if (b < a && b < c)
			{
				const uint32_t x = a;
				a = b, b = c, c = x;
			}
			else if (c < a && c < b)
			{
				const uint32_t x = c;
				c = b, b = a, a = x;
			}
			r = make_uint4(a, b, c, 1u);
		}
		tri[t] = r;
	}
}

__device__ __forceinline__ uint32_t tri_hash(uint4 r)
{
	return mix32(r.x * 0x9e3779b1u ^ mix32(r.y) ^ mix32(r.z * 0x85ebca6bu));
}

__device__ __forceinline__ bool same_tri(uint4 a, uint4 b)
{
	return a.x == b.x && a.y == b.y && a.z == b.z;
}

// step 2: the table slot of a triple ends holding its first triangle
__global__ void k_tri_insert(const uint4* tri, uint32_t tris, uint32_t* table, uint32_t mask)
{
	for (uint32_t t = blockIdx.x * kThreads + threadIdx.x; t < tris; t += gridDim.x * kThreads)
	{
		const uint4 r = tri[t];
		if (!r.w)
			continue;
		uint32_t slot = tri_hash(r) & mask;
		for (uint32_t probe = 0; probe <= mask; ++probe)
		{
			const uint32_t old = atomicCAS(&table[slot], kNone, t);
			if (old == kNone)
				break;
			if (same_tri(tri[old], r))
			{
				atomicMin(&table[slot], t);
				break;
			}
			slot = (slot + 1) & mask;
		}
	}
}

// step 3: a triangle is kept when it is the first of its triple
__global__ void k_tri_keep(const uint4* tri, uint32_t tris, const uint32_t* table, uint32_t mask, uint32_t* keep)
{
	for (uint32_t t = blockIdx.x * kThreads + threadIdx.x; t < tris; t += gridDim.x * kThreads)
	{
		const uint4 r = tri[t];
		uint32_t k = 0;
		if (r.w)
		{
			uint32_t slot = tri_hash(r) & mask;
			for (uint32_t probe = 0; probe <= mask; ++probe)
			{
				const uint32_t e = table[slot];
				if (e == kNone)
					break;
				if (same_tri(tri[e], r))
				{
					k = e == t ? 1u : 0u;
					break;
				}
				slot = (slot + 1) & mask;
			}
		}
		keep[t] = k;
	}
}

// step 4: kept triangles in input order, and the result error to host memory
__global__ void k_tri_write(const uint4* tri, const uint32_t* keep, const uint32_t* pos_out, uint32_t tris, uint32_t* destination,
                            const uint32_t* error_bits, uint32_t* host_error)
{
	if (blockIdx.x == 0 && threadIdx.x == 0)
		*host_error = *error_bits;
	for (uint32_t t = blockIdx.x * kThreads + threadIdx.x; t < tris; t += gridDim.x * kThreads)
	{
		if (!keep[t])
			continue;
		const uint4 r = tri[t];
		const uint32_t o = pos_out[t] * 3;
		destination[o + 0] = r.x;
		destination[o + 1] = r.y;
		destination[o + 2] = r.z;
	}
}

static float cell_scale_of(int grid_size)
{
	return (float)(grid_size - 1);
}

void launch_sloppy_count(hipStream_t s, const SloppyBuffers& b, int grid_size, int second_grid_size)
{
	const uint32_t tris = b.index_count / 3;
	const unsigned int groups = std::min(div_up(tris ? tris : 1, kCountThreads), kCountGroups);
	const float first = cell_scale_of(grid_size), second = cell_scale_of(second_grid_size);
	unsigned long long* parts = reinterpret_cast<unsigned long long*>(b.count_parts);
	if (second_grid_size)
		k_sloppy_count<2><<<groups, kCountThreads, 0, s>>>(b.indices, tris, b.pos, b.lock, first, second, parts, b.count_done, b.host_counts);
	else
		k_sloppy_count<1><<<groups, kCountThreads, 0, s>>>(b.indices, tris, b.pos, b.lock, first, 0.f, parts, b.count_done, b.host_counts);
}

size_t sloppy_count_parts()
{
	return kCountGroups;
}

void launch_sloppy_cells(hipStream_t s, const SloppyBuffers& b, int grid_size, uint32_t* host_cell_count)
{
	const uint32_t n = b.vertex_count;
	k_sloppy_ids<<<grid_for(n), kThreads, 0, s>>>(b.pos, b.lock, n, cell_scale_of(grid_size), b.ids);
	fill_u32(s, b.vtable, kNone, b.vtable_size);
	k_vtable_insert<<<grid_for(n), kThreads, 0, s>>>(b.ids, n, b.vtable, b.vtable_size - 1);
	k_vtable_rep<<<grid_for(n), kThreads, 0, s>>>(b.ids, n, b.vtable, b.vtable_size - 1, b.rep, b.cell_scan);
	scan_exclusive(s, b.cell_scan, b.cell_scan, n, nullptr, host_cell_count, b.scan_temp);
	k_cells<<<grid_for(n), kThreads, 0, s>>>(b.rep, b.cell_scan, n, b.cells, b.cell_first);
}

static int bits_for(uint32_t max_value)
{
	int bits = 1;
	while (bits < 32 && (max_value >> bits) != 0)
		++bits;
	return bits;
}

void launch_sloppy_quadrics(hipStream_t s, const SloppyBuffers& b, uint32_t cell_count)
{
	const uint32_t tris = b.index_count / 3, n = b.vertex_count;
	if (tris)
	{
		k_cell_entries<<<grid_for(tris), kThreads, 0, s>>>(b.indices, tris, b.cells, cell_count, b.entry_keys, b.single_bits);
		radix_sort_pairs(s, b.entry_keys, b.entry_vals, b.entry_keys_alt, b.entry_vals_alt, 3 * (size_t)tris, nullptr, bits_for(cell_count),
		                 b.sort_temp, true);
	}
	k_cell_runs<<<grid_for((size_t)cell_count + 1), kThreads, 0, s>>>(b.entry_keys, 3 * tris, cell_count, b.cell_off);
	// 16 lanes a cell, a wavefront for each where the cells are few and long
	if (3 * (size_t)tris / cell_count < kLongCell)
		k_cell_quadrics<16><<<grid_for(16 * (size_t)cell_count), kThreads, 0, s>>>(b.entry_vals, b.cell_off, cell_count, b.indices, b.single_bits, b.pos, b.cq);
	else
		k_cell_quadrics<64><<<grid_for(64 * (size_t)cell_count), kThreads, 0, s>>>(b.entry_vals, b.cell_off, cell_count, b.indices, b.single_bits, b.pos, b.cq);
	fill_u32(s, reinterpret_cast<uint32_t*>(b.best), kNone, 2 * (size_t)cell_count);
	k_cell_best<<<grid_for(n), kThreads, 0, s>>>(b.cells, b.cq, b.pos, n, reinterpret_cast<unsigned long long*>(b.best));
	k_cell_final<<<grid_for(cell_count), kThreads, 0, s>>>(reinterpret_cast<const unsigned long long*>(b.best), b.cell_first, b.cq, b.pos, cell_count,
	                                                       b.cell_remap, b.error_bits);
}

void launch_sloppy_filter(hipStream_t s, const SloppyBuffers& b, uint32_t* destination, uint32_t* host_kept, uint32_t* host_error)
{
	const uint32_t tris = b.index_count / 3;
	k_tri_canon<<<grid_for(tris), kThreads, 0, s>>>(b.indices, tris, b.cells, b.cell_remap, b.tri);
	fill_u32(s, b.ttable, kNone, b.ttable_size);
	k_tri_insert<<<grid_for(tris), kThreads, 0, s>>>(b.tri, tris, b.ttable, b.ttable_size - 1);
	k_tri_keep<<<grid_for(tris), kThreads, 0, s>>>(b.tri, tris, b.ttable, b.ttable_size - 1, b.keep);
	// the entry arrays are free again: the exclusive scan of the keep flags goes to entry_keys
	scan_exclusive(s, b.keep, b.entry_keys, tris, nullptr, host_kept, b.scan_temp);
	k_tri_write<<<grid_for(tris), kThreads, 0, s>>>(b.tri, b.keep, b.entry_keys, tris, destination, b.error_bits, host_error);
}

} // namespace mhip
