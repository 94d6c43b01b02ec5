// Setup kernels of the edge-collapse simplifier: sparse remap, position remap and wedge
// rings, corner CSR, vertex classification, rescale, and the ordered quadric gathers.
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

// number of bits needed to hold values < n
static int key_bits(size_t n)
{
	int b = 0;
	while (b < 32 && ((size_t)1 << b) < n)
		++b;
	return b;
}

// ------------------------------------------------------------------------------------------
// input validation: any index >= vertex_count sets the flag

__global__ void k_check_indices(const uint32_t* ib, size_t n, size_t limit, uint32_t* flag)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	bool bad = j < n && ib[j] >= limit;
	if (__ballot(bad) && __lane_id() == 0)
		atomicOr(flag, 1u);
}

void launch_check_indices(hipStream_t s, const uint32_t* ib, size_t index_count, size_t vertex_count, uint32_t* flag)
{
	if (index_count)
		k_check_indices<<<grid_for(index_count), kThreads, 0, s>>>(ib, index_count, vertex_count, flag);
}

// the device scalars of a call (the box reductions empty, everything else 0) and the n words at
// `zeroed`
__global__ void __launch_bounds__(kThreads) k_call_init(CallScalars* sc, uint32_t* zeroed, size_t n)
{
	for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (size_t)gridDim.x * kThreads)
		zeroed[i] = 0;
	if (blockIdx.x)
		return;
	uint32_t* w = reinterpret_cast<uint32_t*>(sc);
	for (size_t i = threadIdx.x; i < sizeof(CallScalars) / 4; i += kThreads)
		w[i] = 0;
	__syncthreads();
	if (threadIdx.x < 3)
		sc->box_min[threadIdx.x] = ~0ull;
}

void launch_call_init(hipStream_t s, CallScalars* sc, uint32_t* zeroed, size_t n)
{
	const unsigned int grid = grid_for(n);
	k_call_init<<<grid < 1024 ? grid : 1024, kThreads, 0, s>>>(sc, zeroed, n);
}

// the call's copy of the indices with the range check; with `counts`, each corner also takes its
// slot in its vertex's list (order_corners below)
__global__ void k_load_indices(const uint32_t* in, uint32_t* out, size_t n, size_t limit, uint32_t* counts, uint32_t* slot, uint32_t* flag)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	const uint32_t v = j < n ? in[j] : 0;
	const bool bad = j < n && v >= limit;
	if (__ballot(bad) && __lane_id() == 0)
		atomicOr(flag, 1u);
	if (j >= n)
		return;
	out[j] = v;
	if (counts && !bad)
		slot[j] = atomicAdd(&counts[v], 1u);
}

void launch_load_indices(hipStream_t s, const uint32_t* in, uint32_t* out, size_t index_count, size_t vertex_count, uint32_t* counts, uint32_t* slot,
                         uint32_t* flag)
{
	if (index_count)
		k_load_indices<<<grid_for(index_count), kThreads, 0, s>>>(in, out, index_count, vertex_count, counts, slot, flag);
}

// ------------------------------------------------------------------------------------------
// sparse remap (src/simplifier.cpp:242-294): dense id = order of first occurrence

__global__ void k_first_occurrence(const uint32_t* ib, size_t n, uint32_t* first)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (j < n)
		atomicMin(&first[ib[j]], (uint32_t)j);
}

__global__ void k_first_flags(const uint32_t* ib, size_t n, const uint32_t* first, uint32_t* flags)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (j < n)
		flags[j] = first[ib[j]] == (uint32_t)j;
}

__global__ void k_sparse_write(const uint32_t* ib_in, uint32_t* ib_out, size_t n, const uint32_t* first, const uint32_t* dense, uint32_t* sparse_remap)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= n)
		return;
	uint32_t v = ib_in[j];
	uint32_t f = first[v];
	if (f == (uint32_t)j)
		sparse_remap[dense[j]] = v;
	ib_out[j] = dense[f];
}

void launch_sparse_remap(hipStream_t s, const uint32_t* indices_in, uint32_t* indices_out, size_t index_count, size_t vertex_count,
                         uint32_t* first, uint32_t* flags, uint32_t* dense, uint32_t* sparse_remap, uint32_t* unique_count, uint32_t* temp)
{
	fill_u32(s, first, kNone, vertex_count);
	if (index_count == 0)
	{
		HIP_CHECK(hipMemsetAsync(unique_count, 0, sizeof(uint32_t), s));
		return;
	}
	k_first_occurrence<<<grid_for(index_count), kThreads, 0, s>>>(indices_in, index_count, first);
	k_first_flags<<<grid_for(index_count), kThreads, 0, s>>>(indices_in, index_count, first, flags);
	scan_exclusive(s, flags, dense, index_count, nullptr, unique_count, temp);
	k_sparse_write<<<grid_for(index_count), kThreads, 0, s>>>(indices_in, indices_out, index_count, first, dense, sparse_remap);
}

// ------------------------------------------------------------------------------------------
// positions, their box (the rescale's, src/simplifier.cpp:549-603) and the empty hash table in one
// sweep.  The reference keeps the first element (in vertex order) that compares below the running
// minimum, so among +0/-0 ties the earliest wins: reduce (ordered key, index) pairs, then read the
// winning element's own bits.  The workgroup that finishes last turns the box into the extent.

__device__ __forceinline__ float comp(float4 p, int k)
{
	return k == 0 ? p.x : (k == 1 ? p.y : p.z);
}

constexpr int kGatherThreads = 512;
constexpr unsigned int kGatherBlocks = 512;

__global__ void __launch_bounds__(kGatherThreads) k_gather_positions(const float* positions, size_t stride, const uint32_t* sparse_remap, float4* praw,
                                                                     size_t n, uint32_t* table, size_t table_size, CallScalars* sc)
{
	constexpr int kWaves = kGatherThreads / 64;
	__shared__ uint64_t red[6][kWaves];
	__shared__ bool s_last;
	const size_t step = (size_t)gridDim.x * kGatherThreads, first = (size_t)blockIdx.x * kGatherThreads + threadIdx.x;
	for (size_t i = first; i < table_size; i += step)
		table[i] = kNone;
	uint64_t mn[3], mx[3];
#pragma unroll
	for (int k = 0; k < 3; ++k)
	{
		mn[k] = ~0ull;
		mx[k] = 0ull;
	}
	for (size_t i = first; i < n; i += step)
	{
		const size_t ri = sparse_remap ? sparse_remap[i] : i;
		const float* p = positions + ri * stride;
		const float c[3] = {p[0], p[1], p[2]};
		praw[i] = make_float4(c[0], c[1], c[2], 0.f);
#pragma unroll
		for (int k = 0; k < 3; ++k)
		{
			if (c[k] != c[k])
				continue;
			const uint64_t key = (uint64_t)ordered_key(c[k]) << 32;
			const uint64_t a = key | (uint64_t)(uint32_t)i;
			const uint64_t b = key | (uint64_t)(0xffffffffu - (uint32_t)i);
			mn[k] = a < mn[k] ? a : mn[k];
			mx[k] = b > mx[k] ? b : mx[k];
		}
	}
	const int wave = threadIdx.x >> 6;
#pragma unroll
	for (int k = 0; k < 3; ++k)
	{
		const uint64_t a = wave_min64(mn[k]), b = wave_max64(mx[k]);
		if (__lane_id() == 0)
		{
			red[k][wave] = a;
			red[3 + k][wave] = b;
		}
	}
	__syncthreads();
	if (threadIdx.x < 3)
	{
		const int k = threadIdx.x;
		uint64_t a = ~0ull, b = 0ull;
		for (int w = 0; w < kWaves; ++w)
		{
			a = red[k][w] < a ? red[k][w] : a;
			b = red[3 + k][w] > b ? red[3 + k][w] : b;
		}
		// a workgroup inside the box found so far adds nothing (same-address atomics serialise)
		if (a < __hip_atomic_load(&sc->box_min[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
			atomicMin((unsigned long long*)&sc->box_min[k], (unsigned long long)a);
		if (b > __hip_atomic_load(&sc->box_max[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
			atomicMax((unsigned long long*)&sc->box_max[k], (unsigned long long)b);
	}
	// this workgroup's part of the box, before it counts itself done
	wait_for_memory();
	__syncthreads();
	if (threadIdx.x == 0)
		s_last = atomicAdd(&sc->box_done, 1u) + 1 == gridDim.x;
	__syncthreads();
	if (!s_last || threadIdx.x)
		return;
	float lo[3], hi[3];
	for (int k = 0; k < 3; ++k)
	{
		const uint64_t a = __hip_atomic_load(&sc->box_min[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		const uint64_t b = __hip_atomic_load(&sc->box_max[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		lo[k] = FLT_MAX;
		hi[k] = -FLT_MAX;
		// the caller's own bits of the winning element
		auto value = [&](uint32_t i) { return positions[(size_t)(sparse_remap ? sparse_remap[i] : i) * stride + k]; };
		if (a != ~0ull)
		{
			const float v = value((uint32_t)a);
			lo[k] = FLT_MAX > v ? v : FLT_MAX;
		}
		if (b != 0ull)
		{
			const float v = value(0xffffffffu - (uint32_t)b);
			hi[k] = -FLT_MAX < v ? v : -FLT_MAX;
		}
	}
	float extent = 0.f;
	extent = (hi[0] - lo[0]) < extent ? extent : (hi[0] - lo[0]);
	extent = (hi[1] - lo[1]) < extent ? extent : (hi[1] - lo[1]);
	extent = (hi[2] - lo[2]) < extent ? extent : (hi[2] - lo[2]);
	for (int k = 0; k < 3; ++k)
		sc->lo[k] = lo[k];
	sc->extent = extent;
	sc->scale = extent == 0 ? 0.f : 1.f / extent;
}

void launch_gather_positions(hipStream_t s, Mesh& m, const float* positions, size_t stride_floats, const uint32_t* sparse_remap, uint32_t* table,
                             size_t table_size)
{
	const size_t n = m.vertex_count;
	const unsigned int grid = div_up(n ? n : 1, kGatherThreads);
	k_gather_positions<<<grid < kGatherBlocks ? grid : kGatherBlocks, kGatherThreads, 0, s>>>(positions, stride_floats, sparse_remap, m.praw, n, table,
	                                                                                        table_size, m.sc);
}

__device__ __forceinline__ float4 rescaled(float4 p, const CallScalars* sc)
{
	const float scale = sc->scale;
	return make_float4((p.x - sc->lo[0]) * scale, (p.y - sc->lo[1]) * scale, (p.z - sc->lo[2]) * scale, 0.f);
}

__global__ void k_rescale(const float4* praw, size_t n, const CallScalars* sc, float4* pos)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		pos[i] = rescaled(praw[i], sc);
}

void launch_rescale(hipStream_t s, Mesh& m)
{
	if (m.vertex_count)
		k_rescale<<<grid_for(m.vertex_count), kThreads, 0, s>>>(m.praw, m.vertex_count, m.sc, m.pos);
}

// ------------------------------------------------------------------------------------------
// k_corner_order compares every corner of a list of more than kNet with every other, in the wavefront
// that has the list: pair_steps of its loop, one list after the other.  Where one wavefront's lists come
// to more than kPairSteps, the mesh's lists are made by sorts instead, and the open edges of all lists
// above kNet by a table, linear in the corners.  The two meet at 1000-1400 steps (calls on a hub of 400
// corners, 2500 steps, beside 200 triangles 835 us by pairs, 699 sorted; beside 320 thousand 2657 and
// 2533; on a hub of 200, 625 steps, 565 and 570, 2483 and 2551; 64 positions of 140 corners each, whose
// primaries are neighbours: 1441 us by pairs).  By pairs, the 300 thousand corners that padding with
// (0,0,0) triangles gives a vertex would take half a minute.
constexpr int kNet = 8; // corners that the sorting network takes
constexpr uint32_t kPairSteps = 1280;
constexpr uint32_t kLongVertexLists = 1, kLongClassLists = 2; // of CallScalars::long_lists

__device__ __forceinline__ uint32_t pair_steps(uint32_t corners)
{
	// capped far beyond kPairSteps, so that the sum over a wavefront stays in 32 bits
	const uint32_t c = corners < 4096 ? corners : 4096;
	return c <= kNet ? 0 : (c <= 64 ? c : c * c / 64);
}

// position remap (src/simplifier.cpp:111-240).  remap[i] = lowest index whose xyz compare
// equal as floats (+0 == -0; NaN equals nothing).  Linear-probing table keyed by the
// canonical bits; a slot holds one equality class, and atomicMin leaves its lowest index.

__device__ __forceinline__ bool has_nan(float4 p)
{
	return p.x != p.x || p.y != p.y || p.z != p.z;
}

__device__ __forceinline__ uint32_t canon(float f)
{
	uint32_t u = __float_as_uint(f);
	return u == 0x80000000u ? 0u : u;
}

__device__ __forceinline__ uint32_t pos_hash(float4 p)
{
	uint64_t h = (uint64_t)canon(p.x) * 0x9E3779B97F4A7C15ull;
	h ^= (uint64_t)canon(p.y) * 0xC2B2AE3D27D4EB4Full;
	h ^= (uint64_t)canon(p.z) * 0x165667B19E3779F9ull;
	h ^= h >> 29;
	return (uint32_t)h ^ (uint32_t)(h >> 32);
}

__device__ __forceinline__ bool same_pos(float4 a, float4 b)
{
	return a.x == b.x && a.y == b.y && a.z == b.z;
}

__global__ void k_hash_insert(const float4* pos, size_t n, uint32_t* table, uint32_t mask)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	float4 p = pos[i];
	if (has_nan(p))
		return;
	uint32_t slot = pos_hash(p) & mask;
	for (uint32_t probe = 0; probe <= mask; ++probe)
	{
		uint32_t old = atomicCAS(&table[slot], kNone, (uint32_t)i);
		if (old == kNone)
			return;
		if (same_pos(pos[old], p))
		{
			atomicMin(&table[slot], (uint32_t)i);
			return;
		}
		slot = (slot + 1) & mask;
	}
}

// each vertex's primary, its rescaled position, a wedge ring of its own and no pending ranks; sc
// counts the secondaries and says whether the corner lists are long (kPairSteps).  By vertex, a
// wavefront here holds the counts of one there; by class, every secondary adds its corners to its
// class, and what that adds to the steps of the class to those of the wavefront with the primary
__global__ void __launch_bounds__(kThreads) k_hash_lookup(const float4* praw, size_t n, const uint32_t* table, uint32_t mask, uint32_t* remap,
                                                          uint32_t* wedge, float4* pos, ulonglong2* pend0, ulonglong2* pend1, const uint32_t* counts,
                                                          uint32_t* class_extra, uint32_t* class_steps, CallScalars* sc)
{
	__shared__ uint32_t secondaries;
	if (threadIdx.x == 0)
		secondaries = 0;
	__syncthreads();
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	uint32_t result = (uint32_t)i;
	uint32_t corners = 0, own_steps = 0;
	bool long_class = false;
	if (i < n)
	{
		corners = counts[i];
		const float4 p = praw[i];
		if (!has_nan(p))
		{
			uint32_t slot = pos_hash(p) & mask;
			for (uint32_t probe = 0; probe <= mask; ++probe)
			{
				uint32_t e = table[slot];
				if (e == kNone)
					break; // unreachable: i itself was inserted
				if (e == (uint32_t)i || same_pos(praw[e], p))
				{
					result = e;
					break;
				}
				slot = (slot + 1) & mask;
			}
		}
		remap[i] = result;
		wedge[i] = (uint32_t)i;
		pos[i] = rescaled(p, sc);
		// round minima start as "no entry" (tag of epoch 0, rank all-ones)
		pend0[i] = make_ulonglong2(~0ull, ~0ull);
		pend1[i] = make_ulonglong2(~0ull, ~0ull);
		own_steps = pair_steps(corners);
		if (result != (uint32_t)i && corners)
		{
			const uint32_t before = counts[result] + atomicAdd(&class_extra[result], corners);
			const uint32_t more = pair_steps(before + corners) - pair_steps(before);
			long_class = more && atomicAdd(&class_steps[result / 64], more) + more > kPairSteps;
		}
	}
	if (__ballot(own_steps != 0))
	{
		// the primaries' own part of the classes' steps, and this wavefront's by vertex
		uint32_t primary = result == (uint32_t)i ? own_steps : 0;
		for (int o = 32; o > 0; o >>= 1)
		{
			own_steps += __shfl_xor(own_steps, o, 64);
			primary += __shfl_xor(primary, o, 64);
		}
		if (__lane_id() == 0)
		{
			long_class |= primary && atomicAdd(&class_steps[i / 64], primary) + primary > kPairSteps;
			if (own_steps > kPairSteps)
				atomicOr(&sc->long_lists, kLongVertexLists);
		}
	}
	if (__ballot(long_class) && __lane_id() == 0)
		atomicOr(&sc->long_lists, kLongClassLists);
	const uint64_t second = __ballot(result != (uint32_t)i);
	if (second && __lane_id() == 0)
		atomicAdd(&secondaries, (uint32_t)__popcll(second));
	__syncthreads();
	if (threadIdx.x == 0 && secondaries)
		atomicAdd(&sc->secondary_count, secondaries);
}

void launch_position_remap(hipStream_t s, Mesh& m, uint32_t* table, size_t table_size, const uint32_t* counts, uint32_t* class_extra,
                           uint32_t* class_steps)
{
	size_t n = m.vertex_count;
	if (!n)
		return;
	k_hash_insert<<<grid_for(n), kThreads, 0, s>>>(m.praw, n, table, (uint32_t)(table_size - 1));
	k_hash_lookup<<<grid_for(n), kThreads, 0, s>>>(m.praw, n, table, (uint32_t)(table_size - 1), m.remap, m.wedge, m.pos,
	                                               reinterpret_cast<ulonglong2*>(m.pend[0]), reinterpret_cast<ulonglong2*>(m.pend[1]), counts, class_extra,
	                                               class_steps, m.sc);
}

// wedge rings: for a class r < a_1 < ... < a_m, wedge[r] = a_m, wedge[a_k] = a_{k-1}, wedge[a_1] = r
// (the list buildPositionRemap forms by inserting each secondary after its primary,
// src/simplifier.cpp:229-239).  Secondaries are compacted in index order, stably sorted by
// class, and linked to their predecessor.

__global__ void k_secondary_flags(const uint32_t* remap, size_t n, uint32_t* flags)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		flags[i] = remap[i] != (uint32_t)i;
}

__global__ void k_secondary_compact(const uint32_t* remap, size_t n, const uint32_t* flags, const uint32_t* offs, uint32_t* keys, uint32_t* vals)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n && flags[i])
	{
		keys[offs[i]] = remap[i];
		vals[offs[i]] = (uint32_t)i;
	}
}

__global__ void k_wedge_link(const uint32_t* keys, const uint32_t* vals, size_t n, uint32_t* wedge)
{
	size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (p >= n)
		return;
	uint32_t r = keys[p];
	uint32_t i = vals[p];
	wedge[i] = (p > 0 && keys[p - 1] == r) ? vals[p - 1] : r;
	if (p + 1 == n || keys[p + 1] != r)
		wedge[r] = i;
}

void launch_wedges(hipStream_t s, Mesh& m, size_t secondaries, uint32_t* flags, uint32_t* scratch_a, uint32_t* scratch_b, uint32_t* scratch_c,
                   uint32_t* scratch_d)
{
	size_t n = m.vertex_count;
	if (!secondaries)
		return; // every ring is a vertex of its own
	k_secondary_flags<<<grid_for(n), kThreads, 0, s>>>(m.remap, n, flags);
	scan_exclusive(s, flags, scratch_a, n, nullptr, nullptr, m.temp);
	k_secondary_compact<<<grid_for(n), kThreads, 0, s>>>(m.remap, n, flags, scratch_a, scratch_b, scratch_c);
	radix_sort_pairs(s, scratch_b, scratch_c, scratch_d, scratch_a, secondaries, nullptr, key_bits(n), m.temp);
	k_wedge_link<<<grid_for(secondaries), kThreads, 0, s>>>(scratch_b, scratch_c, secondaries, m.wedge);
}

// ------------------------------------------------------------------------------------------
// Corner lists: each vertex's (or class's) corners in corner order, the order in which the reference
// visits its triangles.  One atomic per corner hands it a slot in its list, in any order; the scan
// of the counts and a placement make the lists, and each is then put in order where it lies: up to
// eight corners by a sorting network in registers, more by the wavefront, every corner's place the
// number of smaller ones.  (Sorting all corners by vertex with three radix digits took 370 us for
// the 3.9 M of icosphere L8 and the open edges 140; lists and open edges now take 300 with the index
// copy and check, 250 of it the count's and the placement's scattered words.)  Meshes with long lists
// (kPairSteps) do take that sort, and a table of edges answers for the open ones.

__global__ void k_corner_count(const uint32_t* ib, size_t n, const uint32_t* remap, uint32_t* counts, uint32_t* slot)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= n)
		return;
	uint32_t v = ib[j];
	if (remap)
		v = remap[v];
	slot[j] = atomicAdd(&counts[v], 1u);
}

__global__ void k_corner_place(const uint32_t* ib, size_t n, const uint32_t* remap, const uint32_t* off, const uint32_t* slot, uint32_t* placed)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= n)
		return;
	uint32_t v = ib[j];
	if (remap)
		v = remap[v];
	placed[off[v] + slot[j]] = (uint32_t)j;
}

struct CornerArgs
{
	const uint32_t* ib;
	const uint32_t* off;
	const uint32_t* placed;
	uint32_t* corners;
	uint32_t* openout;
	uint32_t* openinc;
	uint2* adj; // (next, prev) per listed corner, or null
	size_t n;
	uint32_t longest; // longer lists are sorted already
};

// the vertices after and before corner j in its triangle
__device__ __forceinline__ uint2 corner_neighbours(const uint32_t* ib, uint32_t j)
{
	const uint32_t t = j / 3, c = j - t * 3;
	return make_uint2(ib[t * 3 + (c == 2 ? 0 : c + 1)], ib[t * 3 + (c == 0 ? 2 : c - 1)]);
}

__device__ __forceinline__ void compare_exchange(uint32_t& a, uint32_t& b)
{
	const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
	a = lo;
	b = hi;
}

__device__ __forceinline__ uint32_t open_end(uint32_t v, bool self, uint32_t count, uint32_t last)
{
	return (self || count > 1) ? v : (count == 1 ? last : kNone);
}

// kOpen: also the open half-edges per vertex (src/simplifier.cpp:379-400): an outgoing edge v->t is
// open when t has no edge t->v, an incoming edge u->v when v has no edge v->u.  The opposite of
// either half-edge lies in a triangle around v as well, where the other vertex comes before v
// (t->v) or after it (v->u), so v's own list answers both.  Result: none, the single other endpoint,
// or v itself when there are several open edges or a self edge.
template <bool kOpen>
__global__ void __launch_bounds__(kThreads) k_corner_order(CornerArgs a)
{
	const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
	const uint32_t v = (uint32_t)i, lane = __lane_id();
	const uint32_t b = i < a.n ? a.off[i] : 0, e = i < a.n ? a.off[i + 1] : 0, len = e - b;
	if (i < a.n && len <= kNet)
	{
		uint32_t c[kNet];
#pragma unroll
		for (int q = 0; q < kNet; ++q)
			c[q] = (uint32_t)q < len ? a.placed[b + q] : kNone;
		constexpr uint8_t net[19][2] = {{0, 1}, {2, 3}, {4, 5}, {6, 7}, {0, 2}, {1, 3}, {4, 6}, {5, 7}, {1, 2}, {5, 6},
		                                {0, 4}, {3, 7}, {1, 5}, {2, 6}, {1, 4}, {3, 6}, {2, 4}, {3, 5}, {3, 4}};
#pragma unroll
		for (int k = 0; k < 19; ++k)
			compare_exchange(c[net[k][0]], c[net[k][1]]);
#pragma unroll
		for (int q = 0; q < kNet; ++q)
			if ((uint32_t)q < len)
				a.corners[b + q] = c[q];
		if (kOpen)
		{
			uint2 nb[kNet];
#pragma unroll
			for (int q = 0; q < kNet; ++q)
				nb[q] = (uint32_t)q < len ? corner_neighbours(a.ib, c[q]) : make_uint2(kNone, kNone);
			uint32_t outs = 0, out_last = kNone, ins = 0, in_last = kNone;
			bool self = false;
#pragma unroll
			for (int q = 0; q < kNet; ++q)
			{
				if ((uint32_t)q >= len)
					continue;
				if (a.adj)
					a.adj[b + q] = nb[q];
				bool opposite_out = false, opposite_in = false;
#pragma unroll
				for (int r = 0; r < kNet; ++r)
				{
					opposite_out |= nb[r].y == nb[q].x;
					opposite_in |= nb[r].x == nb[q].y;
				}
				if (nb[q].x == v)
					self = true;
				else if (!opposite_out)
				{
					outs++;
					out_last = nb[q].x;
				}
				if (nb[q].y == v)
					self = true;
				else if (!opposite_in)
				{
					ins++;
					in_last = nb[q].y;
				}
			}
			a.openout[v] = open_end(v, self, outs, out_last);
			a.openinc[v] = open_end(v, self, ins, in_last);
		}
	}
	if (kOpen && len > a.longest)
	{
		// a sorted list; k_table_edges finds its open edges, starting from none
		a.openout[v] = kNone;
		a.openinc[v] = kNone;
	}
	for (uint64_t left = __ballot(len > kNet && len <= a.longest); left; left &= left - 1)
	{
		const int from = __builtin_ctzll(left);
		const uint32_t w = __builtin_amdgcn_readlane(v, from), wb = __builtin_amdgcn_readlane(b, from), we = __builtin_amdgcn_readlane(e, from);
		uint32_t outs = 0, out_last = kNone, ins = 0, in_last = kNone;
		bool self = false;
		for (uint32_t x0 = wb; x0 < we; x0 += 64)
		{
			const bool in = x0 + lane < we;
			const uint32_t cx = in ? a.placed[x0 + lane] : kNone;
			const uint2 nx = kOpen && in ? corner_neighbours(a.ib, cx) : make_uint2(kNone, kNone);
			uint32_t place = 0;
			bool opposite_out = false, opposite_in = false;
			for (uint32_t y0 = wb; y0 < we; y0 += 64)
			{
				const bool iny = y0 + lane < we;
				const uint32_t cy = iny ? a.placed[y0 + lane] : kNone;
				const uint2 ny = kOpen && iny ? corner_neighbours(a.ib, cy) : make_uint2(kNone, kNone);
				const uint32_t m = we - y0 < 64 ? we - y0 : 64;
				for (uint32_t k = 0; k < m; ++k)
				{
					place += (uint32_t)__builtin_amdgcn_readlane(cy, k) < cx ? 1u : 0u;
					if (kOpen)
					{
						opposite_out |= (uint32_t)__builtin_amdgcn_readlane(ny.y, k) == nx.x;
						opposite_in |= (uint32_t)__builtin_amdgcn_readlane(ny.x, k) == nx.y;
					}
				}
			}
			if (in)
			{
				a.corners[wb + place] = cx;
				if (kOpen && a.adj)
					a.adj[wb + place] = nx;
			}
			if (kOpen)
			{
				const uint64_t out_mask = __ballot(in && nx.x != w && !opposite_out), in_mask = __ballot(in && nx.y != w && !opposite_in);
				self |= __ballot(in && (nx.x == w || nx.y == w)) != 0;
				if (out_mask)
					out_last = __builtin_amdgcn_readlane(nx.x, __builtin_ctzll(out_mask));
				if (in_mask)
					in_last = __builtin_amdgcn_readlane(nx.y, __builtin_ctzll(in_mask));
				outs += (uint32_t)__popcll(out_mask);
				ins += (uint32_t)__popcll(in_mask);
			}
		}
		if (kOpen && (int)lane == from)
		{
			a.openout[w] = open_end(w, self, outs, out_last);
			a.openinc[w] = open_end(w, self, ins, in_last);
		}
	}
}

// Lists by sorting, for meshes with long ones: every corner's vertex as the key, its place as the
// value, both arrays in `corners` and `keys` and the sort's other halves in the candidate lists.
// The time is linear in the corners (a sweep per byte of the vertex ids).

__global__ void k_corner_keys(const uint32_t* ib, size_t n, const uint32_t* remap, uint32_t* keys)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= n)
		return;
	const uint32_t v = ib[j];
	keys[j] = remap ? remap[v] : v;
}

static void sort_corners(hipStream_t s, Mesh& m, const uint32_t* remap, uint32_t* keys, uint32_t* corners)
{
	const size_t n = m.index_count;
	uint32_t* keys_alt = reinterpret_cast<uint32_t*>(m.list[0]);
	uint32_t* vals_alt = keys_alt + n;
	k_corner_keys<<<grid_for(n), kThreads, 0, s>>>(m.ib[0], n, remap, keys);
	radix_sort_pairs(s, keys, corners, keys_alt, vals_alt, n, nullptr, std::max(1, key_bits(m.vertex_count)), m.temp, true);
}

// Open edges of sorted lists above kNet, the rule of k_corner_order: a table holds the directed edges at
// their vertices, two per corner, and each corner looks for the opposites of its own two.  The
// candidate lists hold the table: 4 * (I + 4) slots, rounded down to a power of two, for at most I
// different edges, so that every search ends at an empty slot soon.

struct EdgeTable
{
	unsigned long long* slots; // from << 32 | to; ~0: empty
	uint32_t mask;
};

__device__ __forceinline__ uint32_t edge_hash(uint64_t edge)
{
	edge *= 0x9E3779B97F4A7C15ull;
	return (uint32_t)(edge >> 32) ^ (uint32_t)edge;
}

__device__ __forceinline__ void edge_insert(const EdgeTable& t, uint32_t from, uint32_t to)
{
	const unsigned long long edge = (unsigned long long)from << 32 | to;
	uint32_t slot = edge_hash(edge) & t.mask;
	for (uint32_t probe = 0; probe <= t.mask; ++probe)
	{
		// read before it is written: the corners of a padded list all bring the same edge
		unsigned long long old = __hip_atomic_load(&t.slots[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		if (old == ~0ull)
			old = atomicCAS(&t.slots[slot], ~0ull, edge);
		if (old == ~0ull || old == edge)
			return;
		slot = (slot + 1) & t.mask;
	}
}

__device__ __forceinline__ bool edge_known(const EdgeTable& t, uint32_t from, uint32_t to)
{
	const unsigned long long edge = (unsigned long long)from << 32 | to;
	uint32_t slot = edge_hash(edge) & t.mask;
	for (uint32_t probe = 0; probe <= t.mask; ++probe)
	{
		const unsigned long long at = t.slots[slot];
		if (at == edge)
			return true;
		if (at == ~0ull)
			return false;
		slot = (slot + 1) & t.mask;
	}
	return false;
}

// one more open edge of a vertex: the first is named, any other makes it the vertex itself
__device__ __forceinline__ void open_add(uint32_t* open, uint32_t v, uint32_t end)
{
	if (__hip_atomic_load(&open[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == v)
		return;
	if (end == v || atomicCAS(&open[v], kNone, end) != kNone)
		(void)__hip_atomic_exchange(&open[v], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <bool kInsert>
__global__ void k_table_edges(CornerArgs a, size_t n, EdgeTable t)
{
	size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= n)
		return;
	const uint32_t v = a.ib[j];
	if (a.off[v + 1] - a.off[v] <= a.longest)
		return;
	const uint2 nb = corner_neighbours(a.ib, (uint32_t)j);
	if (kInsert)
	{
		if (nb.x != v)
			edge_insert(t, v, nb.x);
		if (nb.y != v)
			edge_insert(t, nb.y, v);
		return;
	}
	if (nb.x == v || nb.y == v)
	{
		open_add(a.openout, v, v);
		open_add(a.openinc, v, v);
	}
	if (nb.x != v && !edge_known(t, nb.x, v))
		open_add(a.openout, v, nb.x);
	if (nb.y != v && !edge_known(t, v, nb.y))
		open_add(a.openinc, v, nb.y);
}

__global__ void k_list_neighbours(const uint32_t* ib, const uint32_t* corners, size_t n, uint2* adj)
{
	size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (p < n)
		adj[p] = corner_neighbours(ib, corners[p]);
}

static void table_open_edges(hipStream_t s, Mesh& m, const CornerArgs& a)
{
	const size_t n = m.index_count;
	size_t slots = 1;
	while (slots * 2 <= 4 * (n + 4) && slots < (size_t)1 << 32)
		slots *= 2;
	const EdgeTable t{reinterpret_cast<unsigned long long*>(m.list[0]), (uint32_t)(slots - 1)};
	fill_u32(s, reinterpret_cast<uint32_t*>(t.slots), kNone, 2 * slots);
	k_table_edges<true><<<grid_for(n), kThreads, 0, s>>>(a, n, t);
	k_table_edges<false><<<grid_for(n), kThreads, 0, s>>>(a, n, t);
	if (a.adj)
		k_list_neighbours<<<grid_for(n), kThreads, 0, s>>>(m.ib[0], a.corners, n, a.adj);
}

// the counts (one word per list) become offsets (one more)
static void corner_offsets(hipStream_t s, Mesh& m, uint32_t* offsets)
{
	scan_exclusive(s, offsets, offsets, m.vertex_count, nullptr, offsets + m.vertex_count, m.temp);
}

void launch_corner_count(hipStream_t s, Mesh& m, const uint32_t* remap, uint32_t* counts, uint32_t* slot)
{
	if (m.index_count)
		k_corner_count<<<grid_for(m.index_count), kThreads, 0, s>>>(m.ib[0], m.index_count, remap, counts, slot);
}

void launch_corner_lists(hipStream_t s, Mesh& m, uint32_t long_lists, bool with_adjacency, uint32_t* offsets, const uint32_t* slot, uint32_t* placed,
                         uint32_t* corners)
{
	if (!m.vertex_count)
		return;
	const bool sorted = (long_lists & kLongVertexLists) != 0;
	corner_offsets(s, m, offsets);
	if (sorted)
		sort_corners(s, m, nullptr, placed, corners);
	else if (m.index_count)
		k_corner_place<<<grid_for(m.index_count), kThreads, 0, s>>>(m.ib[0], m.index_count, nullptr, offsets, slot, placed);
	const CornerArgs a{m.ib[0],   offsets, sorted ? corners : placed, corners, m.loop[0], m.loopback[0], with_adjacency ? m.adj[1] : nullptr,
	                   m.vertex_count, sorted ? (uint32_t)kNet : kNone};
	k_corner_order<true><<<grid_for(m.vertex_count), kThreads, 0, s>>>(a);
	if (sorted)
		table_open_edges(s, m, a);
}

void launch_welded_corner_lists(hipStream_t s, Mesh& m, uint32_t long_lists, uint32_t* offsets, uint32_t* slot, uint32_t* placed, uint32_t* corners)
{
	if (!m.vertex_count)
		return;
	fill_u32(s, offsets, 0, (size_t)m.vertex_count + 1);
	launch_corner_count(s, m, m.remap, offsets, slot);
	corner_offsets(s, m, offsets);
	if (long_lists & kLongClassLists)
	{
		sort_corners(s, m, m.remap, placed, corners);
		return;
	}
	if (m.index_count)
		k_corner_place<<<grid_for(m.index_count), kThreads, 0, s>>>(m.ib[0], m.index_count, m.remap, offsets, slot, placed);
	const CornerArgs a{m.ib[0], offsets, placed, corners, nullptr, nullptr, nullptr, m.vertex_count, kNone};
	k_corner_order<false><<<grid_for(m.vertex_count), kThreads, 0, s>>>(a);
}

// hasEdge over the wedges of a, src/simplifier.cpp:345-362
__device__ __forceinline__ bool has_edge_wedged(const uint32_t* off, const uint2* adj, uint32_t a, uint32_t b, const uint32_t* remap, const uint32_t* wedge)
{
	uint32_t rb = remap[b];
	uint32_t v = a;
	do
	{
		for (uint32_t p = off[v], e = off[v + 1]; p < e; ++p)
			if (remap[adj[p].x] == rb)
				return true;
		v = wedge[v];
	} while (v != a);
	return false;
}

// classifyVertices primary rules, src/simplifier.cpp:406-470
__device__ __forceinline__ uint8_t classify_primary(const uint32_t* remap, const uint32_t* wedge, const uint32_t* loop, const uint32_t* loopback, uint32_t i)
{
	uint8_t k;
	if (wedge[i] == i)
	{
		uint32_t oi = loopback[i], oo = loop[i];
		if (oi == kNone && oo == kNone)
			k = kManifold;
		else if (oi != kNone && oo != kNone && remap[oi] == remap[oo] && oi != i)
			k = kSeam;
		else if (oi != i && oo != i)
			k = kBorder;
		else
			k = kLocked;
	}
	else if (wedge[wedge[i]] == i)
	{
		uint32_t w = wedge[i];
		uint32_t iv = loopback[i], ov = loop[i];
		uint32_t iw = loopback[w], ow = loop[w];
		bool open = iv != kNone && iv != i && ov != kNone && ov != i && iw != kNone && iw != w && ow != kNone && ow != w;
		if (open && remap[iv] == remap[ow] && remap[ov] == remap[iw] && remap[iv] != remap[ov])
			k = kSeam;
		else
			k = kLocked;
	}
	else
		k = kLocked;
	return k;
}

__global__ void k_classify_primary(const uint32_t* remap, const uint32_t* wedge, const uint32_t* loop, const uint32_t* loopback, size_t n, uint8_t* kind)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n && remap[i] == (uint32_t)i)
		kind[i] = classify_primary(remap, wedge, loop, loopback, (uint32_t)i);
}

// permissive mode, src/simplifier.cpp:481-515 (primaries; wedges copy later)
__global__ void k_permissive(const uint32_t* off, const uint2* adj, const uint32_t* remap, const uint32_t* wedge, const uint8_t* vertex_lock,
                             const uint32_t* sparse_remap, size_t n, uint8_t* kind)
{
	size_t ii = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (ii >= n)
		return;
	uint32_t i = (uint32_t)ii;
	if (remap[i] != i || (kind[i] != kSeam && kind[i] != kLocked))
		return;

	bool protect = false;
	uint32_t v = i;
	do
	{
		uint32_t rv = sparse_remap ? sparse_remap[v] : v;
		protect |= vertex_lock && (vertex_lock[rv] & kVertexProtect) != 0;
		v = wedge[v];
	} while (v != i);

	do
	{
		for (uint32_t p = off[v], e = off[v + 1]; p < e && !protect; ++p)
			protect |= !has_edge_wedged(off, adj, adj[p].x, v, remap, wedge);
		v = wedge[v];
	} while (v != i);

	if (!protect)
		kind[i] = kComplex;
}

// vertex_lock Lock bit, src/simplifier.cpp:517-525 (marks the primary)
__global__ void k_lock_mark(const uint32_t* remap, const uint8_t* vertex_lock, const uint32_t* sparse_remap, size_t n, uint8_t* kind)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	size_t ri = sparse_remap ? sparse_remap[i] : i;
	if (vertex_lock[ri] & kVertexLock)
		kind[remap[i]] = kLocked;
}

// every wedge takes its primary's final kind; LockBorder turns Border into Locked
// (src/simplifier.cpp:470-477, 527-536; the Border->Locked map is idempotent, so primaries
// updating in place race harmlessly with wedges reading them).  Counted on the way: the primaries
// of each kind, and the corners of the manifold and seam vertices (boundEdgeCollapses, 1292-1308).
// kDirect: nothing changes a kind between the primary rules and here, and no vertex has a second
// wedge, so each vertex takes the rules' kind itself.
template <bool kDirect>
__global__ void __launch_bounds__(kThreads) k_kind_finalize(const uint32_t* remap, const uint32_t* wedge, const uint32_t* loop, const uint32_t* loopback,
                                                            const uint32_t* off, size_t n, uint32_t options, uint8_t* kind, CallScalars* sc)
{
	__shared__ uint32_t h[7];
	if (threadIdx.x < 7)
		h[threadIdx.x] = 0;
	__syncthreads();
	uint32_t local[7] = {0, 0, 0, 0, 0, 0, 0};
	for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (size_t)gridDim.x * kThreads)
	{
		const uint32_t r = kDirect ? (uint32_t)i : remap[i];
		uint8_t k = kDirect ? classify_primary(remap, wedge, loop, loopback, (uint32_t)i) : kind[r];
		if ((options & kOptLockBorder) && k == kBorder)
			k = kLocked;
		kind[i] = k;
		if (r == (uint32_t)i)
		{
#pragma unroll
			for (int q = 0; q < 5; ++q)
				local[q] += k == q;
			local[5]++;
		}
		local[6] += (k == kManifold || k == kSeam) ? off[i + 1] - off[i] : 0u;
	}
#pragma unroll
	for (int q = 0; q < 7; ++q)
	{
		uint32_t v = local[q];
		for (int o = 32; o > 0; o >>= 1)
			v += __shfl_xor(v, o, 64);
		if (__lane_id() == 0 && v)
			atomicAdd(&h[q], v);
	}
	__syncthreads();
	if (threadIdx.x < 7 && h[threadIdx.x])
		atomicAdd(threadIdx.x < 6 ? &sc->kind_counts[threadIdx.x] : &sc->dual_count, h[threadIdx.x]);
}

void launch_classify(hipStream_t s, Mesh& m, const uint32_t* raw_off, bool secondaries, const uint8_t* vertex_lock, const uint32_t* sparse_remap,
                     uint32_t options)
{
	size_t n = m.vertex_count;
	if (!n)
		return;
	uint32_t* loop = m.loop[0];
	uint32_t* loopback = m.loopback[0];
	const unsigned int grid = std::min(grid_for(n), 1024u);
	if (!secondaries && !vertex_lock && !(options & kOptPermissive))
	{
		k_kind_finalize<true><<<grid, kThreads, 0, s>>>(m.remap, m.wedge, loop, loopback, raw_off, n, options, m.kind, m.sc);
		return;
	}
	k_classify_primary<<<grid_for(n), kThreads, 0, s>>>(m.remap, m.wedge, loop, loopback, n, m.kind);
	if (options & kOptPermissive)
		k_permissive<<<grid_for(n), kThreads, 0, s>>>(raw_off, m.adj[1], m.remap, m.wedge, vertex_lock, sparse_remap, n, m.kind);
	if (vertex_lock)
		k_lock_mark<<<grid_for(n), kThreads, 0, s>>>(m.remap, vertex_lock, sparse_remap, n, m.kind);
	k_kind_finalize<false><<<grid, kThreads, 0, s>>>(m.remap, m.wedge, loop, loopback, raw_off, n, options, m.kind, m.sc);
}

// rescaleAttributes, src/simplifier.cpp:605-621 (only attributes with weight > 0)

__global__ void k_rescale_attributes(const float* attrs, size_t stride, const uint32_t* sparse_remap, size_t n, uint32_t count, AttrMap map, float* va)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	size_t ri = sparse_remap ? sparse_remap[i] : i;
	const float* a = attrs + ri * stride;
	for (uint32_t k = 0; k < count; ++k)
		va[i * count + k] = a[map.index[k]] * map.weight[k];
}

void launch_rescale_attributes(hipStream_t s, Mesh& m, const float* attributes, size_t stride_floats, const uint32_t* sparse_remap,
                               const uint32_t* attr_index, const float* attr_weight)
{
	if (!m.vertex_count || !m.attr_count)
		return;
	AttrMap map;
	for (uint32_t k = 0; k < m.attr_count; ++k)
	{
		map.index[k] = attr_index[k];
		map.weight[k] = attr_weight[k];
	}
	k_rescale_attributes<<<grid_for(m.vertex_count), kThreads, 0, s>>>(attributes, stride_floats, sparse_remap, m.vertex_count, m.attr_count, map, m.va);
}

// ------------------------------------------------------------------------------------------
// vertex quadrics (src/simplifier.cpp:1057-1157), and the first pass's welded adjacency (the lists
// are read here anyway).  One thread per primary r walks r's
// corners in (triangle, corner) order and adds, as the reference's three sequential fills
// do: every face quadric, then the regularising point quadric, then the border/seam edge
// quadrics in (triangle, edge, endpoint) order.  No float atomics; each sum starts at +0.

__device__ __forceinline__ bool edge_loop_qualifies(const uint8_t* kind, const uint32_t* loop, const uint32_t* loopback, uint32_t i0, uint32_t i1, float& weight)
{
	uint8_t k0 = kind[i0], k1 = kind[i1];
	bool b0 = k0 == kBorder || k0 == kSeam;
	bool b1 = k1 == kBorder || k1 == kSeam;
	if (!b0 && !b1)
		return false;
	if (b0 && loop[i0] != i1)
		return false;
	if (b1 && loopback[i1] != i0)
		return false;
	weight = (k0 == kBorder || k1 == kBorder) ? 10.f : 0.5f;
	return true;
}

__global__ void k_vertex_quadrics(const uint32_t* ib, const float4* pos, const uint32_t* remap, const uint8_t* kind, const uint32_t* loop,
                                  const uint32_t* loopback, const uint32_t* woff, const uint32_t* wcorners, const uint8_t* vertex_lock,
                                  const uint32_t* sparse_remap, size_t n, float factor, Quad* vq, Grad* vg, uint2* adj_range, uint2* adj, uint64_t index_count,
                                  CallScalars* sc)
{
	size_t ri = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (ri >= n)
		return;
	uint32_t r = (uint32_t)ri;
	// boundEdgeCollapses (src/simplifier.cpp:1292-1308) from the dual count: the first pick reads it here
	if (r == 0)
	{
		const uint64_t c = index_count - sc->dual_count / 2 + 3;
		sc->pick_capacity = c < 0xffffffffull ? (uint32_t)c : 0xffffffffu;
	}
	const uint32_t begin = woff[r], end = woff[r + 1];
	adj_range[r] = make_uint2(begin, end); // empty for a secondary: the lists are keyed by primaries
	Quad Q;
	quad_zero(Q);
	if (remap[r] != r)
	{
		store_quad(vq, r, Q);
		return;
	}
	Grad GV = {0.f, 0.f, 0.f, 0.f};

	// kChunk corners' gathers in flight at a time; the sums stay in corner order
	constexpr int kChunk = 4;
	for (uint32_t p0 = begin; p0 < end; p0 += kChunk)
	{
		uint32_t t[kChunk], c[kChunk];
#pragma unroll
		for (int q = 0; q < kChunk; ++q)
		{
			const uint32_t j = wcorners[p0 + q < end ? p0 + q : begin];
			t[q] = j / 3;
			c[q] = j - t[q] * 3;
		}
		uint32_t i[kChunk][3];
#pragma unroll
		for (int q = 0; q < kChunk; ++q)
#pragma unroll
			for (int k = 0; k < 3; ++k)
				i[q][k] = ib[t[q] * 3 + k];
		V3 p[kChunk][3];
#pragma unroll
		for (int q = 0; q < kChunk; ++q)
#pragma unroll
			for (int k = 0; k < 3; ++k)
				p[q][k] = load_pos(pos, i[q][k]);
#pragma unroll
		for (int q = 0; q < kChunk; ++q)
		{
			if (p0 + q >= end)
				continue;
			// the first pass's adjacency: the corner's next and previous classes
			adj[p0 + q] = make_uint2(remap[c[q] == 0 ? i[q][1] : (c[q] == 1 ? i[q][2] : i[q][0])], remap[c[q] == 0 ? i[q][2] : (c[q] == 1 ? i[q][0] : i[q][1])]);
			Quad F;
			quad_from_triangle(F, p[q][0], p[q][1], p[q][2], 1.f);
			quad_add(Q, F);
			if (vg)
			{
				// volume gradients of the position solve, summed in the same corner order
				Grad G;
				grad_volume(G, p[q][0], p[q][1], p[q][2]);
				grad_add(GV, G);
			}
		}
	}
	if (vg)
		vg[r] = GV;

	{
		size_t rr = sparse_remap ? sparse_remap[r] : r;
		bool priority = vertex_lock && (vertex_lock[rr] & kVertexPriority) != 0;
		V3 v = load_pos(pos, r);
		float w = Q.w * (priority ? 1.0f : factor);
		Quad P;
		quad_from_point(P, v.x, v.y, v.z, w);
		quad_add(Q, P);
	}

	// a manifold vertex has no open edge, and only open edges qualify below (loop and loopback are
	// the open edges of the set-up)
	uint32_t last_t = kNone;
	for (uint32_t p = kind[r] == kManifold ? end : begin; p < end; ++p)
	{
		uint32_t t = wcorners[p] / 3;
		if (t == last_t)
			continue;
		last_t = t;
		uint32_t tri[3] = {ib[t * 3 + 0], ib[t * 3 + 1], ib[t * 3 + 2]};
		for (int e = 0; e < 3; ++e)
		{
			uint32_t i0 = tri[e];
			uint32_t i1 = tri[e == 2 ? 0 : e + 1];
			uint32_t i2 = tri[e == 0 ? 2 : e - 1];
			bool at0 = remap[i0] == r, at1 = remap[i1] == r;
			if (!at0 && !at1)
				continue;
			float weight;
			if (!edge_loop_qualifies(kind, loop, loopback, i0, i1, weight))
				continue;
			Quad E;
			quad_edge_term(E, load_pos(pos, i0), load_pos(pos, i1), load_pos(pos, i2), weight);
			if (at0)
				quad_add(Q, E);
			if (at1)
				quad_add(Q, E);
		}
	}

	store_quad(vq, r, Q);
}

void launch_vertex_quadrics(hipStream_t s, Mesh& m, const uint32_t* welded_off, const uint32_t* welded_corners, const uint8_t* vertex_lock,
                            const uint32_t* sparse_remap, uint32_t options)
{
	size_t n = m.vertex_count;
	if (!n)
		return;
	float factor = (options & kOptRegularizeLight) ? 1e-2f : ((options & kOptRegularize) ? 1e-1f : 1e-7f);
	k_vertex_quadrics<<<grid_for(n), kThreads, 0, s>>>(m.ib[0], m.pos, m.remap, m.kind, m.loop[0], m.loopback[0], welded_off, welded_corners,
	                                                   vertex_lock, sparse_remap, n, factor, m.vq, m.vg, m.adj_range[0], m.adj[0],
	                                                   (uint64_t)m.index_count, m.sc);
}

// attribute quadrics and gradients (src/simplifier.cpp:1159-1179), per wedge (not welded),
// triangles in order.  N is the attribute count when it is small enough for registers.
template <int N>
__global__ void k_attribute_quadrics(const uint32_t* ib, const float4* pos, const float* va, const uint32_t* off, const uint32_t* corners,
                                     size_t n, int count, Quad* aq, Grad* ag)
{
	size_t ii = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (ii >= n)
		return;
	uint32_t i = (uint32_t)ii;
	const int A = N > 0 ? N : count;

	Quad Q;
	quad_zero(Q);
	Grad G[N > 0 ? N : 1];
	if (N > 0)
		for (int k = 0; k < A; ++k)
			G[k] = Grad{0.f, 0.f, 0.f, 0.f};
	else
		for (int k = 0; k < A; ++k)
			ag[(size_t)i * A + k] = Grad{0.f, 0.f, 0.f, 0.f};

	for (uint32_t p = off[i], e = off[i + 1]; p < e; ++p)
	{
		uint32_t t = corners[p] / 3;
		uint32_t i0 = ib[t * 3 + 0], i1 = ib[t * 3 + 1], i2 = ib[t * 3 + 2];
		AttrFrame f = attr_frame(load_pos(pos, i0), load_pos(pos, i1), load_pos(pos, i2));

		Quad QA;
		quad_zero(QA);
		QA.w = f.w;
		const float* a0 = va + (size_t)i0 * A;
		const float* a1 = va + (size_t)i1 * A;
		const float* a2 = va + (size_t)i2 * A;
		for (int k = 0; k < A; ++k)
		{
			Grad g;
			attr_term(QA, g, f, a0[k], a1[k], a2[k]);
			if (N > 0)
				grad_add(G[k], g);
			else
			{
				Grad acc = ag[(size_t)i * A + k];
				grad_add(acc, g);
				ag[(size_t)i * A + k] = acc;
			}
		}
		quad_add(Q, QA);
	}

	store_quad(aq, i, Q);
	if (N > 0)
		for (int k = 0; k < A; ++k)
			ag[(size_t)i * A + k] = G[k];
}

void launch_attribute_quadrics(hipStream_t s, Mesh& m, const uint32_t* raw_off, const uint32_t* raw_corners)
{
	size_t n = m.vertex_count;
	int A = (int)m.attr_count;
	if (!n || !A)
		return;
	unsigned int g = grid_for(n);
	switch (A)
	{
#define CASE(K) \
	case K: \
		k_attribute_quadrics<K><<<g, kThreads, 0, s>>>(m.ib[0], m.pos, m.va, raw_off, raw_corners, n, A, m.aq, m.ag); \
		break;
		CASE(1)
		CASE(2)
		CASE(3)
		CASE(4)
		CASE(5)
		CASE(6)
		CASE(7)
		CASE(8)
#undef CASE
	default:
		k_attribute_quadrics<0><<<g, kThreads, 0, s>>>(m.ib[0], m.pos, m.va, raw_off, raw_corners, n, A, m.aq, m.ag);
	}
}

} // namespace mhip
