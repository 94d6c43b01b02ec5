// The Prune option (src/simplifier.cpp:1866-2024): connected components of the welded mesh,
// each component's error (the squared radius of its vertices around their mean), and the removal
// of whole components whose error is at or below a cutoff.
//
// Components come from a lock-free union-find that always hooks the larger root under the
// smaller, so every root is the lowest primary of its component, exactly as the reference's
// sequential union (buildComponents) leaves it; ids are then numbered in root order.  The error
// sums run sequentially per component over its vertices in index order, which is the reference's
// accumulation order, so the values match bit for bit.
#include "kernels.h"
#include "prims.h"

namespace mhip
{

static constexpr int kPruneThreads = 256;

static inline unsigned int prune_grid(size_t n)
{
	return div_up(n ? n : 1, kPruneThreads);
}

// root of x with path halving; parent[v] <= v always holds, so a stale read still yields an
// ancestor and every concurrent halving store keeps the trees valid
__device__ __forceinline__ uint32_t uf_root(uint32_t* parent, uint32_t x)
{
	for (;;)
	{
		uint32_t p = __atomic_load_n(&parent[x], __ATOMIC_RELAXED);
		if (p == x)
			return x;
		uint32_t g = __atomic_load_n(&parent[p], __ATOMIC_RELAXED);
		if (g != p)
			__atomic_store_n(&parent[x], g, __ATOMIC_RELAXED);
		x = g;
	}
}

__device__ __forceinline__ void uf_union(uint32_t* parent, uint32_t a, uint32_t b)
{
	for (;;)
	{
		uint32_t ra = uf_root(parent, a), rb = uf_root(parent, b);
		if (ra == rb)
			return;
		uint32_t hi = ra > rb ? ra : rb, lo = ra > rb ? rb : ra;
		if (atomicCAS(&parent[hi], hi, lo) == hi)
			return;
		// hi was hooked by another thread meanwhile: retry from the new roots
	}
}

// The unions start from a forest that already holds most of the mesh: every corner's parent is the
// lowest corner it shares a triangle with (a vertex of its component, never above itself), and each
// vertex then follows its chain to the end.  What is left for the edges below is mostly a
// comparison of two equal roots; from single vertices the same edges fought over a few roots
// (0.96 ms for the edges on 182 k vertices in 201 components; the three kernels take 0.14 ms).
__global__ void k_uf_hook(const uint32_t* ib, size_t tris, const uint32_t* remap, uint32_t* parent)
{
	size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= tris)
		return;
	const uint32_t v[3] = {remap[ib[t * 3 + 0]], remap[ib[t * 3 + 1]], remap[ib[t * 3 + 2]]};
	const uint32_t ab = v[0] < v[1] ? v[0] : v[1];
	const uint32_t lo = ab < v[2] ? ab : v[2];
#pragma unroll
	for (int k = 0; k < 3; ++k)
		if (v[k] != lo && __atomic_load_n(&parent[v[k]], __ATOMIC_RELAXED) > lo)
			atomicMin(&parent[v[k]], lo);
}

__global__ void k_uf_compress(uint32_t* parent, size_t n)
{
	size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (v < n)
		__atomic_store_n(&parent[v], uf_root(parent, (uint32_t)v), __ATOMIC_RELAXED);
}

// buildComponents (src/simplifier.cpp:1866-1908): union over the welded edges of every triangle
// (two edges connect its three corners)
__global__ void k_uf_edges(const uint32_t* ib, size_t tris, const uint32_t* remap, uint32_t* parent)
{
	size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= tris)
		return;
	uint32_t a = remap[ib[t * 3 + 0]], b = remap[ib[t * 3 + 1]], c = remap[ib[t * 3 + 2]];
	uf_union(parent, a, b);
	uf_union(parent, b, c);
}

__global__ void k_uf_roots(const uint32_t* remap, size_t n, uint32_t* parent, uint32_t* roots, uint32_t* flags)
{
	size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (v >= n)
		return;
	bool primary = remap[v] == (uint32_t)v;
	uint32_t r = primary ? uf_root(parent, (uint32_t)v) : 0;
	roots[v] = r;
	flags[v] = primary && r == (uint32_t)v;
}

__global__ void k_component_ids(const uint32_t* remap, size_t n, const uint32_t* roots, const uint32_t* root_ids, uint32_t* comp)
{
	size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (v >= n)
		return;
	comp[v] = root_ids[roots[remap[v]]];
}

void launch_components(hipStream_t s, Mesh& m, size_t index_count, uint32_t* comp, uint32_t* scratch[5])
{
	const size_t V = m.vertex_count, T = index_count / 3;
	HIP_CHECK(hipMemsetAsync(&m.sc->component_count, 0, sizeof(uint32_t), s));
	if (!V)
		return;
	uint32_t* parent = scratch[0];
	uint32_t* roots = scratch[1];
	uint32_t* ids = scratch[2];
	iota_u32(s, parent, V);
	if (T)
	{
		k_uf_hook<<<prune_grid(T), kPruneThreads, 0, s>>>(m.ib[0], T, m.remap, parent);
		k_uf_compress<<<prune_grid(V), kPruneThreads, 0, s>>>(parent, V);
		k_uf_edges<<<prune_grid(T), kPruneThreads, 0, s>>>(m.ib[0], T, m.remap, parent);
	}
	k_uf_roots<<<prune_grid(V), kPruneThreads, 0, s>>>(m.remap, V, parent, roots, ids);
	scan_exclusive(s, ids, ids, V, nullptr, &m.sc->component_count, m.temp);
	k_component_ids<<<prune_grid(V), kPruneThreads, 0, s>>>(m.remap, V, roots, ids, comp);
}

__global__ void k_copy_u32(const uint32_t* in, uint32_t* out, size_t n)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		out[i] = in[i];
}

// start of every component's run in the component-sorted vertex list (every component has its
// root, so no run is empty); off[count] = n
__global__ void k_component_offsets(const uint32_t* sorted_comp, size_t n, uint32_t* off)
{
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	uint32_t c = sorted_comp[i];
	if (i == 0 || sorted_comp[i - 1] != c)
		off[c] = (uint32_t)i;
	if (i + 1 == n)
		off[c + 1] = (uint32_t)n;
}

// measureComponents (src/simplifier.cpp:1910-1968): mean, then the largest squared distance.  The
// sums are serial chains in vertex order, which is what fixes their bits.  A component of up to
// kShortComponent vertices is one thread's; a longer one is appended to `longs` for the kernel
// below (a thread that walks it alone pays a gather per vertex: 46 ms for one of 160 k vertices).
constexpr uint32_t kShortComponent = 32;

// the vertex count as the reference accumulates it: w += 1.f stops growing at 2^24
__device__ __forceinline__ float component_weight(uint32_t n)
{
	return n < (1u << 24) ? (float)n : 16777216.f;
}

__device__ __forceinline__ float component_distance(float4 p, float sx, float sy, float sz)
{
	float dx = p.x - sx, dy = p.y - sy, dz = p.z - sz;
	return dx * dx + dy * dy + dz * dz;
}

__global__ void k_measure_short(const uint32_t* off, const uint32_t* verts, const float4* pos, const uint32_t* count_dev, float* cerr,
                                uint32_t* min_bits, uint32_t* longs, uint32_t* long_count)
{
	size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (c >= *count_dev)
		return;
	const uint32_t b = off[c], e = off[c + 1];
	if (e - b > kShortComponent)
	{
		longs[atomicAdd(long_count, 1u)] = (uint32_t)c;
		return;
	}
	float sx = 0.f, sy = 0.f, sz = 0.f;
	for (uint32_t i = b; i < e; ++i)
	{
		float4 p = pos[verts[i]];
		sx += p.x;
		sy += p.y;
		sz += p.z;
	}
	float w = component_weight(e - b);
	float iw = w == 0.f ? 0.f : 1.f / w;
	sx *= iw;
	sy *= iw;
	sz *= iw;
	float r2 = 0.f;
	for (uint32_t i = b; i < e; ++i)
	{
		float r = component_distance(pos[verts[i]], sx, sy, sz);
		r2 = r2 < r ? r : r2;
	}
	cerr[c] = r2;
	// non-negative floats order like their bit patterns
	atomicMin(min_bits, __float_as_uint(r2));
}

// One workgroup per long component.  Its vertices come in tiles: every thread gathers the next
// tile's positions while three wavefronts, one per coordinate, add the current one from LDS (each
// 16-byte read feeds four links of the chain, so the chain runs at the latency of the add rather
// than of a gather).  The distances have no order (a running maximum that skips NaN): all threads.
// One component of 160 k vertices: 0.63 ms (46 ms by one thread), bound by the chain of adds (about
// eight cycles a link).
constexpr int kLongThreads = 1024;
constexpr int kLongPer = 4;
constexpr int kLongTile = kLongThreads * kLongPer;

__global__ void __launch_bounds__(kLongThreads) k_measure_long(const uint32_t* off, const uint32_t* verts, const float4* pos, const uint32_t* longs,
                                                               const uint32_t* long_count, float* cerr, uint32_t* min_bits)
{
	__shared__ __align__(16) float tile[3][kLongTile];
	__shared__ float mean[3];
	__shared__ uint32_t best;
	const uint32_t n = *long_count;
	const uint32_t wave = threadIdx.x >> 6;
	for (uint32_t q = blockIdx.x; q < n; q += gridDim.x)
	{
		const uint32_t c = longs[q], b = off[c], e = off[c + 1];
		float4 p[kLongPer];
		auto fetch = [&](uint32_t at) {
#pragma unroll
			for (int k = 0; k < kLongPer; ++k)
			{
				const uint32_t i = at + k * kLongThreads + threadIdx.x;
				p[k] = i < e ? pos[verts[i]] : make_float4(0.f, 0.f, 0.f, 0.f);
			}
		};
		fetch(b);
		float sum = 0.f;
		for (uint32_t at = b; at < e; at += kLongTile)
		{
#pragma unroll
			for (int k = 0; k < kLongPer; ++k)
			{
				tile[0][k * kLongThreads + threadIdx.x] = p[k].x;
				tile[1][k * kLongThreads + threadIdx.x] = p[k].y;
				tile[2][k * kLongThreads + threadIdx.x] = p[k].z;
			}
			__syncthreads();
			if (at + kLongTile < e)
				fetch(at + kLongTile);
			if (wave < 3)
			{
				const float* t = tile[wave];
				const uint32_t len = e - at < (uint32_t)kLongTile ? e - at : (uint32_t)kLongTile;
				uint32_t i = 0;
				for (; i + 32 <= len; i += 32)
				{
					float4 v[8];
#pragma unroll
					for (int k = 0; k < 8; ++k)
						v[k] = *reinterpret_cast<const float4*>(t + i + 4 * k);
#pragma unroll
					for (int k = 0; k < 8; ++k)
					{
						sum += v[k].x;
						sum += v[k].y;
						sum += v[k].z;
						sum += v[k].w;
					}
				}
				for (; i < len; ++i)
					sum += t[i];
			}
			__syncthreads();
		}
		if (wave < 3 && __lane_id() == 0)
		{
			const float w = component_weight(e - b);
			mean[wave] = sum * (1.f / w);
		}
		if (threadIdx.x == 0)
			best = 0;
		__syncthreads();
		const float sx = mean[0], sy = mean[1], sz = mean[2];
		float r2 = 0.f;
		for (uint32_t at = b; at < e; at += kLongTile)
		{
			fetch(at);
#pragma unroll
			for (int k = 0; k < kLongPer; ++k)
			{
				const float r = component_distance(p[k], sx, sy, sz);
				if (at + k * kLongThreads + threadIdx.x < e)
					r2 = r2 < r ? r : r2;
			}
		}
		uint32_t bits = __float_as_uint(r2);
#pragma unroll
		for (int o = 32; o > 0; o >>= 1)
		{
			uint32_t x = __shfl_xor(bits, o, 64);
			bits = x > bits ? x : bits;
		}
		if (__lane_id() == 0)
			atomicMax(&best, bits);
		__syncthreads();
		if (threadIdx.x == 0)
		{
			cerr[c] = __uint_as_float(best);
			atomicMin(min_bits, best);
		}
		__syncthreads();
	}
}

__global__ void k_set_u32(uint32_t* p, uint32_t value)
{
	*p = value;
}

static int bits_for(size_t n)
{
	int b = 1;
	while (b < 32 && (size_t(1) << b) < n)
		++b;
	return b;
}

void launch_measure_components(hipStream_t s, Mesh& m, const uint32_t* comp, float* cerr, uint32_t* scratch[5])
{
	const size_t V = m.vertex_count;
	k_set_u32<<<1, 1, 0, s>>>(&m.sc->prune_min_bits, 0x7f7fffffu); // FLT_MAX
	if (!V)
		return;
	uint32_t* keys = scratch[0];
	uint32_t* vals = scratch[1];
	uint32_t* keys_alt = scratch[2];
	uint32_t* vals_alt = scratch[3];
	uint32_t* off = scratch[4];
	k_copy_u32<<<prune_grid(V), kPruneThreads, 0, s>>>(comp, keys, V);
	// stable: each component's vertices stay in index order (the reference's summation order)
	radix_sort_pairs(s, keys, vals, keys_alt, vals_alt, V, nullptr, bits_for(V), m.temp, true);
	k_component_offsets<<<prune_grid(V), kPruneThreads, 0, s>>>(keys, V, off);
	// the sorted keys are not needed any more: their space holds the list of long components
	k_set_u32<<<1, 1, 0, s>>>(&m.sc->work[0], 0u);
	k_measure_short<<<prune_grid(V), kPruneThreads, 0, s>>>(off, vals, m.pos, &m.sc->component_count, cerr, &m.sc->prune_min_bits, keys, &m.sc->work[0]);
	const size_t most = V / (kShortComponent + 1);
	if (most)
		k_measure_long<<<(unsigned int)(most < 512 ? most : 512), kLongThreads, 0, s>>>(off, vals, m.pos, keys, &m.sc->work[0], cerr, &m.sc->prune_min_bits);
}

// pruneComponents (src/simplifier.cpp:1970-2024)
__global__ void k_prune_keep(const uint32_t* ib, size_t tris, const uint32_t* comp, const float* cerr, float cutoff, uint32_t* keep,
                             uint32_t* min_bits)
{
	size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	// the smallest kept error (non-negative floats order like their bits): one atomic per
	// wavefront, so every lane stays to the reduction
	uint32_t bits = 0xffffffffu;
	if (t < tris)
	{
		float e = cerr[comp[ib[t * 3]]];
		bool k = e > cutoff;
		keep[t] = k;
		if (k)
			bits = __float_as_uint(e);
	}
#pragma unroll
	for (int o = 32; o > 0; o >>= 1)
	{
		uint32_t x = __shfl_xor(bits, o, 64);
		bits = x < bits ? x : bits;
	}
	if (__lane_id() == 0 && bits != 0xffffffffu)
		atomicMin(min_bits, bits);
}

__global__ void k_prune_write(const uint32_t* ib, size_t tris, const uint32_t* keep, const uint32_t* off, uint32_t* out)
{
	size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= tris || !keep[t])
		return;
	size_t o = (size_t)off[t] * 3;
	out[o + 0] = ib[t * 3 + 0];
	out[o + 1] = ib[t * 3 + 1];
	out[o + 2] = ib[t * 3 + 2];
}

void launch_prune_triangles(hipStream_t s, Mesh& m, size_t tri_count, const uint32_t* comp, const float* cerr, float cutoff)
{
	HIP_CHECK(hipMemsetAsync(&m.sc->next_triangles, 0, sizeof(uint32_t), s));
	k_set_u32<<<1, 1, 0, s>>>(&m.sc->prune_min_bits, 0x7f7fffffu);
	if (!tri_count)
		return;
	const uint32_t* in = m.ib[m.ib_cur];
	uint32_t* out = m.ib[m.ib_cur ^ 1];
	k_prune_keep<<<prune_grid(tri_count), kPruneThreads, 0, s>>>(in, tri_count, comp, cerr, cutoff, m.tri_cnt, &m.sc->prune_min_bits);
	// keep flags are read by the scatter after the scan overwrites tri_off only
	scan_exclusive(s, m.tri_cnt, m.tri_off, tri_count, nullptr, &m.sc->next_triangles, m.temp);
	k_prune_write<<<prune_grid(tri_count), kPruneThreads, 0, s>>>(in, tri_count, m.tri_cnt, m.tri_off, out);
	m.ib_cur ^= 1;
}

__global__ void k_component_max(const float* cerr, const uint32_t* count_dev, float cutoff, uint32_t* max_bits)
{
	size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (c >= *count_dev)
		return;
	float e = cerr[c];
	if (e > 0.f && e <= cutoff)
		atomicMax(max_bits, __float_as_uint(e));
}

void launch_component_max(hipStream_t s, Mesh& m, const float* cerr, float cutoff)
{
	HIP_CHECK(hipMemsetAsync(&m.sc->prune_max_bits, 0, sizeof(uint32_t), s));
	if (m.vertex_count)
		k_component_max<<<prune_grid(m.vertex_count), kPruneThreads, 0, s>>>(cerr, &m.sc->component_count, cutoff, &m.sc->prune_max_bits);
}

} // namespace mhip
