// Graph stages on the device: SCC decomposition, condensation heights and the
// canonical vertex order.
//
// Replaces transition_graph::reorganize_vertices (reference
// cuda/src/transition_graph.cu:123-202), the GARDENIA FW-BW-trim SCC solver it
// calls (cuda/src/sga/two_phase.cu:12-145, bitset.cu, wcc.cu) and the
// topological_labelling / reorganize kernels (kernels/transition_graph.cu:3-52).
//
// The state graph is an orientation of (a subgraph of) the N-cube, so the
// graph is never stored as an adjacency list here: the neighbours of v are
// v ^ (1 << i), v -> v^(1<<i) iff bit i of mask[v], and v^(1<<i) -> v iff bit
// i of mask[v ^ (1 << i)].  One wavefront owns a 6-sub-cube (64 consecutive
// states), so the moves along bits 0..5 stay in registers (cross-lane
// shuffles) and each pass relaxes to a wave-local fixpoint before it touches
// HBM again; moves along bits >= 6 read the neighbouring sub-cube, which is
// a contiguous, coalesced 256-byte block.
//
// SCCs: rounds on classes of vertices that hold whole SCCs (at first one class).
// A round drops the edges between classes, trims, and gives every vertex two
// colours in one fixpoint: the minimum vertex that reaches it and the minimum that
// it reaches.  Where the two agree they name the vertex's SCC by its minimum
// vertex, the canonical SCC id, so the output is deterministic (the reference's
// atomicCAS pivots, bitset.cu:415-423, are not); the colour pairs of the others are
// the next round's classes (an SCC has one pair).  The pairs part a class from both
// sides, which takes half the rounds of one colour with a closure after it (20
// nodes: 6 instead of 11; 16 nodes: 6 instead of 12), and a round has two fixpoints
// instead of three.  Passes read the neighbours' labels only, the edges of a round
// being two bit masks per vertex.  20 nodes: 4.8 to 2.7 ms with the heights below.
//
// Heights: 1 + the largest height of a successor, terminal SCCs 1 (what rounds that
// label every SCC whose successors are labelled give, topological_labelling), by
// relaxation from 1 everywhere: a pass of a wave relaxes its sub-cube to a fixpoint,
// so it advances a chain by several levels.
//
// Up to 4096 states one workgroup does all of it in LDS, the order included: there a
// pass is a fraction of a microsecond, and launches and round trips were the time.
//
// Order: [terminal SCCs by ascending id | transient SCCs by (height desc, id
// desc)], vertices ascending inside an SCC (transition_graph.cu:170-198).

#include <rocprim/device/device_radix_sort.hpp>

#include "cube.hip.hpp"

namespace esl {

constexpr int gblock = 256;

// ---- the edges of a round: bit i of x (y) is set when the neighbour along bit i is
// active, in v's class (the colour pair of the last round; null in the first) and has
// an edge into v (from v)
template <int HMAX>
__global__ __launch_bounds__(gblock) void k_edges(int N, int64_t n, const uint32_t* __restrict__ mask,
												  const int32_t* __restrict__ scc, const int2* __restrict__ cls,
												  uint2* __restrict__ edges)
{
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	const bool valid = v < n;
	const bool active = valid && scc[v] < 0;
	uint2 e = make_uint2(0u, 0u);
	if (__any(active))
	{
		const uint32_t mv = valid ? mask[v] : 0u;
		const int2 cv = cls && active ? cls[v] : make_int2(-1, -1);
		const uint64_t act = __ballot(active);
		if (HMAX > 0)
		{
			uint32_t mu[HMAX > 0 ? HMAX : 1];
			int32_t su[HMAX > 0 ? HMAX : 1];
			int2 cu[HMAX > 0 ? HMAX : 1];
			const int64_t vv = valid ? v : 0; // lanes past n read vertex 0's neighbours, unused
#pragma unroll
			for (int j = 0; j < HMAX; ++j)
			{
				const int64_t u = vv ^ (int64_t(1) << high_bit(j, N));
				mu[j] = mask[u];
				su[j] = scc[u];
				cu[j] = cv;
			}
			if (cls)
#pragma unroll
				for (int j = 0; j < HMAX; ++j)
					cu[j] = cls[vv ^ (int64_t(1) << high_bit(j, N))];
#pragma unroll
			for (int j = 0; j < HMAX; ++j)
			{
				const int i = 6 + j;
				const bool ok = i < N && su[j] < 0 && cu[j].x == cv.x && cu[j].y == cv.y;
				e.x |= ok ? mu[j] & (1u << i) : 0u;
				e.y |= ok ? mv & (1u << i) : 0u;
			}
		}
		const int lim = N < 6 ? N : 6;
		for (int i = 0; i < lim; ++i)
		{
			const uint32_t mu = __shfl_xor(mv, 1 << i, wave);
			const int cx = __shfl_xor(cv.x, 1 << i, wave), cy = __shfl_xor(cv.y, 1 << i, wave);
			const bool ok = (act >> (lane_id() ^ (1 << i)) & 1) && cx == cv.x && cy == cv.y;
			e.x |= ok ? mu & (1u << i) : 0u;
			e.y |= ok ? mv & (1u << i) : 0u;
		}
		if (!active)
			e = make_uint2(0u, 0u);
	}
	if (valid)
		edges[v] = e;
}

// ---- trimming: a vertex without an active in- or out-neighbour is a singleton SCC
template <int HMAX>
__global__ __launch_bounds__(gblock) void k_trim(int N, int64_t n, const uint2* __restrict__ edges,
												 int32_t* __restrict__ scc, int32_t* __restrict__ changed,
												 const int32_t* __restrict__ prev)
{
	if (converged(prev))
		return;
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	const bool valid = v < n;
	bool active = valid && scc[v] < 0;
	if (!__any(active))
		return;
	const uint2 e = valid ? edges[v] : make_uint2(0u, 0u);
	bool gin = false, gout = false;
	if (HMAX > 0)
	{
		int32_t su[HMAX > 0 ? HMAX : 1];
		const int64_t vv = valid ? v : 0;
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
			su[j] = scc[vv ^ (int64_t(1) << high_bit(j, N))];
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
		{
			const int i = 6 + j;
			const bool ua = i < N && su[j] < 0;
			gin |= ua && ((e.x >> i) & 1u);
			gout |= ua && ((e.y >> i) & 1u);
		}
	}
	const int lim = N < 6 ? N : 6;
	bool trimmed = false;
	for (;;)
	{
		const uint64_t act = __ballot(active);
		bool in = gin, out = gout;
		for (int i = 0; i < lim; ++i)
		{
			const bool ua = act >> (lane_id() ^ (1 << i)) & 1;
			in |= ua && ((e.x >> i) & 1u);
			out |= ua && ((e.y >> i) & 1u);
		}
		const bool t = active && !(in && out);
		if (!__any(t))
			break;
		if (t)
		{
			active = false;
			trimmed = true;
		}
	}
	if (trimmed)
	{
		scc[v] = (int32_t)v;
		changed[0] = 1;
	}
}

// an active vertex starts with itself as both colours, others have none (and, being
// the largest value, none to give)
__global__ __launch_bounds__(gblock) void k_color_init(int64_t n, const int32_t* __restrict__ scc,
													   int2* __restrict__ col)
{
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	if (v < n)
	{
		const int32_t c = scc[v] < 0 ? (int32_t)v : INT32_MAX;
		col[v] = make_int2(c, c);
	}
}

// ---- both colours along the round's edges: x[v] = min(x[v], x[u]) for u -> v,
// y[v] = min(y[v], y[u]) for v -> u
template <int HMAX>
__global__ __launch_bounds__(gblock) void k_color(int N, int64_t n, const uint2* __restrict__ edges,
												  int2* __restrict__ col, int32_t* __restrict__ changed,
												  const int32_t* __restrict__ prev)
{
	if (converged(prev))
		return;
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	const bool valid = v < n;
	const uint2 e = valid ? edges[v] : make_uint2(0u, 0u);
	if (!__any((e.x | e.y) != 0u))
		return;
	const int2 c0 = valid ? col[v] : make_int2(INT32_MAX, INT32_MAX);
	const bool active = c0.x != INT32_MAX; // trimmed vertices have edges still
	int2 c = c0;
	if (HMAX > 0)
	{
		int2 cu[HMAX > 0 ? HMAX : 1];
		const int64_t vv = valid ? v : 0;
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
			cu[j] = col[vv ^ (int64_t(1) << high_bit(j, N))];
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
		{
			const int i = 6 + j;
			if (active && i < N && ((e.x >> i) & 1u))
				c.x = min(c.x, cu[j].x);
			if (active && i < N && ((e.y >> i) & 1u))
				c.y = min(c.y, cu[j].y);
		}
	}
	const int lim = N < 6 ? N : 6;
	for (;;)
	{
		int2 nc = c;
		for (int i = 0; i < lim; ++i)
		{
			const int cx = __shfl_xor(c.x, 1 << i, wave), cy = __shfl_xor(c.y, 1 << i, wave);
			if (active && ((e.x >> i) & 1u))
				nc.x = min(nc.x, cx);
			if (active && ((e.y >> i) & 1u))
				nc.y = min(nc.y, cy);
		}
		const bool ch = nc.x != c.x || nc.y != c.y;
		c = nc;
		if (!__any(ch))
			break;
	}
	if (c.x != c0.x || c.y != c0.y)
	{
		col[v] = c;
		changed[0] = 1;
	}
}

__global__ __launch_bounds__(gblock) void k_assign(int64_t n, int32_t* __restrict__ scc, const int2* __restrict__ col,
												   int32_t* __restrict__ remaining)
{
	__shared__ int s_left;
	if (threadIdx.x == 0)
		s_left = 0;
	__syncthreads();
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	int left = 0;
	if (v < n && scc[v] < 0)
	{
		const int2 c = col[v];
		if (c.x == c.y)
			scc[v] = c.x;
		else
			left = 1;
	}
	const int cnt = __popcll(__ballot(left));
	if (lane_id() == 0 && cnt)
		atomicAdd(&s_left, cnt);
	__syncthreads();
	if (threadIdx.x == 0 && s_left)
		atomicAdd(remaining, s_left);
}

// ---- heights, kept at the roots: h[r] = max(h[r], 1 + h of every successor SCC)
__global__ __launch_bounds__(gblock) void k_height_init(int64_t n, int32_t* __restrict__ h)
{
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	if (v < n)
		h[v] = 1;
}

template <int HMAX>
__global__ __launch_bounds__(gblock) void k_height(int N, int64_t n, const uint32_t* __restrict__ mask,
												   const int32_t* __restrict__ scc, int32_t* __restrict__ h,
												   int32_t* __restrict__ changed, const int32_t* __restrict__ prev)
{
	if (converged(prev))
		return;
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	const bool valid = v < n;
	const int64_t vv = valid ? v : 0;
	const uint32_t mv = valid ? mask[v] : 0u;
	const int32_t r = scc[vv];
	const int32_t h0 = h[r];
	int32_t c = h0;
	if (HMAX > 0)
	{
		int32_t rw[HMAX > 0 ? HMAX : 1], hw[HMAX > 0 ? HMAX : 1];
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
			rw[j] = scc[vv ^ (int64_t(1) << high_bit(j, N))];
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
			hw[j] = h[rw[j]]; // every lane gathers, so the loads are issued together
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
			if (6 + j < N && ((mv >> (6 + j)) & 1u) && rw[j] != r)
				c = max(c, hw[j] + 1);
	}
	const int lim = N < 6 ? N : 6;
	uint32_t out = 0; // edges along the low bits into other SCCs
	for (int i = 0; i < lim; ++i)
	{
		const int32_t ru = __shfl_xor(r, 1 << i, wave);
		out |= ru != r ? mv & (1u << i) : 0u;
	}
	for (;;)
	{
		int32_t nc = c;
		for (int i = 0; i < lim; ++i)
		{
			const int32_t cu = __shfl_xor(c, 1 << i, wave);
			if ((out >> i) & 1u)
				nc = max(nc, cu + 1);
		}
		const bool ch = nc != c;
		c = nc;
		if (!__any(ch))
			break;
	}
	const bool up = c > h0;
	if (up)
		changed[0] = 1;
	if (up && r == (int32_t)v)
		atomicMax(h + r, c);
	// the other members of an SCC: one atomic per wave, and none for a height that others
	// have reported since (a million members of one SCC took 1.5 ms)
	for (uint64_t m = __ballot(up && r != (int32_t)v); m;)
	{
		const int lead = __ffsll((unsigned long long)m) - 1;
		const int32_t rl = __shfl(r, lead, wave);
		const uint64_t same = m & __ballot(r == rl);
		const int32_t mx = wave_max((same >> lane_id() & 1) ? c : 0);
		if (lane_id() == lead && mx > __hip_atomic_load(h + rl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
			atomicMax(h + rl, mx);
		m &= ~same;
	}
}

// info[0] = max height, info[1] = SCCs of height 1 (both zeroed before)
__global__ __launch_bounds__(gblock) void k_height_stats(int64_t n, const int32_t* __restrict__ scc,
														 const int32_t* __restrict__ h, int32_t* __restrict__ info)
{
	__shared__ int s_max[gblock / wave], s_cnt[gblock / wave];
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	const int32_t hv = v < n && scc[v] == (int32_t)v ? h[v] : 0;
	const int mx = wave_max(hv), cnt = __popcll(__ballot(hv == 1));
	if (lane_id() == 0)
		s_max[threadIdx.x / wave] = mx, s_cnt[threadIdx.x / wave] = cnt;
	__syncthreads();
	if (threadIdx.x == 0)
	{
		int m = 0, t = 0;
		for (int i = 0; i < gblock / wave; ++i)
			m = max(m, s_max[i]), t += s_cnt[i];
		if (m)
			atomicMax(info, m);
		if (t)
			atomicAdd(info + 1, t);
	}
}

// ---- the whole stage for n <= 4096 states, by one workgroup: state arrays in LDS, up
// to 4 vertices per thread.  Passes update in place: all relaxations are monotone.  A
// pass is vector instructions on one compute unit, some 10 per vertex and bit: with 4096
// states the stage is 1.7 to 2.4 times as fast as by launches (12 networks), with 8192
// 0.7 to 1.5 times, so the line lies between.
constexpr int gs_block = 1024, gs_v = 4, gs_bits = 12;
constexpr int64_t gs_max = gs_block * gs_v;
constexpr int gs_none = 0xffff; // no SCC yet

inline size_t graph_small_lds(int64_t n) { return (size_t)n * (2 * sizeof(uint32_t) + sizeof(uint32_t) + sizeof(uint16_t)); }

// info: SCCs, terminal SCCs, max height, rounds, passes
__global__ __launch_bounds__(gs_block) void k_graph_small(int N, const uint32_t* __restrict__ mask,
														  int32_t* __restrict__ scc, int32_t* __restrict__ rank,
														  int32_t* __restrict__ height, int32_t* __restrict__ reordered,
														  int32_t* __restrict__ offsets, int32_t* __restrict__ info)
{
	extern __shared__ __align__(16) unsigned char gs_smem[];
	__shared__ int s_red[gs_block / wave + 1], s_max, s_term;
	const int n = 1 << N, t = threadIdx.x;
	uint64_t* const s_key = reinterpret_cast<uint64_t*>(gs_smem); // in the order, where these two were
	uint32_t* const s_mask = reinterpret_cast<uint32_t*>(gs_smem);
	uint32_t* const s_cls = s_mask + n;
	uint32_t* const s_col = s_cls + n; // colours x | y << 16, then heights of the roots
	uint16_t* const s_scc = reinterpret_cast<uint16_t*>(s_col + n);
	int rounds = 0, passes = 0;
	uint32_t in[gs_v], out[gs_v];
	if (t == 0)
		s_max = s_term = 0;
	for (int v = t; v < n; v += gs_block)
	{
		s_mask[v] = mask[v];
		s_cls[v] = 0;
		s_scc[v] = (uint16_t)gs_none;
	}
	__syncthreads();
	for (;;)
	{
		++rounds;
#pragma unroll
		for (int q = 0; q < gs_v; ++q)
		{
			const int v = t + q * gs_block;
			in[q] = out[q] = 0;
			if (v >= n || s_scc[v] != gs_none)
				continue;
			const uint32_t mv = s_mask[v], cv = s_cls[v];
#pragma unroll
			for (int i = 0; i < gs_bits; ++i)
			{
				const int u = v ^ (1 << i);
				if (i < N && s_scc[u] == gs_none && s_cls[u] == cv)
				{
					in[q] |= s_mask[u] & (1u << i);
					out[q] |= mv & (1u << i);
				}
			}
		}
		__syncthreads();
		for (int ch = 1; ch;)
		{
			ch = 0;
			++passes;
#pragma unroll
			for (int q = 0; q < gs_v; ++q)
			{
				const int v = t + q * gs_block;
				if (v >= n || s_scc[v] != gs_none)
					continue;
				uint32_t act = 0;
#pragma unroll
				for (int i = 0; i < gs_bits; ++i)
					if (i < N)
						act |= s_scc[v ^ (1 << i)] == gs_none ? 1u << i : 0u;
				if (!(in[q] & act) || !(out[q] & act))
				{
					s_scc[v] = (uint16_t)v;
					ch = 1;
				}
			}
			ch = __syncthreads_or(ch);
		}
		for (int v = t; v < n; v += gs_block)
			s_col[v] = s_scc[v] == gs_none ? (uint32_t)v | (uint32_t)v << 16 : 0xffffffffu;
		__syncthreads();
		for (int ch = 1; ch;)
		{
			ch = 0;
			++passes;
#pragma unroll
			for (int q = 0; q < gs_v; ++q)
			{
				const int v = t + q * gs_block;
				if (v >= n || s_scc[v] != gs_none)
					continue;
				const uint32_t c0 = s_col[v];
				uint32_t x = c0 & 0xffffu, y = c0 >> 16;
#pragma unroll
				for (int i = 0; i < gs_bits; ++i)
				{
					if (i >= N)
						continue;
					const uint32_t cu = s_col[v ^ (1 << i)];
					if ((in[q] >> i) & 1u)
						x = min(x, cu & 0xffffu);
					if ((out[q] >> i) & 1u)
						y = min(y, cu >> 16);
				}
				const uint32_t c = x | y << 16;
				if (c != c0)
				{
					s_col[v] = c;
					ch = 1;
				}
			}
			ch = __syncthreads_or(ch);
		}
		int left = 0;
		for (int v = t; v < n; v += gs_block)
		{
			if (s_scc[v] != gs_none)
				continue;
			const uint32_t c = s_col[v];
			if ((c & 0xffffu) == c >> 16)
				s_scc[v] = (uint16_t)(c & 0xffffu);
			else
			{
				s_cls[v] = c;
				left = 1;
			}
		}
		if (!__syncthreads_or(left))
			break;
	}

	// heights; out: edges into other SCCs
#pragma unroll
	for (int q = 0; q < gs_v; ++q)
	{
		const int v = t + q * gs_block;
		out[q] = 0;
		if (v >= n)
			continue;
#pragma unroll
		for (int i = 0; i < gs_bits; ++i)
			if (i < N)
				out[q] |= s_scc[v ^ (1 << i)] != s_scc[v] ? s_mask[v] & (1u << i) : 0u;
		s_col[v] = 1;
	}
	__syncthreads();
	for (int ch = 1; ch;)
	{
		ch = 0;
		++passes;
#pragma unroll
		for (int q = 0; q < gs_v; ++q)
		{
			const int v = t + q * gs_block;
			if (v >= n || !out[q])
				continue;
			const int r = s_scc[v];
			const uint32_t h0 = s_col[r];
			uint32_t c = h0;
#pragma unroll
			for (int i = 0; i < gs_bits; ++i)
				if ((out[q] >> i) & 1u)
					c = max(c, s_col[s_scc[v ^ (1 << i)]] + 1);
			if (c > h0)
			{
				atomicMax(s_col + r, c);
				ch = 1;
			}
		}
		ch = __syncthreads_or(ch);
	}
	int mx = 0, term = 0;
	for (int v = t; v < n; v += gs_block)
		if (s_scc[v] == v)
		{
			mx = max(mx, (int)s_col[v]);
			term += s_col[v] == 1;
		}
	mx = wave_max(mx), term = wave_sum(term);
	if (lane_id() == 0)
	{
		atomicMax(&s_max, mx);
		atomicAdd(&s_term, term);
	}
	__syncthreads();

	// the canonical order: (height class, SCC, vertex) in 64 bits, sorted in place
	const int H = s_max;
	for (int v = t; v < n; v += gs_block)
	{
		const int r = s_scc[v], hv = (int)s_col[r];
		const uint64_t hi = hv == 1 ? 0 : H + 1 - hv, lo = hv == 1 ? r : n - 1 - r;
		s_key[v] = hi << 2 * gs_bits | lo << gs_bits | (uint64_t)v;
		scc[v] = r;
		height[v] = hv;
	}
	__syncthreads();
	for (int k = 2; k <= n; k <<= 1)
		for (int j = k >> 1; j > 0; j >>= 1)
		{
			for (int i = t; i < n / 2; i += gs_block)
			{
				const int a = 2 * i - (i & (j - 1)), b = a + j;
				const uint64_t x = s_key[a], y = s_key[b];
				if ((x > y) == ((a & k) == 0))
				{
					s_key[a] = y;
					s_key[b] = x;
				}
			}
			__syncthreads();
		}
	const int per = (n + gs_block - 1) / gs_block, p0 = t * per, p1 = min(n, p0 + per);
	int first = 0, S;
	for (int p = p0; p < p1; ++p)
		first += p == 0 || s_key[p] >> gs_bits != s_key[p - 1] >> gs_bits;
	int k = block_excl_scan<gs_block>(first, s_red, S) - 1;
	for (int p = p0; p < p1; ++p)
	{
		const int v = (int)(s_key[p] & (gs_max - 1));
		if (p == 0 || s_key[p] >> gs_bits != s_key[p - 1] >> gs_bits)
			offsets[++k] = p;
		reordered[p] = v;
		rank[v] = k;
	}
	if (t == 0)
	{
		offsets[S] = n;
		info[0] = S, info[1] = s_term, info[2] = H, info[3] = rounds, info[4] = passes;
	}
}

// ---- canonical order
// root key: terminal -> (0, id); transient -> (H + 1 - h, n - 1 - id), the id in N bits
__global__ __launch_bounds__(gblock) void k_root_keys(int N, int64_t n, const int32_t* __restrict__ scc,
													  const int32_t* __restrict__ h, int32_t H,
													  const int32_t* __restrict__ root_pos,
													  uint64_t* __restrict__ keys, int32_t* __restrict__ vals)
{
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	if (v >= n)
		return;
	const int32_t r = scc[v];
	if (r != (int32_t)v)
		return;
	const int32_t hv = h[v];
	const uint64_t hi = hv == 1 ? 0ull : (uint64_t)(H + 1 - hv);
	const uint64_t lo = hv == 1 ? (uint64_t)v : (uint64_t)(n - 1 - v);
	const int32_t p = root_pos[v];
	keys[p] = (hi << N) | lo;
	vals[p] = (int32_t)v;
}

__global__ __launch_bounds__(gblock) void k_is_root(int64_t n, const int32_t* __restrict__ scc,
													int32_t* __restrict__ flag)
{
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	if (v < n)
		flag[v] = scc[v] == (int32_t)v ? 1 : 0;
}

__global__ __launch_bounds__(gblock) void k_rank_roots(int64_t S, const int32_t* __restrict__ sorted_roots,
													   int32_t* __restrict__ rank)
{
	const int64_t k = (int64_t)blockIdx.x * gblock + threadIdx.x;
	if (k >= S)
		return;
	rank[sorted_roots[k]] = (int32_t)k; // rank is indexed by root vertex here
}

// sccs_offsets from the vertices sorted by SCC rank: offsets[k] = first position of rank k
__global__ __launch_bounds__(gblock) void k_seg_bounds(int64_t n, int64_t S, const uint32_t* __restrict__ sorted_keys,
													   int32_t* __restrict__ offsets)
{
	const int64_t p = (int64_t)blockIdx.x * gblock + threadIdx.x;
	if (p >= n)
		return;
	const uint32_t k = sorted_keys[p];
	if (p == 0 || sorted_keys[p - 1] != k)
		offsets[k] = (int32_t)p;
	if (p == n - 1)
		offsets[S] = (int32_t)n;
}

__global__ __launch_bounds__(gblock) void k_vertex_keys(int64_t n, const int32_t* __restrict__ scc,
														const int32_t* __restrict__ h,
														const int32_t* __restrict__ root_rank,
														uint32_t* __restrict__ keys, int32_t* __restrict__ vals,
														int32_t* __restrict__ vrank, int32_t* __restrict__ vheight)
{
	const int64_t v = (int64_t)blockIdx.x * gblock + threadIdx.x;
	if (v >= n)
		return;
	const int32_t r = scc[v];
	const int32_t k = root_rank[r];
	keys[v] = (uint32_t)k;
	vals[v] = (int32_t)v;
	vrank[v] = k;
	vheight[v] = h[r];
}

namespace {

struct pass_flags
{
	ctx_t& c;
	int32_t* d;
	explicit pass_flags(ctx_t& ctx) : c(ctx), d(ctx.flags.get()) {}
	void clear(int k) { ESL_HIP(hipMemsetAsync(d + k, 0, sizeof(int32_t), c.stream)); }
	int32_t read(int k)
	{
		ESL_HIP(hipMemcpyAsync(c.h_flags + k, d + k, sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
		ESL_HIP(hipStreamSynchronize(c.stream));
		return c.h_flags[k];
	}
};

// one launch and one round trip: 10 nodes 0.14 ms, by passes over device memory 1.52
void graph_small(ctx_t& c, graph_t& g)
{
	const size_t lds = graph_small_lds(g.n);
	ESL_HIP(hipFuncSetAttribute((const void*)k_graph_small, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
	g.offsets.ensure(g.n + 1); // as many SCCs as states at most
	int32_t* d = c.flags.get();
	ESL_HIP(hipEventRecord(c.ev[2], c.stream));
	timed_launch(c, "k_graph_small", 24.0 * g.n, [&] {
		k_graph_small<<<1, gs_block, lds, c.stream>>>(g.N, g.mask.get(), g.scc.get(), g.rank.get(), g.height.get(),
													  g.reordered.get(), g.offsets.get(), d);
	});
	ESL_HIP(hipGetLastError());
	ESL_HIP(hipEventRecord(c.ev[3], c.stream));
	static_assert((gs_max + 1) * sizeof(int32_t) <= stage_bytes, "the offsets fit the staging buffer");
	int32_t* h_off = reinterpret_cast<int32_t*>(c.h_stage);
	ESL_HIP(hipMemcpyAsync(c.h_flags, d, 5 * sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
	ESL_HIP(hipMemcpyAsync(h_off, g.offsets.get(), (g.n + 1) * sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
	ESL_HIP(hipStreamSynchronize(c.stream));
	++g.host_syncs;
	float ms = 0;
	ESL_HIP(hipEventElapsedTime(&ms, c.ev[2], c.ev[3]));
	g.stage_ms[1] = ms;
	g.S = c.h_flags[0];
	g.T = c.h_flags[1];
	g.H = c.h_flags[2];
	g.scc_rounds = c.h_flags[3];
	g.mask_passes = c.h_flags[4];
	g.h_offsets.assign(h_off, h_off + g.S + 1);
	g.n_t = g.h_offsets[g.T];
	g.reorganized = true;
}

} // namespace

void graph_reorganize(ctx_t& c, graph_t& g)
{
	const int N = g.N;
	const int64_t n = g.n;
	const int nb = ceil_div(n, gblock);
	pass_flags fl(c);

	g.scc.ensure(n);
	g.rank.ensure(n);
	g.height.ensure(n);
	g.reordered.ensure(n);
	g.mask_passes = g.scc_rounds = g.host_syncs = 0;
	if (n <= gs_max && graph_small_lds(n) + 4096 <= (size_t)c.lds_per_block)
	{
		graph_small(c, g);
		return;
	}
	dbuf<int2> col, cls;
	col.ensure(n);
	cls.ensure(n);
	dbuf<uint2> edges;
	edges.ensure(n);

	ESL_HIP(hipEventRecord(c.ev[2], c.stream));
	ESL_HIP(hipMemsetAsync(g.scc.get(), 0xff, n * sizeof(int32_t), c.stream));

	const int max_passes = 1 << 20;
	const int pass_group = 8;	   // fixpoint passes per host round trip, after the first
	int hint[3] = { 8, 8, 8 }; // first-group sizes of the three fixpoints
	int64_t prev_left = n + 1;
	auto count = [&](fixpoint_t f) {
		g.mask_passes += f.passes;
		g.host_syncs += f.syncs;
	};
	for (int round = 0;; ++round)
	{
		++g.scc_rounds;
		++g.mask_passes;
		timed_launch(c, "k_edges", (round ? 24.0 : 16.0) * n, [&] {
			ESL_HMAX_DISPATCH(N, k_edges,
							  <<<nb, gblock, 0, c.stream>>>(N, n, g.mask.get(), g.scc.get(),
															round ? cls.get() : nullptr, edges.get()));
		});
		// algorithmic bytes of a pass: edges and the labels it reads and writes
		count(fixpoint(c, hint[0], pass_group, max_passes, "trim", [&](int32_t* f, const int32_t* pf) {
			timed_launch(c, "k_trim", 16.0 * n, [&] {
				ESL_HMAX_DISPATCH(N, k_trim, <<<nb, gblock, 0, c.stream>>>(N, n, edges.get(), g.scc.get(), f, pf));
			});
		}));
		k_color_init<<<nb, gblock, 0, c.stream>>>(n, g.scc.get(), col.get());
		count(fixpoint(c, hint[1], pass_group, max_passes, "colouring", [&](int32_t* f, const int32_t* pf) {
			timed_launch(c, "k_color", 24.0 * n, [&] {
				ESL_HMAX_DISPATCH(N, k_color, <<<nb, gblock, 0, c.stream>>>(N, n, edges.get(), col.get(), f, pf));
			});
		}));
		fl.clear(1);
		timed_launch(c, "k_assign", 16.0 * n,
					 [&] { k_assign<<<nb, gblock, 0, c.stream>>>(n, g.scc.get(), col.get(), fl.d + 1); });
		ESL_HIP(hipGetLastError());
		const int32_t left = fl.read(1);
		++g.host_syncs;
		if (!left)
			break;
		// every round removes at least the SCC of the smallest active vertex
		if (left >= prev_left)
			throw error(ESL_E_DEVICE, "SCC round made no progress");
		prev_left = left;
		std::swap(col, cls);
	}

	// heights (per root)
	dbuf<int32_t> is_root, root_pos;
	is_root.ensure(n);
	root_pos.ensure(n + 1);
	k_is_root<<<nb, gblock, 0, c.stream>>>(n, g.scc.get(), is_root.get());
	exclusive_scan_i32(c, is_root.get(), root_pos.get(), n);
	dbuf<int32_t> hroot;
	hroot.ensure(n);
	k_height_init<<<nb, gblock, 0, c.stream>>>(n, hroot.get());
	count(fixpoint(c, hint[2], 16, max_passes, "height relaxation", [&](int32_t* f, const int32_t* pf) {
		timed_launch(c, "k_height", 16.0 * n, [&] {
			ESL_HMAX_DISPATCH(N, k_height,
							  <<<nb, gblock, 0, c.stream>>>(N, n, g.mask.get(), g.scc.get(), hroot.get(), f, pf));
		});
	}));
	constexpr int hinfo = 2;
	ESL_HIP(hipMemsetAsync(fl.d + hinfo, 0, 2 * sizeof(int32_t), c.stream));
	k_height_stats<<<nb, gblock, 0, c.stream>>>(n, g.scc.get(), hroot.get(), fl.d + hinfo);
	ESL_HIP(hipGetLastError());
	ESL_HIP(hipMemcpyAsync(c.h_flags + hinfo, fl.d + hinfo, 2 * sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
	ESL_HIP(hipMemcpyAsync(c.h_flags + hinfo + 2, root_pos.get() + n, sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
	ESL_HIP(hipStreamSynchronize(c.stream));
	++g.host_syncs;
	g.H = c.h_flags[hinfo];
	g.T = c.h_flags[hinfo + 1];
	const int32_t S = c.h_flags[hinfo + 2], T = (int32_t)g.T;
	g.S = S;

	// sort roots by key
	dbuf<uint64_t> rkeys, rkeys_out;
	dbuf<int32_t> rvals, rvals_out;
	rkeys.ensure(S);
	rkeys_out.ensure(S);
	rvals.ensure(S);
	rvals_out.ensure(S);
	k_root_keys<<<nb, gblock, 0, c.stream>>>(N, n, g.scc.get(), hroot.get(), g.H, root_pos.get(), rkeys.get(),
											 rvals.get());
	ESL_HIP(hipGetLastError());
	unsigned key_bits = N; // a key is at most (H + 1) << N
	while ((int64_t(1) << (key_bits - N)) < (int64_t)g.H + 2)
		++key_bits;
	size_t tmp_bytes = 0;
	ESL_HIP(rocprim::radix_sort_pairs(nullptr, tmp_bytes, rkeys.get(), rkeys_out.get(), rvals.get(),
									  rvals_out.get(), (size_t)S, 0, key_bits, c.stream));
	dbuf<uint8_t> tmp;
	tmp.ensure(tmp_bytes);
	ESL_HIP(rocprim::radix_sort_pairs(tmp.get(), tmp_bytes, rkeys.get(), rkeys_out.get(), rvals.get(),
									  rvals_out.get(), (size_t)S, 0, key_bits, c.stream));
	dbuf<int32_t> root_rank;
	root_rank.ensure(n);
	k_rank_roots<<<ceil_div(S, gblock), gblock, 0, c.stream>>>(S, rvals_out.get(), root_rank.get());

	// stable sort of the vertices by their SCC's rank
	dbuf<uint32_t> vkeys, vkeys_out;
	dbuf<int32_t> vvals;
	vkeys.ensure(n);
	vkeys_out.ensure(n);
	vvals.ensure(n);
	k_vertex_keys<<<nb, gblock, 0, c.stream>>>(n, g.scc.get(), hroot.get(), root_rank.get(), vkeys.get(),
											   vvals.get(), g.rank.get(), g.height.get());
	ESL_HIP(hipGetLastError());
	unsigned end_bit = 1;
	while ((int64_t(1) << end_bit) < (int64_t)S)
		++end_bit;
	tmp_bytes = 0;
	ESL_HIP(rocprim::radix_sort_pairs(nullptr, tmp_bytes, vkeys.get(), vkeys_out.get(), vvals.get(),
									  g.reordered.get(), (size_t)n, 0, end_bit, c.stream));
	tmp.ensure(tmp_bytes);
	ESL_HIP(rocprim::radix_sort_pairs(tmp.get(), tmp_bytes, vkeys.get(), vkeys_out.get(), vvals.get(),
									  g.reordered.get(), (size_t)n, 0, end_bit, c.stream));
	g.offsets.ensure(S + 1);
	k_seg_bounds<<<nb, gblock, 0, c.stream>>>(n, S, vkeys_out.get(), g.offsets.get());
	ESL_HIP(hipGetLastError());
	ESL_HIP(hipEventRecord(c.ev[3], c.stream));
	g.h_offsets.resize(S + 1);
	ESL_HIP(hipMemcpyAsync(g.h_offsets.data(), g.offsets.get(), (S + 1) * sizeof(int32_t), hipMemcpyDeviceToHost,
						   c.stream));
	ESL_HIP(hipStreamSynchronize(c.stream));
	++g.host_syncs;
	float ms = 0;
	ESL_HIP(hipEventElapsedTime(&ms, c.ev[2], c.ev[3]));
	g.stage_ms[1] = ms;
	g.n_t = g.h_offsets[T];
	g.reorganized = true;
}

// ---- graph stage results supplied by the caller (a stored .symb file)

// rank[v] = index of v's SCC in the canonical order, scc[v] = its minimum vertex
// (the first of the SCC's block, vertices being ascending inside a block)
__global__ __launch_bounds__(gblock) void k_import_rank(int64_t n, int64_t S, const int32_t* __restrict__ offsets,
														const int32_t* __restrict__ reordered, int32_t* __restrict__ rank,
														int32_t* __restrict__ scc)
{
	const int64_t p = (int64_t)blockIdx.x * gblock + threadIdx.x;
	if (p >= n)
		return;
	int64_t lo = 0, hi = S; // offsets[lo] <= p < offsets[hi]
	while (hi - lo > 1)
	{
		const int64_t mid = (lo + hi) / 2;
		if (offsets[mid] <= p)
			lo = mid;
		else
			hi = mid;
	}
	const int32_t v = reordered[p];
	rank[v] = (int32_t)lo;
	scc[v] = reordered[offsets[lo]];
}

void graph_import(ctx_t& c, graph_t& g, const int32_t* h_reordered, const int32_t* h_offsets, int64_t S, int64_t T)
{
	const int64_t n = g.n;
	if (S < 1 || T < 1 || T > S || S > n)
		throw error(ESL_E_ARG, "graph import: bad SCC counts");
	if (h_offsets[0] != 0 || h_offsets[S] != n)
		throw error(ESL_E_ARG, "graph import: offsets must start at 0 and end at the state count");
	for (int64_t k = 0; k < S; ++k)
		if (h_offsets[k + 1] <= h_offsets[k])
			throw error(ESL_E_ARG, "graph import: empty or decreasing SCC block");
	std::vector<uint8_t> seen(n, 0);
	for (int64_t k = 0; k < S; ++k)
		for (int32_t p = h_offsets[k]; p < h_offsets[k + 1]; ++p)
		{
			const int32_t v = h_reordered[p];
			if (v < 0 || v >= n || seen[v])
				throw error(ESL_E_ARG, "graph import: reordered vertices are not a permutation");
			seen[v] = 1;
			if (p > h_offsets[k] && v <= h_reordered[p - 1])
				throw error(ESL_E_ARG, "graph import: vertices must ascend inside an SCC");
		}
	g.reordered.ensure(n);
	g.offsets.ensure(S + 1);
	g.rank.ensure(n);
	g.scc.ensure(n);
	ESL_HIP(hipMemcpyAsync(g.reordered.get(), h_reordered, n * sizeof(int32_t), hipMemcpyHostToDevice, c.stream));
	ESL_HIP(hipMemcpyAsync(g.offsets.get(), h_offsets, (S + 1) * sizeof(int32_t), hipMemcpyHostToDevice, c.stream));
	k_import_rank<<<ceil_div(n, gblock), gblock, 0, c.stream>>>(n, S, g.offsets.get(), g.reordered.get(),
																g.rank.get(), g.scc.get());
	ESL_HIP(hipGetLastError());
	ESL_HIP(hipStreamSynchronize(c.stream));
	g.h_offsets.assign(h_offsets, h_offsets + S + 1);
	g.S = S;
	g.T = T;
	g.n_t = h_offsets[T];
	g.H = 0; // heights are not stored
	g.stage_ms[1] = 0.0;
	g.sol = solution_t{};
	g.reorganized = true;
}

} // namespace esl
