// Numeric stages on the device: stationary vector lim exp(K t) x0.
//
// Replaces solver::solve (reference cuda/src/solver.cu:102-334) and
// solve_system / splu / refactor (cuda/src/linear_system_solve.cu:249-626).
//
// The reference builds the kinetic matrix as CSC (scatter_rows_data,
// kernels/solver.cu:4-45), factors it per SCC (dense cuSOLVER getrf for SCCs up
// to 20,000 states, host sparse LU above) and solves one right-hand side per
// terminal SCC.  On random networks at N = 20 single SCCs hold 10^5..10^6
// states and an LU of such a block fills in by two to three orders of
// magnitude, so this path does three things instead:
//
// 1. Operator without stored values.  K[s, t] = rate(t -> s) is a function of
//    the flip mask and the 2N rates only: t = s ^ (1 << i), t -> s iff bit i of
//    mask[t], rate = rates[2i + (s > t ? 0 : 1)] (kernels/solver.cu:33-36).
//    Every product reads the 4-byte mask and the vector, never a value array.
// 2. Exact pruning (x* is unchanged):
//    - states not reachable from supp(x0) end with probability 0;
//    - a transient state whose successors all lead to one terminal SCC sends
//      all its mass there; only "ambiguous" transient states (reaching two or
//      more terminal SCCs) enter a linear system.  Predecessors of an
//      ambiguous state are ambiguous, so that system is closed:
//          (D - A_AA) v = x0_A          (v = expected time spent per state),
//      and terminal SCC j receives y_j = x0 mass that starts in or is bound
//      for j plus the rate-weighted flow v_t * rate(t -> s) of every edge
//      leaving A towards j.  This is R L x0 of solver.cu:302-309 through the
//      single right-hand side N w = x0_nt (w = -v).
//    - a terminal SCC of one state has pi = 1.
// 3. Terminal kernels: for every reachable terminal SCC C of two or more
//    states, K_C pi = 0 with the row of an anchor state a replaced by e_a
//    (pi_a = 1), normalised afterwards.  The anchor is the state of largest
//    mass after a few damped Jacobi sweeps of the singular system, chosen per
//    rate set.
//
// Both systems are solved together, for every rate set of a batch, by BiCGStab on
// the system reduced by one parity class of the states (reduced.hip.hpp), in FP64.
// An explicit restart length, a preconditioner or a pinned schedule asks for restarted
// GMRES with ILU(0) or Jacobi instead, which also finishes the sets that the reduced
// solver leaves: in FP64, or (precision 1) in FP32 cycles on the FP64 residual
// (iterative refinement) until that meets the tolerance.
//
// Vectors are set-major ([set][unknown]); the shared structure (mask, maps,
// unknown list) is a few tens of MB and stays in the 256 MB Infinity Cache
// while the sets stream through.

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <cstdio>
#include <memory>
#include <mutex>
#include <thread>
#include <type_traits>

#include "cube.hip.hpp"
#include "esl_internal.hpp"

namespace esl {

constexpr int sblock = 256;
constexpr int max_rhs_terms = 64; // reachable terminal SCCs tracked by bit masks

// ============================================================================
// setup: reachability, terminal masks, unknown set

__global__ __launch_bounds__(sblock) void k_reach_init(int64_t n, const double* __restrict__ x0,
													   uint8_t* __restrict__ reach)
{
	const int64_t v = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (v < n)
		reach[v] = x0[v] > 0.0 ? 1 : 0;
}

// v is reached if an in-neighbour is (wave-local fixpoint over bits 0..5).
template <int HMAX>
__global__ __launch_bounds__(sblock) void k_reach(int N, int64_t n, const uint32_t* __restrict__ mask,
												  uint8_t* __restrict__ reach, int32_t* __restrict__ changed,
												  const int32_t* __restrict__ prev)
{
	if (converged(prev))
		return;
	const int64_t v = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const bool valid = v < n;
	const uint32_t mv = valid ? mask[v] : 0u;
	const bool r0 = valid && reach[v];
	bool r = r0;
	if (HMAX > 0 && __any(valid && !r))
	{
		uint32_t mu[HMAX > 0 ? HMAX : 1];
		uint8_t ru[HMAX > 0 ? HMAX : 1];
		const int64_t vv = valid ? v : 0; // lanes past n read vertex 0's neighbours, unused
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
		{
			const int64_t u = vv ^ (int64_t(1) << high_bit(j, N));
			mu[j] = mask[u];
			ru[j] = reach[u];
		}
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
			r |= valid && 6 + j < N && ((mu[j] >> (6 + j)) & 1u) && ru[j];
	}
	const int lim = N < 6 ? N : 6;
	for (;;)
	{
		bool nr = r;
		for (int i = 0; i < lim; ++i)
		{
			const int ru = __shfl_xor((int)r, 1 << i, wave);
			const uint32_t mu = __shfl_xor(mv, 1 << i, wave);
			if (valid && ru && ((mu >> i) & 1u))
				nr = true;
		}
		const bool ch = nr != r;
		r = nr;
		if (!__any(ch))
			break;
	}
	if (r && !r0)
	{
		reach[v] = 1;
		changed[0] = 1;
	}
}

// per terminal SCC k (canonical rank < T): reached if any of its states is
__global__ __launch_bounds__(sblock) void k_term_reached(int64_t n_t, const int32_t* __restrict__ reordered,
														 const int32_t* __restrict__ rank,
														 const uint8_t* __restrict__ reach,
														 int32_t* __restrict__ reached)
{
	const int64_t p = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (p >= n_t)
		return;
	const int32_t s = reordered[p];
	if (reach[s])
		reached[rank[s]] = 1;
}

// tm[s]: bit j set iff s reaches reachable terminal SCC j (j = compact index)
__global__ __launch_bounds__(sblock) void k_tm_init(int64_t n, const int32_t* __restrict__ rank, int64_t T,
													const int32_t* __restrict__ jmap,
													const uint8_t* __restrict__ reach, uint64_t* __restrict__ tm)
{
	const int64_t v = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (v >= n)
		return;
	uint64_t m = 0;
	const int32_t k = rank[v];
	if (reach[v] && k < T)
	{
		const int32_t j = jmap[k];
		if (j >= 0 && j < max_rhs_terms)
			m = 1ull << j;
	}
	tm[v] = m;
}

// pull over out-neighbours: tm[v] |= tm[w] for v -> w (reachable transient v)
template <int HMAX>
__global__ __launch_bounds__(sblock) void k_tm(int N, int64_t n, const uint32_t* __restrict__ mask,
											   const int32_t* __restrict__ rank, int64_t T,
											   const uint8_t* __restrict__ reach, uint64_t* __restrict__ tm,
											   int32_t* __restrict__ changed, const int32_t* __restrict__ prev)
{
	if (converged(prev))
		return;
	const int64_t v = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const bool valid = v < n;
	const bool act = valid && reach[v] && rank[v] >= T;
	const uint32_t mv = valid ? mask[v] : 0u;
	const uint64_t m0 = valid ? tm[v] : 0ull;
	uint64_t m = m0;
	if (HMAX > 0 && __any(act))
	{
		uint64_t mu[HMAX > 0 ? HMAX : 1];
		const int64_t vv = valid ? v : 0;
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
			mu[j] = tm[vv ^ (int64_t(1) << high_bit(j, N))];
#pragma unroll
		for (int j = 0; j < HMAX; ++j)
			if (act && 6 + j < N && ((mv >> (6 + j)) & 1u))
				m |= mu[j];
	}
	const int lim = N < 6 ? N : 6;
	for (;;)
	{
		uint64_t nm = m;
		for (int i = 0; i < lim; ++i)
		{
			const uint64_t mw = __shfl_xor(m, 1 << i, wave);
			if (act && ((mv >> i) & 1u))
				nm |= mw;
		}
		const bool ch = nm != m;
		m = nm;
		if (!__any(ch))
			break;
	}
	if (act && m != m0)
	{
		tm[v] = m;
		changed[0] = 1;
	}
}

// ambiguous transient: reachable and reaching >= 2 terminal SCCs (or every
// reachable transient state when more than 64 terminal SCCs are reached)
__global__ __launch_bounds__(sblock) void k_amb_flag(int64_t n, const int32_t* __restrict__ rank, int64_t T,
													 const uint8_t* __restrict__ reach,
													 const uint64_t* __restrict__ tm, int fallback,
													 int32_t* __restrict__ flag)
{
	const int64_t v = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (v >= n)
		return;
	int f = 0;
	if (reach[v] && rank[v] >= T)
		f = fallback ? 1 : (__popcll(tm[v]) >= 2);
	flag[v] = f;
}

// terminal-system unknowns first (canonical order), then ambiguous states ascending
__global__ __launch_bounds__(sblock) void k_fill_unknowns(int64_t n, const int32_t* __restrict__ flag,
														  const int32_t* __restrict__ fpos, int64_t base,
														  int32_t* __restrict__ ulist, int32_t* __restrict__ ucls,
														  int32_t* __restrict__ pos)
{
	const int64_t v = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (v >= n || !flag[v])
		return;
	const int64_t u = base + fpos[v];
	ulist[u] = (int32_t)v;
	ucls[u] = -1;
	pos[v] = (int32_t)u;
}

__global__ __launch_bounds__(sblock) void k_fill_term_unknowns(int64_t count, const int32_t* __restrict__ states,
															   const int32_t* __restrict__ seg_of,
															   int32_t* __restrict__ ulist,
															   int32_t* __restrict__ ucls, int32_t* __restrict__ pos)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (u >= count)
		return;
	const int32_t s = states[u];
	ulist[u] = s;
	ucls[u] = seg_of[u];
	pos[s] = (int32_t)u;
}

// Target of the x0 mass of a state that needs no linear solve: the terminal
// SCC it lies in, or the one an unambiguous transient state is bound for
// (compact index j < Tr); -1 for states without mass, unreachable ones and
// ambiguous ones.  The sums y0[j] are taken on the host in state order, so
// they do not depend on the launch.
__global__ __launch_bounds__(sblock) void k_target_of(int64_t n, const int32_t* __restrict__ rank, int64_t T,
													  const int32_t* __restrict__ jmap,
													  const uint8_t* __restrict__ reach,
													  const uint64_t* __restrict__ tm, const int32_t* __restrict__ amb,
													  const double* __restrict__ x0, int Tr, int32_t* __restrict__ tgt,
													  int32_t* __restrict__ has)
{
	const int64_t v = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (v >= n)
		return;
	int j = -1;
	if (reach[v] && !amb[v] && x0[v] != 0.0)
	{
		const int32_t k = rank[v];
		if (k < T)
			j = jmap[k];
		else if (Tr == 1)
			j = 0; // one reachable terminal SCC: every reachable state ends there
		else if (tm[v])
			j = __ffsll((unsigned long long)tm[v]) - 1;
	}
	tgt[v] = j;
	has[v] = j >= 0 ? 1 : 0;
}

__global__ __launch_bounds__(sblock) void k_target_pack(int64_t n, const int32_t* __restrict__ tgt,
														const int32_t* __restrict__ at, const double* __restrict__ x0,
														int32_t* __restrict__ j, double* __restrict__ x)
{
	const int64_t v = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (v >= n || tgt[v] < 0)
		return;
	j[at[v]] = tgt[v];
	x[at[v]] = x0[v];
}

// ============================================================================
// per-set coefficients

struct sys_t
{
	int N;
	int64_t nU;		   // unknowns
	int64_t nUt;	   // terminal-system unknowns (prefix of the unknown list)
	int B;			   // rate sets
	const uint32_t* mask;
	const int32_t* ulist; // state of unknown u
	const int32_t* ucls;  // terminal-system segment of u, -1 for ambiguous transient
	const int32_t* pos;	  // unknown of a state, -1 outside the systems
	const double* rates;  // [B][2N]
	const int32_t* anchor; // [B][n_seg] unknown index of the anchor of each segment
	const double* invd;	   // [B][nU] 1/D' (1 for anchors)
	int transpose;		   // 0: couple in-neighbours (flow of mass); 1: out-neighbours (absorption probabilities)
	int64_t rate_stride;   // doubles between the rate vectors of consecutive sets (2N, or 0 when shared)
};

__device__ __forceinline__ double rate_of(const double* __restrict__ r, int i, bool up)
{
	return r[2 * i + (up ? 0 : 1)];
}

// D_s = total out-rate of state s (all its transitions; up flips use rates[2i], down rates[2i+1])
__device__ __forceinline__ double out_rate_s(uint32_t s, uint32_t m, const double* __restrict__ r)
{
	double d = 0.0;
	while (m)
	{
		const int i = __ffs(m) - 1;
		m &= m - 1;
		d += r[2 * i + ((s >> i) & 1u)];
	}
	return d;
}

// invd[b][u] = 1 / D_s (1 for the anchor of the set's segment)
__global__ __launch_bounds__(sblock) void k_invd(sys_t S, int n_seg, double* __restrict__ invd)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	if (u >= S.nU)
		return;
	const int32_t s = S.ulist[u];
	const int32_t cls = S.ucls[u];
	double v;
	if (cls >= 0 && S.anchor[(int64_t)b * n_seg + cls] == (int32_t)u)
		v = 1.0;
	else
		v = 1.0 / out_rate_s((uint32_t)s, S.mask[s], S.rates + (int64_t)b * S.rate_stride);
	invd[(int64_t)b * S.nU + u] = v;
}

// coupled in-neighbours of s inside the systems, with the coefficient
// rate(t -> s) / D'_t applied to the preconditioned variable z_t.
template <typename T, typename F>
__device__ __forceinline__ void for_coupled(const sys_t& S, int b, uint32_t s, int32_t cls, F&& f)
{
	const double* __restrict__ r = S.rates + (int64_t)b * S.rate_stride;
	if (S.transpose)
	{
		// out-neighbours d of s: coefficient rate(s -> d), up iff bit i of s is 0
		uint32_t m = S.mask[s];
		while (m)
		{
			const int i = __ffs(m) - 1;
			m &= m - 1;
			const int32_t ud = S.pos[s ^ (1u << i)];
			if (ud < 0)
				continue;
			f(ud, rate_of(r, i, ((s >> i) & 1u) == 0));
		}
		return;
	}
	for (int i = 0; i < S.N; ++i)
	{
		const uint32_t t = s ^ (1u << i);
		if (!((S.mask[t] >> i) & 1u))
			continue;
		const int32_t ut = S.pos[t];
		if (ut < 0)
			continue;
		const int32_t ct = S.ucls[ut];
		if ((ct < 0) != (cls < 0))
			continue;
		f(ut, rate_of(r, i, ((s >> i) & 1u) != 0));
	}
}

// W = A_p V:  w_u = v_u - sum_t rate(t -> s) invd_t v_t   (anchor rows: w = v)
template <typename T>
__global__ __launch_bounds__(sblock) void k_apply(sys_t S, int n_seg, const T* __restrict__ V,
												  T* __restrict__ W)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	if (u >= S.nU)
		return;
	const T* __restrict__ vb = V + (int64_t)b * S.nU;
	const double* __restrict__ ib = S.invd + (int64_t)b * S.nU;
	const int32_t s = S.ulist[u];
	const int32_t cls = S.ucls[u];
	double acc = (double)vb[u];
	const bool anchor = cls >= 0 && S.anchor[(int64_t)b * n_seg + cls] == (int32_t)u;
	if (!anchor)
		for_coupled<T>(S, b, (uint32_t)s, cls, [&](int32_t ut, double rate) { acc -= rate * ib[ut] * (double)vb[ut]; });
	W[(int64_t)b * S.nU + u] = (T)acc;
}

// residual in FP64: r = rhs - A_p z, and per-block partial sums of r^2 and rhs^2
__global__ __launch_bounds__(sblock) void k_residual(sys_t S, int n_seg, const double* __restrict__ rhs,
													 const double* __restrict__ z, double* __restrict__ r,
													 double* __restrict__ part)
{
	__shared__ double s_red[2][sblock / wave + 1];
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	double rr = 0.0, bb = 0.0;
	if (u < S.nU)
	{
		const double* __restrict__ zb = z + (int64_t)b * S.nU;
		const double* __restrict__ ib = S.invd + (int64_t)b * S.nU;
		const int32_t s = S.ulist[u];
		const int32_t cls = S.ucls[u];
		double acc = zb[u];
		const bool anchor = cls >= 0 && S.anchor[(int64_t)b * n_seg + cls] == (int32_t)u;
		if (!anchor)
			for_coupled<double>(S, b, (uint32_t)s, cls,
								[&](int32_t ut, double rate) { acc -= rate * ib[ut] * zb[ut]; });
		const double bv = rhs[(int64_t)b * S.nU + u];
		const double res = bv - acc;
		if (r)
			r[(int64_t)b * S.nU + u] = res;
		rr = res * res;
		bb = bv * bv;
	}
	rr = block_sum<sblock>(rr, s_red[0]);
	bb = block_sum<sblock>(bb, s_red[1]);
	if (threadIdx.x == 0)
	{
		part[((int64_t)b * gridDim.x + blockIdx.x) * 2 + 0] = rr;
		part[((int64_t)b * gridDim.x + blockIdx.x) * 2 + 1] = bb;
	}
}

// out[b][k] = sum over blocks of part[b][blk][k]  (one wave per (b, k))
__global__ __launch_bounds__(wave) void k_reduce_parts(const double* __restrict__ part, int nblk, int K,
													   double* __restrict__ out, int64_t ostride, int accumulate)
{
	const int k = blockIdx.x;
	const int b = blockIdx.y;
	double s = 0.0;
	for (int i = threadIdx.x; i < nblk; i += wave)
		s += part[((int64_t)b * nblk + i) * K + k];
	s = wave_sum(s);
	if (threadIdx.x == 0)
		out[(int64_t)b * ostride + k] = accumulate ? out[(int64_t)b * ostride + k] + s : s;
}

// per-set GMRES state (one thread per set)
struct gm_state_t
{
	double* H;	   // [B][(m+1) * m]  column j at H[j*(m+1) + i]
	double* cs;	   // [B][m]
	double* sn;	   // [B][m]
	double* g;	   // [B][m+1]
	double* c1;	   // [B][m+1] first-pass coefficients
	double* c2;	   // [B][m+1] second-pass coefficients
	double* hn;	   // [B] norm of the new vector
	double* beta;  // [B]
	double* bnorm; // [B]
	double* res;   // [B] current residual estimate / |rhs|
	int32_t* live; // [B] 1 while the set iterates in this cycle
	int32_t* act;  // [B] 1 when the set started this cycle above the tolerance
	int32_t* kb;   // [B] Arnoldi steps the set took in this cycle
	double* res0;  // [B] relative residual at the start of the cycle
};

// start of a cycle: beta = |r|, g = (beta, 0..), live = beta > tol*|rhs|
__global__ void k_gm_start(int B, int m, gm_state_t st, const double* __restrict__ rr_bb, double tol,
						   double* __restrict__ vscale)
{
	const int b = blockIdx.x * blockDim.x + threadIdx.x;
	if (b >= B)
		return;
	const double beta = sqrt(rr_bb[(int64_t)b * 2 + 0]);
	const double bn = sqrt(rr_bb[(int64_t)b * 2 + 1]);
	st.beta[b] = beta;
	st.bnorm[b] = bn;
	for (int i = 0; i <= m; ++i)
		st.g[(int64_t)b * (m + 1) + i] = 0.0;
	st.g[(int64_t)b * (m + 1)] = beta;
	const double rel = bn > 0.0 ? beta / bn : beta;
	st.res[b] = rel;
	st.res0[b] = rel;
	const int live = rel > tol ? 1 : 0;
	st.live[b] = live;
	st.act[b] = live;
	st.kb[b] = 0;
	vscale[b] = live ? beta : 0.0; // V_0 = r / beta (0 when the set is done)
}

// H[:, j] = c1 + c2, H[j+1, j] = |w|, Givens update, residual estimate; a set
// stops iterating (and drops out of the Arnoldi kernels) once its estimate
// reaches max(tol_half, rtol * its residual at the start of the cycle)
__global__ void k_gm_givens(int B, int m, int j, gm_state_t st, double tol_half, double rtol)
{
	const int b = blockIdx.x * blockDim.x + threadIdx.x;
	if (b >= B)
		return;
	double* H = st.H + (int64_t)b * (m + 1) * m;
	double* col = H + (int64_t)j * (m + 1);
	double* cs = st.cs + (int64_t)b * m;
	double* sn = st.sn + (int64_t)b * m;
	double* g = st.g + (int64_t)b * (m + 1);
	if (!st.live[b])
	{
		for (int i = 0; i <= m; ++i)
			col[i] = 0.0;
		col[j] = 1.0;
		cs[j] = 1.0;
		sn[j] = 0.0;
		st.hn[b] = 0.0;
		return;
	}
	st.kb[b] = j + 1;
	for (int i = 0; i <= j; ++i)
		col[i] = st.c1[(int64_t)b * (m + 1) + i] + st.c2[(int64_t)b * (m + 1) + i];
	const double hn = sqrt(st.hn[b]);
	col[j + 1] = hn;
	st.hn[b] = hn;
	for (int i = 0; i < j; ++i)
	{
		const double a = col[i], c = col[i + 1];
		col[i] = cs[i] * a + sn[i] * c;
		col[i + 1] = -sn[i] * a + cs[i] * c;
	}
	const double a = col[j], c = col[j + 1];
	const double rnorm = hypot(a, c);
	double cj = 1.0, sj = 0.0;
	if (rnorm > 0.0)
	{
		cj = a / rnorm;
		sj = c / rnorm;
	}
	cs[j] = cj;
	sn[j] = sj;
	col[j] = rnorm;
	col[j + 1] = 0.0;
	g[j + 1] = -sj * g[j];
	g[j] = cj * g[j];
	const double bn = st.bnorm[b];
	const double rel = fabs(g[j + 1]) / (bn > 0.0 ? bn : 1.0);
	st.res[b] = rel;
	if (!(hn > 0.0) || !(rnorm > 0.0) || rel <= fmax(tol_half, rtol * st.res0[b]))
		st.live[b] = 0;
}

// y = H(0:k,0:k)^-1 g(0:k)  written into c1
__global__ void k_gm_solve_y(int B, int m, int k, gm_state_t st)
{
	const int b = blockIdx.x * blockDim.x + threadIdx.x;
	if (b >= B)
		return;
	const double* H = st.H + (int64_t)b * (m + 1) * m;
	const double* g = st.g + (int64_t)b * (m + 1);
	double* y = st.c1 + (int64_t)b * (m + 1);
	k = min(k, st.kb[b]); // the set's own steps in this cycle
	for (int i = k - 1; i >= 0; --i)
	{
		double s = g[i];
		for (int l = i + 1; l < k; ++l)
			s -= H[(int64_t)l * (m + 1) + i] * y[l];
		const double d = H[(int64_t)i * (m + 1) + i];
		y[i] = d != 0.0 ? s / d : 0.0;
	}
	for (int i = k; i <= m; ++i)
		y[i] = 0.0;
}

__global__ __launch_bounds__(sblock) void k_fill_value(int64_t count, double v, double* __restrict__ p)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count)
		p[i] = v;
}

template <typename T>
__global__ __launch_bounds__(sblock) void k_zero(int64_t count, T* __restrict__ p)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count)
		p[i] = (T)0;
}

// the dense final vectors: one 16-byte non-temporal store per thread.  The
// fill runs beside the solve kernel, whose spilled Krylov basis lives in the
// caches: streaming stores leave the caches to it (N=20 bench, fill and solve
// overlapped: 2.96 -> 2.46 ms per step).  16-byte stores beat 8-byte ones
// (6.9 against 6.4 TB/s alone); grid-stride loops were slower.
typedef double zero2_t __attribute__((ext_vector_type(2)));
__global__ __launch_bounds__(sblock) void k_zero2(int64_t count2, double2* __restrict__ p)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count2)
	{
		const zero2_t z = { 0.0, 0.0 };
		__builtin_nontemporal_store(z, (zero2_t*)p + i);
	}
}

// ============================================================================
// anchors: damped Jacobi sweeps p <- p/2 + (sum_t rate(t->s) p_t / D_s)/2 on
// every terminal segment, then the argmax of each segment per set.

// one block per (segment, set): anchor = smallest unknown index of maximal p
__global__ __launch_bounds__(sblock) void k_anchor_pick(int64_t nUt, const int32_t* __restrict__ seg_off,
														const double* __restrict__ p, int n_seg,
														int32_t* __restrict__ anchor)
{
	__shared__ double s_v[sblock];
	__shared__ int32_t s_i[sblock];
	const int k = blockIdx.x;
	const int b = blockIdx.y;
	const int32_t a = seg_off[k], e = seg_off[k + 1];
	double best = -1.0;
	int32_t bi = a;
	for (int32_t u = a + threadIdx.x; u < e; u += sblock)
	{
		const double v = p[(int64_t)b * nUt + u];
		if (v > best)
		{
			best = v;
			bi = u;
		}
	}
	s_v[threadIdx.x] = best;
	s_i[threadIdx.x] = bi;
	__syncthreads();
	for (int w = sblock / 2; w > 0; w >>= 1)
	{
		if (threadIdx.x < w)
		{
			const double v2 = s_v[threadIdx.x + w];
			const int32_t i2 = s_i[threadIdx.x + w];
			if (v2 > s_v[threadIdx.x] || (v2 == s_v[threadIdx.x] && i2 < s_i[threadIdx.x]))
			{
				s_v[threadIdx.x] = v2;
				s_i[threadIdx.x] = i2;
			}
		}
		__syncthreads();
	}
	if (threadIdx.x == 0)
		anchor[(int64_t)b * n_seg + k] = s_i[0];
}

// The anchor choice in one launch when the terminal unknowns fit in LDS: one
// workgroup per rate set runs the same damped Jacobi sweeps as k_anchor_sweep
// (in-neighbours from the coupling lists, summed in their order) and the pick
// of k_anchor_pick.  Dynamic LDS: p, p', D (nUt doubles each), row pointers
// (nUt + 1 int32), neighbour (uint16) and rate code (uint8) per coupling.
__global__ __launch_bounds__(sblock) void k_anchor_lds(sys_t S, const int32_t* __restrict__ gptr,
													   const int32_t* __restrict__ gnu, const uint8_t* __restrict__ gnr,
													   const int32_t* __restrict__ seg_off, int n_seg, int sweeps,
													   int32_t* __restrict__ anchor)
{
	extern __shared__ __align__(16) unsigned char smem[];
	__shared__ double s_rates[64];
	__shared__ double s_v[sblock];
	__shared__ int32_t s_i[sblock];
	const int nUt = (int)S.nUt;
	const int b = blockIdx.x;
	const int tid = threadIdx.x;
	double* p = (double*)smem;
	double* pn = p + nUt;
	double* d = pn + nUt;
	int32_t* ptr = (int32_t*)(d + nUt);
	const int nnz = gptr[nUt];
	uint16_t* nu = (uint16_t*)(ptr + nUt + 1);
	uint8_t* nc = (uint8_t*)(nu + nnz);
	for (int i = tid; i < 2 * S.N; i += sblock)
		s_rates[i] = S.rates[(int64_t)b * S.rate_stride + i];
	__syncthreads();
	for (int u = tid; u < nUt; u += sblock)
	{
		const uint32_t st = (uint32_t)S.ulist[u];
		p[u] = 1.0;
		d[u] = out_rate_s(st, S.mask[st], s_rates);
		ptr[u] = gptr[u];
	}
	if (tid == 0)
		ptr[nUt] = nnz;
	for (int k = tid; k < nnz; k += sblock)
	{
		nu[k] = (uint16_t)gnu[k];
		nc[k] = gnr[k];
	}
	__syncthreads();
	for (int it = 0; it < sweeps; ++it)
	{
		for (int u = tid; u < nUt; u += sblock)
		{
			double inflow = 0.0;
			for (int k = ptr[u]; k < ptr[u + 1]; ++k)
				inflow += s_rates[nc[k] & 63] * p[nu[k]];
			pn[u] = 0.5 * p[u] + 0.5 * inflow / d[u];
		}
		__syncthreads();
		double* t = p;
		p = pn;
		pn = t;
	}
	for (int k = 0; k < n_seg; ++k)
	{
		const int32_t a = seg_off[k], e = seg_off[k + 1];
		double best = -1.0;
		int32_t bi = a;
		for (int32_t u = a + tid; u < e; u += sblock)
			if (p[u] > best)
			{
				best = p[u];
				bi = u;
			}
		s_v[tid] = best;
		s_i[tid] = bi;
		__syncthreads();
		for (int w = sblock / 2; w > 0; w >>= 1)
		{
			if (tid < w)
			{
				const double v2 = s_v[tid + w];
				const int32_t i2 = s_i[tid + w];
				if (v2 > s_v[tid] || (v2 == s_v[tid] && i2 < s_i[tid]))
				{
					s_v[tid] = v2;
					s_i[tid] = i2;
				}
			}
			__syncthreads();
		}
		if (tid == 0)
			anchor[(int64_t)b * n_seg + k] = s_i[0];
		__syncthreads();
	}
}

// right-hand sides: anchors -> 1, other terminal unknowns -> 0, ambiguous -> x0
__global__ __launch_bounds__(sblock) void k_rhs(sys_t S, int n_seg, const double* __restrict__ x0,
												double* __restrict__ rhs)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	if (u >= S.nU)
		return;
	const int32_t cls = S.ucls[u];
	double v;
	if (cls >= 0)
		v = S.anchor[(int64_t)b * n_seg + cls] == (int32_t)u ? 1.0 : 0.0;
	else
		v = x0[S.ulist[u]];
	rhs[(int64_t)b * S.nU + u] = v;
}

// k_invd, k_rhs and a zero start vector in one launch (the plan's set-up sits on
// the path between the anchor choice and the solve)
__global__ __launch_bounds__(sblock) void k_sys_setup(sys_t S, int n_seg, const double* __restrict__ x0,
													  double* __restrict__ invd, double* __restrict__ rhs,
													  double* __restrict__ z)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	if (u >= S.nU)
		return;
	const int32_t s = S.ulist[u];
	const int32_t cls = S.ucls[u];
	const bool anchor = cls >= 0 && S.anchor[(int64_t)b * n_seg + cls] == (int32_t)u;
	const int64_t i = (int64_t)b * S.nU + u;
	invd[i] = anchor ? 1.0 : 1.0 / out_rate_s((uint32_t)s, S.mask[s], S.rates + (int64_t)b * S.rate_stride);
	rhs[i] = cls >= 0 ? (anchor ? 1.0 : 0.0) : x0[s];
	z[i] = 0.0;
}

// ============================================================================
// assembly of the final vector

// Exit edges of the ambiguous set: edges t -> s from an ambiguous unknown u
// (state t) to a state s outside the systems' ambiguous part, with the
// terminal SCC j their mass goes to.  Rate independent, built once per plan;
// listed per u in bit order, then sorted by j on the host (stable), so the
// per-set sums run in a fixed order.
__device__ __forceinline__ int exit_target(const sys_t& S, const int32_t* __restrict__ rank, int64_t T,
										   const int32_t* __restrict__ jmap, const uint64_t* __restrict__ tm,
										   uint32_t s)
{
	const int32_t us = S.pos[s];
	if (us >= (int32_t)S.nUt)
		return -1; // stays ambiguous
	const int32_t k = rank[s];
	if (k < T)
		return jmap[k];
	return __ffsll((unsigned long long)tm[s]) - 1;
}

__global__ __launch_bounds__(sblock) void k_exit_count(sys_t S, const int32_t* __restrict__ rank, int64_t T,
													   const int32_t* __restrict__ jmap,
													   const uint64_t* __restrict__ tm, int32_t* __restrict__ cnt)
{
	const int64_t a = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (a >= S.nU - S.nUt)
		return;
	const uint32_t t = (uint32_t)S.ulist[S.nUt + a];
	uint32_t m = S.mask[t];
	int c = 0;
	while (m)
	{
		const int i = __ffs(m) - 1;
		m &= m - 1;
		c += exit_target(S, rank, T, jmap, tm, t ^ (1u << i)) >= 0 ? 1 : 0;
	}
	cnt[a] = c;
}

__global__ __launch_bounds__(sblock) void k_exit_fill(sys_t S, const int32_t* __restrict__ rank, int64_t T,
													  const int32_t* __restrict__ jmap,
													  const uint64_t* __restrict__ tm,
													  const int32_t* __restrict__ ptr, int32_t* __restrict__ ej,
													  int32_t* __restrict__ eu, uint8_t* __restrict__ er)
{
	const int64_t a = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (a >= S.nU - S.nUt)
		return;
	const int64_t u = S.nUt + a;
	const uint32_t t = (uint32_t)S.ulist[u];
	uint32_t m = S.mask[t];
	int32_t at = ptr[a];
	while (m)
	{
		const int i = __ffs(m) - 1;
		m &= m - 1;
		const int j = exit_target(S, rank, T, jmap, tm, t ^ (1u << i));
		if (j < 0)
			continue;
		ej[at] = j;
		eu[at] = (int32_t)u;
		er[at] = (uint8_t)(2 * i + ((t >> i) & 1u)); // up flip: rates[2i], down: rates[2i + 1]
		++at;
	}
}

// y[b][j] = flow from the ambiguous set into terminal SCC j for set b: the sum
// over j's exit edges of v_t * rate, v = z * invd (expected time in t).  One
// workgroup per (j, set), fixed summation order.
__global__ __launch_bounds__(sblock) void k_exit_sum(sys_t S, const int32_t* __restrict__ ex_off,
													 const int32_t* __restrict__ ex_u, const uint8_t* __restrict__ ex_r,
													 const double* __restrict__ z, int Tr, double* __restrict__ y)
{
	__shared__ double s_red[sblock / wave + 1];
	const int j = blockIdx.x;
	const int b = blockIdx.y;
	const double* __restrict__ r = S.rates + (int64_t)b * S.rate_stride;
	const int64_t off = (int64_t)b * S.nU;
	double acc = 0.0;
#pragma unroll 8 // one latency per 8 terms of a thread
	for (int32_t e = ex_off[j] + threadIdx.x; e < ex_off[j + 1]; e += sblock)
	{
		const int32_t u = ex_u[e];
		acc += z[off + u] * S.invd[off + u] * r[ex_r[e]];
	}
	acc = block_sum<sblock>(acc, s_red);
	if (threadIdx.x == 0)
		y[(int64_t)b * Tr + j] = acc;
}

// segment sums of pi (= z * invd) over each terminal segment, per set
__global__ __launch_bounds__(sblock) void k_seg_sum(int64_t nU, const int32_t* __restrict__ seg_off,
													const double* __restrict__ z, const double* __restrict__ invd,
													int n_seg, double* __restrict__ sums)
{
	__shared__ double s_red[sblock / wave + 1];
	const int k = blockIdx.x;
	const int b = blockIdx.y;
	double acc = 0.0;
	// one latency per 16 terms of a thread instead of one per term (524,288 states in one
	// segment: 512 to 160 us), added in the same order
#pragma unroll 16
	for (int32_t u = seg_off[k] + threadIdx.x; u < seg_off[k + 1]; u += sblock)
		acc += z[(int64_t)b * nU + u] * invd[(int64_t)b * nU + u];
	acc = block_sum<sblock>(acc, s_red);
	if (threadIdx.x == 0)
		sums[(int64_t)b * n_seg + k] = acc;
}

// final[b][s] for every terminal state s of a reached terminal SCC
__global__ __launch_bounds__(sblock) void k_final(int64_t n, int64_t n_t, const int32_t* __restrict__ reordered,
												  const int32_t* __restrict__ rank, const int32_t* __restrict__ jmap,
												  const int32_t* __restrict__ segmap, const int32_t* __restrict__ pos,
												  const double* __restrict__ z, const double* __restrict__ invd,
												  const double* __restrict__ segsum, int n_seg, int64_t nU,
												  const double* __restrict__ y, int Tr, double* __restrict__ out)
{
	const int64_t p = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	if (p >= n_t)
		return;
	const int32_t s = reordered[p];
	const int32_t k = rank[s];
	const int32_t j = jmap[k];
	if (j < 0)
		return;
	double pi = 1.0;
	const int32_t sg = segmap[k];
	if (sg >= 0)
	{
		const int32_t u = pos[s];
		pi = z[(int64_t)b * nU + u] * invd[(int64_t)b * nU + u] / segsum[(int64_t)b * n_seg + sg];
	}
	out[(int64_t)b * n + s] = pi * y[(int64_t)b * Tr + j];
}

__global__ __launch_bounds__(sblock) void k_y_total(int B, int Tr, const double* __restrict__ y0,
													double* __restrict__ y)
{
	const int i = blockIdx.x * sblock + threadIdx.x;
	if (i >= B * Tr)
		return;
	y[i] += y0[i % Tr];
}


// ============================================================================
// Compressed coupling structure of the systems (shared by every set): for each
// unknown u the coupled neighbours k -- in-neighbours for the forward (mass
// flow) system, out-neighbours for the transposed (absorption) one -- with
// the rate index of the off-diagonal entry M[u, k] (bits 0..5) and a flag
// (bit 6) telling whether the mirrored entry M[k, u] exists.  Neighbours of
// smaller state come first (ILU lower part).  M[u, k] = -rates[idx]; the
// mirrored entry uses rates[idx ^ 1].

constexpr int nbr_rev_flag = 64;

__device__ __forceinline__ int coupled_list(const sys_t& S, int64_t u, int32_t* out_u, uint8_t* out_r, int& n_low)
{
	const uint32_t s = (uint32_t)S.ulist[u];
	const int32_t cls = S.ucls[u];
	int cnt = 0;
	n_low = 0;
	for (int pass = 0; pass < 2; ++pass) // 0: neighbours below s, 1: above
		for (int i = 0; i < S.N; ++i)
		{
			const bool below = (s >> i) & 1u; // s ^ (1 << i) < s
			if (below != (pass == 0))
				continue;
			const uint32_t k = s ^ (1u << i);
			bool edge, rev;
			int idx;
			if (S.transpose)
			{
				edge = (S.mask[s] >> i) & 1u; // u -> k
				rev = (S.mask[k] >> i) & 1u;
				idx = 2 * i + (below ? 1 : 0); // u -> k is a down flip when k < s
			}
			else
			{
				edge = (S.mask[k] >> i) & 1u; // k -> u
				rev = (S.mask[s] >> i) & 1u;
				idx = 2 * i + (below ? 0 : 1); // k -> u is an up flip when k < s
			}
			if (!edge)
				continue;
			const int32_t uk = S.pos[k];
			if (uk < 0)
				continue;
			if (!S.transpose && ((S.ucls[uk] < 0) != (cls < 0)))
				continue;
			if (out_u)
			{
				out_u[cnt] = uk;
				out_r[cnt] = (uint8_t)(idx | (rev ? nbr_rev_flag : 0));
			}
			++cnt;
			if (pass == 0)
				++n_low;
		}
	return cnt;
}

__global__ __launch_bounds__(sblock) void k_nbr_count(sys_t S, int32_t* __restrict__ cnt)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (u >= S.nU)
		return;
	int lo;
	cnt[u] = coupled_list(S, u, nullptr, nullptr, lo);
}

__global__ __launch_bounds__(sblock) void k_nbr_fill(sys_t S, const int32_t* __restrict__ ptr,
													 int32_t* __restrict__ nbr_u, uint8_t* __restrict__ nbr_r,
													 int32_t* __restrict__ mid, int32_t* __restrict__ lvl_key)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (u >= S.nU)
		return;
	int lo;
	const int32_t b = ptr[u];
	coupled_list(S, u, nbr_u + b, nbr_r + b, lo);
	mid[u] = b + lo;
	lvl_key[u] = __popc((uint32_t)S.ulist[u]);
}

struct levels_t
{
	int n; // levels (N + 1)
	int off[34];
};

struct nbr_t
{
	const int32_t* ptr; // nU + 1
	const int32_t* mid; // end of the lower part of each row
	const int32_t* nu;	// neighbour unknowns
	const uint8_t* nr;	// rate index | mirrored flag
	const int32_t* lvl; // unknowns grouped by popcount of their state
	levels_t L;
	// the same lists with rows in level order, packed for the LDS-resident
	// kernels (built only for systems that fit them, else null)
	const uint32_t* hdr; // [nU] first record | lower count << 16 | count << 24 (7 bits)
	const uint32_t* rec; // [nnz] neighbour position | rate code << 16
};

// One damped Jacobi sweep of the anchor choice (the sweeps and the pick are
// described with k_anchor_pick).  The in-neighbours are read from the coupling lists (a terminal unknown's
// list holds exactly its in-neighbours in its own SCC, with their rate codes),
// four at a time, so their loads are in flight together.
__global__ __launch_bounds__(sblock) void k_anchor_sweep(sys_t S, nbr_t G, const double* __restrict__ p_in,
														 double* __restrict__ p_out)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	if (u >= S.nUt)
		return;
	const double* r = S.rates + (int64_t)b * S.rate_stride;
	const int32_t s = S.ulist[u];
	const double* pb = p_in + (int64_t)b * S.nUt;
	double inflow = 0.0;
	int32_t e = G.ptr[u];
	const int32_t e1 = G.ptr[u + 1];
	for (; e + 4 <= e1; e += 4)
	{
		double rv[4], pv[4];
#pragma unroll
		for (int k = 0; k < 4; ++k)
		{
			rv[k] = r[G.nr[e + k] & 63];
			pv[k] = pb[G.nu[e + k]];
		}
#pragma unroll
		for (int k = 0; k < 4; ++k)
			inflow += rv[k] * pv[k];
	}
	for (; e < e1; ++e)
		inflow += r[G.nr[e] & 63] * pb[G.nu[e]];
	const double d = out_rate_s((uint32_t)s, S.mask[s], r);
	p_out[(int64_t)b * S.nUt + u] = 0.5 * pb[u] + 0.5 * inflow / d;
}


// ============================================================================
// One workgroup per rate set: the whole restarted GMRES of that set in one
// launch.  For systems up to a few tens of thousands of unknowns per set this
// keeps every reduction inside the workgroup (no partial sums through HBM, no
// host round trip per iteration); a batch of rate sets is one launch of
// n_sets workgroups.  The iterate x (FP64) is unpreconditioned; right
// preconditioning by Jacobi or by ILU(0).  ILU(0) of these matrices has the
// pattern of M and, ordered by state, dependencies only between states whose
// popcounts differ by one: its triangular solves are level-scheduled over the
// N + 1 popcount levels (one workgroup barrier per level).  The Krylov basis
// lives in global memory (it stays in L2); the Hessenberg matrix and the
// rotations live in LDS.

constexpr int pblock = 256;
constexpr int pwaves = pblock / wave;
constexpr int pm_max = 64;  // restart length cap of the per-set solvers (Hessenberg in LDS)
constexpr int dw_max = 128; // restart length cap of the device-wide solver (Hessenberg in global memory)

struct pgm_out_t
{
	int32_t* iters;	  // [B]
	int32_t* cycles;  // [B]
	double* res;	  // [B] final relative FP64 residual
	int32_t* stalled; // [B] 1 when FP32 cycles stopped reducing the FP64 residual
	uint64_t* tspan;  // [B][2] device wall clock when the set's workgroup started and ended
};

struct pgm_scratch_t
{
	double* r;	   // [B][nU] residual / FP64 correction
	double* udiag; // [B][nU] ILU(0) pivots
	double* t;	   // [B][nU] preconditioned basis vector, FP64 here (the LDS-resident kernels keep it, and
				   // the inverse pivots, in the basis precision)
	void* V;	   // [B][m+1][nU] Krylov basis (FP64 or FP32)
};

// sum over the workgroup of one value per thread, result broadcast
__device__ __forceinline__ double pg_sum(double v, double* lds)
{
	v = wave_sum(v);
	__syncthreads();
	if (lane_id() == 0)
		lds[threadIdx.x / wave] = v;
	__syncthreads();
	double t = 0.0;
	for (int w = 0; w < pwaves; ++w)
		t += lds[w];
	return t;
}

__device__ __forceinline__ bool is_anchor(const sys_t& S, int n_seg, int b, int64_t u)
{
	const int32_t cls = S.ucls[u];
	return cls >= 0 && S.anchor[(int64_t)b * n_seg + cls] == (int32_t)u;
}

// y = M x for one row (FP64): D'_u x_u - sum rate x_k; anchor rows give x_u
template <typename X>
__device__ __forceinline__ double row_apply(const sys_t& S, const nbr_t& G, int n_seg, int b, int64_t u,
											const X* __restrict__ x, const double* __restrict__ r)
{
	if (is_anchor(S, n_seg, b, u))
		return (double)x[u];
	double acc = (double)x[u] / S.invd[(int64_t)b * S.nU + u];
	for (int32_t e = G.ptr[u]; e < G.ptr[u + 1]; ++e)
		acc -= r[G.nr[e] & 63] * (double)x[G.nu[e]];
	return acc;
}

// in place: v <- P^{-1} v with the ILU(0) factors (level-scheduled sweeps)
template <typename X>
__device__ void ilu_apply(const sys_t& S, const nbr_t& G, int n_seg, int b, const double* __restrict__ ud,
						  const double* __restrict__ r, X* __restrict__ v)
{
	for (int l = 0; l < G.L.n; ++l)
	{
		const int a = G.L.off[l], e = G.L.off[l + 1];
		if (a == e)
			continue;
		for (int q = a + threadIdx.x; q < e; q += pblock)
		{
			const int32_t u = G.lvl[q];
			if (is_anchor(S, n_seg, b, u))
				continue; // y_a = v_a
			double y = (double)v[u];
			for (int32_t k = G.ptr[u]; k < G.mid[u]; ++k)
			{
				const int32_t uk = G.nu[k];
				y += r[G.nr[k] & 63] / ud[uk] * (double)v[uk];
			}
			v[u] = (X)y;
		}
		__threadfence_block();
		__syncthreads();
	}
	for (int l = G.L.n - 1; l >= 0; --l)
	{
		const int a = G.L.off[l], e = G.L.off[l + 1];
		if (a == e)
			continue;
		for (int q = a + threadIdx.x; q < e; q += pblock)
		{
			const int32_t u = G.lvl[q];
			if (is_anchor(S, n_seg, b, u))
				continue; // z_a = y_a / 1
			double z = (double)v[u];
			for (int32_t k = G.mid[u]; k < G.ptr[u + 1]; ++k)
				z += r[G.nr[k] & 63] * (double)v[G.nu[k]];
			v[u] = (X)(z / ud[u]);
		}
		__threadfence_block();
		__syncthreads();
	}
}

template <typename T, bool ILU>
__global__ __launch_bounds__(pblock) void k_gmres_set(sys_t S, nbr_t G, int n_seg, const double* __restrict__ rhs,
													  double* __restrict__ zio, pgm_scratch_t sc, int m, double tol,
													  int max_iters, pgm_out_t out, double inner_rtol)
{
	__shared__ double s_H[(pm_max + 1) * pm_max];
	__shared__ double s_cs[pm_max], s_sn[pm_max], s_g[pm_max + 1], s_c[pm_max + 1];
	__shared__ double s_part[(pm_max + 1) * pwaves];
	__shared__ double s_red[pwaves];
	__shared__ double s_scalar[4];
	__shared__ double s_rates[64];

	const int b = blockIdx.x;
	const uint64_t t_begin = wall_clock64();
	const int64_t nU = S.nU;
	const int64_t off = (int64_t)b * nU;
	const double* __restrict__ rb = rhs + off;
	double* __restrict__ x = zio + off; // holds z = D' x on entry and exit, x inside
	double* __restrict__ rr_ = sc.r + off;
	double* __restrict__ ud = sc.udiag + off;
	const double* __restrict__ ib = S.invd + off;
	double* __restrict__ t = sc.t + off; // preconditioned vector, always FP64
	T* __restrict__ V = (T*)sc.V + (int64_t)b * (m + 1) * nU;
	for (int i = threadIdx.x; i < 2 * S.N; i += pblock)
		s_rates[i] = S.rates[(int64_t)b * S.rate_stride + i];
	for (int64_t u = threadIdx.x; u < nU; u += pblock)
		x[u] *= ib[u];
	__syncthreads();

	if (ILU)
	{
		// pivots: u_ss = D'_s - sum over lower k with a mirrored entry of M[s,k] M[k,s] / u_kk
		for (int l = 0; l < G.L.n; ++l)
		{
			const int a = G.L.off[l], e = G.L.off[l + 1];
			if (a == e)
				continue;
			for (int q = a + threadIdx.x; q < e; q += pblock)
			{
				const int32_t u = G.lvl[q];
				double d = 1.0 / ib[u];
				if (!is_anchor(S, n_seg, b, u))
					for (int32_t k = G.ptr[u]; k < G.mid[u]; ++k)
					{
						const int code = G.nr[k];
						const int32_t uk = G.nu[k];
						if ((code & nbr_rev_flag) && !is_anchor(S, n_seg, b, uk))
							d -= s_rates[code & 63] * s_rates[(code & 63) ^ 1] / ud[uk];
					}
				ud[u] = d;
			}
			__threadfence_block();
			__syncthreads();
		}
	}

	int iters = 0, cycles = 0, stalled = 0;
	double rel = 0.0, rel_prev = 0.0;
	for (;;)
	{
		double rr = 0.0, bb = 0.0;
		for (int64_t u = threadIdx.x; u < nU; u += pblock)
		{
			const double res = rb[u] - row_apply<double>(S, G, n_seg, b, u, x, s_rates);
			rr_[u] = res;
			rr += res * res;
			bb += rb[u] * rb[u];
		}
		rr = pg_sum(rr, s_red);
		bb = pg_sum(bb, s_red);
		const double beta = sqrt(rr);
		const double bn = bb > 0.0 ? sqrt(bb) : 1.0;
		rel = beta / bn;
		if (rel <= tol || iters >= max_iters)
			break;
		if (sizeof(T) == 4 && cycles > 0 && !(rel < 0.9 * rel_prev))
		{
			// an FP32 cycle that does not reduce the FP64 residual: undo it if it
			// made things worse and leave the set to the FP64 solver
			if (!(rel <= rel_prev))
			{
				for (int64_t u = threadIdx.x; u < nU; u += pblock)
					x[u] -= t[u];
				rel = rel_prev;
			}
			stalled = 1;
			__threadfence_block();
			__syncthreads();
			break;
		}
		rel_prev = rel;
		// an FP32 cycle stops once its estimate has dropped by inner_rtol (what
		// FP32 arithmetic can deliver); the FP64 residual decides what follows
		const double inner_target = fmax(0.5 * tol, sizeof(T) == 4 ? inner_rtol * rel : 0.0);
		++cycles;
		const double inv_beta = 1.0 / beta;
		for (int64_t u = threadIdx.x; u < nU; u += pblock)
			V[u] = (T)(rr_[u] * inv_beta);
		if (threadIdx.x == 0)
		{
			for (int i = 0; i <= m; ++i)
				s_g[i] = 0.0;
			s_g[0] = beta;
		}
		__threadfence_block();
		__syncthreads();

		int k = 0;
		for (int j = 0; j < m; ++j)
		{
			const T* __restrict__ Vj = V + (int64_t)j * nU;
			T* __restrict__ W = V + (int64_t)(j + 1) * nU;
			// t = P^{-1} V_j
			if (ILU)
			{
				for (int64_t u = threadIdx.x; u < nU; u += pblock)
					t[u] = (double)Vj[u];
				__threadfence_block();
				__syncthreads();
				ilu_apply<double>(S, G, n_seg, b, ud, s_rates, t);
			}
			else
			{
				for (int64_t u = threadIdx.x; u < nU; u += pblock)
					t[u] = (double)Vj[u] * ib[u];
				__threadfence_block();
				__syncthreads();
			}
			for (int64_t u = threadIdx.x; u < nU; u += pblock)
				W[u] = (T)row_apply<double>(S, G, n_seg, b, u, t, s_rates);
			__threadfence_block();
			__syncthreads();
			// classical Gram-Schmidt, twice in FP64 and once in FP32 cycles (as in
			// the LDS-resident kernels); coefficients accumulate in s_H[:, j]
			constexpr int passes = sizeof(T) == 4 ? 1 : 2;
			for (int pass = 0; pass < passes; ++pass)
			{
				for (int i = 0; i <= j; ++i)
				{
					const T* __restrict__ Vi = V + (int64_t)i * nU;
					double d = 0.0;
					for (int64_t u = threadIdx.x; u < nU; u += pblock)
						d += (double)W[u] * (double)Vi[u];
					d = wave_sum(d);
					if (lane_id() == 0)
						s_part[i * pwaves + threadIdx.x / wave] = d;
				}
				__syncthreads();
				if (threadIdx.x <= j)
				{
					double tt = 0.0;
					for (int w = 0; w < pwaves; ++w)
						tt += s_part[threadIdx.x * pwaves + w];
					s_c[threadIdx.x] = tt;
					s_H[j * (pm_max + 1) + threadIdx.x] = (pass == 0 ? 0.0 : s_H[j * (pm_max + 1) + threadIdx.x]) + tt;
				}
				__syncthreads();
				double w2 = 0.0;
				for (int64_t u = threadIdx.x; u < nU; u += pblock)
				{
					double w = (double)W[u];
					for (int i = 0; i <= j; ++i)
						w -= s_c[i] * (double)V[(int64_t)i * nU + u];
					const T wt = (T)w;
					W[u] = wt;
					w2 += (double)wt * (double)wt;
				}
				w2 = pg_sum(w2, s_red);
				if (pass == passes - 1 && threadIdx.x == 0)
					s_scalar[0] = sqrt(w2);
				__threadfence_block();
				__syncthreads();
			}
			if (threadIdx.x == 0)
			{
				double* col = s_H + j * (pm_max + 1);
				const double hn = s_scalar[0];
				col[j + 1] = hn;
				for (int i = 0; i < j; ++i)
				{
					const double a = col[i], c = col[i + 1];
					col[i] = s_cs[i] * a + s_sn[i] * c;
					col[i + 1] = -s_sn[i] * a + s_cs[i] * c;
				}
				const double a = col[j], c = col[j + 1];
				const double rn = hypot(a, c);
				const double cj = rn > 0.0 ? a / rn : 1.0, sj = rn > 0.0 ? c / rn : 0.0;
				s_cs[j] = cj;
				s_sn[j] = sj;
				col[j] = rn;
				col[j + 1] = 0.0;
				s_g[j + 1] = -sj * s_g[j];
				s_g[j] = cj * s_g[j];
				s_scalar[1] = fabs(s_g[j + 1]) / bn;
				s_scalar[2] = (hn > 0.0 && rn > 0.0) ? 1.0 / hn : 0.0;
			}
			__syncthreads();
			const double scale = s_scalar[2];
			for (int64_t u = threadIdx.x; u < nU; u += pblock)
				W[u] = (T)((double)W[u] * scale);
			__threadfence_block();
			__syncthreads();
			++iters;
			k = j + 1;
			if (s_scalar[1] <= inner_target || scale == 0.0 || iters >= max_iters)
				break;
		}
		// y = H^-1 g;  x += P^{-1} (sum_i y_i V_i)   (FP64)
		if (threadIdx.x == 0)
			for (int i = k - 1; i >= 0; --i)
			{
				double tt = s_g[i];
				for (int l = i + 1; l < k; ++l)
					tt -= s_H[l * (pm_max + 1) + i] * s_c[l];
				const double d = s_H[i * (pm_max + 1) + i];
				s_c[i] = d != 0.0 ? tt / d : 0.0;
			}
		__syncthreads();
		// the correction stays in t until the next residual has been checked
		for (int64_t u = threadIdx.x; u < nU; u += pblock)
		{
			double acc = 0.0;
			for (int i = 0; i < k; ++i)
				acc += s_c[i] * (double)V[(int64_t)i * nU + u];
			t[u] = ILU ? acc : acc * ib[u];
		}
		__threadfence_block();
		__syncthreads();
		if (ILU)
			ilu_apply<double>(S, G, n_seg, b, ud, s_rates, t);
		for (int64_t u = threadIdx.x; u < nU; u += pblock)
			x[u] += t[u];
		__threadfence_block();
		__syncthreads();
	}
	for (int64_t u = threadIdx.x; u < nU; u += pblock)
		x[u] /= ib[u];
	if (threadIdx.x == 0)
	{
		out.iters[b] = iters;
		out.cycles[b] = cycles;
		out.res[b] = rel;
		out.stalled[b] = stalled;
		out.tspan[2 * b] = t_begin;
		out.tspan[2 * b + 1] = wall_clock64();
	}
}

#include "reduced.hip.hpp"

// ============================================================================
// LDS-resident variant of k_gmres_set for systems of up to 2048 unknowns per
// set (the common case: one terminal SCC of ~1000 states, many rate sets).
// The ILU(0) sweeps are chains of dependent reads, one chain per popcount
// level; from global memory every level pays several L2 round trips.  Here the
// coupling structure (shared by all sets, 16-bit indices), the inverse pivots
// and the vector being preconditioned live in LDS, so a level costs LDS
// latency plus one workgroup barrier.  Each thread owns the unknowns
// u = threadIdx.x + i * pblock (i < UPT): the Arnoldi vector w and D' of its
// own rows stay in registers, and the basis entries of those rows (a private
// per-thread array, or global memory) are only ever touched by the thread that
// owns the row, so they need no barrier.  Same method and results as
// k_gmres_set (ILU(0) only).

struct lds_plan_t
{
	int off_H, off_g, off_c, off_part, off_t, off_iu, off_hdr, off_rec, bytes;
};

__host__ __device__ inline int lds_take(int& o, int64_t bytes)
{
	const int at = o;
	o += (int)((bytes + 15) / 16 * 16);
	return at;
}

// The rotated Hessenberg matrix is upper triangular: column j (rows 0..j)
// starts at hcol(j) of a packed array.  While column j is formed its
// subdiagonal entry would sit at hcol(j) + j + 1 = hcol(j + 1), the first entry
// of the next column, which is written only after that entry has been rotated
// away.
__host__ __device__ inline int hcol(int j) { return j * (j + 1) / 2; }

// dynamic LDS carve-up for nU unknowns, nnz couplings, restart m, vectors of psize bytes
inline lds_plan_t lds_plan(int64_t nU, int64_t nnz, int m, int psize)
{
	lds_plan_t p{};
	int o = 0;
	p.off_H = lds_take(o, 8 * (int64_t)(hcol(m) + 1));
	p.off_g = lds_take(o, 8 * (int64_t)(m + 1));
	p.off_c = lds_take(o, 8 * (int64_t)(m + 1));
	p.off_part = lds_take(o, 8 * (int64_t)(m + 1) * pwaves);
	p.off_t = lds_take(o, psize * nU);
	p.off_iu = lds_take(o, psize * nU);
	p.off_hdr = lds_take(o, 4 * nU);
	p.off_rec = lds_take(o, 4 * (nnz + 4));
	p.bytes = o;
	return p;
}

constexpr int lds_max_unknowns = 2048;
constexpr int lds_static_bytes = 1024; // upper bound of the kernel's static LDS

// The coupling structure of one set in LDS.  Rows are numbered by their
// position p in the popcount-level order (G.lvl), so a level is a contiguous
// range of rows and a neighbour is reached without an index translation:
//   hdr[p] = first record | lower-neighbour count << 16 | neighbour count << 24
//            | anchor flag << 31
//   rec[k] = neighbour position | (rate index | mirrored flag) << 16
// (lower neighbours first, each part in the order of the coupling lists).
// The anchor flag is set per rate set in LDS, and an anchor's counts are set to
// zero there: its row of M is the identity and its pivot is 1, so the sweeps
// and the row product handle it without a branch.  Four zero records follow
// the last one, so a batch of four records never reads past the array.
constexpr uint32_t hdr_anchor = 1u << 31;
struct lds_view_t
{
	const uint32_t* hdr;
	const uint32_t* rec;
	const double* rates;
	__device__ bool anchor(int p) const { return hdr[p] >> 31; }
};
__device__ __forceinline__ int hdr_first(uint32_t h) { return h & 0xffff; }
__device__ __forceinline__ int hdr_low(uint32_t h) { return (h >> 16) & 0xff; }
__device__ __forceinline__ int hdr_count(uint32_t h) { return (h >> 24) & 0x7f; }

// s + sign * sum over records k0..k1-1 of rate * y[neighbour], added in record
// order.  The records of a row are loaded four at a time (records past k1
// belong to the next rows or to the zero padding, so their positions are in
// range; their terms are dropped by a select): a row of up to four neighbours
// costs two dependent LDS round trips instead of two per neighbour.
template <int SIGN, typename Y>
__device__ __forceinline__ double rec_sum(const lds_view_t& v, int k0, int k1, const Y* __restrict__ y, double s)
{
	for (int k = k0; k < k1; k += 4)
	{
		uint32_t r[4];
#pragma unroll
		for (int i = 0; i < 4; ++i)
			r[i] = v.rec[k + i];
		double rt[4];
		Y yv[4];
#pragma unroll
		for (int i = 0; i < 4; ++i)
		{
			rt[i] = v.rates[(r[i] >> 16) & 63];
			yv[i] = y[r[i] & 0xffff];
		}
		// keep the eight loads together (the scheduler would otherwise
		// interleave them with the products, one round trip per term)
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int i = 0; i < 4; ++i)
		{
			const double term = rt[i] * (double)yv[i];
			s += k + i < k1 ? (SIGN > 0 ? term : -term) : 0.0;
		}
	}
	return s;
}

// The factors of ILU(0) on these matrices.  There is no fill except on the
// diagonal, so P = L1 U1 with L1 = I + L D~^{-1} and U1 = D~ + U, where L and
// U are the strict lower and upper parts of M and D~ the pivots (iu = D~^{-1}).
// In place on LDS, one workgroup barrier per non-empty level:
//   lsolve: y = L1^{-1} t,  y_p = t_p + sum_lower rate * iu_k y_k, stored
//           scaled, t_p <- iu_p y_p, so a neighbour costs one value load.  The
//           lowest non-empty level has no lower neighbours and is skipped: its
//           rows must hold iu_p t_p on entry (rows below lsolve_lowest(...)).
//   usolve: t <- U1^{-1} t,  x_p = iu_p (t_p + sum_upper rate * x_k)
// The bound of the next level is read while the current one is processed.
// first row above the lowest non-empty level
__device__ __forceinline__ int lsolve_lowest(int nl, const int* __restrict__ loff)
{
	for (int l = 0; l < nl; ++l)
		if (loff[l] < loff[l + 1])
			return loff[l + 1];
	return loff[nl];
}

template <typename P>
__device__ void lsolve_lds(int nl, const int* __restrict__ loff, const lds_view_t& v, const P* __restrict__ iu,
						   P* __restrict__ t)
{
	const int tid = threadIdx.x;
	int a = loff[0], e = loff[1];
	bool first = true;
	for (int l = 0; l < nl; ++l)
	{
		const int e2 = loff[l + 2 <= nl ? l + 2 : nl];
		if (a < e)
		{
			if (!first)
			{
				for (int q = a + tid; q < e; q += pblock)
				{
					const uint32_t h = v.hdr[q];
					const double tq = (double)t[q], iq = (double)iu[q];
					const int k0 = hdr_first(h);
					t[q] = (P)(iq * rec_sum<1>(v, k0, k0 + hdr_low(h), t, tq));
				}
				__syncthreads();
			}
			first = false;
		}
		a = e;
		e = e2;
	}
}

template <typename P>
__device__ void usolve_lds(int nl, const int* __restrict__ loff, const lds_view_t& v, const P* __restrict__ iu,
						   P* __restrict__ t)
{
	const int tid = threadIdx.x;
	int a = loff[nl - 1], e = loff[nl];
	for (int l = nl - 1; l >= 0; --l)
	{
		const int a2 = loff[l > 0 ? l - 1 : 0];
		if (a < e)
		{
			for (int q = a + tid; q < e; q += pblock)
			{
				const uint32_t h = v.hdr[q];
				const double tq = (double)t[q], iq = (double)iu[q];
				const int k0 = hdr_first(h);
				t[q] = (P)(iq * rec_sum<1>(v, k0 + hdr_low(h), k0 + hdr_count(h), t, tq));
			}
			__syncthreads();
		}
		e = a;
		a = a2;
	}
}

// row p of M applied to a vector y (rows in level order) held in LDS or global
// memory (FP64 sum)
template <typename Y>
__device__ __forceinline__ double row_lds(const lds_view_t& v, int p, double d, const Y* __restrict__ y)
{
	const uint32_t h = v.hdr[p];
	const int k0 = hdr_first(h);
	return rec_sum<-1>(v, k0, k0 + hdr_count(h), y, d * (double)y[p]);
}

// value of v in lane i of the wavefront (i uniform)
__device__ __forceinline__ double lane_value(double v, int i)
{
	const int lo = __builtin_amdgcn_readlane(__double2loint(v), i);
	const int hi = __builtin_amdgcn_readlane(__double2hiint(v), i);
	return __hiloint2double(hi, lo);
}

constexpr int dot_chunk = 8; // basis vectors per batch of dot products / updates

// Partial dots of w (the thread's own rows) with V_0..V_j, reduced over each
// wavefront: s_part[ii * pwaves + wave] = sum over the wave's rows.  Eight
// basis vectors at a time: their loads are issued together (indices clamped to
// j, so no branches) and the eight values are reduced across the wave by a
// transposed butterfly (halve the values per lane at distances 32, 16, 8, then
// three plain steps): 10 shuffles per eight dots instead of 48.
template <typename T, int UPT>
__device__ __forceinline__ void wave_dots(const T* __restrict__ V, int nU, int j, const double (&w)[UPT],
										  double* __restrict__ s_part)
{
	const int tid = threadIdx.x, lane = tid & (wave - 1), wv = tid / wave;
	for (int c0 = 0; c0 <= j; c0 += dot_chunk)
	{
		double v[dot_chunk];
#pragma unroll
		for (int q = 0; q < dot_chunk; ++q)
		{
			const int ii = c0 + q;
			const T* __restrict__ Vi = V + (int64_t)(ii <= j ? ii : j) * nU;
			double d = 0.0;
#pragma unroll
			for (int i = 0; i < UPT; ++i)
			{
				const int u = tid + i * pblock;
				if (u < nU)
					d += w[i] * (double)Vi[u];
			}
			v[q] = ii <= j ? d : 0.0;
		}
		{
			const bool hi = lane & 32;
#pragma unroll
			for (int k = 0; k < 4; ++k)
			{
				const double send = hi ? v[k] : v[k + 4];
				const double keep = hi ? v[k + 4] : v[k];
				v[k] = keep + __shfl_xor(send, 32, wave);
			}
		}
		{
			const bool hi = lane & 16;
#pragma unroll
			for (int k = 0; k < 2; ++k)
			{
				const double send = hi ? v[k] : v[k + 2];
				const double keep = hi ? v[k + 2] : v[k];
				v[k] = keep + __shfl_xor(send, 16, wave);
			}
		}
		{
			const bool hi = lane & 8;
			const double send = hi ? v[0] : v[1];
			const double keep = hi ? v[1] : v[0];
			v[0] = keep + __shfl_xor(send, 8, wave);
		}
		v[0] += __shfl_xor(v[0], 4, wave);
		v[0] += __shfl_xor(v[0], 2, wave);
		v[0] += __shfl_xor(v[0], 1, wave);
		const int idx = ((lane >> 5) & 1) * 4 + ((lane >> 4) & 1) * 2 + ((lane >> 3) & 1);
		if ((lane & 7) == 0 && c0 + idx <= j)
			s_part[(c0 + idx) * pwaves + wv] = v[0];
	}
}

// w -= sum_ii c[ii] V_ii over ii = 0..j on the own rows (loads batched as above)
template <typename T, int UPT>
__device__ __forceinline__ void wave_update(const T* __restrict__ V, int nU, int j, const double* __restrict__ c,
											double (&w)[UPT])
{
	const int tid = threadIdx.x;
	for (int c0 = 0; c0 <= j; c0 += dot_chunk)
	{
#pragma unroll
		for (int q = 0; q < dot_chunk; ++q)
		{
			const int ii = c0 + q;
			const T* __restrict__ Vi = V + (int64_t)(ii <= j ? ii : j) * nU;
			const double cc = ii <= j ? c[ii] : 0.0;
#pragma unroll
			for (int i = 0; i < UPT; ++i)
			{
				const int u = tid + i * pblock;
				if (u < nU)
					w[i] -= cc * (double)Vi[u];
			}
		}
	}
}

// The same two operations on a Krylov basis held as a per-thread array:
// vb[ii][i] is row tid + i * pblock of basis vector ii (MR + 1 vectors; vectors
// past j are skipped by a uniform branch).
template <int UPT, int MR>
__device__ __forceinline__ void reg_dots(const float (&vb)[MR + 1][UPT], int j, const double (&w)[UPT],
										 double* __restrict__ s_part)
{
	const int tid = threadIdx.x, lane = tid & (wave - 1), wv = tid / wave;
#pragma unroll
	for (int c0 = 0; c0 <= MR; c0 += dot_chunk)
	{
		if (c0 > j)
			break;
		double v[dot_chunk];
#pragma unroll
		for (int q = 0; q < dot_chunk; ++q)
		{
			const int ii = c0 + q <= MR ? c0 + q : MR;
			double d = 0.0;
#pragma unroll
			for (int i = 0; i < UPT; ++i)
				d += w[i] * (double)vb[ii][i];
			v[q] = c0 + q <= j ? d : 0.0;
		}
		{
			const bool hi = lane & 32;
#pragma unroll
			for (int k = 0; k < 4; ++k)
			{
				const double send = hi ? v[k] : v[k + 4];
				const double keep = hi ? v[k + 4] : v[k];
				v[k] = keep + __shfl_xor(send, 32, wave);
			}
		}
		{
			const bool hi = lane & 16;
#pragma unroll
			for (int k = 0; k < 2; ++k)
			{
				const double send = hi ? v[k] : v[k + 2];
				const double keep = hi ? v[k + 2] : v[k];
				v[k] = keep + __shfl_xor(send, 16, wave);
			}
		}
		{
			const bool hi = lane & 8;
			const double send = hi ? v[0] : v[1];
			const double keep = hi ? v[1] : v[0];
			v[0] = keep + __shfl_xor(send, 8, wave);
		}
		v[0] += __shfl_xor(v[0], 4, wave);
		v[0] += __shfl_xor(v[0], 2, wave);
		v[0] += __shfl_xor(v[0], 1, wave);
		const int idx = ((lane >> 5) & 1) * 4 + ((lane >> 4) & 1) * 2 + ((lane >> 3) & 1);
		if ((lane & 7) == 0 && c0 + idx <= j)
			s_part[(c0 + idx) * pwaves + wv] = v[0];
	}
}

template <int UPT, int MR>
__device__ __forceinline__ void reg_update(const float (&vb)[MR + 1][UPT], int j, const double* __restrict__ c,
										   double (&w)[UPT])
{
#pragma unroll
	for (int ii = 0; ii <= MR; ++ii)
	{
		if (ii > j)
			break;
		const double cc = c[ii];
#pragma unroll
		for (int i = 0; i < UPT; ++i)
			w[i] -= cc * (double)vb[ii][i];
	}
}

// MR > 0: the FP32 basis of the thread's rows is a private per-thread array
// (restart length at most MR); MR = 0: the basis lives in global memory.
// Inside the kernel every vector is indexed by level position (thread tid owns
// positions tid + i pblock); the FP64 iterate and the right-hand side are
// gathered into that order at the start (per-set scratch r and udiag) and the
// result is scattered back at the end.
template <typename T, int UPT, int MR>
__device__ __forceinline__ void gmres_lds_body(const sys_t& S, const nbr_t& G, int n_seg, const double* __restrict__ rhs,
											   double* __restrict__ zio, const pgm_scratch_t& sc, int m, double tol,
											   int max_iters, const pgm_out_t& out, const lds_plan_t& lp,
											   double inner_rtol)
{
	using P = T; // precision of the LDS vectors (preconditioned vector, inverse pivots)
	extern __shared__ __align__(16) unsigned char smem[];
	double* s_H = (double*)(smem + lp.off_H);
	double* s_g = (double*)(smem + lp.off_g);
	double* s_c = (double*)(smem + lp.off_c);
	double* s_part = (double*)(smem + lp.off_part);
	P* s_t = (P*)(smem + lp.off_t);
	P* s_iu = (P*)(smem + lp.off_iu);
	uint32_t* s_hdr = (uint32_t*)(smem + lp.off_hdr);
	uint32_t* s_rec = (uint32_t*)(smem + lp.off_rec);
	__shared__ double s_red[pwaves];
	__shared__ double s_nrm[pwaves];
	__shared__ double s_scalar[4];
	__shared__ double s_rates[64];
	__shared__ int s_loff[34];

	const int b = blockIdx.x;
	const uint64_t t_begin = wall_clock64();
	const int tid = threadIdx.x, lane = tid & (wave - 1), wv = tid / wave;
	const int nU = (int)S.nU;
	const int nl = G.L.n;
	const int64_t off = (int64_t)b * nU;
	double* __restrict__ xp = sc.r + off;	   // FP64 iterate x = D'^{-1} z
	double* __restrict__ rbp = sc.udiag + off; // right-hand side
	double* __restrict__ corr = sc.t + off;	   // last correction (undone when an FP32 cycle made things worse)
	T* __restrict__ V = (T*)sc.V + (int64_t)b * (m + 1) * nU;
	static_assert(MR == 0 || sizeof(T) == 4, "the private basis is FP32");
	float vb[MR > 0 ? MR + 1 : 1][UPT];
#pragma unroll
	for (int ii = 0; ii < (MR > 0 ? MR + 1 : 1); ++ii)
#pragma unroll
		for (int i = 0; i < UPT; ++i)
			vb[ii][i] = 0.0f;

	// ---- coupling structure, rates, level bounds into LDS
	const int nnz = G.ptr[nU];
	for (int k = tid; k < nnz + 4; k += pblock)
		s_rec[k] = k < nnz ? G.rec[k] : 0u;
	for (int i = tid; i < 2 * S.N; i += pblock)
		s_rates[i] = S.rates[(int64_t)b * S.rate_stride + i];
	for (int i = tid; i <= nl; i += pblock)
		s_loff[i] = G.L.off[i];
	// ---- own rows: headers with the anchor flag, D', x and b in level order
	double dg[UPT];
	double bb = 0.0;
#pragma unroll
	for (int i = 0; i < UPT; ++i)
	{
		const int p = tid + i * pblock;
		dg[i] = 1.0;
		if (p < nU)
		{
			const int u = G.lvl[p];
			const double ibu = S.invd[off + u];
			const double r = rhs[off + u];
			dg[i] = 1.0 / ibu;
			xp[p] = zio[off + u] * ibu;
			rbp[p] = r;
			bb += r * r;
			s_iu[p] = (P)dg[i]; // D' until the pivots replace it
			const uint32_t h = G.hdr[p];
			s_hdr[p] = is_anchor(S, n_seg, b, u) ? (h & 0xffffu) | hdr_anchor : h;
		}
	}
	__threadfence_block();
	bb = pg_sum(bb, s_red);
	const double bn = bb > 0.0 ? sqrt(bb) : 1.0;
	const lds_view_t lv{ s_hdr, s_rec, s_rates };

	// ---- inverse ILU(0) pivots, level by level
	for (int l = 0; l < nl; ++l)
	{
		const int a = s_loff[l], e = s_loff[l + 1];
		if (a == e)
			continue;
		for (int q = a + tid; q < e; q += pblock)
		{
			double d = (double)s_iu[q];
			const uint32_t h = s_hdr[q];
			if (!(h & hdr_anchor))
			{
				const int k0 = hdr_first(h), k1 = k0 + hdr_low(h);
				for (int k = k0; k < k1; ++k)
				{
					const uint32_t r = s_rec[k];
					const int code = (r >> 16) & 0xff;
					const int pk = r & 0xffff;
					if ((code & nbr_rev_flag) && !lv.anchor(pk))
						d -= s_rates[code & 63] * s_rates[(code & 63) ^ 1] * (double)s_iu[pk];
				}
			}
			s_iu[q] = (P)(1.0 / d);
		}
		__syncthreads();
	}

	const int lowest = lsolve_lowest(nl, s_loff);
	int iters = 0, cycles = 0, stalled = 0;
	double rel = 0.0, rel_prev = 0.0;
	for (;;)
	{
		// FP64 residual of the own rows
		double ro[UPT];
		double rr = 0.0;
#pragma unroll
		for (int i = 0; i < UPT; ++i)
		{
			const int p = tid + i * pblock;
			ro[i] = 0.0;
			if (p < nU)
			{
				ro[i] = rbp[p] - row_lds<double>(lv, p, dg[i], xp);
				rr += ro[i] * ro[i];
			}
		}
		rr = pg_sum(rr, s_red);
		const double beta = sqrt(rr);
		rel = beta / bn;
		if (rel <= tol || iters >= max_iters)
			break;
		if (sizeof(T) == 4 && cycles > 0 && !(rel < 0.9 * rel_prev))
		{
			// an FP32 cycle that does not reduce the FP64 residual: undo it if it
			// made things worse and leave the set to the FP64 solver
			if (!(rel <= rel_prev))
			{
#pragma unroll
				for (int i = 0; i < UPT; ++i)
				{
					const int p = tid + i * pblock;
					if (p < nU)
						xp[p] -= corr[p];
				}
				rel = rel_prev;
			}
			stalled = 1;
			break;
		}
		rel_prev = rel;
		// an FP32 cycle stops once its estimate has dropped by inner_rtol (what
		// FP32 arithmetic can deliver); the FP64 residual decides what follows
		const double inner_target = fmax(0.5 * tol, sizeof(T) == 4 ? inner_rtol * rel : 0.0);
		++cycles;
		// GMRES on the split-preconditioned system L1^{-1} M U1^{-1} (y = U1 x):
		// the cycle starts from the preconditioned residual L1^{-1} r
#pragma unroll
		for (int i = 0; i < UPT; ++i)
		{
			const int p = tid + i * pblock;
			if (p < nU)
				s_t[p] = (P)(p < lowest ? (double)s_iu[p] * ro[i] : ro[i]);
		}
		__syncthreads();
		lsolve_lds<P>(nl, s_loff, lv, s_iu, s_t);
		double rp = 0.0;
#pragma unroll
		for (int i = 0; i < UPT; ++i)
		{
			const int p = tid + i * pblock;
			ro[i] = p < nU ? (double)s_t[p] / (double)s_iu[p] : 0.0;
			rp += ro[i] * ro[i];
		}
		const double beta_p = sqrt(pg_sum(rp, s_red));
		const double inv_beta = 1.0 / beta_p;
		// the Arnoldi estimate |g| / beta_p scales the FP64 relative residual
		const double est_scale = rel / beta_p;
		T vj[UPT];
#pragma unroll
		for (int i = 0; i < UPT; ++i)
		{
			const int p = tid + i * pblock;
			vj[i] = (T)(ro[i] * inv_beta);
			if constexpr (MR > 0)
				vb[0][i] = (float)vj[i];
			else if (p < nU)
				V[p] = vj[i];
		}
		// wavefront 0 applies the Givens rotations: lane i keeps rotation i of
		// this cycle, g_run is the last entry of the rotated right-hand side
		double g_run = beta_p, cs_l = 1.0, sn_l = 0.0;

		int k = 0;
		for (int j = 0; j < m; ++j)
		{
			// w = L1^{-1} M U1^{-1} v_j without a product by M (Eisenstat): with
			// M = L1 D~ + U1 + (D - 2 D~),
			//   x = U1^{-1} v,  w = D~ x + L1^{-1} (v + (D - 2 D~) x)
#pragma unroll
			for (int i = 0; i < UPT; ++i)
			{
				const int p = tid + i * pblock;
				if (p < nU)
					s_t[p] = (P)vj[i];
			}
			__syncthreads();
			usolve_lds<P>(nl, s_loff, lv, s_iu, s_t);
			double w[UPT]; // D~ x until the forward solve is added
#pragma unroll
			for (int i = 0; i < UPT; ++i)
			{
				const int p = tid + i * pblock;
				w[i] = 0.0;
				if (p < nU)
				{
					const double x = (double)s_t[p], iq = (double)s_iu[p], dt = 1.0 / iq;
					w[i] = dt * x;
					const double z = (double)vj[i] + (dg[i] - 2.0 * dt) * x;
					s_t[p] = (P)(p < lowest ? iq * z : z);
				}
			}
			__syncthreads();
			lsolve_lds<P>(nl, s_loff, lv, s_iu, s_t);
#pragma unroll
			for (int i = 0; i < UPT; ++i)
			{
				const int p = tid + i * pblock;
				if (p < nU)
					w[i] += (double)s_t[p] / (double)s_iu[p];
			}
			// classical Gram-Schmidt, twice in FP64 and once in FP32 cycles
			// (an FP32 basis is orthogonal to FP32 accuracy either way, and
			// the FP64 residual that ends each cycle corrects what the cycle
			// leaves: the second pass cost 18 % of the kernel and saved no
			// iterations); lane i <= j of wavefront 0 accumulates H(i, j) in hc
			double hc = 0.0;
			constexpr int passes = sizeof(T) == 4 ? 1 : 2;
			for (int pass = 0; pass < passes; ++pass)
			{
				if constexpr (MR > 0)
					reg_dots<UPT, MR>(vb, j, w, s_part);
				else
					wave_dots<T, UPT>(V, nU, j, w, s_part);
				__syncthreads();
				if (tid <= j)
				{
					double tt = 0.0;
					for (int q = 0; q < pwaves; ++q)
						tt += s_part[tid * pwaves + q];
					s_c[tid] = tt;
					hc += tt;
				}
				__syncthreads();
				if constexpr (MR > 0)
					reg_update<UPT, MR>(vb, j, s_c, w);
				else
					wave_update<T, UPT>(V, nU, j, s_c, w);
			}
			double w2 = 0.0;
#pragma unroll
			for (int i = 0; i < UPT; ++i)
				w2 += w[i] * w[i];
			w2 = wave_sum(w2);
			if (lane == 0)
				s_nrm[wv] = w2;
			__syncthreads();
			if (wv == 0)
			{
				double nn = 0.0;
				for (int q = 0; q < pwaves; ++q)
					nn += s_nrm[q];
				const double hn = sqrt(nn);
				// rotations 0..j-1 applied to column j, the running entry in a register
				double a = lane_value(hc, 0);
				double hv = hc;
				for (int i = 0; i < j; ++i)
				{
					const double c = lane_value(hc, i + 1);
					const double ci = lane_value(cs_l, i), si = lane_value(sn_l, i);
					const double ni = ci * a + si * c;
					if (lane == i)
						hv = ni;
					a = -si * a + ci * c;
				}
				const double rn = hypot(a, hn);
				const double cj = rn > 0.0 ? a / rn : 1.0, sj = rn > 0.0 ? hn / rn : 0.0;
				if (lane == j)
				{
					hv = rn;
					cs_l = cj;
					sn_l = sj;
				}
				if (lane <= j)
					s_H[hcol(j) + lane] = hv;
				if (lane == 0)
				{
					s_g[j] = cj * g_run;
					s_scalar[1] = fabs(sj * g_run) * est_scale;
					s_scalar[2] = (hn > 0.0 && rn > 0.0) ? 1.0 / hn : 0.0;
				}
				g_run = -sj * g_run;
			}
			__syncthreads();
			const double scale = s_scalar[2];
			T* __restrict__ Vn = V + (int64_t)(j + 1) * nU;
#pragma unroll
			for (int i = 0; i < UPT; ++i)
			{
				const int p = tid + i * pblock;
				vj[i] = (T)(w[i] * scale);
				if constexpr (MR == 0)
					if (p < nU)
						Vn[p] = vj[i];
			}
			if constexpr (MR > 0)
			{
#pragma unroll
				for (int ii = 1; ii <= MR; ++ii)
					if (ii == j + 1)
#pragma unroll
						for (int i = 0; i < UPT; ++i)
							vb[ii][i] = (float)vj[i];
			}
			++iters;
			k = j + 1;
			if (s_scalar[1] <= inner_target || scale == 0.0 || iters >= max_iters)
				break;
		}
		// y = R^{-1} g;  x += U1^{-1} (sum_i y_i V_i)
		if (tid == 0)
			for (int i = k - 1; i >= 0; --i)
			{
				double tt = s_g[i];
				for (int l = i + 1; l < k; ++l)
					tt -= s_H[hcol(l) + i] * s_c[l];
				const double d = s_H[hcol(i) + i];
				s_c[i] = d != 0.0 ? tt / d : 0.0;
			}
		__syncthreads();
#pragma unroll
		for (int i = 0; i < UPT; ++i)
		{
			const int p = tid + i * pblock;
			if (p < nU)
			{
				double acc = 0.0;
				if constexpr (MR > 0)
				{
#pragma unroll
					for (int ii = 0; ii <= MR; ++ii)
					{
						if (ii >= k)
							break;
						acc += s_c[ii] * (double)vb[ii][i];
					}
				}
				else
					for (int ii = 0; ii < k; ++ii)
						acc += s_c[ii] * (double)V[(int64_t)ii * nU + p];
				s_t[p] = (P)acc;
			}
		}
		__syncthreads();
		usolve_lds<P>(nl, s_loff, lv, s_iu, s_t);
#pragma unroll
		for (int i = 0; i < UPT; ++i)
		{
			const int p = tid + i * pblock;
			if (p < nU)
			{
				const double cu = (double)s_t[p];
				corr[p] = cu;
				xp[p] += cu;
			}
		}
		__threadfence_block();
		__syncthreads();
	}
	// z = D' x, back in the unknown order of the caller
#pragma unroll
	for (int i = 0; i < UPT; ++i)
	{
		const int p = tid + i * pblock;
		if (p < nU)
		{
			const int u = G.lvl[p];
			zio[off + u] = xp[p] / S.invd[off + u];
		}
	}
	if (tid == 0)
	{
		out.iters[b] = iters;
		out.cycles[b] = cycles;
		out.res[b] = rel;
		out.stalled[b] = stalled;
		out.tspan[2 * b] = t_begin;
		out.tspan[2 * b + 1] = wall_clock64();
	}
}

// The variants differ in where the FP32 Krylov basis of a set lives: in global
// memory (MR = 0), or as a per-thread array of MR + 1 vectors of its own rows
// (MR > 0).  The compiler keeps such an array in lane-private (scratch) memory
// once registers run out; limited to 128 VGPRs (4 waves per SIMD, 4 workgroups
// per CU, the LDS limit as well) this measured fastest on MI355X: 2.56 ms for
// 1024 sets of 1022 unknowns against 2.88 ms with 256 VGPRs (2 workgroups per
// CU) and 3.97 ms with the basis in global memory.
template <typename T, int UPT>
__global__ __launch_bounds__(pblock) void k_gmres_lds(sys_t S, nbr_t G, int n_seg, const double* __restrict__ rhs,
													  double* __restrict__ zio, pgm_scratch_t sc, int m, double tol,
													  int max_iters, pgm_out_t out, lds_plan_t lp, double inner_rtol)
{
	gmres_lds_body<T, UPT, 0>(S, G, n_seg, rhs, zio, sc, m, tol, max_iters, out, lp, inner_rtol);
}

// 8 rows per thread (up to 2048 unknowns): LDS already limits these to 2
// workgroups per CU
template <int MR>
__global__ __launch_bounds__(pblock) __attribute__((amdgpu_waves_per_eu(2))) void k_gmres_priv8(
	sys_t S, nbr_t G, int n_seg, const double* __restrict__ rhs, double* __restrict__ zio, pgm_scratch_t sc, int m,
	double tol, int max_iters, pgm_out_t out, lds_plan_t lp, double inner_rtol)
{
	gmres_lds_body<float, 8, MR>(S, G, n_seg, rhs, zio, sc, m, tol, max_iters, out, lp, inner_rtol);
}

template <int MR>
__global__ __launch_bounds__(pblock) __attribute__((amdgpu_waves_per_eu(4))) void k_gmres_priv(
	sys_t S, nbr_t G, int n_seg, const double* __restrict__ rhs, double* __restrict__ zio, pgm_scratch_t sc, int m,
	double tol, int max_iters, pgm_out_t out, lds_plan_t lp, double inner_rtol)
{
	gmres_lds_body<float, 4, MR>(S, G, n_seg, rhs, zio, sc, m, tol, max_iters, out, lp, inner_rtol);
}

// The same kernel with 170 registers (3 workgroups per CU): the basis of restart
// 24 (100 floats per thread) then stays in registers, and a batch of more sets
// than slots refills the slots that fast sets free.
template <int MR>
__global__ __launch_bounds__(pblock) __attribute__((amdgpu_waves_per_eu(3))) void k_gmres_priv_o3(
	sys_t S, nbr_t G, int n_seg, const double* __restrict__ rhs, double* __restrict__ zio, pgm_scratch_t sc, int m,
	double tol, int max_iters, pgm_out_t out, lds_plan_t lp, double inner_rtol)
{
	gmres_lds_body<float, 4, MR>(S, G, n_seg, rhs, zio, sc, m, tol, max_iters, out, lp, inner_rtol);
}

// Anchor choice from the level-ordered packed records of the LDS-resident
// solver: the damped Jacobi sweeps of k_anchor_sweep (p' = p/2 + inflow/(2D))
// over every unknown of the set in LDS, then per segment the unknown of
// largest mass, ties to the smallest index (k_anchor_pick).  Masses are kept
// in FP32 (they only rank the states), sums in FP64; 1/D of the own rows stays
// in registers and the records of a row are read four at a time.  Rows of
// other segments and ambiguous rows are swept along: their lists hold rows of
// their own part only.  Dynamic LDS: headers, records (+ 4 zero), two FP32
// mass vectors.
template <int UPT>
__global__ __launch_bounds__(pblock) void k_anchor_lvl(sys_t S, nbr_t G, const int32_t* __restrict__ seg_off, int n_seg,
													   int sweeps, int32_t* __restrict__ anchor)
{
	extern __shared__ __align__(16) unsigned char smem[];
	const int nU = (int)S.nU;
	const int nnz = G.ptr[nU];
	uint32_t* s_hdr = (uint32_t*)smem;
	uint32_t* s_rec = s_hdr + nU;
	float* pa = (float*)(s_rec + nnz + 4);
	float* pb = pa + nU;
	__shared__ double s_rates[64];
	__shared__ double s_v[pwaves];
	__shared__ int32_t s_i[pwaves];
	const int b = blockIdx.x, tid = threadIdx.x, lane = tid & (wave - 1), wv = tid / wave;
	for (int k = tid; k < nnz + 4; k += pblock)
		s_rec[k] = k < nnz ? G.rec[k] : 0u;
	for (int i = tid; i < 64; i += pblock)
		s_rates[i] = i < 2 * S.N ? S.rates[(int64_t)b * S.rate_stride + i] : 0.0;
	__syncthreads();
	double invd[UPT];
	int uu[UPT];
#pragma unroll
	for (int i = 0; i < UPT; ++i)
	{
		const int p = tid + i * pblock;
		invd[i] = 0.0;
		uu[i] = -1;
		if (p < nU)
		{
			const int u = G.lvl[p];
			const uint32_t st = (uint32_t)S.ulist[u];
			uu[i] = u;
			s_hdr[p] = G.hdr[p];
			invd[i] = 1.0 / out_rate_s(st, S.mask[st], s_rates);
			pa[p] = 1.0f;
		}
	}
	__syncthreads();
	const lds_view_t lv{ s_hdr, s_rec, s_rates };
	for (int it = 0; it < sweeps; ++it)
	{
		double in[UPT];
#pragma unroll
		for (int i = 0; i < UPT; ++i)
		{
			const int p = tid + i * pblock;
			in[i] = 0.0;
			if (p < nU)
			{
				const uint32_t h = lv.hdr[p];
				in[i] = rec_sum<1>(lv, hdr_first(h), hdr_first(h) + hdr_count(h), pa, 0.0);
			}
		}
#pragma unroll
		for (int i = 0; i < UPT; ++i)
		{
			const int p = tid + i * pblock;
			if (p < nU)
				pb[p] = (float)(0.5 * (double)pa[p] + 0.5 * in[i] * invd[i]);
		}
		__syncthreads();
		float* t = pa;
		pa = pb;
		pb = t;
	}
	for (int k = 0; k < n_seg; ++k)
	{
		const int32_t a = seg_off[k], e = seg_off[k + 1];
		double best = -1.0;
		int32_t bi = a;
#pragma unroll
		for (int i = 0; i < UPT; ++i)
			if (uu[i] >= a && uu[i] < e)
			{
				const double v = (double)pa[tid + i * pblock];
				if (v > best || (v == best && uu[i] < bi))
				{
					best = v;
					bi = uu[i];
				}
			}
		for (int o = wave / 2; o > 0; o >>= 1)
		{
			const double v2 = __shfl_xor(best, o, wave);
			const int32_t i2 = __shfl_xor(bi, o, wave);
			if (v2 > best || (v2 == best && i2 < bi))
			{
				best = v2;
				bi = i2;
			}
		}
		if (lane == 0)
		{
			s_v[wv] = best;
			s_i[wv] = bi;
		}
		__syncthreads();
		if (tid == 0)
		{
			for (int w = 1; w < pwaves; ++w)
				if (s_v[w] > best || (s_v[w] == best && s_i[w] < bi))
				{
					best = s_v[w];
					bi = s_i[w];
				}
			anchor[(int64_t)b * n_seg + k] = bi;
		}
		__syncthreads();
	}
}

// ============================================================================
// element-wise updates of the device-wide solver (any layout)

__global__ __launch_bounds__(sblock) void k_axpy1(int64_t count, const double* __restrict__ a, double* __restrict__ x)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count)
		x[i] += a[i];
}

// x <- x - a (undoes a correction); a is kept for that purpose: b <- a first
__global__ __launch_bounds__(sblock) void k_axpy1_keep(int64_t count, const double* __restrict__ a,
													   double* __restrict__ x, double* __restrict__ keep)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count)
	{
		keep[i] = a[i];
		x[i] += a[i];
	}
}

__global__ __launch_bounds__(sblock) void k_sub1(int64_t count, const double* __restrict__ a, double* __restrict__ x)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count)
		x[i] -= a[i];
}

// z <-> x conversions of the iterate (z = D' x is the convention outside the solvers)
__global__ __launch_bounds__(sblock) void k_scale_invd(int64_t count, const double* __restrict__ invd,
													   double* __restrict__ v, int divide)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count)
		v[i] = divide ? v[i] / invd[i] : v[i] * invd[i];
}

// ============================================================================
// Device-wide GMRES, set-minor layout.  Every vector is [row][set]: the B
// values of one row sit side by side, and rows are numbered in popcount-level
// order (row q = unknown lvl[q]), so a level is one contiguous range of rows.
// A row kernel maps consecutive lanes to the sets of one row (then the next
// row): the row's coupling list is read once per row (the same address for
// all its lanes) and each neighbour's values for all sets are one contiguous
// load -- in the set-major layout the same neighbour read was one isolated
// 8-byte access per set.  Per-set reductions use blocks of R * B threads
// (B <= 1024) with thread t bound to set t % B for the whole grid-stride loop,
// and fixed-order sums: results do not depend on scheduling.

// coupling lists with rows and neighbours in level order
struct wnbr_t
{
	const int32_t* ptr; // [nU + 1]
	const int32_t* mid; // [nU] end of the lower (previous level) part
	const int32_t* nu;	// [nnz] neighbour row (level order)
	const uint8_t* nr;	// [nnz] rate index | mirrored flag
	const int32_t* lvl; // [nU] row -> unknown
	levels_t L;
};

__global__ __launch_bounds__(sblock) void k_w_inv(int64_t nU, const int32_t* __restrict__ lvl, int32_t* __restrict__ inv)
{
	const int64_t q = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (q < nU)
		inv[lvl[q]] = (int32_t)q;
}

__global__ __launch_bounds__(sblock) void k_w_count(int64_t nU, nbr_t G, int32_t* __restrict__ cnt)
{
	const int64_t q = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (q < nU)
	{
		const int32_t u = G.lvl[q];
		cnt[q] = G.ptr[u + 1] - G.ptr[u];
	}
}

__global__ __launch_bounds__(sblock) void k_w_fill(int64_t nU, nbr_t G, const int32_t* __restrict__ inv,
												   const int32_t* __restrict__ wptr, int32_t* __restrict__ wmid,
												   int32_t* __restrict__ wnu, uint8_t* __restrict__ wnr)
{
	const int64_t q = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (q >= nU)
		return;
	const int32_t u = G.lvl[q];
	const int32_t a = G.ptr[u], at = wptr[q];
	wmid[q] = at + (G.mid[u] - a);
	for (int32_t e = a; e < G.ptr[u + 1]; ++e)
	{
		wnu[at + (e - a)] = inv[G.nu[e]];
		wnr[at + (e - a)] = G.nr[e];
	}
}

// set-major plan vectors -> set-minor solver vectors: right-hand side, iterate
// x = invd * z, 1/D' and the anchor flag of every (row, set)
__global__ __launch_bounds__(sblock) void k_w_gather(sys_t S, int n_seg, const int32_t* __restrict__ lvl,
													 const double* __restrict__ rhs, const double* __restrict__ z,
													 double* __restrict__ wrhs, double* __restrict__ wx,
													 double* __restrict__ winvd, uint8_t* __restrict__ wanc)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int B = S.B;
	if (i >= S.nU * B)
		return;
	const int64_t q = i / B;
	const int b = (int)(i - q * B);
	const int32_t u = lvl[q];
	const int64_t o = (int64_t)b * S.nU + u;
	const double iv = S.invd[o];
	wrhs[i] = rhs[o];
	wx[i] = z[o] * iv;
	winvd[i] = iv;
	wanc[i] = is_anchor(S, n_seg, b, u) ? 1 : 0;
}

// z = x / invd back into the plan's set-major layout
__global__ __launch_bounds__(sblock) void k_w_scatter(int64_t nU, int B, const int32_t* __restrict__ lvl,
													  const double* __restrict__ wx, const double* __restrict__ winvd,
													  double* __restrict__ z)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= nU * B)
		return;
	const int64_t q = i / B;
	const int b = (int)(i - q * B);
	z[(int64_t)b * nU + lvl[q]] = wx[i] / winvd[i];
}

// rows [q0, q1) x B sets as a flat range: the row and set of flat index i
__device__ __forceinline__ void w_row_set(int64_t i, int B, int64_t q0, int64_t& q, int& b)
{
	const int64_t rr = i / B;
	b = (int)(i - rr * B);
	q = q0 + rr;
}

// rates transposed for the set-minor kernels: rt[code * B + b] = rate `code`
// of set b, so the lanes of a row (consecutive sets) read consecutive words
__global__ __launch_bounds__(sblock) void k_w_rates(const double* __restrict__ rates, int64_t rstride, int ncode,
													int B, double* __restrict__ rt)
{
	const int i = blockIdx.x * sblock + threadIdx.x;
	if (i >= ncode * B)
		return;
	const int code = i / B, b = i - code * B;
	rt[i] = rates[(int64_t)b * rstride + code];
}

// y = M x for (row q, set b): D'_u x - sum rate x_k; anchor rows give x
template <typename X>
__device__ __forceinline__ double w_row_apply(const wnbr_t& G, int B, int64_t q, int b, const double* __restrict__ rt,
											  const double* __restrict__ winvd, const uint8_t* __restrict__ wanc,
											  const X* __restrict__ x)
{
	const int64_t i = q * B + b;
	if (wanc[i])
		return (double)x[i];
	double acc = (double)x[i] / winvd[i];
	int32_t e = G.ptr[q];
	const int32_t e1 = G.ptr[q + 1];
	// four neighbours' loads in flight at a time; the sum keeps its order
	for (; e + 4 <= e1; e += 4)
	{
		double xv[4], rv[4];
#pragma unroll
		for (int k = 0; k < 4; ++k)
		{
			xv[k] = (double)x[(int64_t)G.nu[e + k] * B + b];
			rv[k] = rt[(G.nr[e + k] & 63) * B + b];
		}
#pragma unroll
		for (int k = 0; k < 4; ++k)
			acc -= rv[k] * xv[k];
	}
	for (; e < e1; ++e)
		acc -= rt[(G.nr[e] & 63) * B + b] * (double)x[(int64_t)G.nu[e] * B + b];
	return acc;
}

template <typename X, typename Y>
__global__ __launch_bounds__(sblock) void k_w_apply(wnbr_t G, int64_t nU, int B, const double* __restrict__ rt,
													const double* __restrict__ winvd,
													const uint8_t* __restrict__ wanc, const Y* __restrict__ t,
													X* __restrict__ W, const int32_t* __restrict__ live)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= nU * B)
		return;
	int64_t q;
	int b;
	w_row_set(i, B, 0, q, b);
	if (!live[b])
		return;
	W[i] = (X)w_row_apply<Y>(G, B, q, b, rt, winvd, wanc, t);
}

__global__ __launch_bounds__(sblock) void k_w_residual(wnbr_t G, int64_t nU, int B, const double* __restrict__ rt,
													   const double* __restrict__ winvd,
													   const uint8_t* __restrict__ wanc,
													   const double* __restrict__ rhs, const double* __restrict__ x,
													   double* __restrict__ r)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= nU * B)
		return;
	int64_t q;
	int b;
	w_row_set(i, B, 0, q, b);
	r[i] = rhs[i] - w_row_apply<double>(G, B, q, b, rt, winvd, wanc, x);
}

template <typename X>
__global__ __launch_bounds__(sblock) void k_w_jacobi(int64_t count, int B, const double* __restrict__ winvd,
													 X* __restrict__ v, const int32_t* __restrict__ live)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= count || !live[i % B])
		return;
	v[i] = (X)((double)v[i] * winvd[i]);
}

// inverse ILU(0) pivots of the rows of one level (the previous level's are final)
__global__ __launch_bounds__(sblock) void k_w_ilu_pivot(wnbr_t G, int B, int l, const double* __restrict__ rt,
														const double* __restrict__ winvd,
														const uint8_t* __restrict__ wanc, double* __restrict__ ud)
{
	const int64_t q0 = G.L.off[l];
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= (G.L.off[l + 1] - q0) * B)
		return;
	int64_t q;
	int b;
	w_row_set(i, B, q0, q, b);
	const int64_t at = q * B + b;
	double d = 1.0 / winvd[at];
	if (!wanc[at])
		for (int32_t e = G.ptr[q]; e < G.mid[q]; ++e)
		{
			const int code = G.nr[e];
			const int64_t k = (int64_t)G.nu[e] * B + b;
			if ((code & nbr_rev_flag) && !wanc[k])
				d -= rt[(code & 63) * B + b] * rt[((code & 63) ^ 1) * B + b] * ud[k];
		}
	ud[at] = 1.0 / d; // the sweeps multiply by inverse pivots (no division per neighbour)
}

template <typename X>
__global__ __launch_bounds__(sblock) void k_w_ilu_fwd(wnbr_t G, int B, int l, const double* __restrict__ rt,
													  const uint8_t* __restrict__ wanc,
													  const double* __restrict__ ud, const X* src, X* v,
													  const int32_t* __restrict__ live)
{
	// v's rows of level l from src's (src may be v): the forward sweep reads every
	// row once, so it also moves the vector into the sweep's output
	const int64_t q0 = G.L.off[l];
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= (G.L.off[l + 1] - q0) * B)
		return;
	int64_t q;
	int b;
	w_row_set(i, B, q0, q, b);
	const int64_t at = q * B + b;
	if (!live[b])
		return;
	if (wanc[at])
	{
		v[at] = src[at];
		return;
	}
	double y = (double)src[at];
	int32_t e = G.ptr[q];
	const int32_t e1 = G.mid[q];
	for (; e + 4 <= e1; e += 4) // four neighbours' loads in flight; the sum keeps its order
	{
		double rv[4], uv[4], vv[4];
#pragma unroll
		for (int k = 0; k < 4; ++k)
		{
			const int64_t at_k = (int64_t)G.nu[e + k] * B + b;
			rv[k] = rt[(G.nr[e + k] & 63) * B + b];
			uv[k] = ud[at_k];
			vv[k] = (double)v[at_k];
		}
#pragma unroll
		for (int k = 0; k < 4; ++k)
			y += rv[k] * uv[k] * vv[k];
	}
	for (; e < e1; ++e)
	{
		const int64_t k = (int64_t)G.nu[e] * B + b;
		y += rt[(G.nr[e] & 63) * B + b] * ud[k] * (double)v[k];
	}
	v[at] = (X)y;
}

template <typename X>
__global__ __launch_bounds__(sblock) void k_w_ilu_bwd(wnbr_t G, int B, int l, const double* __restrict__ rt,
													  const uint8_t* __restrict__ wanc,
													  const double* __restrict__ ud, X* __restrict__ v,
													  const int32_t* __restrict__ live)
{
	const int64_t q0 = G.L.off[l];
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= (G.L.off[l + 1] - q0) * B)
		return;
	int64_t q;
	int b;
	w_row_set(i, B, q0, q, b);
	const int64_t at = q * B + b;
	if (!live[b] || wanc[at])
		return;
	double z = (double)v[at];
	int32_t e = G.mid[q];
	const int32_t e1 = G.ptr[q + 1];
	for (; e + 4 <= e1; e += 4) // four neighbours' loads in flight; the sum keeps its order
	{
		double rv[4], vv[4];
#pragma unroll
		for (int k = 0; k < 4; ++k)
		{
			rv[k] = rt[(G.nr[e + k] & 63) * B + b];
			vv[k] = (double)v[(int64_t)G.nu[e + k] * B + b];
		}
#pragma unroll
		for (int k = 0; k < 4; ++k)
			z += rv[k] * vv[k];
	}
	for (; e < e1; ++e)
		z += rt[(G.nr[e] & 63) * B + b] * (double)v[(int64_t)G.nu[e] * B + b];
	v[at] = (X)(z * ud[at]);
}

// per-set sums over rows: a block of R * B threads, thread t works for set
// t % B on rows blockIdx.x * R + t / B + k * gridDim.x * R; the R partials of a
// set are added in row order into part[blk][b][i]
__device__ __forceinline__ void w_block_sets(double v, int B, int R, double* s_red, double* __restrict__ part,
											 int64_t slot)
{
	// the R values of set b (threads b, b + B, ...) folded in halves: a fixed
	// order, log2(R) barriers instead of R serial additions by one thread
	s_red[threadIdx.x] = v;
	__syncthreads();
	const int i = (int)threadIdx.x / B;
	for (int r = R; r > 1;)
	{
		const int h = (r + 1) / 2;
		if (i < r - h)
			s_red[threadIdx.x] += s_red[threadIdx.x + h * B];
		__syncthreads();
		r = h;
	}
	if ((int)threadIdx.x < B)
		part[slot] = s_red[threadIdx.x];
	__syncthreads();
}

// partial sums of r^2 and rhs^2 per set: part[blk][b][2]
__global__ __launch_bounds__(1024) void k_w_norms(int64_t nU, int B, int R, const double* __restrict__ r,
												  const double* __restrict__ rhs, double* __restrict__ part)
{
	__shared__ double s_red[1024];
	const int b = threadIdx.x % B;
	double rr = 0.0, bb = 0.0;
	if ((int)threadIdx.x < B * R)
		for (int64_t q = (int64_t)blockIdx.x * R + threadIdx.x / B; q < nU; q += (int64_t)gridDim.x * R)
		{
			const double v = r[q * B + b], w = rhs[q * B + b];
			rr += v * v;
			bb += w * w;
		}
	const int64_t base = ((int64_t)blockIdx.x * B + b) * 2;
	w_block_sets(rr, B, R, s_red, part, base + 0);
	w_block_sets(bb, B, R, s_red, part, base + 1);
}

// partial dots: part[blk][b][i] = sum_rows W * V_i, i < K; eight basis
// vectors per pass over the rows, so W is read once per eight
template <typename T>
__global__ __launch_bounds__(1024) void k_w_dots(int64_t nU, int B, int R, int K, const T* __restrict__ W,
												 const T* __restrict__ V, int64_t vstride, double* __restrict__ part,
												 const int32_t* __restrict__ live)
{
	constexpr int C = 8;
	__shared__ double s_red[1024];
	const int b = threadIdx.x % B;
	const bool on = (int)threadIdx.x < B * R && live[b];
	for (int i0 = 0; i0 < K; i0 += C)
	{
		double d[C];
#pragma unroll
		for (int c = 0; c < C; ++c)
			d[c] = 0.0;
		if (on)
		{
			// two rows per step: both rows' loads are in flight together
			const int64_t step = (int64_t)gridDim.x * R;
			int64_t q = (int64_t)blockIdx.x * R + threadIdx.x / B;
			for (; q + step < nU; q += 2 * step)
			{
				const int64_t a0 = q * B + b, a1 = (q + step) * B + b;
				const double w0 = (double)W[a0], w1 = (double)W[a1];
#pragma unroll
				for (int c = 0; c < C; ++c)
					if (i0 + c < K)
					{
						const T* Vc = V + (int64_t)(i0 + c) * vstride;
						d[c] += w0 * (double)Vc[a0] + w1 * (double)Vc[a1];
					}
			}
			if (q < nU)
			{
				const int64_t a0 = q * B + b;
				const double w0 = (double)W[a0];
#pragma unroll
				for (int c = 0; c < C; ++c)
					if (i0 + c < K)
						d[c] += w0 * (double)V[(int64_t)(i0 + c) * vstride + a0];
			}
		}
#pragma unroll
		for (int c = 0; c < C; ++c)
			if (i0 + c < K)
				w_block_sets(d[c], B, R, s_red, part, ((int64_t)blockIdx.x * B + b) * K + i0 + c);
	}
}

// W -= sum_i c[b][i] V_i; partial sums of |W|^2 per set: part[blk][b]
template <typename T>
__global__ __launch_bounds__(1024) void k_w_orth(int64_t nU, int B, int R, int K, T* __restrict__ W,
												 const T* __restrict__ V, int64_t vstride,
												 const double* __restrict__ ct, double* __restrict__ part,
												 const int32_t* __restrict__ live)
{
	__shared__ double s_red[1024];
	const int b = threadIdx.x % B;
	double w2 = 0.0;
	if ((int)threadIdx.x < B * R && live[b])
	{
		// two rows per step: both rows' loads are in flight together
		const int64_t step = (int64_t)gridDim.x * R;
		int64_t q = (int64_t)blockIdx.x * R + threadIdx.x / B;
		for (; q + step < nU; q += 2 * step)
		{
			const int64_t a0 = q * B + b, a1 = (q + step) * B + b;
			double w0 = (double)W[a0], w1 = (double)W[a1];
			for (int i = 0; i < K; ++i)
			{
				const double ci = ct[i * B + b];
				const T* Vi = V + i * vstride;
				w0 -= ci * (double)Vi[a0];
				w1 -= ci * (double)Vi[a1];
			}
			const T t0 = (T)w0, t1 = (T)w1;
			W[a0] = t0;
			W[a1] = t1;
			w2 += (double)t0 * (double)t0 + (double)t1 * (double)t1;
		}
		if (q < nU)
		{
			const int64_t at = q * B + b;
			double w = (double)W[at];
			for (int i = 0; i < K; ++i)
				w -= ct[i * B + b] * (double)V[i * vstride + at];
			const T wt = (T)w;
			W[at] = wt;
			w2 += (double)wt * (double)wt;
		}
	}
	w_block_sets(w2, B, R, s_red, part, (int64_t)blockIdx.x * B + b);
}

// out[b * ostride + i] = sum over blocks of part[blk][b][i]  (one wave per
// (i, b)); outt (if not null) gets the same values transposed, outt[i * B + b]
// out[b][i] = sum over the blocks k of part[k][b][i] (i < K), one workgroup per
// set: thread t adds block rows t / K, t / K + G, ... (G = 256 / K groups) of
// column i = t % K, so each group reads the K contiguous values of a block
// row; the groups' sums are then added in group order (a fixed order)
constexpr int wred_threads = 256;

__global__ __launch_bounds__(wred_threads) void k_w_reduce(const double* __restrict__ part, int nblk, int B, int K,
														   double* __restrict__ out, int64_t ostride,
														   double* __restrict__ outt)
{
	__shared__ double s_sum[wred_threads];
	const int b = blockIdx.x;
	const int G = wred_threads / K; // K <= wred_threads
	const int i = threadIdx.x % K, gi = threadIdx.x / K;
	double s = 0.0;
	if (gi < G)
		for (int k = gi; k < nblk; k += G)
			s += part[((int64_t)k * B + b) * K + i];
	s_sum[threadIdx.x] = s;
	__syncthreads();
	if ((int)threadIdx.x < K)
	{
		double t = 0.0;
		for (int q = 0; q < G; ++q)
			t += s_sum[q * K + threadIdx.x];
		out[(int64_t)b * ostride + threadIdx.x] = t;
		if (outt)
			outt[(int64_t)threadIdx.x * B + b] = t;
	}
}

// yt[j * B + b] = y[b][j], j <= m (the combination weights, transposed)
__global__ __launch_bounds__(sblock) void k_w_transpose_y(int B, int m, const double* __restrict__ y,
														  double* __restrict__ yt)
{
	const int i = blockIdx.x * sblock + threadIdx.x;
	if (i >= B * (m + 1))
		return;
	const int j = i / B, b = i - j * B;
	yt[i] = y[(int64_t)b * (m + 1) + j];
}

template <typename T>
__global__ __launch_bounds__(sblock) void k_w_cast_scale(int64_t count, int B, const double* __restrict__ r,
														 const double* __restrict__ scale, T* __restrict__ out)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= count)
		return;
	const double s = scale[i % B];
	out[i] = (T)(s > 0.0 ? r[i] / s : 0.0);
}

template <typename T, typename O>
__global__ __launch_bounds__(sblock) void k_w_copy_live(int64_t count, int B, const T* __restrict__ a,
														O* __restrict__ out, const int32_t* __restrict__ live)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count && live[i % B])
		out[i] = (O)a[i];
}

template <typename T>
__global__ __launch_bounds__(sblock) void k_w_scale(int64_t count, int B, const T* __restrict__ W,
													const double* __restrict__ hnorm, T* __restrict__ Vn,
													const int32_t* __restrict__ live)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= count)
		return;
	const int b = (int)(i % B);
	if (!live[b])
		return;
	const double h = hnorm[b];
	Vn[i] = (T)((double)W[i] * (h > 0.0 ? 1.0 / h : 0.0));
}

// z += sum_{i < k_b} y[b][i] V_i  (yt = y transposed: yt[i * B + b])
template <typename T>
__global__ __launch_bounds__(sblock) void k_w_combine(int64_t count, int B, int k, const T* __restrict__ V,
													  int64_t vstride, const double* __restrict__ yt,
													  double* __restrict__ z, const int32_t* __restrict__ kb)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i >= count)
		return;
	const int b = (int)(i % B);
	const int kk = min(k, kb[b]);
	if (kk == 0)
		return;
	double acc = z[i];
	for (int j = 0; j < kk; ++j)
		acc += yt[j * B + b] * (double)V[j * vstride + i];
	z[i] = acc;
}

// ============================================================================
// full mode: terminal kernels of every terminal SCC and the absorption
// probabilities X[j, c] of every transient state (solution_term /
// solution_nonterm of solver.cu:102-300)

__global__ __launch_bounds__(sblock) void k_fill_u8(int64_t n, uint8_t v, uint8_t* __restrict__ p)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < n)
		p[i] = v;
}

// rhs[j][u] = sum over edges c -> d leaving the ambiguous set of rate(c -> d)
// when d is bound for terminal SCC j (transposed system, absorption probabilities)
__global__ __launch_bounds__(sblock) void k_rhs_absorb(sys_t S, const int32_t* __restrict__ rank, int64_t T,
													   const uint64_t* __restrict__ tm, double* __restrict__ rhs)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int j = blockIdx.y;
	if (u >= S.nU)
		return;
	const double* r = S.rates;
	const uint32_t c = (uint32_t)S.ulist[u];
	uint32_t m = S.mask[c];
	double acc = 0.0;
	while (m)
	{
		const int i = __ffs(m) - 1;
		m &= m - 1;
		const uint32_t d = c ^ (1u << i);
		if (S.pos[d] >= 0)
			continue;
		const int32_t k = rank[d];
		const int t = k < T ? k : (__ffsll((unsigned long long)tm[d]) - 1);
		if (t == j)
			acc += rate_of(r, i, ((c >> i) & 1u) == 0);
	}
	rhs[(int64_t)j * S.nU + u] = acc;
}

__global__ __launch_bounds__(sblock) void k_times_invd(int64_t count, const double* __restrict__ z,
													   const double* __restrict__ invd, double* __restrict__ out)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count)
		out[i] = z[i] * invd[i];
}


// warm start: p[b][u] = predicted mass of the terminal-system unknown u
// (warm holds [set][n_t] values over the terminal states in canonical order)
__global__ __launch_bounds__(sblock) void k_warm_gather(int64_t nUt, int64_t n_t, const int32_t* __restrict__ tpos,
														const double* __restrict__ warm, double* __restrict__ p)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	if (u >= nUt)
		return;
	const double v = warm[(int64_t)b * n_t + tpos[u]];
	p[(int64_t)b * nUt + u] = v > 0.0 ? v : 0.0;
}

// initial iterate z = D' x with x_u = p_u / p_anchor on the terminal systems
__global__ __launch_bounds__(sblock) void k_warm_z(sys_t S, int n_seg, const double* __restrict__ p,
												   double* __restrict__ z)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	if (u >= S.nUt)
		return;
	const int32_t k = S.ucls[u];
	const int32_t a = S.anchor[(int64_t)b * n_seg + k];
	const double pa = p[(int64_t)b * S.nUt + a];
	const double x = pa > 0.0 ? p[(int64_t)b * S.nUt + u] / pa : (u == a ? 1.0 : 0.0);
	z[(int64_t)b * S.nU + u] = x / S.invd[(int64_t)b * S.nU + u];
}

// ============================================================================
// Exact fallback: FP64 dense LU with partial pivoting of one diagonal block of
// one set's system (the systems are block diagonal: one block per terminal
// segment, one for the ambiguous states), for sets whose Krylov solve missed
// the tolerance.  Column-major s x s matrix, right-looking and blocked by
// lu_nb columns: panel factorisation (one workgroup), row interchanges of the
// other columns, triangular solve of the block row, and the trailing update
// A22 -= L21 U12 in 64 x 64 tiles staged through LDS.  Replaces the
// reference's dense getrf path (linear_system_solve.cu:69-88, 249-325;
// sparse_utils.cu:268-291), which factors without pivoting.

constexpr int lu_nb = 32;
constexpr int lu_panel_threads = 1024;
constexpr int64_t lu_max_block = 16384; // 2 GiB of FP64 matrix

// A = M restricted to block [u0, u0 + s) of set b (x variables: diagonal D'_u,
// off-diagonal -rate; anchor rows e_u); x = the block of the right-hand side
__global__ __launch_bounds__(sblock) void k_lu_assemble(sys_t S, nbr_t G, int n_seg, int b, int64_t u0, int s,
														double* __restrict__ A, const double* __restrict__ rhs,
														double* __restrict__ x, int32_t* __restrict__ flag)
{
	const int i = blockIdx.x * sblock + threadIdx.x;
	if (i >= s)
		return;
	const int64_t u = u0 + i;
	const int64_t off = (int64_t)b * S.nU;
	x[i] = rhs[off + u];
	if (is_anchor(S, n_seg, b, u))
	{
		A[(int64_t)i * s + i] = 1.0;
		return;
	}
	const double* __restrict__ r = S.rates + (int64_t)b * S.rate_stride;
	A[(int64_t)i * s + i] = 1.0 / S.invd[off + u];
	for (int32_t e = G.ptr[u]; e < G.ptr[u + 1]; ++e)
	{
		const int64_t k = (int64_t)G.nu[e] - u0;
		if (k < 0 || k >= s)
		{
			atomicOr(flag, 2); // a coupling leaves the block: the block split is wrong
			continue;
		}
		A[k * s + i] -= r[G.nr[e] & 63];
	}
}

// factorises columns [j0, j0 + jb) of rows [j0, s): pivot search, row swap
// inside the panel, scaling and the rank-1 updates of the panel's own columns
__global__ __launch_bounds__(lu_panel_threads) void k_lu_panel(double* __restrict__ A, int s, int j0, int jb,
															   int32_t* __restrict__ ipiv, int32_t* __restrict__ flag)
{
	__shared__ double s_val[lu_panel_threads / wave];
	__shared__ int s_idx[lu_panel_threads / wave];
	__shared__ double s_prow[lu_nb];
	__shared__ int s_piv;
	const int64_t lda = s;
	const int nw = lu_panel_threads / wave;
	for (int jj = 0; jj < jb; ++jj)
	{
		const int j = j0 + jj;
		double* __restrict__ colj = A + (int64_t)j * lda;
		double best = -1.0;
		int bi = j;
		for (int i = j + threadIdx.x; i < s; i += lu_panel_threads)
		{
			const double v = fabs(colj[i]);
			if (v > best)
			{
				best = v;
				bi = i;
			}
		}
		for (int d = wave / 2; d > 0; d >>= 1)
		{
			const double ov = __shfl_xor(best, d);
			const int oi = __shfl_xor(bi, d);
			if (ov > best || (ov == best && oi < bi))
			{
				best = ov;
				bi = oi;
			}
		}
		if (lane_id() == 0)
		{
			s_val[threadIdx.x / wave] = best;
			s_idx[threadIdx.x / wave] = bi;
		}
		__syncthreads();
		if (threadIdx.x == 0)
		{
			double bv = s_val[0];
			int bx = s_idx[0];
			for (int w = 1; w < nw; ++w)
				if (s_val[w] > bv || (s_val[w] == bv && s_idx[w] < bx))
				{
					bv = s_val[w];
					bx = s_idx[w];
				}
			if (!(bv > 0.0))
				atomicOr(flag, 1); // singular (or not finite)
			s_piv = bx;
			ipiv[j] = bx;
		}
		__syncthreads();
		const int p = s_piv;
		if (p != j)
			for (int k = threadIdx.x; k < jb; k += lu_panel_threads)
			{
				double* c = A + (int64_t)(j0 + k) * lda;
				const double t = c[j];
				c[j] = c[p];
				c[p] = t;
			}
		__syncthreads();
		if (threadIdx.x < jb)
			s_prow[threadIdx.x] = A[(int64_t)(j0 + threadIdx.x) * lda + j];
		__syncthreads();
		const double d = s_prow[jj];
		const double inv = d != 0.0 ? 1.0 / d : 0.0;
		for (int i = j + 1 + threadIdx.x; i < s; i += lu_panel_threads)
		{
			const double l = colj[i] * inv;
			colj[i] = l;
			for (int kk = jj + 1; kk < jb; ++kk)
				A[(int64_t)(j0 + kk) * lda + i] -= l * s_prow[kk];
		}
		__syncthreads();
	}
}

// the panel's row interchanges applied to every column outside the panel
__global__ __launch_bounds__(sblock) void k_lu_swap(double* __restrict__ A, int s, int j0, int jb,
													const int32_t* __restrict__ ipiv)
{
	const int c = blockIdx.x * sblock + threadIdx.x;
	if (c >= s || (c >= j0 && c < j0 + jb))
		return;
	double* __restrict__ col = A + (int64_t)c * s;
	for (int jj = 0; jj < jb; ++jj)
	{
		const int j = j0 + jj, p = ipiv[j];
		if (p != j)
		{
			const double t = col[j];
			col[j] = col[p];
			col[p] = t;
		}
	}
}

// U12 = L11^{-1} A12: one thread per column right of the panel, the unit
// lower triangle L11 in LDS
__global__ __launch_bounds__(sblock) void k_lu_trsm(double* __restrict__ A, int s, int j0, int jb)
{
	__shared__ double sL[lu_nb][lu_nb + 1];
	for (int q = threadIdx.x; q < lu_nb * lu_nb; q += sblock)
	{
		const int i = q % lu_nb, k = q / lu_nb;
		sL[i][k] = (i < jb && k < jb) ? A[(int64_t)(j0 + k) * s + j0 + i] : 0.0;
	}
	__syncthreads();
	const int c = j0 + jb + blockIdx.x * sblock + threadIdx.x;
	if (c >= s)
		return;
	double* __restrict__ col = A + (int64_t)c * s + j0;
	double x[lu_nb];
#pragma unroll
	for (int i = 0; i < lu_nb; ++i)
	{
		double v = i < jb ? col[i] : 0.0;
#pragma unroll
		for (int k = 0; k < i; ++k)
			v -= sL[i][k] * x[k];
		x[i] = v;
		if (i < jb)
			col[i] = v;
	}
}

// A22 -= L21 U12 on the trailing (s - j0 - jb)^2 block, one 64 x 64 tile per
// workgroup, 4 x 4 results per thread
__global__ __launch_bounds__(sblock) void k_lu_gemm(double* __restrict__ A, int s, int j0, int jb)
{
	__shared__ double sL[lu_nb][64 + 1];
	__shared__ double sU[lu_nb][64 + 1];
	const int base = j0 + jb;
	const int r0 = base + blockIdx.x * 64, c0 = base + blockIdx.y * 64;
	for (int q = threadIdx.x; q < lu_nb * 64; q += sblock)
	{
		const int r = q % 64, k = q / 64; // rows contiguous in a column of L21
		sL[k][r] = (k < jb && r0 + r < s) ? A[(int64_t)(j0 + k) * s + r0 + r] : 0.0;
		const int kk = q % lu_nb, cc = q / lu_nb; // U12 column cc, rows contiguous
		sU[kk][cc] = (kk < jb && c0 + cc < s) ? A[(int64_t)(c0 + cc) * s + j0 + kk] : 0.0;
	}
	__syncthreads();
	const int tr = threadIdx.x % 16, tc = threadIdx.x / 16;
	double acc[4][4] = {};
	for (int k = 0; k < jb; ++k)
	{
		double a[4], bb[4];
#pragma unroll
		for (int i = 0; i < 4; ++i)
		{
			a[i] = sL[k][tr + 16 * i];
			bb[i] = sU[k][tc + 16 * i];
		}
#pragma unroll
		for (int i = 0; i < 4; ++i)
#pragma unroll
			for (int j = 0; j < 4; ++j)
				acc[i][j] += a[i] * bb[j];
	}
#pragma unroll
	for (int j = 0; j < 4; ++j)
	{
		const int c = c0 + tc + 16 * j;
		if (c >= s)
			continue;
#pragma unroll
		for (int i = 0; i < 4; ++i)
		{
			const int r = r0 + tr + 16 * i;
			if (r < s)
				A[(int64_t)c * s + r] -= acc[i][j];
		}
	}
}

// x <- A^{-1} x with the factors: the interchanges, then forward substitution
// with unit L and back substitution with U, x in LDS (s <= lu_max_block)
__global__ __launch_bounds__(lu_panel_threads) void k_lu_solve(const double* __restrict__ A, int s,
															   const int32_t* __restrict__ ipiv, double* __restrict__ x)
{
	extern __shared__ double sx[];
	for (int i = threadIdx.x; i < s; i += lu_panel_threads)
		sx[i] = x[i];
	__syncthreads();
	if (threadIdx.x == 0)
		for (int j = 0; j < s; ++j)
		{
			const int p = ipiv[j];
			if (p != j)
			{
				const double t = sx[j];
				sx[j] = sx[p];
				sx[p] = t;
			}
		}
	__syncthreads();
	for (int j = 0; j < s; ++j)
	{
		const double xj = sx[j];
		const double* __restrict__ col = A + (int64_t)j * s;
		for (int i = j + 1 + threadIdx.x; i < s; i += lu_panel_threads)
			sx[i] -= col[i] * xj;
		__syncthreads();
	}
	for (int j = s - 1; j >= 0; --j)
	{
		const double* __restrict__ col = A + (int64_t)j * s;
		const double xj = sx[j] / col[j];
		__syncthreads();
		if (threadIdx.x == 0)
			sx[j] = xj;
		for (int i = threadIdx.x; i < j; i += lu_panel_threads)
			sx[i] -= col[i] * xj;
		__syncthreads();
	}
	for (int i = threadIdx.x; i < s; i += lu_panel_threads)
		x[i] = sx[i];
}

// r = rhs - M x on the block, M applied through the coupling structure (the
// LU overwrote its copy); used for iterative refinement with the factors
__global__ __launch_bounds__(sblock) void k_lu_residual(sys_t S, nbr_t G, int n_seg, int b, int64_t u0, int s,
														const double* __restrict__ x, const double* __restrict__ rhs,
														double* __restrict__ r)
{
	const int i = blockIdx.x * sblock + threadIdx.x;
	if (i >= s)
		return;
	const int64_t u = u0 + i;
	const int64_t off = (int64_t)b * S.nU;
	double mx;
	if (is_anchor(S, n_seg, b, u))
		mx = x[i];
	else
	{
		const double* __restrict__ rt = S.rates + (int64_t)b * S.rate_stride;
		mx = x[i] / S.invd[off + u];
		for (int32_t e = G.ptr[u]; e < G.ptr[u + 1]; ++e)
		{
			const int64_t k = (int64_t)G.nu[e] - u0;
			if (k >= 0 && k < s) // k_lu_assemble flags couplings that leave the block
				mx -= rt[G.nr[e] & 63] * x[k];
		}
	}
	r[i] = rhs[off + u] - mx;
}

__global__ __launch_bounds__(sblock) void k_lu_axpy(int s, const double* __restrict__ dx, double* __restrict__ x)
{
	const int i = blockIdx.x * sblock + threadIdx.x;
	if (i < s)
		x[i] += dx[i];
}

// z = D' x on the block (the solvers' convention outside the kernels)
__global__ __launch_bounds__(sblock) void k_lu_store(sys_t S, int b, int64_t u0, int s, const double* __restrict__ x,
													 double* __restrict__ z)
{
	const int i = blockIdx.x * sblock + threadIdx.x;
	if (i >= s)
		return;
	const int64_t at = (int64_t)b * S.nU + u0 + i;
	z[at] = x[i] / S.invd[at];
}

// ============================================================================
// host driver

namespace {

// Device arrays to the host with one wait, through the context's pinned staging
// buffer while they fit it.
struct readback_t
{
	struct item_t
	{
		void* to;
		size_t at, bytes;
	};
	ctx_t& c;
	std::vector<item_t> items;
	size_t used = 0;
	explicit readback_t(ctx_t& x) : c(x) {}
	template <typename T>
	void add(std::vector<T>& h, const T* d, size_t count)
	{
		h.resize(count);
		if (!count)
			return;
		const size_t bytes = count * sizeof(T);
		void* to = h.data();
		if (used + bytes <= c.h_stage_bytes)
		{
			items.push_back({ to, used, bytes });
			to = c.h_stage + used;
			used += (bytes + 15) / 16 * 16;
		}
		ESL_HIP(hipMemcpyAsync(to, d, bytes, hipMemcpyDeviceToHost, c.stream));
	}
	void wait()
	{
		ESL_HIP(hipStreamSynchronize(c.stream));
		for (const item_t& i : items)
			std::memcpy(i.to, c.h_stage + i.at, i.bytes);
		items.clear();
		used = 0;
	}
};

template <typename T>
void read_host(ctx_t& c, std::vector<T>& h, const T* d, size_t count)
{
	readback_t r(c);
	r.add(h, d, count);
	r.wait();
}

// terminal masks to their fixpoint
void propagate_masks(ctx_t& c, const graph_t& g, const uint8_t* reach, uint64_t* tmask)
{
	int hint = 4;
	fixpoint(c, hint, 8, 1 << 24, "terminal-mask propagation", [&](int32_t* f, const int32_t* pf) {
		ESL_HMAX_DISPATCH(g.N, k_tm,
						  <<<ceil_div(g.n, sblock), sblock, 0, c.stream>>>(g.N, g.n, g.mask.get(), g.rank.get(), g.T,
																		   reach, tmask, f, pf));
	});
}

template <typename T>
void write_dev(ctx_t& c, T* d, const std::vector<T>& h)
{
	if (!h.empty())
		ESL_HIP(hipMemcpyAsync(d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, c.stream));
}

// device time between marks on the stream, by the context's events; read once at the end
struct timer_t
{
	static constexpr int first = 4, most = 8;
	ctx_t& c;
	int marks = 0;
	explicit timer_t(ctx_t& x) : c(x) { mark(); }
	void mark()
	{
		if (marks < most)
			ESL_HIP(hipEventRecord(c.ev[first + marks++], c.stream));
	}
	void read(double* ms)
	{
		ESL_HIP(hipEventSynchronize(c.ev[first + marks - 1]));
		for (int i = 0; i + 1 < marks; ++i)
		{
			float t = 0;
			ESL_HIP(hipEventElapsedTime(&t, c.ev[first + i], c.ev[first + i + 1]));
			ms[i] = t;
		}
	}
};


// coupling structure of the per-set solver (see k_nbr_fill)
struct nbr_store_t
{
	bool ready = false;
	dbuf<int32_t> ptr, mid, nu, lvl;
	dbuf<uint8_t> nr;
	dbuf<uint32_t> hdr, rec;
	bool packed = false; // hdr / rec built
	levels_t L{};
	int64_t nnz = 0, nnz_t = 0; // of all rows, of the terminal rows
	// the same lists with rows and neighbours in level order (set-minor
	// device-wide solver), built on first use
	mutable dbuf<int32_t> wptr, wmid, wnu;
	mutable dbuf<uint8_t> wnr;
	mutable bool wready = false;
	// the same lists in parity-class order (reduced.hip.hpp)
	dbuf<int32_t> rptr, rrow;
	dbuf<uint4> rrec;
	int64_t nE = 0, nR = 0, rgroups = 0;
	rb_t rview() const { return rb_t{ (int)nE, (int)nR, rptr.get(), rrow.get(), rrec.get() }; }
	nbr_t view() const
	{
		return nbr_t{ ptr.get(), mid.get(), nu.get(), nr.get(), lvl.get(), L,
					  packed ? hdr.get() : nullptr, packed ? rec.get() : nullptr };
	}
	wnbr_t wview() const { return wnbr_t{ wptr.get(), wmid.get(), wnu.get(), wnr.get(), lvl.get(), L }; }
};

void build_wnbr(ctx_t& c, int64_t nU, const nbr_store_t& st)
{
	if (st.wready)
		return;
	const nbr_t G = st.view();
	const int nb = ceil_div(nU, sblock);
	dbuf<int32_t> inv, cnt;
	inv.ensure(nU);
	cnt.ensure(nU);
	st.wptr.ensure(nU + 1);
	st.wmid.ensure(nU);
	st.wnu.ensure(std::max<int64_t>(st.nnz, 1));
	st.wnr.ensure(std::max<int64_t>(st.nnz, 1));
	k_w_inv<<<nb, sblock, 0, c.stream>>>(nU, G.lvl, inv.get());
	k_w_count<<<nb, sblock, 0, c.stream>>>(nU, G, cnt.get());
	exclusive_scan_i32(c, cnt.get(), st.wptr.get(), nU);
	k_w_fill<<<nb, sblock, 0, c.stream>>>(nU, G, inv.get(), st.wptr.get(), st.wmid.get(), st.wnu.get(), st.wnr.get());
	ESL_HIP(hipGetLastError());
	ESL_HIP(hipStreamSynchronize(c.stream));
	st.wready = true;
}

// coupling lists in parity-class order from the lists by unknown; opos: exclusive
// scan of the odd-parity flags, n_odd their total
void build_rb(ctx_t& c, const sys_t& S, nbr_store_t& st, const int32_t* opos, int64_t n_odd, int32_t* cnt)
{
	const int64_t nU = S.nU;
	const int nb = ceil_div(nU, sblock);
	const int elim = n_odd > nU - n_odd ? 1 : 0; // the larger class is eliminated
	st.nE = elim ? n_odd : nU - n_odd;
	st.nR = nU - st.nE;
	dbuf<int32_t> inv;
	inv.ensure(nU);
	st.rptr.ensure(nU + 1);
	st.rrow.ensure(nU);
	k_rb_place<<<nb, sblock, 0, c.stream>>>(nU, (int)st.nE, elim, S.ulist, opos, st.ptr.get(), st.rrow.get(), inv.get(),
											cnt);
	exclusive_scan_i32(c, cnt, st.rptr.get(), nU);
	// groups of four per row: at most one of each row is not full; and one past the last,
	// for loads ahead
	st.rrec.ensure((size_t)(st.nnz / 4 + nU) + 1);
	k_rb_fill<<<nb, sblock, 0, c.stream>>>(nU, 2 * S.N, st.rrow.get(), inv.get(), st.ptr.get(), st.nu.get(), st.nr.get(),
										   st.rptr.get(), st.rrec.get());
	ESL_HIP(hipGetLastError());
}

void build_nbr(ctx_t& c, const sys_t& S, nbr_store_t& st)
{
	const int64_t nU = S.nU;
	const int nb = ceil_div(nU, sblock);
	dbuf<int32_t> cnt, lvl_key, opos;
	cnt.ensure(nU);
	lvl_key.ensure(nU);
	opos.ensure(nU + 1);
	st.ptr.ensure(nU + 1);
	st.mid.ensure(nU);
	st.lvl.ensure(nU);
	k_rb_parity<<<nb, sblock, 0, c.stream>>>(nU, S.ulist, cnt.get());
	exclusive_scan_i32(c, cnt.get(), opos.get(), nU);
	k_nbr_count<<<nb, sblock, 0, c.stream>>>(S, cnt.get());
	exclusive_scan_i32(c, cnt.get(), st.ptr.get(), nU);
	readback_t rd(c);
	std::vector<int32_t> h_nnz, h_odd, h_groups, h_nnz_t;
	rd.add(h_nnz, st.ptr.get() + nU, 1);
	rd.add(h_odd, opos.get() + nU, 1);
	rd.wait();
	const int32_t nnz = h_nnz[0], n_odd = h_odd[0];
	st.nnz = nnz;
	st.nu.ensure(std::max(nnz, 1));
	st.nr.ensure(std::max(nnz, 1));
	k_nbr_fill<<<nb, sblock, 0, c.stream>>>(S, st.ptr.get(), st.nu.get(), st.nr.get(), st.mid.get(), lvl_key.get());
	build_rb(c, S, st, opos.get(), n_odd, cnt.get());
	// unknowns grouped by popcount level (counting sort on the host: N + 1 buckets)
	const bool pack = nU <= lds_max_unknowns && nnz < 65536 && S.N < 128;
	std::vector<int32_t> h_key, h_ptr, h_mid, h_nu;
	std::vector<uint8_t> h_nr;
	rd.add(h_groups, st.rptr.get() + nU, 1);
	rd.add(h_nnz_t, st.ptr.get() + S.nUt, 1);
	rd.add(h_key, lvl_key.get(), (size_t)nU);
	if (pack)
	{
		rd.add(h_ptr, st.ptr.get(), (size_t)nU + 1);
		rd.add(h_mid, st.mid.get(), (size_t)nU);
		rd.add(h_nu, st.nu.get(), (size_t)nnz);
		rd.add(h_nr, st.nr.get(), (size_t)nnz);
	}
	rd.wait();
	st.rgroups = h_groups[0];
	st.nnz_t = h_nnz_t[0];
	st.L = levels_t{};
	st.L.n = S.N + 1;
	std::vector<int32_t> h_cnt(st.L.n + 1, 0), h_lvl(nU);
	for (int32_t k : h_key)
		h_cnt[k + 1]++;
	for (int l = 0; l < st.L.n; ++l)
		h_cnt[l + 1] += h_cnt[l];
	for (int l = 0; l <= st.L.n; ++l)
		st.L.off[l] = h_cnt[l];
	std::vector<int32_t> fill(h_cnt.begin(), h_cnt.end() - 1);
	for (int64_t u = 0; u < nU; ++u)
		h_lvl[fill[h_key[u]]++] = (int32_t)u;
	write_dev(c, st.lvl.get(), h_lvl);
	// level-ordered packed records for the LDS-resident kernels: positions and
	// record offsets must fit 16 bits, counts 7 bits (a row has at most N
	// neighbours)
	st.packed = false;
	if (pack)
	{
		std::vector<int32_t> pos(nU);
		for (int64_t p = 0; p < nU; ++p)
			pos[h_lvl[p]] = (int32_t)p;
		std::vector<uint32_t> h_hdr(nU), h_rec(std::max<int64_t>(nnz, 1));
		uint32_t at = 0;
		for (int64_t p = 0; p < nU; ++p)
		{
			const int32_t u = h_lvl[p];
			const uint32_t n_low = (uint32_t)(h_mid[u] - h_ptr[u]), cnt = (uint32_t)(h_ptr[u + 1] - h_ptr[u]);
			h_hdr[p] = at | n_low << 16 | cnt << 24;
			for (int32_t k = h_ptr[u]; k < h_ptr[u + 1]; ++k)
				h_rec[at++] = (uint32_t)pos[h_nu[k]] | (uint32_t)h_nr[k] << 16;
		}
		st.hdr.ensure(nU);
		st.rec.ensure(h_rec.size());
		write_dev(c, st.hdr.get(), h_hdr);
		write_dev(c, st.rec.get(), h_rec);
		st.packed = true;
	}
	ESL_HIP(hipStreamSynchronize(c.stream));
	st.ready = true;
}


// Device-wide GMRES(m) on the set-minor layout (the k_w_* kernels): the method
// of gmres_t -- FP64 iterate x, right preconditioning by Jacobi or the
// level-scheduled ILU(0), classical Gram-Schmidt (twice in FP64, once in FP32
// cycles), FP64 residual at every restart -- with every vector [row][set] in
// level order.  enter() gathers the plan's set-major right-hand side and
// iterate, leave() scatters the iterate back.  At most 1024 sets (one
// reduction block holds every set).  The preconditioned Arnoldi vector has the
// basis type (FP32 in FP32 cycles); pivots, the iterate, residuals and the
// correction of each cycle are FP64.
template <typename T>
struct gmres_w_t
{
	ctx_t& c;
	const sys_t& S;
	const nbr_store_t& NB;
	int n_seg, m;
	bool ilu;
	int64_t nU;
	int B, R, nred;
	wnbr_t G;
	dbuf<T> V, W;
	dbuf<T> t;		  // preconditioned Arnoldi vector
	dbuf<double> keep; // FP32 cycles: the last correction, undone if it raised the residual
	dbuf<double> r, ud, wrhs, wx, winvd; // ud: inverse ILU(0) pivots
	dbuf<double> rt, ct, yt; // rates, Gram-Schmidt coefficients, combination weights: [index][set]
	dbuf<uint8_t> wanc;
	dbuf<double> H, cs, sn, g, c1, c2, hn, beta, bnorm, res, vscale, part, rr, res0;
	dbuf<int32_t> live, act, kb;
	gm_state_t st{};
	std::vector<double> h_res;
	int iters = 0, cycles = 0;
	double final_res = 0.0;

	gmres_w_t(ctx_t& ctx, const sys_t& sys, const nbr_store_t& nb, int nseg, int restart, bool use_ilu)
		: c(ctx), S(sys), NB(nb), n_seg(nseg), m(restart), ilu(use_ilu), nU(sys.nU), B(sys.B)
	{
		if (B > 1024)
			throw error(ESL_E_ARG, "the device-wide solver takes at most 1024 rate sets per call");
		build_wnbr(c, nU, NB);
		G = NB.wview();
		// reduction kernels: B x R threads per workgroup (up to 1024), at most 512
		// workgroups (two per CU), so the per-block partial sums stay small
		R = std::max(1, 1024 / B);
		nred = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(nU, R), 512));
		const size_t cnt = (size_t)nU * B;
		V.ensure((size_t)(m + 1) * cnt);
		W.ensure(cnt);
		t.ensure(cnt);
		if (sizeof(T) == 4)
			keep.ensure(cnt);
		r.ensure(cnt);
		ud.ensure(cnt);
		wrhs.ensure(cnt);
		wx.ensure(cnt);
		winvd.ensure(cnt);
		wanc.ensure(cnt);
		H.ensure((size_t)B * (m + 1) * m);
		cs.ensure((size_t)B * m);
		sn.ensure((size_t)B * m);
		g.ensure((size_t)B * (m + 1));
		c1.ensure((size_t)B * (m + 1));
		c2.ensure((size_t)B * (m + 1));
		hn.ensure(B);
		beta.ensure(B);
		bnorm.ensure(B);
		res.ensure(B);
		vscale.ensure(B);
		live.ensure(B);
		act.ensure(B);
		kb.ensure(B);
		res0.ensure(B);
		part.ensure((size_t)nred * B * std::max(m + 1, 2) + 16);
		rr.ensure((size_t)B * 2);
		rt.ensure((size_t)64 * B);
		ct.ensure((size_t)(m + 1) * B);
		yt.ensure((size_t)(m + 1) * B);
		st = gm_state_t{ H.get(),	 cs.get(),	  sn.get(),	  g.get(),	 c1.get(),	c2.get(),
						 hn.get(),	 beta.get(), bnorm.get(), res.get(), live.get(), act.get(),
						 kb.get(),	 res0.get() };
		h_res.resize(B);
		if (sizeof(T) == 4) // one Gram-Schmidt pass: the second-pass coefficients stay zero
			k_zero<double><<<ceil_div(B * (m + 1), sblock), sblock, 0, c.stream>>>(B * (m + 1), c2.get());
	}

	int grid(int64_t count) const { return (int)ceil_div(count, sblock); }

	// plan vectors (set-major, z = D' x) -> solver vectors; ILU(0) pivots
	void enter(const double* rhs, const double* z)
	{
		k_w_gather<<<grid(nU * B), sblock, 0, c.stream>>>(S, n_seg, G.lvl, rhs, z, wrhs.get(), wx.get(), winvd.get(),
														   wanc.get());
		k_w_rates<<<grid(2 * S.N * B), sblock, 0, c.stream>>>(S.rates, S.rate_stride, 2 * S.N, B, rt.get());
		if (ilu)
			for (int l = 0; l < G.L.n; ++l)
			{
				const int cntl = G.L.off[l + 1] - G.L.off[l];
				if (cntl)
					k_w_ilu_pivot<<<grid((int64_t)cntl * B), sblock, 0, c.stream>>>(G, B, l, rt.get(), winvd.get(),
																					 wanc.get(), ud.get());
			}
		ESL_HIP(hipGetLastError());
	}

	void leave(double* z)
	{
		k_w_scatter<<<grid(nU * B), sblock, 0, c.stream>>>(nU, B, G.lvl, wx.get(), winvd.get(), z);
		ESL_HIP(hipGetLastError());
	}

	double max_res()
	{
		read_host(c, h_res, res.get(), (size_t)B);
		double mx = 0.0;
		for (double v : h_res)
			mx = std::max(mx, std::isnan(v) ? 1e300 : v);
		return mx;
	}

	// Liveness after Arnoldi step j is copied to pinned memory with an event and
	// read one step later, so the host never waits for the step it just
	// enqueued: the device runs step j while the host checks step j - 1.
	struct live_mirror_t
	{
		int32_t* h = nullptr; // [2][B]
		hipEvent_t ev[2] = { nullptr, nullptr };
		~live_mirror_t()
		{
			if (h)
				(void)hipHostFree(h);
			for (hipEvent_t e : ev)
				if (e)
					(void)hipEventDestroy(e);
		}
	} lm;

	void post_live(int j)
	{
		if (!lm.h)
		{
			ESL_HIP(hipHostMalloc((void**)&lm.h, 2 * (size_t)B * sizeof(int32_t), hipHostMallocDefault));
			for (hipEvent_t& e : lm.ev)
				ESL_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
		}
		ESL_HIP(hipMemcpyAsync(lm.h + (j & 1) * B, live.get(), (size_t)B * sizeof(int32_t), hipMemcpyDeviceToHost,
							   c.stream));
		ESL_HIP(hipEventRecord(lm.ev[j & 1], c.stream));
	}

	// whether any set was still live after step j (posted by post_live(j))
	bool live_after(int j)
	{
		ESL_HIP(hipEventSynchronize(lm.ev[j & 1]));
		const int32_t* f = lm.h + (j & 1) * B;
		for (int b = 0; b < B; ++b)
			if (f[b])
				return true;
		return false;
	}

	// v <- P^{-1} src for the sets with flags[b] != 0 (src may be v)
	template <typename X>
	void precondition(const X* src, X* v, const int32_t* flags)
	{
		if (!ilu)
		{
			if (src != v)
				k_w_copy_live<X, X><<<grid(nU * B), sblock, 0, c.stream>>>(nU * B, B, src, v, flags);
			k_w_jacobi<X><<<grid(nU * B), sblock, 0, c.stream>>>(nU * B, B, winvd.get(), v, flags);
			return;
		}
		for (int l = 0; l < G.L.n; ++l)
		{
			const int cntl = G.L.off[l + 1] - G.L.off[l];
			if (cntl)
				k_w_ilu_fwd<X><<<grid((int64_t)cntl * B), sblock, 0, c.stream>>>(G, B, l, rt.get(), wanc.get(),
																				 ud.get(), src, v, flags);
		}
		for (int l = G.L.n - 1; l >= 0; --l)
		{
			const int cntl = G.L.off[l + 1] - G.L.off[l];
			if (cntl)
				k_w_ilu_bwd<X><<<grid((int64_t)cntl * B), sblock, 0, c.stream>>>(G, B, l, rt.get(), wanc.get(),
																				 ud.get(), v, flags);
		}
	}

	bool solve(double tol, int max_iters, double inner_rtol = 0.0)
	{
		double prev = 0.0;
		const int64_t cnt = nU * B;
		const int gq = grid(cnt);
		const int64_t vstride = cnt;
		const int sb = ceil_div(B, 64);
		const int bs = B * R;
		for (;;)
		{
			k_w_residual<<<gq, sblock, 0, c.stream>>>(G, nU, B, rt.get(), winvd.get(), wanc.get(), wrhs.get(),
													  wx.get(), r.get());
			k_w_norms<<<nred, bs, 0, c.stream>>>(nU, B, R, r.get(), wrhs.get(), part.get());
			k_w_reduce<<<B, wred_threads, 0, c.stream>>>(part.get(), nred, B, 2, rr.get(), 2, nullptr);
			k_gm_start<<<sb, 64, 0, c.stream>>>(B, m, st, rr.get(), tol, vscale.get());
			ESL_HIP(hipGetLastError());
			final_res = max_res();
			if (final_res <= tol)
				return true;
			if (sizeof(T) == 4 && cycles > 0 && !(final_res < 0.9 * prev))
			{
				if (!(final_res <= prev))
				{
					k_sub1<<<gq, sblock, 0, c.stream>>>(cnt, keep.get(), wx.get());
					ESL_HIP(hipGetLastError());
					final_res = prev;
				}
				return false;
			}
			prev = final_res;
			if (iters >= max_iters)
				return false; // the caller checks every set's residual
			++cycles;
			k_w_cast_scale<T><<<gq, sblock, 0, c.stream>>>(cnt, B, r.get(), vscale.get(), V.get());
			int k = 0;
			for (int j = 0; j < m; ++j)
			{
				const T* Vj = V.get() + (int64_t)j * vstride;
				precondition<T>(Vj, t.get(), live.get());
				// algorithmic bytes: t read, W written, coupling structure and 1/D' read
				timed_launch(c, "k_w_apply", (double)cnt * (2.0 * sizeof(T) + 8.0) + 12.0 * nU + 5.0 * NB.nnz, [&] {
					k_w_apply<T, T><<<gq, sblock, 0, c.stream>>>(G, nU, B, rt.get(), winvd.get(), wanc.get(), t.get(),
																 W.get(), live.get());
				});
				const double dbytes = (double)cnt * sizeof(T) * (j + 2);
				timed_launch(c, "k_w_dots", dbytes, [&] {
					k_w_dots<T><<<nred, bs, 0, c.stream>>>(nU, B, R, j + 1, W.get(), V.get(), vstride, part.get(),
														   live.get());
				});
				k_w_reduce<<<B, wred_threads, 0, c.stream>>>(part.get(), nred, B, j + 1, c1.get(), m + 1,
																   ct.get());
				timed_launch(c, "k_w_orth", dbytes + (double)cnt * sizeof(T), [&] {
					k_w_orth<T><<<nred, bs, 0, c.stream>>>(nU, B, R, j + 1, W.get(), V.get(), vstride, ct.get(),
														   part.get(), live.get());
				});
				if (sizeof(T) != 4)
				{
					k_w_dots<T><<<nred, bs, 0, c.stream>>>(nU, B, R, j + 1, W.get(), V.get(), vstride, part.get(),
														   live.get());
					k_w_reduce<<<B, wred_threads, 0, c.stream>>>(part.get(), nred, B, j + 1, c2.get(), m + 1,
																	   ct.get());
					k_w_orth<T><<<nred, bs, 0, c.stream>>>(nU, B, R, j + 1, W.get(), V.get(), vstride, ct.get(),
														   part.get(), live.get());
				}
				k_w_reduce<<<B, wred_threads, 0, c.stream>>>(part.get(), nred, B, 1, hn.get(), 1, nullptr);
				k_gm_givens<<<sb, 64, 0, c.stream>>>(B, m, j, st, 0.5 * tol, sizeof(T) == 4 ? inner_rtol : 0.0);
				k_w_scale<T><<<gq, sblock, 0, c.stream>>>(cnt, B, W.get(), hn.get(), V.get() + (int64_t)(j + 1) * vstride,
														  live.get());
				ESL_HIP(hipGetLastError());
				++iters;
				k = j + 1;
				post_live(j);
				if (j > 0 && !live_after(j - 1))
				{
					// every set had stopped after step j - 1: step j changed nothing that
					// is used (dead sets keep their column count), so it is not counted
					--iters;
					k = j;
					break;
				}
				if (iters >= max_iters)
					break;
			}
			// x += P^{-1} (sum_i y_i V_i) in FP64
			k_gm_solve_y<<<sb, 64, 0, c.stream>>>(B, m, k, st);
			k_w_transpose_y<<<grid((int64_t)B * (m + 1)), sblock, 0, c.stream>>>(B, m, c1.get(), yt.get());
			k_zero<double><<<gq, sblock, 0, c.stream>>>(cnt, r.get());
			k_w_combine<T><<<gq, sblock, 0, c.stream>>>(cnt, B, k, V.get(), vstride, yt.get(), r.get(), kb.get());
			precondition<double>(r.get(), r.get(), act.get());
			if (sizeof(T) == 4) // keep the correction in t until the next residual has been checked
				k_axpy1_keep<<<gq, sblock, 0, c.stream>>>(cnt, r.get(), wx.get(), keep.get());
			else
				k_axpy1<<<gq, sblock, 0, c.stream>>>(cnt, r.get(), wx.get());
			ESL_HIP(hipGetLastError());
		}
	}
};

// Buffers of a device-wide reduced solve: nine vectors of unknowns x sets (1 GB for 64
// sets of 221,184 unknowns), so they are the call's, not the plan's; a pool of the context
// keeps its bound of them.  Kept with every plan, they made several large plans run out
// of memory.
struct rbw_ws_t
{
	ctx_t& ctx;
	dbuf<double> x, b, c, dj, res, keep, part, norms, pick_v, pa;
	dbuf<double> vec; // the vectors of the cycle: six on the kept rows, one on the others
	dbuf<rbw_set_t> st;
	dbuf<int32_t> undo, pick_u, seg_rows;
	explicit rbw_ws_t(ctx_t& c) : ctx(c) {}
	rbw_ws_t(const rbw_ws_t&) = delete;
	rbw_ws_t& operator=(const rbw_ws_t&) = delete;
	~rbw_ws_t()
	{
		const pool_scope_t scope(ctx.wide);
		if (ctx.wide_shared)
			(void)hipStreamSynchronize(ctx.stream); // the next owner may be on another stream
		for (dbuf<double>* d : { &x, &b, &c, &dj, &res, &keep, &part, &norms, &pick_v, &pa, &vec })
			d->reset();
		st.reset();
		for (dbuf<int32_t>* d : { &undo, &pick_u, &seg_rows })
			d->reset();
	}
	void reserve(int64_t nE, int64_t nR, int B, int nblk, int n_seg, int slices)
	{
		const pool_scope_t scope(ctx.wide);
		const size_t cU = (size_t)(nE + nR) * B, cR = (size_t)nR * B, cE = (size_t)nE * B;
		for (dbuf<double>* d : { &x, &b, &c, &res, &keep })
			d->ensure(cU);
		dj.ensure(cR);
		part.ensure((size_t)nblk * B * 5);
		norms.ensure((size_t)2 * B);
		vec.ensure(6 * cR + cE);
		pick_v.ensure((size_t)slices * n_seg * B);
		pick_u.ensure((size_t)slices * n_seg * B);
		pa.ensure((size_t)n_seg * B);
		seg_rows.ensure((size_t)2 * (n_seg + 1));
		st.ensure(B);
		undo.ensure((size_t)2 * B);
	}
};

// Device-wide BiCGStab on the parity-reduced system (the k_rbw_* kernels) for up
// to 1024 sets.  The host drives the cycles: it reads the FP64 residuals, decides
// per set (converged, another cycle, undone, stalled) and enqueues the iterations,
// checking liveness one iteration late so that the device never waits for it.
struct bicg_w_t
{
	ctx_t& c;
	const sys_t& S;
	const nbr_store_t& NB;
	rbw_ws_t& ws;
	int n_seg, B, W;
	rb_t G;
	rbw_geo_t geo{};
	int nbR, nbE, nbU, chunks, slices = 1;
	double *X, *R, *RH, *P, *V, *T2, *TE;
	std::vector<double> h_res; // relative residuals of the last check
	int iters = 0, cycles = 0;
	double final_res = 0.0;
	static constexpr int live_ev = timer_t::first + timer_t::most; // the context's events of the last two iterations
	static_assert(live_ev + 2 <= (int)(sizeof(ctx_t::ev) / sizeof(hipEvent_t)), "as many events");
	rb_setup_t su{};	// segments and anchors, where these may be moved
	bool moved = false; // anchors were

	bicg_w_t(ctx_t& ctx, const sys_t& sys, const nbr_store_t& nb, rbw_ws_t& w, int nseg)
		: c(ctx), S(sys), NB(nb), ws(w), n_seg(nseg), B(sys.B), G(nb.rview())
	{
		if (2 * B > live_words)
			throw error(ESL_E_ARG, "the device-wide solver takes at most 1024 rate sets per call");
		// up to 64 sets (an even share) side by side, two to a lane where the batch is
		// even, and as many rows as fill the block
		W = B % 2 ? 1 : 2;
		geo.B = B;
		geo.bs = ceil_div(ceil_div(B, ceil_div(B, rbw_sets)), W) * W;
		chunks = ceil_div(B, geo.bs);
		geo.L = geo.bs / W;
		geo.R = std::max(1, rbw_threads / geo.L);
		geo.ncode = 2 * S.N;
		geo.rates = S.rates;
		geo.rstride = S.rate_stride;
		auto blocks = [&](int64_t rows) {
			const int64_t k = std::max<int64_t>(1, std::min<int64_t>(ceil_div(rows, geo.R), std::max(8, 2048 / chunks)));
			return (int)(k > 8 ? k / 8 * 8 : k);
		};
		nbR = blocks(G.nR);
		nbE = blocks(G.nE);
		nbU = blocks((int64_t)G.nE + G.nR);
		slices = (int)std::max<int64_t>(1, std::min<int64_t>(64, S.nUt / (64 * std::max(1, n_seg))));
		ws.reserve(G.nE, G.nR, B, std::max(nbR, nbU), n_seg, slices);
		const size_t cR = (size_t)G.nR * B;
		X = ws.vec.get();
		R = X + cR;
		RH = R + cR;
		P = RH + cR;
		V = P + cR;
		T2 = V + cR;
		TE = T2 + cR;
		h_res.assign(B, 0.0);
	}

	// a kernel over row blocks, for W sets per lane (pick(W) names it); K sums per set
	// go through LDS, over the rates' place
	template <typename F, typename... A>
	void rows(int nb, int K, bool rates, F pick, A... args)
	{
		const int nt = geo.L * geo.R;
		const size_t lds = std::max((size_t)K * W * nt, rates ? (size_t)(geo.ncode + 1) * geo.bs : 0) * sizeof(double);
		if (W == 2)
			pick(two{})<<<dim3(nb, chunks), nt, lds, c.stream>>>(args...);
		else
			pick(one{})<<<dim3(nb, chunks), nt, lds, c.stream>>>(args...);
	}
	using one = std::integral_constant<int, 1>;
	using two = std::integral_constant<int, 2>;

	// set-up from the rates alone: coefficients, anchors (into anchor[b][seg]), start
	// vector and right-hand side
	void enter(const rb_setup_t& setup)
	{
		movable(setup);
		rows(nbU, 0, true, [](auto w) { return k_rbw_coef<decltype(w)::value>; }, S, G, geo, su, ws.c.get(), TE, P);
		if (su.n_seg)
		{
			for (int it = 0; it < rb_sweeps; ++it)
			{
				timed_launch(c, "k_rbw_sweep", 24.0 * G.nE * B, [&] {
					rows(nbE, 0, true, [](auto w) { return k_rbw_sweep<decltype(w)::value, false>; }, G, geo, ws.c.get(), P, TE);
				});
				timed_launch(c, "k_rbw_sweep", 32.0 * G.nR * B, [&] {
					rows(nbR, 0, true, [](auto w) { return k_rbw_sweep<decltype(w)::value, true>; }, G, geo, ws.c.get(), TE, P);
				});
			}
			pick(TE, P, nullptr);
		}
		rows(nbU, 0, false, [](auto w) { return k_rbw_start<decltype(w)::value>; }, S, G, geo, n_seg, su.x0, TE, P, ws.pa.get(), ws.c.get(), ws.x.get(), ws.b.get());
		diag();
	}

	// from the plan's vectors (another system, set up set-major)
	void enter(const double* rhs, const double* z)
	{
		const dim3 gt(ceil_div(S.nU, rbw_tile), ceil_div(B, rbw_tile));
		k_rbw_enter<<<gt, sblock, 0, c.stream>>>(S, G, n_seg, rhs, z, ws.x.get(), ws.b.get(), ws.c.get());
		diag();
	}

	// the segments, so that their anchors can be picked and moved
	void movable(const rb_setup_t& setup)
	{
		su = setup;
		if (su.n_seg)
			k_rbw_seg_rows<<<ceil_div(su.n_seg + 1, sblock), sblock, 0, c.stream>>>(G, su.n_seg, su.seg_off,
																					 ws.seg_rows.get());
	}

	// the rows of largest value in mE, mR as anchors, of every set or (replacing bad ones) of
	// the sets of `only`
	void pick(const double* mE, const double* mR, const int32_t* only)
	{
		const int nt = geo.L * geo.R;
		const size_t lds = (size_t)W * nt * 12;
		const dim3 gp(slices * su.n_seg, chunks);
		if (W == 2)
			k_rbw_pick<2><<<gp, nt, lds, c.stream>>>(G, geo, su.n_seg, slices, ws.seg_rows.get(), mE, mR, ws.pick_v.get(),
													 ws.pick_u.get());
		else
			k_rbw_pick<1><<<gp, nt, lds, c.stream>>>(G, geo, su.n_seg, slices, ws.seg_rows.get(), mE, mR, ws.pick_v.get(),
													 ws.pick_u.get());
		k_rbw_anchor<<<ceil_div(su.n_seg * B, sblock), sblock, 0, c.stream>>>(
			B, su.n_seg, slices, ws.pick_v.get(), ws.pick_u.get(), su.anchor, ws.pa.get(), only, ws.undo.get() + B);
	}

	// The anchors of the sets with a mark in `which` [B] moved where they are bad (k_rb_move);
	// returns which sets' were.  Other sets keep their iterates and coefficients, bit for bit.
	std::vector<int32_t> move_anchors(std::vector<int32_t> which)
	{
		which.resize((size_t)2 * B, 0);
		write_dev(c, ws.undo.get(), which);
		const int32_t* only = ws.undo.get();
		pick(ws.x.get(), ws.x.get() + (size_t)G.nE * B, only);
		rows(nbU, 0, true, [](auto w) { return k_rbw_coef<decltype(w)::value>; }, S, G, geo, su, ws.c.get(), TE, P);
		rows(nbU, 0, false, [](auto w) { return k_rbw_move<decltype(w)::value>; }, S, G, geo, n_seg, ws.pa.get(), only, ws.c.get(), ws.x.get(), ws.b.get());
		diag();
		std::vector<int32_t> got;
		read_host(c, got, ws.undo.get() + B, (size_t)B);
		return got;
	}

	void diag()
	{
		rows(nbR, 0, true, [](auto w) { return k_rbw_diag<decltype(w)::value>; }, G, geo, ws.c.get(), ws.dj.get());
		ESL_HIP(hipGetLastError());
	}

	void leave(double* z, double* invd)
	{
		const dim3 gt(ceil_div(S.nU, rbw_tile), ceil_div(B, rbw_tile));
		k_rbw_leave<<<gt, sblock, 0, c.stream>>>(S, G, ws.x.get(), ws.c.get(), ws.dj.get(), z, invd);
		ESL_HIP(hipGetLastError());
	}

	bool live_after(int j)
	{
		ESL_HIP(hipEventSynchronize(c.ev[live_ev + (j & 1)]));
		const int32_t* f = c.h_live + (size_t)(j & 1) * B;
		return std::any_of(f, f + B, [](int32_t v) { return v != 0; });
	}

	// two products by S for every live set
	void iteration(int j, double aim)
	{
		const rbw_set_t* st = ws.st.get();
		const double *cc = ws.c.get(), *dj = ws.dj.get();
		double* part = ws.part.get();
		int32_t* live = c.h_live + (size_t)(j & 1) * B;
		// algorithmic bytes: each vector and coefficient the step reads or writes once
		const double eb = 8.0 * G.nE * B, rb = 8.0 * G.nR * B, st_b = 16.0 * NB.rgroups;
		for (int half = 0; half < 2; ++half)
		{
			timed_launch(c, "k_rbw_te", rb + 2.0 * eb + st_b, [&] {
				rows(nbE, 0, true, [](auto w) { return k_rbw_te<decltype(w)::value>; }, G, geo, cc, half ? R : P, TE, st);
			});
			timed_launch(c, "k_rbw_mul", eb + 5.0 * rb + st_b, [&] {
				if (half)
				{
					rows(nbR, 5, true, [](auto w) { return k_rbw_mul<decltype(w)::value, true>; }, G, geo, cc, dj, TE, R, RH, T2, st, part);
				}
				else
				{
					rows(nbR, 1, true, [](auto w) { return k_rbw_mul<decltype(w)::value, false>; }, G, geo, cc, dj, TE, P, RH, V, st, part);
				}
			});
			if (half)
			{
				k_rbw_reduce<3><<<B, sblock, 0, c.stream>>>(part, nbR, B, ws.st.get(), nullptr, live, aim);
				timed_launch(c, "k_rbw_update", 8.0 * rb, [&] {
					rows(nbR, 0, false, [](auto w) { return k_rbw_update<decltype(w)::value>; }, (int64_t)G.nR, geo, X, R, P, V, T2, st);
				});
			}
			else
			{
				k_rbw_reduce<2><<<B, sblock, 0, c.stream>>>(part, nbR, B, ws.st.get(), nullptr, nullptr, 0.0);
				timed_launch(c, "k_rbw_s", 3.0 * rb, [&] {
					rows(nbR, 0, false, [](auto w) { return k_rbw_s<decltype(w)::value>; }, (int64_t)G.nR, geo, R, V, st);
				});
			}
		}
		ESL_HIP(hipGetLastError());
		ESL_HIP(hipEventRecord(c.ev[live_ev + (j & 1)], c.stream));
	}

	// false when sets are left above the tolerance
	bool solve(double tol, int max_iters)
	{
		std::vector<double> norms, prev(B, 0.0);
		std::vector<rbw_set_t> hs(B);
		std::vector<int32_t> undo(B, 0), fails(B, 0), compare(B, 0), tried(B, 0);
		const double* cc = ws.c.get();
		for (;;)
		{
			rows(nbU, 2, true, [](auto w) { return k_rbw_residual<decltype(w)::value>; }, G, geo, cc, ws.dj.get(), ws.b.get(), ws.x.get(), ws.res.get(), ws.part.get());
			k_rbw_reduce<0><<<B, sblock, 0, c.stream>>>(ws.part.get(), nbU, B, ws.st.get(), ws.norms.get(), nullptr, 0.0);
			ESL_HIP(hipGetLastError());
			read_host(c, norms, ws.norms.get(), (size_t)2 * B);
			bool any_undo = false, any_live = false, all = true;
			final_res = 0.0;
			for (int b = 0; b < B; ++b)
			{
				const double beta = std::sqrt(norms[2 * b]), bn = norms[2 * b + 1] > 0.0 ? std::sqrt(norms[2 * b + 1]) : 1.0;
				double rel = beta / bn;
				undo[b] = 0;
				hs[b] = rbw_set_t{};
				bool go = false;
				if (!(rel <= tol))
				{
					if (compare[b] && !(rel < 0.9 * prev[b]))
					{
						++fails[b];
						if (!(rel <= prev[b])) // worse: back to the iterate before the cycle
						{
							undo[b] = 1;
							any_undo = true;
							rel = prev[b];
						}
					}
					else if (compare[b])
						fails[b] = 0;
					go = fails[b] < rb_max_fails && !undo[b];
				}
				compare[b] = go;
				prev[b] = rel;
				h_res[b] = rel;
				all = all && rel <= tol;
				final_res = std::max(final_res, std::isnan(rel) ? 1e300 : rel);
				if (go)
				{
					hs[b].est = rel;
					hs[b].scale = beta;
					hs[b].live = 1;
					hs[b].fails = fails[b];
					any_live = true;
				}
			}
			if (any_undo)
			{
				write_dev(c, ws.undo.get(), undo);
				k_rbw_undo<<<ceil_div(S.nU * B, sblock), sblock, 0, c.stream>>>(S.nU * B, B, ws.keep.get(), ws.x.get(),
																				ws.undo.get());
				ESL_HIP(hipGetLastError());
				ESL_HIP(hipStreamSynchronize(c.stream));
				bool more = false;
				for (int b = 0; b < B; ++b)
				{
					compare[b] = 0; // every set's residual is taken again before the next cycle
					more = more || (h_res[b] > tol && fails[b] < rb_max_fails);
				}
				if (more)
					continue;
			}
			if (su.n_seg)
			{
				std::vector<int32_t> which(B, 0);
				for (int b = 0; b < B; ++b)
					which[b] = !(h_res[b] <= tol) && fails[b] >= rb_max_fails && !tried[b];
				if (std::any_of(which.begin(), which.end(), [](int32_t v) { return v != 0; }))
				{
					const std::vector<int32_t> got = move_anchors(which);
					bool again = false;
					for (int b = 0; b < B; ++b)
					{
						tried[b] |= which[b];
						if (!got[b])
							continue;
						fails[b] = 0;
						again = moved = true;
					}
					if (again)
					{
						std::fill(compare.begin(), compare.end(), 0); // as after an undone cycle
						continue;
					}
				}
			}
			if (all || !any_live || iters >= max_iters)
				return all;
			++cycles;
			write_dev(c, ws.st.get(), hs);
			const rbw_set_t* st = ws.st.get();
			rows(nbE, 0, false, [](auto w) { return k_rbw_te0<decltype(w)::value>; }, G, geo, cc, ws.res.get(), TE, st);
			rows(nbR, 3, true, [](auto w) { return k_rbw_init<decltype(w)::value>; }, G, geo, cc, ws.res.get(), TE, R, RH, P, X, st, ws.part.get());
			k_rbw_reduce<1><<<B, sblock, 0, c.stream>>>(ws.part.get(), nbR, B, ws.st.get(), nullptr, nullptr, 0.0);
			ESL_HIP(hipGetLastError());
			for (int j = 0; 2 * j < rb_cycle_products; ++j)
			{
				iteration(j, rb_aim * tol);
				iters += 2;
				if (j > 0 && !live_after(j - 1))
				{
					iters -= 2; // every set had stopped before iteration j
					break;
				}
				if (iters >= max_iters)
					break;
			}
			rows(nbR, 0, false, [](auto w) { return k_rbw_correct<decltype(w)::value, true>; }, G, geo, cc, ws.res.get(), X, ws.x.get(), ws.keep.get(), st);
			rows(nbE, 0, true, [](auto w) { return k_rbw_correct<decltype(w)::value, false>; }, G, geo, cc, ws.res.get(), X, ws.x.get(), ws.keep.get(), st);
			ESL_HIP(hipGetLastError());
		}
	}
};

// Systems up to this size per set run as one workgroup per set; larger ones
// device-wide.  Measured on MI355X: 128 sets of 32,724 unknowns take 115 ms per
// set-workgroup and 50 ms device-wide, 128 sets of 239,616 unknowns 2.4 s and
// 1.0 s, while systems of a few thousand unknowns are fastest per set at any
// batch size.  esl_plan_autotune measures the choice for a given batch.
int64_t per_set_max_unknowns(int B)
{
	(void)B;
	return 4096;
}

// algorithmic bytes of one per-set launch: the coupling structure once
// (row pointers, neighbour index and code), then per set the right-hand side,
// the iterate (read and written) and 1/D'.
double gmres_set_bytes(const sys_t& S, int64_t nnz)
{
	return (double)S.nU * 12.0 + (double)nnz * 5.0 + (double)S.B * S.nU * (8.0 + 16.0 + 8.0);
}

// Solves A_p z = rhs for every set of S (z holds the initial guess): one
// workgroup per set when the system is small, device-wide otherwise.
struct krylov_result_t
{
	double resid = 0.0;
	int iters = 0, cycles = 0;
	int sets_iterated = 0; // sets whose initial iterate missed the tolerance
	int fp64_fallback = 0; // sets finished in FP64 after their FP32 cycles stalled
	int finished = 0;	   // sets that a second launch finished (their vectors changed after the first)
	int missed = 0;		   // sets above the tolerance
	int64_t iters_sum = 0; // iterations summed over the sets
	int exact = 0;		   // sets solved by the exact dense LU
};

// device scratch of the per-set kernels (pointers only)
struct pss_view_t
{
	double *r = nullptr, *udiag = nullptr, *res = nullptr, *t = nullptr;
	double* xk = nullptr; // reduced solver: the iterate before the last cycle
	int32_t *its = nullptr, *cyc = nullptr, *stl = nullptr;
	uint64_t* tspan = nullptr; // [B][2] start / end wall clock of each set's workgroup
	float* Vf = nullptr;  // FP32 basis (precision 1)
	double* Vd = nullptr; // FP64 basis (precision 0, and the FP64 finish of precision 1)
};

// per-set outcome of a solve: relative FP64 residual, Krylov iterations and
// how the set was finished (0 Krylov at the asked precision, 1 FP64 Krylov
// after stalled FP32 cycles, 2 exact dense LU, -1 above the tolerance)
struct set_results_t
{
	std::vector<double> res;
	std::vector<int32_t> its, method;
	std::vector<uint64_t> tspan; // per-set start / end wall clock of the last per-set launch (empty otherwise)
};

std::string sci(double v)
{
	char buf[32];
	std::snprintf(buf, sizeof buf, "%.3e", v);
	return buf;
}

// per-set results of the last launch: max / sums over the sets, and the host
// copies of the per-set residuals, iteration and cycle counts
// The per-set outputs of a launch (residuals, start / end clocks, iterations,
// cycles) in one staged copy: the arrays go back to back into the context's
// pinned buffer, enqueued behind the launch so that one wait covers both, where
// a copy per array into pageable memory costs a host round trip each.  Returns
// false (nothing enqueued) when the batch does not fit the buffer.
bool stage_set_outputs(ctx_t& c, const pss_view_t& sc, int B)
{
	const size_t nb = (size_t)std::max(B, 0);
	if (!c.h_stage || nb == 0 || nb * 32 > c.h_stage_bytes)
		return false;
	unsigned char* p = c.h_stage;
	ESL_HIP(hipMemcpyAsync(p, sc.res, 8 * nb, hipMemcpyDeviceToHost, c.stream));
	ESL_HIP(hipMemcpyAsync(p + 8 * nb, sc.tspan, 16 * nb, hipMemcpyDeviceToHost, c.stream));
	ESL_HIP(hipMemcpyAsync(p + 24 * nb, sc.its, 4 * nb, hipMemcpyDeviceToHost, c.stream));
	ESL_HIP(hipMemcpyAsync(p + 28 * nb, sc.cyc, 4 * nb, hipMemcpyDeviceToHost, c.stream));
	return true;
}

// staged: stage_set_outputs already enqueued the copies for this view and batch
void read_set_outputs(ctx_t& c, const pss_view_t& sc, int B, std::vector<double>& res, std::vector<int32_t>& its,
					  std::vector<int32_t>& cyc, std::vector<uint64_t>* tspan, bool staged)
{
	const size_t nb = (size_t)std::max(B, 0);
	if (staged || stage_set_outputs(c, sc, B))
	{
		ESL_HIP(hipStreamSynchronize(c.stream));
		const unsigned char* p = c.h_stage;
		const double* h_res = reinterpret_cast<const double*>(p);
		const uint64_t* h_ts = reinterpret_cast<const uint64_t*>(p + 8 * nb);
		const int32_t* h_its = reinterpret_cast<const int32_t*>(p + 24 * nb);
		const int32_t* h_cyc = h_its + nb;
		res.assign(h_res, h_res + nb);
		its.assign(h_its, h_its + nb);
		cyc.assign(h_cyc, h_cyc + nb);
		if (tspan)
			tspan->assign(h_ts, h_ts + 2 * nb);
		return;
	}
	read_host(c, res, sc.res, nb);
	read_host(c, its, sc.its, nb);
	read_host(c, cyc, sc.cyc, nb);
	if (tspan)
		read_host(c, *tspan, sc.tspan, 2 * nb);
}

krylov_result_t collect_sets(ctx_t& c, const pss_view_t& sc, int B, double tol, bool check,
							 std::vector<double>* h_res_out = nullptr, std::vector<int32_t>* h_its_out = nullptr,
							 std::vector<uint64_t>* tspan_out = nullptr, bool staged = false)
{
	krylov_result_t kr;
	std::vector<int32_t> h_its, h_cyc;
	std::vector<double> h_res;
	read_set_outputs(c, sc, B, h_res, h_its, h_cyc, tspan_out, staged);
	for (int b = 0; b < B; ++b)
	{
		kr.resid = std::max(kr.resid, std::isnan(h_res[b]) ? 1e300 : h_res[b]);
		kr.iters = std::max(kr.iters, h_its[b]);
		kr.cycles = std::max(kr.cycles, h_cyc[b]);
		kr.sets_iterated += h_cyc[b] > 0 ? 1 : 0;
		kr.missed += (h_res[b] <= tol) ? 0 : 1;
		kr.iters_sum += h_its[b];
	}
	if (check && !(kr.resid <= tol))
		throw error(ESL_E_NUMERIC, "the solve did not reach the tolerance: relative residual " + sci(kr.resid) +
									   " after " + std::to_string(kr.iters) + " iterations");
	if (h_res_out)
		*h_res_out = std::move(h_res);
	if (h_its_out)
		*h_its_out = std::move(h_its);
	return kr;
}

// scratch of the per-set kernels, grown on demand and reused
struct per_set_scratch_t
{
	dbuf<double> r, udiag, res, t, xk;
	dbuf<int32_t> its, cyc, stl;
	dbuf<uint64_t> tspan;
	dbuf<float> Vf;
	dbuf<double> Vd;
	// reduced: for the reduced solver, which keeps no basis
	void reserve(int B, int64_t nU, int m, int precision, bool reduced)
	{
		nU = std::max<int64_t>(nU, 1);
		r.ensure((size_t)B * nU);
		udiag.ensure((size_t)B * nU);
		res.ensure(B);
		its.ensure(B);
		cyc.ensure(B);
		stl.ensure(B);
		tspan.ensure((size_t)2 * B);
		t.ensure((size_t)B * nU);
		if (reduced)
			xk.ensure((size_t)B * nU);
		else if (precision == 1)
			Vf.ensure((size_t)B * (m + 1) * nU);
		else
			Vd.ensure((size_t)B * (m + 1) * nU);
	}
	pss_view_t view() const
	{
		return pss_view_t{ r.get(),	  udiag.get(), res.get(),	t.get(),  xk.get(), its.get(),
						   cyc.get(), stl.get(),   tspan.get(), Vf.get(), Vd.get() };
	}
};

// schedules of a plan (esl_plan_autotune): how a run solves its systems
enum : int
{
	path_lds = 0,	  // per set, GMRES, system in LDS (private per-thread FP32 basis where it fits)
	path_global = 1,  // per set, GMRES from global memory
	path_wide = 2,	  // device-wide, GMRES
	path_lds_mem = 3, // as 0 with the basis in global memory
	path_lds_o3 = 4,  // as 0 with 3 workgroups per CU
	path_reduced = 5  // per set, BiCGStab on the parity-reduced system
};

// The reduced solver's kernel for this system and batch, or null when another
// path or a preconditioner of GMRES is asked for by name, or none fits.
const bicg_variant_t* reduced_variant(const ctx_t& c, const sys_t& S, const nbr_store_t& nb, const esl_solve_opts& o,
									  int path)
{
	if (path != path_reduced || o.preconditioner != 0)
		return nullptr;
	return rb_variant(nb.nE, nb.nR, nb.rgroups, S.B, (size_t)std::min(c.lds_per_block, 160 * 1024));
}

// one launch: the solve of every set, one workgroup per set (no host synchronisation)
// path: the schedule; path_reduced falls back to path_lds where no reduced variant fits
// su: the reduced solver's set-up from the rates (x0 null: the plan's vectors are set up)
void launch_per_set(ctx_t& c, const sys_t& S, const nbr_store_t& nb, int n_seg, const double* rhs, double* z,
					const esl_solve_opts& o, const pss_view_t& sc, int path, const rb_setup_t& su = {})
{
	const int B = S.B;
	const int m = std::min(std::max(o.restart > 0 ? o.restart : 32, 2), pm_max);
	const int nseg1 = std::max(n_seg, 1);
	const bool ilu = o.preconditioner != 1; // ILU(0) unless Jacobi is asked for
	const nbr_t G = nb.view();
	pgm_out_t po{ sc.its, sc.cyc, sc.res, sc.stl, sc.tspan };
	const double by = gmres_set_bytes(S, nb.nnz);
	if (const bicg_variant_t* v = reduced_variant(c, S, nb, o, path))
	{
		const size_t lds = rb_lds_bytes(S.nU, nb.rgroups, v->lrec);
		const bicg_set_fn fn = v->fn;
		if (lds > 48 * 1024)
			ESL_HIP(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
		const rb_scratch_t sp{ sc.r, sc.udiag, sc.t, sc.xk };
		timed_launch(c, "k_bicg_set", by, [&] {
			fn<<<B, v->blk, lds, c.stream>>>(S, nb.rview(), nseg1, rhs, z, sp, su, o.tol, o.max_iters, po);
		});
		ESL_HIP(hipGetLastError());
		return;
	}
	const bool allow_reg = path != path_lds_mem;
	if (path != path_global && ilu && nb.packed)
	{
		// LDS-resident kernel when its structure, pivots and vector fit
		const int psize = o.precision == 1 ? 4 : 8;
		const lds_plan_t lp = lds_plan(S.nU, nb.nnz, m, psize);
		if (lp.bytes + lds_static_bytes <= std::min(c.lds_per_block, 160 * 1024))
		{
			const bool small = S.nU <= 4 * pblock;
			if (lp.bytes > 48 * 1024)
			{
				const void* fns[13] = { (const void*)k_gmres_lds<float, 4>,  (const void*)k_gmres_lds<float, 8>,
										(const void*)k_gmres_lds<double, 4>, (const void*)k_gmres_lds<double, 8>,
										(const void*)k_gmres_priv<32>,		 (const void*)k_gmres_priv<24>,
										(const void*)k_gmres_priv<16>,		 (const void*)k_gmres_priv8<32>,
										(const void*)k_gmres_priv8<24>,		 (const void*)k_gmres_priv8<16>,
										(const void*)k_gmres_priv_o3<32>,	 (const void*)k_gmres_priv_o3<24>,
										(const void*)k_gmres_priv_o3<16> };
				for (const void* f : fns)
					ESL_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lp.bytes));
			}
			if (o.precision == 1 && !small && m <= 32 && allow_reg)
			{
				pgm_scratch_t sp{ sc.r, sc.udiag, sc.t, sc.Vf };
				timed_launch(c, "k_gmres_priv8<float>", by, [&] {
					if (m <= 16)
						k_gmres_priv8<16><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol,
																			  o.max_iters, po, lp, o.inner_rtol);
					else if (m <= 24)
						k_gmres_priv8<24><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol,
																			  o.max_iters, po, lp, o.inner_rtol);
					else
						k_gmres_priv8<32><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol,
																			  o.max_iters, po, lp, o.inner_rtol);
				});
			}
			else if (o.precision == 1 && small && m <= 32 && allow_reg)
			{
				// the FP32 basis of each thread's rows as a private array
				pgm_scratch_t sp{ sc.r, sc.udiag, sc.t, sc.Vf };
#define ESL_PRIV_LAUNCH(KERNEL)                                                                                \
	do                                                                                                         \
	{                                                                                                          \
		if (m <= 16)                                                                                           \
			KERNEL<16><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol, o.max_iters, po, lp, \
														  o.inner_rtol);                                      \
		else if (m <= 24)                                                                                      \
			KERNEL<24><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol, o.max_iters, po, lp, \
														  o.inner_rtol);                                      \
		else                                                                                                   \
			KERNEL<32><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol, o.max_iters, po, lp, \
														  o.inner_rtol);                                      \
	} while (0)
				timed_launch(c, path == path_lds_o3 ? "k_gmres_priv_o3<float>" : "k_gmres_priv<float>", by, [&] {
					if (path == path_lds_o3)
						ESL_PRIV_LAUNCH(k_gmres_priv_o3);
					else
						ESL_PRIV_LAUNCH(k_gmres_priv);
				});
#undef ESL_PRIV_LAUNCH
			}
			else if (o.precision == 1)
			{
				pgm_scratch_t sp{ sc.r, sc.udiag, sc.t, sc.Vf };
				timed_launch(c, "k_gmres_lds<float>", by, [&] {
					if (small)
						k_gmres_lds<float, 4><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol,
																				 o.max_iters, po, lp, o.inner_rtol);
					else
						k_gmres_lds<float, 8><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol,
																				 o.max_iters, po, lp, o.inner_rtol);
				});
			}
			else
			{
				pgm_scratch_t sp{ sc.r, sc.udiag, sc.t, sc.Vd };
				timed_launch(c, "k_gmres_lds<double>", by, [&] {
					if (small)
						k_gmres_lds<double, 4><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol,
																				  o.max_iters, po, lp, o.inner_rtol);
					else
						k_gmres_lds<double, 8><<<B, pblock, lp.bytes, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol,
																				  o.max_iters, po, lp, o.inner_rtol);
				});
			}
			ESL_HIP(hipGetLastError());
			return;
		}
	}
	if (o.precision == 1)
	{
		pgm_scratch_t sp{ sc.r, sc.udiag, sc.t, sc.Vf };
		timed_launch(c, ilu ? "k_gmres_set<float,ilu>" : "k_gmres_set<float,jacobi>", by, [&] {
			if (ilu)
				k_gmres_set<float, true><<<B, pblock, 0, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol, o.max_iters,
																	 po, o.inner_rtol);
			else
				k_gmres_set<float, false><<<B, pblock, 0, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol,
																	  o.max_iters, po, o.inner_rtol);
		});
	}
	else
	{
		pgm_scratch_t sp{ sc.r, sc.udiag, sc.t, sc.Vd };
		timed_launch(c, ilu ? "k_gmres_set<double,ilu>" : "k_gmres_set<double,jacobi>", by, [&] {
			if (ilu)
				k_gmres_set<double, true><<<B, pblock, 0, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol, o.max_iters,
																	  po, o.inner_rtol);
			else
				k_gmres_set<double, false><<<B, pblock, 0, c.stream>>>(S, G, nseg1, rhs, z, sp, m, o.tol,
																	   o.max_iters, po, o.inner_rtol);
		});
	}
	ESL_HIP(hipGetLastError());
}

// Reads the per-set results of a launch_per_set.  Sets that the reduced solver leaves
// above the tolerance get their bad anchors moved (k_rb_move) and another go; what it
// still leaves starts over with GMRES, as where that is asked for by name (FP32 cycles
// with refinement in mixed precision).  Sets that missed the tolerance with GMRES in mixed
// precision (their FP32 cycles stalled) are finished by FP64 GMRES from their current
// iterate; sets that already converged leave it at their first residual check.
// basis(precision) gives the scratch with a basis of that precision (it may grow it).
// Nothing is thrown here: sets still above the tolerance are counted in kr.missed and
// marked in `out` (method -1) for the caller's fallback.
template <typename F>
krylov_result_t finish_per_set(ctx_t& c, const sys_t& S, const nbr_store_t& nb, int n_seg, const double* rhs,
							   double* z, esl_solve_opts o, const pss_view_t& sc, bool reduced, rb_setup_t su,
							   F&& basis, set_results_t* out = nullptr, bool staged = false)
{
	ESL_HIP(hipStreamSynchronize(c.stream));
	const int B = S.B;
	set_results_t sr;
	sr.method.assign(B, 0);
	krylov_result_t kr = collect_sets(c, sc, B, o.tol, false, &sr.res, &sr.its, &sr.tspan, staged);
	if (reduced && su.n_seg && kr.missed > 0)
	{
		k_rb_move<<<B, sblock, 0, c.stream>>>(S, su, sc.res, o.tol, z, sc.stl);
		ESL_HIP(hipGetLastError());
		std::vector<int32_t> moved;
		read_host(c, moved, sc.stl, (size_t)B);
		const int n_moved = (int)std::count(moved.begin(), moved.end(), 1);
		if (n_moved)
		{
			su.x0 = nullptr;
			su.only = sc.stl;
			launch_per_set(c, S, nb, n_seg, rhs, z, o, sc, path_reduced, su);
			std::vector<double> res2;
			std::vector<int32_t> its2;
			const krylov_result_t k2 = collect_sets(c, sc, B, o.tol, false, &res2, &its2);
			for (int b = 0; b < B; ++b)
				if (moved[b])
				{
					sr.res[b] = res2[b];
					sr.its[b] += its2[b];
					kr.iters = std::max(kr.iters, sr.its[b]);
					kr.iters_sum += its2[b];
				}
			kr.finished += n_moved;
			kr.missed = k2.missed;
			kr.resid = k2.resid;
			kr.cycles += k2.cycles;
		}
	}
	if (reduced && kr.missed > 0)
		k_rb_restart<<<dim3(ceil_div(S.nU, sblock), B), sblock, 0, c.stream>>>(S, std::max(n_seg, 1), sc.res, o.tol, z,
																				 nullptr);
	if (reduced && kr.missed > 0 && o.precision == 1)
	{
		const pss_view_t sf = basis(1);
		launch_per_set(c, S, nb, n_seg, rhs, z, o, sf, path_lds);
		std::vector<double> res2;
		std::vector<int32_t> its2;
		const krylov_result_t k2 = collect_sets(c, sf, B, o.tol, false, &res2, &its2);
		for (int b = 0; b < B; ++b)
		{
			sr.res[b] = res2[b];
			sr.its[b] += its2[b];
		}
		kr.finished += kr.missed;
		kr.missed = k2.missed;
		kr.resid = k2.resid;
		kr.iters += k2.iters;
		kr.cycles += k2.cycles;
		kr.iters_sum += k2.iters_sum;
	}
	if ((o.precision == 1 || reduced) && kr.missed > 0)
	{
		const bool mixed = o.precision == 1;
		o.precision = 0;
		const pss_view_t sd = basis(0);
		launch_per_set(c, S, nb, n_seg, rhs, z, o, sd, path_lds);
		ESL_HIP(hipStreamSynchronize(c.stream));
		std::vector<double> res2;
		std::vector<int32_t> its2;
		const krylov_result_t k2 = collect_sets(c, sd, B, o.tol, false, &res2, &its2);
		for (int b = 0; b < B; ++b)
		{
			if (!(sr.res[b] <= o.tol) && mixed)
				sr.method[b] = 1;
			sr.res[b] = res2[b];
			sr.its[b] += its2[b];
		}
		kr.finished += kr.missed;
		kr.fp64_fallback = mixed ? kr.missed : 0;
		kr.missed = k2.missed;
		kr.resid = k2.resid;
		kr.iters += k2.iters;
		kr.cycles += k2.cycles;
		kr.iters_sum += k2.iters_sum;
	}
	for (int b = 0; b < B; ++b)
		if (!(sr.res[b] <= o.tol))
			sr.method[b] = -1;
	if (out)
		*out = std::move(sr);
	return kr;
}

// everything a solve needs that does not depend on the rates
struct plan_t
{
	static uint64_t next_id()
	{
		static std::atomic<uint64_t> n{ 0 };
		return ++n;
	}
	const uint64_t id = next_id();
	graph_t* g = nullptr;
	dbuf<double> x0;
	dbuf<uint8_t> reach;
	dbuf<uint64_t> tmask;
	dbuf<int32_t> amb, pos, ulist, ucls, d_jmap, d_segmap, d_seg_off, d_tpos;
	std::vector<int32_t> jmap, segmap, seg_off, seg_src;
	int Tr = 0, n_seg = 0;
	bool fallback = false;
	int64_t nU = 0, nUt = 0, nA = 0;
	dbuf<double> y0;
	// exit edges of the ambiguous set sorted by target (k_exit_sum): segment
	// offsets (host and device), unknown and rate index of each edge
	std::vector<int32_t> ex_off;
	dbuf<int32_t> d_ex_off, ex_u;
	dbuf<uint8_t> ex_r;
	int64_t n_exit = 0;
	nbr_store_t nbr;
	// per-run buffers (grown to the largest batch seen)
	dbuf<double> p0, p1, invd, rhs, z, y, segsum;
	dbuf<int32_t> anchor;
	per_set_scratch_t scr;
	// the buffers the run being enqueued uses: the ones above (plan_reserve), or
	// slices of the library's static scratch (plan_run_noalloc)
	struct run_bufs_t
	{
		double *p0 = nullptr, *p1 = nullptr, *invd = nullptr, *rhs = nullptr, *z = nullptr, *y = nullptr,
			   *segsum = nullptr;
		int32_t* anchor = nullptr;
		pss_view_t ps;
	} rb;
	void use_own_bufs()
	{
		rb = run_bufs_t{ p0.get(), p1.get(), invd.get(), rhs.get(), z.get(), y.get(), segsum.get(),
						 anchor.get(), scr.view() };
	}
	int anchor_sweeps = 32;
	size_t anchor_lds = 0; // dynamic LDS of k_anchor_lds, 0 when the terminal unknowns do not fit
	size_t anchor_lvl = 0; // dynamic LDS of k_anchor_lvl, 0 without packed records
	int64_t epoch = 0; // bumped whenever a per-run buffer is reallocated
	// schedule chosen by plan_autotune, used when a solve asks for restart 0
	struct tune_t
	{
		bool set = false;
		int path = 0; // path_lds ... path_reduced
		int m = 32;
	} tune;
	int path = 0; // the schedule of the run being enqueued
	set_results_t results; // per-set outcome of the last run (esl_plan_set_results)
	double ms[3] = { 0, 0, 0 };
	// captured numeric sequence and the arguments it was captured with
	struct gkey_t
	{
		int B = 0;
		const double* rates = nullptr;
		double* fin = nullptr;
		const double* warm = nullptr;
		int precision = 0, preconditioner = 0, m = 0;
		double tol = 0, inner_rtol = 0;
		int max_iters = 0;
		int64_t epoch = 0;
		int path = 0;
		bool operator==(const gkey_t& o) const
		{
			return B == o.B && rates == o.rates && fin == o.fin && warm == o.warm && precision == o.precision &&
				   preconditioner == o.preconditioner && m == o.m && tol == o.tol && inner_rtol == o.inner_rtol &&
				   max_iters == o.max_iters && epoch == o.epoch && path == o.path;
		}
	};
	gkey_t gkey{};
	bool gprof = false; // captured with profiling events
	hipGraphExec_t gexec = nullptr;
	std::vector<hipEvent_t> gev;			   // events recorded by the graph
	std::vector<prof_t::pending_t> gpend;	   // kernels timed inside the graph
	plan_t() = default;
	plan_t(const plan_t&) = delete;
	plan_t& operator=(const plan_t&) = delete;
	void drop_graph()
	{
		if (gexec)
			(void)hipGraphExecDestroy(gexec);
		gexec = nullptr;
		for (auto e : gev)
			(void)hipEventDestroy(e);
		gev.clear();
		gpend.clear();
	}
	~plan_t() { drop_graph(); }
	sys_t sys(int B, const double* rates) const;
	rb_setup_t setup(const double* warm) const
	{
		return rb_setup_t{ x0.get(), d_seg_off.get(), n_seg,	rb.anchor, rb.invd, rb.rhs, n_seg ? warm : nullptr,
						   d_tpos.get(), g->n_t, nullptr };
	}
};


// Restart length of the device-wide solver for cb sets of nU unknowns: the
// caller's (at most dw_max), or by default 32, lowered while the basis in FP64
// (what a stalled FP32 solve falls back to) would exceed half of the free
// device memory.  Longer restarts pay off on some systems and not on others
// (MI355X, FP32 cycles + FP64 refinement, sets/s at restart 32 -> 64): N=22
// seed 0, 1,769,472 unknowns: 27 -> 37 (241 -> 128 iterations per set; at 96
// and 128 the cycles end at their FP32 accuracy target first, 37.6); N=22
// seed 8, 221,184 unknowns: 203 -> 377; N=20 seeds 4 / 7, 524,288 unknowns:
// 132 -> 79 and 236 -> 153; the uneven 8-network batch: 4.66 k -> 2.66 k.
// So the default stays 32 and callers (or the autotuner) ask for more.
int dw_restart(int requested, int64_t nU, int cb)
{
	int m = requested > 0 ? std::min(std::max(requested, 2), dw_max) : 32;
	if (requested > 0)
		return m;
	size_t free_b = 0, total_b = 0;
	if (hipMemGetInfo(&free_b, &total_b) != hipSuccess)
		free_b = 0;
	while (m > 8 && (double)(m + 1) * (double)nU * cb * sizeof(double) > 0.5 * (double)free_b)
		m /= 2;
	return m;
}

// throw_on_miss = false leaves sets above the tolerance to the caller (kr.missed);
// setup: the reduced solver may move anchors, and where it has x0 sets itself up (rhs, z
// and S.invd need no values)
krylov_result_t krylov_solve(ctx_t& c, const sys_t& S, int n_seg, const double* rhs_p, double* z_p,
							 const esl_solve_opts& opts, const nbr_store_t* prebuilt = nullptr, bool device_wide = false,
							 bool throw_on_miss = true, std::vector<double>* set_res = nullptr,
							 int path = path_reduced, const rb_setup_t* setup = nullptr)
{
	krylov_result_t kr;
	const int64_t nU = S.nU;
	const int B = S.B;
	const double tol = opts.tol > 0 ? opts.tol : 1e-13;
	const int max_iters = opts.max_iters > 0 ? opts.max_iters : 20000;
	const int restart = std::min(std::max(opts.restart > 0 ? opts.restart : 32, 2), dw_max);
	if (opts.restart > 0 && path == path_reduced)
		path = path_lds;
	if (!device_wide && nU <= per_set_max_unknowns(B))
	{
		const int m = std::min(restart, pm_max);
		nbr_store_t local;
		if (!prebuilt)
			build_nbr(c, S, local);
		const nbr_store_t& nb = prebuilt ? *prebuilt : local;
		per_set_scratch_t sc;
		esl_solve_opts o = opts;
		o.tol = tol;
		o.max_iters = max_iters;
		o.restart = m;
		const bool reduced = reduced_variant(c, S, nb, o, path) != nullptr;
		sc.reserve(B, nU, m, opts.precision, reduced);
		launch_per_set(c, S, nb, n_seg, rhs_p, z_p, o, sc.view(), path);
		kr = finish_per_set(c, S, nb, n_seg, rhs_p, z_p, o, sc.view(), reduced, setup ? *setup : rb_setup_t{}, [&](int prec) {
			sc.reserve(B, nU, m, prec, false);
			return sc.view();
		});
		if (kr.missed && throw_on_miss)
			throw error(ESL_E_NUMERIC, "the solve did not reach the tolerance: relative residual " + sci(kr.resid) +
										   " after " + std::to_string(kr.iters) + " iterations");
	}
	else
	{
		// device-wide solver on the set-minor layout, at most 1024 sets at a time
		nbr_store_t local;
		if (!prebuilt)
			build_nbr(c, S, local);
		const nbr_store_t& nb = prebuilt ? *prebuilt : local;
		const bool ilu = opts.preconditioner != 1;
		const int nseg1 = std::max(n_seg, 1);
		std::vector<double> res_all;
		dbuf<double> d_res;
		for (int b0 = 0; b0 < B; b0 += 1024)
		{
			const int cb = std::min(1024, B - b0);
			sys_t Sc = S;
			Sc.B = cb;
			Sc.rates = S.rates + (int64_t)b0 * S.rate_stride;
			Sc.anchor = S.anchor + (int64_t)b0 * nseg1;
			Sc.invd = S.invd + (int64_t)b0 * nU;
			const double* rhs_c = rhs_p + (int64_t)b0 * nU;
			double* z_c = z_p + (int64_t)b0 * nU;
			bool done = false;
			int it = 0, cy = 0;
			std::vector<double> cres;
			double cmax = 0.0;
			const bool reduced = path == path_reduced && opts.preconditioner == 0;
			if (reduced)
			{
				rbw_ws_t ws(c);
				bicg_w_t gm(c, Sc, nb, ws, nseg1);
				rb_setup_t su = setup ? *setup : rb_setup_t{};
				if (su.n_seg)
					su.anchor += (int64_t)b0 * nseg1;
				if (su.warm)
					su.warm += (int64_t)b0 * su.n_t;
				if (su.x0)
					gm.enter(su);
				else
				{
					gm.enter(rhs_c, z_c);
					gm.movable(su);
				}
				done = gm.solve(tol, max_iters);
				const bool anew = su.x0 || gm.moved; // anchors, and what goes with them, are the solver's
				if (anew)
					k_rhs<<<dim3(ceil_div(nU, sblock), cb), sblock, 0, c.stream>>>(Sc, nseg1, su.x0,
																				   su.rhs + (int64_t)b0 * nU);
				gm.leave(z_c, anew ? su.invd + (int64_t)b0 * nU : nullptr);
				cres = std::move(gm.h_res);
				cmax = gm.final_res;
				it = gm.iters;
				cy = gm.cycles;
			}
			const int it_r = it; // products of the reduced solver: GMRES has max_iters beside them
			if (reduced && !done)
			{
				d_res.ensure(cb);
				write_dev(c, d_res.get(), cres);
				k_rb_restart<<<dim3(ceil_div(nU, sblock), cb), sblock, 0, c.stream>>>(
					Sc, nseg1, d_res.get(), tol, z_c, setup ? setup->invd + (int64_t)b0 * nU : nullptr);
				ESL_HIP(hipStreamSynchronize(c.stream));
			}
			if (!done && opts.precision == 1)
			{
				gmres_w_t<float> gm(c, Sc, nb, nseg1, dw_restart(opts.restart, nU, cb), ilu);
				gm.enter(rhs_c, z_c);
				done = gm.solve(tol, max_iters, opts.inner_rtol);
				gm.leave(z_c);
				cres = gm.h_res; // the residuals of its last check
				cmax = gm.final_res;
				it += gm.iters;
				cy += gm.cycles;
				if (!done)
					kr.fp64_fallback += cb;
			}
			if (!done)
			{
				// FP64 from the current iterate (also what an FP32 solve that stalled falls back to)
				gmres_w_t<double> gm(c, Sc, nb, nseg1, dw_restart(opts.restart, nU, cb), ilu);
				gm.enter(rhs_c, z_c);
				const bool done64 = gm.solve(tol, std::max(max_iters - (it - it_r), 1));
				gm.leave(z_c);
				cres = gm.h_res;
				cmax = gm.final_res;
				it += gm.iters;
				cy += gm.cycles;
				if (!done64)
				{
					if (throw_on_miss)
						throw error(ESL_E_NUMERIC, "the solve did not reach the tolerance: relative residual " +
													   sci(cmax) + " after " + std::to_string(it) + " iterations");
					kr.missed += cb; // an upper bound: the caller reads every set's residual
				}
			}
			res_all.insert(res_all.end(), cres.begin(), cres.end());
			kr.resid = std::max(kr.resid, cmax);
			kr.iters = std::max(kr.iters, it);
			kr.cycles = std::max(kr.cycles, cy);
			kr.sets_iterated += cy > 0 ? cb : 0;
			kr.iters_sum += (int64_t)it * cb; // the sets of a chunk iterate together
		}
		if (set_res)
			*set_res = std::move(res_all);
		ESL_HIP(hipGetLastError());
	}
	return kr;
}

} // namespace

// ---- plan: the rate-independent part of a solve -----------------------------

void plan_build(ctx_t& c, graph_t& g, const double* d_x0, plan_t& P)
{
	if (!g.reorganized)
		throw error(ESL_E_STATE, "esl_graph_reorganize must run before a solve");
	const int N = g.N;
	const int64_t n = g.n;
	const int64_t T = g.T;
	const int64_t n_t = g.n_t;
	const int nb = ceil_div(n, sblock);
	timer_t tm_(c);
	P.g = &g;
	P.x0.ensure(n);
	ESL_HIP(hipMemcpyAsync(P.x0.get(), d_x0, n * sizeof(double), hipMemcpyDeviceToDevice, c.stream));

	// ---- reachability from supp(x0)
	P.reach.ensure(n);
	k_reach_init<<<nb, sblock, 0, c.stream>>>(n, P.x0.get(), P.reach.get());
	int hint = 4;
	fixpoint(c, hint, 8, 1 << 24, "reachability", [&](int32_t* f, const int32_t* pf) {
		ESL_HMAX_DISPATCH(N, k_reach, <<<nb, sblock, 0, c.stream>>>(N, n, g.mask.get(), P.reach.get(), f, pf));
	});
	tm_.mark();

	// ---- reachable terminal SCCs, compact index j, segments of size >= 2
	dbuf<int32_t> reached;
	reached.ensure(std::max<int64_t>(T, 1));
	ESL_HIP(hipMemsetAsync(reached.get(), 0, T * sizeof(int32_t), c.stream));
	if (n_t)
		k_term_reached<<<ceil_div(n_t, sblock), sblock, 0, c.stream>>>(n_t, g.reordered.get(), g.rank.get(),
																		 P.reach.get(), reached.get());
	// with few terminal states their order comes along, in the same wait (plan of 32,768
	// terminal states 463 us with, 483 without; 64,512: 587 and 576, most are not needed)
	std::vector<int32_t> h_reached, h_reord;
	readback_t rd(c);
	rd.add(h_reached, reached.get(), (size_t)T);
	if (n_t <= 16384)
		rd.add(h_reord, g.reordered.get(), (size_t)n_t);
	rd.wait();
	P.jmap.assign(T, -1);
	P.segmap.assign(T, -1);
	P.seg_off.assign(1, 0);
	P.seg_src.clear();
	P.Tr = 0;
	P.n_seg = 0;
	for (int64_t k = 0; k < T; ++k)
	{
		if (!h_reached[k])
			continue;
		P.jmap[k] = P.Tr++;
		const int32_t sz = g.h_offsets[k + 1] - g.h_offsets[k];
		if (sz >= 2)
		{
			P.segmap[k] = P.n_seg++;
			P.seg_off.push_back(P.seg_off.back() + sz);
			P.seg_src.push_back(g.h_offsets[k]);
		}
	}
	P.fallback = P.Tr > max_rhs_terms;
	P.d_jmap.ensure(std::max<int64_t>(T, 1));
	P.d_segmap.ensure(std::max<int64_t>(T, 1));
	write_dev(c, P.d_jmap.get(), P.jmap);
	write_dev(c, P.d_segmap.get(), P.segmap);

	// ---- terminal masks and ambiguous set
	P.tmask.ensure(n);
	k_tm_init<<<nb, sblock, 0, c.stream>>>(n, g.rank.get(), T, P.d_jmap.get(), P.reach.get(), P.tmask.get());
	if (!P.fallback && P.Tr > 1)
		propagate_masks(c, g, P.reach.get(), P.tmask.get());
	P.amb.ensure(n);
	dbuf<int32_t> fpos;
	fpos.ensure(n + 1);
	int32_t nA = 0;
	if (P.Tr > 1)
	{
		k_amb_flag<<<nb, sblock, 0, c.stream>>>(n, g.rank.get(), T, P.reach.get(), P.tmask.get(), P.fallback ? 1 : 0,
												P.amb.get());
		exclusive_scan_i32(c, P.amb.get(), fpos.get(), n);
		std::vector<int32_t> h_nA;
		read_host(c, h_nA, fpos.get() + n, 1);
		nA = h_nA[0];
	}
	else
		ESL_HIP(hipMemsetAsync(P.amb.get(), 0, n * sizeof(int32_t), c.stream));
	P.nA = nA;
	tm_.mark();

	// ---- unknowns: terminal segments (canonical order) then ambiguous states
	P.nUt = P.seg_off.back();
	P.nU = P.nUt + nA;
	P.pos.ensure(n);
	P.ulist.ensure(P.nU + 1);
	P.ucls.ensure(P.nU + 1);
	P.d_seg_off.ensure(P.seg_off.size());
	ESL_HIP(hipMemsetAsync(P.pos.get(), 0xff, n * sizeof(int32_t), c.stream));
	write_dev(c, P.d_seg_off.get(), P.seg_off);
	// what is copied to the device stays until the wait at the end
	std::vector<int32_t> states, seg_of, tpos, s_u;
	std::vector<uint8_t> s_r;
	std::vector<double> h_y0;
	dbuf<int32_t> d_states, d_segof;
	if (P.nUt)
	{
		if (n_t > 16384)
			read_host(c, h_reord, g.reordered.get(), (size_t)n_t);
		states.resize(P.nUt), seg_of.resize(P.nUt), tpos.resize(P.nUt);
		for (int k = 0; k < P.n_seg; ++k)
			for (int32_t q = 0; q < P.seg_off[k + 1] - P.seg_off[k]; ++q)
			{
				states[P.seg_off[k] + q] = h_reord[P.seg_src[k] + q];
				seg_of[P.seg_off[k] + q] = k;
				tpos[P.seg_off[k] + q] = P.seg_src[k] + q;
			}
		P.d_tpos.ensure(P.nUt);
		write_dev(c, P.d_tpos.get(), tpos);
		d_states.ensure(P.nUt);
		d_segof.ensure(P.nUt);
		write_dev(c, d_states.get(), states);
		write_dev(c, d_segof.get(), seg_of);
		k_fill_term_unknowns<<<ceil_div(P.nUt, sblock), sblock, 0, c.stream>>>(
			P.nUt, d_states.get(), d_segof.get(), P.ulist.get(), P.ucls.get(), P.pos.get());
	}
	if (nA)
		k_fill_unknowns<<<nb, sblock, 0, c.stream>>>(n, P.amb.get(), fpos.get(), P.nUt, P.ulist.get(), P.ucls.get(),
													 P.pos.get());

	// ---- x0 mass needing no solve, summed on the host in state order
	P.y0.ensure(std::max(P.Tr, 1));
	if (P.Tr)
	{
		// the states with such mass, packed in state order: 32,768 of a million with five of
		// 20 nodes fixed, and 12 MB to the host otherwise (3.6 of 10.5 ms of such a model)
		dbuf<int32_t> tgt, has, at, mj;
		dbuf<double> mx;
		tgt.ensure(n);
		has.ensure(n);
		at.ensure(n + 1);
		k_target_of<<<nb, sblock, 0, c.stream>>>(n, g.rank.get(), T, P.d_jmap.get(), P.reach.get(), P.tmask.get(),
												  P.amb.get(), P.x0.get(), P.Tr, tgt.get(), has.get());
		exclusive_scan_i32(c, has.get(), at.get(), n);
		std::vector<int32_t> h_count, h_j;
		std::vector<double> h_x;
		// few states: packed into arrays for all of them, read with their number in one wait
		// (plan of 10 nodes 430 us so, 507 with a wait for the number; 13 nodes 444 and 506, 17
		// nodes 937 and 903, 20 nodes 1,358 and 576)
		const bool few = n <= 8192;
		int64_t count = n;
		if (!few)
		{
			read_host(c, h_count, at.get() + n, 1);
			count = h_count[0];
		}
		mj.ensure(std::max<int64_t>(count, 1));
		mx.ensure(std::max<int64_t>(count, 1));
		k_target_pack<<<nb, sblock, 0, c.stream>>>(n, tgt.get(), at.get(), P.x0.get(), mj.get(), mx.get());
		ESL_HIP(hipGetLastError());
		if (few)
			rd.add(h_count, at.get() + n, 1);
		rd.add(h_j, mj.get(), (size_t)count);
		rd.add(h_x, mx.get(), (size_t)count);
		rd.wait();
		count = h_count[0];
		h_y0.assign(P.Tr, 0.0);
		for (int64_t i = 0; i < count; ++i)
			h_y0[h_j[i]] += h_x[i];
		write_dev(c, P.y0.get(), h_y0);
	}
	// ---- exit edges of the ambiguous set, by target terminal SCC
	P.ex_off.assign(std::max(P.Tr, 0) + 1, 0);
	P.n_exit = 0;
	if (P.Tr && nA)
	{
		sys_t S = P.sys(1, nullptr);
		const int gA = ceil_div(nA, sblock);
		dbuf<int32_t> cnt, ptr;
		cnt.ensure(nA);
		ptr.ensure(nA + 1);
		k_exit_count<<<gA, sblock, 0, c.stream>>>(S, g.rank.get(), T, P.d_jmap.get(), P.tmask.get(), cnt.get());
		exclusive_scan_i32(c, cnt.get(), ptr.get(), nA);
		std::vector<int32_t> h_E;
		read_host(c, h_E, ptr.get() + nA, 1);
		const int32_t E = h_E[0];
		dbuf<int32_t> ej, eu;
		dbuf<uint8_t> er;
		ej.ensure(std::max(E, 1));
		eu.ensure(std::max(E, 1));
		er.ensure(std::max(E, 1));
		k_exit_fill<<<gA, sblock, 0, c.stream>>>(S, g.rank.get(), T, P.d_jmap.get(), P.tmask.get(), ptr.get(),
												 ej.get(), eu.get(), er.get());
		ESL_HIP(hipGetLastError());
		std::vector<int32_t> h_j, h_u;
		std::vector<uint8_t> h_r;
		rd.add(h_j, ej.get(), (size_t)E);
		rd.add(h_u, eu.get(), (size_t)E);
		rd.add(h_r, er.get(), (size_t)E);
		rd.wait();
		// stable counting sort by target
		for (int32_t e = 0; e < E; ++e)
		{
			if (h_j[e] < 0 || h_j[e] >= P.Tr)
				throw error(ESL_E_DEVICE, "exit edge with a target outside the reached terminal SCCs");
			P.ex_off[h_j[e] + 1]++;
		}
		for (int j = 0; j < P.Tr; ++j)
			P.ex_off[j + 1] += P.ex_off[j];
		std::vector<int32_t> fill(P.ex_off.begin(), P.ex_off.end() - 1);
		s_u.resize(E), s_r.resize(E);
		for (int32_t e = 0; e < E; ++e)
		{
			const int32_t at = fill[h_j[e]]++;
			s_u[at] = h_u[e];
			s_r[at] = h_r[e];
		}
		P.ex_u.ensure(std::max(E, 1));
		P.ex_r.ensure(std::max(E, 1));
		P.d_ex_off.ensure(P.Tr + 1);
		write_dev(c, P.ex_u.get(), s_u);
		write_dev(c, P.ex_r.get(), s_r);
		write_dev(c, P.d_ex_off.get(), P.ex_off);
		P.n_exit = E;
	}
	// ---- coupling structure of the per-set solver
	P.nbr.ready = false;
	P.anchor_lds = 0;
	P.anchor_lvl = 0;
	if (P.nU)
	{
		sys_t S = P.sys(1, nullptr);
		build_nbr(c, S, P.nbr);
		if (P.nUt > 0 && P.nUt <= 4096)
		{
			const size_t bytes = 24 * (size_t)P.nUt + 4 * (size_t)(P.nUt + 1) + 3 * (size_t)P.nbr.nnz_t + 16;
			const size_t static_bytes = 64 * 8 + sblock * 12 + 256;
			if (bytes + static_bytes <= (size_t)std::min(c.lds_per_block, 160 * 1024))
			{
				P.anchor_lds = bytes;
				if (bytes > 48 * 1024)
					ESL_HIP(hipFuncSetAttribute((const void*)k_anchor_lds, hipFuncAttributeMaxDynamicSharedMemorySize,
												(int)bytes));
			}
		}
		// with the solver's packed records: headers, records and two FP32 mass vectors
		if (P.nbr.packed && P.n_seg > 0)
		{
			const size_t bytes = 12 * (size_t)P.nU + 4 * ((size_t)P.nbr.nnz + 4) + 16;
			if (bytes + 1024 <= (size_t)std::min(c.lds_per_block, 160 * 1024))
			{
				P.anchor_lvl = bytes;
				if (bytes > 48 * 1024)
					for (const void* f : { (const void*)k_anchor_lvl<4>, (const void*)k_anchor_lvl<8> })
						ESL_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
			}
		}
	}
	tm_.mark();
	tm_.read(P.ms);
}

sys_t plan_t::sys(int B, const double* rates) const
{
	sys_t S{};
	S.N = g->N;
	S.nU = nU;
	S.nUt = nUt;
	S.B = B;
	S.mask = g->mask.get();
	S.ulist = ulist.get();
	S.ucls = ucls.get();
	S.pos = pos.get();
	S.rates = rates;
	S.rate_stride = 2 * g->N;
	S.transpose = 0;
	S.anchor = rb.anchor;
	S.invd = rb.invd;
	return S;
}

// whether a per-set run of the plan takes the reduced solver
bool plan_reduced(const ctx_t& c, const plan_t& P, int B, const esl_solve_opts& o)
{
	sys_t S{};
	S.nU = P.nU;
	S.B = B;
	return P.nU > 0 && reduced_variant(c, S, P.nbr, o, P.path) != nullptr;
}

// The numeric part for B rate sets: anchors, coefficients and start vector
// (setup), the Krylov solves, then absorption masses and the final vector
// (post).  No host synchronisation inside, so with the per-set solver the whole
// sequence can be captured into a HIP graph; results are checked afterwards.
void plan_enqueue_setup(ctx_t& c, plan_t& P, int B, const double* d_rates, const esl_solve_opts& o)
{
	const int64_t n_t = P.g->n_t;
	const int64_t nU = P.nU, nUt = P.nUt;
	const int n_seg = P.n_seg, nseg1 = std::max(n_seg, 1);
	sys_t S = P.sys(B, d_rates);
	const bool warm = o.warm_pi != nullptr && n_seg > 0;
	if (n_seg)
	{
		const dim3 gt(ceil_div(nUt, sblock), B);
		if (warm)
			// the prediction picks the anchors (no Jacobi sweeps)
			k_warm_gather<<<gt, sblock, 0, c.stream>>>(nUt, n_t, P.d_tpos.get(), o.warm_pi, P.rb.p0);
		else if (P.anchor_lvl)
		{
			// sweeps and pick in one launch on the solver's level-ordered records
			timed_launch(c, "k_anchor_lvl", 8.0 * B * nUt, [&] {
				if (nU <= 4 * pblock)
					k_anchor_lvl<4><<<B, pblock, P.anchor_lvl, c.stream>>>(S, P.nbr.view(), P.d_seg_off.get(), n_seg,
																		   P.anchor_sweeps, P.rb.anchor);
				else
					k_anchor_lvl<8><<<B, pblock, P.anchor_lvl, c.stream>>>(S, P.nbr.view(), P.d_seg_off.get(), n_seg,
																		   P.anchor_sweeps, P.rb.anchor);
			});
		}
		else if (P.anchor_lds)
		{
			// sweeps and pick in one launch, the terminal unknowns in LDS
			timed_launch(c, "k_anchor_lds", 8.0 * B * nUt, [&] {
				k_anchor_lds<<<B, sblock, P.anchor_lds, c.stream>>>(S, P.nbr.ptr.get(), P.nbr.nu.get(),
																	 P.nbr.nr.get(), P.d_seg_off.get(), n_seg,
																	 P.anchor_sweeps, P.rb.anchor);
			});
		}
		else
		{
			k_fill_value<<<ceil_div((int64_t)B * nUt, sblock), sblock, 0, c.stream>>>((int64_t)B * nUt, 1.0,
																					  P.rb.p0);
			double *pa = P.rb.p0, *pb = P.rb.p1;
			for (int it = 0; it < P.anchor_sweeps; ++it)
			{
				timed_launch(c, "k_anchor_sweep", 16.0 * B * nUt, [&] {
					k_anchor_sweep<<<gt, sblock, 0, c.stream>>>(S, P.nbr.view(), pa, pb);
				});
				std::swap(pa, pb);
			}
			if (pa != P.rb.p0)
				std::swap(P.rb.p0, P.rb.p1); // the mass after the last sweep
		}
		if (warm || (!P.anchor_lds && !P.anchor_lvl))
			k_anchor_pick<<<dim3(n_seg, B), sblock, 0, c.stream>>>(nUt, P.d_seg_off.get(), P.rb.p0, n_seg,
																	 P.rb.anchor);
	}
	if (nU)
	{
		const dim3 gu(ceil_div(nU, sblock), B);
		k_sys_setup<<<gu, sblock, 0, c.stream>>>(S, nseg1, P.x0.get(), P.rb.invd, P.rb.rhs, P.rb.z);
		if (warm)
			k_warm_z<<<dim3(ceil_div(nUt, sblock), B), sblock, 0, c.stream>>>(S, n_seg, P.rb.p0, P.rb.z);
	}
	ESL_HIP(hipGetLastError());
}

// the dense final vectors zeroed (algorithmic bytes: written once)
void enqueue_final_fill(ctx_t& c, int B, int64_t n, double* d_final)
{
	timed_launch(c, "k_zero<final>", 8.0 * B * n, [&] {
		const int64_t count = (int64_t)B * n;
		if (count % 2 == 0 && ((uintptr_t)d_final & 15) == 0)
			k_zero2<<<ceil_div(count / 2, sblock), sblock, 0, c.stream>>>(count / 2, (double2*)d_final);
		else
			k_zero<double><<<ceil_div(count, sblock), sblock, 0, c.stream>>>(count, d_final);
	});
}

// clear: the final vectors still have to be zeroed here (false when the fill
// ran on its own stream)
void plan_enqueue_post(ctx_t& c, plan_t& P, int B, const double* d_rates, double* d_final, bool clear = true)
{
	graph_t& g = *P.g;
	const int64_t n = g.n, n_t = g.n_t, T = g.T;
	const int64_t nU = P.nU;
	const int n_seg = P.n_seg, nseg1 = std::max(n_seg, 1), Tr = P.Tr;
	sys_t S = P.sys(B, d_rates);
	if (Tr)
	{
		if (P.nA)
			k_exit_sum<<<dim3(Tr, B), sblock, 0, c.stream>>>(S, P.d_ex_off.get(), P.ex_u.get(), P.ex_r.get(), P.rb.z,
															 Tr, P.rb.y);
		else
			k_zero<double><<<ceil_div((int64_t)B * Tr, sblock), sblock, 0, c.stream>>>((int64_t)B * Tr, P.rb.y);
		k_y_total<<<ceil_div((int64_t)B * Tr, sblock), sblock, 0, c.stream>>>(B, Tr, P.y0.get(), P.rb.y);
	}
	if (n_seg)
		k_seg_sum<<<dim3(n_seg, B), sblock, 0, c.stream>>>(nU, P.d_seg_off.get(), P.rb.z, P.rb.invd, n_seg,
														  P.rb.segsum);
	if (clear)
		enqueue_final_fill(c, B, n, d_final);
	if (n_t && Tr)
		k_final<<<dim3(ceil_div(n_t, sblock), B), sblock, 0, c.stream>>>(
			n, n_t, g.reordered.get(), g.rank.get(), P.d_jmap.get(), P.d_segmap.get(), P.pos.get(), P.rb.z,
			P.rb.invd, P.rb.segsum, nseg1, nU, P.rb.y, Tr, d_final);
	ESL_HIP(hipGetLastError());
}

// fork_fill: the final-vector fill (HBM-write bound) runs on its own stream
// beside the anchor, set-up and solve kernels (LDS and latency bound); the
// final scatter waits for it.  Both slow down while they share HBM, but the
// pair ends sooner than the two in sequence (N=20 bench: 3.19 -> 2.95 ms).
void plan_enqueue(ctx_t& c, plan_t& P, int B, const double* d_rates, double* d_final, const esl_solve_opts& o,
				  bool fork_fill = false)
{
	const bool fork = fork_fill && P.nU > 0;
	if (fork)
	{
		if (!c.fill_s)
		{
			ESL_HIP(hipStreamCreateWithFlags(&c.fill_s, hipStreamNonBlocking));
			for (hipEvent_t& e : c.fill_ev)
				ESL_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
		}
		const hipStream_t main = c.stream;
		ESL_HIP(hipEventRecord(c.fill_ev[0], main));
		ESL_HIP(hipStreamWaitEvent(c.fill_s, c.fill_ev[0], 0));
		c.stream = c.fill_s;
		try
		{
			enqueue_final_fill(c, B, P.g->n, d_final);
		}
		catch (...)
		{
			c.stream = main;
			throw;
		}
		c.stream = main;
		ESL_HIP(hipEventRecord(c.fill_ev[1], c.fill_s));
	}
	rb_setup_t su{};
	if (plan_reduced(c, P, B, o)) // sets itself up
		su = P.setup(o.warm_pi);
	else
		plan_enqueue_setup(c, P, B, d_rates, o);
	if (P.nU)
		launch_per_set(c, P.sys(B, d_rates), P.nbr, P.n_seg, P.rb.rhs, P.rb.z, o, P.rb.ps, P.path, su);
	if (fork)
		ESL_HIP(hipStreamWaitEvent(c.stream, c.fill_ev[1], 0));
	plan_enqueue_post(c, P, B, d_rates, d_final, !fork);
}

void plan_reserve_(plan_t& P, int B, int m, int precision, bool reduced, bool masses);

// The schedule of a run: the tuned one when the caller asks for restart 0, else
// the reduced solver -- unless a restart length asks for GMRES.
int run_path(const plan_t& P, const esl_solve_opts& o)
{
	if (o.restart == 0 && P.tune.set)
		return P.tune.path;
	return o.restart <= 0 ? path_reduced : path_lds;
}

// whether a run is per set (one workgroup per rate set) or device-wide
bool runs_per_set(const plan_t& P, int B, bool tuned)
{
	if (P.nU == 0 || (tuned && P.tune.path != path_wide && P.tune.path != path_reduced))
		return true;
	return !(tuned && P.tune.path == path_wide) && P.nU <= per_set_max_unknowns(B);
}

// grows the per-run buffers; a captured graph holds their addresses, so any
// reallocation bumps the plan's epoch (part of every graph key).  masses: for a run that
// sets up GMRES (the reduced solvers set themselves up)
void plan_reserve(plan_t& P, int B, int m, int precision, bool reduced, bool masses)
{
	auto ptrs = [&] {
		return std::vector<const void*>{ P.p0.get(),	 P.p1.get(),	  P.anchor.get(), P.invd.get(),
										 P.rhs.get(),	 P.z.get(),		  P.y.get(),	  P.segsum.get(),
										 P.scr.r.get(),	  P.scr.udiag.get(), P.scr.res.get(),
										 P.scr.t.get(), P.scr.its.get(), P.scr.cyc.get(), P.scr.stl.get(),
										 P.scr.tspan.get(), P.scr.xk.get(), P.scr.Vf.get(), P.scr.Vd.get() };
	};
	const auto before = ptrs();
	plan_reserve_(P, B, m, precision, reduced, masses);
	if (ptrs() != before)
		++P.epoch;
}

void plan_reserve_(plan_t& P, int B, int m, int precision, bool reduced, bool masses)
{
	const int64_t nU = std::max<int64_t>(P.nU, 1), nUt = std::max<int64_t>(P.nUt, 1);
	if (masses)
	{
		P.p0.ensure((size_t)B * nUt);
		P.p1.ensure((size_t)B * nUt);
	}
	P.anchor.ensure((size_t)B * std::max(P.n_seg, 1));
	P.invd.ensure((size_t)B * nU);
	P.rhs.ensure((size_t)B * nU);
	P.z.ensure((size_t)B * nU);
	P.y.ensure((size_t)B * std::max(P.Tr, 1));
	P.segsum.ensure((size_t)B * std::max(P.n_seg, 1));
	if (m > 0) // 0: the device-wide solvers keep their own buffers
		P.scr.reserve(B, nU, m, precision, reduced);
	P.use_own_bufs();
}

// relative FP64 residual ||rhs - A_p z||_2 / ||rhs||_2 of every set, from the
// mask-based operator (independent of the solvers' coupling structure)
std::vector<double> set_residuals(ctx_t& c, const sys_t& S, int n_seg, const double* rhs, const double* z)
{
	const int B = S.B;
	std::vector<double> out(B, 0.0);
	if (S.nU == 0)
		return out;
	const int nblk = ceil_div(S.nU, sblock);
	dbuf<double> part, rr;
	part.ensure((size_t)B * nblk * 2);
	rr.ensure((size_t)B * 2);
	k_residual<<<dim3(nblk, B), sblock, 0, c.stream>>>(S, std::max(n_seg, 1), rhs, z, nullptr, part.get());
	k_reduce_parts<<<dim3(2, B), wave, 0, c.stream>>>(part.get(), nblk, 2, rr.get(), 2, 0);
	ESL_HIP(hipGetLastError());
	std::vector<double> h;
	read_host(c, h, rr.get(), (size_t)B * 2);
	for (int b = 0; b < B; ++b)
	{
		const double r2 = h[2 * b], b2 = h[2 * b + 1];
		out[b] = b2 > 0 ? std::sqrt(r2 / b2) : (r2 > 0 ? INFINITY : 0.0);
	}
	return out;
}

// the diagonal blocks (first unknown, size) of every set's system: one per
// terminal segment, one for the ambiguous states
std::vector<std::pair<int64_t, int64_t>> plan_blocks(const plan_t& P)
{
	std::vector<std::pair<int64_t, int64_t>> bl;
	for (int k = 0; k < P.n_seg; ++k)
		bl.push_back({ P.seg_off[k], P.seg_off[k + 1] - P.seg_off[k] });
	if (P.nA > 0)
		bl.push_back({ P.nUt, P.nA });
	return bl;
}

// Exact FP64 solve of the systems of `sets` (indices into the batch) by dense
// LU with partial pivoting, block by block, with two steps of iterative
// refinement; z of those sets receives D' x.  Returns false, changing nothing,
// when a block exceeds lu_max_block unknowns.
bool exact_solve_sets(ctx_t& c, plan_t& P, int B, const double* d_rates, const std::vector<int>& sets)
{
	const auto blocks = plan_blocks(P);
	int64_t smax = 0;
	for (auto& bl : blocks)
		smax = std::max(smax, bl.second);
	if (smax == 0 || sets.empty())
		return true;
	if (smax > lu_max_block)
		return false;
	dbuf<double> A, x, r;
	dbuf<int32_t> ipiv, flag;
	A.ensure((size_t)smax * smax);
	x.ensure(smax);
	r.ensure(smax);
	ipiv.ensure(smax);
	flag.ensure(1);
	k_zero<int32_t><<<1, sblock, 0, c.stream>>>(1, flag.get());
	if (smax * (int64_t)sizeof(double) > 48 * 1024)
		ESL_HIP(hipFuncSetAttribute((const void*)k_lu_solve, hipFuncAttributeMaxDynamicSharedMemorySize,
									(int)(smax * sizeof(double))));
	const sys_t S = P.sys(B, d_rates);
	const nbr_t G = P.nbr.view();
	const int nseg1 = std::max(P.n_seg, 1);
	for (int b : sets)
		for (auto& bl : blocks)
		{
			const int64_t u0 = bl.first;
			const int sz = (int)bl.second;
			const int gs = ceil_div(sz, sblock);
			const size_t lds = (size_t)sz * sizeof(double);
			k_zero<double><<<ceil_div((int64_t)sz * sz, sblock), sblock, 0, c.stream>>>((int64_t)sz * sz, A.get());
			k_lu_assemble<<<gs, sblock, 0, c.stream>>>(S, G, nseg1, b, u0, sz, A.get(), P.rb.rhs, x.get(),
													   flag.get());
			for (int j0 = 0; j0 < sz; j0 += lu_nb)
			{
				const int jb = std::min(lu_nb, sz - j0);
				k_lu_panel<<<1, lu_panel_threads, 0, c.stream>>>(A.get(), sz, j0, jb, ipiv.get(), flag.get());
				k_lu_swap<<<gs, sblock, 0, c.stream>>>(A.get(), sz, j0, jb, ipiv.get());
				const int rest = sz - j0 - jb;
				if (rest > 0)
				{
					k_lu_trsm<<<ceil_div(rest, sblock), sblock, 0, c.stream>>>(A.get(), sz, j0, jb);
					const int t = ceil_div(rest, 64);
					k_lu_gemm<<<dim3(t, t), sblock, 0, c.stream>>>(A.get(), sz, j0, jb);
				}
			}
			k_lu_solve<<<1, lu_panel_threads, lds, c.stream>>>(A.get(), sz, ipiv.get(), x.get());
			for (int it = 0; it < 2; ++it) // iterative refinement with the factors
			{
				k_lu_residual<<<gs, sblock, 0, c.stream>>>(S, G, nseg1, b, u0, sz, x.get(), P.rb.rhs, r.get());
				k_lu_solve<<<1, lu_panel_threads, lds, c.stream>>>(A.get(), sz, ipiv.get(), r.get());
				k_lu_axpy<<<gs, sblock, 0, c.stream>>>(sz, r.get(), x.get());
			}
			k_lu_store<<<gs, sblock, 0, c.stream>>>(S, b, u0, sz, x.get(), P.rb.z);
			ESL_HIP(hipGetLastError());
		}
	int32_t h_flag = 0;
	ESL_HIP(hipMemcpyAsync(&h_flag, flag.get(), sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
	ESL_HIP(hipStreamSynchronize(c.stream));
	if (h_flag & 2)
		throw error(ESL_E_DEVICE, "exact solve: a coupling crosses the diagonal blocks of the system");
	if (h_flag & 1)
		throw error(ESL_E_NUMERIC, "exact solve: a system matrix is singular");
	return true;
}

// After the Krylov solves of a run: sets above the tolerance (every set when
// exact_fallback is 2) are solved by the exact dense LU when allow_lu and their
// blocks fit, the final vectors are rebuilt when a set changed (or `rebuild`),
// and the per-set outcome is stored in the plan.  A set still above the
// tolerance fails the call with ESL_E_NUMERIC, after every set's final vector
// has been written.
void plan_finish_sets(ctx_t& c, plan_t& P, int B, const double* d_rates, double* d_final, const esl_solve_opts& o,
					  krylov_result_t& kr, set_results_t sr, bool rebuild, bool allow_lu)
{
	std::vector<int> todo;
	if (P.nU > 0 && o.exact_fallback >= 1)
		for (int b = 0; b < B; ++b)
			if (o.exact_fallback == 2 || !(sr.res[b] <= o.tol))
				todo.push_back(b);
	bool fits = true;
	if (!todo.empty() && allow_lu)
	{
		fits = exact_solve_sets(c, P, B, d_rates, todo);
		if (fits)
		{
			const auto res = set_residuals(c, P.sys(B, d_rates), P.n_seg, P.rb.rhs, P.rb.z);
			for (int b : todo)
			{
				sr.res[b] = res[b];
				sr.method[b] = 2;
			}
			kr.exact = (int)todo.size();
			rebuild = true;
		}
	}
	if (rebuild)
	{
		plan_enqueue_post(c, P, B, d_rates, d_final);
		ESL_HIP(hipStreamSynchronize(c.stream));
	}
	int missed = 0;
	double worst = 0.0;
	for (int b = 0; b < B; ++b)
	{
		worst = std::max(worst, std::isnan(sr.res[b]) ? 1e300 : sr.res[b]);
		if (!(sr.res[b] <= o.tol))
		{
			sr.method[b] = -1;
			++missed;
		}
	}
	kr.resid = worst;
	kr.missed = missed;
	P.results = std::move(sr);
	if (missed)
	{
		std::string why;
		if (o.exact_fallback < 1)
			why = " (exact fallback off)";
		else if (!allow_lu)
			why = " (no exact fallback in this entry point)";
		else if (!fits)
			why = " (a system block exceeds the exact solver's " + std::to_string(lu_max_block) + " unknowns)";
		throw error(ESL_E_NUMERIC, std::to_string(missed) + " of " + std::to_string(B) +
									   " rate sets missed the tolerance " + sci(o.tol) + ": worst relative residual " +
									   sci(worst) + why);
	}
}

// per-set outcome when there is nothing to solve
set_results_t trivial_results(int B)
{
	set_results_t sr;
	sr.res.assign(B, 0.0);
	sr.its.assign(B, 0);
	sr.method.assign(B, 0);
	return sr;
}

void plan_run(ctx_t& c, plan_t& P, int B, const double* d_rates, double* d_final, const esl_solve_opts& o_in,
			  esl_solve_report& rep)
{
	esl_solve_opts o = o_in;
	if (o.tol <= 0)
		o.tol = 1e-13;
	if (o.max_iters <= 0)
		o.max_iters = 20000;
	// host wall time of the call (the stream is idle at its end); device events
	// would add their creation and one more host round trip to every solve
	const auto t_start = std::chrono::steady_clock::now();
	const bool tuned = o.restart == 0 && P.tune.set;
	if (tuned && P.tune.path != path_reduced)
		o.restart = P.tune.m;
	P.path = run_path(P, o_in);
	const int m = std::min(std::max(o.restart > 0 ? o.restart : 32, 2), pm_max);
	const bool per_set = runs_per_set(P, B, tuned);
	rep.terminals_reached = P.Tr;
	rep.unknowns = P.nU;
	rep.reachable = -1;
	krylov_result_t kr;
	if (per_set)
	{
		const bool reduced = plan_reduced(c, P, B, o);
		plan_reserve(P, B, m, o.precision, reduced, !reduced);
		const bool use_graph = o.graph != 0;
		if (use_graph)
		{
			const plan_t::gkey_t key{ B,		   d_rates,	  d_final,	   o.warm_pi,  o.precision,
									  o.preconditioner, m,		  o.tol,	   o.inner_rtol, o.max_iters,
									  P.epoch,		   P.path };
			if (!P.gexec || !(P.gkey == key) || P.gprof != c.prof.on)
			{
				P.drop_graph();
				hipGraph_t graph;
				if (c.prof.on)
				{
					// timing events become nodes of the graph; booked after every replay
					ESL_HIP(hipStreamSynchronize(c.stream));
					c.prof.flush();
					c.prof.capture_events = &P.gev;
					c.prof.capture_pending = &P.gpend;
				}
				ESL_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
				try
				{
					plan_enqueue(c, P, B, d_rates, d_final, o, true);
				}
				catch (...)
				{
					(void)hipStreamEndCapture(c.stream, &graph);
					c.prof.capture_events = nullptr;
					c.prof.capture_pending = nullptr;
					throw;
				}
				c.prof.capture_events = nullptr;
				c.prof.capture_pending = nullptr;
				ESL_HIP(hipStreamEndCapture(c.stream, &graph));
				ESL_HIP(hipGraphInstantiate(&P.gexec, graph, nullptr, nullptr, 0));
				(void)hipGraphDestroy(graph);
				P.gkey = key;
				P.gprof = c.prof.on;
			}
			ESL_HIP(hipGraphLaunch(P.gexec, c.stream));
		}
		else
			plan_enqueue(c, P, B, d_rates, d_final, o, true);
		// the per-set outputs follow the launch on the stream: one wait for both
		const bool staged = P.nU > 0 && stage_set_outputs(c, P.rb.ps, B);
		ESL_HIP(hipStreamSynchronize(c.stream));
		if (use_graph && c.prof.on)
			c.prof.book(P.gpend);
		if (P.nU > 0)
		{
			esl_solve_opts of = o;
			of.restart = m;
			set_results_t sr;
			kr = finish_per_set(c, P.sys(B, d_rates), P.nbr, P.n_seg, P.rb.rhs, P.rb.z, of, P.rb.ps, reduced, P.setup(nullptr), [&](int prec) {
				plan_reserve(P, B, m, prec, false, false); // captured graphs are told of a basis that moved
				return P.rb.ps;
			}, &sr, staged);
			// the final vectors are rebuilt when a second launch finished sets
			plan_finish_sets(c, P, B, d_rates, d_final, of, kr, std::move(sr), kr.finished > 0, true);
		}
		else
			P.results = trivial_results(B);
	}
	else
	{
		// one large system: device-wide, driven from the host
		const bool reduced = P.path == path_reduced && o.preconditioner == 0;
		plan_reserve(P, B, 0, 0, reduced, !reduced);
		const rb_setup_t su = P.setup(o.warm_pi);
		if (!reduced)
			plan_enqueue_setup(c, P, B, d_rates, o);
		set_results_t sr;
		kr = krylov_solve(c, P.sys(B, d_rates), P.n_seg, P.rb.rhs, P.rb.z, o, &P.nbr, true, false, &sr.res, P.path,
						  reduced ? &su : nullptr);
		plan_enqueue_post(c, P, B, d_rates, d_final);
		if ((int)sr.res.size() != B)
			sr.res = set_residuals(c, P.sys(B, d_rates), P.n_seg, P.rb.rhs, P.rb.z);
		sr.its.assign(B, kr.iters);
		sr.method.assign(B, kr.fp64_fallback ? 1 : 0);
		plan_finish_sets(c, P, B, d_rates, d_final, o, kr, std::move(sr), false, true);
	}
	rep.residual = kr.resid;
	rep.iterations = kr.iters;
	rep.refinements = kr.cycles;
	rep.sets_iterated = kr.sets_iterated;
	rep.fp64_fallback = kr.fp64_fallback;
	rep.iterations_sum = kr.iters_sum;
	rep.exact_solves = kr.exact;
	ESL_HIP(hipStreamSynchronize(c.stream));
	rep.ms_stage[3] = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
	rep.ms_total = rep.ms_stage[3];
}

void solve_run(ctx_t& c, graph_t& g, const solve_args_t& a, esl_solve_report& rep)
{
	plan_t P;
	plan_build(c, g, a.d_x0, P);
	rep.ms_stage[0] = P.ms[0];
	rep.ms_stage[1] = P.ms[1];
	rep.ms_stage[2] = P.ms[2];
	plan_run(c, P, a.n_sets, a.d_rates, a.d_final, a.opts, rep);
	rep.ms_total = P.ms[0] + P.ms[1] + P.ms[2] + rep.ms_stage[3];
}

// ---- opaque plan handles for the C ABI
void* plan_create(ctx_t& c, graph_t& g, const double* d_x0)
{
	auto P = std::make_unique<plan_t>();
	plan_build(c, g, d_x0, *P);
	return P.release();
}

void plan_destroy(void* p) { delete static_cast<plan_t*>(p); }

void plan_solve(ctx_t& c, void* p, int B, const double* d_rates, double* d_final, const esl_solve_opts& o,
				esl_solve_report& rep)
{
	plan_run(c, *static_cast<plan_t*>(p), B, d_rates, d_final, o, rep);
}

// ---- the solve that allocates nothing: every per-run buffer of a plan is a
// slice of one static device array.  Each GPU the library runs on holds its own
// copy of the array until the process ends; calls on one GPU share it (and
// race when they overlap), and each call rewrites what it reads.

static __device__ __align__(256) unsigned char scratch[noalloc_scratch_bytes];

namespace {
std::mutex noalloc_mu;
void* noalloc_dev_ptr[max_devices] = {}; // device address of `scratch`, per device
} // namespace

void noalloc_init(ctx_t& c)
{
	std::lock_guard<std::mutex> lk(noalloc_mu);
	if (c.device < 0 || c.device >= max_devices)
		throw error(ESL_E_ARG, "device index " + std::to_string(c.device) + " is beyond the library's table");
	if (!noalloc_dev_ptr[c.device])
	{
		void* ptr = nullptr;
		ESL_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch))); // the calling thread has c.device current
		noalloc_dev_ptr[c.device] = ptr;
	}
	c.noalloc_scratch = noalloc_dev_ptr[c.device];
}

namespace {
// bump allocator over [base, base + cap): 256-byte aligned slices
struct carve_t
{
	uintptr_t base, at;
	template <typename T>
	T* take(size_t count)
	{
		at = (at + 255) & ~(uintptr_t)255;
		T* p = reinterpret_cast<T*>(at);
		at += std::max<size_t>(count, 1) * sizeof(T);
		return p;
	}
	size_t used() const { return (size_t)(at - base); }
};

// the per-run buffers of B sets at restart m; the basis is sized for FP64
// (precision 1 keeps its FP32 basis in the same slice and reuses it for the
// FP64 finish of stalled sets)
plan_t::run_bufs_t carve_run_bufs(const plan_t& P, int B, int m, carve_t& cv)
{
	const size_t nU = (size_t)std::max<int64_t>(P.nU, 1), nUt = (size_t)std::max<int64_t>(P.nUt, 1);
	const size_t nseg = (size_t)std::max(P.n_seg, 1), Tr = (size_t)std::max(P.Tr, 1);
	plan_t::run_bufs_t rb;
	rb.p0 = cv.take<double>(B * nUt);
	rb.p1 = cv.take<double>(B * nUt);
	rb.anchor = cv.take<int32_t>(B * nseg);
	rb.invd = cv.take<double>(B * nU);
	rb.rhs = cv.take<double>(B * nU);
	rb.z = cv.take<double>(B * nU);
	rb.y = cv.take<double>(B * Tr);
	rb.segsum = cv.take<double>(B * nseg);
	rb.ps.r = cv.take<double>(B * nU);
	rb.ps.udiag = cv.take<double>(B * nU);
	rb.ps.t = cv.take<double>(B * nU);
	rb.ps.res = cv.take<double>(B);
	rb.ps.its = cv.take<int32_t>(B);
	rb.ps.cyc = cv.take<int32_t>(B);
	rb.ps.stl = cv.take<int32_t>(B);
	rb.ps.tspan = cv.take<uint64_t>((size_t)2 * B);
	rb.ps.Vd = cv.take<double>((size_t)B * (m + 1) * nU);
	rb.ps.Vf = reinterpret_cast<float*>(rb.ps.Vd);
	rb.ps.xk = rb.ps.Vd; // the reduced solver keeps no basis
	return rb;
}

// profiling off for the call (its event pool would grow), restored on exit
struct prof_pause_t
{
	ctx_t& c;
	bool was;
	explicit prof_pause_t(ctx_t& x) : c(x), was(x.prof.on) { c.prof.on = false; }
	~prof_pause_t() { c.prof.on = was; }
};
} // namespace

void plan_solve_noalloc(ctx_t& c, void* p, int B, const double* d_rates, double* d_final, const esl_solve_opts& o_in,
						esl_solve_report& rep)
{
	plan_t& P = *static_cast<plan_t*>(p);
	if (!c.noalloc_scratch)
		throw error(ESL_E_STATE, "the static scratch of this context's device was not set up");
	esl_solve_opts o = o_in;
	if (o.tol <= 0)
		o.tol = 1e-13;
	if (o.max_iters <= 0)
		o.max_iters = 20000;
	const bool tuned = o.restart == 0 && P.tune.set;
	if (tuned && P.tune.path != path_reduced)
		o.restart = P.tune.m;
	const int m = std::min(std::max(o.restart > 0 ? o.restart : 32, 2), pm_max);
	o.restart = m;
	const bool per_set = runs_per_set(P, B, tuned);
	if (!per_set)
		throw error(ESL_E_ARG, "the no-allocation solve runs the per-set solvers only; this plan's system (" +
								   std::to_string(P.nU) + " unknowns per set) needs the device-wide solver");
	carve_t dry{ 0, 0 };
	(void)carve_run_bufs(P, B, m, dry);
	if (dry.used() > noalloc_scratch_bytes)
		throw error(ESL_E_ARG, std::to_string(B) + " rate sets of this plan at restart " + std::to_string(m) +
								   " need " + std::to_string(dry.used()) + " bytes of scratch; the static scratch holds " +
								   std::to_string(noalloc_scratch_bytes) + " (use fewer sets per call)");
	const uintptr_t base = reinterpret_cast<uintptr_t>(c.noalloc_scratch);
	carve_t cv{ base, base };
	prof_pause_t pause(c);
	P.rb = carve_run_bufs(P, B, m, cv);
	P.path = run_path(P, o_in);
	rep.terminals_reached = P.Tr;
	rep.unknowns = P.nU;
	rep.reachable = -1;
	krylov_result_t kr;
	try
	{
		ESL_HIP(hipEventRecord(c.ev[0], c.stream));
		plan_enqueue(c, P, B, d_rates, d_final, o, false);
		if (P.nU > 0)
		{
			const pss_view_t ps = P.rb.ps;
			set_results_t sr;
			kr = finish_per_set(c, P.sys(B, d_rates), P.nbr, P.n_seg, P.rb.rhs, P.rb.z, o, ps,
								plan_reduced(c, P, B, o), P.setup(nullptr), [&](int) { return ps; }, &sr);
			// no exact fallback here (its dense matrix would need an allocation)
			plan_finish_sets(c, P, B, d_rates, d_final, o, kr, std::move(sr), kr.finished > 0, false);
		}
		else
			P.results = trivial_results(B);
		ESL_HIP(hipEventRecord(c.ev[1], c.stream));
		ESL_HIP(hipEventSynchronize(c.ev[1]));
		float ms = 0;
		ESL_HIP(hipEventElapsedTime(&ms, c.ev[0], c.ev[1]));
		rep.ms_stage[3] = rep.ms_total = ms;
	}
	catch (...)
	{
		P.use_own_bufs();
		throw;
	}
	P.use_own_bufs(); // pointers only: later runs of the plan use its own buffers again
	rep.residual = kr.resid;
	rep.iterations = kr.iters;
	rep.refinements = kr.cycles;
	rep.sets_iterated = kr.sets_iterated;
	rep.fp64_fallback = kr.fp64_fallback;
	rep.iterations_sum = kr.iters_sum;
}

// ---- several plans (distinct networks) in one call: their per-set solves run
// concurrently on forked streams, optionally captured as one HIP graph
struct multi_graph_t
{
	std::vector<uint64_t> plans; // plan_t::id: an address may name another plan later
	std::vector<int> B;
	std::vector<const double*> rates;
	std::vector<double*> fin;
	std::vector<int64_t> epochs;
	std::vector<int> ms, paths;
	int precision = 0, preconditioner = 0, max_iters = 0;
	double tol = 0, inner_rtol = 0;
	bool prof = false;
	hipGraphExec_t exec = nullptr;
	std::vector<hipEvent_t> gev;
	std::vector<prof_t::pending_t> gpend;
	bool same(const multi_graph_t& o) const
	{
		return plans == o.plans && B == o.B && rates == o.rates && fin == o.fin && epochs == o.epochs &&
			   ms == o.ms && paths == o.paths && precision == o.precision && preconditioner == o.preconditioner &&
			   max_iters == o.max_iters && tol == o.tol &&
			   inner_rtol == o.inner_rtol && prof == o.prof;
	}
	~multi_graph_t()
	{
		if (exec)
			(void)hipGraphExecDestroy(exec);
		for (auto e : gev)
			(void)hipEventDestroy(e);
	}
};

void multi_graph_free(void* p) { delete static_cast<multi_graph_t*>(p); }

void ensure_aux(ctx_t& c, int n)
{
	while ((int)c.aux.size() < n)
	{
		hipStream_t s;
		ESL_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
		c.aux.push_back(s);
	}
	while ((int)c.aux_ev.size() < n + 1)
	{
		hipEvent_t e;
		ESL_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
		c.aux_ev.push_back(e);
	}
}

void many_per_set(ctx_t& c, const std::vector<int>& conc, void* const* plans, const int* B,
				  const double* const* d_rates, double* const* d_final, const esl_solve_opts& o,
				  std::vector<esl_solve_opts>& po, esl_solve_report* reps);

// A context of its own (stream, events, flags; profiling off) for a host thread
// that drives one device-wide solve while the calling thread drives the rest.
struct child_ctx_t
{
	ctx_t c;
	explicit child_ctx_t(const ctx_t& parent)
	{
		c.device = parent.device;
		c.lds_per_block = parent.lds_per_block;
		c.wall_khz = parent.wall_khz;
		c.wide = parent.wide;
		c.wide_shared = true;
		c.pool->other = c.wide;
		ESL_HIP(hipSetDevice(c.device));
		ESL_HIP(hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking));
		for (auto& e : c.ev)
			ESL_HIP(hipEventCreate(&e));
		c.flags.ensure(flag_words);
		ESL_HIP(hipHostMalloc((void**)&c.h_flags, (flag_words + live_words) * sizeof(int32_t), hipHostMallocDefault));
		c.h_live = c.h_flags + flag_words;
		c.h_stage_bytes = stage_bytes;
		ESL_HIP(hipHostMalloc((void**)&c.h_stage, c.h_stage_bytes, hipHostMallocDefault));
	}
	~child_ctx_t()
	{
		(void)hipSetDevice(c.device);
		if (c.stream)
		{
			(void)hipStreamSynchronize(c.stream);
			(void)hipStreamDestroy(c.stream);
		}
		c.pool->clear(true); // plans may hold buffers of it: freed directly from here on
		for (auto& e : c.ev)
			if (e)
				(void)hipEventDestroy(e);
		if (c.h_flags)
			(void)hipHostFree(c.h_flags);
		if (c.h_stage)
			(void)hipHostFree(c.h_stage);
	}
	child_ctx_t(const child_ctx_t&) = delete;
	child_ctx_t& operator=(const child_ctx_t&) = delete;
};

// Several plans (distinct networks) in one call.  Plans solved per set run
// concurrently on forked streams of the calling thread (one HIP graph with
// graph = 1); each plan that needs the host-driven device-wide solver runs at
// the same time on a host thread and stream of its own.
void plan_solve_many(ctx_t& c, int np, void* const* plans, const int* B, const double* const* d_rates,
					 double* const* d_final, const esl_solve_opts& o_in, esl_solve_report* reps)
{
	esl_solve_opts o = o_in;
	if (o.tol <= 0)
		o.tol = 1e-13;
	if (o.max_iters <= 0)
		o.max_iters = 20000;
	std::vector<int> conc, wide;
	std::vector<esl_solve_opts> po(np, o); // per plan: the tuned restart length when asked for
	for (int i = 0; i < np; ++i)
	{
		plan_t& P = *static_cast<plan_t*>(plans[i]);
		reps[i] = esl_solve_report{};
		const bool tuned = o_in.restart == 0 && P.tune.set;
		P.path = run_path(P, o_in);
		po[i].restart = std::min(std::max(tuned ? P.tune.m : (o.restart > 0 ? o.restart : 32), 2), pm_max);
		if (runs_per_set(P, B[i], tuned))
			conc.push_back(i);
		else // one large system: its device-wide solver is driven from the host
			wide.push_back(i);
	}
	// No capture beside the host threads below, which allocate and free: a program
	// that alternates between such batches would capture anew on every call while
	// they run.  One such run ended in a host segmentation fault whose cause is not
	// known, and what a replay saves is microseconds beside milliseconds of device-wide
	// solves.
	if (!wide.empty())
		o.graph = 0;
	// the device-wide plans, each on a host thread of its own, joined before return
	std::vector<std::unique_ptr<child_ctx_t>> kids;
	if (!wide.empty())
		ESL_HIP(hipStreamSynchronize(c.stream)); // what its solves left in the pool may go to another stream
	for (size_t k = 0; k < wide.size(); ++k)
		kids.push_back(std::make_unique<child_ctx_t>(c));
	std::vector<std::exception_ptr> errs(wide.size());
	std::vector<std::thread> workers;
	for (size_t k = 0; k < wide.size(); ++k)
		workers.emplace_back([&, k] {
			try
			{
				const int i = wide[k];
				const pool_scope_t scope(kids[k]->c.pool);
				ESL_HIP(hipSetDevice(kids[k]->c.device));
				plan_run(kids[k]->c, *static_cast<plan_t*>(plans[i]), B[i], d_rates[i], d_final[i], o_in, reps[i]);
			}
			catch (...)
			{
				errs[k] = std::current_exception();
			}
		});
	auto join_all = [&] {
		for (std::thread& t : workers)
			if (t.joinable())
				t.join();
		workers.clear();
	};
	try
	{
		many_per_set(c, conc, plans, B, d_rates, d_final, o, po, reps);
	}
	catch (...)
	{
		join_all();
		throw;
	}
	join_all();
	for (const std::exception_ptr& e : errs)
		if (e)
			std::rethrow_exception(e);
}

// the per-set plans of plan_solve_many: concurrent on forked streams
void many_per_set(ctx_t& c, const std::vector<int>& conc, void* const* plans, const int* B,
				  const double* const* d_rates, double* const* d_final, const esl_solve_opts& o,
				  std::vector<esl_solve_opts>& po, esl_solve_report* reps)
{
	if (conc.empty())
		return;
	for (int i : conc)
	{
		plan_t& P = *static_cast<plan_t*>(plans[i]);
		const bool reduced = plan_reduced(c, P, B[i], po[i]);
		plan_reserve(P, B[i], po[i].restart, o.precision, reduced, !reduced);
	}
	ensure_aux(c, (int)conc.size());
	timer_t tm_(c);
	auto enqueue_all = [&] {
		const hipStream_t main = c.stream;
		ESL_HIP(hipEventRecord(c.aux_ev[0], main));
		for (size_t k = 0; k < conc.size(); ++k)
		{
			const int i = conc[k];
			ESL_HIP(hipStreamWaitEvent(c.aux[k], c.aux_ev[0], 0));
			c.stream = c.aux[k];
			try
			{
				plan_enqueue(c, *static_cast<plan_t*>(plans[i]), B[i], d_rates[i], d_final[i], po[i]);
			}
			catch (...)
			{
				c.stream = main;
				throw;
			}
			c.stream = main;
			ESL_HIP(hipEventRecord(c.aux_ev[k + 1], c.aux[k]));
			ESL_HIP(hipStreamWaitEvent(main, c.aux_ev[k + 1], 0));
		}
	};
	if (o.graph)
	{
		multi_graph_t key;
		for (int i : conc)
		{
			key.plans.push_back(static_cast<plan_t*>(plans[i])->id);
			key.B.push_back(B[i]);
			key.rates.push_back(d_rates[i]);
			key.fin.push_back(d_final[i]);
			key.epochs.push_back(static_cast<plan_t*>(plans[i])->epoch);
			key.ms.push_back(po[i].restart);
			key.paths.push_back(static_cast<plan_t*>(plans[i])->path);
		}
		key.precision = o.precision;
		key.preconditioner = o.preconditioner;
		key.max_iters = o.max_iters;
		key.tol = o.tol;
		key.inner_rtol = o.inner_rtol;
		key.prof = c.prof.on;
		multi_graph_t* mg = static_cast<multi_graph_t*>(c.multi);
		if (!mg || !mg->same(key))
		{
			if (c.multi_free && c.multi)
				c.multi_free(c.multi);
			c.multi = nullptr;
			mg = new multi_graph_t(std::move(key));
			c.multi = mg;
			c.multi_free = multi_graph_free;
			if (c.prof.on)
			{
				ESL_HIP(hipStreamSynchronize(c.stream));
				c.prof.flush();
				c.prof.capture_events = &mg->gev;
				c.prof.capture_pending = &mg->gpend;
			}
			hipGraph_t graph;
			ESL_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
			try
			{
				enqueue_all();
			}
			catch (...)
			{
				(void)hipStreamEndCapture(c.stream, &graph);
				c.prof.capture_events = nullptr;
				c.prof.capture_pending = nullptr;
				c.multi_free(c.multi);
				c.multi = nullptr;
				throw;
			}
			c.prof.capture_events = nullptr;
			c.prof.capture_pending = nullptr;
			ESL_HIP(hipStreamEndCapture(c.stream, &graph));
			const hipError_t ie = hipGraphInstantiate(&mg->exec, graph, nullptr, nullptr, 0);
			(void)hipGraphDestroy(graph);
			if (ie != hipSuccess)
			{
				c.multi_free(c.multi);
				c.multi = nullptr;
				ESL_HIP(ie);
			}
		}
		ESL_HIP(hipGraphLaunch(mg->exec, c.stream));
		ESL_HIP(hipStreamSynchronize(c.stream));
		if (c.prof.on)
			c.prof.book(mg->gpend);
	}
	else
		enqueue_all();
	ESL_HIP(hipStreamSynchronize(c.stream));
	for (int i : conc)
	{
		plan_t& P = *static_cast<plan_t*>(plans[i]);
		esl_solve_report& rep = reps[i];
		rep.terminals_reached = P.Tr;
		rep.unknowns = P.nU;
		rep.reachable = -1;
		if (P.nU > 0)
		{
			const esl_solve_opts& of = po[i];
			set_results_t sr;
			krylov_result_t kr =
				finish_per_set(c, P.sys(B[i], d_rates[i]), P.nbr, P.n_seg, P.rb.rhs, P.rb.z, of, P.rb.ps,
							   plan_reduced(c, P, B[i], of), P.setup(nullptr), [&](int prec) {
					plan_reserve(P, B[i], of.restart, prec, false, false);
					return P.rb.ps;
				}, &sr);
			plan_finish_sets(c, P, B[i], d_rates[i], d_final[i], of, kr, std::move(sr), kr.finished > 0, true);
			rep.exact_solves = kr.exact;
			rep.residual = kr.resid;
			rep.iterations = kr.iters;
			rep.refinements = kr.cycles;
			rep.sets_iterated = kr.sets_iterated;
			rep.fp64_fallback = kr.fp64_fallback;
			rep.iterations_sum = kr.iters_sum;
		}
	}
	tm_.mark();
	double ms = 0.0;
	tm_.read(&ms);
	for (int i : conc)
	{
		reps[i].ms_stage[3] = ms;
		reps[i].ms_total = ms;
	}
}

// out[b][i] = final[b][reordered[i]], i < n_t: the final vectors on the terminal
// states in canonical order (the layout of a warm start and of surrogate targets)
__global__ __launch_bounds__(sblock) void k_gather_terminal(int64_t n, int64_t n_t, const int32_t* __restrict__ reordered,
															const double* __restrict__ fin, double* __restrict__ out)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int64_t b = blockIdx.y;
	if (i < n_t)
		out[b * n_t + i] = fin[b * n + reordered[i]];
}

void plan_gather_terminal(ctx_t& c, const void* p, int B, const double* d_final, double* d_out)
{
	const plan_t& P = *static_cast<const plan_t*>(p);
	const graph_t& g = *P.g;
	if (g.n_t == 0)
		return;
	k_gather_terminal<<<dim3(ceil_div(g.n_t, sblock), B), sblock, 0, c.stream>>>(g.n, g.n_t, g.reordered.get(),
																				  d_final, d_out);
	ESL_HIP(hipGetLastError());
	ESL_HIP(hipStreamSynchronize(c.stream));
}

// Times candidate schedules of a plan on the caller's own batch and keeps the
// fastest one that meets the tolerance: per-set LDS-resident / per-set from
// global memory / device-wide / per-set LDS-resident with the basis in global
// memory / per-set LDS-resident with the private basis at 3 workgroups per CU,
// restart length 16 / 24 / 32 / 64, and the reduced solver.  Each candidate runs once untimed
// (graph capture, buffer growth), then two timed blocks of four runs (the
// better block's mean).  The
// chosen schedule then runs once more, so d_final holds its results.  Later
// solves use the choice when they ask for restart 0.
void plan_autotune(ctx_t& c, void* p, int B, const double* d_rates, double* d_final, const esl_solve_opts& o_in,
				   int32_t choice[2], double* best_ms)
{
	plan_t& P = *static_cast<plan_t*>(p);
	esl_solve_opts o = o_in;
	o.restart = 0;
	o.exact_fallback = 0; // a schedule that misses the tolerance is skipped, not rescued
	struct cand_t
	{
		int path, m;
	};
	std::vector<cand_t> cands;
	const bool ilu = o.preconditioner != 1;
	if (P.nU == 0)
		cands.push_back({ 0, 32 });
	else
		for (int m : { 16, 24, 32, 64 })
		{
			cands.push_back({ 0, m });
			if (ilu && P.nU <= lds_max_unknowns) // otherwise path 1 is path 0
				cands.push_back({ 1, m });
			if (ilu && o.precision == 1 && P.nU <= lds_max_unknowns && m <= 32) // otherwise path 3 is path 0
				cands.push_back({ 3, m });
			if (ilu && o.precision == 1 && P.nU <= 4 * pblock && m <= 32) // the private-basis kernel at 3 WG per CU
				cands.push_back({ 4, m });
			cands.push_back({ 2, m });
		}
	if (P.nU > 0 && o.preconditioner == 0)
		cands.push_back({ path_reduced, 32 }); // keeps no basis: the restart length does not matter
	const plan_t::tune_t saved = P.tune;
	plan_t::tune_t best_t{};
	double best = 1e300;
	for (const cand_t& cd : cands)
	{
		P.tune = plan_t::tune_t{ true, cd.path, cd.m };
		try
		{
			esl_solve_report rep{};
			plan_run(c, P, B, d_rates, d_final, o, rep);
			// the better of two blocks of four back-to-back runs (mean per run):
			// single runs vary by about 5 %, and the best single run favours
			// whichever candidate had one lucky run over the steady-state rate
			double t = 1e300;
			for (int blk = 0; blk < 2; ++blk)
			{
				const auto t0 = std::chrono::steady_clock::now();
				for (int r = 0; r < 4; ++r)
					plan_run(c, P, B, d_rates, d_final, o, rep);
				t = std::min(t, std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count() /
									4.0);
			}
			if (t < best)
			{
				best = t;
				best_t = P.tune;
			}
		}
		catch (const error& e)
		{
			// a schedule that does not converge or does not fit is skipped
			if (e.code != ESL_E_NUMERIC && e.code != ESL_E_OOM)
			{
				P.tune = saved;
				throw;
			}
			(void)hipGetLastError();
		}
	}
	if (!best_t.set)
	{
		P.tune = saved;
		throw error(ESL_E_NUMERIC, "autotune: no schedule reached the tolerance");
	}
	P.tune = best_t;
	{
		esl_solve_report rep{};
		esl_solve_opts of = o_in;
		of.restart = 0; // the tuned schedule, with the caller's fallback setting
		plan_run(c, P, B, d_rates, d_final, of, rep);
	}
	choice[0] = P.tune.path;
	choice[1] = P.tune.m;
	*best_ms = best;
}

void plan_set_schedule(void* p, int path, int restart)
{
	plan_t& P = *static_cast<plan_t*>(p);
	if (path < 0)
		P.tune = plan_t::tune_t{};
	else
		P.tune = plan_t::tune_t{ true, path, std::min(std::max(restart, 2), path == 2 ? dw_max : pm_max) };
}

void plan_set_results(const void* p, int B, double* res, int32_t* its, int32_t* method)
{
	const plan_t& P = *static_cast<const plan_t*>(p);
	if (P.results.res.empty())
		throw error(ESL_E_STATE, "no solve has run on this plan");
	if ((size_t)B != P.results.res.size())
		throw error(ESL_E_ARG, "n_sets (" + std::to_string(B) + ") differs from the last solve's (" +
								   std::to_string(P.results.res.size()) + ")");
	for (int b = 0; b < B; ++b)
	{
		if (res)
			res[b] = P.results.res[b];
		if (its)
			its[b] = P.results.its[b];
		if (method)
			method[b] = P.results.method[b];
	}
}

// per-set start / end of the last per-set launch in ms after its first start
void plan_set_times(const void* p, int B, double wall_khz, double* start_ms, double* end_ms)
{
	const plan_t& P = *static_cast<const plan_t*>(p);
	const auto& t = P.results.tspan;
	if (t.size() != (size_t)2 * B)
		throw error(ESL_E_STATE, "the last solve of this plan recorded no per-set times for " + std::to_string(B) +
									 " sets (it ran device-wide or with another batch size)");
	uint64_t t0 = UINT64_MAX;
	for (int b = 0; b < B; ++b)
		t0 = std::min(t0, t[2 * b]);
	for (int b = 0; b < B; ++b)
	{
		if (start_ms)
			start_ms[b] = (double)(t[2 * b] - t0) / wall_khz;
		if (end_ms)
			end_ms[b] = (double)(t[2 * b + 1] - t0) / wall_khz;
	}
}

void plan_info(const void* p, int64_t info[8])
{
	const plan_t& P = *static_cast<const plan_t*>(p);
	info[0] = P.nU;
	info[1] = P.nUt;
	info[2] = P.nA;
	info[3] = P.Tr;
	info[4] = P.n_seg;
	info[5] = P.nbr.nnz;
	info[6] = P.g ? P.g->n_t : 0;
	info[7] = P.tune.set ? (int64_t)P.tune.path * 1000 + P.tune.m : -1;
}

// solution_term and solution_nonterm in the reference layout (one rate set).
void solution_full(ctx_t& c, graph_t& g, const double* d_rates, const esl_solve_opts& opts_in)
{
	esl_solve_opts opts = opts_in;
	opts.precision = 0;
	const int N = g.N;
	const int64_t n = g.n, T = g.T, n_t = g.n_t;
	const int nb = ceil_div(n, sblock);
	solution_t& sol = g.sol;
	sol = solution_t{};
	std::vector<int32_t> h_reord;
	read_host(c, h_reord, g.reordered.get(), (size_t)n);

	// ---- (a) pi of every terminal SCC (row-replaced systems, no pruning)
	std::vector<int32_t> seg_off(1, 0), seg_src, segmap(T, -1);
	int n_seg = 0;
	for (int64_t k = 0; k < T; ++k)
	{
		const int32_t sz = g.h_offsets[k + 1] - g.h_offsets[k];
		if (sz >= 2)
		{
			segmap[k] = n_seg++;
			seg_off.push_back(seg_off.back() + sz);
			seg_src.push_back(g.h_offsets[k]);
		}
	}
	sol.term_indptr.assign(g.h_offsets.begin(), g.h_offsets.begin() + T + 1);
	sol.term_indices.assign(h_reord.begin(), h_reord.begin() + n_t);
	sol.term_data.assign(n_t, 1.0);
	dbuf<int32_t> pos;
	pos.ensure(n);
	if (n_seg)
	{
		const int64_t nUt = seg_off.back();
		std::vector<int32_t> states(nUt), seg_of(nUt);
		for (int k = 0; k < n_seg; ++k)
			for (int32_t q = 0; q < seg_off[k + 1] - seg_off[k]; ++q)
			{
				states[seg_off[k] + q] = h_reord[seg_src[k] + q];
				seg_of[seg_off[k] + q] = k;
			}
		dbuf<int32_t> ulist, ucls, d_seg_off, anchor;
		ulist.ensure(nUt);
		ucls.ensure(nUt);
		d_seg_off.ensure(seg_off.size());
		anchor.ensure(n_seg);
		write_dev(c, ulist.get(), states);
		write_dev(c, ucls.get(), seg_of);
		write_dev(c, d_seg_off.get(), seg_off);
		ESL_HIP(hipMemsetAsync(pos.get(), 0xff, n * sizeof(int32_t), c.stream));
		dbuf<int32_t> d_states;
		d_states.ensure(nUt);
		write_dev(c, d_states.get(), states);
		k_fill_term_unknowns<<<ceil_div(nUt, sblock), sblock, 0, c.stream>>>(nUt, d_states.get(), ucls.get(),
																			 ulist.get(), ucls.get(), pos.get());
		sys_t S{};
		S.N = N;
		S.nU = S.nUt = nUt;
		S.B = 1;
		S.mask = g.mask.get();
		S.ulist = ulist.get();
		S.ucls = ucls.get();
		S.pos = pos.get();
		S.rates = d_rates;
		S.rate_stride = 2 * N;
		S.transpose = 0;
		nbr_store_t nb; // the coupling lists serve the anchor sweeps and the solve
		build_nbr(c, S, nb);
		dbuf<double> p0, p1;
		p0.ensure(nUt);
		p1.ensure(nUt);
		write_dev(c, p0.get(), std::vector<double>(nUt, 1.0));
		for (int it = 0; it < 32; ++it)
		{
			k_anchor_sweep<<<dim3(ceil_div(nUt, sblock), 1), sblock, 0, c.stream>>>(S, nb.view(), p0.get(),
																				   p1.get());
			std::swap(p0, p1);
		}
		k_anchor_pick<<<dim3(n_seg, 1), sblock, 0, c.stream>>>(nUt, d_seg_off.get(), p0.get(), n_seg, anchor.get());
		S.anchor = anchor.get();
		dbuf<double> invd, rhs, z, segsum, pi;
		invd.ensure(nUt);
		rhs.ensure(nUt);
		z.ensure(nUt);
		segsum.ensure(n_seg);
		pi.ensure(nUt);
		S.invd = invd.get();
		const dim3 gu(ceil_div(nUt, sblock), 1);
		k_invd<<<gu, sblock, 0, c.stream>>>(S, n_seg, invd.get());
		k_rhs<<<gu, sblock, 0, c.stream>>>(S, n_seg, nullptr, rhs.get());
		k_zero<double><<<ceil_div(nUt, sblock), sblock, 0, c.stream>>>(nUt, z.get());
		ESL_HIP(hipGetLastError());
		const rb_setup_t su{ nullptr, d_seg_off.get(), n_seg, anchor.get(), invd.get(), rhs.get(), nullptr, nullptr, 0, nullptr };
		krylov_solve(c, S, n_seg, rhs.get(), z.get(), opts, &nb, false, true, nullptr, path_reduced, &su);
		k_seg_sum<<<dim3(n_seg, 1), sblock, 0, c.stream>>>(nUt, d_seg_off.get(), z.get(), invd.get(), n_seg,
														  segsum.get());
		k_times_invd<<<ceil_div(nUt, sblock), sblock, 0, c.stream>>>(nUt, z.get(), invd.get(), pi.get());
		std::vector<double> h_pi, h_sum;
		read_host(c, h_pi, pi.get(), nUt);
		read_host(c, h_sum, segsum.get(), n_seg);
		for (int k = 0; k < n_seg; ++k)
			for (int32_t q = 0; q < seg_off[k + 1] - seg_off[k]; ++q)
				sol.term_data[seg_src[k] + q] = h_pi[seg_off[k] + q] / h_sum[k];
	}

	// ---- (b) absorption probabilities X[j, c] of every transient state
	sol.nonterm_indptr.assign(1, 0);
	const int64_t n_nt = n - n_t;
	if (n_nt == 0 || T == 1)
	{
		for (int64_t j = 0; j < T; ++j)
		{
			for (int32_t p = g.h_offsets[j]; p < g.h_offsets[j + 1]; ++p)
			{
				sol.nonterm_indices.push_back(h_reord[p]);
				sol.nonterm_data.push_back(1.0);
			}
			for (int64_t p = n_t; p < n; ++p)
			{
				sol.nonterm_indices.push_back(h_reord[p]);
				sol.nonterm_data.push_back(1.0);
			}
			sol.nonterm_indptr.push_back((int32_t)sol.nonterm_indices.size());
		}
		sol.valid = true;
		return;
	}
	const bool fallback = T > max_rhs_terms;
	if (T > 65535)
		throw error(ESL_E_ARG, "full solution export supports at most 65535 terminal SCCs (one right-hand side "
							   "per terminal SCC in one launch dimension)");
	dbuf<uint8_t> reach;
	reach.ensure(n);
	k_fill_u8<<<nb, sblock, 0, c.stream>>>(n, 1, reach.get());
	std::vector<int32_t> jmap(T);
	for (int64_t k = 0; k < T; ++k)
		jmap[k] = (int32_t)k;
	dbuf<int32_t> d_jmap;
	d_jmap.ensure(T);
	write_dev(c, d_jmap.get(), jmap);
	dbuf<uint64_t> tmask;
	tmask.ensure(n);
	k_tm_init<<<nb, sblock, 0, c.stream>>>(n, g.rank.get(), T, d_jmap.get(), reach.get(), tmask.get());
	if (!fallback)
		propagate_masks(c, g, reach.get(), tmask.get());
	dbuf<int32_t> amb, fpos;
	amb.ensure(n);
	fpos.ensure(n + 1);
	k_amb_flag<<<nb, sblock, 0, c.stream>>>(n, g.rank.get(), T, reach.get(), tmask.get(), fallback ? 1 : 0,
											amb.get());
	exclusive_scan_i32(c, amb.get(), fpos.get(), n);
	int32_t nA = 0;
	ESL_HIP(hipMemcpyAsync(&nA, fpos.get() + n, sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
	ESL_HIP(hipStreamSynchronize(c.stream));
	std::vector<uint64_t> h_tm;
	read_host(c, h_tm, tmask.get(), (size_t)n);
	std::vector<int32_t> h_pos(n, -1);
	std::vector<double> h_x; // [T][nA]
	if (nA)
	{
		dbuf<int32_t> ulist, ucls;
		ulist.ensure(nA);
		ucls.ensure(nA);
		ESL_HIP(hipMemsetAsync(pos.get(), 0xff, n * sizeof(int32_t), c.stream));
		k_fill_unknowns<<<nb, sblock, 0, c.stream>>>(n, amb.get(), fpos.get(), 0, ulist.get(), ucls.get(),
													 pos.get());
		sys_t S{};
		S.N = N;
		S.nU = nA;
		S.nUt = 0;
		S.B = (int)T;
		S.mask = g.mask.get();
		S.ulist = ulist.get();
		S.ucls = ucls.get();
		S.pos = pos.get();
		S.rates = d_rates;
		S.rate_stride = 0; // every right-hand side shares the rates
		S.transpose = 1;
		dbuf<int32_t> anchor;
		anchor.ensure(1);
		S.anchor = anchor.get();
		dbuf<double> invd, rhs, z;
		invd.ensure((size_t)T * nA);
		rhs.ensure((size_t)T * nA);
		z.ensure((size_t)T * nA);
		S.invd = invd.get();
		const dim3 gu(ceil_div(nA, sblock), (unsigned)T);
		k_invd<<<gu, sblock, 0, c.stream>>>(S, 1, invd.get());
		k_rhs_absorb<<<gu, sblock, 0, c.stream>>>(S, g.rank.get(), T, tmask.get(), rhs.get());
		k_zero<double><<<ceil_div((int64_t)T * nA, sblock), sblock, 0, c.stream>>>((int64_t)T * nA, z.get());
		ESL_HIP(hipGetLastError());
		krylov_solve(c, S, 0, rhs.get(), z.get(), opts);
		dbuf<double> x;
		x.ensure((size_t)T * nA);
		k_times_invd<<<ceil_div((int64_t)T * nA, sblock), sblock, 0, c.stream>>>((int64_t)T * nA, z.get(), invd.get(),
																				  x.get());
		read_host(c, h_x, x.get(), (size_t)T * nA);
		read_host(c, h_pos, pos.get(), (size_t)n);
	}
	std::vector<int32_t> h_rank;
	read_host(c, h_rank, g.rank.get(), (size_t)n);
	for (int64_t j = 0; j < T; ++j)
	{
		for (int32_t p = g.h_offsets[j]; p < g.h_offsets[j + 1]; ++p)
		{
			sol.nonterm_indices.push_back(h_reord[p]);
			sol.nonterm_data.push_back(1.0);
		}
		for (int64_t p = n_t; p < n; ++p)
		{
			const int32_t cst = h_reord[p];
			const int32_t u = h_pos[cst];
			double v;
			if (u >= 0)
			{
				if (!fallback && !((h_tm[cst] >> j) & 1ull))
					continue;
				v = h_x[(size_t)j * nA + u];
				if (v == 0.0)
					continue;
			}
			else
			{
				const int t = __builtin_ffsll((long long)h_tm[cst]) - 1;
				if (t != j)
					continue;
				v = 1.0;
			}
			sol.nonterm_indices.push_back(cst);
			sol.nonterm_data.push_back(v);
		}
		sol.nonterm_indptr.push_back((int32_t)sol.nonterm_indices.size());
	}
	sol.valid = true;
}

} // namespace esl
