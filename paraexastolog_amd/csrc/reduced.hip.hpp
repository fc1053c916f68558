// Per-set solver on the parity-reduced system (included by solve.hip).
//
// Every coupling flips one bit of the state, so it joins a state of even to a
// state of odd popcount: the systems are two-coloured,
//     M = [ D_E  -A_ER ]      rows E: one parity class (the larger),
//         [ -A_RE  D_R ]      rows R: the other.
// The E unknowns are eliminated exactly (D_E is diagonal), which leaves
//     S x_R = b_R + A_RE D_E^{-1} b_E,   S = D_R - A_RE D_E^{-1} A_ER
// on half the unknowns, and x_E = D_E^{-1} (b_E + A_ER x_R).  A product by S
// costs what a product by M costs and has two phases, so two workgroup
// barriers, where a preconditioned step with ILU(0) has one per popcount level
// and sweep.  BiCGStab on S, scaled from the left by the inverse of its
// diagonal, needs no basis: five vectors of half length per set, in registers.
//
// It replaces restarted GMRES with ILU(0) as the default method of the per-set
// solver (that one stays for sets on which this method stalls, and for callers
// that ask for a restart length or a preconditioner).  At 1e-12 a set of N = 20
// seed 0 (1,022 unknowns) takes 66-90 products by S against 30 by M with ILU(0),
// but a product costs three barriers and one reduction where a preconditioned step
// has 22 levels and a Gram-Schmidt pass.  Bound: the latency of that chain.
// Measured on MI355X, GMRES with ILU(0) -> this: one set in FP64 853 -> 89 us; 250
// sets of 2,048 unknowns in FP64 6,600 -> 385 us; 1,024 sets of 1,022 unknowns in
// mixed precision, beside the fill of the final vectors, 2,130 -> 912 us.

// coupling lists with rows in class order: row q < nE is an eliminated unknown,
// row nE + o a kept one; a neighbour is named by its index inside the other
// class.  Lists are padded to groups of four records with null records (rate
// code rb_null, whose rate is zero; neighbour 0), so a group is one 16-byte load
// and needs no bounds test.
struct rb_t
{
	int nE = 0, nR = 0;
	const int32_t* ptr = nullptr; // [nU + 1] first group of each row
	const int32_t* row = nullptr; // [nU] row -> unknown
	const uint4* rec = nullptr;	  // neighbour | rate code << 25 | mirrored << 31
};
constexpr int rb_null = 63; // 2N <= 52 rate codes are in use
constexpr uint32_t rb_index = (1u << 25) - 1; // a parity class has at most 2^25 states (N <= 26)
__device__ __forceinline__ int rb_code(uint32_t r) { return (r >> 25) & 63; }

__global__ __launch_bounds__(sblock) void k_rb_parity(int64_t nU, const int32_t* __restrict__ ulist,
													  int32_t* __restrict__ odd)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (u < nU)
		odd[u] = __popc((uint32_t)ulist[u]) & 1;
}

// unknowns -> rows (ascending unknowns inside a class); inv[u] = index inside its
// class, cnt[row] = groups of four couplings
__global__ __launch_bounds__(sblock) void k_rb_place(int64_t nU, int nE, int elim, const int32_t* __restrict__ ulist,
													 const int32_t* __restrict__ opos,
													 const int32_t* __restrict__ gptr, int32_t* __restrict__ row,
													 int32_t* __restrict__ inv, int32_t* __restrict__ cnt)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (u >= nU)
		return;
	const int par = __popc((uint32_t)ulist[u]) & 1;
	const int32_t idx = par ? opos[u] : (int32_t)u - opos[u];
	const int32_t q = par == elim ? idx : nE + idx;
	inv[u] = idx;
	row[q] = (int32_t)u;
	cnt[q] = (gptr[u + 1] - gptr[u] + 3) / 4;
}

__global__ __launch_bounds__(sblock) void k_rb_fill(int64_t nU, const int32_t* __restrict__ row,
													const int32_t* __restrict__ inv, const int32_t* __restrict__ gptr,
													const int32_t* __restrict__ gnu, const uint8_t* __restrict__ gnr,
													const int32_t* __restrict__ rptr, uint4* __restrict__ rec)
{
	const int64_t q = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (q >= nU)
		return;
	const int32_t u = row[q];
	int32_t e = gptr[u];
	const int32_t e1 = gptr[u + 1];
	for (int32_t g = rptr[q]; g < rptr[q + 1]; ++g)
	{
		uint32_t r[4];
		for (int k = 0; k < 4; ++k, ++e)
		{
			r[k] = (uint32_t)rb_null << 25;
			if (e < e1)
			{
				const uint32_t code = gnr[e];
				r[k] = (uint32_t)inv[gnu[e]] | (code & 63u) << 25 | (code & nbr_rev_flag ? 1u << 31 : 0u);
			}
		}
		rec[g] = make_uint4(r[0], r[1], r[2], r[3]);
	}
}

// s + sum over the groups of a row (first group | groups << 24) of rate * y[neighbour], in list order
template <typename Y>
__device__ __forceinline__ double rb_sum(const uint4* __restrict__ rec, const double* __restrict__ rates, uint32_t h,
										 const Y* __restrict__ y, double s)
{
	const int g1 = (int)(h & 0xffffff) + (int)(h >> 24);
	for (int g = (int)(h & 0xffffff); g < g1; ++g)
	{
		const uint4 q = rec[g];
		const double r0 = rates[rb_code(q.x)], r1 = rates[rb_code(q.y)];
		const double r2 = rates[rb_code(q.z)], r3 = rates[rb_code(q.w)];
		const Y y0 = y[q.x & rb_index], y1 = y[q.y & rb_index];
		const Y y2 = y[q.z & rb_index], y3 = y[q.w & rb_index];
		// the eight loads together: one LDS round trip per group instead of one per term
		__builtin_amdgcn_sched_barrier(0);
		s += r0 * (double)y0;
		s += r1 * (double)y1;
		s += r2 * (double)y2;
		s += r3 * (double)y3;
	}
	return s;
}

// v plus the value of v in the lane that a DPP control names (zero past a row's end)
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_add(double v)
{
	const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
	const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
	return v + __hiloint2double(hi, lo);
}
constexpr int dpp_shr1 = 0x111, dpp_shr2 = 0x112, dpp_shr4 = 0x114, dpp_shr8 = 0x118, dpp_bcast15 = 0x142,
			  dpp_bcast31 = 0x143;

// sum over the wavefront, valid in lane 63.  Six data-parallel-primitive adds:
// no LDS round trip, where a shuffle butterfly makes twelve for a double.
__device__ __forceinline__ double wave_sum63(double v)
{
	v = dpp_add<dpp_shr1>(v);
	v = dpp_add<dpp_shr2>(v);
	v = dpp_add<dpp_shr4>(v);
	v = dpp_add<dpp_shr8>(v);
	v = dpp_add<dpp_bcast15, 0xa>(v);
	v = dpp_add<dpp_bcast31, 0xc>(v);
	return v;
}

__device__ __forceinline__ double read_lane(double v, int i)
{
	return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), i),
							__builtin_amdgcn_readlane(__double2loint(v), i));
}

constexpr int rb_part = 128; // doubles of one reduction buffer (K <= 8 sums of up to 16 wavefronts)

// v[k] <- sum over the workgroup (K values at once, one barrier, fixed order).
// Every wavefront adds the per-wavefront partials of all K values in its lanes:
// one LDS read and log2(wavefronts) adds.  `part` must not be reused before
// another barrier has passed (callers alternate between two).
template <int BLK, int K>
__device__ __forceinline__ void rb_block_sums(double (&v)[K], double* part)
{
	constexpr int nw = BLK / wave;
#pragma unroll
	for (int k = 0; k < K; ++k)
		v[k] = wave_sum63(v[k]);
	if constexpr (nw == 1)
	{
#pragma unroll
		for (int k = 0; k < K; ++k)
			v[k] = read_lane(v[k], wave - 1);
	}
	else
	{
		const int lane = threadIdx.x & (wave - 1);
		if (lane == wave - 1)
#pragma unroll
			for (int k = 0; k < K; ++k)
				part[k * nw + threadIdx.x / wave] = v[k];
		__syncthreads();
#pragma unroll
		for (int k0 = 0; k0 < K; k0 += wave / nw)
		{
			double t = part[k0 * nw + lane]; // lanes past K * nw read words of the buffer that are not used
			t = dpp_add<dpp_shr1>(t);
			if constexpr (nw > 2)
				t = dpp_add<dpp_shr2>(t);
			if constexpr (nw > 4)
				t = dpp_add<dpp_shr4>(t);
			if constexpr (nw > 8)
				t = dpp_add<dpp_shr8>(t);
#pragma unroll
			for (int k = k0; k < K && k < k0 + wave / nw; ++k)
				v[k] = read_lane(t, (k - k0 + 1) * nw - 1);
		}
	}
}

__device__ __forceinline__ bool rb_finite(double v) { return fabs(v) < 1e300; }

// weight of row o in the shadow vector of a cycle after `fails` cycles that did
// not reduce the residual: 1 at first (the residual itself), then the residual
// with weights in [0.5, 1.5), then values in [-0.5, 0.5) of their own.  A cycle
// whose shadow vector is orthogonal to its first product breaks down; another
// shadow vector does not.
__device__ __forceinline__ double rb_shadow(int o, int fails, double r)
{
	if (fails == 0)
		return r;
	uint32_t h = (uint32_t)o * 2654435761u + 12345u;
	h ^= h >> 15;
	h *= 0x85ebca6bu;
	h ^= h >> 13;
	const double w = (double)(h & 1023u) / 1024.0;
	return fails == 1 ? r * (0.5 + w) : w - 0.5;
}

struct rb_scratch_t
{
	double* x;	// [B][nU] iterate, in row order
	double* b;	// [B][nU] right-hand side, in row order
	double* rE; // [B][nU] residual of the eliminated rows
	double* xk; // [B][nU] iterate before the last cycle
};

// Where a cycle that starts at the relative residual rel stops: a tenth of the
// tolerance, in as many equal drops as cycles that each reduce by inner_rtol
// would need (what FP32 vectors can deliver; 0: in one).  Aiming at the tolerance
// itself leaves the last cycle's residual just below it; the extra decade costs
// one product in twelve and keeps the error of the result where GMRES had it.
__device__ __forceinline__ double rb_target(double rel, double tol, double inner_rtol)
{
	const double end = 0.1 * tol;
	if (!(inner_rtol > 0.0) || rel * inner_rtol <= end)
		return end;
	const double cycles = ceil(log(rel / end) / -log(inner_rtol) - 1e-3);
	return rel * exp(-log(rel / end) / fmax(cycles, 1.0));
}

constexpr int rb_max_fails = 3;		 // cycles without progress before a set is left to GMRES
constexpr int rb_cycle_products = 200; // products by S per cycle, so that rounding cannot drift for long

// One workgroup of BLK threads solves one rate set; thread t owns the rows
// t + i BLK (i < RPT) of both classes.  LREC: the coupling records are copied to
// LDS, else they are read from global memory (shared by all sets, so from L2).
template <typename T, int BLK, int RPT, bool LREC>
__device__ __forceinline__ void bicg_set_body(const sys_t& S, const rb_t& G, int n_seg, const double* __restrict__ rhs,
											  double* __restrict__ zio, const rb_scratch_t& sc, double tol,
											  int max_iters, const pgm_out_t& out, double inner_rtol)
{
	extern __shared__ __align__(16) unsigned char smem[];
	__shared__ double s_part[2][rb_part];
	__shared__ double s_rates[64];
	const int b = blockIdx.x, tid = threadIdx.x;
	const uint64_t t_begin = wall_clock64();
	const int nE = G.nE, nR = G.nR, nU = nE + nR;
	const int64_t off = (int64_t)b * nU;
	T* s_g = (T*)smem;	 // [nR] the vector being multiplied
	T* s_te = s_g + nR;	 // [nE] its image on the eliminated rows
	uint4* s_rec = (uint4*)(smem + ((size_t)nU * sizeof(T) + 15) / 16 * 16);
	double* __restrict__ xp = sc.x + off;
	double* __restrict__ bp = sc.b + off;
	double* __restrict__ rEp = sc.rE + off;
	double* __restrict__ xk = sc.xk + off;
	const uint4* rec = LREC ? s_rec : G.rec;

	for (int i = tid; i < 64; i += BLK)
		s_rates[i] = i < 2 * S.N ? S.rates[(int64_t)b * S.rate_stride + i] : 0.0;
	if (LREC)
	{
		const int groups = G.ptr[nU];
		for (int g = tid; g < groups; g += BLK)
			s_rec[g] = G.rec[g];
	}
	// own rows: coupling groups (none for an anchor, whose row is the identity),
	// 1 / D of the eliminated ones, D and 1 / diag(S) of the kept ones
	uint32_t hE[RPT], hR[RPT];
	double cE[RPT], dR[RPT], jR[RPT];
	double bb = 0.0;
#pragma unroll
	for (int i = 0; i < RPT; ++i)
	{
		const int e = tid + i * BLK;
		hE[i] = 0;
		cE[i] = 0.0;
		if (e < nE)
		{
			const int u = G.row[e];
			const bool anc = is_anchor(S, n_seg, b, u);
			const int g0 = G.ptr[e];
			hE[i] = anc ? 0u : (uint32_t)g0 | (uint32_t)(G.ptr[e + 1] - g0) << 24;
			cE[i] = S.invd[off + u];
			xp[e] = zio[off + u] * cE[i];
			const double r = rhs[off + u];
			bp[e] = r;
			bb += r * r;
			s_te[e] = anc ? (T)0 : (T)cE[i];
		}
	}
	__syncthreads();
#pragma unroll
	for (int i = 0; i < RPT; ++i)
	{
		const int o = tid + i * BLK;
		hR[i] = 0;
		dR[i] = jR[i] = 0.0;
		if (o < nR)
		{
			const int u = G.row[nE + o];
			const int g0 = G.ptr[nE + o];
			hR[i] = is_anchor(S, n_seg, b, u) ? 0u : (uint32_t)g0 | (uint32_t)(G.ptr[nE + o + 1] - g0) << 24;
			const double iv = S.invd[off + u];
			dR[i] = 1.0 / iv;
			xp[nE + o] = zio[off + u] * iv;
			const double r = rhs[off + u];
			bp[nE + o] = r;
			bb += r * r;
			// diag(S): D less what leaves the row and comes straight back
			double d = dR[i];
			const int g1 = (int)(hR[i] & 0xffffff) + (int)(hR[i] >> 24);
			for (int g = (int)(hR[i] & 0xffffff); g < g1; ++g)
			{
				const uint4 q = rec[g];
				const uint32_t qq[4] = { q.x, q.y, q.z, q.w };
#pragma unroll
				for (int k = 0; k < 4; ++k)
					if (qq[k] >> 31)
						d -= s_rates[rb_code(qq[k])] * s_rates[rb_code(qq[k]) ^ 1] * (double)s_te[qq[k] & rb_index];
			}
			jR[i] = 1.0 / (d > 0.0 ? d : dR[i]);
		}
	}
	__threadfence_block();
	double sums[5];
	{
		double s1[1] = { bb };
		rb_block_sums<BLK>(s1, s_part[1]);
		bb = s1[0];
	}
	const double bn = bb > 0.0 ? sqrt(bb) : 1.0;
	__syncthreads();

	int iters = 0, cycles = 0, stalled = 0, fails = 0;
	bool compare = false; // rel_prev is the residual before the last cycle
	double rel = 0.0, rel_prev = 0.0;
	for (;;)
	{
		// FP64 residual of the own rows of both classes
		double ro[RPT];
		double rr[1] = { 0.0 };
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int e = tid + i * BLK;
			if (e < nE)
			{
				const double r = bp[e] - (xp[e] / cE[i] - rb_sum(rec, s_rates, hE[i], xp + nE, 0.0));
				rEp[e] = r;
				rr[0] += r * r;
			}
			ro[i] = 0.0;
			if (e < nR)
			{
				ro[i] = bp[nE + e] - (dR[i] * xp[nE + e] - rb_sum(rec, s_rates, hR[i], xp, 0.0));
				rr[0] += ro[i] * ro[i];
			}
		}
		rb_block_sums<BLK>(rr, s_part[0]);
		const double beta = sqrt(rr[0]);
		rel = beta / bn;
		if (rel <= tol || iters >= max_iters)
			break;
		if (compare && !(rel < 0.9 * rel_prev))
		{
			// a cycle that did not reduce the residual: undo it if it made things
			// worse, and go on with another shadow vector a few times
			++fails;
			if (!(rel <= rel_prev))
			{
#pragma unroll
				for (int i = 0; i < RPT; ++i)
				{
					const int e = tid + i * BLK;
					if (e < nE)
						xp[e] = xk[e];
					if (e < nR)
						xp[nE + e] = xk[nE + e];
				}
				rel = rel_prev;
				__threadfence_block();
				__syncthreads();
			}
			if (fails >= rb_max_fails)
			{
				stalled = 1;
				break;
			}
			if (rel == rel_prev) // undone: its residual is needed again
			{
				compare = false;
				continue;
			}
		}
		else
			fails = compare ? 0 : fails;
		compare = true;
		rel_prev = rel;
		const double inner_target = rb_target(rel, tol, sizeof(T) == 4 ? inner_rtol : 0.0);
		++cycles;
		const double inv_beta = 1.0 / beta;
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int e = tid + i * BLK;
			if (e < nE)
				s_te[e] = (T)(cE[i] * rEp[e] * inv_beta);
		}
		__syncthreads();
		T r[RPT], rh[RPT], p[RPT], v[RPT], x[RPT];
		double s2[2] = { 0.0, 0.0 };
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int o = tid + i * BLK;
			r[i] = (T)(jR[i] * rb_sum(rec, s_rates, hR[i], s_te, ro[i] * inv_beta));
			rh[i] = o < nR ? (T)rb_shadow(o, fails, (double)r[i]) : (T)0;
			p[i] = r[i];
			x[i] = (T)0;
			s2[0] += (double)r[i] * (double)r[i];
			s2[1] += (double)rh[i] * (double)r[i];
		}
		rb_block_sums<BLK>(s2, s_part[1]);
		double rho = s2[1];
		const double est = s2[0] > 0.0 ? rel / sqrt(s2[0]) : 0.0; // |r| -> relative residual
		int left = s2[0] > 0.0 ? rb_cycle_products : 0;
		while (left > 0)
		{
			// v = J S p
#pragma unroll
			for (int i = 0; i < RPT; ++i)
				if (tid + i * BLK < nR)
					s_g[tid + i * BLK] = p[i];
			__syncthreads();
#pragma unroll
			for (int i = 0; i < RPT; ++i)
				if (tid + i * BLK < nE)
					s_te[tid + i * BLK] = (T)(cE[i] * rb_sum(rec, s_rates, hE[i], s_g, 0.0));
			__syncthreads();
			double s1[1] = { 0.0 };
#pragma unroll
			for (int i = 0; i < RPT; ++i)
			{
				v[i] = (T)(jR[i] * (dR[i] * (double)p[i] - rb_sum(rec, s_rates, hR[i], s_te, 0.0)));
				s1[0] += (double)rh[i] * (double)v[i];
			}
			rb_block_sums<BLK>(s1, s_part[0]);
			++iters;
			--left;
			const double alpha = rho / s1[0];
			if (!rb_finite(alpha))
				break;
			// s = r - alpha v (in r), t = J S s
#pragma unroll
			for (int i = 0; i < RPT; ++i)
			{
				r[i] = (T)((double)r[i] - alpha * (double)v[i]);
				if (tid + i * BLK < nR)
					s_g[tid + i * BLK] = r[i];
			}
			__syncthreads();
#pragma unroll
			for (int i = 0; i < RPT; ++i)
				if (tid + i * BLK < nE)
					s_te[tid + i * BLK] = (T)(cE[i] * rb_sum(rec, s_rates, hE[i], s_g, 0.0));
			__syncthreads();
			T t[RPT];
#pragma unroll
			for (int k = 0; k < 5; ++k)
				sums[k] = 0.0;
#pragma unroll
			for (int i = 0; i < RPT; ++i)
			{
				t[i] = (T)(jR[i] * (dR[i] * (double)r[i] - rb_sum(rec, s_rates, hR[i], s_te, 0.0)));
				const double td = (double)t[i], sd = (double)r[i], hd = (double)rh[i];
				sums[0] += td * sd;
				sums[1] += td * td;
				sums[2] += sd * sd;
				sums[3] += hd * sd;
				sums[4] += hd * td;
			}
			rb_block_sums<BLK>(sums, s_part[1]);
			++iters;
			--left;
			double omega = sums[1] > 0.0 ? sums[0] / sums[1] : 0.0;
			if (!rb_finite(omega))
				omega = 0.0;
			const double rr2 = fmax(sums[2] - omega * (2.0 * sums[0] - omega * sums[1]), 0.0);
			const double rho1 = sums[3] - omega * sums[4];
			const double beta_b = (rho1 / rho) * (alpha / omega);
			const bool stop = sqrt(rr2) * est <= inner_target || omega == 0.0 || !rb_finite(beta_b) || beta_b == 0.0 ||
							  iters >= max_iters;
			rho = rho1;
#pragma unroll
			for (int i = 0; i < RPT; ++i)
			{
				x[i] = (T)((double)x[i] + alpha * (double)p[i] + omega * (double)r[i]);
				r[i] = (T)((double)r[i] - omega * (double)t[i]);
				p[i] = (T)((double)r[i] + beta_b * ((double)p[i] - omega * (double)v[i]));
			}
			if (stop)
				break;
		}
		// x_R += |r| x, then x_E from the rows that were eliminated, in FP64; the
		// last pass over s_g ended before the barriers of the reduction above
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int o = tid + i * BLK;
			if (o < nR)
			{
				s_g[o] = x[i];
				const double x0 = xp[nE + o];
				xk[nE + o] = x0;
				xp[nE + o] = x0 + beta * (double)x[i];
			}
		}
		__syncthreads();
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int e = tid + i * BLK;
			if (e < nE)
			{
				const double x0 = xp[e];
				xk[e] = x0;
				xp[e] = x0 + cE[i] * (rEp[e] + beta * rb_sum(rec, s_rates, hE[i], s_g, 0.0));
			}
		}
		__threadfence_block();
		__syncthreads();
	}
	// z = D' x, back in the unknown order of the caller
	for (int q = tid; q < nU; q += BLK)
	{
		const int u = G.row[q];
		zio[off + u] = xp[q] / S.invd[off + u];
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

template <typename T, int BLK, int RPT, bool LREC>
__global__ __launch_bounds__(BLK, BLK >= 1024 || LREC ? 4 : 2) void k_bicg_set(
	sys_t S, rb_t G, int n_seg, const double* __restrict__ rhs, double* __restrict__ zio, rb_scratch_t sc, double tol,
	int max_iters, pgm_out_t out, double inner_rtol)
{
	bicg_set_body<T, BLK, RPT, LREC>(S, G, n_seg, rhs, zio, sc, tol, max_iters, out, inner_rtol);
}

using bicg_set_fn = void (*)(sys_t, rb_t, int, const double*, double*, rb_scratch_t, double, int, pgm_out_t, double);
struct bicg_variant_t
{
	bicg_set_fn fn[2]; // FP64, FP32 vectors
	int blk, rows;	   // threads, rows of the larger class at most
	bool lrec;
};

// The variants, smallest first.  A batch of more sets than compute units takes
// two rows per thread, so that several sets share a CU; up to that many sets
// each has a CU to itself, and one row per thread shortens its chain.
constexpr int rb_cus = 256;
constexpr size_t rb_lds_static = 3072; // upper bound of the kernel's static LDS
// dynamic LDS of one set: the vector being multiplied, its image, the records
inline size_t rb_lds_bytes(int64_t nU, int64_t groups, int precision, bool lrec)
{
	return ((size_t)nU * (precision == 1 ? 4 : 8) + 15) / 16 * 16 + (lrec ? (size_t)groups * 16 : 0);
}
inline const bicg_variant_t* rb_variant(int64_t nE, int64_t nR, int64_t groups, int precision, int B, size_t lds_max)
{
#define ESL_RB(BLK, RPT, LREC)                                                                                       \
	{ { k_bicg_set<double, BLK, RPT, LREC>, k_bicg_set<float, BLK, RPT, LREC> }, BLK, BLK * RPT, LREC }
	static const bicg_variant_t few[] = { ESL_RB(64, 1, true),	 ESL_RB(256, 1, true),	 ESL_RB(512, 1, true),
										  ESL_RB(1024, 1, true), ESL_RB(1024, 2, false), ESL_RB(1024, 4, false) };
	static const bicg_variant_t many[] = { ESL_RB(64, 2, true), ESL_RB(256, 2, true), ESL_RB(512, 2, true),
										   ESL_RB(1024, 2, false), ESL_RB(1024, 4, false) };
#undef ESL_RB
	const int64_t rows = nE > nR ? nE : nR;
	auto pick = [&](const bicg_variant_t* v, int n) -> const bicg_variant_t* {
		for (int i = 0; i < n; ++i)
			if (rows <= v[i].rows && rb_lds_bytes(nE + nR, groups, precision, v[i].lrec) + rb_lds_static <= lds_max)
				return v + i;
		return nullptr;
	};
	return B <= rb_cus ? pick(few, sizeof few / sizeof *few) : pick(many, sizeof many / sizeof *many);
}
