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
// diagonal, needs no basis: five vectors of half length per set, in registers (the
// kernels of 1,024 threads with four and two rows a thread spill 104 and 6 of them, the one
// of 512 threads with two rows 2).
//
// It replaces restarted GMRES with ILU(0) as the default method of the per-set
// solver (that one stays for sets on which this method stalls, and for callers
// that ask for a restart length or a preconditioner).  At 1e-12 a set of N = 20
// seed 0 (1,022 unknowns) takes 40-90 products by S against 30 by M with ILU(0),
// but a product costs three barriers and one reduction where a preconditioned step
// has 22 levels and a Gram-Schmidt pass.  Bound: the latency of that chain.
// Vectors are FP64 in both precisions: in FP32 the recurrences lose so much that
// the same sets take 90 products on average and up to 288 instead of 62 and 158
// (1,024 sets: 912 us against 453), and larger systems up to three times as many.
// Measured on MI355X, GMRES with ILU(0) -> this: one set in FP64 853 -> 89 us; 250
// sets of 2,048 unknowns in FP64 6,600 -> 385 us; 1,024 sets of 1,022 unknowns in
// mixed precision, beside the fill of the final vectors, 2,130 -> 453 us.

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

__global__ __launch_bounds__(sblock) void k_rb_fill(int64_t nU, int null_code, const int32_t* __restrict__ row,
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
			r[k] = (uint32_t)null_code << 25;
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
__device__ __forceinline__ double rb_sum(const uint4* __restrict__ rec, const double* __restrict__ rates, uint32_t h,
										 const double* __restrict__ y, double s)
{
	const int g1 = (int)(h & 0xffffff) + (int)(h >> 24);
	for (int g = (int)(h & 0xffffff); g < g1; ++g)
	{
		const uint4 q = rec[g];
		const double r0 = rates[rb_code(q.x)], r1 = rates[rb_code(q.y)];
		const double r2 = rates[rb_code(q.z)], r3 = rates[rb_code(q.w)];
		const double y0 = y[q.x & rb_index], y1 = y[q.y & rb_index];
		const double y2 = y[q.z & rb_index], y3 = y[q.w & rb_index];
		// the eight loads together: one LDS round trip per group instead of one per term
		__builtin_amdgcn_sched_barrier(0);
		s += r0 * y0;
		s += r1 * y1;
		s += r2 * y2;
		s += r3 * y3;
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

// A cycle ends at a tenth of the tolerance: aiming at the tolerance itself leaves
// the residual just below it, and the extra decade costs one product in twelve and
// keeps the error of the result below what GMRES left.
constexpr double rb_aim = 0.1;

// A cycle also ends when rho, the product of the residual with the shadow vector, is no
// more than this part of their norms: its bits are rounding then, and so are the steps
// made of it.  Such cycles crept or diverged until they ran out of products: the slowest
// of 257 sets of 11,772 undecided states took 1,004 products and takes 178 now, the call
// 37.4 and 9.1 ms (13.4 with GMRES).  On 80 networks, 8 of them with such sets at all, no
// mean number of products grew.
constexpr double rb_lost = 1e-16;

constexpr int rb_max_fails = 3;		 // cycles without progress before a set is left to GMRES
constexpr int rb_cycle_products = 500; // products by S per cycle, so that rounding cannot drift for long

// What a solve that starts from the rates alone sets up by itself: the anchors
// [B][n_seg], and from them 1 / D' and the right-hand side that other methods and
// checks read.  Anchors that turn out to be bad are moved there too.
struct rb_setup_t
{
	const double* x0; // [2^N]; null: anchors, 1 / D', right-hand side and start vector are given
	const int32_t* seg_off;
	int n_seg;
	int32_t* anchor;
	double *invd, *rhs;
	const double* warm;	 // [B][n_t] predicted final vectors on the terminal states, or null
	const int32_t* tpos; // terminal unknown -> its place there
	int64_t n_t;
	const int32_t* only; // per set: whether the per-set kernel solves it; null: all
	// mass that the sweeps start from on a terminal unknown
	__device__ __forceinline__ double mass(int b, int32_t u) const
	{
		return warm ? fmax(warm[(int64_t)b * n_t + tpos[u]], 0.0) : 1.0;
	}
};

// Anchor sweeps: damped Jacobi sweeps (as in k_anchor_sweep) taken class by class.
// E rows: m = inflow / D; R rows: m = (m + inflow / D) / 2.  One pair moves the mass
// as far as two sweeps over all rows, so half as many do.  They start from equal
// masses or from a prediction, which they smooth (a stationary vector stays as it is).
// Inside the solve kernel, on the records it holds anyway, they and the set-up cost
// 10 us of its 98 (one set of 1,022 unknowns) where the anchor kernel took 78 and the
// set-up 6; 250 sets of 2,048 unknowns: 0 of 384 against 180 and 10.
constexpr int rb_sweeps = 16;

// the largest mass of the workgroup and its unknown, ties to the smallest unknown
template <int BLK>
__device__ __forceinline__ void rb_block_argmax(double& v, int32_t& u, double* s_v, int32_t* s_u)
{
#pragma unroll
	for (int o = wave / 2; o > 0; o >>= 1)
	{
		const double v2 = __shfl_xor(v, o, wave);
		const int32_t u2 = __shfl_xor(u, o, wave);
		if (v2 > v || (v2 == v && u2 < u))
		{
			v = v2;
			u = u2;
		}
	}
	if constexpr (BLK > wave)
	{
		__syncthreads();
		if (lane_id() == 0)
		{
			s_v[threadIdx.x / wave] = v;
			s_u[threadIdx.x / wave] = u;
		}
		__syncthreads();
		for (int w = 0; w < BLK / wave; ++w)
			if (s_v[w] > v || (s_v[w] == v && s_u[w] < u))
			{
				v = s_v[w];
				u = s_u[w];
			}
	}
}

// One workgroup of BLK threads solves one rate set; thread t owns the rows
// t + i BLK (i < RPT) of both classes.  LREC: the coupling records are copied to
// LDS, else they are read from global memory (shared by all sets, so from L2).
template <int BLK, int RPT, bool LREC>
__device__ __forceinline__ void bicg_set_body(const sys_t& S, const rb_t& G, int n_seg, const double* __restrict__ rhs,
											  double* __restrict__ zio, const rb_scratch_t& sc,
											  const rb_setup_t& su, double tol, int max_iters, const pgm_out_t& out)
{
	extern __shared__ __align__(16) unsigned char smem[];
	__shared__ double s_part[2][rb_part];
	__shared__ double s_rates[64];
	const int b = blockIdx.x, tid = threadIdx.x;
	if (su.only && !su.only[b])
		return;
	const uint64_t t_begin = wall_clock64();
	const int nE = G.nE, nR = G.nR, nU = nE + nR;
	const int64_t off = (int64_t)b * nU;
	double* s_g = (double*)smem;	 // [nR] the vector being multiplied
	double* s_te = s_g + nR;	 // [nE] its image on the eliminated rows
	uint4* s_rec = (uint4*)(smem + ((size_t)nU * sizeof(double) + 15) / 16 * 16);
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
	auto groups_of = [&](int q) { return (uint32_t)G.ptr[q] | (uint32_t)(G.ptr[q + 1] - G.ptr[q]) << 24; };
	if (su.x0)
	{
		// from the rates alone: the anchor of a segment is its row of largest mass
		// after the sweeps, and the masses relative to it are the start vector (a start
		// from the anchor alone leaves a residual with one or two nonzeros, on which
		// the first cycle breaks down); undecided states start from zero
		int32_t uE[RPT], uR[RPT], kE[RPT], kR[RPT];
		__syncthreads(); // the rates
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int e = tid + i * BLK;
			hE[i] = hR[i] = 0;
			cE[i] = dR[i] = 0.0;
			kE[i] = kR[i] = -1;
			if (e < nE)
			{
				uE[i] = G.row[e];
				kE[i] = S.ucls[uE[i]];
				const uint32_t st = (uint32_t)S.ulist[uE[i]];
				cE[i] = 1.0 / out_rate_s(st, S.mask[st], s_rates);
				hE[i] = groups_of(e);
			}
			if (e < nR)
			{
				uR[i] = G.row[nE + e];
				kR[i] = S.ucls[uR[i]];
				const uint32_t st = (uint32_t)S.ulist[uR[i]];
				dR[i] = out_rate_s(st, S.mask[st], s_rates);
				hR[i] = groups_of(nE + e);
				s_g[e] = kR[i] >= 0 ? su.mass(b, uR[i]) : 0.0;
			}
		}
		__syncthreads();
		for (int it = 0; it < (su.n_seg ? rb_sweeps : 0); ++it)
		{
#pragma unroll
			for (int i = 0; i < RPT; ++i)
				if (tid + i * BLK < nE)
					s_te[tid + i * BLK] = cE[i] * rb_sum(rec, s_rates, hE[i], s_g, 0.0);
			__syncthreads();
#pragma unroll
			for (int i = 0; i < RPT; ++i)
				if (tid + i * BLK < nR)
				{
					const int o = tid + i * BLK;
					s_g[o] = 0.5 * s_g[o] + 0.5 * (rb_sum(rec, s_rates, hR[i], s_te, 0.0) / dR[i]);
				}
			__syncthreads();
		}
		// undecided states
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int e = tid + i * BLK;
			if (e < nE && kE[i] < 0)
			{
				const double r = su.x0[S.ulist[uE[i]]];
				su.invd[off + uE[i]] = cE[i];
				su.rhs[off + uE[i]] = bp[e] = r;
				xp[e] = 0.0;
				bb += r * r;
			}
			if (e < nR && kR[i] < 0)
			{
				const double r = su.x0[S.ulist[uR[i]]];
				su.invd[off + uR[i]] = 1.0 / dR[i];
				su.rhs[off + uR[i]] = bp[nE + e] = r;
				xp[nE + e] = 0.0;
				bb += r * r;
			}
		}
		// segments
		for (int k = 0; k < su.n_seg; ++k)
		{
			double best = -1.0;
			int32_t bu = INT32_MAX;
#pragma unroll
			for (int i = 0; i < RPT; ++i)
			{
				const int e = tid + i * BLK;
				if (kE[i] == k && (s_te[e] > best || (s_te[e] == best && uE[i] < bu)))
				{
					best = s_te[e];
					bu = uE[i];
				}
				if (kR[i] == k && (s_g[e] > best || (s_g[e] == best && uR[i] < bu)))
				{
					best = s_g[e];
					bu = uR[i];
				}
			}
			rb_block_argmax<BLK>(best, bu, s_part[0], (int32_t*)s_part[1]);
			if (tid == 0)
				su.anchor[(int64_t)b * su.n_seg + k] = bu;
			const double inv = best > 0.0 ? 1.0 / best : 0.0;
#pragma unroll
			for (int i = 0; i < RPT; ++i)
			{
				const int e = tid + i * BLK;
				if (kE[i] == k)
				{
					const bool anc = uE[i] == bu;
					if (anc)
					{
						hE[i] = 0;
						cE[i] = 1.0;
						bb += 1.0;
					}
					xp[e] = anc ? 1.0 : s_te[e] * inv;
					su.invd[off + uE[i]] = cE[i];
					su.rhs[off + uE[i]] = bp[e] = anc ? 1.0 : 0.0;
				}
				if (kR[i] == k)
				{
					const bool anc = uR[i] == bu;
					if (anc)
					{
						hR[i] = 0;
						dR[i] = 1.0;
						bb += 1.0;
					}
					xp[nE + e] = anc ? 1.0 : s_g[e] * inv;
					su.invd[off + uR[i]] = 1.0 / dR[i];
					su.rhs[off + uR[i]] = bp[nE + e] = anc ? 1.0 : 0.0;
				}
			}
		}
		__syncthreads();
	}
	else
	{
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int e = tid + i * BLK;
			hE[i] = hR[i] = 0;
			cE[i] = dR[i] = 0.0;
			for (int cls = 0; cls < 2; ++cls)
			{
				if (e >= (cls ? nR : nE))
					continue;
				const int q = cls ? nE + e : e, u = G.row[q];
				const uint32_t h = is_anchor(S, n_seg, b, u) ? 0u : groups_of(q);
				const double iv = S.invd[off + u], r = rhs[off + u];
				if (cls)
				{
					hR[i] = h;
					dR[i] = 1.0 / iv;
				}
				else
				{
					hE[i] = h;
					cE[i] = iv;
				}
				xp[q] = zio[off + u] * iv;
				bp[q] = r;
				bb += r * r;
			}
		}
		__syncthreads();
	}
	// diag(S): D less what leaves the row and comes straight back (not through an
	// anchor, whose row takes nothing in)
#pragma unroll
	for (int i = 0; i < RPT; ++i)
		if (tid + i * BLK < nE)
			s_te[tid + i * BLK] = hE[i] >> 24 ? cE[i] : 0.0;
	__syncthreads();
#pragma unroll
	for (int i = 0; i < RPT; ++i)
	{
		jR[i] = 0.0;
		if (tid + i * BLK < nR)
		{
			double d = dR[i];
			const int g1 = (int)(hR[i] & 0xffffff) + (int)(hR[i] >> 24);
			for (int g = (int)(hR[i] & 0xffffff); g < g1; ++g)
			{
				const uint4 q = rec[g];
				const uint32_t qq[4] = { q.x, q.y, q.z, q.w };
#pragma unroll
				for (int k = 0; k < 4; ++k)
					if (qq[k] >> 31)
						d -= s_rates[rb_code(qq[k])] * s_rates[rb_code(qq[k]) ^ 1] * s_te[qq[k] & rb_index];
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
		++cycles;
		const double inv_beta = 1.0 / beta;
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int e = tid + i * BLK;
			if (e < nE)
				s_te[e] = cE[i] * rEp[e] * inv_beta;
		}
		__syncthreads();
		double r[RPT], rh[RPT], p[RPT], v[RPT], x[RPT];
		double s2[3] = { 0.0, 0.0, 0.0 };
#pragma unroll
		for (int i = 0; i < RPT; ++i)
		{
			const int o = tid + i * BLK;
			r[i] = jR[i] * rb_sum(rec, s_rates, hR[i], s_te, ro[i] * inv_beta);
			rh[i] = o < nR ? rb_shadow(o, fails, r[i]) : 0.0;
			p[i] = r[i];
			x[i] = 0.0;
			s2[0] += r[i] * r[i];
			s2[1] += rh[i] * r[i];
			s2[2] += rh[i] * rh[i];
		}
		rb_block_sums<BLK>(s2, s_part[1]);
		double rho = s2[1];
		const double lost2 = rb_lost * rb_lost * s2[2];
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
					s_te[tid + i * BLK] = cE[i] * rb_sum(rec, s_rates, hE[i], s_g, 0.0);
			__syncthreads();
			double s1[1] = { 0.0 };
#pragma unroll
			for (int i = 0; i < RPT; ++i)
			{
				v[i] = jR[i] * (dR[i] * p[i] - rb_sum(rec, s_rates, hR[i], s_te, 0.0));
				s1[0] += rh[i] * v[i];
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
				r[i] -= alpha * v[i];
				if (tid + i * BLK < nR)
					s_g[tid + i * BLK] = r[i];
			}
			__syncthreads();
#pragma unroll
			for (int i = 0; i < RPT; ++i)
				if (tid + i * BLK < nE)
					s_te[tid + i * BLK] = cE[i] * rb_sum(rec, s_rates, hE[i], s_g, 0.0);
			__syncthreads();
			double t[RPT];
#pragma unroll
			for (int k = 0; k < 5; ++k)
				sums[k] = 0.0;
#pragma unroll
			for (int i = 0; i < RPT; ++i)
			{
				t[i] = jR[i] * (dR[i] * r[i] - rb_sum(rec, s_rates, hR[i], s_te, 0.0));
				const double td = t[i], sd = r[i], hd = rh[i];
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
			// without branches, so that it is done beside the updates below
			const bool stop = (sqrt(rr2) * est <= rb_aim * tol) | (omega == 0.0) | !rb_finite(beta_b) | (beta_b == 0.0) |
							  (rho1 * rho1 <= lost2 * rr2) | (iters >= max_iters);
			rho = rho1;
#pragma unroll
			for (int i = 0; i < RPT; ++i)
			{
				x[i] += alpha * p[i] + omega * r[i];
				r[i] -= omega * t[i];
				p[i] = r[i] + beta_b * (p[i] - omega * v[i]);
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
				xp[nE + o] = x0 + beta * x[i];
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

template <int BLK, int RPT, bool LREC>
__global__ __launch_bounds__(BLK, 4) void k_bicg_set(
	sys_t S, rb_t G, int n_seg, const double* __restrict__ rhs, double* __restrict__ zio, rb_scratch_t sc, rb_setup_t su,
	double tol, int max_iters, pgm_out_t out)
{
	bicg_set_body<BLK, RPT, LREC>(S, G, n_seg, rhs, zio, sc, su, tol, max_iters, out);
}

// Moves bad anchors, for the sets above the tolerance.  A segment's solution is scaled
// to 1 at its anchor, the row of largest mass after the sweeps.  Where the rates part
// a segment into regions that exchange little mass, the sweeps can end before the mass
// has settled; the anchor is then a row with a thousandth of the largest entry or
// less, and the rounding of D x alone keeps the residual, which is relative to the
// anchor's 1, above a tolerance of 1e-12 (about two sets in a million of 2,048 unknowns
// with log-uniform rates in [0.1, 10]: entries of 700 to 6,600 times the anchor's).
// No method gets below that; the same iterate divided by its largest entry, with the
// anchor there, has a residual of 1e-15.  Rare, so in a kernel of its own, one
// workgroup per set, on the set-major vectors.
constexpr double rb_bad_anchor = 2.0; // an anchor is moved to an entry more than this many times its own
__global__ __launch_bounds__(sblock) void k_rb_move(sys_t S, rb_setup_t su, const double* __restrict__ res, double tol,
													double* __restrict__ z, int32_t* __restrict__ moved)
{
	__shared__ double s_v[sblock / wave];
	__shared__ int32_t s_u[sblock / wave];
	const int b = blockIdx.x, tid = threadIdx.x;
	const int64_t off = (int64_t)b * S.nU;
	int any = 0;
	for (int k = 0; k < su.n_seg && !(res[b] <= tol); ++k)
	{
		const int32_t old = su.anchor[(int64_t)b * su.n_seg + k], u1 = su.seg_off[k + 1];
		double best = -1.0;
		int32_t bu = INT32_MAX;
		for (int32_t u = su.seg_off[k] + tid; u < u1; u += sblock)
		{
			const double x = z[off + u] * su.invd[off + u];
			if (x > best)
			{
				best = x;
				bu = u;
			}
		}
		rb_block_argmax<sblock>(best, bu, s_v, s_u);
		if (!(best > rb_bad_anchor) || !rb_finite(best) || bu == old)
			continue;
		any = 1;
		for (int32_t u = su.seg_off[k] + tid; u < u1; u += sblock)
		{
			const double v = z[off + u] / best;
			z[off + u] = v;
			if (u == old)
			{
				const uint32_t st = (uint32_t)S.ulist[u];
				const double d = out_rate_s(st, S.mask[st], S.rates + (int64_t)b * S.rate_stride);
				z[off + u] = v * d; // D' was 1 here
				su.invd[off + u] = 1.0 / d;
				su.rhs[off + u] = 0.0;
			}
			if (u == bu)
				z[off + u] = su.invd[off + u] = su.rhs[off + u] = 1.0;
		}
		if (tid == 0)
			su.anchor[(int64_t)b * su.n_seg + k] = bu;
	}
	if (tid == 0)
		moved[b] = any;
}

// For GMRES to take over the sets above the tolerance: zero for them and, where `invd` is
// given, 1 / D' as GMRES sets it up (the device-wide solver's differs in the last bit),
// other iterates kept.  It then starts as where it is asked for by name, so it meets a
// bound on its iterations, or a tolerance near the rounding, as it does there.
__global__ __launch_bounds__(sblock) void k_rb_restart(sys_t S, int n_seg, const double* __restrict__ res, double tol,
													   double* __restrict__ z, double* __restrict__ invd)
{
	const int64_t u = (int64_t)blockIdx.x * sblock + threadIdx.x;
	const int b = blockIdx.y;
	if (u >= S.nU)
		return;
	const int64_t i = (int64_t)b * S.nU + u;
	const bool left = !(res[b] <= tol);
	if (!invd)
	{
		if (left)
			z[i] = 0.0;
		return;
	}
	const uint32_t st = (uint32_t)S.ulist[u];
	const double x = z[i] * invd[i];
	const double iv =
		is_anchor(S, n_seg, b, u) ? 1.0 : 1.0 / out_rate_s(st, S.mask[st], S.rates + (int64_t)b * S.rate_stride);
	invd[i] = iv;
	z[i] = left ? 0.0 : x / iv;
}

using bicg_set_fn = void (*)(sys_t, rb_t, int, const double*, double*, rb_scratch_t, rb_setup_t, double, int, pgm_out_t);
struct bicg_variant_t
{
	bicg_set_fn fn;
	int blk, rows; // threads, rows of the larger class at most
	bool lrec;
};

// The variants, smallest first.  A batch of more sets than compute units takes
// two rows per thread, so that several sets share a CU; up to that many sets
// each has a CU to itself, and one row per thread shortens its chain.  One row / two
// rows, us per call: 2,048 unknowns 390 / 411 for 256 sets, 462 / 417 for 257, 1,107 / 880
// for 1,024; 936 unknowns, whose sets share a CU either way, 221 / 258 for 256, 230 / 260
// for 512, 303 / 288 for 1,024; 696 unknowns 227 / 296, 266 / 299, 476 / 428.
constexpr int rb_cus = 256; // of the MI355X
constexpr size_t rb_lds_static = 3072; // upper bound of the kernel's static LDS
// dynamic LDS of one set: the vector being multiplied, its image, the records
inline size_t rb_lds_bytes(int64_t nU, int64_t groups, bool lrec)
{
	return ((size_t)nU * 8 + 15) / 16 * 16 + (lrec ? (size_t)groups * 16 : 0);
}
inline const bicg_variant_t* rb_variant(int64_t nE, int64_t nR, int64_t groups, int B, size_t lds_max)
{
#define ESL_RB(BLK, RPT, LREC)                                                                                       \
	{ k_bicg_set<BLK, RPT, LREC>, BLK, BLK * RPT, LREC }
	static const bicg_variant_t few[] = { ESL_RB(64, 1, true),	 ESL_RB(256, 1, true),	 ESL_RB(512, 1, true),
										  ESL_RB(1024, 1, true), ESL_RB(1024, 2, false), ESL_RB(1024, 4, false) };
	static const bicg_variant_t many[] = { ESL_RB(64, 2, true), ESL_RB(256, 2, true), ESL_RB(512, 2, true),
										   ESL_RB(1024, 2, false), ESL_RB(1024, 4, false) };
#undef ESL_RB
	const int64_t rows = nE > nR ? nE : nR;
	auto pick = [&](const bicg_variant_t* v, int n) -> const bicg_variant_t* {
		for (int i = 0; i < n; ++i)
			if (rows <= v[i].rows && rb_lds_bytes(nE + nR, groups, v[i].lrec) + rb_lds_static <= lds_max)
				return v + i;
		return nullptr;
	};
	return B <= rb_cus ? pick(few, sizeof few / sizeof *few) : pick(many, sizeof many / sizeof *many);
}

// ============================================================================
// The same method device-wide, for systems too large for one workgroup.  Vectors
// are [row][set] with rows in class order; a lane takes W (2, or 1 for an odd batch)
// neighbouring sets of a row, a block up to 64 sets of R rows at a time.  A row's
// records are read once per set pair, its neighbours' values are contiguous
// 16-byte loads, and the rates of the block's sets sit in LDS.  A block owns a
// contiguous range of rows, and blocks are dealt to the eight XCDs in contiguous
// runs: most neighbours of a row (its low bits) then lie in what the same XCD's L2
// holds.  Two products by S are eight launches and no host round trip; a step of
// GMRES with ILU(0) was two launches per popcount level, a product by M and two
// passes over up to 32 basis vectors.  Measured: 64 sets of 221,184 unknowns 138 ms
// -> 59 ms, 16 sets of 524,288 unknowns 73 -> 24 ms.  Bound: the products' gathers
// (64 sets of 221,184 unknowns: 78 us for 113 MB of compulsory vectors and eleven
// neighbours a row), then the vector updates at 7 TB/s through the Infinity Cache.
// One set per lane with rates from global memory took 110 us.

constexpr int rbw_threads = 256; // threads of a block at most
constexpr int rbw_sets = 64;	 // sets of a block at most

struct rbw_geo_t
{
	int B, bs, L, R; // sets, sets per block, lanes per row, rows per step; block = L * R threads
	int ncode;		 // 2N
	const double* rates;
	int64_t rstride;
};

// contiguous share of `rows` for this block; XCD i (blockIdx.x % 8) gets the i-th eighth of the blocks
__device__ __forceinline__ void rbw_rows(int64_t rows, int64_t& q0, int64_t& q1)
{
	const int64_t nb = gridDim.x;
	int64_t k = blockIdx.x;
	if (nb % 8 == 0)
		k = (k % 8) * (nb / 8) + k / 8;
	q0 = rows * k / nb;
	q1 = rows * (k + 1) / nb;
}

// the thread's row of a step, its first set, and whether that set exists (W divides B)
#define ESL_RBW_THREAD                                                                                               \
	const int t_row = (int)threadIdx.x / geo.L, bl = (int)threadIdx.x % geo.L * W;                                   \
	const int b = (int)blockIdx.y * geo.bs + bl, B = geo.B;                                                          \
	const bool in = bl < geo.bs && b < B

template <int W>
struct rbw_vec_t
{
	double v[W];
};
template <int W>
__device__ __forceinline__ rbw_vec_t<W> rbw_load(const double* __restrict__ p)
{
	rbw_vec_t<W> r;
	if constexpr (W == 2)
	{
		const double2 d = *(const double2*)p;
		r.v[0] = d.x;
		r.v[1] = d.y;
	}
	else
		r.v[0] = *p;
	return r;
}
template <int W>
__device__ __forceinline__ void rbw_store(double* __restrict__ p, const rbw_vec_t<W>& r)
{
	if constexpr (W == 2)
		*(double2*)p = make_double2(r.v[0], r.v[1]);
	else
		*p = r.v[0];
}

// rates of the block's sets into LDS, [code][set of the block]; code 2N (null records) is zero
__device__ __forceinline__ double* rbw_lds_rates(const rbw_geo_t& geo)
{
	extern __shared__ __align__(16) unsigned char smem[];
	double* s = (double*)smem;
	for (int i = threadIdx.x; i < (geo.ncode + 1) * geo.bs; i += blockDim.x)
	{
		const int k = i % geo.bs, code = i / geo.bs, b = (int)blockIdx.y * geo.bs + k;
		s[i] = code < geo.ncode && b < geo.B ? geo.rates[(int64_t)b * geo.rstride + code] : 0.0;
	}
	__syncthreads();
	return s;
}

// sum over the couplings of row q for W sets; the next group's records are loaded
// while this one's values are
template <int W>
__device__ __forceinline__ rbw_vec_t<W> rbw_sum(const rb_t& G, int64_t q, int b, int bl, const rbw_geo_t& geo,
												const double* __restrict__ rt, const double* __restrict__ y)
{
	rbw_vec_t<W> s{};
	int g = G.ptr[q];
	const int g1 = G.ptr[q + 1];
	uint4 c = G.rec[g];
	const double* __restrict__ yb = y + b;
	const double* __restrict__ rb = rt + bl;
	const uint32_t B = (uint32_t)geo.B, bs = (uint32_t)geo.bs;
	while (g < g1)
	{
		const uint4 nx = G.rec[++g];
		const auto y0 = rbw_load<W>(yb + (uint64_t)(c.x & rb_index) * B), y1 = rbw_load<W>(yb + (uint64_t)(c.y & rb_index) * B);
		const auto y2 = rbw_load<W>(yb + (uint64_t)(c.z & rb_index) * B), y3 = rbw_load<W>(yb + (uint64_t)(c.w & rb_index) * B);
		const auto r0 = rbw_load<W>(rb + rb_code(c.x) * bs), r1 = rbw_load<W>(rb + rb_code(c.y) * bs);
		const auto r2 = rbw_load<W>(rb + rb_code(c.z) * bs), r3 = rbw_load<W>(rb + rb_code(c.w) * bs);
#pragma unroll
		for (int w = 0; w < W; ++w)
			s.v[w] += r0.v[w] * y0.v[w] + r1.v[w] * y1.v[w] + (r2.v[w] * y2.v[w] + r3.v[w] * y3.v[w]);
		c = nx;
	}
	return s;
}

// per-set sums of a block: the R partials of a set folded in halves (a fixed
// order), into part[blk][b][k].  Reuses the dynamic LDS from its start.
template <int W, int K>
__device__ __forceinline__ void rbw_block_sums(const rbw_geo_t& geo, const double (&v)[K][W], bool on, int b, int t_row,
											   double* __restrict__ part)
{
	extern __shared__ __align__(16) unsigned char smem[];
	double* s = (double*)smem; // [K][W][blockDim]
	const int nt = blockDim.x;
	__syncthreads();
#pragma unroll
	for (int k = 0; k < K; ++k)
#pragma unroll
		for (int w = 0; w < W; ++w)
			s[(k * W + w) * nt + threadIdx.x] = on ? v[k][w] : 0.0;
	for (int r = geo.R; r > 1;)
	{
		const int h = (r + 1) / 2;
		__syncthreads();
		if (t_row < r - h)
#pragma unroll
			for (int k = 0; k < K * W; ++k)
				s[k * nt + threadIdx.x] += s[k * nt + threadIdx.x + h * geo.L];
		r = h;
	}
	__syncthreads();
	if (t_row == 0 && on)
#pragma unroll
		for (int w = 0; w < W; ++w)
#pragma unroll
			for (int k = 0; k < K; ++k)
				part[((int64_t)blockIdx.x * geo.B + b + w) * K + k] = s[(k * W + w) * nt + threadIdx.x];
}

// state of a set through a cycle
struct rbw_set_t
{
	double rho, alpha, omega, beta; // BiCGStab
	double est;						// |r| -> relative residual
	double lost2;					// square of rb_lost times the norm of the shadow vector
	double scale;					// norm of the FP64 residual (the cycle solves for x / scale)
	int32_t live, upd, fails, pad;
};

// ---- start

// c = 1 / D of every row, and the masses the anchor sweeps start from (0 on
// ambiguous rows)
template <int W>
__global__ void k_rbw_coef(sys_t S, rb_t G, rbw_geo_t geo, rb_setup_t su, double* __restrict__ c,
						   double* __restrict__ mE, double* __restrict__ mR)
{
	const double* rt = rbw_lds_rates(geo);
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(S.nU, q0, q1);
	if (!in)
		return;
	for (int64_t q = q0 + t_row; q < q1; q += geo.R)
	{
		const int32_t u = G.row[q];
		const uint32_t s = (uint32_t)S.ulist[u];
		rbw_vec_t<W> d{}, m;
		for (uint32_t k = S.mask[s]; k; k &= k - 1)
		{
			const int i = __ffs(k) - 1;
#pragma unroll
			for (int w = 0; w < W; ++w)
				d.v[w] += rt[(2 * i + ((s >> i) & 1u)) * geo.bs + bl + w];
		}
#pragma unroll
		for (int w = 0; w < W; ++w)
		{
			d.v[w] = 1.0 / d.v[w];
			m.v[w] = S.ucls[u] >= 0 ? su.mass(b + w, u) : 0.0;
		}
		rbw_store<W>(c + q * B + b, d);
		rbw_store<W>((q < G.nE ? mE + q * B : mR + (q - G.nE) * B) + b, m);
	}
}

// one class of an anchor sweep (rb_sweeps)
template <int W, bool KEPT>
__global__ void k_rbw_sweep(rb_t G, rbw_geo_t geo, const double* __restrict__ c, const double* __restrict__ from,
							double* __restrict__ to)
{
	const double* rt = rbw_lds_rates(geo);
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(KEPT ? G.nR : G.nE, q0, q1);
	if (!in)
		return;
	for (int64_t o = q0 + t_row; o < q1; o += geo.R)
	{
		const int64_t q = KEPT ? G.nE + o : o;
		auto s = rbw_sum<W>(G, q, b, bl, geo, rt, from);
		const auto cc = rbw_load<W>(c + q * B + b);
		rbw_vec_t<W> m{};
		if (KEPT)
			m = rbw_load<W>(to + o * B + b);
#pragma unroll
		for (int w = 0; w < W; ++w)
			s.v[w] = KEPT ? 0.5 * m.v[w] + 0.5 * (cc.v[w] * s.v[w]) : cc.v[w] * s.v[w];
		rbw_store<W>(to + o * B + b, s);
	}
}

// index inside its class of the first unknown >= u, for each segment's bounds:
// off[0][k] eliminated rows, off[1][k] kept rows
__global__ __launch_bounds__(sblock) void k_rbw_seg_rows(rb_t G, int n_seg, const int32_t* __restrict__ seg_off,
														 int32_t* __restrict__ off)
{
	const int k = blockIdx.x * sblock + threadIdx.x;
	if (k > n_seg)
		return;
	for (int cls = 0; cls < 2; ++cls)
	{
		// rows of a class ascend in the unknowns
		const int32_t* r = G.row + (cls ? G.nE : 0);
		int lo = 0, hi = cls ? G.nR : G.nE;
		while (lo < hi)
		{
			const int mid = (lo + hi) / 2;
			if (r[mid] < seg_off[k])
				lo = mid + 1;
			else
				hi = mid;
		}
		off[cls * (n_seg + 1) + k] = lo;
	}
}

// largest mass of a slice of a segment per set, ties to the smallest unknown:
// block (segment and slice, set chunk) -> pv / pu[slice][seg][b]
template <int W>
__global__ void k_rbw_pick(rb_t G, rbw_geo_t geo, int n_seg, int slices, const int32_t* __restrict__ off,
						   const double* __restrict__ mE, const double* __restrict__ mR, double* __restrict__ pv,
						   int32_t* __restrict__ pu)
{
	extern __shared__ __align__(16) unsigned char smem[];
	ESL_RBW_THREAD;
	const int k = blockIdx.x / slices, sl = blockIdx.x % slices, nt = blockDim.x;
	double* s_v = (double*)smem;				   // [W][blockDim]
	int32_t* s_u = (int32_t*)(s_v + W * nt); // [W][blockDim]
	double best[W];
	int32_t bu[W];
#pragma unroll
	for (int w = 0; w < W; ++w)
	{
		best[w] = -1.0;
		bu[w] = INT32_MAX;
	}
	for (int cls = 0; cls < 2 && in; ++cls)
	{
		const int64_t a = off[cls * (n_seg + 1) + k], n = off[cls * (n_seg + 1) + k + 1] - a;
		const int64_t o0 = a + n * sl / slices, o1 = a + n * (sl + 1) / slices;
		for (int64_t o = o0 + t_row; o < o1; o += geo.R)
		{
			const auto m = rbw_load<W>((cls ? mR : mE) + o * B + b);
			const int32_t u = G.row[cls ? G.nE + o : o];
#pragma unroll
			for (int w = 0; w < W; ++w)
				if (m.v[w] > best[w] || (m.v[w] == best[w] && u < bu[w]))
				{
					best[w] = m.v[w];
					bu[w] = u;
				}
		}
	}
#pragma unroll
	for (int w = 0; w < W; ++w)
	{
		s_v[w * nt + threadIdx.x] = best[w];
		s_u[w * nt + threadIdx.x] = bu[w];
	}
	__syncthreads();
	if (t_row == 0 && in)
#pragma unroll
		for (int w = 0; w < W; ++w)
		{
			for (int r = 1; r < geo.R; ++r)
			{
				const double v = s_v[w * nt + threadIdx.x + r * geo.L];
				const int32_t u = s_u[w * nt + threadIdx.x + r * geo.L];
				if (v > best[w] || (v == best[w] && u < bu[w]))
				{
					best[w] = v;
					bu[w] = u;
				}
			}
			const int64_t at = ((int64_t)sl * n_seg + k) * B + b + w;
			pv[at] = best[w];
			pu[at] = bu[w];
		}
}

// slices -> anchor[b][seg] and its mass pa[seg][b].  Where anchors are moved (k_rb_move;
// `only` null otherwise) for the sets of `only`: bad ones are replaced and the set
// marked in `moved`, the others' mass is 1.
__global__ __launch_bounds__(sblock) void k_rbw_anchor(int B, int n_seg, int slices, const double* __restrict__ pv,
													   const int32_t* __restrict__ pu, int32_t* __restrict__ anchor,
													   double* __restrict__ pa, const int32_t* __restrict__ only,
													   int32_t* __restrict__ moved)
{
	const int i = blockIdx.x * sblock + threadIdx.x;
	if (i >= n_seg * B)
		return;
	const int k = i / B, b = i - k * B;
	if (only && !only[b])
		return;
	double best = -1.0;
	int32_t bu = INT32_MAX;
	for (int s = 0; s < slices; ++s)
	{
		const int64_t at = ((int64_t)s * n_seg + k) * B + b;
		if (pv[at] > best || (pv[at] == best && pu[at] < bu))
		{
			best = pv[at];
			bu = pu[at];
		}
	}
	if (only)
	{
		if (!(best > rb_bad_anchor) || !rb_finite(best) || anchor[(int64_t)b * n_seg + k] == bu)
		{
			pa[i] = 1.0;
			return;
		}
		moved[b] = 1;
	}
	anchor[(int64_t)b * n_seg + k] = bu;
	pa[i] = best;
}

// after k_rbw_anchor moved anchors and k_rbw_coef made the coefficients anew: the anchors'
// coefficients of every set, and the iterate and right-hand side of the sets of `only`
template <int W>
__global__ void k_rbw_move(sys_t S, rb_t G, rbw_geo_t geo, int n_seg, const double* __restrict__ pa,
						   const int32_t* __restrict__ only, double* __restrict__ c, double* __restrict__ x,
						   double* __restrict__ wb)
{
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(S.nU, q0, q1);
	if (!in)
		return;
	for (int64_t q = q0 + t_row; q < q1; q += geo.R)
	{
		const int32_t u = G.row[q], k = S.ucls[u];
		if (k < 0)
			continue;
		for (int w = 0; w < W; ++w)
		{
			const int64_t i = q * B + b + w;
			const bool anchor = S.anchor[(int64_t)(b + w) * n_seg + k] == u;
			if (anchor)
				c[i] = 0.0;
			if (only[b + w])
			{
				x[i] = anchor ? 1.0 : x[i] / pa[(int64_t)k * B + b + w];
				wb[i] = anchor ? 1.0 : 0.0;
			}
		}
	}
}

// start vector, right-hand side and anchors (c <- 0: the row is the identity).
// Terminal rows start from their masses relative to the anchor's, ambiguous ones
// from zero.  A start from the anchor alone would leave a residual with one or two
// nonzeros, on which the first cycle breaks down.
template <int W>
__global__ void k_rbw_start(sys_t S, rb_t G, rbw_geo_t geo, int n_seg, const double* __restrict__ x0,
							const double* __restrict__ mE, const double* __restrict__ mR, const double* __restrict__ pa,
							double* __restrict__ c, double* __restrict__ x, double* __restrict__ wb)
{
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(S.nU, q0, q1);
	if (!in)
		return;
	for (int64_t q = q0 + t_row; q < q1; q += geo.R)
	{
		const int32_t u = G.row[q], k = S.ucls[u];
		rbw_vec_t<W> xv{}, bv{};
		if (k < 0)
		{
			const double v = x0[S.ulist[u]];
#pragma unroll
			for (int w = 0; w < W; ++w)
				bv.v[w] = v;
		}
		else
		{
			const auto m = rbw_load<W>((q < G.nE ? mE + q * B : mR + (q - G.nE) * B) + b);
#pragma unroll
			for (int w = 0; w < W; ++w)
			{
				const double p = pa[(int64_t)k * B + b + w];
				xv.v[w] = p > 0.0 ? m.v[w] / p : 0.0;
				if (S.anchor[(int64_t)(b + w) * n_seg + k] == u)
				{
					xv.v[w] = bv.v[w] = 1.0;
					c[q * B + b + w] = 0.0;
				}
			}
		}
		rbw_store<W>(x + q * B + b, xv);
		rbw_store<W>(wb + q * B + b, bv);
	}
}

constexpr int rbw_tile = 32; // rows (and sets) of a transposed tile

// or from a system that is set up: plan vectors (set-major) -> solver vectors, through
// LDS tiles so that both sides are read and written along their rows
__global__ __launch_bounds__(sblock) void k_rbw_enter(sys_t S, rb_t G, int n_seg, const double* __restrict__ rhs,
													  const double* __restrict__ z, double* __restrict__ wx,
													  double* __restrict__ wb, double* __restrict__ wc)
{
	__shared__ double s_x[rbw_tile][rbw_tile + 1], s_b[rbw_tile][rbw_tile + 1], s_c[rbw_tile][rbw_tile + 1];
	const int64_t nU = S.nU, q0 = (int64_t)blockIdx.x * rbw_tile;
	const int b0 = blockIdx.y * rbw_tile, tx = threadIdx.x % rbw_tile, ty = threadIdx.x / rbw_tile;
	constexpr int step = sblock / rbw_tile;
	const int64_t q = q0 + tx;
	const int32_t u = q < nU ? G.row[q] : 0;
	for (int j = ty; j < rbw_tile && q < nU; j += step)
		if (b0 + j < S.B)
		{
			const int b = b0 + j;
			const int64_t o = (int64_t)b * nU + u;
			const double iv = S.invd[o];
			s_x[j][tx] = z[o] * iv;
			s_b[j][tx] = rhs[o];
			s_c[j][tx] = is_anchor(S, n_seg, b, u) ? 0.0 : iv;
		}
	__syncthreads();
	for (int j = ty; j < rbw_tile; j += step)
		if (q0 + j < nU && b0 + tx < S.B)
		{
			const int64_t i = (q0 + j) * S.B + b0 + tx;
			wx[i] = s_x[tx][j];
			wb[i] = s_b[tx][j];
			wc[i] = s_c[tx][j];
		}
}

// z = D' x and 1 / D' (1 for anchors) back into the plan's layout
__global__ __launch_bounds__(sblock) void k_rbw_leave(sys_t S, rb_t G, const double* __restrict__ wx,
													  const double* __restrict__ wc, const double* __restrict__ dj,
													  double* __restrict__ z, double* __restrict__ invd)
{
	__shared__ double s_x[rbw_tile][rbw_tile + 1], s_c[rbw_tile][rbw_tile + 1];
	const int64_t nU = S.nU, q0 = (int64_t)blockIdx.x * rbw_tile;
	const int b0 = blockIdx.y * rbw_tile, tx = threadIdx.x % rbw_tile, ty = threadIdx.x / rbw_tile;
	constexpr int step = sblock / rbw_tile;
	for (int j = ty; j < rbw_tile; j += step)
		if (q0 + j < nU && b0 + tx < S.B)
		{
			const int64_t i = (q0 + j) * S.B + b0 + tx;
			double cc = wc[i];
			if (cc != 0.0 && q0 + j >= G.nE)
				cc /= dj[i - (int64_t)G.nE * S.B]; // J / (D J)
			s_x[j][tx] = wx[i];
			s_c[j][tx] = cc != 0.0 ? cc : 1.0;
		}
	__syncthreads();
	const int64_t q = q0 + tx;
	const int32_t u = q < nU ? G.row[q] : 0;
	for (int j = ty; j < rbw_tile && q < nU; j += step)
		if (b0 + j < S.B)
		{
			const int64_t o = (int64_t)(b0 + j) * nU + u;
			z[o] = s_x[tx][j] / s_c[tx][j];
			if (invd)
				invd[o] = s_c[tx][j];
		}
}

// kept rows: J = 1 / diag(S) in place of 1 / D (0 for an anchor), and D J (1 for an anchor)
template <int W>
__global__ void k_rbw_diag(rb_t G, rbw_geo_t geo, double* __restrict__ c, double* __restrict__ dj)
{
	const double* rt = rbw_lds_rates(geo);
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(G.nR, q0, q1);
	if (!in)
		return;
	for (int64_t o = q0 + t_row; o < q1; o += geo.R)
	{
		const int64_t q = G.nE + o;
		auto cc = rbw_load<W>(c + q * B + b);
		rbw_vec_t<W> back{}, dv;
		for (int g = G.ptr[q]; g < G.ptr[q + 1]; ++g)
		{
			const uint4 r4 = G.rec[g];
			const uint32_t r[4] = { r4.x, r4.y, r4.z, r4.w };
#pragma unroll
			for (int k = 0; k < 4; ++k)
				if (r[k] >> 31) // an anchor's coefficient is zero, so its mirrored entry counts nothing
				{
					const auto ce = rbw_load<W>(c + (int64_t)(r[k] & rb_index) * B + b);
#pragma unroll
					for (int w = 0; w < W; ++w)
						back.v[w] += rt[rb_code(r[k]) * geo.bs + bl + w] * rt[(rb_code(r[k]) ^ 1) * geo.bs + bl + w] * ce.v[w];
				}
		}
#pragma unroll
		for (int w = 0; w < W; ++w)
		{
			const bool anchor = cc.v[w] == 0.0;
			const double D = 1.0 / cc.v[w], d = D - back.v[w];
			const double J = 1.0 / (d > 0.0 ? d : D);
			cc.v[w] = anchor ? 0.0 : J;
			dv.v[w] = anchor ? 1.0 : D * J;
		}
		rbw_store<W>(c + q * B + b, cc);
		rbw_store<W>(dj + o * B + b, dv);
	}
}

// ---- cycles

// FP64 residual of every row; partial sums of r^2 and b^2
template <int W>
__global__ void k_rbw_residual(rb_t G, rbw_geo_t geo, const double* __restrict__ c, const double* __restrict__ dj,
							   const double* __restrict__ wb, const double* __restrict__ x, double* __restrict__ r,
							   double* __restrict__ part)
{
	const double* rt = rbw_lds_rates(geo);
	ESL_RBW_THREAD;
	const int64_t nE = G.nE, nU = nE + G.nR;
	int64_t q0, q1;
	rbw_rows(nU, q0, q1);
	double sum[2][W] = {};
	if (in)
		for (int64_t q = q0 + t_row; q < q1; q += geo.R)
		{
			const int64_t i = q * B + b;
			const auto cc = rbw_load<W>(c + i), bv = rbw_load<W>(wb + i), xv = rbw_load<W>(x + i);
			const auto s = rbw_sum<W>(G, q, b, bl, geo, rt, q < nE ? x + nE * B : x);
			rbw_vec_t<W> d, res;
			if (q >= nE)
				d = rbw_load<W>(dj + i - nE * B);
#pragma unroll
			for (int w = 0; w < W; ++w)
			{
				const double D = q < nE ? 1.0 / cc.v[w] : d.v[w] / cc.v[w];
				res.v[w] = cc.v[w] != 0.0 ? bv.v[w] - (D * xv.v[w] - s.v[w]) : bv.v[w] - xv.v[w];
				sum[0][w] += res.v[w] * res.v[w];
				sum[1][w] += bv.v[w] * bv.v[w];
			}
			rbw_store<W>(r + i, res);
		}
	rbw_block_sums<W, 2>(geo, sum, in, b, t_row, part);
}

// whether any of the thread's sets is in the cycle (others run along, unused)
template <int W>
__device__ __forceinline__ bool rbw_live(const rbw_set_t* __restrict__ st, int b)
{
	bool l = st[b].live != 0;
	if constexpr (W == 2)
		l = l || st[b + 1].live != 0;
	return l;
}

// t_E at the start of a cycle: r_E / (D scale)
template <int W>
__global__ void k_rbw_te0(rb_t G, rbw_geo_t geo, const double* __restrict__ c, const double* __restrict__ r,
						  double* __restrict__ te, const rbw_set_t* __restrict__ st)
{
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(G.nE, q0, q1);
	if (!in || !rbw_live<W>(st, b))
		return;
	double inv[W];
#pragma unroll
	for (int w = 0; w < W; ++w)
		inv[w] = st[b + w].live ? 1.0 / st[b + w].scale : 0.0;
	for (int64_t q = q0 + t_row; q < q1; q += geo.R)
	{
		const int64_t i = q * B + b;
		const auto cc = rbw_load<W>(c + i);
		auto rv = rbw_load<W>(r + i);
#pragma unroll
		for (int w = 0; w < W; ++w)
			rv.v[w] *= (cc.v[w] != 0.0 ? cc.v[w] : 1.0) * inv[w];
		rbw_store<W>(te + i, rv);
	}
}

// start of a cycle: r = J (r_R + A t_E) / scale, shadow vector, p = r, x = 0; sums of r.r, rh.r
// and rh.rh
template <int W>
__global__ void k_rbw_init(rb_t G, rbw_geo_t geo, const double* __restrict__ c, const double* __restrict__ res,
						   const double* __restrict__ te, double* __restrict__ r, double* __restrict__ rh,
						   double* __restrict__ p, double* __restrict__ x, const rbw_set_t* __restrict__ st,
						   double* __restrict__ part)
{
	const double* rt = rbw_lds_rates(geo);
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(G.nR, q0, q1);
	double sum[3][W] = {};
	if (in && rbw_live<W>(st, b))
	{
		double inv[W];
		int fails[W];
#pragma unroll
		for (int w = 0; w < W; ++w)
		{
			inv[w] = st[b + w].live ? 1.0 / st[b + w].scale : 0.0;
			fails[w] = st[b + w].fails;
		}
		for (int64_t o = q0 + t_row; o < q1; o += geo.R)
		{
			const int64_t q = G.nE + o, i = o * B + b;
			const auto J = rbw_load<W>(c + q * B + b), rv = rbw_load<W>(res + q * B + b);
			const auto s = rbw_sum<W>(G, q, b, bl, geo, rt, te);
			rbw_vec_t<W> g, h;
#pragma unroll
			for (int w = 0; w < W; ++w)
			{
				g.v[w] = rv.v[w] * inv[w];
				if (J.v[w] != 0.0)
					g.v[w] = J.v[w] * (g.v[w] + s.v[w]);
				h.v[w] = rb_shadow((int)o, fails[w], g.v[w]);
				sum[0][w] += g.v[w] * g.v[w];
				sum[1][w] += h.v[w] * g.v[w];
				sum[2][w] += h.v[w] * h.v[w];
			}
			rbw_store<W>(r + i, g);
			rbw_store<W>(p + i, g);
			rbw_store<W>(rh + i, h);
			rbw_store<W>(x + i, rbw_vec_t<W>{});
		}
	}
	rbw_block_sums<W, 3>(geo, sum, in, b, t_row, part);
}

// t_E = 1/D (A y) on the eliminated rows
template <int W>
__global__ void k_rbw_te(rb_t G, rbw_geo_t geo, const double* __restrict__ c, const double* __restrict__ y,
						 double* __restrict__ te, const rbw_set_t* __restrict__ st)
{
	const double* rt = rbw_lds_rates(geo);
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(G.nE, q0, q1);
	if (!in || !rbw_live<W>(st, b))
		return;
	for (int64_t q = q0 + t_row; q < q1; q += geo.R)
	{
		const auto cc = rbw_load<W>(c + q * B + b);
		auto s = rbw_sum<W>(G, q, b, bl, geo, rt, y);
#pragma unroll
		for (int w = 0; w < W; ++w)
			s.v[w] *= cc.v[w];
		rbw_store<W>(te + q * B + b, s);
	}
}

// out = J S y on the kept rows.  FULL false: with the sum rh.out (v of the step);
// true: with out.y, out.out, y.y, rh.y, rh.out (t of the step)
template <int W, bool FULL>
__global__ void k_rbw_mul(rb_t G, rbw_geo_t geo, const double* __restrict__ c, const double* __restrict__ dj,
						  const double* __restrict__ te, const double* __restrict__ y, const double* __restrict__ rh,
						  double* __restrict__ out, const rbw_set_t* __restrict__ st, double* __restrict__ part)
{
	constexpr int K = FULL ? 5 : 1;
	const double* rt = rbw_lds_rates(geo);
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(G.nR, q0, q1);
	double sum[K][W] = {};
	if (in && rbw_live<W>(st, b))
		for (int64_t o = q0 + t_row; o < q1; o += geo.R)
		{
			const int64_t q = G.nE + o, i = o * B + b;
			const auto J = rbw_load<W>(c + q * B + b), d = rbw_load<W>(dj + i), yv = rbw_load<W>(y + i),
					   hv = rbw_load<W>(rh + i);
			auto s = rbw_sum<W>(G, q, b, bl, geo, rt, te);
#pragma unroll
			for (int w = 0; w < W; ++w)
			{
				const double t = d.v[w] * yv.v[w] - J.v[w] * s.v[w];
				s.v[w] = t;
				if constexpr (FULL)
				{
					sum[0][w] += t * yv.v[w];
					sum[1][w] += t * t;
					sum[2][w] += yv.v[w] * yv.v[w];
					sum[3][w] += hv.v[w] * yv.v[w];
					sum[4][w] += hv.v[w] * t;
				}
				else
					sum[0][w] += hv.v[w] * t;
			}
			rbw_store<W>(out + i, s);
		}
	rbw_block_sums<W, K>(geo, sum, in, b, t_row, part);
}

// s = r - alpha v, in place
template <int W>
__global__ void k_rbw_s(int64_t nR, rbw_geo_t geo, double* __restrict__ r, const double* __restrict__ v,
						const rbw_set_t* __restrict__ st)
{
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(nR, q0, q1);
	if (!in || !rbw_live<W>(st, b))
		return;
	double alpha[W];
#pragma unroll
	for (int w = 0; w < W; ++w)
		alpha[w] = st[b + w].live ? st[b + w].alpha : 0.0;
	for (int64_t o = q0 + t_row; o < q1; o += geo.R)
	{
		const auto vv = rbw_load<W>(v + o * B + b);
		auto rv = rbw_load<W>(r + o * B + b);
#pragma unroll
		for (int w = 0; w < W; ++w)
			if (alpha[w] != 0.0)
				rv.v[w] -= alpha[w] * vv.v[w];
		rbw_store<W>(r + o * B + b, rv);
	}
}

// x += alpha p + omega s;  r = s - omega t;  p = r + beta (p - omega v)
template <int W>
__global__ void k_rbw_update(int64_t nR, rbw_geo_t geo, double* __restrict__ x, double* __restrict__ r,
							 double* __restrict__ p, const double* __restrict__ v, const double* __restrict__ t,
							 const rbw_set_t* __restrict__ st)
{
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(nR, q0, q1);
	if (!in)
		return;
	bool upd[W], any = false;
	double alpha[W], omega[W], beta[W];
#pragma unroll
	for (int w = 0; w < W; ++w)
	{
		upd[w] = st[b + w].upd != 0;
		any = any || upd[w];
		alpha[w] = st[b + w].alpha;
		omega[w] = st[b + w].omega;
		beta[w] = st[b + w].beta;
	}
	if (!any)
		return;
	for (int64_t o = q0 + t_row; o < q1; o += geo.R)
	{
		const int64_t i = o * B + b;
		auto xv = rbw_load<W>(x + i), rv = rbw_load<W>(r + i), pv = rbw_load<W>(p + i);
		const auto vv = rbw_load<W>(v + i), tv = rbw_load<W>(t + i);
#pragma unroll
		for (int w = 0; w < W; ++w)
			if (upd[w])
			{
				xv.v[w] += alpha[w] * pv.v[w] + omega[w] * rv.v[w];
				rv.v[w] -= omega[w] * tv.v[w];
				pv.v[w] = rv.v[w] + beta[w] * (pv.v[w] - omega[w] * vv.v[w]);
			}
		rbw_store<W>(x + i, xv);
		rbw_store<W>(r + i, rv);
		rbw_store<W>(p + i, pv);
	}
}

// end of a cycle, FP64: KEPT: x_R += scale dx, else x_E += 1/D (r_E + scale A dx);
// keep receives the iterate before
template <int W, bool KEPT>
__global__ void k_rbw_correct(rb_t G, rbw_geo_t geo, const double* __restrict__ c, const double* __restrict__ res,
							  const double* __restrict__ dx, double* __restrict__ x, double* __restrict__ keep,
							  const rbw_set_t* __restrict__ st)
{
	const double* rt = KEPT ? nullptr : rbw_lds_rates(geo);
	ESL_RBW_THREAD;
	int64_t q0, q1;
	rbw_rows(KEPT ? G.nR : G.nE, q0, q1);
	if (!in)
		return;
	double scale[W];
	bool any = false;
#pragma unroll
	for (int w = 0; w < W; ++w)
	{
		scale[w] = st[b + w].scale;
		any = any || scale[w] > 0.0;
	}
	if (!any)
		return;
	for (int64_t o = q0 + t_row; o < q1; o += geo.R)
	{
		const int64_t i = (KEPT ? G.nE + o : o) * B + b;
		auto xv = rbw_load<W>(x + i);
		rbw_store<W>(keep + i, xv);
		rbw_vec_t<W> d, cc{}, rv{};
		if (KEPT)
			d = rbw_load<W>(dx + o * B + b);
		else
		{
			cc = rbw_load<W>(c + i);
			rv = rbw_load<W>(res + i);
			d = rbw_sum<W>(G, o, b, bl, geo, rt, dx);
		}
#pragma unroll
		for (int w = 0; w < W; ++w)
			if (scale[w] > 0.0)
				xv.v[w] += KEPT			   ? scale[w] * d.v[w]
						   : cc.v[w] != 0.0 ? cc.v[w] * (rv.v[w] + scale[w] * d.v[w])
											: rv.v[w];
		rbw_store<W>(x + i, xv);
	}
}

// the iterate before the last cycle, for the sets of `undo`
__global__ __launch_bounds__(sblock) void k_rbw_undo(int64_t count, int B, const double* __restrict__ keep,
													 double* __restrict__ x, const int32_t* __restrict__ undo)
{
	const int64_t i = (int64_t)blockIdx.x * sblock + threadIdx.x;
	if (i < count && undo[i % B])
		x[i] = keep[i];
}

// sums over the blocks of part[blk][b][K] (one workgroup per set, fixed order),
// then that set's scalars.  STEP 0: residual norms to out[b][2]; 1: start of a
// cycle; 2: alpha; 3: omega, beta and whether the set goes on, also into the
// host's mirror.
template <int STEP>
__global__ __launch_bounds__(sblock) void k_rbw_reduce(const double* __restrict__ part, int nblk, int B,
													   rbw_set_t* __restrict__ st, double* __restrict__ out,
													   int32_t* __restrict__ h_live, double aim)
{
	constexpr int K = STEP == 2 ? 1 : STEP == 3 ? 5 : STEP == 1 ? 3 : 2;
	__shared__ double s_part[rb_part];
	const int b = blockIdx.x;
	const bool on = STEP == 0 || st[b].live;
	if (STEP == 3 && !on)
	{
		if (threadIdx.x == 0)
		{
			st[b].upd = 0;
			h_live[b] = 0;
		}
		return;
	}
	if (!on)
		return;
	double v[K];
#pragma unroll
	for (int k = 0; k < K; ++k)
		v[k] = 0.0;
	for (int i = threadIdx.x; i < nblk; i += sblock)
#pragma unroll
		for (int k = 0; k < K; ++k)
			v[k] += part[((int64_t)i * B + b) * K + k];
	rb_block_sums<sblock>(v, s_part);
	if (threadIdx.x != 0)
		return;
	if constexpr (STEP == 0)
	{
		out[2 * b] = v[0];
		out[2 * b + 1] = v[1];
	}
	else if constexpr (STEP == 1)
	{
		rbw_set_t& s = st[b];
		s.rho = v[1];
		s.lost2 = rb_lost * rb_lost * v[2];
		s.est = v[0] > 0.0 ? s.est / sqrt(v[0]) : 0.0; // the host left the relative residual here
		if (!(v[0] > 0.0))
			s.live = 0; // nothing left on the kept rows: the correction solves the eliminated ones
	}
	else if constexpr (STEP == 2)
	{
		rbw_set_t& s = st[b];
		s.alpha = s.rho / v[0];
		if (!rb_finite(s.alpha))
			s.live = 0;
	}
	else
	{
		rbw_set_t& s = st[b];
		double omega = v[1] > 0.0 ? v[0] / v[1] : 0.0;
		if (!rb_finite(omega))
			omega = 0.0;
		const double rr = fmax(v[2] - omega * (2.0 * v[0] - omega * v[1]), 0.0);
		const double rho1 = v[3] - omega * v[4];
		const double beta = (rho1 / s.rho) * (s.alpha / omega);
		const bool stop = sqrt(rr) * s.est <= aim || omega == 0.0 || !rb_finite(beta) || beta == 0.0 ||
						  rho1 * rho1 <= s.lost2 * rr;
		s.omega = omega;
		s.beta = stop ? 0.0 : beta;
		s.rho = rho1;
		s.upd = 1;
		s.live = stop ? 0 : 1;
		h_live[b] = s.live;
	}
}
