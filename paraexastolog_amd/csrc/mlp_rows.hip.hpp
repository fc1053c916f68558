// The surrogate network in two kernels per training step and one per forward
// pass, for inputs and hidden layers up to 256 wide, at most 4 hidden layers and
// 2048 outputs (what LDS holds for 16 rows); other shapes run layer by layer.
//
// k_mlp_rows takes 4 or 16 rows through the whole network, and back: the rows'
// activations, GELU derivatives and output gradients stay in LDS and registers,
// so the only operands that come from memory are the weights, once each way.
// k_mlp_update multiplies the rows' activations by their gradients, tile by tile
// of the weights, and applies Adam to the tile it holds.
//
// Products are v_mfma_f32_16x16x32_bf16: lane l holds A[l % 16][8 (l / 16) + 0..7],
// B[8 (l / 16) + 0..7][l % 16] and C[4 (l / 16) + 0..3][l % 16].  Operands come from
// memory as fragments: 16 x 32 tiles of 1 KB in the order in which the lanes take
// them, one 16-byte load per lane.  The weights have such copies for both directions,
// rounded to BF16 as the products always did, kept beside the FP32 masters and
// rewritten by the update; activations and gradients are stored so by k_mlp_rows, with
// rows as the summed index.  The sums that probabilities, gradients and parameters come
// from are those of the layer-by-layer kernels, their splits of k included, and were the
// same bits on 13 shapes (widths and outputs that are no multiple of a tile, 1 to 4,096
// rows, three training steps); a row's loss, which is only reported, is added in another
// order and differed in its last bit on three.  The order matters: training amplifies a
// difference in the last bit (an activation on the other side of a BF16 rounding,
// through Adam's quotient) to 4e-5 of the parameters in 64 steps.
//
// What bounds them: a workgroup reads all weights, 2.6 MB there and back, at the 64 bytes
// per clock of its compute unit's cache (17 us), beside vector work and barriers; the
// update moves parameters, moments and copies (18 MB) and waits for memory three times.
// 512 x (32-256-256-256-2048), per training step: 23 launches of 3 to 10 us, each a few
// memory latencies long, 138 us; two launches of 33.5 and 12.8 us, 51 us with the gaps.
// 4096 rows forward: four products and a softmax, 83 us; one launch of 28 us, 36 to 37 us
// as a call, of which 33 MB of probabilities take 7.
#pragma once

namespace esl {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

constexpr int mr_layers = 4;   // hidden layers
constexpr int mr_width = 256;  // inputs, hidden width
constexpr int mr_out = 2048;   // outputs: 16 waves x 8 tiles x 16
constexpr int mr_block = 1024; // a wave per 16 hidden columns
constexpr int mr_waves = mr_block / wave;
constexpr int mr_tile = 512; // shorts of a fragment
constexpr int mr_ktq = 8;	 // fragments loaded ahead
constexpr int mr_sum_ld = 260; // a row of k_mlp_rows' partial sums

struct mlp_net_t
{
	int n_in, hidden, layers, n_out;
	int kt0, kth, kto; // 32-wide tiles of the input, the padded hidden width and the output
	float* params;
	short* ops;
	int64_t w[mr_layers + 1], b[mr_layers + 1];	  // into params
	int64_t wf[mr_layers + 1], wb[mr_layers + 1]; // into ops: [n / 16][k / 32] of W, [k / 16][n / 32] of W^T
	__host__ __device__ int in_tiles(int l) const { return l == 0 ? kt0 : kth; }
	__host__ __device__ int out_tiles(int l) const { return l == layers ? kto : kth; }
	__host__ __device__ int rows_of(int l) const { return l == 0 ? n_in : hidden; }
	__host__ __device__ int cols_of(int l) const { return l == layers ? n_out : hidden; }
	__host__ __device__ int biases() const { return layers * hidden + n_out; }
};

struct mlp_batch_t
{
	int rows, rt; // rows, tiles of 32 rows
	const float *x, *tg;
	float* P;
	double* Pd;	 // instead of P
	short* frag; // activations and gradients, [32 rows][16 columns] fragments
	int64_t xf[mr_layers + 1], zf[mr_layers + 1]; // input and output gradient of weight layer l
	float *dz, *loss_rows; // output gradients of all layers in FP32, [rows][biases]
	int zc, xc[mr_layers + 1]; // 32-wide tiles per partial sum: over the outputs; over the rows, per weight layer
};

__device__ __forceinline__ f32x4_t mfma16(bf16x8_t a, bf16x8_t b, f32x4_t c)
{
	return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint2 pack_bf16(const float v[4])
{
	return make_uint2((uint32_t)(uint16_t)to_bf16(v[0]) | ((uint32_t)(uint16_t)to_bf16(v[1]) << 16),
					  (uint32_t)(uint16_t)to_bf16(v[2]) | ((uint32_t)(uint16_t)to_bf16(v[3]) << 16));
}

// LDS of k_mlp_rows: two activation buffers, two sets of per-wave row values, the partial
// sums of the softmax, and with training the GELU derivatives and, in the sums' place
// later, the output gradients
inline size_t mlp_rows_lds(const mlp_net_t& m, int rb, bool train)
{
	const size_t sums = (size_t)rb * mr_sum_ld * sizeof(float), d = (size_t)rb * (32 * m.kto + 8) * sizeof(short);
	return (size_t)2 * rb * (32 * std::max(m.kt0, m.kth) + 8) * sizeof(short) + (size_t)2 * mr_waves * rb * sizeof(float) +
		   (train ? (size_t)m.layers * rb * 32 * m.kth * sizeof(float) + std::max(sums, d) : sums);
}

template <int E>
__device__ __forceinline__ void put_bf16(short* d, const float (&v)[E])
{
	if constexpr (E == 4)
		*reinterpret_cast<uint2*>(d) = pack_bf16(v);
	else
		for (int i = 0; i < E; ++i)
			d[i] = to_bf16(v[i]);
}

// E rows per group of 16 lanes, 4 E per workgroup.  With E = 4 a lane has the four rows of
// its C fragment.  A workgroup's time is that of its vector instructions (some 50 per row
// and output) and of its weights (1 MB each way for 2048 outputs, at the rate of one
// compute unit's cache), so few rows are spread over more compute units (512 rows
// of the above: 49.5 us with E = 4, 33.5 with E = 1): with E = 1 group
// g of the 16 rows of A repeats row g, every lane has one element per tile, and the
// products' unused rows cost nothing.  KT: padded hidden width / 32; TPW: most output
// tiles per wave.
template <int E, int KT, int TPW, bool TRAIN>
__global__ __launch_bounds__(mr_block) void k_mlp_rows(mlp_net_t m, mlp_batch_t q)
{
	extern __shared__ __align__(16) unsigned char mr_smem[];
	constexpr int rb = 4 * E; // rows of a workgroup
	constexpr int ht = 2 * KT; // 16-column tiles of a hidden layer: waves that own one
	const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / wave), l = lane_id(), g = l >> 4, c = l & 15;
	const int lda = 32 * max(m.kt0, KT) + 8, ldd = 32 * m.kto + 8;
	short* const sa = reinterpret_cast<short*>(mr_smem);
	float* const s_red = reinterpret_cast<float*>(sa + 2 * rb * lda);
	float* const s_gg = s_red + 2 * mr_waves * rb;
	short* const s_d = reinterpret_cast<short*>(s_gg + (TRAIN ? m.layers * rb * 32 * KT : 0));
	float* const s_sum = reinterpret_cast<float*>(s_d);
	const int r0 = blockIdx.x * rb, rl = r0 + E * g; // this lane's rows: rl + 0 .. E - 1
	const int ar = E * (c >> 2) + (c & 3) % E;		 // row of this lane's A operand
	// where they lie in a fragment over rows
	const int64_t rtile = r0 / 32;
	const int rpos = (16 * (((r0 & 31) + E * g) >> 3) + c) * 8 + ((r0 + E * g) & 7);
	const bool own = w < ht;
	const int n = 16 * w + c; // hidden column of a wave that owns one
	const int ntile = 2 * m.kto; // a wave computes every 16th tile of the output
	auto frag = [&](const short* t, int k) { return *reinterpret_cast<const bf16x8_t*>(t + k * mr_tile + 8 * l); };
	auto out_tile = [&](int j) {
		return m.ops + m.wf[m.layers] + (int64_t)min(w + mr_waves * j, ntile - 1) * KT * mr_tile;
	};

	// a layer's weights and bias (after the last, the wave's first output tile) are on their way
	// before the rows are staged and while the previous layer's activation is evaluated
	bf16x8_t wr[KT];
	float bv = 0.0f;
	auto ahead = [&](int y) {
		if (y < m.layers && !own)
			return;
		const short* W = y == m.layers ? out_tile(0) : m.ops + m.wf[y] + (int64_t)w * m.in_tiles(y) * mr_tile;
#pragma unroll
		for (int k = 0; k < KT; ++k)
			if (y > 0 || k < m.kt0)
				wr[k] = frag(W, k);
		if (n < m.cols_of(y))
			bv = m.params[m.b[y] + n];
	};
	ahead(0);
	{
		const int k0p = 32 * m.kt0;
		for (int i = threadIdx.x; i < rb * k0p; i += mr_block)
		{
			const int r = i / k0p, k = i - r * k0p;
			const float v = r0 + r < q.rows && k < m.n_in ? q.x[(int64_t)(r0 + r) * m.n_in + k] : 0.0f;
			sa[r * lda + k] = to_bf16(v);
		}
	}
	__syncthreads();
	if constexpr (TRAIN)
		for (int t = w; t < 2 * m.kt0; t += mr_waves)
		{ // as operand of the first weights' gradient
			const short* s = sa + E * g * lda + 16 * t + c;
			short* d = q.frag + q.xf[0] + (rtile * 2 * m.kt0 + t) * mr_tile + rpos;
#pragma unroll
			for (int i = 0; i < E; ++i)
				d[i] = s[i * lda];
		}

	// hidden layers: a wave computes 16 columns
	int p = 0;
	for (int y = 0; y < m.layers; ++y)
	{
		const short* s = sa + p * rb * lda + ar * lda + 8 * g;
		f32x4_t acc = { 0.0f, 0.0f, 0.0f, 0.0f };
		if (own)
		{
#pragma unroll
			for (int k = 0; k < KT; ++k)
				if (y > 0 || k < m.kt0)
					acc = mfma16(*reinterpret_cast<const bf16x8_t*>(s + 32 * k), wr[k], acc);
			if (y == 0)
				for (int k = KT; k < m.kt0; ++k)
					acc = mfma16(*reinterpret_cast<const bf16x8_t*>(s + 32 * k),
								 frag(m.ops + m.wf[0] + (int64_t)w * m.kt0 * mr_tile, k), acc);
		}
		const float b = bv;
		ahead(y + 1);
		if (own)
		{
			float a[E];
#pragma unroll
			for (int i = 0; i < E; ++i)
			{
				const float z = acc[i] + b;
				float du;
				const float sg = gelu_sigma(z, du);
				a[i] = rl + i < q.rows ? z * sg : 0.0f;
				if constexpr (TRAIN)
					s_gg[E * ((y * ht + w) * wave + l) + i] = sg + 2.0f * z * sg * (1.0f - sg) * du;
			}
			short* d = sa + (p ^ 1) * rb * lda + E * g * lda + n;
#pragma unroll
			for (int i = 0; i < E; ++i)
				d[i * lda] = to_bf16(a[i]);
			if constexpr (TRAIN)
				put_bf16<E>(q.frag + q.xf[y + 1] + (rtile * ht + w) * mr_tile + rpos, a);
		}
		p ^= 1;
		__syncthreads();
	}

	// logits: the next tile's weights are loaded before a tile is multiplied.  The rows'
	// operand is read from LDS for each tile (the fence keeps it out of registers, which
	// hold two tiles of weights instead); past the last tile the last one is repeated.
	float acc[TPW][E];
	{
		const short* s = sa + p * rb * lda + ar * lda + 8 * g;
#pragma unroll
		for (int j = 0; j < TPW; ++j)
		{
			bf16x8_t wn[KT];
			float bn = 0.0f;
			if (j + 1 < TPW)
			{
				bn = m.params[m.b[m.layers] + min(16 * (w + mr_waves * (j + 1)) + c, m.n_out - 1)];
				const short* W = out_tile(j + 1);
#pragma unroll
				for (int k = 0; k < KT; ++k)
					wn[k] = frag(W, k);
			}
			asm volatile("" ::: "memory");
			f32x4_t v = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
			for (int k = 0; k < KT; ++k)
				v = mfma16(*reinterpret_cast<const bf16x8_t*>(s + 32 * k), wr[k], v);
#pragma unroll
			for (int i = 0; i < E; ++i)
				acc[j][i] = v[i] + bv;
			bv = bn;
			if (j + 1 < TPW)
#pragma unroll
				for (int k = 0; k < KT; ++k)
					wr[k] = wn[k];
		}
	}
	auto col = [&](int j) { return 16 * (w + mr_waves * j) + c; };
	auto live = [&](int j) { return col(j) < m.n_out; };
	// with few rows the targets are on their way during the softmax
	constexpr bool early = TRAIN && E == 1;
	float tv[early ? TPW : 1][E];
	auto target = [&](int j, float (&d)[E]) {
		const float* const tg = q.tg + (int64_t)r0 * m.n_out;
#pragma unroll
		for (int i = 0; i < E; ++i)
			d[i] = tg[min(E * g + i, q.rows - 1 - r0) * m.n_out + min(col(j), m.n_out - 1)];
	};
	if constexpr (early)
#pragma unroll
		for (int j = 0; j < TPW; ++j)
			target(j, tv[j]);
	float mx[E];
#pragma unroll
	for (int i = 0; i < E; ++i)
		mx[i] = -INFINITY;
#pragma unroll
	for (int j = 0; j < TPW; ++j)
	{
		const bool in = live(j);
#pragma unroll
		for (int i = 0; i < E; ++i)
		{
			if (in)
				mx[i] = fmaxf(mx[i], acc[j][i]);
		}
	}
	// values of this lane's rows over the wave's 16 lanes of columns, then over the waves
	auto rows_put = [&](float (&v)[E], float* s, auto op) {
#pragma unroll
		for (int d = 1; d < 16; d <<= 1)
#pragma unroll
			for (int i = 0; i < E; ++i)
				v[i] = op(v[i], __shfl_xor(v[i], d, wave));
		if (c == 0)
#pragma unroll
			for (int i = 0; i < E; ++i)
				s[w * rb + E * g + i] = v[i];
	};
	auto op_max = [](float a, float b) { return fmaxf(a, b); };
	auto op_add = [](float a, float b) { return a + b; };
	rows_put(mx, s_red, op_max);
	__syncthreads();
	// a row's maximum: the waves' by 16 lanes each, then between those
	{
		float v[E];
#pragma unroll
		for (int i = 0; i < E; ++i)
			v[i] = s_red[c * rb + E * g + i];
#pragma unroll
		for (int d = 1; d < 16; d <<= 1)
#pragma unroll
			for (int i = 0; i < E; ++i)
				v[i] = fmaxf(v[i], __shfl_xor(v[i], d, wave));
#pragma unroll
		for (int i = 0; i < E; ++i)
			mx[i] = v[i];
	}
	float sm[E] = {};
#pragma unroll
	for (int j = 0; j < TPW; ++j)
		if (live(j))
#pragma unroll
			for (int i = 0; i < E; ++i)
				sm[i] += __expf(acc[j][i] - mx[i]);
	// the 256 partial sums of a row (columns a stride of 256 apart) in the order of a
	// 256-thread workgroup's sum; wave w adds those of row w
#pragma unroll
	for (int i = 0; i < E; ++i)
		s_sum[(E * g + i) * mr_sum_ld + 16 * w + c] = sm[i];
	__syncthreads();
	if (w < rb)
	{
		float t = 0.0f;
#pragma unroll
		for (int k = 0; k < 4; ++k)
			t += wave_sum(s_sum[w * mr_sum_ld + wave * k + l]);
		if (l == 0)
			s_red[mr_waves * rb + w] = t;
	}
	__syncthreads();
	float lse[E];
#pragma unroll
	for (int i = 0; i < E; ++i)
		lse[i] = mx[i] + logf(s_red[mr_waves * rb + E * g + i]);

	if constexpr (!TRAIN)
	{
#pragma unroll
		for (int j = 0; j < TPW; ++j)
			if (live(j))
#pragma unroll
				for (int i = 0; i < E; ++i)
					if (rl + i < q.rows)
					{
						const float pv = __expf(acc[j][i] - lse[i]);
						const int64_t o0 = (int64_t)r0 * m.n_out;
						const int o = (E * g + i) * m.n_out + col(j);
						if (q.Pd)
							q.Pd[o0 + o] = (double)pv;
						else
							q.P[o0 + o] = pv;
					}
		return;
	}
	else
	{
		float* const dz = q.dz + (int64_t)r0 * m.biases();
		// a tile of gradients: its fragment, its operand in LDS, and in FP32 for the column sums
		auto put = [&](const float (&v)[E], short* fr, short* lds, int ld, int o, bool in) {
			put_bf16<E>(fr + rpos, v);
			if (lds)
			{
#pragma unroll
				for (int i = 0; i < E; ++i)
					lds[(E * g + i) * ld] = to_bf16(v[i]);
			}
#pragma unroll
			for (int i = 0; i < E; ++i)
				if (in && rl + i < q.rows)
					dz[(E * g + i) * m.biases() + o] = v[i];
		};
		float loss[E] = {};
#pragma unroll
		for (int j = 0; j < TPW; ++j)
		{
			const int t = w + mr_waves * j;
			if (t >= ntile)
				continue;
			const bool in = live(j);
			float d[E];
			if constexpr (!early)
				target(j, tv[0]);
#pragma unroll
			for (int i = 0; i < E; ++i)
			{
				const bool ok = in && rl + i < q.rows;
				const float e = acc[j][i] - lse[i], ti = tv[early ? j : 0][i];
				d[i] = ok ? (__expf(e) - ti) / (float)q.rows : 0.0f;
				if (ok && ti > 0.0f)
					loss[i] -= ti * e;
			}
			put(d, q.frag + q.zf[m.layers] + (rtile * ntile + t) * mr_tile, s_d + col(j), ldd,
				m.layers * m.hidden + col(j), in);
		}
		rows_put(loss, s_red, op_add); // the maxima there were read before the last barrier
		__syncthreads();
		if (threadIdx.x < rb && r0 + (int)threadIdx.x < q.rows)
		{
			float t = 0.0f;
			for (int k = 0; k < mr_waves; ++k)
				t += s_red[k * rb + threadIdx.x];
			q.loss_rows[r0 + threadIdx.x] = t;
		}

		// back through the layers: the gradient of hidden layer y's output, times its GELU derivative
		// the weights from hidden layer y to the one below, on their way a layer ahead
		auto below = [&](int y) {
			if (own && y > 1)
#pragma unroll
				for (int k = 0; k < KT; ++k)
					wr[k] = frag(m.ops + m.wb[y - 1] + (int64_t)w * KT * mr_tile, k);
		};
		below(m.layers);
		f32x4_t tot = { 0.0f, 0.0f, 0.0f, 0.0f };
		if (own)
		{
			const short* s = s_d + ar * ldd + 8 * g;
			const short* W = m.ops + m.wb[m.layers] + (int64_t)w * m.kto * mr_tile + 8 * l;
			for (int k0 = 0; k0 < m.kto; k0 += q.zc)
			{
				const int ke = min(m.kto, k0 + q.zc);
				f32x4_t v = { 0.0f, 0.0f, 0.0f, 0.0f };
				int k = k0;
				for (; k + mr_ktq <= ke; k += mr_ktq)
#pragma unroll
					for (int e = 0; e < mr_ktq; ++e)
						v = mfma16(*reinterpret_cast<const bf16x8_t*>(s + 32 * (k + e)),
								   *reinterpret_cast<const bf16x8_t*>(W + (k + e) * mr_tile), v);
				for (; k < ke; ++k)
					v = mfma16(*reinterpret_cast<const bf16x8_t*>(s + 32 * k),
							   *reinterpret_cast<const bf16x8_t*>(W + k * mr_tile), v);
#pragma unroll
				for (int i = 0; i < 4; ++i)
					tot[i] += v[i];
			}
		}
		for (int y = m.layers; y >= 1; --y)
		{
			if (own)
			{
				float d[E];
#pragma unroll
				for (int i = 0; i < E; ++i)
					d[i] = rl + i < q.rows ? tot[i] * s_gg[E * (((y - 1) * ht + w) * wave + l) + i] : 0.0f;
				put(d, q.frag + q.zf[y - 1] + (rtile * ht + w) * mr_tile,
					y > 1 ? sa + p * rb * lda + n : nullptr, lda, (y - 1) * m.hidden + n, n < m.hidden);
			}
			if (y == 1)
				break;
			__syncthreads();
			if (own)
			{
				const short* s = sa + p * rb * lda + ar * lda + 8 * g;
				tot = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
				for (int k = 0; k < KT; ++k)
					tot = mfma16(*reinterpret_cast<const bf16x8_t*>(s + 32 * k), wr[k], tot);
			}
			below(y - 1);
			p ^= 1;
		}
	}
}

struct mlp_adam_t
{
	float *m1, *m2, *grads; // grads: written instead of the Adam step
	float* loss;
	int accumulate;
	float lr, b1, b2, eps, c1, c2;
};

// Gradients of 16 x 32 weights per wave, summed over the rows (fragments straight from
// memory: an operand tile is used by a few waves only, and there are fewer waves than
// the chip holds, so their loads are what there is to overlap; 32 x 32 weights per wave
// took 14.9 us instead of 12.8), and the Adam
// step on them.  Then workgroups for 32 biases each (column sums of the gradients) and one for
// the loss.
template <bool ADAM>
__global__ __launch_bounds__(256) void k_mlp_update(mlp_net_t m, mlp_batch_t q, mlp_adam_t a, int tiles)
{
	__shared__ float s_part[256];
	const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / wave), l = lane_id(), g = l >> 4, c = l & 15;
	const int tile_blocks = (tiles + 3) / 4;
	if ((int)blockIdx.x < tile_blocks)
	{
		int t = blockIdx.x * 4 + w, y = 0;
		if (t >= tiles)
			return;
		while (t >= 2 * m.in_tiles(y) * m.out_tiles(y))
		{
			t -= 2 * m.in_tiles(y) * m.out_tiles(y);
			++y;
		}
		const int it = 2 * m.in_tiles(y), ot = m.out_tiles(y); // tiles of 16 inputs, of 32 outputs
		const int mt = t % it, nt = t / it;
		const int M = m.rows_of(y), N = m.cols_of(y);
		const int row = 16 * mt + 4 * g, cl = 32 * nt + c; // of this lane's first element
		const int64_t o0 = m.w[y] + (int64_t)16 * mt * N + 32 * nt;
		float pv[2][4], m1[2][4], m2[2][4];
#pragma unroll
		for (int j = 0; j < 2; ++j)
#pragma unroll
			for (int e = 0; e < 4; ++e)
			{
				const bool in = ADAM && row + e < M && cl + 16 * j < N;
				const int o = (4 * g + e) * N + c + 16 * j;
				pv[j][e] = in ? m.params[o0 + o] : 0.0f;
				m1[j][e] = in ? a.m1[o0 + o] : 0.0f;
				m2[j][e] = in ? a.m2[o0 + o] : 0.0f;
			}
		const short* X = q.frag + q.xf[y] + (int64_t)mt * mr_tile;
		const short* Z = q.frag + q.zf[y] + (int64_t)2 * nt * mr_tile;
		const int64_t xs = (int64_t)it * mr_tile, zs = (int64_t)2 * ot * mr_tile;
		auto ld = [&](const short* s) { return *reinterpret_cast<const bf16x8_t*>(s + 8 * l); };
		// 8 tiles of 32 rows at a time, the next 8 loaded before they are multiplied (past the
		// end the last tile again, unused); a partial sum ends every xc tiles
		const int xc = q.xc[y];
		f32x4_t tot[2] = {}, v[2] = {};
		bf16x8_t x[mr_ktq], z[mr_ktq][2];
		auto fetch = [&](int k, bf16x8_t (&fx)[mr_ktq], bf16x8_t (&fz)[mr_ktq][2]) {
#pragma unroll
			for (int f = 0; f < mr_ktq; ++f)
			{
				const int kk = min(k + f, q.rt - 1);
				fx[f] = ld(X + kk * xs);
				fz[f][0] = ld(Z + kk * zs), fz[f][1] = ld(Z + kk * zs + mr_tile);
			}
		};
		fetch(0, x, z);
		for (int k0 = 0; k0 < q.rt; k0 += mr_ktq)
		{
			bf16x8_t xn[mr_ktq], zn[mr_ktq][2];
			if (k0 + mr_ktq < q.rt)
				fetch(k0 + mr_ktq, xn, zn);
#pragma unroll
			for (int f = 0; f < mr_ktq; ++f)
			{
				if (k0 + f >= q.rt)
					break;
				v[0] = mfma16(x[f], z[f][0], v[0]), v[1] = mfma16(x[f], z[f][1], v[1]);
				if ((k0 + f + 1) % xc == 0 || k0 + f + 1 == q.rt)
				{
					tot[0] += v[0], tot[1] += v[1];
					v[0] = v[1] = f32x4_t{ 0.0f, 0.0f, 0.0f, 0.0f };
				}
			}
#pragma unroll
			for (int f = 0; f < mr_ktq; ++f)
				x[f] = xn[f], z[f][0] = zn[f][0], z[f][1] = zn[f][1];
		}
#pragma unroll
		for (int j = 0; j < 2; ++j)
		{
			float nv[4];
#pragma unroll
			for (int e = 0; e < 4; ++e)
			{
				nv[e] = 0.0f;
				if (row + e >= M || cl + 16 * j >= N)
					continue;
				const int o = (4 * g + e) * N + c + 16 * j;
				if constexpr (ADAM)
				{
					nv[e] = adam_step(pv[j][e], tot[j][e], m1[j][e], m2[j][e], a.lr, a.b1, a.b2, a.eps, a.c1, a.c2);
					m.params[o0 + o] = nv[e];
					a.m1[o0 + o] = m1[j][e];
					a.m2[o0 + o] = m2[j][e];
				}
				else
					a.grads[o0 + o] = tot[j][e];
			}
			if constexpr (ADAM)
			{
				// the operand copies: k = 16 (mt % 2) + 4 g + e and n = 16 j + c within 32 x 32 weights
				const uint2 pk = pack_bf16(nv);
				short* f = m.ops + m.wf[y] + ((int64_t)(2 * nt + j) * (it / 2) + mt / 2) * mr_tile;
				*reinterpret_cast<uint2*>(f + (16 * (2 * (mt & 1) + (g >> 1)) + c) * 8 + 4 * (g & 1)) = pk;
				if (y > 0)
				{
					short* b = m.ops + m.wb[y] + ((int64_t)mt * ot + nt) * mr_tile +
							   (16 * (2 * j + (c >> 3)) + 4 * g) * 8 + (c & 7);
					b[0] = (short)(pk.x & 0xffff), b[8] = (short)(pk.x >> 16);
					b[16] = (short)(pk.y & 0xffff), b[24] = (short)(pk.y >> 16);
				}
			}
		}
		return;
	}
	const int nb = m.biases(), bias_blocks = (nb + 31) / 32, bb = blockIdx.x - tile_blocks;
	if (bb < bias_blocks)
	{
		// 32 biases, 8 slices of consecutive rows
		const int i = bb * 32 + (threadIdx.x & 31), sl = threadIdx.x >> 5;
		const int per = (q.rows + 7) / 8, re = min(q.rows, (sl + 1) * per);
		float t = 0.0f;
		if (i < nb)
		{
#pragma unroll 32
			for (int r = sl * per; r < re; ++r)
				t += q.dz[(int64_t)r * nb + i];
		}
		s_part[threadIdx.x] = t;
		__syncthreads();
		if (sl || i >= nb)
			return;
		t = 0.0f;
		for (int k = 0; k < 8; ++k)
			t += s_part[32 * k + threadIdx.x];
		const int y = min(i / m.hidden, m.layers);
		const int64_t o = m.b[y] + i - y * m.hidden;
		if constexpr (ADAM)
		{
			float m1 = a.m1[o], m2 = a.m2[o];
			m.params[o] = adam_step(m.params[o], t, m1, m2, a.lr, a.b1, a.b2, a.eps, a.c1, a.c2);
			a.m1[o] = m1;
			a.m2[o] = m2;
		}
		else
			a.grads[o] = t;
		return;
	}
	float t = 0.0f;
	for (int i = threadIdx.x; i < q.rows; i += 256)
		t += q.loss_rows[i];
	t = block_sum<256>(t, s_part);
	if (threadIdx.x == 0)
		a.loss[0] = a.accumulate ? a.loss[0] + t : t;
}

// the operand copies from the parameters (padding zero): a wave per fragment
__global__ __launch_bounds__(256) void k_mlp_operands(mlp_net_t m, int frags)
{
	int t = blockIdx.x * 4 + threadIdx.x / wave;
	const int l = lane_id();
	if (t >= frags)
		return;
	for (int y = 0; y <= m.layers; ++y)
		for (int back = 0; back < (y > 0 ? 2 : 1); ++back)
		{
			const int it = m.in_tiles(y), ot = m.out_tiles(y);
			if (t >= 2 * it * ot)
			{
				t -= 2 * it * ot;
				continue;
			}
			const int kt = back ? ot : it; // tiles of the summed index
			const int M = m.rows_of(y), N = m.cols_of(y);
			const int outer = 16 * (t / kt) + (l & 15), k = 32 * (t % kt) + 8 * (l >> 4);
			short* d = m.ops + (back ? m.wb[y] : m.wf[y]) + (int64_t)t * mr_tile + 8 * l;
#pragma unroll
			for (int j = 0; j < 8; ++j)
			{
				const int r = back ? outer : k + j, n = back ? k + j : outer;
				d[j] = r < M && n < N ? to_bf16(m.params[m.w[y] + (int64_t)r * N + n]) : (short)0;
			}
			return;
		}
}

} // namespace esl
