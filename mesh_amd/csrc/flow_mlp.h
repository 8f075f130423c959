// Dense layers and circle maps shared by the U(1) learned flows (flow.hip:
// coupling layers on links, pcflow.hip: coupling layers on plaquettes).
//
// Per layer an MLP NI -> 64 -> 64 -> 10 (tanh) turns NI context features of
// an active variable into the parameters of a circle diffeomorphism
//   h(a) = g(wrap(a - t)) + t,  g(u) = sum_k w_k 2 atan(s_k tan(u / 2))
// (a mixture of NK = 4 non-compact projections; s_k = exp(clamp(y_k, -8, 8)),
// w = softmax(y_{4..7}), t = atan2(y_9, y_8)).  The dense layers run on FP32
// MFMA (v_mfma_f32_16x16x4_f32) in 16-row tiles, one tile per wavefront; the
// backward pass forms the weight gradients as MFMA tile products.
//
// Parameters of one layer, in order: W1 [NI][64], b1 [64], W2 [64][64],
// b2 [64], W3 [64][10], b3 [10].
#pragma once

#include <cstddef>

#include "mesh_internal.h"
#include "rng_dev.h"

namespace flow_mlp {

constexpr int NK = 4;          // mixture components
constexpr int NH = 64;         // hidden width
constexpr int NO = 2 * NK + 2; // outputs
constexpr float PI_F = 3.14159265358979323846f;
constexpr float TWO_PI_F = 6.28318530717958647692f;

typedef float f4 __attribute__((ext_vector_type(4)));

template <int NI> struct Layout
{
	static_assert(NI % 4 == 0 && NI <= 48, "features: a multiple of 4, at most 48");
	static constexpr int XS = (NI + 15) / 16 * 16; // feature row stride of a tile
	static constexpr int OW1 = 0, OB1 = OW1 + NI * NH, OW2 = OB1 + NH, OB2 = OW2 + NH * NH, OW3 = OB2 + NH,
	                     OB3 = OW3 + NH * NO, NP = OB3 + NO;
};

// orders the LDS accesses of one wavefront (no cross-wavefront wait)
__device__ __forceinline__ void wave_sync()
{
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float wrapf(float a)
{
	a = a - TWO_PI_F * floorf((a + PI_F) * (1.0f / TWO_PI_F));
	return a >= PI_F ? a - TWO_PI_F : (a < -PI_F ? a + TWO_PI_F : a);
}

// D(16x16) = sum_k A(i,k) B(k,n), A(i,k) = A[i*sai + k*sak], B(k,n) = B[k*sbk + n*sbn],
// k < K (multiple of 4).  Lane l supplies A(l%16, k0 + l/16) and
// B(k0 + l/16, l%16); it receives D(4*(l/16) + j, l%16), j < 4.
__device__ __forceinline__ f4 tile_mm(const float *A, int sai, int sak, const float *B, int sbk, int sbn, int K)
{
	int l = threadIdx.x & 63, i = l & 15, kk = l >> 4;
	f4 acc = {0.f, 0.f, 0.f, 0.f};
	for (int k0 = 0; k0 < K; k0 += 4)
		acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[i * sai + (k0 + kk) * sak], B[(k0 + kk) * sbk + i * sbn], acc,
		                                           0, 0, 0);
	return acc;
}

// LDS image of one layer's weights (W3/b3 padded to 16 columns)
template <int NI> struct LW
{
	float w1[NI * NH], b1[NH], w2[NH * NH], b2[NH], w3[NH * 16], b3[16];
};

template <int NI> __device__ void load_weights(LW<NI> &lw, const float *__restrict__ p)
{
	using Y = Layout<NI>;
	for (int i = threadIdx.x; i < NI * NH; i += blockDim.x)
		lw.w1[i] = p[Y::OW1 + i];
	for (int i = threadIdx.x; i < NH * NH; i += blockDim.x)
		lw.w2[i] = p[Y::OW2 + i];
	for (int i = threadIdx.x; i < NH * 16; i += blockDim.x)
	{
		int k = i / 16, n = i % 16;
		lw.w3[i] = n < NO ? p[Y::OW3 + k * NO + n] : 0.f;
	}
	for (int i = threadIdx.x; i < NH; i += blockDim.x)
	{
		lw.b1[i] = p[Y::OB1 + i];
		lw.b2[i] = p[Y::OB2 + i];
	}
	for (int i = threadIdx.x; i < 16; i += blockDim.x)
		lw.b3[i] = i < NO ? p[Y::OB3 + i] : 0.f;
}

// per-wavefront tile scratch: features (row stride XS; the columns from NI on
// must be finite), two hidden layers h1, h2() and the outputs y().  SEP = false
// (kernels without a backward pass, which needs every layer's values) puts h2
// over h1 and the outputs over the features, each consumed by then: 5 KB less
// LDS per tile.
template <int NI, bool SEP = true> struct Tile
{
	float x[16 * Layout<NI>::XS], h1[16 * NH];
	float h2s[SEP ? 16 * NH : 1];
	float ys[SEP ? 16 * 16 : 1];
	__device__ float *h2() { return SEP ? h2s : h1; }
	__device__ float *y() { return SEP ? ys : x; }
};

// One layer's parameters held in registers (two floats a lane per chunk) so
// that the next layer's global loads overlap the current layer's work; NP is
// even for every NI, so each layer starts 8-byte aligned.  store() writes the
// LDS image: w1, b1, w2, b2 in the parameters' own order, W3/b3 into their
// 16-column padding (the pad stays as zero_pad() left it).
template <int NI, int THREADS> struct WeightRegs
{
	using Y = Layout<NI>;
	static_assert(Y::NP % 2 == 0 && Y::OW3 % 2 == 0 && Y::OB3 % 2 == 0 && NO % 2 == 0, "pairs of parameters");
	static constexpr int NC = Y::NP / 2;
	static constexpr int PER = (NC + THREADS - 1) / THREADS;
	float2 v[PER];

	__device__ void load(const float *__restrict__ p)
	{
		const float2 *q = reinterpret_cast<const float2 *>(p);
		for (int i = 0; i < PER; ++i)
		{
			const int c = threadIdx.x + i * THREADS;
			if (c < NC)
				v[i] = q[c];
		}
	}
	__device__ void store(LW<NI> &lw) const
	{
		static_assert(offsetof(LW<NI>, w3) == Y::OW3 * sizeof(float), "w1, b1, w2, b2 as in the parameters");
		float2 *head = reinterpret_cast<float2 *>(&lw);
		for (int i = 0; i < PER; ++i)
		{
			const int c = threadIdx.x + i * THREADS, idx = 2 * c;
			if (c >= NC)
				break;
			if (idx < Y::OW3)
				head[c] = v[i];
			else if (idx < Y::OB3)
			{
				const int k = (idx - Y::OW3) / NO, n = idx - Y::OW3 - k * NO;
				*reinterpret_cast<float2 *>(&lw.w3[k * 16 + n]) = v[i];
			}
			else
				*reinterpret_cast<float2 *>(&lw.b3[idx - Y::OB3]) = v[i];
		}
	}
};

// zero the W3/b3 padding columns NO..15 once per kernel (store() never writes them)
template <int NI> __device__ void zero_pad(LW<NI> &lw)
{
	for (int i = threadIdx.x; i < NH * 16; i += blockDim.x)
		if (i % 16 >= NO)
			lw.w3[i] = 0.f;
	if (threadIdx.x < 16 && threadIdx.x >= NO)
		lw.b3[threadIdx.x] = 0.f;
}

// tanh from the hardware exponential and reciprocal: absolute error a few
// 1e-7, saturating to +-1 (e = inf or 0)
__device__ __forceinline__ float tanh_fast(float x)
{
	const float e = __expf(2.f * x);
	return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + e);
}

template <bool FAST> __device__ __forceinline__ float act(float x) { return FAST ? tanh_fast(x) : tanhf(x); }

// MLP forward of one tile: h1 = tanh(x W1 + b1), h2 = tanh(h1 W2 + b2), y = h2 W3 + b3
// (FAST: tanh_fast; a flow uses one choice in all of its kernels)
template <int NI, bool FAST = false, bool SY = true> __device__ void mlp_forward(LW<NI> const &lw, Tile<NI, SY> &T)
{
	constexpr int XS = Layout<NI>::XS;
	int l = threadIdx.x & 63, c = l & 15, rq = (l >> 4) * 4;
	for (int n0 = 0; n0 < NH; n0 += 16)
	{
		f4 d = tile_mm(T.x, XS, 1, lw.w1 + n0, NH, 1, NI);
		for (int j = 0; j < 4; ++j)
			T.h1[(rq + j) * NH + n0 + c] = act<FAST>(d[j] + lw.b1[n0 + c]);
	}
	wave_sync();
	if constexpr (SY)
		for (int n0 = 0; n0 < NH; n0 += 16)
		{
			f4 d = tile_mm(T.h1, NH, 1, lw.w2 + n0, NH, 1, NH);
			for (int j = 0; j < 4; ++j)
				T.h2()[(rq + j) * NH + n0 + c] = act<FAST>(d[j] + lw.b2[n0 + c]);
		}
	else
	{
		// h2() is h1's storage: all four column blocks of h1 W2 first
		f4 d2[NH / 16];
		for (int n0 = 0; n0 < NH; n0 += 16)
			d2[n0 / 16] = tile_mm(T.h1, NH, 1, lw.w2 + n0, NH, 1, NH);
		wave_sync();
		for (int n0 = 0; n0 < NH; n0 += 16)
			for (int j = 0; j < 4; ++j)
				T.h2()[(rq + j) * NH + n0 + c] = act<FAST>(d2[n0 / 16][j] + lw.b2[n0 + c]);
	}
	wave_sync();
	f4 d = tile_mm(T.h2(), NH, 1, lw.w3, 16, 1, NH);
	for (int j = 0; j < 4; ++j)
		T.y()[(rq + j) * 16 + c] = d[j] + lw.b3[c];
	wave_sync();
}

// ---- the MLP on one wavefront with the activations in registers -----------
//
// A 16-row tile is computed transposed, Y^T = W^T X^T: the weights are the
// MFMA's A operand (lane l: output column l % 16 of a block), the activations
// its B operand (lane l: row l % 16).  The product leaves row l % 16's columns
// 16 b + 4 (l / 16) + j in acc[b][j] of lane l, and the next layer takes its
// contraction index in just that order -- step (b, j) contracts the columns
// 16 b + 4 q + j, q = 0..3, one per quarter of the wavefront -- so every lane
// already holds the B operand of the next product and no activation goes
// through LDS.  (With the tile's activations in LDS, rows 64 floats apart,
// the 16 rows of an A operand fell on one bank and each product read them
// again for each block of columns.)  Only the weights are read from LDS, each
// once per tile: rows padded to WS (W3S) floats, 4 WS = 16 (mod 64), put the
// four quarters of a read on different banks.
constexpr int WS = NH + 4;  // row stride of W1 and W2
constexpr int W3S = 20;     // row stride of W3 (columns NO..15 zero)
constexpr int YS = 20;      // row stride of a tile's outputs

// LDS image of one layer's weights
template <int NI> struct alignas(16) LWP
{
	float w1[NI * WS], b1[NH], w2[NH * WS], b2[NH], w3[NH * W3S], b3[16];
};

// One layer's parameters held in registers (two floats a lane per chunk) so
// that the next layer's global loads overlap the current layer's work; NP is
// even for every NI, so each layer starts 8-byte aligned.  store() writes the
// LDS image (the pad columns of W3/b3 stay as zero_pad() left them).
template <int NI, int THREADS> struct WeightRegsP
{
	using Y = Layout<NI>;
	static_assert(Y::NP % 2 == 0 && Y::OB1 % 2 == 0 && Y::OW2 % 2 == 0 && Y::OB2 % 2 == 0 && Y::OW3 % 2 == 0 &&
	                  Y::OB3 % 2 == 0 && NO % 2 == 0,
	              "pairs of parameters");
	static constexpr int NC = Y::NP / 2;
	static constexpr int PER = (NC + THREADS - 1) / THREADS;
	float2 v[PER];

	__device__ void load(const float *__restrict__ p)
	{
		const float2 *q = reinterpret_cast<const float2 *>(p);
#pragma unroll
		for (int i = 0; i < PER; ++i)
		{
			const int c = threadIdx.x + i * THREADS;
			if (c < NC)
				v[i] = q[c];
		}
	}
	__device__ void store(LWP<NI> &lw) const
	{
#pragma unroll
		for (int i = 0; i < PER; ++i)
		{
			const int c = threadIdx.x + i * THREADS, x = 2 * c;
			if (c >= NC)
				break;
			float *dst;
			if (x < Y::OB1)
				dst = lw.w1 + (x / NH) * WS + x % NH;
			else if (x < Y::OW2)
				dst = lw.b1 + (x - Y::OB1);
			else if (x < Y::OB2)
				dst = lw.w2 + ((x - Y::OW2) / NH) * WS + (x - Y::OW2) % NH;
			else if (x < Y::OW3)
				dst = lw.b2 + (x - Y::OB2);
			else if (x < Y::OB3)
				dst = lw.w3 + ((x - Y::OW3) / NO) * W3S + (x - Y::OW3) % NO;
			else
				dst = lw.b3 + (x - Y::OB3);
			*reinterpret_cast<float2 *>(dst) = v[i];
		}
	}
};

// zero the W3/b3 padding columns NO..15 once per kernel (store() never writes them)
template <int NI> __device__ void zero_pad(LWP<NI> &lw)
{
	for (int i = threadIdx.x; i < NH * 16; i += blockDim.x)
		if (i % 16 >= NO)
			lw.w3[(i / 16) * W3S + i % 16] = 0.f;
	if (threadIdx.x < 16 && threadIdx.x >= NO)
		lw.b3[threadIdx.x] = 0.f;
}

// act() of one block of pre-activations
template <bool FAST> __device__ __forceinline__ f4 act4(f4 a)
{
	return f4{act<FAST>(a[0]), act<FAST>(a[1]), act<FAST>(a[2]), act<FAST>(a[3])};
}

// MLP forward of one tile: lane l holds row l % 16; x[s] is its feature
// row(s), the four lanes of a row holding NI / 4 different features each.
// h1[b][j], h2[b][j]: hidden columns 16 b + 4 (l / 16) + j; the return value:
// outputs 4 (l / 16) + j.
//
// AHEAD (kernels with one wavefront a SIMD): the weights come a chunk of 16
// ahead of their products; the scheduling barriers keep the loads there, which
// left alone are placed two products before their use, so that each pair of
// products waits out the LDS.  16^2 sample, 256 chains: 47.2 -> 43.7 us; with
// more wavefronts its registers cost more (32^2 propose 210 -> 228 us).
template <int NI, bool FAST, bool AHEAD, class ROW>
__device__ __forceinline__ f4 mlp_rows(LWP<NI> const &lw, const float (&x)[NI / 4], ROW row, f4 (&h1)[4], f4 (&h2)[4])
{
	constexpr int NS = NI / 4, C1 = (NS + 3) / 4; // steps and chunks of the first layer
	const int l = threadIdx.x & 63, i = l & 15, q4 = (l >> 4) * 4;
	const float *w2 = lw.w2 + q4 * WS + i, *w3 = lw.w3 + q4 * W3S + i;
	float w[2][16];
	// chunk c of the weights: C1 of W1, four of W2 (one for each block of 16 of h1's columns), W3
	auto load = [&](int c, float (&d)[16]) {
#pragma unroll
		for (int s = 0; s < 4; ++s)
			if (c < C1)
			{
				if (4 * c + s < NS)
#pragma unroll
					for (int b = 0; b < 4; ++b)
						d[4 * s + b] = lw.w1[row(4 * c + s) * WS + i + 16 * b];
			}
			else if (c < C1 + 4)
#pragma unroll
				for (int b = 0; b < 4; ++b)
					d[4 * s + b] = w2[(16 * (c - C1) + s) * WS + 16 * b];
			else
#pragma unroll
				for (int b = 0; b < 4; ++b)
					d[4 * s + b] = w3[(16 * b + s) * W3S];
	};
	auto mm = [](float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); };
#pragma unroll
	for (int b = 0; b < 4; ++b)
	{
		h1[b] = *reinterpret_cast<const f4 *>(lw.b1 + 16 * b + q4);
		h2[b] = *reinterpret_cast<const f4 *>(lw.b2 + 16 * b + q4);
	}
	// two chains: the products of one block of columns are each other's input
	f4 y0 = *reinterpret_cast<const f4 *>(lw.b3 + q4), y1 = {0.f, 0.f, 0.f, 0.f};
	if (AHEAD)
		load(0, w[0]);
#pragma unroll
	for (int c = 0; c < C1 + 5; ++c)
	{
		if (!AHEAD)
			load(c, w[c & 1]);
		else if (c < C1 + 4)
			load(c + 1, w[(c + 1) & 1]);
		if (AHEAD)
			__builtin_amdgcn_sched_barrier(0);
		float (&d)[16] = w[c & 1];
		const int k = c - C1;
		if (k < 0)
		{
#pragma unroll
			for (int s = 0; s < 4; ++s)
				if (4 * c + s < NS)
#pragma unroll
					for (int b = 0; b < 4; ++b)
						h1[b] = mm(d[4 * s + b], x[4 * c + s], h1[b]);
			if (k == -1)
				h1[0] = act4<FAST>(h1[0]);
		}
		else if (k < 3)
		{
#pragma unroll
			for (int j = 0; j < 4; ++j)
#pragma unroll
				for (int b = 0; b < 4; ++b)
					h2[b] = mm(d[4 * j + b], h1[k][j], h2[b]);
			h1[k + 1] = act4<FAST>(h1[k + 1]);
		}
		else if (k == 3)
		{
#pragma unroll
			for (int b = 0; b < 4; ++b)
			{
#pragma unroll
				for (int j = 0; j < 4; ++j)
					h2[b] = mm(d[4 * j + b], h1[3][j], h2[b]);
				h2[b] = act4<FAST>(h2[b]);
			}
		}
		else
		{
#pragma unroll
			for (int b = 0; b < 4; b += 2)
#pragma unroll
				for (int j = 0; j < 4; ++j)
				{
					y0 = mm(d[4 * j + b], h2[b][j], y0);
					y1 = mm(d[4 * j + b + 1], h2[b + 1][j], y1);
				}
		}
	}
	return y0 + y1;
}

// outputs of mlp_rows to y[row * YS + column] (one wavefront's scratch, 16 YS floats)
__device__ __forceinline__ void put_outputs(float *y, f4 v)
{
	const int l = threadIdx.x & 63;
	*reinterpret_cast<f4 *>(y + (l & 15) * YS + (l >> 4) * 4) = v;
}

// transform parameters from the MLP outputs
struct NCP
{
	float s[NK], w[NK], t, ta, tb;
};

__device__ __forceinline__ NCP ncp_params(const float *y)
{
	NCP p;
	float m = y[NK];
	for (int k = 1; k < NK; ++k)
		m = fmaxf(m, y[NK + k]);
	float z = 0.f;
	for (int k = 0; k < NK; ++k)
	{
		p.s[k] = expf(fminf(fmaxf(y[k], -8.f), 8.f));
		p.w[k] = expf(y[NK + k] - m);
		z += p.w[k];
	}
	for (int k = 0; k < NK; ++k)
		p.w[k] /= z;
	p.ta = y[2 * NK];
	p.tb = y[2 * NK + 1];
	p.t = atan2f(p.tb, p.ta);
	return p;
}

// g(u), g'(u) of the mixture
__device__ __forceinline__ void ncp_eval(NCP const &p, float u, float &G, float &Gp)
{
	float c = cosf(0.5f * u), sn = sinf(0.5f * u);
	G = 0.f;
	Gp = 0.f;
	for (int k = 0; k < NK; ++k)
	{
		float d = fmaf(c, c, p.s[k] * p.s[k] * sn * sn);
		G = fmaf(p.w[k], 2.f * atan2f(p.s[k] * sn, c), G);
		Gp = fmaf(p.w[k], p.s[k] / d, Gp);
	}
}

// u = g^-1(target): g is increasing on [-pi, pi] with g(+-pi) = +-pi, so
// Newton steps inside a bracket that every evaluation narrows, bisection when
// a step leaves it, until a step or the bracket is below 2e-7 max(1, |u|)
// (an FP32 ulp of u is up to 2.4e-7 here, so an absolute bound could not stop
// an iterate that alternates between neighbouring floats; at most 40
// evaluations).  Returns u, and g'(u) in Gp.
__device__ __forceinline__ float ncp_inverse(NCP const &p, float target, float &Gp)
{
	float lo = -PI_F, hi = PI_F, u = target, G;
	for (int b = 0; b < 40; ++b)
	{
		ncp_eval(p, u, G, Gp);
		float f = G - target;
		if (f == 0.f)
			break;
		if (f < 0.f)
			lo = u;
		else
			hi = u;
		if (hi - lo <= 2e-7f * fmaxf(1.f, fabsf(u)))
			break;
		float un = u - f / Gp;
		if (un > lo && un < hi)
		{
			bool done = fabsf(un - u) <= 2e-7f * fmaxf(1.f, fabsf(un));
			u = un;
			if (done)
				break;
		}
		else
			u = 0.5f * (lo + hi);
	}
	ncp_eval(p, u, G, Gp);
	return u;
}

// ---- elementary functions of the quad maps below, for the ranges they meet.
// The maps were held by these: the library's sincosf and atan2f carry the
// reduction of huge arguments, infinities and zeros, about 90 and 60 VALU
// instructions a call against 24 and 27 here.  Coefficients: minimax fits
// (reweighted least squares) of (sin r - r) / r^3 and (cos r - 1 + r^2 / 2) /
// r^4 over |r| <= pi / 4 and of (atan q - q) / q^3 over [0, 1]; largest errors
// in FP32 0.66 ulp (sin), 1.22 ulp (cos), 0.88 ulp (atan).

// n / d to within an ulp, for d and 1 / d in the normal range
__device__ __forceinline__ float div1(float n, float d)
{
	const float r = __builtin_amdgcn_rcpf(d), q = n * r;
	return fmaf(fmaf(-q, d, n), r, q);
}

constexpr float HALF_PI_HI = 1.57079637050628662109f, HALF_PI_LO = -4.37113900018624283e-8f;

// sin and cos for |x| up to a few turns (NaN gives NaN)
__device__ __forceinline__ void sincos1(float x, float &sn, float &cs)
{
	const float q = rintf(x * 0.63661977236758134f);
	float r = fmaf(-q, HALF_PI_HI, x);
	r = fmaf(-q, HALF_PI_LO, r);
	const float r2 = r * r;
	const float s = fmaf(r * r2, fmaf(fmaf(-0.00019516977772582322f, r2, 0.008332176133990288f), r2,
	                                  -0.16666655242443085f), r);
	const float c = fmaf(r2 * r2, fmaf(fmaf(2.443809171381872e-05f, r2, -0.0013887364184483886f), r2,
	                                   0.04166664555668831f), fmaf(-0.5f, r2, 1.f));
	const int i = (int)q;
	const bool odd = i & 1;
	sn = __int_as_float(__float_as_int(odd ? c : s) ^ ((i & 2) << 30));
	cs = __int_as_float(__float_as_int(odd ? s : c) ^ (((i + 1) & 2) << 30));
}

// atan2(y, x) for finite arguments, the larger of them a normal number whose
// reciprocal is one too
__device__ __forceinline__ float atan2_1(float y, float x)
{
	const float ax = fabsf(x), ay = fabsf(y);
	const float q = div1(fminf(ax, ay), fmaxf(ax, ay)), q2 = q * q;
	float p = fmaf(-0.0018272141460329294f, q2, 0.011064446531236172f);
	p = fmaf(p, q2, -0.031455714255571365f);
	p = fmaf(p, q2, 0.0582345649600029f);
	p = fmaf(p, q2, -0.0841946005821228f);
	p = fmaf(p, q2, 0.10957576334476471f);
	p = fmaf(p, q2, -0.1426524519920349f);
	p = fmaf(p, q2, 0.19998638331890106f);
	p = fmaf(p, q2, -0.33333301544189453f);
	const float a = fmaf(q * q2, p, q);
	// pi/2 -+ a where |y| > |x|, pi - a for x < 0 below that
	const bool steep = ay > ax, neg = x < 0.f;
	const float k = steep ? HALF_PI_HI : (neg ? 2.f * HALF_PI_HI : 0.f);
	const float t = fmaf(k, HALF_PI_LO / HALF_PI_HI, steep != neg ? -a : a);
	return copysignf(k + t, y);
}

// ---- the mixture on a quad of lanes: lane k (= lane % 4) of a quad holds
// component k; sums over the quad pair lanes (0,1)(2,3) and then the pairs,
// with commutative adds, so that every lane of the quad holds the same bits.
// A quad is active or inactive as a whole.
static_assert(NK == 4, "one mixture component per lane of a quad");

template <int CTRL> __device__ __forceinline__ float quad_swap(float v)
{
	return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float quad_sum(float v)
{
	v += quad_swap<0xB1>(v); // quad_perm [1, 0, 3, 2]
	return v + quad_swap<0x4E>(v); // quad_perm [2, 3, 0, 1]
}

struct NCPq
{
	float s, w, t;
};

// component lane % 4 of the transform with MLP outputs y
__device__ __forceinline__ NCPq ncpq_params(const float *y)
{
	const int k = threadIdx.x & 3;
	const float m = fmaxf(fmaxf(y[NK], y[NK + 1]), fmaxf(y[NK + 2], y[NK + 3]));
	const float e = expf(y[NK + k] - m);
	NCPq p;
	p.w = e / quad_sum(e);
	p.s = expf(fminf(fmaxf(y[k], -8.f), 8.f));
	p.t = atan2f(y[2 * NK + 1], y[2 * NK]);
	return p;
}

// g(u), g'(u) of the mixture, every lane of the quad
__device__ __forceinline__ void ncpq_eval(NCPq const &p, float u, float &G, float &Gp)
{
	float sn, c;
	sincos1(0.5f * u, sn, c);
	const float d = fmaf(c, c, p.s * p.s * sn * sn); // e^-16 .. e^16
	G = quad_sum(p.w * (2.f * atan2_1(p.s * sn, c)));
	Gp = quad_sum(p.w * div1(p.s, d));
}

__device__ __forceinline__ float quad_min(float v)
{
	v = fminf(v, quad_swap<0xB1>(v));
	return fminf(v, quad_swap<0x4E>(v));
}
__device__ __forceinline__ float quad_max(float v)
{
	v = fmaxf(v, quad_swap<0xB1>(v));
	return fmaxf(v, quad_swap<0x4E>(v));
}

// u = g^-1(target), the evaluations on the quad (the bracket and the iterates
// are uniform over it).  g is a convex combination of the increasing maps
// g_k, so the root lies between the smallest and the largest closed-form
// component inverse g_k^-1(target) = 2 atan2(sin(target/2), s_k cos(target/2))
// (widened by a few ulps against their rounding); Newton starts from their
// w-weighted mean and continues as ncp_inverse.  It also stops once
// |g(u) - target| is at the rounding level of g (2.5e-7 max(1, |target|)):
// where g' is small the residual is noise and further steps would only wander
// inside the noise band (u is then as accurate as the output determines it).
__device__ __forceinline__ float ncpq_inverse(NCPq const &p, float target, float &Gp)
{
	float st, ct;
	sincos1(0.5f * target, st, ct);
	const float uk = fminf(fmaxf(2.f * atan2_1(st, p.s * ct), -PI_F), PI_F);
	float lo = quad_min(uk), hi = quad_max(uk), u = quad_sum(p.w * uk), G;
	lo = fmaxf(-PI_F, lo - 5e-7f * fmaxf(1.f, fabsf(lo)));
	hi = fminf(PI_F, hi + 5e-7f * fmaxf(1.f, fabsf(hi)));
	u = fminf(fmaxf(u, lo), hi);
	bool fresh = false; // G, Gp belong to the current u
	for (int b = 0; b < 40; ++b)
	{
		ncpq_eval(p, u, G, Gp);
		fresh = true;
		float f = G - target;
		if (fabsf(f) <= 2.5e-7f * fmaxf(1.f, fabsf(target)))
			break;
		if (f < 0.f)
			lo = u;
		else
			hi = u;
		if (hi - lo <= 2e-7f * fmaxf(1.f, fabsf(u)))
			break;
		float un = u - f * __builtin_amdgcn_rcpf(Gp);
		fresh = false;
		if (un > lo && un < hi)
		{
			bool done = fabsf(un - u) <= 2e-7f * fmaxf(1.f, fabsf(un));
			u = un;
			if (done)
				break;
		}
		else
			u = 0.5f * (lo + hi);
	}
	if (!fresh)
		ncpq_eval(p, u, G, Gp);
	return u;
}

// Adjoints of L = A (g(u) + t) - log g'(u), u = wrap(a - t), for one active
// variable a with MLP outputs y: dy[16] = dL/dy (through s, w and t), and
// the return value dL/da.
__device__ __forceinline__ float ncp_adjoint(const float *y, float u, float A, float (&dy)[16])
{
	NCP p = ncp_params(y);
	float cc = cosf(0.5f * u), sn = sinf(0.5f * u);
	float Gp = 0.f, Gpp = 0.f, gk[NK], gpk[NK], dgs[NK], dgps[NK];
	for (int k = 0; k < NK; ++k)
	{
		float s2 = p.s[k] * p.s[k];
		float d = fmaf(cc, cc, s2 * sn * sn);
		gk[k] = 2.f * atan2f(p.s[k] * sn, cc);
		gpk[k] = p.s[k] / d;
		dgs[k] = 2.f * sn * cc / d;
		dgps[k] = (cc * cc - s2 * sn * sn) / (d * d);
		Gp = fmaf(p.w[k], gpk[k], Gp);
		Gpp = fmaf(p.w[k], -p.s[k] * (s2 - 1.f) * sn * cc / (d * d), Gpp);
	}
	float iG = 1.f / Gp;
	float dLdt = A * (1.f - Gp) + Gpp * iG;
	float dLdw[NK], sw = 0.f;
	for (int k = 0; k < 16; ++k)
		dy[k] = 0.f;
	for (int k = 0; k < NK; ++k)
	{
		dLdw[k] = A * gk[k] - gpk[k] * iG;
		sw = fmaf(p.w[k], dLdw[k], sw);
		float dLds = p.w[k] * (A * dgs[k] - dgps[k] * iG);
		dy[k] = (y[k] > -8.f && y[k] < 8.f) ? p.s[k] * dLds : 0.f;
	}
	for (int k = 0; k < NK; ++k)
		dy[NK + k] = p.w[k] * (dLdw[k] - sw);
	float r2 = fmaf(p.ta, p.ta, p.tb * p.tb) + 1e-20f;
	dy[2 * NK] = dLdt * (-p.tb / r2);
	dy[2 * NK + 1] = dLdt * (p.ta / r2);
	return A * Gp - Gpp * iG;
}

// Weight-gradient accumulators of one wavefront (lane-owned tile fragments)
template <int NI> struct Grad
{
	static constexpr int NX = Layout<NI>::XS / 16;
	f4 w1[NX * 4], w2[16], w3[4];
	float b1, b2, b3;
	__device__ void zero()
	{
		for (int q = 0; q < NX * 4; ++q)
			w1[q] = f4{0.f, 0.f, 0.f, 0.f};
		for (int q = 0; q < 16; ++q)
			w2[q] = f4{0.f, 0.f, 0.f, 0.f};
		for (int q = 0; q < 4; ++q)
			w3[q] = f4{0.f, 0.f, 0.f, 0.f};
		b1 = b2 = b3 = 0.f;
	}
};

// MLP backward of one tile whose T.y() holds dL/dy (and T.x, T.h1, T.h2() the
// forward values): accumulates the weight gradients into G and writes
// dL/dx of rows r0 .. r0+15 (r < nrows) to dx[r * NI + feature]
template <int NI>
__device__ void mlp_backward(LW<NI> const &lw, Tile<NI> &T, Grad<NI> &G, float *__restrict__ dx, int r0, int nrows)
{
	constexpr int XS = Layout<NI>::XS;
	const int l = threadIdx.x & 63, lc = l & 15, rq = (l >> 4) * 4;
	// dW3 += H2^T dY, db3
	for (int i0 = 0; i0 < NH; i0 += 16)
		G.w3[i0 / 16] += tile_mm(T.h2() + i0, 1, NH, T.y(), 16, 1, 16);
	if (l < 16)
		for (int rr = 0; rr < 16; ++rr)
			G.b3 += T.y()[rr * 16 + l];
	// dA2 = (dY W3^T) * (1 - h2^2), into h2
	f4 dh2[4];
	for (int n0 = 0; n0 < NH; n0 += 16)
		dh2[n0 / 16] = tile_mm(T.y(), 16, 1, lw.w3 + n0 * 16, 1, 16, 16);
	wave_sync();
	for (int n0 = 0; n0 < NH; n0 += 16)
		for (int j = 0; j < 4; ++j)
		{
			float hv = T.h2()[(rq + j) * NH + n0 + lc];
			T.h2()[(rq + j) * NH + n0 + lc] = dh2[n0 / 16][j] * (1.f - hv * hv);
		}
	wave_sync();
	// dW2 += H1^T dA2, db2
	for (int i0 = 0; i0 < NH; i0 += 16)
		for (int n0 = 0; n0 < NH; n0 += 16)
			G.w2[(i0 / 16) * 4 + n0 / 16] += tile_mm(T.h1 + i0, 1, NH, T.h2() + n0, NH, 1, 16);
	for (int rr = 0; rr < 16; ++rr)
		G.b2 += T.h2()[rr * NH + l];
	// dA1 = (dA2 W2^T) * (1 - h1^2), into h1
	f4 dh1[4];
	for (int n0 = 0; n0 < NH; n0 += 16)
		dh1[n0 / 16] = tile_mm(T.h2(), NH, 1, lw.w2 + n0 * NH, 1, NH, NH);
	wave_sync();
	for (int n0 = 0; n0 < NH; n0 += 16)
		for (int j = 0; j < 4; ++j)
		{
			float hv = T.h1[(rq + j) * NH + n0 + lc];
			T.h1[(rq + j) * NH + n0 + lc] = dh1[n0 / 16][j] * (1.f - hv * hv);
		}
	wave_sync();
	// dW1 += X^T dA1, db1
	for (int i0 = 0; i0 < XS; i0 += 16)
		for (int n0 = 0; n0 < NH; n0 += 16)
			G.w1[(i0 / 16) * 4 + n0 / 16] += tile_mm(T.x + i0, 1, XS, T.h1 + n0, NH, 1, 16);
	for (int rr = 0; rr < 16; ++rr)
		G.b1 += T.h1[rr * NH + l];
	// dX = dA1 W1^T (feature columns < NI)
	for (int n0 = 0; n0 < XS; n0 += 16)
	{
		f4 dxt = tile_mm(T.h1, NH, 1, lw.w1 + n0 * NH, 1, NH, NH);
		for (int j = 0; j < 4; ++j)
		{
			int r = r0 + rq + j, f = n0 + lc;
			if (f < NI && r < nrows)
				dx[(long)r * NI + f] = dxt[j];
		}
	}
	wave_sync();
}

// the four wavefronts' accumulators, added in wavefront order, into the
// layer's per-configuration gradient pl[0 .. NP)
template <int NI> __device__ void store_grad(Grad<NI> const &G, float *__restrict__ pl)
{
	using Y = Layout<NI>;
	constexpr int XS = Y::XS;
	const int w = threadIdx.x >> 6, l = threadIdx.x & 63, lc = l & 15, rq = (l >> 4) * 4;
	for (int ww = 0; ww < 4; ++ww)
	{
		if (w == ww)
		{
			for (int i0 = 0; i0 < XS; i0 += 16)
				for (int n0 = 0; n0 < NH; n0 += 16)
					for (int j = 0; j < 4; ++j)
					{
						int k = i0 + rq + j, n = n0 + lc;
						if (k < NI)
						{
							float *dst = pl + Y::OW1 + k * NH + n;
							*dst = (ww ? *dst : 0.f) + G.w1[(i0 / 16) * 4 + n0 / 16][j];
						}
					}
			for (int i0 = 0; i0 < NH; i0 += 16)
				for (int n0 = 0; n0 < NH; n0 += 16)
					for (int j = 0; j < 4; ++j)
					{
						float *dst = pl + Y::OW2 + (i0 + rq + j) * NH + n0 + lc;
						*dst = (ww ? *dst : 0.f) + G.w2[(i0 / 16) * 4 + n0 / 16][j];
					}
			for (int i0 = 0; i0 < NH; i0 += 16)
				for (int j = 0; j < 4; ++j)
					if (lc < NO)
					{
						float *dst = pl + Y::OW3 + (i0 + rq + j) * NO + lc;
						*dst = (ww ? *dst : 0.f) + G.w3[i0 / 16][j];
					}
			pl[Y::OB1 + l] = (ww ? pl[Y::OB1 + l] : 0.f) + G.b1;
			pl[Y::OB2 + l] = (ww ? pl[Y::OB2 + l] : 0.f) + G.b2;
			if (l < NO)
				pl[Y::OB3 + l] = (ww ? pl[Y::OB3 + l] : 0.f) + G.b3;
		}
		__syncthreads();
	}
}

// initial weights of n parameters (layers of NP each): W ~ N(0, 1/fan_in) for
// the hidden layers, the last layer 1e-2 of that (identical components would
// receive identical gradients for ever) with the bias of the identity
// transform (s_k = 1, w uniform, t = 0)
template <int NI> __device__ void init_param(int i, float *p, uint64_t seed, uint32_t tag)
{
	using Y = Layout<NI>;
	int o = i % Y::NP;
	float v = 0.f;
	double sd = 0.0;
	if (o >= Y::OW1 && o < Y::OB1)
		sd = 1.0 / sqrt((double)NI);
	else if (o >= Y::OW2 && o < Y::OB2)
		sd = 1.0 / sqrt((double)NH);
	else if (o >= Y::OW3 && o < Y::OB3)
		sd = 1e-2 / sqrt((double)NH);
	if (sd > 0)
	{
		mesh_dev::u4 ctr = {(uint32_t)i, 0u, 0u, tag};
		mesh_dev::u4 r = mesh_dev::philox4x32_10(ctr, (uint32_t)seed, (uint32_t)(seed >> 32));
		double z0, z1;
		mesh_dev::normal_pair(r, &z0, &z1);
		v = (float)(z0 * sd);
	}
	if (o == Y::OB3 + 2 * NK)
		v = 1.f;
	p[i] = v;
}

} // namespace flow_mlp
