// Dense layers and circle maps shared by the U(1) learned flows (flow.hip:
// coupling layers on links, pcflow.hip: coupling layers on plaquettes).
//
// Per layer an MLP NI -> 64 -> 64 -> 10 (tanh) turns NI context features of
// an active variable into the parameters of a circle diffeomorphism
//   h(a) = g(wrap(a - t)) + t,  g(u) = sum_k w_k 2 atan(s_k tan(u / 2))
// (a mixture of NK = 4 non-compact projections; s_k = exp(clamp(y_k, -8, 8)),
// w = softmax(y_{4..7}), t = atan2(y_9, y_8)).  The dense layers run on FP32
// MFMA (v_mfma_f32_16x16x4_f32), or on BF16 MFMA with every number split in three,
// in 16-row tiles, one tile per wavefront, with the activations in registers; the
// backward pass forms the weight gradients as MFMA products over the rows of four
// tiles.
//
// Parameters of one layer, in order: W1 [NI][64], b1 [64], W2 [64][64],
// b2 [64], W3 [64][10], b3 [10].
#pragma once

#include <cstddef>

#include "mesh_internal.h"
#include "rng_dev.h"
#include "trig_dev.h"

namespace flow_mlp {

using mesh_dev::atan2_1;
using mesh_dev::div1;
using mesh_dev::sincos1;

constexpr int NK = 4;          // mixture components
constexpr int NH = 64;         // hidden width
constexpr int NO = 2 * NK + 2; // outputs
constexpr float PI_F = 3.14159265358979323846f;
constexpr float TWO_PI_F = 6.28318530717958647692f;

typedef float f4 __attribute__((ext_vector_type(4)));

template <int NI> struct Layout
{
	static_assert(NI % 4 == 0 && NI <= 48, "features: a multiple of 4, at most 48");
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

// tanh from the hardware exponential and reciprocal: absolute error a few
// 1e-7, saturating to +-1 (e = inf or 0)
__device__ __forceinline__ float tanh_fast(float x)
{
	const float e = __builtin_amdgcn_exp2f(x * 2.88539008177792681f); // exp(2 x)
	return fmaf(-2.f, __builtin_amdgcn_rcpf(1.f + e), 1.f);
}

template <bool FAST> __device__ __forceinline__ float act(float x) { return FAST ? tanh_fast(x) : tanhf(x); }

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

// two floats of memory that is aligned for one
struct __attribute__((packed, aligned(4))) Pair
{
	float x, y;
};

// One layer's parameters held in registers (two floats a lane per chunk, from
// 4-byte aligned memory) so that the next layer's global loads overlap the
// current layer's work.  store() writes the LDS image (the pad columns of
// W3/b3 stay as zero_pad() left them).
template <int NI, int THREADS> struct WeightRegsP
{
	using Y = Layout<NI>;
	static_assert(Y::NP % 2 == 0 && Y::OB1 % 2 == 0 && Y::OW2 % 2 == 0 && Y::OB2 % 2 == 0 && Y::OW3 % 2 == 0 &&
	                  Y::OB3 % 2 == 0 && NO % 2 == 0,
	              "pairs of parameters");
	static constexpr int NC = Y::NP / 2;
	static constexpr int PER = (NC + THREADS - 1) / THREADS;
	Pair v[PER];

	__device__ void load(const float *__restrict__ p)
	{
		const Pair *q = reinterpret_cast<const Pair *>(p);
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
			*reinterpret_cast<float2 *>(dst) = make_float2(v[i].x, v[i].y);
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
// The weights come a chunk of 16 ahead of their products; the scheduling
// barriers keep the loads there, which left alone are placed two products before
// their use, so that each pair of products waits out the LDS (plaquette flow,
// 16^2 sample, 256 chains: 47.2 -> 43.7 us).
template <int NI, bool FAST, class ROW>
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
	load(0, w[0]);
#pragma unroll
	for (int c = 0; c < C1 + 5; ++c)
	{
		if (c < C1 + 4)
			load(c + 1, w[(c + 1) & 1]);
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

// ---- the same products on the BF16 matrix units, to FP32's precision ------
//
// FP32 MFMA runs on the vector ALUs (the chip's FP32 rate is the same either
// way), so a tile's products and its activations, feature sums and circle maps
// add up; BF16 MFMA has units of its own.  A float is the sum of three BF16
// numbers, each the rounding of what the ones before it leave (8 + 8 + 8 bits
// with signs hold all 24), and of the nine products of two such sums the six
// that reach FP32's rounding are formed and accumulated in FP32: the three
// left out are below 2^-24 of the product.  Against 64 bits, 32 seeds of 64
// chains of a 32^2 proposal round: links 7.0e-7, log q 1.3e-9 of its value (FP32
// MFMA on tiles in LDS with the library's trigonometry: 8.3e-7 and 8.1e-9).  A round
// of 256 chains of 32^2: 224 -> 178 us with weights of order one, 209 -> 160 with the
// initial ones and 5% noise.
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// v[e] = p[0][e] + p[1][e] + p[2][e], two BF16 numbers a word
template <int N> struct Split
{
	typedef __bf16 vec __attribute__((ext_vector_type(N)));
	typedef uint32_t words __attribute__((ext_vector_type(N / 2)));
	words p[3];
	__device__ __forceinline__ vec part(int k) const { return __builtin_bit_cast(vec, p[k]); }
};
// a, b rounded to BF16 in the halves of a word (one instruction), and what it leaves of them
__device__ __forceinline__ uint32_t take_bf16(float &a, float &b)
{
	typedef __bf16 pair __attribute__((ext_vector_type(2)));
	const uint32_t w = __builtin_bit_cast(uint32_t, pair{(__bf16)a, (__bf16)b});
	a -= __uint_as_float(w << 16);
	b -= __uint_as_float(w & 0xffff0000u);
	return w;
}
template <int N> __device__ __forceinline__ Split<N> split(const float (&v)[N])
{
	Split<N> s;
#pragma unroll
	for (int e = 0; e < N; e += 2)
	{
		float a = v[e], b = v[e + 1];
#pragma unroll
		for (int k = 0; k < 3; ++k)
			s.p[k][e / 2] = take_bf16(a, b);
	}
	return s;
}

// LDS image of one layer's weights as the MFMA's A operands: lane l = 16 q + i
// of step t, column block b holds in element e the parts of the weight of
// output column 16 b + i and contraction index (t, q, e) -- for W2 and W3
// column 16 (2t + e / 4) + 4 q + e % 4 of the layer before, for W1 the quarter's
// feature row(q, 8 t + e); the features past the last eight are a step of four
template <int NI> struct alignas(16) LWS
{
	static constexpr int T8 = NI / 4 / 8, R4 = (NI / 4) % 8;
	static_assert(R4 <= 4, "the last features fill a step of four");
	bf8 w1[T8 ? T8 : 1][4][3][64];
	Split<4>::vec w1r[R4 ? 4 : 1][3][64];
	bf8 w2[2][4][3][64], w3[2][3][64];
	float b1[NH], b2[NH], b3[16];
};

// One layer's parameters in registers, the floats of a thread's operand
// fragments, so that the next layer's global loads overlap the current layer's
// work; store() splits them into the LDS image.
template <int NI, int THREADS, class ROW> struct WeightFrags
{
	using Y = Layout<NI>;
	using W = LWS<NI>;
	static constexpr int N2 = 512 / THREADS; // fragments of W2 a thread
	static_assert(W::T8 == 1 && W::R4 > 0 && (THREADS == 256 || THREADS == 512), "one step of eight features and a rest");
	float w1[8], w1r[4], w2[N2][8], w3[8] = {}, b[1] = {}; // (zero past column NO)

	// a fragment's block b (of W1: 0..3) and lane
	static __device__ __forceinline__ bool has_w1() { return threadIdx.x < 256; }
	static __device__ __forceinline__ bool has_w1r() { return THREADS == 256 || threadIdx.x >= 256; }
	static __device__ __forceinline__ bool has_w3() { return threadIdx.x < 128; }

	// (unsigned offsets from the uniform p: one register an address)
	__device__ __forceinline__ void load(const float *__restrict__ p)
	{
		const unsigned l = threadIdx.x & 63, i = l & 15, q = l >> 4, f = (threadIdx.x >> 6) & 3;
		if (has_w1())
#pragma unroll
			for (int e = 0; e < 8; ++e)
				w1[e] = p[Y::OW1 + (unsigned)ROW::row(q, e) * NH + 16 * f + i];
		if (has_w1r())
#pragma unroll
			for (int e = 0; e < 4; ++e)
				w1r[e] = e < W::R4 ? p[Y::OW1 + (unsigned)ROW::row(q, 8 * W::T8 + (e < W::R4 ? e : 0)) * NH + 16 * f + i] : 0.f;
#pragma unroll
		for (int k = 0; k < N2; ++k)
		{
			const unsigned u = (threadIdx.x >> 6) + k * (THREADS / 64), o = (32 * (u >> 2) + 4 * q) * NH + 16 * (u & 3) + i;
#pragma unroll
			for (int e = 0; e < 8; ++e)
				w2[k][e] = p[Y::OW2 + o + (16 * (e / 4) + e % 4) * NH];
		}
		if (has_w3() && i < NO)
		{
			const unsigned o = (32 * (threadIdx.x >> 6) + 4 * q) * NO + i;
#pragma unroll
			for (int e = 0; e < 8; ++e)
				w3[e] = p[Y::OW3 + o + (16 * (e / 4) + e % 4) * NO];
		}
		// the biases: b1, b2, b3 by the first 138 threads
		const unsigned x = threadIdx.x;
		if (x < 2 * NH + NO)
			b[0] = p[x < NH ? Y::OB1 + x : (x < 2 * NH ? Y::OB2 + x - NH : Y::OB3 + x - 2 * NH)];
	}

	// infinite weights as the largest BF16 number: a part of an activation may
	// be 0, and 0 times infinity would not be what the activation times it is
	static __device__ __forceinline__ float finite(float v)
	{
		return fabsf(v) > 3.38953139e38f ? copysignf(3.38953139e38f, v) : v;
	}
	template <int N, class DST> static __device__ __forceinline__ void put(const float (&v)[N], DST *dst, int l)
	{
		float w[N];
#pragma unroll
		for (int e = 0; e < N; ++e)
			w[e] = finite(v[e]);
		const Split<N> s = split<N>(w);
#pragma unroll
		for (int k = 0; k < 3; ++k)
			dst[k][l] = s.part(k);
	}
	__device__ __forceinline__ void store(W &lw) const
	{
		const int l = threadIdx.x & 63, f = (threadIdx.x >> 6) & 3;
		if (has_w1())
			put<8>(w1, lw.w1[0][f], l);
		if (has_w1r())
			put<4>(w1r, lw.w1r[f], l);
#pragma unroll
		for (int k = 0; k < N2; ++k)
		{
			const int u = (threadIdx.x >> 6) + k * (THREADS / 64);
			put<8>(w2[k], lw.w2[u >> 2][u & 3], l);
		}
		if (has_w3())
			put<8>(w3, lw.w3[threadIdx.x >> 6], l);
		const int x = threadIdx.x;
		if (x < NH)
			lw.b1[x] = b[0];
		else if (x < 2 * NH)
			lw.b2[x - NH] = b[0];
		else if (x < 2 * NH + 16)
			lw.b3[x - 2 * NH] = b[0];
	}
};

// mlp_rows on the split weights.  A part of the weights is read once for the
// products it is in (with the activations' parts 0; 1, 0; 2, 1, 0), one part
// ahead of them: the scheduling barriers let arithmetic through but no LDS
// read, which left alone are all placed early and take half the wavefronts'
// registers.
template <int NI, bool FAST>
__device__ __forceinline__ f4 mlp_rows_split(LWS<NI> const &lw, const float (&x)[NI / 4])
{
	using W = LWS<NI>;
	const int l = threadIdx.x & 63, q4 = (l >> 4) * 4;
	// acc[b] += the six products of weight fragments at(b, part) and activation parts s
	auto products = [&](auto at, auto const &s, auto mm, auto &acc) {
		constexpr int B = sizeof(acc) / sizeof(f4);
		decltype(at(0, 0)) w[2][B];
#pragma unroll
		for (int b = 0; b < B; ++b)
			w[0][b] = at(b, 2);
#pragma unroll
		for (int k = 2; k >= 0; --k)
		{
			if (k > 0)
#pragma unroll
				for (int b = 0; b < B; ++b)
					w[(k + 1) & 1][b] = at(b, k - 1);
			__builtin_amdgcn_sched_barrier(1);
#pragma unroll
			for (int j = 2 - k; j >= 0; --j)
#pragma unroll
				for (int b = 0; b < B; ++b)
					acc[b] = mm(w[k & 1][b], s.part(j), acc[b]);
		}
	};
	auto mm8 = [](bf8 a, bf8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); };
	auto mm4 = [](Split<4>::vec a, Split<4>::vec b, f4 c) {
		return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0,
		                                                 0);
	};
	f4 h[4], g[4], y[1];
#pragma unroll
	for (int b = 0; b < 4; ++b)
	{
		h[b] = *reinterpret_cast<const f4 *>(lw.b1 + 16 * b + q4);
		g[b] = *reinterpret_cast<const f4 *>(lw.b2 + 16 * b + q4);
	}
	y[0] = *reinterpret_cast<const f4 *>(lw.b3 + q4);
	float v[8], r[4];
#pragma unroll
	for (int e = 0; e < 8; ++e)
		v[e] = x[e];
#pragma unroll
	for (int e = 0; e < 4; ++e)
		r[e] = e < W::R4 ? x[8 + (e < W::R4 ? e : 0)] : 0.f;
	products([&](int b, int k) { return lw.w1[0][b][k][l]; }, split<8>(v), mm8, h);
	products([&](int b, int k) { return lw.w1r[b][k][l]; }, split<4>(r), mm4, h);
	auto parts = [](f4 a, f4 b) {
		const float v[8] = {act<FAST>(a[0]), act<FAST>(a[1]), act<FAST>(a[2]), act<FAST>(a[3]),
		                    act<FAST>(b[0]), act<FAST>(b[1]), act<FAST>(b[2]), act<FAST>(b[3])};
		return split<8>(v);
	};
#pragma unroll
	for (int t = 0; t < 2; ++t)
		products([&](int b, int k) { return lw.w2[t][b][k][l]; }, parts(h[2 * t], h[2 * t + 1]), mm8, g);
#pragma unroll
	for (int t = 0; t < 2; ++t)
		products([&](int, int k) { return lw.w3[t][k][l]; }, parts(g[2 * t], g[2 * t + 1]), mm8, y);
	return y[0];
}

// outputs of mlp_rows to y[row * YS + column] (one wavefront's scratch, 16 YS floats)
__device__ __forceinline__ void put_outputs(float *y, f4 v)
{
	const int l = threadIdx.x & 63;
	*reinterpret_cast<f4 *>(y + (l & 15) * YS + (l >> 4) * 4) = v;
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
// (widened by a few ulps against their rounding).  Newton starts from their
// w-weighted mean; every evaluation moves one end of the bracket to the iterate,
// a step that leaves the bracket is replaced by its midpoint, and a step or a
// bracket below 2e-7 max(1, |u|) (an FP32 ulp of u is up to 2.4e-7) ends it, or 40
// evaluations.  NEAR: it also stops at |g(u) - target| <= 2.5e-7 max(1, |target|).
// Where |target| is well below 1 that is above g's rounding: on maps whose s_k are
// all small u can be off by 5e-4 (s_k = e^-7.5) where the iteration reaches 5e-7,
// so only the plaquette coupling flow, which has always used it, does.
template <bool NEAR> __device__ __forceinline__ float ncpq_inverse(NCPq const &p, float target, float &Gp)
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
		if (NEAR ? fabsf(f) <= 2.5e-7f * fmaxf(1.f, fabsf(target)) : f == 0.f)
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
// variable a with MLP outputs y[16] on its quad: overwrites y with dL/dy
// (through s, w and t; the columns from NO on zero) and returns dL/da in every
// lane of the quad.  live = false: a row without a variable, dL/dy = 0.  (The
// direction (y_8, y_9) passes dL/dt / r, r its length: a variable that the MLP leaves
// with r of order 1e-3 carries most of a gradient's error, whatever the products'
// rounding.  80 inputs, plaquette flow 16^2 against 64 bits: median 2.4e-7, 95% below
// 4.0e-7, largest 1.8e-5.)
__device__ __forceinline__ float ncpq_adjoint(NCPq const &p, float *y, float u, float A, bool live)
{
	const int k = threadIdx.x & 3;
	float sn, c;
	sincos1(0.5f * u, sn, c);
	const float s2 = p.s * p.s, d = fmaf(c, c, s2 * sn * sn), id = div1(1.f, d);
	const float g = 2.f * atan2_1(p.s * sn, c), gp = p.s * id;
	const float dgs = 2.f * sn * c * id, dgps = (c * c - s2 * sn * sn) * (id * id);
	const float Gp = quad_sum(p.w * gp), Gpp = quad_sum(p.w * (-p.s * (s2 - 1.f) * sn * c * (id * id)));
	const float iG = div1(1.f, Gp);
	const float dLdt = A * (1.f - Gp) + Gpp * iG;
	const float dLdw = A * g - gp * iG, sw = quad_sum(p.w * dLdw);
	const float yk = y[k], ta = y[2 * NK], tb = y[2 * NK + 1];
	const float r2 = fmaf(ta, ta, tb * tb) + 1e-20f;
	wave_sync(); // every lane of the quad has read y
	y[k] = live && yk > -8.f && yk < 8.f ? p.s * (p.w * (A * dgs - dgps * iG)) : 0.f;
	y[NK + k] = live ? p.w * (dLdw - sw) : 0.f;
	y[2 * NK + k] = live && k < 2 ? dLdt * ((k ? ta : -tb) / r2) : 0.f;
	y[2 * NK + 4 + k] = 0.f;
	return A * Gp - Gpp * iG;
}

// ---- backward of four tiles, one on each of a workgroup's four wavefronts
//
// The adjoints run back through the layers in registers just as the
// activations ran forward (mlp_rows).  The weight gradients contract over the
// rows: the tiles' activations and adjoints go to LDS transposed, [column]
// [row], and wavefront w forms block w of the gradient's columns (of W3: of its
// rows) over the 64 rows of all four tiles, so that no sum over the wavefronts
// is left and a wavefront's accumulators are a quarter of the gradient.  Row
// stride TS: 16 consecutive columns are read from 16 different groups of four
// banks, and a column's 16 rows written to 16 banks.
constexpr int TS = 20;

template <int NI> struct BackBuf
{
	alignas(16) float a[4][NH * TS], b[4][NH * TS];
	alignas(16) float y[4][16 * TS]; // outputs of mlp_rows, then dL/dy, then its transpose (YS = TS)
	static_assert(YS == TS && NI <= NH, "the outputs and their transpose share their storage");
};

// gradient accumulators of wavefront w: columns 16 w + l % 16 of W1 (rows: the
// features row(4 b + j) of the lane's quarter) and W2 (rows 16 b + 4 q + j),
// rows 16 w + 4 q + j of W3, and the biases' sums over the lane's rows
template <int NI> struct GradP
{
	static constexpr int NB = (NI / 4 + 3) / 4; // blocks of four features of a quarter
	f4 w1[NB], w2[4], w3;
	float b1, b2, b3;
	__device__ void zero()
	{
#pragma unroll
		for (int b = 0; b < NB; ++b)
			w1[b] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
		for (int b = 0; b < 4; ++b)
			w2[b] = f4{0.f, 0.f, 0.f, 0.f};
		w3 = f4{0.f, 0.f, 0.f, 0.f};
		b1 = b2 = b3 = 0.f;
	}
};

__device__ __forceinline__ f4 mm4(f4 a, f4 b, f4 c)
{
#pragma unroll
	for (int j = 0; j < 4; ++j)
		c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
	return c;
}

// a lane's columns 16 b + 4 q + j of its row to t[column * TS + row]
template <int NB> __device__ __forceinline__ void put_columns(float *t, f4 const (&v)[NB])
{
	const int l = threadIdx.x & 63, q4 = (l >> 4) * 4;
#pragma unroll
	for (int b = 0; b < NB; ++b)
#pragma unroll
		for (int j = 0; j < 4; ++j)
			t[(16 * b + q4 + j) * TS + (l & 15)] = v[b][j];
}

// One round: x, h1, h2 from mlp_rows on this wavefront's tile; B.y[w] holds
// its dL/dy (ncpq_adjoint).  Adds to G and returns in dx[b][j] the adjoint of
// feature row(q, 4 b + j), q the lane's quarter.  Called by all 256 threads.
template <int NI, class ROW>
__device__ __forceinline__ void mlp_rows_backward(LWP<NI> const &lw, BackBuf<NI> &B, const float (&x)[NI / 4], ROW row,
                                                  f4 const (&h1)[4], f4 const (&h2)[4], GradP<NI> &G,
                                                  f4 (&dx)[GradP<NI>::NB])
{
	constexpr int NS = NI / 4, NB = GradP<NI>::NB;
	const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l & 15, q4 = (l >> 4) * 4;
	const f4 zero = {0.f, 0.f, 0.f, 0.f};
	auto sum = [](f4 v) { return (v[0] + v[1]) + (v[2] + v[3]); };
	auto at = [&](const float *t, int c) { return *reinterpret_cast<const f4 *>(t + (c + i) * TS + q4); };
	f4 dy[1] = {*reinterpret_cast<const f4 *>(B.y[w] + i * TS + q4)};
	wave_sync();
	put_columns(B.y[w], dy);
	put_columns(B.a[w], h2);
	__syncthreads();
	// dW3 = H2^T dY, dA2 = (dY W3^T) (1 - h2^2)
	f4 d2[4], d1[4];
#pragma unroll
	for (int t = 0; t < 4; ++t)
	{
		const f4 v = at(B.y[t], 0);
		G.w3 = mm4(at(B.a[t], 16 * w), v, G.w3);
		G.b3 += sum(v);
	}
#pragma unroll
	for (int b = 0; b < 4; ++b)
		d2[b] = mm4(*reinterpret_cast<const f4 *>(lw.w3 + (16 * b + i) * W3S + q4), dy[0], zero) * (1.f - h2[b] * h2[b]);
	__syncthreads();
	put_columns(B.a[w], h1);
	put_columns(B.b[w], d2);
	__syncthreads();
	// dW2 = H1^T dA2, dA1 = (dA2 W2^T) (1 - h1^2)
#pragma unroll
	for (int t = 0; t < 4; ++t)
	{
		const f4 v = at(B.b[t], 16 * w);
		G.b2 += sum(v);
#pragma unroll
		for (int b = 0; b < 4; ++b)
			G.w2[b] = mm4(at(B.a[t], 16 * b), v, G.w2[b]);
	}
#pragma unroll
	for (int b = 0; b < 4; ++b)
	{
		f4 acc = zero;
#pragma unroll
		for (int k = 0; k < 4; ++k)
			acc = mm4(*reinterpret_cast<const f4 *>(lw.w2 + (16 * b + i) * WS + 16 * k + q4), d2[k], acc);
		d1[b] = acc * (1.f - h1[b] * h1[b]);
	}
	__syncthreads();
	f4 xb[NB];
#pragma unroll
	for (int b = 0; b < NB; ++b)
#pragma unroll
		for (int j = 0; j < 4; ++j)
			xb[b][j] = 4 * b + j < NS ? x[4 * b + j] : 0.f;
	put_columns(B.a[w], xb);
	put_columns(B.b[w], d1);
	__syncthreads();
	// dW1 = X^T dA1, dX = dA1 W1^T
#pragma unroll
	for (int t = 0; t < 4; ++t)
	{
		const f4 v = at(B.b[t], 16 * w);
		G.b1 += sum(v);
#pragma unroll
		for (int b = 0; b < NB; ++b)
			G.w1[b] = mm4(at(B.a[t], 16 * b), v, G.w1[b]);
	}
#pragma unroll
	for (int b = 0; b < NB; ++b)
	{
		// row i of the product: feature 4 b + i % 4 of quarter i / 4 (past NS: any, not used)
		const int s = 4 * b + (i & 3), f = row(i >> 2, s < NS ? s : 0);
		f4 acc = zero;
#pragma unroll
		for (int k = 0; k < 4; ++k)
			acc = mm4(*reinterpret_cast<const f4 *>(lw.w1 + f * WS + 16 * k + q4), d1[k], acc);
		dx[b] = acc;
	}
	__syncthreads(); // the buffers are free for the next round
}

// a layer's gradient of one configuration, pl[0 .. NP)
template <int NI, class ROW> __device__ __forceinline__ void store_grad(GradP<NI> const &G, ROW row, float *__restrict__ pl)
{
	using Y = Layout<NI>;
	const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l & 15, q = l >> 4, n = 16 * w + i;
#pragma unroll
	for (int b = 0; b < GradP<NI>::NB; ++b)
#pragma unroll
		for (int j = 0; j < 4; ++j)
			if (4 * b + j < NI / 4)
				pl[Y::OW1 + row(q, 4 * b + j) * NH + n] = G.w1[b][j];
#pragma unroll
	for (int b = 0; b < 4; ++b)
#pragma unroll
		for (int j = 0; j < 4; ++j)
			pl[Y::OW2 + (16 * b + 4 * q + j) * NH + n] = G.w2[b][j];
	if (i < NO)
#pragma unroll
		for (int j = 0; j < 4; ++j)
			pl[Y::OW3 + (16 * w + 4 * q + j) * NO + i] = G.w3[j];
	// the biases' sums over the quarters
	auto quarters = [](float v) {
		v += __shfl_xor(v, 16, 64);
		return v + __shfl_xor(v, 32, 64);
	};
	const float b1 = quarters(G.b1), b2 = quarters(G.b2), b3 = quarters(G.b3);
	if (q == 0)
	{
		pl[Y::OB1 + n] = b1;
		pl[Y::OB2 + n] = b2;
		if (w == 0 && i < NO)
			pl[Y::OB3 + i] = b3;
	}
}

// grad[i] = scale * sum_c partial[c][i], in a fixed order: thread group g of
// four takes the configurations c = g (mod 4), so that four times the loads are
// in flight (one thread an entry left 930 wavefronts of serial loads on the
// chip: 62 us for 256 configurations of 8 layers)
__global__ __launch_bounds__(256) static void k_grad_reduce(int n, const float *__restrict__ partial, int batch,
                                                            float scale, float *__restrict__ grad)
{
	__shared__ double part[4][64];
	const int g = threadIdx.x >> 6, l = threadIdx.x & 63, i = blockIdx.x * 64 + l;
	double s = 0.0;
	if (i < n)
	{
		int c = g;
		for (; c + 28 < batch; c += 32)
		{
			float v[8];
#pragma unroll
			for (int k = 0; k < 8; ++k)
				v[k] = partial[(long)(c + 4 * k) * n + i];
#pragma unroll
			for (int k = 0; k < 8; ++k)
				s += v[k];
		}
		for (; c < batch; c += 4)
			s += partial[(long)c * n + i];
	}
	part[g][l] = s;
	__syncthreads();
	if (g == 0 && i < n)
		grad[i] = (float)((((part[0][l] + part[1][l]) + part[2][l]) + part[3][l]) * scale);
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
