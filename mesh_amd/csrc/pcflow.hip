// Plaquette coupling flow for 2-d U(1): gauge-equivariant coupling layers
// acting on the plaquettes, used as an independence proposal beside HMC (no
// counterpart in the reference; U(1) conventions of u1.hip).
//
// Variables: the V - 1 free plaquettes of an L0 x L1 torus (all but the last,
// P(L0-1, L1-1), which the others fix); the links follow by the integration
// of u1_plaq.h with uniform holonomies and gauge, so the flow acts on
// gauge-invariant variables only and its density over links is gauge
// invariant.
//  * prior: every free plaquette uniform on [-pi, pi);
//  * layer l: mask class m = l % 4; the plaquettes with
//    (x0 mod 2, x1 mod 2) = (m % 2, m / 2) are active (the last excluded),
//    every other one is frozen.  Each active plaquette a moves to
//    h(a) = g(wrap(a - t)) + t with the mixture g of flow_mlp.h, its
//    parameters from an MLP 40 -> 64 -> 64 -> 10 of the frozen 3x3
//    neighbourhood: (cos, sin) of the 8 surrounding plaquettes (1x1 loops),
//    of the 8 1x2 loops formed by neighbouring pairs of them and of the 4
//    L-shaped loops that each 2x2 square of the neighbourhood leaves when its
//    (active) centre is taken out (a loop's angle is the sum of its
//    plaquettes); the last plaquette enters the context as 0 (it is not a
//    variable of the flow);
//  * log q(U) = -sum over layers and active plaquettes of log g'
//    - (V - 1) log 2 pi (prior) - (V + 1) log 2 pi (holonomies, gauge).
// Within a layer the active plaquettes see only frozen ones, so the map is
// triangular with the exact log-determinant above, and it does not perturb
// any plaquette it has not transformed (a link-space coupling layer moves a
// second, passive plaquette with every link it updates).
//
// Kernels: one workgroup per configuration, plaquettes in LDS, the dense layers
// on MFMA (flow_mlp.h): BF16 MFMA on split numbers in the forward and inverse
// kernels, FP32 MFMA in the backward one.
#include "flow_mlp.h"
#include "mesh_internal.h"
#include "rng_dev.h"
#include "u1_plaq.h"

using namespace mesh_dev;
namespace FM = flow_mlp;
using u1_plaq::block_sum;
using u1_plaq::plaqp;
using u1_plaq::wrapd;

namespace {

struct PCGeo : u1_plaq::PGeo
{
	unsigned hm; // ceil(2^20 / (L1 / 2)), see active_xy
};

constexpr int NI = 40; // features: 20 loops, (cos, sin) each
constexpr int NP_LAYER = FM::Layout<NI>::NP;
constexpr int MAX_LAYERS = 64;
constexpr int THREADS = 256; // of the backward kernel
// Forward and inverse run on 512 threads from WIDE_V plaquettes on, where each
// of the eight wavefronts has a tile in a layer (V / 4 >= 8 * 16), unless the
// launch has more workgroups than CUs and two of 256 threads fit a CU's LDS
// (V <= PAIR_V): those run side by side without each other's barriers.  256
// chains, initial weights with 5% noise: sample 32^2 103 us on 256 threads, 90 on 512,
// 64^2 342 and 282; propose (512 workgroups) 32^2 161 and 179, 64^2 772 and 617.
constexpr int WIDE_V = 512, PAIR_V = 1664;
constexpr bool FAST = true; // tanh_fast in every kernel of this flow
constexpr uint32_t TAG_PCFZ = 0x5043465au; // prior, holonomies, gauge
constexpr uint32_t TAG_PCFI = 0x50434649u; // initial weights
constexpr double LOG_2PI = 1.8378770664093454836;

// offset of ring position k = 0..7 around a plaquette, in order around it
__device__ __forceinline__ void ring(int k, int &d0, int &d1)
{
	d0 = (k <= 2) ? -1 : ((k >= 4 && k <= 6) ? 1 : 0);
	d1 = (k == 0 || k == 6 || k == 7) ? -1 : ((k >= 2 && k <= 4) ? 1 : 0);
}

// site (x0, x1) with one periodic step either way
__device__ __forceinline__ int sitew(PCGeo const &g, int x0, int x1)
{
	x0 = x0 < 0 ? x0 + g.L0 : (x0 >= g.L0 ? x0 - g.L0 : x0);
	x1 = x1 < 0 ? x1 + g.L1 : (x1 >= g.L1 ? x1 - g.L1 : x1);
	return x0 * g.L1 + x1;
}

// active plaquette r of mask class m
__device__ __forceinline__ void active_xy(PCGeo const &g, int m, int r, int &x0, int &x1)
{
	// r < 1024 and h <= 512: r / h = r ceil(2^20 / h) >> 20 exactly, since
	// r (h ceil(2^20 / h) - 2^20) < 2^20
	const int h = g.L1 >> 1, i = (int)(((unsigned)r * g.hm) >> 20), j = r - i * h;
	x0 = (m & 1) + 2 * i;
	x1 = (m >> 1) + 2 * j;
}
__device__ __forceinline__ int n_active(PCGeo const &g, int m) { return (g.V >> 2) - (m == 3 ? 1 : 0); }
// (cos, sin) of the sum of two angles
__device__ __forceinline__ float2 cs_add(float2 a, float2 b)
{
	return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.y, b.x, a.x * b.y));
}

__device__ __forceinline__ float2 sincos2(float a)
{
	float s, c;
	FM::sincos1(a, s, c);
	return make_float2(c, s);
}

// LDS of the forward and inverse kernels of NT threads
template <int NT> struct PCSharedF
{
	FM::LWS<NI> lw;
	float y[NT / 64][16 * FM::YS];
	double red[4][NT / 64];
};
// LDS of the backward kernel
struct PCSharedB
{
	FM::LWP<NI> lw;
	FM::BackBuf<NI> buf;
	double red[4][4];
};

// A lane's share of the 20 context loops of its row's plaquette: quarter q of
// the wavefront takes ring plaquettes 2q and 2q + 1, the 1x2 loops (2q, 2q + 1)
// and (2q - 1, 2q) and the L-shaped loop (2q - 1, 2q, 2q + 1), so three gathers
// give its ten features.  rg: the loops' (cos, sin), in that order; row(s): the
// feature index of x[s].
struct LaneLoops
{
	int q, d0[3], d1[3]; // quarter; offsets of ring plaquettes 2q - 1, 2q, 2q + 1
	__device__ LaneLoops()
	{
		q = (threadIdx.x >> 4) & 3;
		ring((2 * q + 7) & 7, d0[0], d1[0]);
		ring(2 * q, d0[1], d1[1]);
		ring(2 * q + 1, d0[2], d1[2]);
	}
	// index of the parameters' feature that is x[s] of quarter q
	static __device__ __forceinline__ int row(int q, int s)
	{
		return s < 4 ? 4 * q + s : (s < 6 ? 12 + 4 * q + s : (s < 8 ? 10 + 2 * ((2 * q + 7) & 7) + s : 24 + 2 * q + s));
	}
	__device__ __forceinline__ void features(PCGeo const &g, const float2 *cs, int x0, int x1, float (&x)[NI / 4]) const
	{
		const float2 a = cs[sitew(g, x0 + d0[0], x1 + d1[0])], b = cs[sitew(g, x0 + d0[1], x1 + d1[1])],
		             c = cs[sitew(g, x0 + d0[2], x1 + d1[2])];
		const float2 p = cs_add(b, c), m = cs_add(a, b), t = cs_add(m, c);
		x[0] = b.x, x[1] = b.y, x[2] = c.x, x[3] = c.y, x[4] = p.x, x[5] = p.y, x[6] = m.x, x[7] = m.y, x[8] = t.x,
		x[9] = t.y;
	}
};

// One layer on the workgroup: wavefront w takes tiles w, w + NT / 64, ... of
// the NA active plaquettes: features and MLP in registers (mlp_rows_split), then the
// circle map on quads (lane 4i + k: row i of the tile, mixture component k),
// to which the outputs go through 1.25 KB of LDS.  Features read only frozen
// plaquettes, so a wavefront may move its active ones while the others still
// read theirs.  INV: apply g^-1 (the inverse pass).  Adds log g' to ld.
template <bool INV, int NT>
__device__ __forceinline__ void layer_apply(PCGeo const &g, LaneLoops const &ll, float *phi, float2 *cs, int m,
                                            PCSharedF<NT> &sh, double &ld)
{
	const int w = threadIdx.x >> 6, l = threadIdx.x & 63, NA = n_active(g, m), ntile = (NA + 15) / 16;
	float *y = sh.y[w];
	for (int tix = w; tix < ntile; tix += NT / 64)
	{
		int x0, x1;
		// rows beyond NA repeat the last one; nothing reads their outputs
		active_xy(g, m, min(tix * 16 + (l & 15), NA - 1), x0, x1);
		float x[NI / 4];
		ll.features(g, cs, x0, x1, x);
		FM::put_outputs(y, FM::mlp_rows_split<NI, FAST>(sh.lw, x));
		FM::wave_sync();
		const int row = l >> 2, r = tix * 16 + row;
		if (r < NA)
		{
			active_xy(g, m, r, x0, x1);
			const int xs = x0 * g.L1 + x1;
			const FM::NCPq p = FM::ncpq_params(&y[row * FM::YS]);
			const float a = FM::wrapf(phi[xs] - p.t);
			float v, Gp;
			if (INV)
				v = FM::ncpq_inverse<true>(p, a, Gp);
			else
				FM::ncpq_eval(p, a, v, Gp);
			if ((l & 3) == 0)
			{
				const float nx = FM::wrapf(v + p.t);
				phi[xs] = nx;
				cs[xs] = sincos2(nx);
				ld += (double)logf(Gp);
			}
		}
		FM::wave_sync();
	}
}

// z uniform -> free plaquettes -> links.  phi_layers (optional): the input of
// every layer; phi_final (optional): the output; theta_out (optional): the
// links.  out[2c + {0,1}] = {log q, S/beta}, S of the links when they are
// formed, else of the plaquettes (the last one = -sum of the free ones).
// LDS: phi[V], cs[V] (then the links' scratch), al[V].
template <int NT>
__device__ __forceinline__ void pc_forward(PCGeo const &g, int nl, const float *__restrict__ params, uint64_t seed,
                                           uint32_t step, float *theta_out, float *phi_layers, float *phi_final,
                                           double *out, int c, float *dyn, PCSharedF<NT> &sh)
{
	float *phi = dyn;
	float2 *cs = reinterpret_cast<float2 *>(dyn + g.V);
	float *al = dyn + 3 * g.V;
	const uint32_t cc = (uint32_t)c << 1;
	FM::WeightFrags<NI, NT, LaneLoops> wr;
	const LaneLoops ll;
	wr.load(params);
	for (int x = threadIdx.x; x < g.V; x += NT)
	{
		const float z = x < g.V - 1 ? u1_plaq::uniform_angle(seed, step, (uint32_t)x, cc, TAG_PCFZ) : 0.f;
		phi[x] = z;
		cs[x] = sincos2(z);
		al[x] = u1_plaq::uniform_angle(seed, step, (uint32_t)x, cc | 1u, TAG_PCFZ);
	}
	double ld = 0.0;
	for (int layer = 0; layer < nl; ++layer)
	{
		__syncthreads(); // the previous layer is done with the weights and the plaquettes
		wr.store(sh.lw);
		if (phi_layers)
			for (int x = threadIdx.x; x < g.V; x += NT)
				phi_layers[((long)c * nl + layer) * g.V + x] = phi[x];
		__syncthreads();
		if (layer + 1 < nl)
			wr.load(params + (long)(layer + 1) * NP_LAYER);
		layer_apply<false, NT>(g, ll, phi, cs, layer & 3, sh, ld);
	}
	__syncthreads();
	if (phi_final)
		for (int x = threadIdx.x; x < g.V; x += NT)
			phi_final[(long)c * g.V + x] = phi[x];
	double v[3] = {ld, 0.0, 0.0}; // log det, S of the free plaquettes, their sum
	for (int x = threadIdx.x; x < g.V - 1; x += NT)
	{
		v[1] += 1.0 - cos1((double)phi[x]);
		v[2] += (double)phi[x];
	}
	block_sum<3>(v, sh.red);
	double S = v[1] + (1.0 - cos(wrapd(-v[2])));
	if (theta_out)
	{
		float *o = theta_out + (long)c * 2 * g.V;
		const float h0 = u1_plaq::uniform_angle(seed, step, (uint32_t)g.V, cc, TAG_PCFZ);
		const float h1 = u1_plaq::uniform_angle(seed, step, (uint32_t)g.V + 1u, cc, TAG_PCFZ);
		float *t = reinterpret_cast<float *>(cs);
		u1_plaq::links_from_plaquettes(g, phi, h0, h1, al, t, o, NT);
		__syncthreads();
		double s[1] = {0.0};
		for (int x = threadIdx.x; x < g.V; x += NT)
		{
			const int x0 = x / g.L1, x1 = x - x0 * g.L1;
			s[0] += 1.0 - cos1((double)plaqp(g, t, x0, x1));
		}
		block_sum<1>(s, sh.red);
		S = s[0];
	}
	if (threadIdx.x == 0)
	{
		out[2 * c + 0] = -v[0] - 2.0 * g.V * LOG_2PI;
		out[2 * c + 1] = S;
	}
}

// log q of given links: plaquettes, then the layers in reverse with g^-1.
// out[2c + {0,1}] = {log q(U), S(U)/beta}; z_out (optional): the prior draws,
// V per configuration (the last 0).  LDS: the links (then cs[V]), phi[V].
template <int NT>
__device__ __forceinline__ void pc_inverse(PCGeo const &g, int nl, const float *__restrict__ params,
                                           const float *__restrict__ theta, float *z_out, double *out, int c,
                                           float *dyn, PCSharedF<NT> &sh)
{
	float *th = dyn;
	float2 *cs = reinterpret_cast<float2 *>(dyn);
	float *phi = dyn + 2 * g.V;
	FM::WeightFrags<NI, NT, LaneLoops> wr;
	const LaneLoops ll;
	wr.load(params + (long)(nl - 1) * NP_LAYER);
	for (int i = threadIdx.x; i < 2 * g.V; i += NT)
		th[i] = theta[(long)c * 2 * g.V + i];
	__syncthreads();
	double v[2] = {0.0, 0.0}; // log det, S
	for (int x = threadIdx.x; x < g.V; x += NT)
	{
		const int x0 = x / g.L1, x1 = x - x0 * g.L1;
		const float tp = plaqp(g, th, x0, x1);
		v[1] += 1.0 - cos_any((double)tp);
		phi[x] = x < g.V - 1 ? FM::wrapf(tp) : 0.f;
	}
	__syncthreads(); // the links are read; cs takes their place
	for (int x = threadIdx.x; x < g.V; x += NT)
		sincos_any(phi[x], cs[x].y, cs[x].x);
	for (int layer = nl - 1; layer >= 0; --layer)
	{
		__syncthreads();
		wr.store(sh.lw);
		__syncthreads();
		if (layer > 0)
			wr.load(params + (long)(layer - 1) * NP_LAYER);
		layer_apply<true, NT>(g, ll, phi, cs, layer & 3, sh, v[0]);
	}
	__syncthreads();
	block_sum<2>(v, sh.red);
	if (threadIdx.x == 0)
	{
		out[2 * c + 0] = -v[0] - 2.0 * g.V * LOG_2PI;
		out[2 * c + 1] = v[1];
	}
	if (z_out)
		for (int x = threadIdx.x; x < g.V; x += NT)
			z_out[(long)c * g.V + x] = phi[x];
}

// The kernels run on 256 or 512 threads (by_width()).
template <int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2)))
void k_pc_forward(PCGeo g, int nl, const float *__restrict__ params, uint64_t seed,
                  uint32_t step, float *theta_out, float *phi_layers,
                  float *phi_final, double *out)
{
	extern __shared__ float dyn[];
	__shared__ PCSharedF<NT> sh;
	pc_forward(g, nl, params, seed, step, theta_out, phi_layers, phi_final, out, blockIdx.x, dyn, sh);
}

template <int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2)))
void k_pc_inverse(PCGeo g, int nl, const float *__restrict__ params,
                  const float *__restrict__ theta, float *z_out, double *out)
{
	extern __shared__ float dyn[];
	__shared__ PCSharedF<NT> sh;
	pc_inverse(g, nl, params, theta, z_out, out, blockIdx.x, dyn, sh);
}

// one MH proposal round in one launch: workgroups 0..batch-1 take log q of
// the current configurations, batch..2 batch-1 draw the proposals, so that on
// small lattices (two workgroups' LDS per CU) the two passes share the CUs
template <int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2)))
void k_pc_propose(PCGeo g, int nl, const float *__restrict__ params, int batch,
                  const float *__restrict__ theta, double *state, uint64_t seed,
                  uint32_t step, float *theta_prop, double *prop_out)
{
	extern __shared__ float dyn[];
	__shared__ PCSharedF<NT> sh;
	if ((int)blockIdx.x < batch)
		pc_inverse(g, nl, params, theta, nullptr, state, blockIdx.x, dyn, sh);
	else
		pc_forward(g, nl, params, seed, step, theta_prop, nullptr, nullptr, prop_out, blockIdx.x - batch, dyn, sh);
}

// gradient of the per-configuration loss beta S - log det (S with the last
// plaquette = -sum of the free ones) with respect to every weight:
// partial[c][layer * NP_LAYER + i].  phi_layers / phi_final from k_pc_forward;
// drs: scratch of (V/4) * 8 floats per configuration, the adjoints of every
// active plaquette's ring.
// LDS: cs[V] (of the current layer's input), phi[V], a[V], gact[V/4].
__global__ __launch_bounds__(THREADS) void k_pc_backward(PCGeo g, int nl, const float *__restrict__ params,
                                                         const float *__restrict__ phi_layers,
                                                         const float *__restrict__ phi_final, float beta,
                                                         float *__restrict__ drs, float *__restrict__ partial)
{
	extern __shared__ float dyn[];
	float2 *cs = reinterpret_cast<float2 *>(dyn);
	float *phi = dyn + 2 * g.V;  // input of the current layer
	float *a = dyn + 3 * g.V;    // adjoint w.r.t. the current layer's output
	float *gact = dyn + 4 * g.V; // adjoint w.r.t. the active plaquettes' input
	__shared__ PCSharedB sh;
	const int c = blockIdx.x, w = threadIdx.x >> 6, l = threadIdx.x & 63;
	float *dr = drs + (long)c * (g.V >> 2) * 8;
	float *part = partial + (long)c * nl * NP_LAYER;
	FM::WeightRegsP<NI, THREADS> wr;
	const LaneLoops ll;
	auto row = [](int q, int s) { return LaneLoops::row(q, s); };
	wr.load(params + (long)(nl - 1) * NP_LAYER);
	FM::zero_pad<NI>(sh.lw);
	for (int x = threadIdx.x; x < g.V; x += THREADS)
		phi[x] = phi_final[(long)c * g.V + x];
	double s[1] = {0.0};
	for (int x = threadIdx.x; x < g.V - 1; x += THREADS)
		s[0] += (double)phi[x];
	block_sum<1>(s, sh.red);
	const float sin_last = (float)sin(wrapd(-s[0]));
	for (int x = threadIdx.x; x < g.V; x += THREADS)
		a[x] = x < g.V - 1 ? beta * (sinf(phi[x]) - sin_last) : 0.f;
	for (int layer = nl - 1; layer >= 0; --layer)
	{
		const int m = layer & 3, NA = n_active(g, m), ntile = (NA + 15) / 16;
		__syncthreads();
		for (int x = threadIdx.x; x < g.V; x += THREADS)
		{
			const float p = phi_layers[((long)c * nl + layer) * g.V + x];
			phi[x] = p;
			cs[x] = sincos2(p);
		}
		wr.store(sh.lw);
		__syncthreads();
		if (layer > 0)
			wr.load(params + (long)(layer - 1) * NP_LAYER);
		FM::GradP<NI> gr;
		gr.zero();
		// four tiles a round; a wavefront past the last tile repeats the last
		// row with dL/dy = 0
		for (int t0 = 0; t0 < ntile; t0 += 4)
		{
			const int r = (t0 + w) * 16 + (l & 15); // this lane's row in the MLP
			int x0, x1;
			active_xy(g, m, min(r, NA - 1), x0, x1);
			float x[NI / 4], *y = sh.buf.y[w];
			ll.features(g, cs, x0, x1, x);
			FM::f4 h1[4], h2[4], dx[FM::GradP<NI>::NB];
			const FM::f4 out = FM::mlp_rows<NI, FAST>(sh.lw, x, [&](int k) { return row(ll.q, k); }, h1, h2);
			FM::put_outputs(y, out);
			FM::wave_sync();
			{
				const int rq = (t0 + w) * 16 + (l >> 2); // its quad's row in the map
				const bool live = rq < NA;
				active_xy(g, m, min(rq, NA - 1), x0, x1);
				const int xs = x0 * g.L1 + x1;
				float *yr = y + (l >> 2) * FM::YS;
				const FM::NCPq p = FM::ncpq_params(yr);
				const float da = FM::ncpq_adjoint(p, yr, FM::wrapf(phi[xs] - p.t), a[xs], live);
				if (live && (l & 3) == 0)
					gact[rq] = da;
			}
			FM::wave_sync();
			FM::mlp_rows_backward<NI>(sh.lw, sh.buf, x, row, h1, h2, gr, dx);
			// the adjoints of the lane's loops' angles, then of ring plaquettes
			// 2q and 2q + 1 (that of 2q - 1 goes to the quarter which holds it)
			float e[5];
#pragma unroll
			for (int k = 0; k < 5; ++k)
				e[k] = fmaf(x[2 * k], dx[(2 * k + 1) / 4][(2 * k + 1) & 3], -x[2 * k + 1] * dx[2 * k / 4][(2 * k) & 3]);
			const float from_next = __shfl(e[3] + e[4], (l + 16) & 63, 64);
			if (r < NA)
				*reinterpret_cast<FM::Pair *>(dr + r * 8 + 2 * ll.q) = // (the caller's workspace)
				    FM::Pair{e[0] + e[2] + e[3] + e[4], e[1] + e[2] + e[4] + from_next};
		}
		__syncthreads();
		FM::store_grad<NI>(gr, row, part + (long)layer * NP_LAYER);
		// adjoints w.r.t. the layer's input: the active plaquettes from gact,
		// the frozen ones gain theirs as ring plaquettes of the active ones,
		// which lie one step along x0, x1 or both (class bits that differ)
		const int h = g.L1 >> 1;
		for (int y = threadIdx.x; y < g.V - 1; y += THREADS)
		{
			const int y0 = y / g.L1, y1 = y - y0 * g.L1;
			const int s0 = (y0 ^ m) & 1, s1 = (y1 ^ (m >> 1)) & 1;
			if (!s0 && !s1)
			{
				a[y] = gact[(y0 >> 1) * h + (y1 >> 1)];
				continue;
			}
			float acc = 0.f;
#pragma unroll
			for (int k = 0; k < 8; ++k)
			{
				int d0, d1;
				ring(k, d0, d1);
				if ((d0 != 0) != (s0 != 0) || (d1 != 0) != (s1 != 0))
					continue;
				const int x = sitew(g, y0 - d0, y1 - d1);
				if (x == g.V - 1)
					continue;
				const int x0 = x / g.L1, x1 = x - x0 * g.L1;
				acc += dr[((x0 >> 1) * h + (x1 >> 1)) * 8 + k];
			}
			a[y] += acc;
		}
	}
}

__global__ void k_pc_init(int n, float *p, uint64_t seed)
{
	int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		FM::init_param<NI>(i, p, seed, TAG_PCFI);
}

int pc_setup(mesh_ctx *ctx, const mesh_grid *g, int batch, int layers, PCGeo *pg, const float *params = nullptr)
{
	if (layers < 1 || layers > MAX_LAYERS)
		return mesh_fail(ctx, MESH_E_ARG, "the plaquette coupling flow has 1 to 64 layers");
	if (!g || g->nd != 2 || g->dims[0] % 2 || g->dims[1] % 2 || g->dims[0] < 4 || g->dims[1] < 4)
		return mesh_fail(ctx, MESH_E_SIZE, "the plaquette coupling flow needs a 2-d lattice with even extents >= 4");
	long V = (long)g->dims[0] * g->dims[1];
	if (V > 4096)
		return mesh_fail(ctx, MESH_E_SIZE, "the plaquette coupling flow holds a configuration in LDS: volume <= 4096");
	if (batch < 1)
		return mesh_fail(ctx, MESH_E_ARG, "batch must be >= 1");
	if ((uintptr_t)params % 8)
		return mesh_fail(ctx, MESH_E_ARG, "the flow's parameters must be 8-byte aligned");
	pg->L0 = g->dims[0];
	pg->L1 = g->dims[1];
	pg->V = (int)V;
	const unsigned h = (unsigned)pg->L1 >> 1;
	pg->hm = ((1u << 20) + h - 1) / h;
	return MESH_OK;
}

template <class K> int set_lds(mesh_ctx *ctx, K kernel, size_t bytes)
{
	MESH_HIP(ctx, hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
	return MESH_OK;
}

// kernel(std::integral_constant<int, threads>) for a launch of so many workgroups
template <class F> int by_width(PCGeo const &g, int blocks, F &&kernel)
{
	if (g.V >= WIDE_V && (blocks <= 256 || g.V > PAIR_V))
		return kernel(std::integral_constant<int, 512>{});
	return kernel(std::integral_constant<int, 256>{});
}

template <int NT> int launch_forward(mesh_ctx *ctx, PCGeo const &g, int batch, int layers, const float *params,
                                     uint64_t seed, uint32_t step, float *theta_out, float *phi_layers,
                                     float *phi_final, double *out)
{
	const size_t lds = 4 * (size_t)g.V * sizeof(float);
	if (int rc = set_lds(ctx, k_pc_forward<NT>, lds))
		return rc;
	k_pc_forward<NT><<<batch, NT, lds, ctx->stream>>>(g, layers, params, seed, step, theta_out, phi_layers, phi_final,
	                                                  out);
	MESH_LAUNCHED(ctx);
	return MESH_OK;
}

} // namespace

extern "C" {

int mesh_pcflow_num_params(int layers) { return layers >= 1 && layers <= MAX_LAYERS ? layers * NP_LAYER : 0; }

int mesh_pcflow_init(mesh_ctx *ctx, int layers, float *params, uint64_t seed)
{
	MESH_CHECK_CTX(ctx);
	if (!params || layers < 1 || layers > MAX_LAYERS)
		return mesh_fail(ctx, MESH_E_ARG, "bad pcflow_init arguments");
	const int n = layers * NP_LAYER;
	k_pc_init<<<(n + 255) / 256, 256, 0, ctx->stream>>>(n, params, seed);
	MESH_LAUNCHED(ctx);
	return MESH_OK;
}

int mesh_pcflow_sample(mesh_ctx *ctx, const mesh_grid *g, int batch, int layers, const float *params, uint64_t seed,
                       uint32_t step, float *theta_out, double *out_dev)
{
	MESH_CHECK_CTX(ctx);
	PCGeo pg;
	if (int rc = pc_setup(ctx, g, batch, layers, &pg, params))
		return rc;
	if (!params || !theta_out || !out_dev)
		return mesh_fail(ctx, MESH_E_ARG, "NULL argument to pcflow_sample");
	return by_width(pg, batch, [&](auto nt) {
		return launch_forward<decltype(nt)::value>(ctx, pg, batch, layers, params, seed, step, theta_out, nullptr,
		                                           nullptr, out_dev);
	});
}

int mesh_pcflow_logq(mesh_ctx *ctx, const mesh_grid *g, int batch, int layers, const float *params,
                     const float *theta, float *z_out, double *out_dev)
{
	MESH_CHECK_CTX(ctx);
	PCGeo pg;
	if (int rc = pc_setup(ctx, g, batch, layers, &pg, params))
		return rc;
	if (!params || !theta || !out_dev)
		return mesh_fail(ctx, MESH_E_ARG, "NULL argument to pcflow_logq");
	return by_width(pg, batch, [&](auto nt) -> int {
		constexpr int NT = decltype(nt)::value;
		const size_t lds = 3 * (size_t)pg.V * sizeof(float);
		if (int rc = set_lds(ctx, k_pc_inverse<NT>, lds))
			return rc;
		k_pc_inverse<NT><<<batch, NT, lds, ctx->stream>>>(pg, layers, params, theta, z_out, out_dev);
		MESH_LAUNCHED(ctx);
		return MESH_OK;
	});
}

int mesh_pcflow_propose(mesh_ctx *ctx, const mesh_grid *g, int batch, int layers, const float *params,
                        const float *theta, double *state_dev, uint64_t seed, uint32_t step, float *theta_prop,
                        double *prop_dev)
{
	MESH_CHECK_CTX(ctx);
	PCGeo pg;
	if (int rc = pc_setup(ctx, g, batch, layers, &pg, params))
		return rc;
	if (!params || !theta || !state_dev || !theta_prop || !prop_dev)
		return mesh_fail(ctx, MESH_E_ARG, "NULL argument to pcflow_propose");
	if (theta == theta_prop || state_dev == prop_dev)
		return mesh_fail(ctx, MESH_E_ARG, "pcflow_propose: the proposals and their log q need their own buffers");
	return by_width(pg, 2 * batch, [&](auto nt) -> int {
		constexpr int NT = decltype(nt)::value;
		const size_t lds = 4 * (size_t)pg.V * sizeof(float);
		if (int rc = set_lds(ctx, k_pc_propose<NT>, lds))
			return rc;
		k_pc_propose<NT><<<2 * batch, NT, lds, ctx->stream>>>(pg, layers, params, batch, theta, state_dev, seed, step,
		                                                      theta_prop, prop_dev);
		MESH_LAUNCHED(ctx);
		return MESH_OK;
	});
}

size_t mesh_pcflow_workspace_bytes(const mesh_grid *g, int batch, int layers)
{
	PCGeo pg;
	if (pc_setup(nullptr, g, batch, layers, &pg))
		return 0;
	size_t n = (size_t)batch * layers * pg.V           // plaquettes per layer
	           + (size_t)batch * pg.V                  // final plaquettes
	           + (size_t)batch * (pg.V / 4) * 8        // adjoints of the active plaquettes' rings
	           + (size_t)batch * layers * NP_LAYER;    // per-configuration gradients
	return n * sizeof(float);
}

int mesh_pcflow_gradient(mesh_ctx *ctx, const mesh_grid *g, int batch, int layers, const float *params, uint64_t seed,
                         uint32_t step, double beta, void *workspace, float *grad, double *out_dev)
{
	MESH_CHECK_CTX(ctx);
	PCGeo pg;
	if (int rc = pc_setup(ctx, g, batch, layers, &pg, params))
		return rc;
	if (!params || !workspace || !grad || !out_dev)
		return mesh_fail(ctx, MESH_E_ARG, "NULL argument to pcflow_gradient");
	float *pl = (float *)workspace;
	float *pf = pl + (size_t)batch * layers * pg.V;
	float *drs = pf + (size_t)batch * pg.V;
	float *part = drs + (size_t)batch * (pg.V / 4) * 8;
	if (int rc = by_width(pg, batch, [&](auto nt) {
		    return launch_forward<decltype(nt)::value>(ctx, pg, batch, layers, params, seed, step, nullptr, pl, pf,
		                                               out_dev);
	    }))
		return rc;
	const size_t lds_b = (4 * (size_t)pg.V + pg.V / 4) * sizeof(float);
	if (int rc = set_lds(ctx, k_pc_backward, lds_b))
		return rc;
	k_pc_backward<<<batch, THREADS, lds_b, ctx->stream>>>(pg, layers, params, pl, pf, (float)beta, drs, part);
	MESH_LAUNCHED(ctx);
	const int n = layers * NP_LAYER;
	FM::k_grad_reduce<<<(n + 63) / 64, 256, 0, ctx->stream>>>(n, part, batch, 1.0f / batch, grad);
	MESH_LAUNCHED(ctx);
	return MESH_OK;
}

int mesh_pcflow_adam(mesh_ctx *ctx, int layers, float *params, const float *grad, float *m, float *v, int t,
                     double lr)
{
	MESH_CHECK_CTX(ctx);
	if (!params || !grad || !m || !v || t < 1 || layers < 1 || layers > MAX_LAYERS)
		return mesh_fail(ctx, MESH_E_ARG, "bad pcflow_adam arguments");
	return mesh_launch_adam(ctx, layers * NP_LAYER, params, grad, m, v, t, lr);
}

} // extern "C"
