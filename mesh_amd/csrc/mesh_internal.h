// Internal declarations shared by the translation units of libmesh_hip.so.
#pragma once
#include "../../include/mesh_hip.h"
#include "su3_dev.h"
#include <hip/hip_runtime.h>
#include <string>
#include <vector>

// kernels timed by the optional per-launch event profiler
enum mesh_prof_kind
{
	PROF_FORCE_UPDATE = 0,
	PROF_LINK_UPDATE,
	PROF_DELTA_H,
	PROF_MOMENTA,
	PROF_PLAQ,
	PROF_LANDAU_OR,
	PROF_FORCE_LINK,
	PROF_MOMENTA_LINK,
	PROF_NKINDS
};

struct mesh_prof_rec
{
	int kind;
	hipEvent_t a, b;
};

struct mesh_ctx
{
	int magic;
	int device;
	hipStream_t stream;
	std::string err;
	// reduction scratch: per-block partial sums (device) and the final values
	// (pinned host memory, and its address for the device)
	double *partials = nullptr;
	size_t partials_cap = 0; // doubles
	double *red_host = nullptr;
	double *red_out = nullptr;
	double *aux = nullptr; // small device buffer (integrator step tables)
	size_t aux_cap = 0;    // doubles
	std::vector<double> aux_host; // host copy of what aux holds
	int xcd_remap = 3;     // block order of the stencil kernels (BlockOrder)
	int rb_tile = 4;       // row-blocks per traversal tile of orders 3 and 4
	int force_variant = -1; // -1: the default kernel (variant 0)
	int fuse_md = 1;        // fuse each momentum step with the next link step
	int compact_p = 1;      // fused trajectory: momenta in 9 reals per link
	void *md_spare = nullptr; // third gauge field for the fused trajectory
	size_t md_spare_bytes = 0;
	int u1_general = 0;       // U(1): site-parallel kernels also for small 2-d lattices
	int float_sums = 0;       // FP32 trajectories: Delta H from the reference's FP32 energy sums
	void *u1_ws = nullptr;    // workspace of the site-parallel U(1) kernels
	size_t u1_ws_bytes = 0;
	// device address of the static scratch array of the no-allocation entry
	// point on this context's device (mesh_scratch_setup)
	double *scratch = nullptr;
	// profiler: events around launches, resolved after a stream sync
	int prof_on = 0;
	std::vector<hipEvent_t> prof_pool;
	std::vector<mesh_prof_rec> prof_pending;
	double prof_ms[PROF_NKINDS] = {};
	long long prof_cnt[PROF_NKINDS] = {};
};

// bracket a launch with events when profiling is on (returns a handle or -1)
int mesh_prof_begin(mesh_ctx *ctx, int kind);
void mesh_prof_end(mesh_ctx *ctx, int handle);
// resolve pending records (call after the stream has been synchronised)
void mesh_prof_collect(mesh_ctx *ctx);

constexpr int MESH_CTX_MAGIC = 0x4d455348;
constexpr int RED_MAX_Q = 18;

int mesh_fail(mesh_ctx *ctx, int code, std::string const &msg);
int mesh_hip_fail(mesh_ctx *ctx, hipError_t e, char const *what);
bool mesh_ctx_ok(mesh_ctx *ctx);

#define MESH_CHECK_CTX(ctx)                                                                        \
	do                                                                                             \
	{                                                                                              \
		if (!mesh_ctx_ok(ctx))                                                                     \
			return MESH_E_STATE;                                                                   \
	} while (0)

#define MESH_HIP(ctx, expr)                                                                        \
	do                                                                                             \
	{                                                                                              \
		hipError_t e_ = (expr);                                                                    \
		if (e_ != hipSuccess)                                                                      \
			return mesh_hip_fail(ctx, e_, #expr);                                                  \
	} while (0)

#define MESH_LAUNCHED(ctx)                                                                         \
	do                                                                                             \
	{                                                                                              \
		hipError_t e_ = hipGetLastError();                                                         \
		if (e_ != hipSuccess)                                                                      \
			return mesh_hip_fail(ctx, e_, "kernel launch");                                        \
	} while (0)

// validates a grid; fills the device geometry descriptor
int mesh_make_geo(mesh_ctx *ctx, const mesh_grid *g, mesh_dev::Geo *geo);
int mesh_check_prec(mesh_ctx *ctx, int prec);
// ensures ctx->partials holds at least n doubles
int mesh_reserve_partials(mesh_ctx *ctx, size_t n);
// copies n host doubles into ctx->aux (grown as needed), on the ctx stream
int mesh_stage_doubles(mesh_ctx *ctx, const double *host, size_t n);
// one Adam step (Kingma & Ba) over n parameters, t >= 1
int mesh_launch_adam(mesh_ctx *ctx, int n, float *params, const float *grad, float *m, float *v, int t, double lr);
// sums nq quantities of nb partials each into host out[nq] (synchronises)
int mesh_finish_reduction(mesh_ctx *ctx, int nb, int nq, double *out);
// the same fixed-order sum of nb partials (nq = 1) into device out_dev, on the
// context's stream, without copying or synchronising
int mesh_reduce_to_device(mesh_ctx *ctx, const double *partials, int nb, double *out_dev);
// resolves the device address of the no-allocation scratch array for the
// context's device (once per device; the device must be current)
int mesh_scratch_setup(mesh_ctx *ctx);

// launch shape of the site-blocked kernels: nb logical blocks; with XCD
// remapping the grid is padded to a multiple of 8
inline int mesh_grid_blocks(mesh_ctx *ctx, int nb) { return ctx->xcd_remap ? ((nb + 7) / 8) * 8 : nb; }
// block-order argument of the stencil kernels (block_order): order | (tile << 4)
inline int mesh_order(mesh_ctx *ctx) { return ctx->xcd_remap | (ctx->rb_tile << 4); }

namespace mesh_dev {

// Workgroups are dispatched round-robin over the 8 XCDs of an MI355X.
// Block order of the stencil kernels (sbk consecutive sites per workgroup,
// i.e. one "row-block" rb of the x2/x3 plane), argument order | (T << 4):
//   0: linear;  1: XCD-contiguous linear;
//   2: cache order for 4-d lattices with sbk | L2*L3 -- each XCD walks its own
//      range of row-blocks and, within it, x0 fastest then x1, so the
//      x0-neighbours of a workgroup were staged by the previous one and the
//      x1-neighbours L0 workgroups earlier, all in the same L2;
//   3: slab order for 4-d lattices with 8 | L0 -- XCD k owns the slab x0 in
//      [k L0/8, (k+1) L0/8) and walks it x0 fastest, then a tile of T
//      row-blocks, then x1, then the next tile, so the x1- and rb-neighbours of
//      a workgroup are at most (L0/8) T workgroups back and only the two x0
//      faces of the slab come from another XCD; T: tile_of(the argument's);
//   4: as 3 with XCD k owning x0 in a quarter (k % 4) and x1 in a half (k / 4)
//      of the lattice (4 | L0, 2 | L1); also order 3's fallback where 8 does
//      not divide L0.
// Where a plane is no whole number of blocks, or the extents allow neither,
// orders 3 and 4 give XCD k the k-th eighth of the blocks in memory order, about
// L0/8 slices of x0, and walk it as the kernel asks (Walk): in memory order, with
// the slices side by side (slice fastest, then the position in the slice, so the
// x0-neighbours of a workgroup are the launches before and after it, to within a
// block), or, where planes are whole blocks, in order 2.
// Returns the memory-order block index (-1: padding workgroup).  The order
// only permutes workgroups; every site's arithmetic is unchanged.  GEO: any
// geometry with nd and L[4] (the SU(3) and SU(2) ones).
// the row-blocks of a tile of orders 3 and 4: the divisor of nb2 (row-blocks of
// a plane) nearest below or just above the one asked for (fused step FP64 40^4, whose
// planes of 25 blocks take 5: 1740 us in memory order, 1485)
inline int tile_of(int nb2, int t)
{
	if (nb2 % t == 0)
		return t;
	if (nb2 % (t + 1) == 0)
		return t + 1;
	while (nb2 % t)
		--t;
	return t;
}

// one launch's order: what does not depend on the workgroup is worked out on the
// host, and a workgroup divides by multiplication (FastDiv); done in the kernel it
// was a chain of scalar divisions before the first load of every workgroup
// (fused step with this and the coordinates' divisions so: 8^4 FP64 13.2 -> 12.7
// us, FP32 11.6 -> 11.2, 12^4 21.3 -> 20.9 and 15.7 -> 15.2; 32^4 FP64 560 -> 563,
// FP32 341 -> 338)
struct BlockOrder
{
	enum Kind
	{
		LINEAR, // memory order
		SLAB,   // orders 3 and 4 on planes of whole blocks
		CHUNK,  // an eighth of memory order an XCD, w slices side by side if S > 0
		CACHE   // order 2
	};
	int kind = LINEAR, nb = 0, nb2 = 1, L1 = 1;
	int halves = 0, X = 1, X1 = 1, T = 1; // SLAB: x0 positions and x1 positions of an XCD, tile
	int chunk = 0, S = 0;                 // CHUNK
	FastDiv by_a, by_b, by_c;             // SLAB: X, T, X1; CHUNK: S; CACHE: L0, L1

	// the memory-order block of workgroup b (-1: padding)
	__host__ __device__ __forceinline__ int at(int b) const
	{
		if (kind == LINEAR)
			return b < nb ? b : -1;
		const int k = b & 7, j = b >> 3;
		if (kind == SLAB)
		{
			if (j >= nb >> 3)
				return -1;
			int t = by_a(j);
			const int x0 = (halves ? k & 3 : k) * X + (j - t * X);
			const int u = by_b(t), v = by_c(u);
			const int rb = (t - u * T) + v * T, x1 = (halves ? (k >> 2) * X1 : 0) + (u - v * X1);
			return (x0 * L1 + x1) * nb2 + rb;
		}
		const int first = k * chunk, o = first + j;
		if (o >= nb)
			return -1;
		if (kind == CACHE)
		{
			const int t = by_a(o), rb = by_b(t);
			return ((o - t * X) * L1 + (t - rb * L1)) * nb2 + rb;
		}
		if (S == 0)
			return o;
		// this XCD's C blocks as slices of S: R positions have w + 1 of them,
		// the others w
		const int C = nb - first < chunk ? nb - first : chunk, w = by_a(C);
		if (w == 0)
			return o;
		const int R = C - w * S;
		if (j < R * (w + 1))
			return first + (j % (w + 1)) * S + j / (w + 1);
		const int i = j - R * (w + 1);
		return first + (i % w) * S + R + i / w;
	}
};

// how orders 3 and 4 walk a lattice that allows neither: slices side by side if a
// slice has at least `side` blocks and an XCD `slices` of them; else order 2 if
// `cache` and planes are whole blocks, else memory order
struct Walk
{
	int side = 129, slices = 1;
	bool cache = false;
};
// (measured on lattices with and without whole planes, a slice of 60 to 1,700
// blocks, an XCD of less than one to six slices)
//
// SU(3) fused step.  FP64: side by side from 300 blocks a slice (28^4, 343 blocks:
// 396 -> 383 us; 36^4, 729: 1121 -> 1059; 44^4 2558 -> 2355; 26^4, 274: 299 -> 304;
// 30x24^3, 216: 245 -> 250); below that, or with fewer than two slices an XCD, order 2
// if a block holds two rows or more (18x16^3 46.6 -> 44.0 us, 18x8x32x32 89.2 -> 84.4,
// 30x32x32x16 285 -> 273, 6x32^3 114.8 -> 111.4; 22x16x16x64, whose blocks are single
// rows, 208 -> 216 us, and 18x24^3, whose rows cross the blocks, 147 -> 153).  FP32,
// with four workgroups a CU and half the bytes, has a slice's neighbours in its L2 for
// longer: side by side from 600 blocks and four slices (36^4 657 -> 633 us, 38^4 976
// -> 921; 34^4, 614, even; 28^4, 343: 223 -> 226; 18x36^3, two slices: 297 -> 309),
// order 2 nowhere (18x32^3 197 -> 200 us, 6x32^3 67.5 -> 71.1).
template <class GEO> inline Walk fused_walk(GEO const &g, bool f64)
{
	if (!f64)
		return {601, 4, false};
	return {301, 2, g.L[3] <= 32 && 64 % g.L[3] == 0};
}
// SU(3) Delta H (blocks of 128 sites).  FP64 reads two fields and leaves its slices
// in memory order (side by side 36^4 974 -> 1038 us, 38^4 1288 -> 1345); order 2 with
// fewer than three slices an XCD (6x32^3 127 -> 120 us, 18x32x32x16 181 -> 173;
// 30x32^3 561 -> 597).  FP32 walks them side by side (36^4 541 -> 513 us, 44^4 1177
// -> 1119, 30x32^3 311 -> 290).
template <class GEO> inline Walk delta_h_walk(GEO const &g, bool f64)
{
	if (!f64)
		return {};
	return {1 << 30, 1, g.L[0] < 24 && g.L[3] <= 32 && 64 % g.L[3] == 0};
}

template <class GEO> inline BlockOrder block_order(GEO const &g, int nb, int sbk, int arg, Walk walk = {})
{
	BlockOrder o;
	const int order = arg & 15;
	o.nb = nb;
	if (order == 0)
		return o;
	const bool planes = g.nd == 4 && (g.L[2] * g.L[3]) % sbk == 0;
	o.nb2 = planes ? (g.L[2] * g.L[3]) / sbk : 1;
	o.L1 = g.L[1];
	const bool slab = order == 3 && planes && (g.L[0] & 7) == 0;
	if (slab || ((order == 4 || order == 3) && planes && (g.L[0] & 3) == 0 && (g.L[1] & 1) == 0))
	{
		// order 4: XCD k owns x0 in a quarter (k % 4) and x1 in a half (k / 4)
		// of the lattice, walked as in order 3
		o.kind = BlockOrder::SLAB;
		o.halves = !slab;
		o.X = g.L[0] >> (slab ? 3 : 2);
		o.X1 = slab ? g.L[1] : g.L[1] >> 1;
		o.T = tile_of(o.nb2, (arg >> 4) > 0 ? arg >> 4 : 1);
		o.by_a = FastDiv(o.X), o.by_b = FastDiv(o.T), o.by_c = FastDiv(o.X1);
		return o;
	}
	o.chunk = (nb + 7) >> 3;
	o.kind = BlockOrder::CHUNK;
	const int slice = g.nd == 4 ? nb / g.L[0] : 0;
	if (order >= 3 && slice >= walk.side && o.chunk >= walk.slices * slice)
	{
		o.S = slice;
		o.by_a = FastDiv(o.S);
	}
	else if (planes && (order == 2 || (order >= 3 && walk.cache)))
	{
		o.kind = BlockOrder::CACHE;
		o.X = g.L[0];
		o.by_a = FastDiv(g.L[0]), o.by_b = FastDiv(g.L[1]);
	}
	return o;
}

// deterministic block sum of NQ doubles; thread 0 writes partials[q*nb + lb]
template <int NQ>
__device__ __forceinline__ void block_sum_store(double (&v)[NQ], double *partials, int nb, int lb)
{
	__shared__ double red[NQ][16];
	int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
	for (int q = 0; q < NQ; ++q)
	{
		double s = v[q];
#pragma unroll
		for (int o = 32; o >= 1; o >>= 1)
			s += __shfl_xor(s, o, 64);
		if (lane == 0)
			red[q][w] = s;
	}
	__syncthreads();
	if (threadIdx.x == 0)
	{
		int nw = (blockDim.x + 63) >> 6;
#pragma unroll
		for (int q = 0; q < NQ; ++q)
		{
			double s = red[q][0];
			for (int i = 1; i < nw; ++i)
				s += red[q][i];
			partials[(long)q * nb + lb] = s;
		}
	}
}

} // namespace mesh_dev
