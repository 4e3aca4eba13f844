// Differentiable FP64 PIC run on gfx950: reverse-mode gradients of the
// time-integrated field energy L = sum_it W(it), W = -(e0/2) sum_g rho_g phi_g,
// with respect to every particle's initial position and velocity.
//
// The forward is the reference loop (sim_step, src/sim.c:482-581, with the
// iteration-0 back half-step of src/mover.c:204-214) on particles that keep
// their index (no tile sorting): per iteration
//   rho = Dep(r)  (interpolate_p2f_rho)      phi = S rho  (MFT_solve)
//   E = D phi     (field_E_compute)          E_p = Gat(E, r)  (interpolate_f2p_E)
//   u' = M (u + h E_p) + h E_p  (Boris, B = (0,0,Bz))   r' = wrap(r + dt' u')
// with the production kernels' arithmetic (picmath.h, the same FFT and E
// stencil kernels).  The reverse sweep applies the transposed maps, given
// the adjoints (lr', lu') of (r', u'):
//   mu = lu' + dt' lr'                 (move; the wrap has derivative 1)
//   lu = M^T mu,  lE_p = h (M^T mu + mu)          (Boris, linear in u and E)
//   lE = Dep(lE_p)                     (gather^T = deposit with CIC weights)
//   psi = D^T lE - e0 rho              (stencil^T; -e0 rho = dW/d(S rho))
//   lrho = S psi                       (S is symmetric: real, even G)
//   lr = lr' + grad Gat(E)(r) . lE_p + c grad Gat(lrho)(r),  c = -q/e0
// (the last two are derivatives of the CIC interpolant with respect to the
// particle position).  The forward keeps every iteration's rho, E and
// positions when they fit fixed budgets, and the reverse reads them.  Otherwise
// states are checkpointed every K iterations and the reverse recomputes each
// segment's positions from its checkpoint (and, without the field history,
// their rho and E).  No counterpart
// in the reference, which has no gradients.
#include "dev.h"
#include "picmath.h"

#include <cmath>
#include <stdlib.h>
#include <string.h>

struct AdjSpecies {
	double h[CPIC_MAX_SPECIES];   // 0.5 dt' q / m
	double tz[CPIC_MAX_SPECIES];  // Bz h
	double sz[CPIC_MAX_SPECIES];  // 2 tz / (1 + tz^2)
	double c[CPIC_MAX_SPECIES];   // -q / e0
};

struct cpic_adj {
	cpic_dev *d;              // grid, FFT tables and stream (a batch of one, no particles)
	Geo g;
	int64_t n;
	int ns;
	AdjSpecies k[2];          // [0]: iteration 0 (dt' = -dt/2), [1]: later iterations
	uint8_t *sp;              // species of each particle, in sorted order
	uint8_t *sp0;             // the same in the caller's order
	int64_t *perm;            // sorted position i holds the caller's particle perm[i]
	double *x, *y, *ux, *uy;  // state
	double *rho[2], *phi, *psi, *lrho;
	double2 *E, *lE;          // lE: two buffers of nodes values (reverse iterations alternate)
	double *lx, *ly, *lux, *luy;
	double *ck;               // checkpoints, 4n doubles each
	int64_t ckcap;
	double *seg;              // positions of one segment's iterations after its first, 2n doubles each
	int64_t segcap;
	double *segf;             // rho and E of one segment's iterations, 3 nodes doubles each
	int64_t segfcap;
	double *hist;             // W per iteration
	int64_t histcap;
	// field history of the last forward (when it fits ADJ_FIELD_HISTORY_MAX
	// and is not switched off): rho of iterations 0..T and E of 0..T-1,
	// which the reverse sweep reads instead of recomputing them
	double *frho, *fE;
	int64_t frhocap, fEcap;   // doubles
	int fhist;                // the last forward kept it
	// position history of the last forward (with the field history, when it
	// fits ADJ_POS_HISTORY_MAX and is not switched off): x, then y of
	// iterations 0..T-1, which leaves the reverse sweep nothing to recompute
	double *ph;
	int64_t phcap;
	int phist, phist_off;
	int fhist_off;            // cpic_adj_set_field_history(a, 0)
	double *wk;               // recompute state of the reverse sweep, and x, y, ux, uy in
	                          // the caller's order on their way in and out: 4n doubles
	hipEvent_t ev[4];         // device work of the last forward [0,1] and backward [2,3]
	int evok;                 // events created
	int evrec;                // bit 0: forward pair recorded, bit 1: backward pair
	int *derr;
	int64_t nsteps;
	int K;
	int have;                 // a forward has run
};

static __device__ __forceinline__ void cic_nodes(const Geo &g, double x, double y, int &i00,
		int &i01, int &i10, int &i11, double &rx, double &ry)
{
	int ix, iy;
	cell64(g, x, y, ix, iy, rx, ry);
	int i1x = ix + 1 == g.nx ? 0 : ix + 1;
	int i1y = iy + 1 == g.ny ? 0 : iy + 1;
	i00 = iy * g.nx + ix;
	i01 = i1y * g.nx + ix;
	i10 = iy * g.nx + i1x;
	i11 = i1y * g.nx + i1x;
}

// Deposits.  The particles are kept sorted by their initial cell (cells taken
// round-robin within each block's chunk), so the ADJ_PPT*CPIC_BLOCK
// consecutive particles of a block lie in a small patch of cells: each block
// accumulates its deposit in LDS over the bounding box of its cells and
// flushes the non-zero nodes with one global atomic each.
// A block whose box is too large or wraps around the grid deposits with
// global atomics directly.
// 4 particles per thread and 1,024 per block: at 8 the kernels hold 100+
// VGPRs (4 waves per SIMD) and the 256^2 adjoint workload runs 10 % slower
#ifndef ADJ_PPT
#define ADJ_PPT 4
#endif
#define ADJ_CHUNK (ADJ_PPT * CPIC_BLOCK)
// Up to ADJ_FEW particles, one workgroup per CU at ADJ_PPT, the depositing
// kernels take one particle per thread instead: a launch is then one
// workgroup's latency, which is shorter with fewer particles in sequence
// (10,240 particles at 64^2: push 11.6 -> 5.8 us, reverse 9.6 -> 7.3 us).
#define ADJ_FEW ((int64_t) 256 * ADJ_CHUNK)
// Particles per thread of the reverse sweep's recompute push, which only
// moves particles (no deposit, no LDS box): at 256^2 (4,194,304 particles)
// 4 per thread make ~2.3 rounds of workgroups, the last a third full;
// smaller blocks of work keep the chip busier to the end
#ifndef MOVE_PPT
#define MOVE_PPT 2
#endif
// 20 KB of double: seven depositing blocks per CU (their 72 VGPRs allow
// seven; a 24 KB box held them to six: forward 15.8 -> 15.7 ms at 256^2);
// the boxes there hold at most ~125 nodes
#ifndef ADJ_BOX_NODES
#define ADJ_BOX_NODES 2560
#endif

// LDS accumulation box of a block: nodes [x0, x0 + w) x [y0, y0 + h) in
// coordinates relative to a reference cell (rx, ry), wrapped into
// [-n/2, n/2).  A block's particles then form one compact box also where
// they straddle the periodic boundary: a chunk of the cell-sorted order
// that ends one grid row and begins the next, or particles that crossed
// x = 0.  (With absolute coordinates such a box spans the whole row, and
// the block fell back to global atomics on a few rows of nodes, which
// serialise: 6-9 % of the blocks at 256^2.)
struct Box {
	int x0, y0, w, h;
	int rx, ry;
	bool lds;
};

// grid sides are powers of two
static __device__ __forceinline__ int rel_wrap(int i, int ref, int n)
{
	int r = (i - ref) & (n - 1);
	return r >= n / 2 ? r - n : r;
}

// Bounding box (plus the CIC +1 node) of the block's cells; ix[u] < 0 marks
// no particle.  Thread 0's first particle (the block's first, which always
// exists) is the reference cell.  s6: six ints of LDS.
template <int U>
static __device__ Box block_box(const Geo &g, const int *ix, const int *iy, int *s6, int cap)
{
	if(threadIdx.x == 0)
	{
		s6[0] = 0x7fffffff;
		s6[1] = -0x7fffffff;
		s6[2] = 0x7fffffff;
		s6[3] = -0x7fffffff;
		s6[4] = ix[0];
		s6[5] = iy[0];
	}
	__syncthreads();
	const int rx = s6[4], ry = s6[5];
	int lox = 0x7fffffff, hix = -0x7fffffff, loy = 0x7fffffff, hiy = -0x7fffffff;
#pragma unroll
	for(int u = 0; u < U; u++)
		if(ix[u] >= 0)
		{
			int ax = rel_wrap(ix[u], rx, g.nx), ay = rel_wrap(iy[u], ry, g.ny);
			lox = min(lox, ax);
			hix = max(hix, ax);
			loy = min(loy, ay);
			hiy = max(hiy, ay);
		}
	// wavefront reduction first: four LDS atomics per wavefront
	for(int off = 32; off > 0; off >>= 1)
	{
		lox = min(lox, __shfl_xor(lox, off));
		hix = max(hix, __shfl_xor(hix, off));
		loy = min(loy, __shfl_xor(loy, off));
		hiy = max(hiy, __shfl_xor(hiy, off));
	}
	if((threadIdx.x & 63) == 0 && hix >= lox)
	{
		atomicMin(&s6[0], lox);
		atomicMax(&s6[1], hix);
		atomicMin(&s6[2], loy);
		atomicMax(&s6[3], hiy);
	}
	__syncthreads();
	Box b;
	b.rx = rx;
	b.ry = ry;
	b.x0 = s6[0];
	b.y0 = s6[2];
	b.w = s6[1] - s6[0] + 2;
	b.h = s6[3] - s6[2] + 2;
	b.lds = s6[1] - s6[0] <= g.nx / 2 && s6[3] - s6[2] <= g.ny / 2 && b.w * b.h <= cap;
	__syncthreads();
	return b;
}

static __device__ __forceinline__ void cell_of(const Geo &g, double x, double y, int &ix, int &iy,
		double &rx, double &ry)
{
	cell64(g, x, y, ix, iy, rx, ry);
}

// box node (dx, dy in {0,1} from cell (ix, iy))
static __device__ __forceinline__ int box_node(const Geo &g, const Box &b, int ix, int iy,
		int dx, int dy)
{
	return (rel_wrap(iy, b.ry, g.ny) - b.y0 + dy) * b.w + (rel_wrap(ix, b.rx, g.nx) - b.x0 + dx);
}

static __device__ __forceinline__ int64_t wrap_node(const Geo &g, int x, int y)
{
	x = x >= g.nx ? x - g.nx : x;
	y = y >= g.ny ? y - g.ny : y;
	return (int64_t) y * g.nx + x;
}

// Adds c * (CIC weights of (rx, ry)) at the 4 nodes of cell (ix, iy) into
// the LDS box or, without one, into the global grid (order of
// src/interpolate.c:259-262).
static __device__ __forceinline__ void dep1(const Geo &g, const Box &b, double *sacc,
		double *__restrict__ rho, int ix, int iy, double rx, double ry, double c)
{
	double dxw = 1.0 - rx, dyw = 1.0 - ry;
	double v00 = (dxw * dyw) * c, v01 = (dxw * ry) * c, v10 = (rx * dyw) * c, v11 = (rx * ry) * c;
	if(b.lds)
	{
		LDS_AS double *l = (LDS_AS double *) sacc;
		lds_add(&l[box_node(g, b, ix, iy, 0, 0)], v00);
		lds_add(&l[box_node(g, b, ix, iy, 0, 1)], v01);
		lds_add(&l[box_node(g, b, ix, iy, 1, 0)], v10);
		lds_add(&l[box_node(g, b, ix, iy, 1, 1)], v11);
	}
	else
	{
		GLB_AS double *m = gptr<double>(rho);
		glb_add(&m[wrap_node(g, ix, iy)], v00);
		glb_add(&m[wrap_node(g, ix, iy + 1)], v01);
		glb_add(&m[wrap_node(g, ix + 1, iy)], v10);
		glb_add(&m[wrap_node(g, ix + 1, iy + 1)], v11);
	}
}

static __device__ void box_zero(const Box &b, double *sacc, int ncomp)
{
	if(b.lds)
		for(int i = threadIdx.x; i < b.w * b.h * ncomp; i += blockDim.x)
			sacc[i] = 0.0;
	__syncthreads();
}

// flushes component k of an LDS box holding ncomp interleaved components
static __device__ void box_flush(const Geo &g, const Box &b, const double *sacc, int ncomp,
		double *__restrict__ out, int out_stride)
{
	__syncthreads();
	if(!b.lds)
		return;
	for(int i = threadIdx.x; i < b.w * b.h; i += blockDim.x)
	{
		int ly = i / b.w, lx = i - ly * b.w;
		int gx = (b.rx + b.x0 + lx) & (g.nx - 1), gy = (b.ry + b.y0 + ly) & (g.ny - 1);
		int64_t gnode = (int64_t) gy * g.nx + gx;
		for(int k = 0; k < ncomp; k++)
		{
			double v = ((const LDS_AS double *) sacc)[i * ncomp + k];
			if(v != 0.0)
				glb_add(&gptr<double>(out)[gnode * out_stride + k], v);
		}
	}
}

// rho += Dep(r) for the particles of the block
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_deposit(Geo g, AdjSpecies k, int64_t n, const uint8_t *__restrict__ sp,
		const double *__restrict__ x, const double *__restrict__ y, double *__restrict__ rho)
{
	__shared__ double sacc[ADJ_BOX_NODES];
	__shared__ int s6[6];
	int64_t p0 = (int64_t) blockIdx.x * ADJ_CHUNK;
	int ix[ADJ_PPT], iy[ADJ_PPT];
	double rx[ADJ_PPT], ry[ADJ_PPT];
#pragma unroll
	for(int u = 0; u < ADJ_PPT; u++)
	{
		int64_t i = p0 + u * CPIC_BLOCK + threadIdx.x;
		ix[u] = -1;
		if(i < n)
		{
			cell_of(g, x[i], y[i], ix[u], iy[u], rx[u], ry[u]);
		}
	}
	Box b = block_box<ADJ_PPT>(g, ix, iy, s6, ADJ_BOX_NODES);
	box_zero(b, sacc, 1);
#pragma unroll
	for(int u = 0; u < ADJ_PPT; u++)
	{
		int64_t i = p0 + u * CPIC_BLOCK + threadIdx.x;
		if(ix[u] >= 0)
			dep1(g, b, sacc, rho, ix[u], iy[u], rx[u], ry[u], k.c[sp[i]]);
	}
	box_flush(g, b, sacc, 1, rho, 1);
}

// gather + Boris + move + wrap, then (DEP) deposit at the new position into
// rho_next; positions are read from (x, y) and written to (xo, yo), which may
// be the same arrays.  PPT particles per thread: ADJ_PPT with the deposit
// (its LDS box spans one sort chunk), MOVE_PPT without
template <bool DEP, int PPT>
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_push(Geo g, AdjSpecies k, int set_r, double dtp, int64_t n,
		const uint8_t *__restrict__ sp, const double *x, const double *y, double *xo,
		double *yo, double *__restrict__ ux, double *__restrict__ uy,
		const double2 *__restrict__ E, double *__restrict__ rho_next, int *derr)
{
	__shared__ double sacc[ADJ_BOX_NODES];
	__shared__ int s6[6];
	bool bad = false, nan_ = false;
	int64_t p0 = (int64_t) blockIdx.x * (PPT * CPIC_BLOCK);
	int ix[PPT], iy[PPT];
	double rx[PPT], ry[PPT];
	// all of the thread's loads first, unconditional: behind a bounds check, or
	// behind the stores of the particle before (which the compiler cannot tell
	// from the positions), each particle's were waited for in turn
	double lpx[PPT], lpy[PPT], lux[PPT], luy[PPT];
	int ls[PPT];
#pragma unroll
	for(int u = 0; u < PPT; u++)
	{
		const int64_t i = min(p0 + u * CPIC_BLOCK + (int) threadIdx.x, n - 1);
		lpx[u] = x[i];
		lpy[u] = y[i];
		lux[u] = ux[i];
		luy[u] = uy[i];
		ls[u] = sp[i];
	}
#pragma unroll
	for(int u = 0; u < PPT; u++)
	{
		int64_t i = p0 + u * CPIC_BLOCK + threadIdx.x;
		ix[u] = -1;
		if(i >= n)
			continue;
		const int s = ls[u];
		int jx, jy;
		double qx, qy;
		double px = lpx[u], py = lpy[u];
		cell_of(g, px, py, jx, jy, qx, qy);
		int j1x = jx + 1 == g.nx ? 0 : jx + 1;
		int j1y = jy + 1 == g.ny ? 0 : jy + 1;
		double dxw = 1.0 - qx, dyw = 1.0 - qy;
		double w00 = dxw * dyw, w01 = dxw * qy, w10 = qx * dyw, w11 = qx * qy;
		double2 e00 = E[(int64_t) jy * g.nx + jx], e01 = E[(int64_t) j1y * g.nx + jx];
		double2 e10 = E[(int64_t) jy * g.nx + j1x], e11 = E[(int64_t) j1y * g.nx + j1x];
		double ex = w00 * e00.x;
		ex = fma(w01, e01.x, ex);
		ex = fma(w10, e10.x, ex);
		ex = fma(w11, e11.x, ex);
		double ey = w00 * e00.y;
		ey = fma(w01, e01.y, ey);
		ey = fma(w10, e10.y, ey);
		ey = fma(w11, e11.y, ey);
		double uu = lux[u], vv = luy[u];
		boris_bz<double>(k.h[s], k.tz[s], k.sz[s], ex, ey, uu, vv);
		if(fabs(uu) > g.umax_x || fabs(vv) > g.umax_y)
			bad = true;
		if(set_r)
		{
			px = wrap64(fma(uu, dtp, px), g.L0);
			py = wrap64(fma(vv, dtp, py), g.L1);
		}
		if(!(isfinite(px) && isfinite(py) && isfinite(uu) && isfinite(vv)))
		{
			nan_ = true;
			px = py = 0.0;
		}
		xo[i] = px;
		yo[i] = py;
		ux[i] = uu;
		uy[i] = vv;
		cell_of(g, px, py, ix[u], iy[u], rx[u], ry[u]);
	}
	if(bad)
		atomicOr(derr, CPIC_DERR_UMAX);
	if(nan_)
		atomicOr(derr, CPIC_DERR_NAN);
	if(!DEP)
		return;
	Box b = block_box<PPT>(g, ix, iy, s6, ADJ_BOX_NODES);
	box_zero(b, sacc, 1);
#pragma unroll
	for(int u = 0; u < PPT; u++)
		if(ix[u] >= 0)
			dep1(g, b, sacc, rho_next, ix[u], iy[u], rx[u], ry[u], k.c[ls[u]]);
	box_flush(g, b, sacc, 1, rho_next, 1);
}

// (ax, ay) += c grad Gat(lrho)(x, y): the derivative of the CIC interpolant
// of lrho at a particle's position, the last term of lr
static __device__ __forceinline__ void rev_b_term(const Geo &g, double c, double x, double y,
		const double *__restrict__ lrho, double &ax, double &ay)
{
	int i00, i01, i10, i11;
	double rx, ry;
	cic_nodes(g, x, y, i00, i01, i10, i11, rx, ry);
	double l00 = lrho[i00], l01 = lrho[i01], l10 = lrho[i10], l11 = lrho[i11];
	double dxw = 1.0 - rx, dyw = 1.0 - ry;
	ax += c * (g.idx * (dyw * (l10 - l00) + ry * (l11 - l01)));
	ay += c * (g.idy * (dxw * (l01 - l00) + rx * (l11 - l10)));
}

// Reverse of move + Boris + gather for one iteration; accumulates the
// gather-weight derivative into (lx, ly) and deposits lE_p into lE.  With
// PEND, first adds the lrho term of the iteration after it (rev_b_term at
// that iteration's positions (bx, by) with its lrho), so that (lx, ly) are
// read and written once for both.
// REV_PPT particles per thread: the kernel keeps six values per particle
// across the box barriers, and 8 per thread would hold it to 3 waves per
// SIMD; 2 rather than 4 make twice the workgroups, so that at 256^2 the last
// of their rounds idles less of the chip (reverse sweep 34.4 -> 33.5 ms).
// A fraction of a round-robin chunk still spans its cells.
#ifndef REV_PPT
#define REV_PPT 2
#endif
#define REV_CHUNK (REV_PPT * CPIC_BLOCK)
static_assert(ADJ_CHUNK % REV_CHUNK == 0, "reverse blocks split the sort's chunks");
#define REV_BOX_NODES 1536          // 2 components: 24 KB
// Device memory the field history of a forward may take (rho and E of every
// iteration, 24 B per node and iteration: 315 MB for 200 iterations at
// 256^2); beyond it the reverse sweep recomputes each segment's fields
#define ADJ_FIELD_HISTORY_MAX ((int64_t) 8 << 30)
// Device memory the position history may take (16 B per particle and
// iteration: 13.4 GB for 200 iterations of 4,194,304 particles), and at most
// half of what is free.  The forward's push writes each iteration's positions
// there instead of in place.  It moves as many bytes, but 67 MB of them per
// iteration to memory that the memory-side cache does not hold yet: push 53.5
// -> 59.8 us, forward 15.9 -> 16.7 ms for 4,194,304 particles and 200 steps.  The
// reverse sweep reads the positions instead of pushing every segment's
// particles again from a checkpoint: 32.0 -> 21.2 ms.  The checkpoints (134 MB
// of copies each there) are not taken.
#define ADJ_POS_HISTORY_MAX ((int64_t) 32 << 30)
template <bool PEND, int PPT>
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_rev_a(Geo g, AdjSpecies k, int set_r, double dtp, int64_t n,
		const uint8_t *__restrict__ sp, const double *__restrict__ x,
		const double *__restrict__ y, const double2 *__restrict__ E, double *__restrict__ lx,
		double *__restrict__ ly, double *__restrict__ lux, double *__restrict__ luy,
		double2 *__restrict__ lE, const double *__restrict__ bx, const double *__restrict__ by,
		const double *__restrict__ lrho)
{
	__shared__ double sacc[2 * REV_BOX_NODES];
	__shared__ int s6[6];
	int64_t p0 = (int64_t) blockIdx.x * (PPT * CPIC_BLOCK);
	int ix[PPT], iy[PPT];
	double rx[PPT], ry[PPT], lex[PPT], ley[PPT];
#pragma unroll
	for(int u = 0; u < PPT; u++)
	{
		int64_t i = p0 + u * CPIC_BLOCK + threadIdx.x;
		ix[u] = -1;
		if(i >= n)
			continue;
		int s = sp[i];
		double mx = lux[i], my = luy[i];
		double ax = lx[i], ay = ly[i];
		if(PEND)
			rev_b_term(g, k.c[s], bx[i], by[i], lrho, ax, ay);
		if(set_r)
		{
			mx = fma(dtp, ax, mx);
			my = fma(dtp, ay, my);
		}
		double h = k.h[s], tz = k.tz[s], sz = k.sz[s];
		double a_ = 1.0 - tz * sz, b_ = sz;
		double nux = a_ * mx - b_ * my;      // M^T mu
		double nuy = b_ * mx + a_ * my;
		lex[u] = h * (nux + mx);
		ley[u] = h * (nuy + my);
		lux[i] = nux;
		luy[i] = nuy;

		cell_of(g, x[i], y[i], ix[u], iy[u], rx[u], ry[u]);
		int i1x = ix[u] + 1 == g.nx ? 0 : ix[u] + 1;
		int i1y = iy[u] + 1 == g.ny ? 0 : iy[u] + 1;
		double dxw = 1.0 - rx[u], dyw = 1.0 - ry[u];
		double2 e00 = E[(int64_t) iy[u] * g.nx + ix[u]], e01 = E[(int64_t) i1y * g.nx + ix[u]];
		double2 e10 = E[(int64_t) iy[u] * g.nx + i1x], e11 = E[(int64_t) i1y * g.nx + i1x];
		// d/dx and d/dy of the CIC interpolants of Ex and Ey
		double gxx = g.idx * (dyw * (e10.x - e00.x) + ry[u] * (e11.x - e01.x));
		double gyx = g.idy * (dxw * (e01.x - e00.x) + rx[u] * (e11.x - e10.x));
		double gxy = g.idx * (dyw * (e10.y - e00.y) + ry[u] * (e11.y - e01.y));
		double gyy = g.idy * (dxw * (e01.y - e00.y) + rx[u] * (e11.y - e10.y));
		lx[i] = ax + (lex[u] * gxx + ley[u] * gxy);
		ly[i] = ay + (lex[u] * gyx + ley[u] * gyy);
	}
	Box b = block_box<PPT>(g, ix, iy, s6, REV_BOX_NODES);
	box_zero(b, sacc, 2);
#pragma unroll
	for(int u = 0; u < PPT; u++)
	{
		if(ix[u] < 0)
			continue;
		double dxw = 1.0 - rx[u], dyw = 1.0 - ry[u];
		double w[4] = {dxw * dyw, dxw * ry[u], rx[u] * dyw, rx[u] * ry[u]};
		const int ddx[4] = {0, 0, 1, 1}, ddy[4] = {0, 1, 0, 1};
#pragma unroll
		for(int c = 0; c < 4; c++)
		{
			if(b.lds)
			{
				LDS_AS double *l = (LDS_AS double *) sacc;
				int nd = box_node(g, b, ix[u], iy[u], ddx[c], ddy[c]);
				lds_add(&l[2 * nd], w[c] * lex[u]);
				lds_add(&l[2 * nd + 1], w[c] * ley[u]);
			}
			else
			{
				GLB_AS double *m = gptr<double>(lE);
				int64_t nd = wrap_node(g, ix[u] + ddx[c], iy[u] + ddy[c]);
				glb_add(&m[2 * nd], w[c] * lex[u]);
				glb_add(&m[2 * nd + 1], w[c] * ley[u]);
			}
		}
	}
	box_flush(g, b, sacc, 2, (double *) lE, 2);
}

// psi = D^T lE - srho * rho, D the central-difference E stencil
// (E_x[i] = (phi[i-1] - phi[i+1]) / 2dx, so (D_x^T a)[i] = (a[i+1] - a[i-1]) / 2dx);
// zeroes lE_zero (the other lE buffer, which the next reverse iteration
// deposits into)
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_field(Geo g, const double2 *__restrict__ lE, const double *__restrict__ rho,
		double srho, double *__restrict__ psi, double2 *__restrict__ lE_zero)
{
	int64_t n = (int64_t) g.nx * g.ny;
	double dx2 = 2 * g.dx, dy2 = 2 * g.dy;
	for(int64_t i = blockIdx.x * (int64_t) blockDim.x + threadIdx.x; i < n;
			i += (int64_t) gridDim.x * blockDim.x)
	{
		int iy = (int) (i >> g.lgnx), ix = (int) (i & (g.nx - 1));
		int xm = ix == 0 ? g.nx - 1 : ix - 1, xp = ix == g.nx - 1 ? 0 : ix + 1;
		int ym = iy == 0 ? g.ny - 1 : iy - 1, yp = iy == g.ny - 1 ? 0 : iy + 1;
		int64_t row = (int64_t) iy * g.nx;
		double lphi = (lE[row + xp].x - lE[row + xm].x) / dx2 +
			(lE[(int64_t) yp * g.nx + ix].y - lE[(int64_t) ym * g.nx + ix].y) / dy2;
		psi[i] = lphi - srho * rho[i];
		lE_zero[i] = make_double2(0.0, 0.0);
	}
}

// lr += c * grad Gat(lrho)(r) for the last iteration of the sweep (the
// others are applied by the next k_adj_rev_a)
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_rev_b(Geo g, AdjSpecies k, int64_t n, const uint8_t *__restrict__ sp,
		const double *__restrict__ x, const double *__restrict__ y,
		const double *__restrict__ lrho, double *__restrict__ lx, double *__restrict__ ly)
{
	for(int64_t i = blockIdx.x * (int64_t) blockDim.x + threadIdx.x; i < n;
			i += (int64_t) gridDim.x * blockDim.x)
	{
		double ax = lx[i], ay = ly[i];
		rev_b_term(g, k.c[sp[i]], x[i], y[i], lrho, ax, ay);
		lx[i] = ax;
		ly[i] = ay;
	}
}

// ------------------------------------------------------ particle order ---
//
// The particles are kept in the order of their initial cell, and within each
// run of ADJ_CHUNK positions the cells are taken round-robin: one particle of
// every cell that still has one, per round, so that the 64 consecutive
// particles of a wavefront lie in different cells and their deposit atomics
// spread over the LDS banks.  The particles of one cell come in the order in
// which the counting reached them, another one in each forward: only sums
// of deposits, whose order is open anyway, see it (sort_by_cell_rr() in host_sort.h
// states the same order of cells sequentially, with the caller's order within
// each).  Counted, scanned and placed on the device;
// 4,194,304 particles at 256^2, a forward and a backward from host arrays:
// 69.4 ms with the order made, applied and undone by 16 host threads, 48.2 ms so.

#define ADJ_SCAN 2048             // cells per block of the scan
#define ADJ_DERR_INPUT 0x100      // derr: a particle outside the box or not finite

// cell[i] of the caller's particle i, rank[i] its number among the particles
// of its cell, cnt[cell] their count
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_cells(Geo g, int64_t n, const double *__restrict__ raw, int32_t *__restrict__ cell,
		int32_t *__restrict__ rank, int32_t *__restrict__ cnt, int *__restrict__ derr)
{
	bool bad = false;
	for(int64_t i = blockIdx.x * (int64_t) blockDim.x + threadIdx.x; i < n;
			i += (int64_t) gridDim.x * blockDim.x)
	{
		const double x = raw[i], y = raw[n + i];
		int c = 0;
		if(x >= 0.0 && x <= g.L0 && y >= 0.0 && y <= g.L1)
			c = min((int) (y * g.idy), g.ny - 1) * g.nx + min((int) (x * g.idx), g.nx - 1);
		else
			bad = true;
		if(!isfinite(raw[2 * n + i]) || !isfinite(raw[3 * n + i]))
			bad = true;
		cell[i] = c;
		rank[i] = atomicAdd(&cnt[c], 1);
	}
	if(bad)
		atomicOr(derr, ADJ_DERR_INPUT);
}

// Sum of v over the threads before this one, and over all of them (into *all).
static __device__ __forceinline__ int64_t block_before(int64_t v, int64_t *s_w, int64_t *all)
{
	const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
	int64_t x = v;
	for(int off = 1; off < 64; off <<= 1)
	{
		int64_t o = __shfl_up((long long) x, off);
		if(lane >= off)
			x += o;
	}
	__syncthreads();
	if(lane == 63)
		s_w[wid] = x;
	__syncthreads();
	int64_t before = x - v, t = 0;
	for(int w = 0; w < nw; w++)
	{
		if(w < wid)
			before += s_w[w];
		t += s_w[w];
	}
	*all = t;
	return before;
}

// Particles in each ADJ_SCAN cells
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_scan_sums(int64_t cells, const int32_t *__restrict__ cnt, int64_t *__restrict__ part)
{
	__shared__ int64_t s_w[CPIC_BLOCK / 64];
	int64_t sum = 0, all;
	for(int64_t k = threadIdx.x; k < ADJ_SCAN; k += CPIC_BLOCK)
	{
		int64_t c = (int64_t) blockIdx.x * ADJ_SCAN + k;
		sum += c < cells ? cnt[c] : 0;
	}
	block_before(sum, s_w, &all);
	if(threadIdx.x == 0)
		part[blockIdx.x] = all;
}

// Exclusive scan of the n sums, one block
__global__ __launch_bounds__(1024)
void k_adj_scan_part(int n, int64_t *__restrict__ part)
{
	__shared__ int64_t s_w[1024 / 64];
	int64_t carry = 0;
	for(int k = 0; k < n; k += 1024)
	{
		const int i = k + (int) threadIdx.x;
		int64_t v = i < n ? part[i] : 0, all;
		int64_t b = block_before(v, s_w, &all);
		if(i < n)
			part[i] = carry + b;
		carry += all;
	}
}

// start[c]: particles in the cells before c
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_scan_starts(int64_t cells, const int32_t *__restrict__ cnt,
		const int64_t *__restrict__ part, int64_t *__restrict__ start)
{
	__shared__ int64_t s_w[CPIC_BLOCK / 64];
	constexpr int PER = ADJ_SCAN / CPIC_BLOCK;
	const int64_t c0 = (int64_t) blockIdx.x * ADJ_SCAN + (int64_t) threadIdx.x * PER;
	int v[PER];
	int64_t sum = 0, all;
	for(int k = 0; k < PER; k++)
	{
		v[k] = c0 + k < cells ? cnt[c0 + k] : 0;
		sum += v[k];
	}
	int64_t at = part[blockIdx.x] + block_before(sum, s_w, &all);
	for(int k = 0; k < PER; k++)
	{
		if(c0 + k < cells)
			start[c0 + k] = at;
		at += v[k];
	}
}

// The particles by cell: position j holds the caller's particle order[j], of
// cell scell[j]
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_place(int64_t n, const int32_t *__restrict__ cell, const int32_t *__restrict__ rank,
		const int64_t *__restrict__ start, int64_t *__restrict__ order,
		int32_t *__restrict__ scell)
{
	for(int64_t i = blockIdx.x * (int64_t) blockDim.x + threadIdx.x; i < n;
			i += (int64_t) gridDim.x * blockDim.x)
	{
		const int c = cell[i];
		const int64_t j = start[c] + rank[i];
		order[j] = i;
		scell[j] = c;
	}
}

// Takes the cells of one chunk round-robin and fetches the state in the
// resulting order.  The r-th particle (from 0) of the chunk's q-th cell follows the
// first r particles of every cell, and the r-th ones of the cells before it.
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_robin(int64_t n, const int64_t *__restrict__ order, const int32_t *__restrict__ scell,
		const double *__restrict__ raw, const uint8_t *__restrict__ sp0,
		int64_t *__restrict__ perm, double *__restrict__ x, double *__restrict__ y,
		double *__restrict__ ux, double *__restrict__ uy, uint8_t *__restrict__ sp)
{
	__shared__ int s_cell[ADJ_CHUNK], s_head[ADJ_CHUNK + 1];
	__shared__ int64_t s_w[CPIC_BLOCK / 64];
	const int64_t c0 = (int64_t) blockIdx.x * ADJ_CHUNK;
	const int m = (int) min((int64_t) ADJ_CHUNK, n - c0);
	for(int j = threadIdx.x; j < m; j += CPIC_BLOCK)
		s_cell[j] = scell[c0 + j];
	__syncthreads();
	// the chunk's cells: s_head[q] is the q-th one's first position
	const int j0 = threadIdx.x * ADJ_PPT;
	int q[ADJ_PPT], heads = 0;
	for(int u = 0; u < ADJ_PPT; u++)
	{
		const int j = j0 + u;
		if(j < m && (j == 0 || s_cell[j] != s_cell[j - 1]))
			heads++;
		q[u] = heads;
	}
	int64_t all;
	const int before = (int) block_before(heads, s_w, &all);
	const int nq = (int) all;
	for(int u = 0; u < ADJ_PPT; u++)
	{
		const int j = j0 + u;
		q[u] += before - 1;
		if(j < m && (j == 0 || s_cell[j] != s_cell[j - 1]))
			s_head[q[u]] = j;
	}
	if(threadIdx.x == 0)
		s_head[nq] = m;
	__syncthreads();
	int r[ADJ_PPT], f[ADJ_PPT];
	for(int u = 0; u < ADJ_PPT; u++)
	{
		r[u] = j0 + u < m ? j0 + u - s_head[q[u]] : 0;
		f[u] = 0;
	}
	for(int k = 0, h = 0; k < nq; k++)
	{
		const int hn = s_head[k + 1], len = hn - h;
		h = hn;
#pragma unroll
		for(int u = 0; u < ADJ_PPT; u++)
			f[u] += min(len, r[u]) + (k < q[u] && len > r[u] ? 1 : 0);
	}
	for(int u = 0; u < ADJ_PPT; u++)
	{
		if(j0 + u >= m)
			continue;
		const int64_t i = order[c0 + j0 + u], o = c0 + f[u];
		perm[o] = i;
		x[o] = raw[i];
		y[o] = raw[n + i];
		ux[o] = raw[2 * n + i];
		uy[o] = raw[3 * n + i];
		sp[o] = sp0[i];
	}
}

// Four arrays in sorted order -> the caller's order (out: 4 arrays of n)
__global__ __launch_bounds__(CPIC_BLOCK)
void k_adj_unsort(int64_t n, const int64_t *__restrict__ perm, const double *__restrict__ a0,
		const double *__restrict__ a1, const double *__restrict__ a2,
		const double *__restrict__ a3, double *__restrict__ out)
{
	for(int64_t j = blockIdx.x * (int64_t) blockDim.x + threadIdx.x; j < n;
			j += (int64_t) gridDim.x * blockDim.x)
	{
		const int64_t i = perm[j];
		out[i] = a0[j];
		out[n + i] = a1[j];
		out[2 * n + i] = a2[j];
		out[3 * n + i] = a3[j];
	}
}

// ---------------------------------------------------------------- host ---

// blocks of the kernels that take ppt particles per thread
static unsigned
blocks_of(int64_t n, int ppt)
{
	return (unsigned) ((n + ppt * CPIC_BLOCK - 1) / (ppt * CPIC_BLOCK));
}

// blocks of the depositing kernels: one per ADJ_CHUNK particles
static int
chunks(int64_t n)
{
	return (int) blocks_of(n, ADJ_PPT);
}

static int
pblocks(int64_t n)
{
	int64_t b = (n + CPIC_BLOCK - 1) / CPIC_BLOCK;
	if(b > 65536)
		b = 65536;
	return b < 1 ? 1 : (int) b;
}

static void
adj_free(cpic_adj *a)
{
	if(!a)
		return;
	if(a->d)
		hipStreamSynchronize(a->d->stream);
	hipFree(a->sp); hipFree(a->sp0); hipFree(a->perm); hipFree(a->x); hipFree(a->y); hipFree(a->ux); hipFree(a->uy);
	hipFree(a->rho[0]); hipFree(a->rho[1]); hipFree(a->phi); hipFree(a->psi); hipFree(a->lrho);
	hipFree(a->E); hipFree(a->lE);
	hipFree(a->lx); hipFree(a->ly); hipFree(a->lux); hipFree(a->luy);
	hipFree(a->ck); hipFree(a->seg); hipFree(a->segf); hipFree(a->hist);
	hipFree(a->frho); hipFree(a->fE); hipFree(a->ph);
	hipFree(a->derr);
	hipFree(a->wk);
	if(a->evok)
		for(int i = 0; i < 4; i++)
			hipEventDestroy(a->ev[i]);
	if(a->d)
		cpic_dev_destroy(a->d);
	free(a);
}

static void
species_consts(const cpic_dev_desc_t *desc, double dtp, AdjSpecies *k)
{
	memset(k, 0, sizeof(*k));
	for(int s = 0; s < desc->nspecies; s++)
	{
		double h = 0.5 * dtp * desc->q[s] / desc->m[s];
		double tz = desc->B[2] * h;
		double sden = fma(tz, tz, 1.0);
		k->h[s] = h;
		k->tz[s] = tz;
		k->sz[s] = 2.0 * tz / sden;
		k->c[s] = -desc->q[s] / desc->e0;
	}
}

extern "C" int
cpic_adj_create(const cpic_dev_desc_t *desc, int64_t n, const int32_t *species,
		cpic_adj_t **out)
{
	cpic_dev_desc_t dd;
	cpic_adj *a;
	int ret;
	if(!desc || !out || n < 1 || !species || desc->precision != 64)
		return CPIC_EINVAL;
	*out = NULL;
	for(int64_t i = 0; i < n; i++)
		if(species[i] < 0 || species[i] >= desc->nspecies)
			return CPIC_EINVAL;
	dd = *desc;
	dd.flags = CPIC_F_NO_DIAG | CPIC_F_NO_GRAPH;
	a = (cpic_adj *) calloc(1, sizeof(*a));
	if(!a)
		return CPIC_ENOMEM;
	if((ret = cpic_dev_create(&dd, &a->d)))
	{
		free(a);
		return ret;
	}
	a->g = a->d->hgeo[0];
	a->n = n;
	a->ns = desc->nspecies;
	species_consts(desc, -desc->dt / 2, &a->k[0]);
	species_consts(desc, desc->dt, &a->k[1]);
	int64_t nodes = (int64_t) a->g.nx * a->g.ny;
	size_t pn = sizeof(double) * (size_t) n, gn = sizeof(double) * (size_t) nodes;
	uint8_t *sp8 = (uint8_t *) malloc((size_t) n);
	if(!sp8)
	{
		adj_free(a);
		return CPIC_ENOMEM;
	}
	for(int64_t i = 0; i < n; i++)
		sp8[i] = (uint8_t) species[i];
	if(hipMalloc(&a->sp, (size_t) n) != hipSuccess ||
			hipMalloc(&a->sp0, (size_t) n) != hipSuccess ||
			hipMemcpy(a->sp0, sp8, (size_t) n, hipMemcpyHostToDevice) != hipSuccess ||
			hipMalloc(&a->perm, sizeof(int64_t) * (size_t) n) != hipSuccess ||
			hipMalloc(&a->wk, 4 * pn) != hipSuccess ||
			hipMalloc(&a->x, pn) != hipSuccess || hipMalloc(&a->y, pn) != hipSuccess ||
			hipMalloc(&a->ux, pn) != hipSuccess || hipMalloc(&a->uy, pn) != hipSuccess ||
			hipMalloc(&a->lx, pn) != hipSuccess || hipMalloc(&a->ly, pn) != hipSuccess ||
			hipMalloc(&a->lux, pn) != hipSuccess || hipMalloc(&a->luy, pn) != hipSuccess ||
			hipMalloc(&a->rho[0], gn) != hipSuccess || hipMalloc(&a->rho[1], gn) != hipSuccess ||
			hipMalloc(&a->phi, gn) != hipSuccess || hipMalloc(&a->psi, gn) != hipSuccess ||
			hipMalloc(&a->lrho, gn) != hipSuccess ||
			hipMalloc(&a->E, 2 * gn) != hipSuccess || hipMalloc(&a->lE, 4 * gn) != hipSuccess ||
			hipMalloc(&a->derr, sizeof(int)) != hipSuccess)
	{
		free(sp8);
		adj_free(a);
		return CPIC_ENOMEM;
	}
	free(sp8);
	for(int i = 0; i < 4; i++)
		if(hipEventCreate(&a->ev[i]) != hipSuccess)
		{
			for(int j = 0; j < i; j++)
				hipEventDestroy(a->ev[j]);
			adj_free(a);
			return CPIC_EHIP;
		}
	a->evok = 1;
	*out = a;
	return 0;
}

extern "C" int
cpic_adj_destroy(cpic_adj_t *a)
{
	if(!a)
		return CPIC_EINVAL;
	hipSetDevice(a->d->device);
	adj_free(a);
	return 0;
}

static int
grow(double **p, int64_t *cap, int64_t want)
{
	if(*cap >= want)
		return 0;
	hipFree(*p);
	*p = NULL;
	*cap = 0;
	if(hipMalloc(p, sizeof(double) * (size_t) want) != hipSuccess)
		return CPIC_ENOMEM;
	*cap = want;
	return 0;
}

static void
release(double **p, int64_t *cap)
{
	if(*p)
		hipFree(*p);
	*p = NULL;
	*cap = 0;
}

static int
zero(cpic_adj *a, double *p, int64_t n)
{
	return cpic_zero(a->d, p, n);
}

static int
deposit(cpic_adj *a, const double *x, const double *y, double *rho)
{
	int ret;
	if((ret = zero(a, rho, (int64_t) a->g.nx * a->g.ny)))
		return ret;
	hipLaunchKernelGGL(k_adj_deposit, dim3(chunks(a->n)), dim3(CPIC_BLOCK), 0, a->d->stream,
			a->g, a->k[1], a->n, a->sp, x, y, rho);
	HIPCHK(hipGetLastError());
	return 0;
}

// phi and E (into E) from rho; with w, the field energy of rho,
// -(e0/2) sum rho phi, is added to *w (zero beforehand; the column pass of
// the solve sums it over the spectrum, sum_k G |rho^(k)|^2 / (nx ny), equal
// to sum rho phi by Parseval); with rho_zero, that (other) buffer is zeroed
// by the solve's last pass
static int
fields(cpic_adj *a, const double *rho, double *w, double *rho_zero, double2 *E)
{
	return cpic_solve_ptr_E(a->d, rho, a->phi, rho_zero, w, E);
}

// one forward iteration from positions (x, y), velocities (ux, uy) and
// rho_in = Dep(r): E of this iteration into E, the moved positions into
// (xo, yo) (may be (x, y)), Dep(r') of the moved particles into rho_out
static int
forward_step(cpic_adj *a, int64_t it, const double *x, const double *y, double *xo,
		double *yo, const double *rho_in, double *rho_out, double2 *E, double *w)
{
	int ret;
	if((ret = fields(a, rho_in, w, rho_out, E)))
		return ret;
	int first = it == 0;
	double dtp = first ? -a->g.dt / 2 : a->g.dt;
	if(a->n <= ADJ_FEW)
		hipLaunchKernelGGL((k_adj_push<true, 1>), dim3(blocks_of(a->n, 1)), dim3(CPIC_BLOCK), 0,
				a->d->stream,
				a->g, a->k[first ? 0 : 1], first ? 0 : 1, dtp, a->n, a->sp, x, y, xo, yo, a->ux,
				a->uy, (const double2 *) E, rho_out, a->derr);
	else
		hipLaunchKernelGGL((k_adj_push<true, ADJ_PPT>), dim3(chunks(a->n)), dim3(CPIC_BLOCK), 0,
				a->d->stream,
				a->g, a->k[first ? 0 : 1], first ? 0 : 1, dtp, a->n, a->sp, x, y, xo, yo, a->ux,
				a->uy, (const double2 *) E, rho_out, a->derr);
	HIPCHK(hipGetLastError());
	return 0;
}

// The particle half of forward_step, for the reverse sweep's recompute with
// a field history: positions (and the velocities in place) of iteration
// it + 1 from those of it with E of it; no deposit
static int
move_step(cpic_adj *a, int64_t it, const double *x, const double *y, double *xo, double *yo,
		const double2 *E)
{
	int first = it == 0;
	double dtp = first ? -a->g.dt / 2 : a->g.dt;
	hipLaunchKernelGGL((k_adj_push<false, MOVE_PPT>),
			dim3(blocks_of(a->n, MOVE_PPT)),
			dim3(CPIC_BLOCK), 0, a->d->stream,
			a->g, a->k[first ? 0 : 1], first ? 0 : 1, dtp, a->n, a->sp, x, y, xo, yo, a->ux,
			a->uy, E, (double *) NULL, a->derr);
	HIPCHK(hipGetLastError());
	return 0;
}

// forward_step in place on the state, on the double-buffered rho[cur] /
// rho[1-cur] and the E array
static int
forward_iter(cpic_adj *a, int64_t it, int *cur, double *w)
{
	int ret, c = *cur;
	if((ret = forward_step(a, it, a->x, a->y, a->x, a->y, a->rho[c], a->rho[1 - c], a->E, w)))
		return ret;
	*cur = 1 - c;
	return 0;
}

static int
adj_derr(cpic_adj *a)
{
	int e = 0;
	HIPCHK(hipMemcpyAsync(&e, a->derr, sizeof(int), hipMemcpyDeviceToHost, a->d->stream));
	HIPCHK(hipStreamSynchronize(a->d->stream));
	if(e & CPIC_DERR_UMAX)
		return CPIC_EUMAX;
	if(e & CPIC_DERR_NAN)
		return CPIC_ENAN;
	return 0;
}

static int
copy_state(cpic_adj *a, double *dst, const double *x, const double *y, const double *ux,
		const double *uy, hipMemcpyKind kind)
{
	size_t pn = sizeof(double) * (size_t) a->n;
	int64_t n = a->n;
	HIPCHK(hipMemcpyAsync(dst, x, pn, kind, a->d->stream));
	HIPCHK(hipMemcpyAsync(dst + n, y, pn, kind, a->d->stream));
	if(ux)
		HIPCHK(hipMemcpyAsync(dst + 2 * n, ux, pn, kind, a->d->stream));
	if(uy)
		HIPCHK(hipMemcpyAsync(dst + 3 * n, uy, pn, kind, a->d->stream));
	return 0;
}

// The caller's particles, in wk, into the state in sorted order (see "particle
// order"); CPIC_EINVAL, with the state as it was, if one is outside the box or
// not finite.  The reverse sweep's buffers hold the intermediate arrays.
static int
sort_in(cpic_adj *a)
{
	const int64_t n = a->n, cells = (int64_t) a->g.nx * a->g.ny;
	int32_t *cell = (int32_t *) a->ly, *rank = cell + n, *scell = (int32_t *) a->lux;
	int32_t *cnt = (int32_t *) a->lrho;
	int64_t *order = (int64_t *) a->lx, *start = (int64_t *) a->psi, *part = (int64_t *) a->rho[1];
	const int sb = (int) ((cells + ADJ_SCAN - 1) / ADJ_SCAN);
	const dim3 block(CPIC_BLOCK), pb(pblocks(n));
	hipStream_t st = a->d->stream;
	int ret, e = 0;
	// cells is even: both grid sides are powers of two from 2 up
	if((ret = zero(a, (double *) cnt, cells / 2)))
		return ret;
	HIPCHK(hipMemsetAsync(a->derr, 0, sizeof(int), st));
	hipLaunchKernelGGL(k_adj_cells, pb, block, 0, st, a->g, n, (const double *) a->wk, cell, rank,
			cnt, a->derr);
	hipLaunchKernelGGL(k_adj_scan_sums, dim3(sb), block, 0, st, cells, cnt, part);
	hipLaunchKernelGGL(k_adj_scan_part, dim3(1), dim3(1024), 0, st, sb, part);
	hipLaunchKernelGGL(k_adj_scan_starts, dim3(sb), block, 0, st, cells, cnt, part, start);
	hipLaunchKernelGGL(k_adj_place, pb, block, 0, st, n, cell, rank, start, order, scell);
	HIPCHK(hipGetLastError());
	HIPCHK(hipMemcpyAsync(&e, a->derr, sizeof(int), hipMemcpyDeviceToHost, st));
	HIPCHK(hipStreamSynchronize(st));
	if(e & ADJ_DERR_INPUT)
		return CPIC_EINVAL;
	hipLaunchKernelGGL(k_adj_robin, dim3(chunks(n)), block, 0, st, n, order, scell,
			(const double *) a->wk, (const uint8_t *) a->sp0, a->perm, a->x, a->y, a->ux, a->uy,
			a->sp);
	HIPCHK(hipGetLastError());
	return 0;
}

// Device arrays in sorted order -> host arrays in the caller's order.
static int
download_unsorted(cpic_adj *a, double *const *src, double *const *dst)
{
	const int64_t n = a->n;
	DlRange r[4];
	int nr = 0;
	hipLaunchKernelGGL(k_adj_unsort, dim3(pblocks(n)), dim3(CPIC_BLOCK), 0, a->d->stream, n,
			(const int64_t *) a->perm, (const double *) src[0], (const double *) src[1],
			(const double *) src[2], (const double *) src[3], a->wk);
	HIPCHK(hipGetLastError());
	for(int c = 0; c < 4; c++)
		if(dst[c])
			r[nr++] = {dst[c], a->wk + c * n, sizeof(double) * (size_t) n};
	return nr ? cpic_download(a->d, nr, r) : 0;
}

// Whether this forward keeps its position history, whose memory is then there.
// The buffers of the way not taken, left by an earlier forward, are given back.
static bool
pos_history(cpic_adj *a, int64_t nsteps)
{
	size_t avail = 0, total = 0;
	const double want = 2.0 * (double) a->n * (double) nsteps;
	const double held = (double) a->phcap + (double) a->ckcap + (double) a->segcap;
	bool keep = a->fhist && !a->phist_off && want * sizeof(double) <= (double) ADJ_POS_HISTORY_MAX;
	if(keep && (double) a->phcap < want)
		keep = hipMemGetInfo(&avail, &total) == hipSuccess &&
			want * sizeof(double) <= 0.5 * ((double) avail + sizeof(double) * held);
	if(keep)
	{
		release(&a->ck, &a->ckcap);
		release(&a->seg, &a->segcap);
		keep = !grow(&a->ph, &a->phcap, (int64_t) want);
	}
	if(!keep)
	{
		// checkpoints instead
		(void) hipGetLastError();
		release(&a->ph, &a->phcap);
	}
	return keep;
}

extern "C" int
cpic_adj_forward(cpic_adj_t *a, const double *x, const double *y, const double *ux,
		const double *uy, int64_t nsteps, int32_t checkpoint_every, double *loss,
		double *energy)
{
	int ret, cur = 0;
	if(!a || !x || !y || !ux || !uy || nsteps < 1 || checkpoint_every < 1)
		return CPIC_EINVAL;
	hipSetDevice(a->d->device);
	int64_t K = checkpoint_every, nck = (nsteps + K - 1) / K, n = a->n;
	if((ret = grow(&a->hist, &a->histcap, nsteps)))
		return ret;
	const size_t pn = sizeof(double) * (size_t) n;
	const DlRange up[4] = {{a->wk, x, pn}, {a->wk + n, y, pn}, {a->wk + 2 * n, ux, pn},
		{a->wk + 3 * n, uy, pn}};
	if((ret = cpic_upload(a->d, 4, up)) || (ret = sort_in(a)))
		return ret;
	a->have = 0;
	a->evrec = 0;             // a backward belongs to the forward before it
	// the field history, when it fits: each iteration's rho and E are
	// written straight into their slots (the solve zeroes the slot the push
	// deposits into), at no extra work in the forward
	const int64_t nodes = (int64_t) a->g.nx * a->g.ny;
	a->fhist = 0;
	if(!a->fhist_off &&
			(double) nodes * (3.0 * (double) nsteps + 1.0) * sizeof(double) <=
			(double) ADJ_FIELD_HISTORY_MAX)
	{
		if(!grow(&a->frho, &a->frhocap, nodes * (nsteps + 1)) &&
				!grow(&a->fE, &a->fEcap, 2 * nodes * nsteps))
			a->fhist = 1;
		else
			(void) hipGetLastError();   // no room: the reverse recomputes instead
	}
	a->phist = pos_history(a, nsteps);
	if(!a->phist && (ret = grow(&a->ck, &a->ckcap, 4 * n * nck)))
		return ret;
	HIPCHK(hipEventRecord(a->ev[0], a->d->stream));
	if((ret = deposit(a, a->x, a->y, a->fhist ? a->frho : a->rho[0])) ||
			(ret = zero(a, a->hist, nsteps)))
		return ret;
	for(int64_t it = 0; it < nsteps; it++)
	{
		if(a->phist && it == 0)
		{
			if((ret = copy_state(a, a->ph, a->x, a->y, NULL, NULL, hipMemcpyDeviceToDevice)))
				return ret;
		}
		else if(!a->phist && it % K == 0)
			if((ret = copy_state(a, a->ck + 4 * n * (it / K), a->x, a->y, a->ux, a->uy,
					hipMemcpyDeviceToDevice)))
				return ret;
		if(a->fhist)
		{
			// with the position history, from its slot to the next one or, the
			// last, to the state
			double *from = a->phist ? a->ph + 2 * n * it : NULL;
			bool last = !a->phist || it + 1 == nsteps;
			ret = forward_step(a, it, from ? from : a->x, from ? from + n : a->y,
					last ? a->x : from + 2 * n, last ? a->y : from + 3 * n, a->frho + nodes * it,
					a->frho + nodes * (it + 1), (double2 *) a->fE + nodes * it, a->hist + it);
		}
		else
			ret = forward_iter(a, it, &cur, a->hist + it);
		if(ret)
			return ret;
	}
	HIPCHK(hipEventRecord(a->ev[1], a->d->stream));
	a->evrec |= 1;
	double *h = (double *) malloc(sizeof(double) * (size_t) nsteps);
	if(!h)
		return CPIC_ENOMEM;
	if(hipMemcpyAsync(h, a->hist, sizeof(double) * nsteps, hipMemcpyDeviceToHost, a->d->stream)
			!= hipSuccess || hipStreamSynchronize(a->d->stream) != hipSuccess)
	{
		free(h);
		return CPIC_EHIP;
	}
	double L = 0.0;
	for(int64_t it = 0; it < nsteps; it++)
		L += h[it];
	if(energy)
		memcpy(energy, h, sizeof(double) * nsteps);
	free(h);
	if(loss)
		*loss = L;
	if((ret = adj_derr(a)))
		return ret;
	a->nsteps = nsteps;
	a->K = (int) K;
	a->have = 1;
	return 0;
}

extern "C" int
cpic_adj_device_ms(cpic_adj_t *a, double *forward_ms, double *backward_ms)
{
	if(!a || !a->evok)
		return CPIC_EINVAL;
	float f = 0.0f, b = 0.0f;
	hipSetDevice(a->d->device);
	if(a->evrec & 1)
		HIPCHK(hipEventElapsedTime(&f, a->ev[0], a->ev[1]));
	if(a->evrec & 2)
		HIPCHK(hipEventElapsedTime(&b, a->ev[2], a->ev[3]));
	if(forward_ms)
		*forward_ms = (a->evrec & 1) ? (double) f : -1.0;
	if(backward_ms)
		*backward_ms = (a->evrec & 2) ? (double) b : -1.0;
	return 0;
}

extern "C" int
cpic_adj_set_field_history(cpic_adj_t *a, int on)
{
	if(!a)
		return CPIC_EINVAL;
	a->fhist_off = !on;
	return 0;
}

extern "C" int
cpic_adj_set_position_history(cpic_adj_t *a, int on)
{
	if(!a)
		return CPIC_EINVAL;
	a->phist_off = !on;
	return 0;
}

extern "C" int
cpic_adj_state(cpic_adj_t *a, double *x, double *y, double *ux, double *uy)
{
	if(!a || !a->have)
		return CPIC_EINVAL;
	hipSetDevice(a->d->device);
	double *src[4] = {a->x, a->y, a->ux, a->uy};
	double *dst[4] = {x, y, ux, uy};
	return download_unsorted(a, src, dst);
}

extern "C" int
cpic_adj_backward(cpic_adj_t *a, double dloss, double *gx, double *gy, double *gux,
		double *guy)
{
	int ret;
	if(!a || !a->have)
		return CPIC_EINVAL;
	hipSetDevice(a->d->device);
	const int64_t n = a->n, T = a->nsteps, K = a->phist ? T : a->K, nodes = (int64_t) a->g.nx * a->g.ny;
	const int fh = a->fhist, ph = a->phist;
	// with the position history one segment is the whole run
	const int64_t nck = ph ? 1 : (T + K - 1) / K;
	// a segment holds at most min(K, T) iterations (the last one T - (nck-1) K),
	// the positions of all but its first in the segment buffer
	const int64_t Kseg = K < T ? K : T;
	if((!ph && (ret = grow(&a->seg, &a->segcap, 2 * n * (Kseg - 1)))) ||
			(!fh && (ret = grow(&a->segf, &a->segfcap, 3 * nodes * Kseg))))
		return ret;
	a->evrec &= ~2;
	HIPCHK(hipEventRecord(a->ev[2], a->d->stream));
	// both lE buffers start at zero; each iteration's k_adj_field zeroes the
	// one the next iteration deposits into
	if((ret = zero(a, a->lx, n)) || (ret = zero(a, a->ly, n)) || (ret = zero(a, a->lux, n)) ||
			(ret = zero(a, a->luy, n)) || (ret = zero(a, (double *) a->lE, 4 * nodes)))
		return ret;
	// keep the forward's final state: the recompute runs on copies
	double *fx = a->x, *fy = a->y, *fux = a->ux, *fuy = a->uy;
	double *wk = a->wk;
	a->x = wk;
	a->y = wk + n;
	a->ux = wk + 2 * n;
	a->uy = wk + 3 * n;
	ret = 0;
	// rho and E of iteration it (in the segment starting at it0), read by
	// the reverse iteration: the forward's field history, or recomputed with
	// the segment's positions below (no deposit or solve again in the
	// reverse iteration either way)
	double *const segf = a->segf, *const frho = a->frho;
	double2 *const fE = (double2 *) a->fE;
	auto seg_rho = [=](int64_t it, int64_t it0) {
		return fh ? frho + nodes * it : segf + 3 * nodes * (it - it0);
	};
	auto seg_E = [=](int64_t it, int64_t it0) {
		return fh ? fE + nodes * it : (double2 *) (segf + 3 * nodes * (it - it0) + nodes);
	};
	for(int64_t sg = nck - 1; sg >= 0 && !ret; sg--)
	{
		int64_t it0 = sg * K, it1 = it0 + K < T ? it0 + K : T;
		// positions (x, then y) of iteration it: the checkpoint's for the
		// segment's first, slot it - it0 - 1 of the segment buffer, which the
		// recompute's pushes write, for the others
		const double *c = ph ? a->ph : a->ck + 4 * n * sg;
		auto slot = [&](int64_t it) -> double * { return a->seg + 2 * n * (it - it0 - 1); };
		auto pos = [&](int64_t it) -> const double * {
			return ph ? a->ph + 2 * n * it : it == it0 ? c : slot(it);
		};
		// velocities only for a segment that moves its particles
		if(!ph && it1 - it0 > 1 &&
				(hipMemcpyAsync(a->ux, c + 2 * n, sizeof(double) * n, hipMemcpyDeviceToDevice,
						a->d->stream) != hipSuccess ||
				hipMemcpyAsync(a->uy, c + 3 * n, sizeof(double) * n, hipMemcpyDeviceToDevice,
						a->d->stream) != hipSuccess))
		{
			ret = CPIC_EHIP;
			break;
		}
		if(ph)
			;                  // positions and fields are there
		else if(fh)
		{
			// positions only, moved by the history's E
			for(int64_t it = it0; it + 1 < it1 && !ret; it++)
				ret = move_step(a, it, pos(it), pos(it) + n, slot(it + 1), slot(it + 1) + n,
						seg_E(it, it0));
		}
		else
		{
			if((ret = deposit(a, pos(it0), pos(it0) + n, seg_rho(it0, it0))))
				break;
			for(int64_t it = it0; it < it1 && !ret; it++)
			{
				if(it + 1 < it1)
					ret = forward_step(a, it, pos(it), pos(it) + n, slot(it + 1), slot(it + 1) + n,
							seg_rho(it, it0), seg_rho(it + 1, it0), seg_E(it, it0),
							(double *) NULL);
				else
					ret = fields(a, seg_rho(it, it0), (double *) NULL, (double *) NULL,
							seg_E(it, it0));
			}
		}
		for(int64_t it = it1 - 1; it >= it0 && !ret; it--)
		{
			const double *sx = pos(it), *sy = sx + n;
			int first = it == 0;
			double dtp = first ? -a->g.dt / 2 : a->g.dt;
			double2 *lE = a->lE + (it & 1) * nodes, *lE_next = a->lE + ((it + 1) & 1) * nodes;
			const bool few = n <= ADJ_FEW, pend = it + 1 < T;
			// the lrho term of iteration it + 1, at its positions: the
			// segment's next slot, or the next checkpoint's
			const double *bx = !pend ? NULL : it + 1 < it1 ? pos(it + 1) : a->ck + 4 * n * (sg + 1);
			auto rev = [&](auto kern, int ppt) {
				hipLaunchKernelGGL(kern, dim3(blocks_of(n, ppt)), dim3(CPIC_BLOCK), 0, a->d->stream,
						a->g, a->k[first ? 0 : 1], first ? 0 : 1, dtp, n, a->sp, sx, sy,
						(const double2 *) seg_E(it, it0), a->lx, a->ly, a->lux, a->luy, lE,
						bx, pend ? bx + n : NULL, (const double *) a->lrho);
			};
			if(few && pend)
				rev(k_adj_rev_a<true, 1>, 1);
			else if(few)
				rev(k_adj_rev_a<false, 1>, 1);
			else if(pend)
				rev(k_adj_rev_a<true, REV_PPT>, REV_PPT);
			else
				rev(k_adj_rev_a<false, REV_PPT>, REV_PPT);
			if(a->d->fft_small)
			{
				if(hipGetLastError() != hipSuccess)
					ret = CPIC_EHIP;
				else
					ret = cpic_solve_transposed_small(a->d, lE, seg_rho(it, it0),
							dloss * a->g.e0, lE_next, a->lrho);
				continue;
			}
			hipLaunchKernelGGL(k_adj_field, dim3(pblocks(nodes)), dim3(CPIC_BLOCK), 0,
					a->d->stream, a->g, (const double2 *) lE, seg_rho(it, it0),
					dloss * a->g.e0, a->psi, lE_next);
			if(hipGetLastError() != hipSuccess)
			{
				ret = CPIC_EHIP;
				break;
			}
			if((ret = cpic_solve_ptr(a->d, a->psi, a->lrho)))
				break;
		}
	}
	// the lrho term of iteration 0 (its positions: the history's or the first
	// checkpoint's)
	const double *r0 = ph ? a->ph : a->ck;
	if(!ret)
	{
		hipLaunchKernelGGL(k_adj_rev_b, dim3(pblocks(n)), dim3(CPIC_BLOCK), 0, a->d->stream,
				a->g, a->k[1], n, a->sp, r0, r0 + n,
				(const double *) a->lrho, a->lx, a->ly);
		if(hipGetLastError() != hipSuccess)
			ret = CPIC_EHIP;
	}
	if(!ret && hipEventRecord(a->ev[3], a->d->stream) == hipSuccess)
		a->evrec |= 2;
	hipStreamSynchronize(a->d->stream);
	a->x = fx;
	a->y = fy;
	a->ux = fux;
	a->uy = fuy;
	if(ret)
		return ret;
	double *src[4] = {a->lx, a->ly, a->lux, a->luy};
	double *dst[4] = {gx, gy, gux, guy};
	if((ret = download_unsorted(a, src, dst)))
		return ret;
	return adj_derr(a);
}
