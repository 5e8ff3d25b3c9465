// sepdev_list.hip -- cell binning and Verlet neighbour-list build.
//
// A rebuild is a short kernel sequence on the library stream:
//   k_bin          cell index per atom (reference formula or floor+wrap),
//                  per-cell counts and slots by wave-aggregated atomics
//   k_scan         one workgroup: exclusive scan of the counts -> cell_start
//   k_scatter      atom -> start of its cell + its slot
//                  (k_scan_scatter: both in one launch, every workgroup
//                  scanning the counts itself, for grids of up to 16352
//                  cells)
//   k_sort_permute a half-wave per cell (a wave for cells of more than 32
//                  atoms on average): order the segment by original atom
//                  index (so the device order and every list are independent
//                  of atomic timing) and move each member's state to its new
//                  cell-sorted index in the spare copy
//                  (k_order: all of these in one launch, for systems of up to
//                  32768 atoms, where it says so)
//   k_build_q      a wave per slab of a cell's atoms (k_build: a workgroup per
//                  cell, for boxes that are not cubic): the stencil's atoms
//                  within the list cutoff, 64 candidates at a time; then copy
//                  the cells' permuted state home
// and a BUILD task for the step's finisher.  With conditional = 1 every
// kernel returns at once unless the device rebuild flag is set, so the
// sequence can sit in a captured graph.
//
// The pair multiset equals the reference's half list of
// source/sepprfrc.c:419-513 (and its exclusion variants :517-700) taken in
// both directions: every half-shell offset s contributes j in cell(i)+s
// ("forward") and cell(i)-s ("backward"), with the reference's
// "m1 != m2 || j2 > j1" rule applied on original indices when the offset
// wraps back onto the home cell.  r2 is formed as the reference does
// (difference, single-image wrap, x2 + y2 + z2 in that order, each
// operation rounded on its own), so the set is identical bit for bit.
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "sepdev_impl.h"

__device__ __forceinline__ void sepk_set_error(sepdev_sys *sys, int code)
{
	atomicCAS(&sys->error, 0, code);
}

__device__ __forceinline__ int sepk_mod(int a, int n)
{
	int r = a % n;
	return r < 0 ? r + n : r;
}

// Linear cell index of a position, or -1 if it falls outside the grid.
__device__ __forceinline__ long sepk_cell_of(const sepk_pos &p, const sepdev_grid &g)
{
	const double q[3] = {p.x / g.l[0], p.y / g.l[1], p.z / g.l[2]};
	int c[3];
	for (int k = 0; k < 3; k++) {
		if (!(fabs(q[k]) < 1.0e9))
			return -1;
		if (g.ref_index)
			c[k] = (int)q[k]; // truncation, as source/sepprfrc.c:403-405
		else
			c[k] = sepk_mod((int)floor(q[k]), g.n[k]);
	}
	const long lin = (long)c[0] + (long)c[1] * g.n[0] + (long)c[2] * g.n[0] * g.n[1];
	const long ncell = (long)g.n[0] * g.n[1] * g.n[2];
	if (lin < 0 || lin >= ncell)
		return -1;
	return lin;
}

#define SEPK_GRID_CAP 2048 // grid-stride launches: at most this many blocks

// Cell index of every atom and its slot among the cell's members.  The
// lanes of a wave that share a cell take their slots with one atomic add per
// distinct cell (atoms arrive in the last build's cell order, so a wave holds
// a handful of runs), which keeps the device-wide atomics to a few per wave.
__global__ void k_bin(const sepk_pos *pos, long n, sepdev_grid g, int *cellid, int *slot,
		      int *count, sepdev_sys *sys, int conditional)
{
	if ((conditional && sys->neighb_flag == 0) || sys->error)
		return;
	// the build's atomic maximum starts here
	if (blockIdx.x == 0 && threadIdx.x == 0)
		sys->max_full = 0;
	const int lane = threadIdx.x & 63;
	const unsigned long long below = (1ull << lane) - 1ull;
	const long stride = (long)gridDim.x * blockDim.x;
	// whole waves iterate together (the bound is rounded up to a wave)
	const long nw = (n + 63) / 64 * 64;
	for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < nw; t += stride) {
		const bool act = t < n;
		long c = 0;
		if (act) {
			const sepk_pos p = pos[t];
			c = sepk_cell_of(p, g);
			if (c < 0) {
				sepk_set_error(sys, SEP_GPU_ECELL);
				c = 0;
			}
			// an atom outside [0, n*l) on some axis (allowed: it is
			// binned by truncation or wrapping) rules out the per-cell
			// image shifts
			const double q[3] = {p.x / g.l[0], p.y / g.l[1], p.z / g.l[2]};
			if (!(q[0] >= 0.0 && q[0] < g.n[0] && q[1] >= 0.0 && q[1] < g.n[1] &&
			      q[2] >= 0.0 && q[2] < g.n[2]))
				sys->unclean = 1;
			cellid[t] = (int)c;
		}
		unsigned long long todo = __ballot(act);
		int my = 0;
		while (todo) {
			const int lead = __ffsll((long long)todo) - 1;
			const int cl = __shfl((int)c, lead, 64);
			const unsigned long long same = __ballot(act && (int)c == cl);
			int base = 0;
			if (lane == lead)
				base = atomicAdd(&count[cl], __popcll(same));
			base = __shfl(base, lead, 64);
			if (act && (int)c == cl)
				my = base + __popcll(same & below);
			todo &= ~same;
		}
		if (act)
			slot[t] = my;
	}
}

// Exclusive scan of count[0..ncell) into start[0..ncell], zeroing count for
// the next rebuild.  One workgroup; each thread scans SEPK_SCAN_ITEMS
// consecutive cells of a pass in registers (one memory round trip per pass).
// It also fixes whether the rest of the rebuild runs: sys->frozen = an error
// is set (by an earlier step, or by this binning), read by the scatter,
// permutation and build kernels, which must all run or all skip (the build
// may itself raise an error while it runs).  The counts are zeroed either
// way, so a later rebuild starts from zero.
#define SEPK_SCAN_ITEMS 16
__global__ __launch_bounds__(1024) void k_scan(int *count, int *start, long ncell,
					       sepdev_sys *sys, int conditional)
{
	if (conditional && sys->neighb_flag == 0)
		return;
	if (threadIdx.x == 0)
		sys->frozen = sys->error != 0;
	__shared__ int wsum[16];
	__shared__ int carry_s;
	const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
	int carry = 0;
	const long pass = 1024L * SEPK_SCAN_ITEMS;
	for (long base = 0; base < ncell; base += pass) {
		const long c0 = base + (long)threadIdx.x * SEPK_SCAN_ITEMS;
		int v[SEPK_SCAN_ITEMS];
		if (c0 + SEPK_SCAN_ITEMS <= ncell) {
			// 16-byte aligned (count comes from hipMalloc, c0 % 16 == 0)
			const int4 *q = (const int4 *)(count + c0);
#pragma unroll
			for (int k = 0; k < SEPK_SCAN_ITEMS / 4; k++) {
				const int4 w = q[k];
				v[4 * k] = w.x;
				v[4 * k + 1] = w.y;
				v[4 * k + 2] = w.z;
				v[4 * k + 3] = w.w;
			}
		} else {
#pragma unroll
			for (int k = 0; k < SEPK_SCAN_ITEMS; k++)
				v[k] = c0 + k < ncell ? count[c0 + k] : 0;
		}
		int tot = 0;
#pragma unroll
		for (int k = 0; k < SEPK_SCAN_ITEMS; k++)
			tot += v[k];
		int x = tot; // inclusive wave scan of the thread totals
		for (int o = 1; o < 64; o <<= 1) {
			const int y = __shfl_up(x, o, 64);
			if (lane >= o)
				x += y;
		}
		if (lane == 63)
			wsum[wid] = x;
		__syncthreads();
		int off = carry;
		for (int w = 0; w < wid; w++)
			off += wsum[w];
		off += x - tot;
#pragma unroll
		for (int k = 0; k < SEPK_SCAN_ITEMS; k++) {
			if (c0 + k < ncell) {
				start[c0 + k] = off;
				count[c0 + k] = 0;
			}
			off += v[k];
		}
		if (threadIdx.x == 1023)
			carry_s = off;
		__syncthreads();
		carry = carry_s;
		__syncthreads();
	}
	if (threadIdx.x == 0)
		start[ncell] = carry;
}

// The scan and the scatter in one launch, for grids of at most
// SEPK_PLACE_CELLS cells: every workgroup scans the cell counts into LDS
// (one pass of SEPK_SCAN_ITEMS cells a thread, as k_scan), the first also
// writes them to start[], and each then places its share of the atoms.  No
// workgroup waits for another.  It fixes sys->frozen as k_scan does; the
// counts, which every workgroup reads, are zeroed by k_sort_permute.
#define SEPK_PLACE_CELLS (1024 * SEPK_SCAN_ITEMS - 32) // 64 KB of LDS with the wave sums
__global__ __launch_bounds__(1024) void k_scan_scatter(const int *count, int *start,
						       const int *cellid, const int *slot, int *order,
						       long ncell, long n, sepdev_sys *sys,
						       int conditional)
{
	if (conditional && sys->neighb_flag == 0)
		return;
	const bool frozen = sys->error != 0;
	if (blockIdx.x == 0 && threadIdx.x == 0)
		sys->frozen = frozen;
	if (frozen)
		return; // the permutation and the build skip as well
	__shared__ int sstart[SEPK_PLACE_CELLS + 1];
	__shared__ int wsum[16];
	const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
	const long c0 = (long)threadIdx.x * SEPK_SCAN_ITEMS;
	int v[SEPK_SCAN_ITEMS];
	if (c0 + SEPK_SCAN_ITEMS <= ncell) {
		// 16-byte aligned (count comes from hipMalloc, c0 % 16 == 0)
		const int4 *q = (const int4 *)(count + c0);
#pragma unroll
		for (int k = 0; k < SEPK_SCAN_ITEMS / 4; k++) {
			const int4 w = q[k];
			v[4 * k] = w.x;
			v[4 * k + 1] = w.y;
			v[4 * k + 2] = w.z;
			v[4 * k + 3] = w.w;
		}
	} else {
#pragma unroll
		for (int k = 0; k < SEPK_SCAN_ITEMS; k++)
			v[k] = c0 + k < ncell ? count[c0 + k] : 0;
	}
	int tot = 0;
#pragma unroll
	for (int k = 0; k < SEPK_SCAN_ITEMS; k++)
		tot += v[k];
	int x = tot; // inclusive wave scan of the thread totals
	for (int o = 1; o < 64; o <<= 1) {
		const int y = __shfl_up(x, o, 64);
		if (lane >= o)
			x += y;
	}
	if (lane == 63)
		wsum[wid] = x;
	__syncthreads();
	int off = 0;
	for (int w = 0; w < wid; w++)
		off += wsum[w];
	off += x - tot;
#pragma unroll
	for (int k = 0; k < SEPK_SCAN_ITEMS; k++) {
		if (c0 + k < ncell)
			sstart[c0 + k] = off;
		off += v[k];
		if (c0 + k == ncell - 1)
			sstart[ncell] = off;
	}
	__syncthreads();
	if (blockIdx.x == 0)
		for (long c = threadIdx.x; c <= ncell; c += blockDim.x)
			start[c] = sstart[c];
	for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n;
	     t += (long)gridDim.x * blockDim.x)
		order[sstart[cellid[t]] + slot[t]] = (int)t;
}

// Atom t -> its place in the cell-sorted order (slot from k_bin).
__global__ void k_scatter(const int *cellid, const int *slot, const int *start, int *order,
			  long n, sepdev_sys *sys, int conditional)
{
	if ((conditional && sys->neighb_flag == 0) || sys->frozen)
		return;
	for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n;
	     t += (long)gridDim.x * blockDim.x)
		order[start[cellid[t]] + slot[t]] = (int)t;
}

// Copies the partner table of atom o in src to slot t of dst, eight
// entries per round trip.
__device__ __forceinline__ void sepk_copy_partners(const sepk_state &src, const sepk_state &dst,
						   long o, long t, long npad)
{
	for (int k0 = 0; k0 < 40; k0 += 8) {
		int p[8];
#pragma unroll
		for (int k = 0; k < 8; k++)
			p[k] = sepk_at(src.partners + (size_t)(k0 + k) * npad, (unsigned)o);
#pragma unroll
		for (int k = 0; k < 8; k++)
			sepk_at(dst.partners + (size_t)(k0 + k) * npad, (unsigned)t) = p[k];
	}
}

// Moves atom o of src to slot t of dst.  Each half of the state is loaded
// whole before any of it is stored, so the move pays two memory round
// trips instead of one per field (source and destination may alias as far
// as the compiler knows).  pending: xn = x and cross_neighb = 0 are owed.
__device__ __forceinline__ void sepk_move_atom(const sepk_state &src, long o,
					       const sepk_state &dst, long t, long npad,
					       bool pending)
{
	const unsigned ou = (unsigned)o, tu = (unsigned)t;
	const sepk_pos p = sepk_at(src.pos, ou);
	{
		const int4 q = sepk_at(src.qpos, ou);
		const double v0 = sepk_at(src.v, ou), v1 = sepk_at(src.v + npad, ou);
		const double v2 = sepk_at(src.v + 2 * npad, ou);
		const double f0 = sepk_at(src.f, ou), f1 = sepk_at(src.f + npad, ou);
		const double f2 = sepk_at(src.f + 2 * npad, ou);
		const double a0 = sepk_at(src.a, ou), a1 = sepk_at(src.a + npad, ou);
		const double a2 = sepk_at(src.a + 2 * npad, ou);
		sepk_at(dst.pos, tu) = p;
		sepk_at(dst.qpos, tu) = q;
		sepk_at(dst.v, tu) = v0;
		sepk_at(dst.v + npad, tu) = v1;
		sepk_at(dst.v + 2 * npad, tu) = v2;
		sepk_at(dst.f, tu) = f0;
		sepk_at(dst.f + npad, tu) = f1;
		sepk_at(dst.f + 2 * npad, tu) = f2;
		sepk_at(dst.a, tu) = a0;
		sepk_at(dst.a + npad, tu) = a1;
		sepk_at(dst.a + 2 * npad, tu) = a2;
	}
	double x0 = sepk_at(src.xn, ou), x1 = sepk_at(src.xn + npad, ou);
	double x2 = sepk_at(src.xn + 2 * npad, ou);
	int n0 = sepk_at(src.cn, ou), n1 = sepk_at(src.cn + npad, ou), n2 = sepk_at(src.cn + 2 * npad, ou);
	const int r0 = sepk_at(src.cr, ou), r1 = sepk_at(src.cr + npad, ou);
	const int r2 = sepk_at(src.cr + 2 * npad, ou);
	const double m = sepk_at(src.m, ou);
	const int mol = sepk_at(src.mol, ou), orig = sepk_at(src.orig, ou);
	const signed char ty = sepk_at(src.type, ou);
	if (pending) {
		x0 = p.x;
		x1 = p.y;
		x2 = p.z;
		n0 = n1 = n2 = 0;
	}
	sepk_at(dst.xn, tu) = x0;
	sepk_at(dst.xn + npad, tu) = x1;
	sepk_at(dst.xn + 2 * npad, tu) = x2;
	sepk_at(dst.cn, tu) = n0;
	sepk_at(dst.cn + npad, tu) = n1;
	sepk_at(dst.cn + 2 * npad, tu) = n2;
	sepk_at(dst.cr, tu) = r0;
	sepk_at(dst.cr + npad, tu) = r1;
	sepk_at(dst.cr + 2 * npad, tu) = r2;
	sepk_at(dst.m, tu) = m;
	sepk_at(dst.mol, tu) = mol;
	sepk_at(dst.orig, tu) = orig;
	sepk_at(dst.type, tu) = ty;
}

// HW lanes per cell (grid-stride over cells; HW = 32: the two halves of a
// wave take two cells, for cells of up to about 32 atoms; HW = 64: a wave
// per cell): rank each member by its original index -- the keys of the
// cell are held one per lane and compared through shuffles within the
// group -- and move its state to start + rank in the spare copy.
template <int HW>
__global__ void k_sort_permute(const int *order, const int *start, sepk_state src,
			       sepk_state dst, int *iperm, long ncell,
			       long npad, sepdev_sys *sys, int conditional,
			       int has_partners, int *count)
{
	if (conditional && sys->neighb_flag == 0)
		return;
	// the counts start from zero at the next rebuild, whether this one runs
	// on or stops here
	for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell;
	     c += (long)gridDim.x * blockDim.x)
		count[c] = 0;
	if (sys->frozen)
		return;
	const int pending = sys->xn_pending;
	static_assert(HW == 32 || HW == 64, "half or whole waves");
	const int hl = threadIdx.x % HW;
	const long halves = (long)gridDim.x * (blockDim.x / HW);
	for (long c = ((long)blockIdx.x * blockDim.x + threadIdx.x) / HW; c < ncell; c += halves) {
		const int s = start[c], e = start[c + 1];
		for (int i0 = s; i0 < e; i0 += HW) {
			const int i = i0 + hl;
			const long o = i < e ? sepk_at(order, (unsigned)i) : 0;
			const int key = i < e ? sepk_at(src.orig, (unsigned)o) : 0;
			int rank = 0;
			for (int b = s; b < e; b += HW) {
				// keys of members b .. b + HW - 1, one per lane of the group
				const unsigned ob = b + hl < e ? (unsigned)sepk_at(order, (unsigned)(b + hl)) : 0u;
				const int kj = b == i0 ? key : (b + hl < e ? sepk_at(src.orig, ob) : 0);
				const int m = min(HW, e - b);
				for (int jj = 0; jj < m; jj++)
					rank += __shfl(kj, jj, HW) < key;
			}
			if (i >= e)
				continue;
			const long t = s + rank;
			sepk_move_atom(src, o, dst, t, npad, pending);
			sepk_at(iperm, (unsigned)key) = (int)t;
			if (has_partners)
				sepk_copy_partners(src, dst, o, t, npad);
		}
	}
}

// The same for cells of more than 64 atoms on average (dense molecular
// boxes): a workgroup per cell (grid-stride over cells).  The cell's keys
// go to LDS once, SEPK_SORT_KEYS at a time, and each thread ranks its
// members against them with broadcast reads, so a cell costs one round
// trip for its keys and one for its moves where a wave per cell pays one
// per 64 keys, and four waves work on it instead of one.  Same ranks, so
// the same permutation as k_sort_permute.
#define SEPK_SORT_KEYS 1024
__global__ __launch_bounds__(SEPK_BLOCK) void k_sort_permute_wg(
	const int *order, const int *start, sepk_state src, sepk_state dst, int *iperm,
	long ncell, long npad, sepdev_sys *sys, int conditional, int has_partners, int *count)
{
	if (conditional && sys->neighb_flag == 0)
		return;
	for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell;
	     c += (long)gridDim.x * blockDim.x)
		count[c] = 0;
	if (sys->frozen)
		return;
	const int pending = sys->xn_pending;
	__shared__ int keys[SEPK_SORT_KEYS];
	for (long c = blockIdx.x; c < ncell; c += gridDim.x) {
		const int s = start[c], e = start[c + 1];
		for (int i0 = s; i0 < e; i0 += SEPK_BLOCK) {
			const int i = i0 + (int)threadIdx.x;
			const long o = i < e ? sepk_at(order, (unsigned)i) : 0;
			const int key = i < e ? sepk_at(src.orig, (unsigned)o) : 0;
			int rank = 0;
			for (int b = s; b < e; b += SEPK_SORT_KEYS) {
				const int m = min(SEPK_SORT_KEYS, e - b);
				__syncthreads(); // the previous keys are no longer read
				for (int q = threadIdx.x; q < m; q += SEPK_BLOCK) {
					const int x = b + q; // a thread's own member: its key
					keys[q] = x == i ? key
							 : sepk_at(src.orig, (unsigned)sepk_at(order, (unsigned)x));
				}
				__syncthreads();
#pragma unroll 4
				for (int jj = 0; jj < m; jj++)
					rank += keys[jj] < key;
			}
			if (i >= e)
				continue;
			const long t = s + rank;
			sepk_move_atom(src, o, dst, t, npad, pending);
			sepk_at(iperm, (unsigned)key) = (int)t;
			if (has_partners)
				sepk_copy_partners(src, dst, o, t, npad);
		}
	}
}

// Binning, scan, sort and permutation in one launch, for systems of up to
// SEPK_ORDER_ATOMS atoms and SEPK_ORDER_CELLS cells: every workgroup bins all
// atoms and scans the cell counts in its LDS, and permutes the cells of its
// own share, so that no workgroup waits for another and the three launches of
// a larger system (k_bin, k_scan_scatter, k_sort_permute) are one.  What it saves
// is two launches in every step, rebuilt or not, and the chain of three kernels'
// memory round trips in a rebuild; what it costs is the reading of every
// position in each of 64 workgroups, 31 us a rebuild at 27000 atoms.  Per step,
// which rebuilds when the flag is set (three launches -> one, us, FP64 LJ liquid at
// T = 1): 4000 atoms 22.4 -> 19.0, 16000 24.0 -> 21.3, 27000 29.0 -> 27.5, 32000
// 30.3 -> 29.0; with a rebuild every fifth step (T = 2) 27000 32.0 -> 31.4, 32000
// 33.7 -> 33.8; water 6000 98 -> 96.1.
// A call that is sure to rebuild (synchronised, brute force) pays the cost each
// time and saves the launches once: 8000 atoms 44.8 -> 41.6, 14000 49.9 -> 50.4,
// 16000 51.5 -> 53.3, 24000 55.7 -> 62.2, 32000 65.3 -> 77.3, so there the line is
// SEPK_ORDER_BUILD; except where the cells hold more than SEPK_ORDER_FULL atoms on
// average, whose ranking by 256 threads a cell takes longer than by 1024 (32768
// atoms in 27 cells 1350 -> 1284, in one 99.3 -> 52.6 ms).
#define SEPK_ORDER_ATOMS 32768
#define SEPK_ORDER_BUILD 16384
#define SEPK_ORDER_FULL 1024
#define SEPK_ORDER_CELLS 4096
#define SEPK_ORDER_GRID 64
#define SEPK_ORDER_KEYS 2048

// Whether q = p / l, from the product with 1 / l, is far enough from a whole
// number and inside the grid for its truncation to be that of the division.
__device__ __forceinline__ bool sepk_plain_cell(double q, int n, int &c)
{
	c = (int)q;
	const double r = q - (double)c;
	return q > 1e-6 && r > 1e-9 && r < 1.0 - 1e-9 && c < n;
}

template <int NMAX>
__global__ __launch_bounds__(1024) void k_order(sepk_state src, sepk_state dst, long nl, long npad,
						sepdev_grid g, int ncell, int *start, int *iperm,
						sepdev_sys *sys, int conditional, int has_partners)
{
	if (conditional && sys->neighb_flag == 0)
		return;
	__shared__ unsigned short cid[NMAX], mem[NMAX];
	__shared__ int sstart[SEPK_ORDER_CELLS + 4], keys[SEPK_ORDER_KEYS];
	__shared__ int fill[SEPK_ORDER_CELLS / SEPK_ORDER_GRID + 1];
	__shared__ int wsum[16], failed, bad;
	const int n = (int)nl, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
	const int pending = sys->xn_pending;
	for (int c = tid; c < ncell; c += 1024)
		sstart[c] = 0;
	// an error set while this runs is an atom outside the grid, which every
	// workgroup finds by itself; one set before is looked at once
	if (tid == 0) {
		const bool err = sys->error != 0;
		failed = bad = err;
		// the build's atomic maximum starts here; after an overflow it
		// stays for the host, which grows the list by it
		if (blockIdx.x == 0 && !err)
			sys->max_full = 0;
	}
	__syncthreads();
	const double il0 = 1.0 / g.l[0], il1 = 1.0 / g.l[1], il2 = 1.0 / g.l[2];
	// whole waves iterate together
	for (int t0 = 0; t0 < n && !failed; t0 += 1024) {
		const int t = t0 + tid;
		int c = -1;
		if (t < n) {
			const sepk_pos p = sepk_at(src.pos, (unsigned)t);
			int cx, cy, cz;
			const bool fx = sepk_plain_cell(p.x * il0, g.n[0], cx),
				   fy = sepk_plain_cell(p.y * il1, g.n[1], cy),
				   fz = sepk_plain_cell(p.z * il2, g.n[2], cz);
			c = cx + (cy + cz * g.n[1]) * g.n[0];
			if (!(fx && fy && fz)) {
				c = (int)sepk_cell_of(p, g);
				if (c < 0) {
					sepk_set_error(sys, SEP_GPU_ECELL);
					bad = 1;
					c = 0;
				}
				// an atom outside [0, n*l) on some axis, as in k_bin
				const double q[3] = {p.x / g.l[0], p.y / g.l[1], p.z / g.l[2]};
				if (!(q[0] >= 0.0 && q[0] < g.n[0] && q[1] >= 0.0 && q[1] < g.n[1] &&
				      q[2] >= 0.0 && q[2] < g.n[2]))
					sys->unclean = 1;
			}
			cid[t] = (unsigned short)c;
		}
		// one LDS atomic per run of lanes in one cell (the atoms arrive in
		// the last build's cell order)
		const int before = __shfl_up(c, 1, 64);
		const unsigned long long head = __ballot(lane == 0 || c != before);
		if (c >= 0 && (head >> lane & 1ull)) {
			const unsigned long long rest = lane == 63 ? 0ull : head >> (lane + 1);
			atomicAdd(&sstart[c], rest ? __builtin_ctzll(rest) + 1 : min(64 - lane, n - t));
		}
	}
	__syncthreads();
	const bool frozen = bad != 0;
	if (blockIdx.x == 0 && tid == 0)
		sys->frozen = frozen;
	if (frozen)
		return; // the build skips as well
	// exclusive scan of the counts, four cells a thread
	{
		static_assert(SEPK_ORDER_CELLS == 4 * 1024, "one pass");
		int v[4], tot = 0;
#pragma unroll
		for (int k = 0; k < 4; k++) {
			v[k] = 4 * tid + k < ncell ? sstart[4 * tid + k] : 0;
			tot += v[k];
		}
		int x = tot; // inclusive wave scan of the thread totals
		for (int o = 1; o < 64; o <<= 1) {
			const int y = __shfl_up(x, o, 64);
			if (lane >= o)
				x += y;
		}
		if (lane == 63)
			wsum[wid] = x;
		__syncthreads();
		int off = x - tot;
		for (int w = 0; w < wid; w++)
			off += wsum[w];
#pragma unroll
		for (int k = 0; k < 4; k++) {
			if (4 * tid + k < ncell)
				sstart[4 * tid + k] = off;
			off += v[k];
		}
		if (tid == 0)
			sstart[ncell] = n;
	}
	// this workgroup's cells [c0, c1): their members, in any order
	const int per = (ncell + (int)gridDim.x - 1) / (int)gridDim.x;
	const int c0 = min((int)blockIdx.x * per, ncell), c1 = min(c0 + per, ncell);
	for (int k = tid; k < per; k += 1024)
		fill[k] = 0;
	__syncthreads();
	if (c0 == c1)
		return;
	const int base = sstart[c0], m = sstart[c1] - base;
	for (int c = c0 + tid; c < c1 + (c1 == ncell ? 1 : 0); c += 1024)
		start[c] = sstart[c];
	for (int t = tid; t < n; t += 1024) {
		const int c = cid[t];
		if (c >= c0 && c < c1)
			mem[sstart[c] - base + atomicAdd(&fill[c - c0], 1)] = (unsigned short)t;
	}
	__syncthreads();
	// Each member ranked by its original index within its cell and moved.  The
	// keys are in LDS, SEPK_ORDER_KEYS at a time where the share holds more (a
	// few very full cells; all atoms in one, where the box has no three cells
	// an axis).  A pair call that rebuilds, 10000 atoms in one cell: 5.2 ms;
	// 11.9 with the keys of such a share read from memory for every member,
	// 9.6 with the three launches; 1000 atoms: 82 us, 108 with the ranking not
	// unrolled, 135 with the three launches.
	for (int i0 = 0; i0 < m; i0 += 1024) {
		const int i = i0 + tid;
		const bool act = i < m;
		const int o = act ? mem[i] : 0, c = act ? cid[o] : c0;
		const int a = sstart[c] - base, b = act ? sstart[c + 1] - base : a;
		const int key = act ? sepk_at(src.orig, (unsigned)o) : 0;
		int rank = 0;
		for (int k0 = 0; k0 < m; k0 += SEPK_ORDER_KEYS) {
			const int kn = min(m - k0, SEPK_ORDER_KEYS);
			if (i0 == 0 || m > SEPK_ORDER_KEYS) { // the same for the workgroup
				__syncthreads(); // the previous keys are no longer read
				for (int q = tid; q < kn; q += 1024)
					keys[q] = k0 + q == i ? key : sepk_at(src.orig, (unsigned)mem[k0 + q]);
				__syncthreads();
			}
			const int e = min(b - k0, kn);
#pragma unroll 4
			for (int j = max(a - k0, 0); j < e; j++)
				rank += keys[j] < key;
		}
		if (!act)
			continue;
		const int t = sstart[c] + rank;
		sepk_move_atom(src, o, dst, t, npad, pending);
		sepk_at(iperm, (unsigned)key) = t;
		if (has_partners)
			sepk_copy_partners(src, dst, o, t, npad);
	}
}

// Partner scan of source/sepprfrc.c:703-731: stops at the first -1 in
// either atom's array.  Partner values are original indices.
__device__ __forceinline__ int sepk_share(const int *P, long npad, long ti, long tj,
					  int base, int cap, int oi, int oj)
{
	for (int k = 0; k < cap; k++) {
		const int a = P[(base + k) * npad + ti], b = P[(base + k) * npad + tj];
		if (a == -1 || b == -1)
			return 0;
		if (a == oj || b == oi)
			return 1;
	}
	return 0;
}

// Copies atom t of the permuted spare state back to the current buffers,
// whose addresses every other kernel (and a captured graph) holds.
__device__ __forceinline__ void sepk_copy_home(const sepk_state &src, const sepk_state &dst,
					       long t, long npad, int has_partners)
{
	sepk_move_atom(src, t, dst, t, npad, false);
	if (has_partners)
		sepk_copy_partners(src, dst, t, t, npad);
}

// Lists come out in stencil-offset order and, within a cell, in device order;
// entry k of atom t goes to slot sepk_entry(k, t, npad).  Cells (and the
// slices of their atoms) are split into one contiguous range per XCD, walked
// with a stride of the range's workgroups or waves.
//
// Quantized build (k_build_q): a cubic box of at least 3 cells an axis with
// every atom inside it, the usual case.  Every coordinate is held as
// floor(x * 65536 / L) mod 2^16 (the upper half of the pair kernels'
// quantized record), x and y in one word and z in the low half of another.  A
// packed 16-bit subtraction gives the minimum-image difference in units of
// u = L / 65536, each component within one unit of the exact one, and two
// saturating packed dot products its square r2q.  With R = r_list / u the
// distance is below r_list - 0.26 u when r2q < floor((R - 2)^2) and above
// r_list + 0.26 u when r2q > ceil((R + 2)^2) (sqrt(3) < 1.74), far outside
// the rounding of the FP64 r2 (a component near half the box, whose sign may
// go either way, has |d| >= L/2 - u > 1.4 r_list); only candidates between
// the two bounds (a shell about 4 u thick: a few in ten thousand) take the
// FP64 test, the reference's own, so the accepted set is the FP64 test's
// exactly.
//
// FP64 build (k_build): every other box, each candidate by the reference's
// test.  SHIFT: with at least 5 cells on every axis and every atom inside
// its own cell, |x_i - x_j| < 2l <= 0.4 L for a target cell reached without
// crossing the box and > L - 2l >= 0.6 L for one reached across it, so the
// reference's single-image wrap (subtract or add L exactly when |d| > L/2) is
// the constant shift of the target cell; d + shift rounds exactly like its
// d - L / d + L, and d + 0 is d.  Otherwise the wrap is evaluated per
// candidate.
#define SEPK_BT 256      // threads of a build workgroup (4 waves)
#define SEPK_BCHUNK 384  // candidates staged at a time, FP64 build
#define SEPK_BHOME 64    // home atoms at a time
// rounds of 64 candidates that a lane holds, quantized build (fewer with the
// same-molecule rule, whose molecule numbers take registers and LDS too)
#define SEPK_QROUNDS(EXCL) ((EXCL) == 3 ? 4 : 5)
#define SEPK_BGRID 1792  // build workgroups at most (a multiple of 8)
#define SEPK_QSLICE 11   // home atoms of a wave, quantized build, in large systems
static_assert(SEPK_BCHUNK % 64 == 0, "candidates are tested 64 at a time");
static_assert(SEPK_BHOME <= 64 * (SEPK_BT / 64), "a wave's home atoms fit its lanes");

struct sepk_build_lds {
	double cx[SEPK_BCHUNK], cy[SEPK_BCHUNK], cz[SEPK_BCHUNK];
	int cj[SEPK_BCHUNK], cm[SEPK_BCHUNK];
	unsigned char co[SEPK_BCHUNK];
	double hx[SEPK_BHOME], hy[SEPK_BHOME], hz[SEPK_BHOME];
	int horig[SEPK_BHOME], hmol[SEPK_BHOME];
	int segjs[SEPDEV_MAX_OFF], segpre[SEPDEV_MAX_OFF + 1];
	int segrule[SEPDEV_MAX_OFF]; // rule when the target is the home cell, else -1
	double segsh[SEPDEV_MAX_OFF][3];
	int hs, h, anyshift;
};

// Bounds of the quantized test, in units of L / 2^16, and of the second one
// for the candidates between them, in units of L / 2^21.
struct sepk_qtest {
	double lo2f, hi2f;
	int lo2, hi2;
	double icell[2], islice; // reciprocals: cells along x and y, slices a cell
};

// Whether the quantized build serves a grid (once its binning finds every
// atom inside the box): three cells of at least r_list an axis, so that
// R <= 21846 and both bounds are below 2^30 (SEPK_QNONE).
static bool sepk_qtest_of(const sepdev_grid &g, sepk_qtest &q)
{
	const double R = sqrt(g.rlist2) * (65536.0 / g.L[0]), Rf = 32.0 * R;
	const bool on = g.n[0] >= 3 && g.n[1] >= 3 && g.n[2] >= 3 && g.noff == 27 &&
			g.L[0] == g.L[1] && g.L[1] == g.L[2] && R > 2.0 && R < 21900.0;
	q.lo2 = on ? (int)floor((R - 2.0) * (R - 2.0)) : 0;
	q.hi2 = on ? (int)ceil((R + 2.0) * (R + 2.0)) : 0;
	q.lo2f = floor((Rf - 2.0) * (Rf - 2.0));
	q.hi2f = ceil((Rf + 2.0) * (Rf + 2.0));
	q.icell[0] = 1.0 / g.n[0];
	q.icell[1] = 1.0 / g.n[1];
	return on;
}

// The build's form of a quantized record (sepk_quant): the upper 21 bits of
// each coordinate, of which the upper 16 are x and y in the low and high
// halves of .x and z in the low half of .y, and the lower 5 of x, y and z in
// bits 16..30 of .y.
__device__ __forceinline__ uint2 sepk_quant21(const int4 &q)
{
	const unsigned lx = (unsigned)q.x >> 11 & 31u, ly = (unsigned)q.y >> 11 & 31u,
		       lz = (unsigned)q.z >> 11 & 31u;
	return make_uint2((unsigned)q.x >> 16 | ((unsigned)q.y & 0xffff0000u),
			  (unsigned)q.z >> 16 | ((lz << 5 | ly) << 5 | lx) << 16);
}

// The 21-bit coordinates of such a record in the upper bits of three words.
__device__ __forceinline__ void sepk_words21(uint2 q, unsigned &x, unsigned &y, unsigned &z)
{
	x = q.x << 16 | (q.y >> 5 & 0xf800u);
	y = (q.x & 0xffff0000u) | (q.y >> 10 & 0xf800u);
	z = q.y << 16 | (q.y >> 15 & 0xf800u);
}

typedef short sepk_short2 __attribute__((ext_vector_type(2)));

// Squared quantized minimum-image distance (16 bits a coordinate, .y without
// the lower bits), saturated at 2^31 - 1.
__device__ __forceinline__ int sepk_r2q(uint2 a, uint2 b)
{
	const sepk_short2 dxy =
		__builtin_bit_cast(sepk_short2, a.x) - __builtin_bit_cast(sepk_short2, b.x);
	const sepk_short2 dz =
		__builtin_bit_cast(sepk_short2, a.y) - __builtin_bit_cast(sepk_short2, b.y);
	return __builtin_amdgcn_sdot2(dz, dz, __builtin_amdgcn_sdot2(dxy, dxy, 0, true), true);
}

// Lane `lane` of v (a wave-uniform lane number) becomes val, whatever the
// execution mask.
__device__ __forceinline__ void sepk_writelane(int &v, int val, int lane)
{
	asm volatile("v_writelane_b32 %0, %1, %2" : "+v"(v) : "s"(val), "{m0}"(lane));
}

// SEP_EXCL_BONDED: whether the pair (t, j) stays in the list.
__device__ __forceinline__ bool sepk_keep_bonded(const sepk_state &s, const sepdev_grid &g, long t,
						 int j, long npad)
{
	const int oi = s.orig[t], oj = s.orig[j];
	int sh = sepk_share(s.partners, npad, t, j, 0, 10, oi, oj);
	if (g.bonded_all)
		sh += sepk_share(s.partners, npad, t, j, 10, 10, oi, oj) +
		      sepk_share(s.partners, npad, t, j, 20, 20, oi, oj);
	// rule 2 is the Coulomb brute-force test of source/sepcoulomb.c:44, which
	// excludes only when exactly one kind of partnership holds
	return g.bonded_all == 2 ? sh != 1 : sh == 0;
}

// Number of set bits of m below this lane.
__device__ __forceinline__ int sepk_rank(unsigned long long m)
{
	return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
					      __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// Orders a wave's accesses to its own LDS row (the hardware executes them in
// order; this keeps the compiler to it).
__device__ __forceinline__ void sepk_wave_lds()
{
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The candidates in `near` (record cq, index j) that are within the list
// cutoff of atom t (record q): by the 21-bit records, and the few that lie
// within two of their units of the cutoff by the reference's FP64 test
// (there the image by rint is the reference's single-image wrap bit for bit,
// sepk_wrap_fast).  One atom in three has a candidate in `near`, one in a
// hundred needs positions from memory: a load here waits for the list
// stores in flight as well.
__device__ __forceinline__ unsigned long long sepk_near_test(const sepk_state &s,
							     const sepdev_grid &g,
							     const sepk_qtest &qt,
							     unsigned long long near, uint2 q,
							     const uint2 *cq, int t, int j)
{
	unsigned ax, ay, az, bx, by, bz;
	sepk_words21(q, ax, ay, az);
	sepk_words21(*cq, bx, by, bz);
	const double ux = (double)((int)(ax - bx) >> 11), uy = (double)((int)(ay - by) >> 11),
		     uz = (double)((int)(az - bz) >> 11);
	const double u2 = fma(ux, ux, fma(uy, uy, uz * uz)); // exact
	unsigned long long in = __ballot(u2 < qt.lo2f) & near;
	const unsigned long long edge = __ballot(u2 <= qt.hi2f) & near & ~in;
	if (edge) {
		bool ok = false;
		if (__builtin_amdgcn_inverse_ballot_w64(edge)) {
			// the address is formed here, not held through the caller's loop
			asm volatile("" : "+v"(j));
			const sepk_pos pi = sepk_at(s.pos, (unsigned)t);
			const sepk_pos pj = sepk_at(s.pos, (unsigned)j);
			const double L = g.L[0], iL = 1.0 / L;
			const double dx = sepk_wrap_fast(pi.x - pj.x, L, iL);
			const double dy = sepk_wrap_fast(pi.y - pj.y, L, iL);
			const double dz = sepk_wrap_fast(pi.z - pj.z, L, iL);
			ok = dx * dx + dy * dy + dz * dz < g.rlist2;
		}
		in |= __ballot(ok);
	}
	return in;
}

// A packed 16-bit difference held within 16 bits.
__device__ __forceinline__ sepk_short2 sepk_sub_sat(sepk_short2 a, sepk_short2 b)
{
	return __builtin_elementwise_sub_sat(a, b);
}

// One wave's LDS of the quantized build.
template <int EXCL>
struct sepk_qwave {
	static constexpr int NR = SEPK_QROUNDS(EXCL), CAP = 64 * NR;
	uint2 cq[CAP];                  // its candidates
	int cj[CAP], cm[EXCL == 3 ? CAP : 1];
	// an atom's accepted ones, the phantom after them
	__align__(16) int row[CAP + SEPK_PAD];
};

// Quantized build: the wave's home atoms tb + i, i the bits of mine (lane i
// holds the record and molecule of atom tb + i) against the nf candidates in
// its LDS, appending the accepted ones to the lists.  Lane i of cnt holds the
// list length of atom tb + i; entries at or beyond cap are counted but not stored.
// last: the entries are padded with the phantom slot to a multiple of
// SEPK_PAD.
// A lane holds one candidate of every round in registers for all of the
// atoms; for one atom all rounds are tested (one ballot a round), the passing
// lanes put their candidate into the LDS row at the number of those before
// them (mbcnt), and the row goes to the list, four slots a lane.
template <int EXCL>
__device__ __forceinline__ void sepk_build_pass(
	sepk_qwave<EXCL> &W, const sepk_state &s, const sepdev_grid &g, const sepk_qtest &qt,
	int nf, int tb, unsigned long long mine, uint2 hq, int hm, long npad, int cap, int phantom, bool last,
	int *nbr, int &cnt)
{
	constexpr int NR = sepk_qwave<EXCL>::NR;
	const int lane = threadIdx.x & 63;
	const int nr = (nf + 63) / 64;
	// this lane's four consecutive slots of 256, and the first of the four
	// entries (SEPK_SUB apart) that they hold
	const size_t lslot = (size_t)(lane / SEPK_SUB) * npad * SEPK_PAD + lane % SEPK_SUB * SEPK_BATCH;
	const int lent = lane / SEPK_SUB * SEPK_PAD + lane % SEPK_SUB;
	static_assert(SEPK_SUB == 4 && SEPK_BATCH == 4, "four slots a lane");
	uint2 cq[NR];
	int cj[NR], cm[NR];
#pragma unroll
	for (int r = 0; r < NR; r++)
		if (r < nr) {
			const int f = 64 * r + lane;
			cq[r] = W.cq[f];
			cq[r].y &= 0xffffu;
			cj[r] = W.cj[f];
			if (EXCL == 3)
				cm[r] = W.cm[f];
		}
	// the candidates of the last round
	const unsigned long long some = nf & 63 ? ~(~0ull << (nf & 63)) : ~0ull;
	for (; mine; mine &= mine - 1ull) {
		const int i = __builtin_ctzll(mine), t = tb + i;
		const uint2 q = make_uint2((unsigned)__builtin_amdgcn_readlane((int)hq.x, i),
					   (unsigned)__builtin_amdgcn_readlane((int)hq.y, i));
		const int mi = EXCL == 3 ? __builtin_amdgcn_readlane(hm, i) : -1;
		int m = 0; // accepted in this pass
#pragma unroll
		for (int r = 0; r < NR; r++) {
			if (r >= nr)
				continue;
			const int r2q = sepk_r2q(make_uint2(q.x, q.y & 0xffffu), cq[r]);
			// the lanes that hold a candidate: the others' records and
			// indices are left over and must reach nothing below
			const unsigned long long held = r == nr - 1 ? some : ~0ull;
			unsigned long long take = __ballot(r2q < qt.lo2) & held;
			const unsigned long long near = __ballot(r2q <= qt.hi2) & held & ~take;
			if (near)
				take |= sepk_near_test(s, g, qt, near, q, W.cq + 64 * r + lane, t, cj[r]);
			take &= __ballot(cj[r] != t); // not the atom itself
			if (EXCL == 3) {
				if (mi != -1)
					take &= __ballot(cm[r] != mi);
			}
			if (__builtin_amdgcn_inverse_ballot_w64(take))
				(W.row + m)[sepk_rank(take)] = cj[r];
			m += __popcll(take);
		}
		sepk_wave_lds();
		if (EXCL == 2) {
			// drop the bonded ones from the row, in place and in order
			int keep = 0;
			for (int b = 0; b < m; b += 64) {
				const int j = W.row[min(b + lane, m - 1)];
				const bool ok = b + lane < m && sepk_keep_bonded(s, g, t, j, npad);
				const unsigned long long in = __ballot(ok);
				sepk_wave_lds();
				if (ok)
					(W.row + keep)[sepk_rank(in)] = j;
				keep += __popcll(in);
				sepk_wave_lds();
			}
			m = keep;
		}
		const int e0 = __builtin_amdgcn_readlane(cnt, i), e1 = e0 + m;
		if (last && e0 == 0) {
			// the whole list at once (up to 256 entries a store)
			if (lane < SEPK_PAD)
				W.row[m + lane] = phantom;
			sepk_wave_lds();
			int *list = nbr + (size_t)t * SEPK_PAD + lslot;
			const int end = min(m, cap);
			for (int b = lent; b < end + lane % SEPK_SUB; b += 64 * SEPK_BATCH) {
				const int *w = W.row + b;
				*(int4 *)list = make_int4(w[0], w[SEPK_SUB], w[2 * SEPK_SUB], w[3 * SEPK_SUB]);
				list += 16 * SEPK_PAD * npad;
			}
		} else {
			const int end = min(last ? (e1 + SEPK_PAD - 1) / SEPK_PAD * SEPK_PAD : e1, cap);
			for (int e = e0 + lane; e < end; e += 64)
				nbr[sepk_entry(e, t, npad)] = e < e1 ? W.row[e - e0] : phantom;
		}
		sepk_wave_lds();
		sepk_writelane(cnt, e1, i);
	}
}

// a / b for 0 <= a < 2^31 and b > 0 from ib = 1 / b: (a + 1/2) / b is at
// least 1 / (2 b) from a whole number, the product's error below 2^-20 / b.
__device__ __forceinline__ int sepk_quotient(int a, double ib)
{
	return (int)(((double)a + 0.5) * ib);
}

// Segment of lane l < 18 of cell c's stencil: cells next to each other along
// x hold consecutive atoms, so the three of a row are one segment, or two
// where the box ends between them (lanes 2 r and 2 r + 1 take row r, in
// stencil order); lane 18: the cell itself.  js, len: first atom, atoms.
__device__ __forceinline__ void sepk_build_segment(const sepdev_grid &g, const sepk_qtest &qt,
						   int c, const int *start, int &js, int &len)
{
	const int lane = threadIdx.x & 63;
	js = len = 0;
	if (lane > 18)
		return;
	const int n0 = g.n[0], n1 = g.n[1], n2 = g.n[2];
	const int zy = sepk_quotient(c, qt.icell[0]), cz = sepk_quotient(zy, qt.icell[1]);
	const int cx = c - zy * n0, cy = zy - cz * n1;
	int row = c, xa = 0, xb = 0;
	if (lane < 18) {
		const int r = lane >> 1;
		int y = cy + r % 3 - 1, z = cz + r / 3 - 1;
		y += y < 0 ? n1 : y >= n1 ? -n1 : 0;
		z += z < 0 ? n2 : z >= n2 ? -n2 : 0;
		row = (y + z * n1) * n0;
		xa = cx - 1; // cells xa .. xb
		xb = cx + 1;
		if (xa < 0 || xb >= n0) {
			const bool two = xb >= n0; // two cells before the end
			xa = lane & 1 ? 0 : two ? n0 - 2 : n0 - 1;
			xb = lane & 1 ? (two ? 0 : 1) : n0 - 1;
		} else if (lane & 1) {
			return;
		}
	}
	js = start[row + xa];
	len = start[row + xb + 1] - js;
}

// Quantized build of home atoms tb + i, i the bits of mine, when some atom
// lies outside the box: the same segments, the reference's FP64 test of every candidate,
// the accepted ones stored as they come (rare: an atom at x == L exactly, or
// a starting configuration that reaches outside).
template <int EXCL>
__device__ void sepk_build_outside(int js, int len, const sepk_state &s, const sepdev_grid &g,
				   int tb, unsigned long long mine, long npad, int cap,
				   int phantom, int *nbr, int &cnt)
{
	const int lane = threadIdx.x & 63;
	for (; mine; mine &= mine - 1ull) {
		const int t = tb + __builtin_ctzll(mine);
		const sepk_pos pi = sepk_at(s.pos, (unsigned)t);
		const int mi = EXCL == 3 ? sepk_at(s.mol, (unsigned)t) : -1;
		int m = 0;
		for (int o = 0; o < 18; o++) {
			const int n = __builtin_amdgcn_readlane(len, o);
			for (int q0 = 0; q0 < n; q0 += 64) {
				const int q = q0 + lane;
				const int j = __builtin_amdgcn_readlane(js, o) + min(q, n - 1);
				const sepk_pos pj = sepk_at(s.pos, (unsigned)j);
				const double dx = sepk_wrap(pi.x - pj.x, g.L[0]);
				const double dy = sepk_wrap(pi.y - pj.y, g.L[1]);
				const double dz = sepk_wrap(pi.z - pj.z, g.L[2]);
				bool in = q < n && j != t && dx * dx + dy * dy + dz * dz < g.rlist2;
				if (EXCL == 3 && mi != -1)
					in = in && sepk_at(s.mol, (unsigned)j) != mi;
				if (EXCL == 2 && in)
					in = sepk_keep_bonded(s, g, t, j, npad);
				const unsigned long long take = __ballot(in);
				const int e = m + sepk_rank(take);
				if (in && e < cap)
					nbr[sepk_entry(e, t, npad)] = j;
				m += __popcll(take);
			}
		}
		const int pad = min((m + SEPK_PAD - 1) / SEPK_PAD * SEPK_PAD, cap);
		if (m + lane < pad)
			nbr[sepk_entry(m + lane, t, npad)] = phantom;
		sepk_writelane(cnt, m, t - tb);
	}
}

// The wave's candidates for home atoms tb + i, i the bits of mine (lane i
// holds the record of atom tb + i): those of the stencil's T atoms that come
// within the list cutoff of the atoms' bounding box (in order, through the
// wave's LDS), sepk_qwave::CAP at a time.
// Segment o of the stencil (the bits of used) starts at candidate pre of the
// wave's T, its atom k at k + off: lane o holds pre and off.
template <int EXCL>
__device__ __forceinline__ void sepk_build_home(
	sepk_qwave<EXCL> &W, unsigned used, int pre, int off, int T, const sepk_state &s,
	const sepdev_grid &g, const sepk_qtest &qt, int tb, unsigned long long mine, uint2 hq,
	int hm, long npad, int cap, int phantom, int *nbr, int &cnt)
{
	constexpr int NR = sepk_qwave<EXCL>::NR, CAP = sepk_qwave<EXCL>::CAP;
	const int lane = threadIdx.x & 63;
	// the box of the atoms: centre and half edges (rounded up)
	const sepk_short2 zero = {0, 0};
	sepk_short2 cxy, hxy, cz, hz;
	{
		typedef unsigned short us2 __attribute__((ext_vector_type(2)));
		// the other lanes stand in for the first of the atoms
		const int one = __builtin_ctzll(mine);
		const bool in = mine >> lane & 1ull;
		const unsigned x1 = (unsigned)__builtin_amdgcn_readlane((int)hq.x, one);
		const unsigned y1 = (unsigned)__builtin_amdgcn_readlane((int)hq.y, one);
		us2 axy = __builtin_bit_cast(us2, in ? hq.x : x1), bxy = axy;
		us2 az = __builtin_bit_cast(us2, (in ? hq.y : y1) & 0xffffu), bz = az;
		for (int o = 32; o > 0; o >>= 1) {
			const unsigned p = __shfl_xor(__builtin_bit_cast(unsigned, axy), o, 64);
			const unsigned q = __shfl_xor(__builtin_bit_cast(unsigned, bxy), o, 64);
			const unsigned u = __shfl_xor(__builtin_bit_cast(unsigned, az), o, 64);
			const unsigned v = __shfl_xor(__builtin_bit_cast(unsigned, bz), o, 64);
			axy = __builtin_elementwise_min(axy, __builtin_bit_cast(us2, p));
			bxy = __builtin_elementwise_max(bxy, __builtin_bit_cast(us2, q));
			az = __builtin_elementwise_min(az, __builtin_bit_cast(us2, u));
			bz = __builtin_elementwise_max(bz, __builtin_bit_cast(us2, v));
		}
		const unsigned a = __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, axy));
		const unsigned b = __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, bxy));
		const int a2 = __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, az));
		const int b2 = __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, bz));
		const int a0 = (int)(a & 0xffffu), a1 = (int)(a >> 16);
		const int b0 = (int)(b & 0xffffu), b1 = (int)(b >> 16);
		cxy = sepk_short2{(short)((a0 + b0) >> 1), (short)((a1 + b1) >> 1)};
		hxy = sepk_short2{(short)min((b0 - a0 + 1) >> 1, 32767), (short)min((b1 - a1 + 1) >> 1, 32767)};
		cz = sepk_short2{(short)((a2 + b2) >> 1), 0};
		hz = sepk_short2{(short)min((b2 - a2 + 1) >> 1, 32767), 0};
	}
	int ko = 0, kn = 0; // this segment's offset, the next one's first candidate
	int nf = 0;
	for (int k0 = 0;; k0 += CAP) {
		const bool end = k0 >= T;
		int jq[NR], mq[NR], nb = 0;
		uint2 cq[NR];
		unsigned long long in[NR];
		if (!end) {
			// the atom of every lane's candidate: the segment is followed
			// along the rounds, the lanes past its end moved to the next
#pragma unroll
			for (int r = 0; r < NR; r++) {
				const int k = min(k0 + 64 * r + lane, T - 1);
				jq[r] = k + ko;
				while (kn <= k0 + 64 * r + 63) { // the next segment starts in this round
					const int o = __builtin_ctz(used);
					ko = __builtin_amdgcn_readlane(off, o);
					jq[r] = k >= kn ? k + ko : jq[r];
					used &= used - 1u;
					kn = used ? __builtin_amdgcn_readlane(pre, __builtin_ctz(used)) : INT_MAX;
				}
			}
			int4 pq[NR];
#pragma unroll
			for (int r = 0; r < NR; r++) {
				pq[r] = sepk_at(s.qpos, (unsigned)jq[r]);
				if (EXCL == 3)
					mq[r] = sepk_at(s.mol, (unsigned)jq[r]);
			}
#pragma unroll
			for (int r = 0; r < NR; r++) {
				// the distance to the box is no larger than to any atom in it,
				// in the same units
				cq[r] = sepk_quant21(pq[r]);
				sepk_short2 dxy = __builtin_bit_cast(sepk_short2, cq[r].x) - cxy;
				sepk_short2 dz = __builtin_bit_cast(sepk_short2, (unsigned)pq[r].z >> 16) - cz;
				dxy = __builtin_elementwise_max(dxy, sepk_sub_sat(zero, dxy));
				dz = __builtin_elementwise_max(dz, sepk_sub_sat(zero, dz));
				dxy = __builtin_elementwise_max(sepk_sub_sat(dxy, hxy), zero);
				dz = __builtin_elementwise_max(sepk_sub_sat(dz, hz), zero);
				const int d2 = __builtin_amdgcn_sdot2(
					dz, dz, __builtin_amdgcn_sdot2(dxy, dxy, 0, true), true);
				in[r] = __ballot(d2 <= qt.hi2 && k0 + 64 * r + lane < T);
				nb += __popcll(in[r]);
			}
		}
		if (end || nf + nb > CAP) {
			sepk_wave_lds();
			sepk_build_pass<EXCL>(W, s, g, qt, nf, tb, mine, hq, hm, npad, cap, phantom, end,
					      nbr, cnt);
			if (end)
				return;
			nf = 0;
		}
#pragma unroll
		for (int r = 0; r < NR; r++) {
			if (__builtin_amdgcn_inverse_ballot_w64(in[r])) {
				const int f = nf + sepk_rank(in[r]);
				W.cq[f] = cq[r];
				W.cj[f] = jq[r];
				if (EXCL == 3)
					W.cm[f] = mq[r];
			}
			nf += __popcll(in[r]);
		}
	}
}

// FP64 build, one round: the 64 staged candidates [q0, q0 + 64) of a chunk
// of kn against the wave's home atoms i = wid, wid + 4, ... < hn, storing the
// accepted ones to their lists, each at the atom's length so far plus its
// rank among the passing lanes.  cnt and cap as above.
// SH: some stencil target of the cell lies across the box (shift adds).
template <bool SHIFT, bool SH, int EXCL>
__device__ __forceinline__ void sepk_build_round(
	sepk_build_lds &L, const sepk_state &s, const sepdev_grid &g, int q0, int kn, long tbase,
	int hn, long npad, int cap, int *nbr, int &cnt)
{
	const int lane = threadIdx.x & 63;
	const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // wave-uniform
	const int q = min(q0 + lane, kn - 1);
	// lanes past the staged candidates take a bound that no distance meets
	const bool valid = lane < kn - q0;
	const int j = L.cj[q];
	const int o = L.co[q];
	const int rule = L.segrule[o];
	const int mj = EXCL == 3 ? L.cm[q] : -1;
	// lanes whose candidate is in the home cell (SHIFT: through offset 0,
	// whose rule is NE)
	const unsigned long long home = __ballot(rule >= 0);
	// original index of a home-cell candidate, for the GT / LT rules
	const int oj = !SHIFT && rule >= SEPDEV_RULE_GT ? s.orig[j] : 0;
	const double px = L.cx[q], py = L.cy[q], pz = L.cz[q];
	const double rl2 = valid ? g.rlist2 : -1.0;
	const int jrel = j - (int)tbase; // the home atom i's own candidate has jrel == i
	double sx = 0.0, sy = 0.0, sz = 0.0;
	if (SH) {
		sx = L.segsh[o][0];
		sy = L.segsh[o][1];
		sz = L.segsh[o][2];
	}
	int kk = 0;
	for (int i = wid; i < hn; i += SEPK_BT / 64, kk++) {
		const long t = tbase + i;
		const int t32 = (int)t;
		double dx, dy, dz;
		if (SHIFT) {
			dx = L.hx[i] - px;
			dy = L.hy[i] - py;
			dz = L.hz[i] - pz;
			if (SH) {
				dx += sx;
				dy += sy;
				dz += sz;
			}
		} else {
			dx = sepk_wrap(L.hx[i] - px, g.L[0]);
			dy = sepk_wrap(L.hy[i] - py, g.L[1]);
			dz = sepk_wrap(L.hz[i] - pz, g.L[2]);
		}
		const double r2 = dx * dx + dy * dy + dz * dz;
		unsigned long long take = __ballot(r2 < rl2);
		if (SHIFT) {
			// the 27-cell stencil reaches the home cell only through
			// offset 0: drop the atom itself
			take &= ~__ballot(jrel == i);
		} else if (take & home) {
			const int oi = L.horig[i];
			const bool drop = rule == SEPDEV_RULE_NE ? j == t32
					  : rule == SEPDEV_RULE_GT ? oj <= oi
								   : oj >= oi;
			take &= ~(__ballot(drop) & home);
		}
		if (EXCL == 3 /* SEP_EXCL_SAME_MOL */) {
			const int mi = L.hmol[i];
			if (mi != -1)
				take &= ~__ballot(mj == mi);
		}
		if (EXCL == 2 /* SEP_EXCL_BONDED */ && take) {
			bool ok = false;
			if (__builtin_amdgcn_inverse_ballot_w64(take))
				ok = sepk_keep_bonded(s, g, t, j, npad);
			take = __ballot(ok);
		}
		if (take) {
			const int e0 = __builtin_amdgcn_readlane(cnt, kk);
			const int e = (int)__builtin_amdgcn_mbcnt_hi(
				(unsigned)(take >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)take, (unsigned)e0));
			if (__builtin_amdgcn_inverse_ballot_w64(take) && e < cap)
				nbr[sepk_entry(e, t, npad)] = j;
			sepk_writelane(cnt, e0 + __popcll(take), kk);
		}
	}
}

// FP64 build: slice `slice` of `nslice` of cell c, its home atoms
// [h * slice / nslice, h * (slice + 1) / nslice), SEPK_BHOME at a time.  The
// stencil cells' segments are staged in LDS SEPK_BCHUNK candidates at a
// time, the home atoms beside them; each wave owns every fourth home atom.
template <bool SHIFT, int EXCL>
__device__ __forceinline__ void sepk_build_cell(
	sepk_build_lds &L, const sepk_state &s, long c, int slice, int nslice,
	const int *start, const sepdev_grid &g, long npad, int cap, int phantom, int *nbr,
	int *cnt, sepdev_sys *sys, int &mymax)
{
	const int lane = threadIdx.x & 63;
	const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // wave-uniform
	const int n0 = g.n[0], n1 = g.n[1], n2 = g.n[2];
	__syncthreads(); // the previous cell's readers are done with the LDS
	if (wid == 0) {
		// stencil segments, their prefix sums and whether any is shifted
		int len = 0;
		bool shifted = false;
		if (lane < g.noff) {
			const int o = lane;
			const unsigned cu = (unsigned)c, zy = cu / (unsigned)n0;
			const int cxi = (int)(cu - zy * (unsigned)n0), czi = (int)(zy / (unsigned)n1);
			const int cyi = (int)zy - czi * n1;
			const int ux = cxi + g.off[o][0], uy = cyi + g.off[o][1], uz = czi + g.off[o][2];
			const int tx = sepk_mod(ux, n0), ty = sepk_mod(uy, n1), tz = sepk_mod(uz, n2);
			const long c2 = tx + (long)ty * n0 + (long)tz * n0 * n1;
			const double sx = ux >= n0 ? -g.L[0] : ux < 0 ? g.L[0] : 0.0;
			const double sy = uy >= n1 ? -g.L[1] : uy < 0 ? g.L[1] : 0.0;
			const double sz = uz >= n2 ? -g.L[2] : uz < 0 ? g.L[2] : 0.0;
			L.segsh[o][0] = sx;
			L.segsh[o][1] = sy;
			L.segsh[o][2] = sz;
			shifted = sx != 0.0 || sy != 0.0 || sz != 0.0;
			const int js = start[c2];
			L.segjs[o] = js;
			len = start[c2 + 1] - js;
			L.segrule[o] = c2 == c ? g.off[o][3] : -1;
		}
		int x = len; // inclusive scan over the segments
		for (int d = 1; d < 64; d <<= 1) {
			const int y = __shfl_up(x, d, 64);
			if (lane >= d)
				x += y;
		}
		if (lane == 0)
			L.segpre[0] = 0;
		if (lane < g.noff)
			L.segpre[lane + 1] = x;
		const unsigned long long sv = __ballot(shifted);
		if (lane == 0) {
			L.anyshift = sv != 0ull;
			L.hs = start[c];
			L.h = start[c + 1] - L.hs;
		}
	}
	__syncthreads();
	const int hs = L.hs, h = L.h, T = L.segpre[g.noff];
	const bool anyshift = L.anyshift;
	// h < 2^24 atoms a cell and nslice <= 64: 32-bit products
	const int hbeg = nslice == 1 ? 0 : (int)((unsigned)(h * slice) / (unsigned)nslice);
	const int hend = nslice == 1 ? h : (int)((unsigned)(h * (slice + 1)) / (unsigned)nslice);
	for (int hb = hbeg; hb < hend; hb += SEPK_BHOME) {
		const int hn = min(hend - hb, SEPK_BHOME);
		int len = 0; // lane kk: list length of the wave's kk-th home atom
		for (int k0 = 0; k0 < T; k0 += SEPK_BCHUNK) {
			const int kn = min(T - k0, SEPK_BCHUNK);
			if (k0 > 0)
				__syncthreads(); // the previous chunk is no longer read
			// stage [k0, k0 + kn): thread x takes candidates x, x + SEPK_BT,
			// ...; each finds its segment by a binary search of the prefix
			// sums and all of its loads are issued before any LDS store
			constexpr int PER = (SEPK_BCHUNK + SEPK_BT - 1) / SEPK_BT;
			int jq[PER], oq[PER];
#pragma unroll
			for (int r = 0; r < PER; r++) {
				const int q = threadIdx.x + r * SEPK_BT;
				const int k = k0 + q;
				int o = 0; // the last segment starting at or before k
#pragma unroll
				for (int step = 16; step > 0; step >>= 1)
					if (o + step < g.noff && L.segpre[o + step] <= k)
						o += step;
				oq[r] = q < kn && q < SEPK_BCHUNK ? o : -1;
				jq[r] = L.segjs[o] + (k - L.segpre[o]);
			}
			sepk_pos pq[PER];
			int mq[PER];
#pragma unroll
			for (int r = 0; r < PER; r++) {
				if (oq[r] >= 0) {
					pq[r] = sepk_at(s.pos, (unsigned)jq[r]);
					if (EXCL == 3)
						mq[r] = sepk_at(s.mol, (unsigned)jq[r]);
				}
			}
#pragma unroll
			for (int r = 0; r < PER; r++) {
				if (oq[r] >= 0) {
					const int q = threadIdx.x + r * SEPK_BT;
					L.cx[q] = pq[r].x;
					L.cy[q] = pq[r].y;
					L.cz[q] = pq[r].z;
					L.cj[q] = jq[r];
					L.co[q] = (unsigned char)oq[r];
					if (EXCL == 3)
						L.cm[q] = mq[r];
				}
			}
			if (k0 == 0)
				for (int i = threadIdx.x; i < hn; i += SEPK_BT) {
					const unsigned t = (unsigned)(hs + hb + i);
					const sepk_pos p = sepk_at(s.pos, t);
					L.hx[i] = p.x;
					L.hy[i] = p.y;
					L.hz[i] = p.z;
					L.horig[i] = sepk_at(s.orig, t);
					L.hmol[i] = EXCL == 3 ? sepk_at(s.mol, t) : -1;
				}
			__syncthreads();
			const long tb = hs + hb;
			for (int q0 = 0; q0 < kn; q0 += 64) {
				if (SHIFT && anyshift)
					sepk_build_round<SHIFT, true, EXCL>(L, s, g, q0, kn, tb, hn, npad, cap,
									    nbr, len);
				else
					sepk_build_round<SHIFT, false, EXCL>(L, s, g, q0, kn, tb, hn, npad, cap,
									     nbr, len);
			}
		}
		// lane kk of each wave: its home atom's count and length bound
		const int i = wid + (SEPK_BT / 64) * lane;
		if (lane < SEPK_BHOME / (SEPK_BT / 64) && i < hn) {
			const long t = hs + hb + i;
			cnt[t] = len < cap ? len : cap;
			if (len > cap)
				sepk_set_error(sys, SEP_GPU_ENEIGHB);
			mymax = max(mymax, len);
		}
		// padding with the phantom slot to a multiple of SEPK_PAD, four
		// atoms a store: lane 16 a + s takes entry s of the last block of
		// the a-th atom of the group when that entry lies in [len, pad)
		const int nk = wid < hn ? (hn - wid + (SEPK_BT / 64) - 1) / (SEPK_BT / 64) : 0;
		for (int g0 = 0; g0 < nk; g0 += 64 / SEPK_PAD) {
			const int kk = g0 + lane / SEPK_PAD;
			const int lk = __shfl(len, kk, 64);
			const int pad = min((lk + SEPK_PAD - 1) / SEPK_PAD * SEPK_PAD, cap);
			const int e = lk / SEPK_PAD * SEPK_PAD + lane % SEPK_PAD;
			if (kk < nk && e >= lk && e < pad)
				nbr[sepk_entry(e, hs + hb + wid + (SEPK_BT / 64) * kk, npad)] = phantom;
		}
		if (hb + SEPK_BHOME < hend)
			__syncthreads(); // the next batch restages the candidates
	}
}

// End of a build kernel: the permuted state of the workgroup's share of the
// cells goes home (in one batch, so its memory round trip is paid once; one
// wave per cell, SEPK_BT / 64 cells at a time), and the largest list length to
// sys->max_full by an atomic maximum (order-independent, so the result is
// deterministic).
__device__ __forceinline__ void sepk_build_end(const sepk_state &s, const sepk_state &home,
					       const int *start, long ncell, long npad,
					       int has_partners, int mymax, sepdev_sys *sys)
{
	const long per = gridDim.x / SEPK_NXCD;
	const long xcd = blockIdx.x % SEPK_NXCD, k = blockIdx.x / SEPK_NXCD;
	const long cper = (ncell + SEPK_NXCD - 1) / SEPK_NXCD;
	const long lo = xcd * cper, hi = min(lo + cper, ncell);
	const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
	for (long c = lo + k + wv * per; c < hi; c += (SEPK_BT / 64) * per) {
		const int a = start[c], b = start[c + 1];
		for (int t = a + ln; t < b; t += 64)
			sepk_copy_home(s, home, t, npad, has_partners);
	}
	for (int o = 32; o > 0; o >>= 1)
		mymax = max(mymax, __shfl_xor(mymax, o, 64));
	__shared__ int bmax;
	if (threadIdx.x == 0)
		bmax = 0;
	__syncthreads();
	if (ln == 0)
		atomicMax(&bmax, mymax);
	__syncthreads();
	if (threadIdx.x == 0 && bmax > 0)
		atomicMax(&sys->max_full, bmax);
}

// Quantized build, persistent over (cell, slice) items, a wave an item
// (nslice per cell): no wave waits for another, so the memory round trips of
// one (cell starts, candidates) hide behind the tests of the others.  A slice
// takes the cell's atoms by their rank in x: a slab whose bounding box only
// about 45 % of the stencil's candidates come near (two slabs a cell; a third
// with four, but the walk over the candidates is then shared by too few).
// Neither the order of the atoms nor that of the lists depends on the slices.
//
// What bounds the build is instruction issue and latency; its bytes are few.
// N = 256000, per rebuild: 190 us with a workgroup a cell, candidates shared
// through LDS, every one tested and each round's handful of accepted ones
// stored at once (a partly filled store and 9 address instructions a round);
// 143 with the accepted ones collected in an LDS row; 138 with the bounding
// box; 130 with a wave an item and slabs of about 11 atoms (a few us more with 6
// and with the whole cell).
template <int EXCL>
__global__ __launch_bounds__(SEPK_BT) __attribute__((amdgpu_waves_per_eu(EXCL == 2 ? 4 : 7))) void k_build_q(
	sepk_state s, sepk_state home, const int *start, sepdev_grid g, sepk_qtest qt, long ncell,
	int nslice, long n, long npad, int cap, int *nbr, int *cnt, sepdev_sys *sys,
	int conditional, int has_partners)
{
	if ((conditional && sys->neighb_flag == 0) || sys->frozen)
		return;
	__shared__ sepk_qwave<EXCL> WV[SEPK_BT / 64];
	const int lane = threadIdx.x & 63;
	const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // wave-uniform
	sepk_qwave<EXCL> &W = WV[wid];
	const bool clean = sys->unclean == 0;
	// items < 2^31 (the host bounds nslice by the atoms a cell)
	const unsigned per = gridDim.x / SEPK_NXCD;
	const unsigned xcd = blockIdx.x % SEPK_NXCD, k = blockIdx.x / SEPK_NXCD;
	const unsigned nitem = (unsigned)ncell * (unsigned)nslice;
	const unsigned iper = (nitem + SEPK_NXCD - 1) / SEPK_NXCD;
	const unsigned ilo = xcd * iper, ihi = min(ilo + iper, nitem);
	int mymax = 0;
	for (unsigned it = ilo + k * (SEPK_BT / 64) + wid; it < ihi; it += per * (SEPK_BT / 64)) {
		const int c = sepk_quotient((int)it, qt.islice);
		const int sl = (int)it - c * nslice;
		int js, len;
		sepk_build_segment(g, qt, c, start, js, len);
		const int hs = __builtin_amdgcn_readlane(js, 18), h = __builtin_amdgcn_readlane(len, 18);
		if (h == 0)
			continue;
		int x = lane < 18 ? len : 0; // inclusive scan over the segments
		for (int d = 1; d < 32; d <<= 1) {
			const int y = __shfl_up(x, d, 64);
			if (lane >= d)
				x += y;
		}
		const unsigned used = (unsigned)__ballot(lane < 18 && len > 0);
		const int T = __builtin_amdgcn_readlane(x, 17);
		// the cell's atoms in nb batches of at most 64 (one, unless it is
		// very full), the cell's slices shared out among the batches: this
		// one is slab `sub` of `nsub` of its batch (or whole batches, every
		// nslice-th, where there are more batches than slices)
		const int nb = (h + SEPK_BHOME - 1) / SEPK_BHOME;
		const bool shared = nb <= nslice;
		int b = shared ? (int)((unsigned)(sl * nb) / (unsigned)nslice) : sl;
		for (; b < nb; b += shared ? nb : nslice) {
			const int s0 = shared ? (b * nslice + nb - 1) / nb : sl;
			const int s1 = shared ? ((b + 1) * nslice + nb - 1) / nb : sl + 1;
			const int sub = sl - s0, nsub = s1 - s0;
			const int ha = (int)((unsigned long)h * b / nb);
			const int hn = (int)((unsigned long)h * (b + 1) / nb) - ha, tb = hs + ha;
			const unsigned ti = (unsigned)(tb + min(lane, hn - 1));
			const uint2 hq = sepk_quant21(sepk_at(s.qpos, ti));
			const int hm = EXCL == 3 ? sepk_at(s.mol, ti) : -1;
			unsigned long long mine = hn < 64 ? ~(~0ull << hn) : ~0ull;
			if (nsub > 1) {
				// the slab's atoms by their rank in x
				const int key = (int)((hq.x & 0xffffu) << 6) | lane;
				int rank = 0;
				for (int j = 0; j < hn; j++)
					rank += __builtin_amdgcn_readlane(key, j) < key;
				mine &= __ballot(rank >= hn * sub / nsub && rank < hn * (sub + 1) / nsub);
				if (!mine)
					continue;
			}
			int m = 0; // lane i: list length of home atom i
			if (clean)
				sepk_build_home<EXCL>(W, used, x - len, js - (x - len), T, s, g, qt, tb, mine, hq,
						      hm, npad, cap, (int)n, nbr, m);
			else
				sepk_build_outside<EXCL>(js, len, s, g, tb, mine, npad, cap, (int)n, nbr, m);
			if (mine >> lane & 1ull) {
				cnt[tb + lane] = m < cap ? m : cap;
				if (m > cap)
					sepk_set_error(sys, SEP_GPU_ENEIGHB);
				mymax = max(mymax, m);
			}
		}
	}
	sepk_build_end(s, home, start, ncell, npad, has_partners, mymax, sys);
}

// FP64 build, persistent over (cell, slice) items, nslice per cell, a
// workgroup an item.
template <int EXCL>
__global__ __launch_bounds__(SEPK_BT) __attribute__((amdgpu_waves_per_eu(EXCL == 2 ? 4 : 7))) void k_build(
	sepk_state s, sepk_state home, const int *start, sepdev_grid g, sepk_qtest, long ncell,
	int nslice, long n, long npad, int cap, int *nbr, int *cnt, sepdev_sys *sys,
	int conditional, int has_partners)
{
	if ((conditional && sys->neighb_flag == 0) || sys->frozen)
		return;
	__shared__ sepk_build_lds L;
	const bool shift = g.shift_ok && sys->unclean == 0;
	const long per = gridDim.x / SEPK_NXCD;
	const long xcd = blockIdx.x % SEPK_NXCD, k = blockIdx.x / SEPK_NXCD;
	const long nitem = ncell * nslice;
	const long iper = (nitem + SEPK_NXCD - 1) / SEPK_NXCD;
	const long ilo = xcd * iper, ihi = min(ilo + iper, nitem);
	int mymax = 0;
	for (long it = ilo + k; it < ihi; it += per) {
		// items < 2^31 (the host bounds nslice by the atoms a cell)
		const long c = nslice == 1 ? it : (long)((unsigned)it / (unsigned)nslice);
		const int sl = (int)(it - c * nslice);
		if (shift)
			sepk_build_cell<true, EXCL>(L, s, c, sl, nslice, start, g, npad, cap, (int)n, nbr,
						    cnt, sys, mymax);
		else
			sepk_build_cell<false, EXCL>(L, s, c, sl, nslice, start, g, npad, cap, (int)n, nbr,
						     cnt, sys, mymax);
	}
	sepk_build_end(s, home, start, ncell, npad, has_partners, mymax, sys);
}

// ---- host side --------------------------------------------------------------

extern "C" int sepdev_reserve_list(sepdev *d, int cap)
{
	if (d->capturing)
		return sepk_fail(SEP_GPU_ESTATE, "list resize during graph capture");
	int lcap = (cap + SEPK_SUB - 1) / SEPK_SUB;
	lcap = (lcap + 7) / 8 * 8;
	if (d->nbr && lcap <= d->lcap)
		return 0;
	SEPK_CHECK(hipStreamSynchronize(d->st));
	if (d->nbr)
		(void)hipFree(d->nbr);
	d->nbr = nullptr;
	SEPK_CHECK(hipMalloc(&d->nbr, (size_t)lcap * SEPK_SUB * d->npad * sizeof(int)));
	SEPK_CHECK(hipMemsetAsync(d->nbr_count, 0, d->npad * sizeof(int), d->st));
	d->lcap = lcap;
	d->cap = lcap * SEPK_SUB;
	d->list_built = 0;
	return 0;
}

extern "C" int sepdev_list_limit(sepdev *d, int cap, int *applied)
{
	if (cap < 0)
		return sepk_fail(SEP_GPU_EARG, "list limit %d", cap);
	// whole batches: a truncated list then ends on a batch boundary, and
	// the pair kernels read no entry the build did not write
	if (cap > 0) {
		cap = cap / SEPK_PAD * SEPK_PAD;
		if (cap < SEPK_PAD)
			cap = SEPK_PAD;
	}
	d->cap_limit = cap;
	if (cap > 0 && (!d->nbr || cap > d->cap)) {
		int rc = sepdev_reserve_list(d, cap);
		if (rc)
			return rc;
	}
	if (applied)
		*applied = cap;
	return 0;
}

extern "C" int sepdev_reset_max_dist(sepdev *d)
{
	// owed to the next leapfrog, which then starts its maximum at zero
	d->max_reset_pending = 1;
	return 0;
}

extern "C" int sepdev_list_capacity(sepdev *d) { return d->nbr ? d->cap : 0; }

extern "C" int sepdev_build_list(sepdev *d, const sepdev_grid *gp, int conditional)
{
	const sepdev_grid &g = *gp;
	if (g.noff <= 0 || g.noff > SEPDEV_MAX_OFF)
		return sepk_fail(SEP_GPU_EARG, "build_list: %d offsets", g.noff);
	for (int k = 0; k < 3; k++)
		if (g.n[k] < 1)
			return sepk_fail(SEP_GPU_EARG, "build_list: %d cells on axis %d", g.n[k], k);
	const long ncell = (long)g.n[0] * g.n[1] * g.n[2];
	if (ncell > (1L << 28))
		return sepk_fail(SEP_GPU_EARG, "build_list: %ld cells", ncell);
	if (g.opt == 2 && !d->s[0].partners)
		return sepk_fail(SEP_GPU_ESTATE, "SEP_EXCL_BONDED needs bonded partners");
	// a recorded pair call reads the current list: launch it before the
	// list can be resized or rebuilt
	int rc = sepk_flush_pair(d);
	if (rc)
		return rc;
	rc = sepk_flush_nh(d);
	if (rc)
		return rc;
	// a rebuild permutes the atoms: a fork point recorded before it (also
	// by the flushed pair call above) must not serve the terms after it
	d->fork_ready = 0;

	// size buffers on the host side of any capture
	if (ncell > d->ncell_cap) {
		if (d->capturing)
			return sepk_fail(SEP_GPU_ESTATE, "cell grid grew during graph capture");
		(void)hipFree(d->cell_count);
		(void)hipFree(d->cell_start);
		SEPK_CHECK(hipMalloc(&d->cell_count, ncell * sizeof(int)));
		SEPK_CHECK(hipMalloc(&d->cell_start, (ncell + 1) * sizeof(int)));
		SEPK_CHECK(hipMemsetAsync(d->cell_count, 0, ncell * sizeof(int), d->st));
		d->ncell_cap = ncell;
	}
	if (!d->nbr) {
		// capacity from the mean density with a generous margin
		const double V = g.L[0] * g.L[1] * g.L[2];
		const double rl = sqrt(g.rlist2);
		double expect = 4.18879020478639 * rl * rl * rl * (double)d->n / V;
		if (!(expect < 1e7))
			expect = 1e7;
		long cap = (long)(2.0 * expect) + 64;
		if (cap > d->n * 4 + 64)
			cap = d->n * 4 + 64;
		if (d->capturing)
			return sepk_fail(SEP_GPU_ESTATE, "list allocated during graph capture");
		if ((rc = sepdev_reserve_list(d, (int)cap)))
			return rc;
	}
	if ((rc = sepk_claim_region(d, SEPK_R_BUILD)))
		return rc;
	sepk_qtest qt;
	const bool qnt = sepk_qtest_of(g, qt);
	if (qnt && (rc = sepk_fresh_qpos(d, g.L)))
		return rc;

	sepk_state &cur = d->s[0];   // current state, fixed addresses
	sepk_state &spare = d->s[1]; // receives the permuted order
	const int hp = cur.partners != nullptr;
	const bool one = conditional || d->n <= SEPK_ORDER_BUILD || d->n > SEPK_ORDER_FULL * ncell;
	if (one && d->n <= SEPK_ORDER_ATOMS && ncell <= SEPK_ORDER_CELLS) {
		const unsigned ob = (unsigned)(ncell < SEPK_ORDER_GRID ? ncell : SEPK_ORDER_GRID);
		(d->n <= SEPK_ORDER_ATOMS / 8 ? k_order<SEPK_ORDER_ATOMS / 8> : k_order<SEPK_ORDER_ATOMS>)<<<ob, 1024, 0, d->st>>>(
			cur, spare, d->n, d->npad, g, (int)ncell, d->cell_start, d->iperm, d->sys,
			conditional, hp);
	} else {
		unsigned nb = sepk_blocks(d->n);
		if (nb > SEPK_GRID_CAP)
			nb = SEPK_GRID_CAP;
		// half a wave per cell when the cells hold 32 atoms or fewer on
		// average, a wave up to 64, a workgroup beyond
		const bool half = d->n <= 32 * ncell, wg = d->n > 64 * ncell;
		long sb = wg ? ncell : (ncell * (half ? 32 : 64) + SEPK_BLOCK - 1) / SEPK_BLOCK;
		if (sb > SEPK_GRID_CAP)
			sb = SEPK_GRID_CAP;
		k_bin<<<nb, SEPK_BLOCK, 0, d->st>>>(cur.pos, d->n, g, d->cellid_old, d->cell_slot,
						    d->cell_count, d->sys,
						    conditional);
		if (ncell <= SEPK_PLACE_CELLS) {
			// one launch: each workgroup scans the counts itself
			long pb = (d->n + 1023) / 1024;
			if (pb > 256)
				pb = 256;
			k_scan_scatter<<<(unsigned)pb, 1024, 0, d->st>>>(
				d->cell_count, d->cell_start, d->cellid_old, d->cell_slot, d->order_tmp, ncell,
				d->n, d->sys, conditional);
		} else {
			k_scan<<<1, 1024, 0, d->st>>>(d->cell_count, d->cell_start, ncell, d->sys,
						      conditional);
			k_scatter<<<nb, SEPK_BLOCK, 0, d->st>>>(d->cellid_old, d->cell_slot,
								d->cell_start, d->order_tmp, d->n, d->sys,
								conditional);
		}
		(wg ? k_sort_permute_wg : half ? k_sort_permute<32> : k_sort_permute<64>)<<<(unsigned)sb, SEPK_BLOCK, 0, d->st>>>(
			d->order_tmp, d->cell_start, cur, spare, d->iperm, ncell, d->npad,
			d->sys, conditional, hp, d->cell_count);
	}
	SEPK_LAUNCH_CHECK();
	// A cell's atoms in nslice slices (the lists do not depend on the
	// split).  FP64, a workgroup a slice: one, unless the cells are few and
	// full: at least 16 atoms a slice, at most SEPK_BHOME, about 1024
	// slices.  Quantized, a wave a slice: about SEPK_QSLICE atoms, fewer
	// where there would not be 2048 slices (N = 27000: 37.5 us a step; 38.5
	// with 4096 slices, 39.4 with a workgroup a cell), 4096 where the cells
	// hold more than 64 atoms, so that slices of several atoms are left (a
	// pair call that rebuilds, us: 16000 atoms in 125 cells 148 -> 121, in 216
	// 97 -> 81, 32000 317 -> 254 and 189 -> 159; 8000 in 125 53 -> 56, so not
	// below.  The FP64 build took 134, 90, 287, 180 and 69).
	const long avg = (d->n + ncell - 1) / ncell;
	const long least = qnt ? (avg + 31) / 32 : (avg + SEPK_BHOME - 1) / SEPK_BHOME;
	const long most = qnt ? avg : (avg + 15) / 16;
	const long fill = ((qnt ? avg > 64 ? 4096 : 2048 : 1024) + ncell - 1) / ncell;
	long nslice = qnt ? (avg + SEPK_QSLICE / 2) / SEPK_QSLICE : 1;
	if (nslice < fill)
		nslice = fill;
	if (nslice > most)
		nslice = most;
	if (nslice < least)
		nslice = least;
	if (nslice < 1)
		nslice = 1;
	if (nslice > 64)
		nslice = 64;
	qt.islice = 1.0 / (double)nslice;
	const long wgs = qnt ? (ncell * nslice + SEPK_BT / 64 - 1) / (SEPK_BT / 64) : ncell * nslice;
	long bb = (wgs + SEPK_NXCD - 1) / SEPK_NXCD * SEPK_NXCD;
	if (bb > SEPK_BGRID)
		bb = SEPK_BGRID;
	auto kb = qnt ? (g.opt == 2 ? k_build_q<2> : g.opt == 3 ? k_build_q<3> : k_build_q<0>)
		      : (g.opt == 2 ? k_build<2> : g.opt == 3 ? k_build<3> : k_build<0>);
	const int capb = d->cap_limit > 0 && d->cap_limit < d->cap ? d->cap_limit : d->cap;
	kb<<<(unsigned)bb, SEPK_BT, 0, d->st>>>(spare, cur, d->cell_start, g, qt, ncell, (int)nslice,
						      d->n, d->npad, capb, d->nbr, d->nbr_count,
						      d->sys, conditional, hp);
	SEPK_LAUNCH_CHECK();
	// clears the rebuild flag and the owed xn reset
	sepk_task f;
	memset(&f, 0, sizeof f);
	f.mode = SEPK_FIN_BUILD;
	f.region = SEPK_R_BUILD;
	f.conditional = conditional;
	if ((rc = sepk_queue_task(d, f)))
		return rc;
	// an unconditional build is finished at once, so the host can check it
	if (!conditional && (rc = sepk_flush_tasks(d)))
		return rc;
	d->grid = g;
	d->list_built = 1;
	return 0;
}
