// sepdev_force.hip -- pair forces over the full neighbour list, the
// Nose-Hoover and leapfrog updates, and list extraction for the host.
//
// Pair kernels: one thread per atom (device order), the full list read in
// its interleaved layout, forces kept in registers and written once per
// atom (no atomics).  Energy and stress are summed per atom, halved (each
// pair is seen from both ends), reduced per block in a fixed order and
// finished by the last block, so repeated runs give identical bits.
#include <float.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "sepdev_impl.h"

int sepk_timer_begin(sepdev *d, sepk_timer *t);
int sepk_timer_end(sepdev *d, sepk_timer *t);

// ---- lazy force reset ------------------------------------------------------

__global__ void k_zero_forces(double *f, long count, const int *err)
{
	long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
	if (t < count && !*err)
		f[t] = 0.0;
}

int sepk_materialize_forces(sepdev *d)
{
	int rc = sepk_flush_pair(d);
	if (rc || (rc = sepk_flush_gathers(d)))
		return rc;
	if (!d->f_zero_pending)
		return 0;
	const long cnt = 3 * d->npad;
	k_zero_forces<<<sepk_blocks(cnt), SEPK_BLOCK, 0, d->st>>>(d->s[0].f, cnt, d->s[0].err);
	SEPK_LAUNCH_CHECK();
	d->f_zero_pending = 0;
	return 0;
}

extern "C" int sepdev_zero_forces(sepdev *d)
{
	// The next force kernel overwrites instead of accumulating; anything
	// else that reads f first materialises the zeros.  Owed gathers would
	// be zeroed with the rest: they are dropped.
	d->f_zero_pending = 1;
	d->ngpend = 0;
	d->gpend_over = 0;
	return 0;
}

// ---- LJ family ---------------------------------------------------------------

// ft = eps48 q^3 (q^3 - aw/2) q and u = eps4 q^3 (q^3 - aw) + ushift with
// q = sig2 / r^2, evaluated as ft = (A q^3 + nB) q^3 q, u = (C q^3 + nD) q^3 + ushift
// (nB = -eps48 aw/2, nD = -eps4 aw)

// Shared epilogue of the list kernels: combine the SEPK_SUB lanes of each
// atom (fixed xor order), write or add its force from lane 0, and leave the
// block's energy + stress row in the pair region.  acc = {e, wxx, wxy, wxz,
// wyy, wyz, wzz}, each summed over the lane's share of the full list.
// The stress of a pair term, sum over listed pairs of f (x) r, is not
// accumulated pair by pair.  With r_ij = x_i - x_j - s_ij (s_ij = L k_ij,
// the periodic shift taken off) and f_ji = -f_ij, the full-list sum is
//     sum_{i,j} f_ij (x) r_ij = 2 sum_i F_i (x) x_i - sum_{i,j} f_ij (x) s_ij,
// so a pair adds to the stress only when it crosses the box (k != 0), and
// each atom adds 2 F_i (x) x_i once, here, from its summed force.  The six
// components are {xx, xy, xz, yy, yz, zz} of f (x) r; the finisher halves
// the full-list sums.  frozen: the device error word is set, and f is left
// as it is.
template <bool OVERWRITE>
__device__ __forceinline__ void sepk_pair_epilogue(
	long t, int sub, long n, long npad, bool act, double fx, double fy, double fz,
	double px, double py, double pz, double (&acc)[7], double *f, double *partial,
	long row, long rows, bool frozen)
{
	fx = sepk_atom_sum(fx);
	fy = sepk_atom_sum(fy);
	fz = sepk_atom_sum(fz);
	if (t < n && sub == 0 && !frozen) {
		if (OVERWRITE) {
			f[t] = fx;
			f[npad + t] = fy;
			f[2 * npad + t] = fz;
		} else if (act) {
			f[t] += fx;
			f[npad + t] += fy;
			f[2 * npad + t] += fz;
		}
	}
	if (act && sub == 0) {
		const double gx = 2.0 * fx, gy = 2.0 * fy, gz = 2.0 * fz;
		acc[1] = fma(gx, px, acc[1]);
		acc[2] = fma(gx, py, acc[2]);
		acc[3] = fma(gx, pz, acc[3]);
		acc[4] = fma(gy, py, acc[4]);
		acc[5] = fma(gy, pz, acc[5]);
		acc[6] = fma(gz, pz, acc[6]);
	}
	sepk_block_partial(acc, partial, row, rows);
}

// Minimum image of d, returning d - L k with the image count k in
// {-1, 0, 1} (the reference's single-image rule, or its FAST form).
template <bool FAST>
__device__ __forceinline__ double sepk_image(double d, double L, double iL, double &k)
{
	// selected, not branched to: the pairs of a batch are evaluated side by
	// side (d - L and d + L are the fma's results for k = 1 and -1)
	k = FAST ? rint(d * iL) : d > 0.5 * L ? 1.0 : d < -0.5 * L ? -1.0 : 0.0;
	return fma(-L, k, d);
}

// Adds one pair's force ft r to the atom and its energy; the stress gets
// only the crossing term -f (x) s (see sepk_pair_epilogue).
__device__ __forceinline__ void sepk_pair_cross(
	double ft, double dx, double dy, double dz, double kx, double ky, double kz, double L0,
	double L1, double L2, double (&acc)[7])
{
	const double sx = kx * L0, sy = ky * L1, sz = kz * L2;
	const double gx = -ft * dx, gy = -ft * dy, gz = -ft * dz;
	acc[1] = fma(gx, sx, acc[1]);
	acc[2] = fma(gx, sy, acc[2]);
	acc[3] = fma(gx, sz, acc[3]);
	acc[4] = fma(gy, sy, acc[4]);
	acc[5] = fma(gy, sz, acc[5]);
	acc[6] = fma(gz, sz, acc[6]);
}

__device__ __forceinline__ void sepk_pair_accumulate(
	double ft, double e, double dx, double dy, double dz, double kx, double ky, double kz,
	double L0, double L1, double L2, double &fx, double &fy, double &fz, double (&acc)[7])
{
	fx = fma(ft, dx, fx);
	fy = fma(ft, dy, fy);
	fz = fma(ft, dz, fz);
	acc[0] += e;
	if (kx != 0.0 || ky != 0.0 || kz != 0.0)
		sepk_pair_cross(ft, dx, dy, dz, kx, ky, kz, L0, L1, L2, acc);
}

// Entries of one lane are taken SEPK_BATCH at a time: every index and
// every neighbour position of the batch is loaded before any is used, so a
// wave keeps SEPK_BATCH gathers in flight instead of one.  Lists are padded
// to whole batches with the phantom slot (NaN position, type 0, charge 0),
// which fails every test, so the loads need neither clamps nor branches; the
// accumulation order is the list order.
//
// Addressing: lane `sub` of atom t reads the SEPK_BATCH indices of its
// batch b as one int4 (sepk_entry, sepk_lane_list); neighbour records are
// fetched with 32-bit byte offsets from the uniform base.
__device__ __forceinline__ const sepk_pos &sepk_rec(const char *base, int j)
{
	return *(const sepk_pos *)(base + (unsigned)j * (unsigned)sizeof(sepk_pos));
}

// 1 / r2 in FP64: hardware reciprocal and two Newton steps (within an ulp of
// the division; the error bar of the FP64 path is 1e-12)
__device__ __forceinline__ double sepk_recip(double r2)
{
	double y = __builtin_amdgcn_rcp(r2);
	double e = fma(-r2, y, 1.0);
	y = fma(y, e, y);
	e = fma(-r2, y, 1.0);
	return fma(y, e, y);
}

// The cutoff test of the mixed LJ loops.  Each quantized coordinate is
// within half a quantization step of the FP64 one, so the quantized r^2 is
// within c.band of the r^2 the plain kernel forms; a pair that close to the
// cutoff is decided on the FP64 records, as the plain kernel decides it.
// (The force of sep_lj and sep_lj_shift jumps by F(rc) = -0.039 at rc = 2.5:
// a pair taken by one form and dropped by the other would put that whole
// jump into the force error of both atoms.)  About one pair in 10^8 lies in
// the band.
template <bool FAST>
__device__ __forceinline__ bool sepk_inside_mixed(const sepk_state &s, long t, unsigned j,
						  double r2, const sepk_lj &c)
{
	if (!(fabs(r2 - c.cf2) < c.band))
		return r2 < c.cf2;
	const sepk_pos pi = s.pos[t], pj = s.pos[j];
	double kx, ky, kz;
	const double dx = sepk_image<FAST>(pi.x - pj.x, c.L0, c.iL0, kx);
	const double dy = sepk_image<FAST>(pi.y - pj.y, c.L1, c.iL1, ky);
	const double dz = sepk_image<FAST>(pi.z - pj.z, c.L2, c.iL2, kz);
	return dx * dx + dy * dy + dz * dz < c.cf2;
}

// One pair of the mixed LJ loop: the FP32 force and energy terms from the
// quantized squared distance r2 (dx, dy, dz in FP64), summed in FP64, and
// the crossing stress when the integer difference wrapped.
__device__ __forceinline__ void sepk_lj_mixed_add(
	const sepk_lj &c, unsigned ux, unsigned vx, unsigned uy, unsigned vy, unsigned uz,
	unsigned vz, int ix, int iy, int iz, double dx, double dy, double dz, double r2,
	double &fx, double &fy, double &fz, double (&acc)[7])
{
	const float q = c.sig2f * __builtin_amdgcn_rcpf((float)r2);
	const float q3 = q * q * q;
	const double ft = (double)(fmaf(c.Af, q3, c.nBf) * q3 * q);
	const double e = (double)fmaf(fmaf(c.Cf, q3, c.nDf), q3, c.ushiftf);
	fx = fma(ft, dx, fx);
	fy = fma(ft, dy, fy);
	fz = fma(ft, dz, fz);
	acc[0] += e;
	const bool bx = (ux < vx) != (ix < 0), by = (uy < vy) != (iy < 0),
		   bz = (uz < vz) != (iz < 0);
	if (bx | by | bz) {
		// k = +1 when the unwrapped difference is >= 2^31 steps (wrapped
		// negative), -1 when it is below -2^31 (wrapped non-negative)
		const double kx = bx ? (ix < 0 ? 1.0 : -1.0) : 0.0;
		const double ky = by ? (iy < 0 ? 1.0 : -1.0) : 0.0;
		const double kz = bz ? (iz < 0 ? 1.0 : -1.0) : 0.0;
		sepk_pair_cross(ft, dx, dy, dz, kx, ky, kz, c.L0, c.L1, c.L2, acc);
	}
}

// One entry of a mixed LJ walk (untyped): the pair of records qi, qj,
// added when inside c.cf2lo; one nearer the cutoff than that sets band and
// is left to sepk_lj_mixed_band.
__device__ __forceinline__ void sepk_lj_mixed_entry(const sepk_lj &c, const int4 &qi,
						    const int4 &qj, double &fx, double &fy,
						    double &fz, double (&acc)[7], bool &band)
{
	if (qj.w == SEPK_QPHANTOM)
		return;
	const unsigned ux = (unsigned)qi.x, vx = (unsigned)qj.x;
	const unsigned uy = (unsigned)qi.y, vy = (unsigned)qj.y;
	const unsigned uz = (unsigned)qi.z, vz = (unsigned)qj.z;
	const int ix = (int)(ux - vx), iy = (int)(uy - vy), iz = (int)(uz - vz);
	const double dx = (double)ix * c.qd0;
	const double dy = (double)iy * c.qd1;
	const double dz = (double)iz * c.qd2;
	const double r2 = dx * dx + dy * dy + dz * dz;
	if (!(r2 < c.cf2lo)) {
		// near the cutoff: decided after the walk
		band |= r2 < c.cf2hi;
		return;
	}
	sepk_lj_mixed_add(c, ux, vx, uy, vy, uz, vz, ix, iy, iz, dx, dy, dz, r2, fx, fy, fz, acc);
}

// The pairs of the mixed loop that lay within c.band of the cutoff (the
// loop left them out and flagged the lane): decided on the FP64 records as
// the plain kernel decides them (sepk_inside_mixed), and added when inside.
// A lane gets here for about one pair in 10^8.
template <bool TYPED, bool FAST>
__device__ __forceinline__ void sepk_lj_mixed_band(
	const sepk_state &s, const int *__restrict__ nbr, const int *__restrict__ cnt, long npad,
	const sepk_lj &c, long t, int sub, signed char ti, int4 qi, double &fx, double &fy,
	double &fz, double (&acc)[7])
{
	const int n = cnt[t];
	for (int e = sub; e < n; e += SEPK_SUB) {
		const unsigned j = (unsigned)nbr[sepk_entry(e, t, npad)];
		const int4 qj = sepk_at(s.qpos, j);
		if (TYPED) {
			const signed char tj = s.type[j];
			if (!((ti == c.t0 && tj == c.t1) || (ti == c.t1 && tj == c.t0)))
				continue;
		}
		if (qj.w == SEPK_QPHANTOM)
			continue;
		const unsigned ux = (unsigned)qi.x, vx = (unsigned)qj.x;
		const unsigned uy = (unsigned)qi.y, vy = (unsigned)qj.y;
		const unsigned uz = (unsigned)qi.z, vz = (unsigned)qj.z;
		const int ix = (int)(ux - vx), iy = (int)(uy - vy), iz = (int)(uz - vz);
		const double dx = (double)ix * c.qd0;
		const double dy = (double)iy * c.qd1;
		const double dz = (double)iz * c.qd2;
		const double r2 = dx * dx + dy * dy + dz * dz;
		if (r2 < c.cf2lo || !(r2 < c.cf2hi) || !sepk_inside_mixed<FAST>(s, t, j, r2, c))
			continue;
		sepk_lj_mixed_add(c, ux, vx, uy, vy, uz, vz, ix, iy, iz, dx, dy, dz, r2, fx, fy, fz,
				  acc);
	}
}

// The pair loop of atom t, lane `sub`: the lane's share of the atom's force
// and of the block's energy and crossing stress, and the position the
// stress identity pairs the summed force with (px, py, pz).
template <bool TYPED, bool MIXED, bool FAST>
__device__ __forceinline__ void sepk_lj_pairs(
	const sepk_state &s, const int *__restrict__ nbr, const int *__restrict__ cnt, long npad,
	const sepk_lj &c, long t, int sub, bool act, signed char ti, double &fx, double &fy,
	double &fz, double (&acc)[7], double &px, double &py, double &pz)
{
	if (MIXED) {
		// positions quantized to the box (sepk_quant): the integer
		// difference is the minimum image, one 16-byte gather per entry;
		// the stress identity uses the quantized positions x~ = u L / 2^32
		// and the image count k of the pair, nonzero when the unwrapped
		// difference borrows differently from the wrapped one
		int4 qi = make_int4(0, 0, 0, SEPK_QPHANTOM);
		if (act) {
			qi = s.qpos[t];
			bool band = false;
			const int nbat = (cnt[t] + SEPK_PAD - 1) / SEPK_PAD;
			const size_t stride = (size_t)npad * SEPK_SUB;
			const int4 *lp = sepk_wave_list(nbr, t, sub);
			const unsigned ln = threadIdx.x & 63;
			// batch 0 goes out with the count (every list allocation
			// holds it), and batch b + 1 while batch b is computed
			int4 jb = sepk_at(lp, ln);
			for (int b = 0; b < nbat; b++) {
				const int j[SEPK_BATCH] = {jb.x, jb.y, jb.z, jb.w};
				int4 qj[SEPK_BATCH];
				signed char tj[SEPK_BATCH];
#pragma unroll
				for (int u = 0; u < SEPK_BATCH; u++) {
					qj[u] = sepk_at(s.qpos, (unsigned)j[u]);
					if (TYPED)
						tj[u] = s.type[(unsigned)j[u]];
				}
				// the wave's last batch reloads itself (a cache hit)
				if (__ballot(b + 1 < nbat))
					lp += stride;
				jb = sepk_at(lp, ln);
#pragma unroll
				for (int u = 0; u < SEPK_BATCH; u++) {
					if (TYPED && !((ti == c.t0 && tj[u] == c.t1) ||
						       (ti == c.t1 && tj[u] == c.t0)))
						continue;
					sepk_lj_mixed_entry(c, qi, qj[u], fx, fy, fz, acc, band);
				}
			}
			if (band)
				sepk_lj_mixed_band<TYPED, FAST>(s, nbr, cnt, npad, c, t, sub, ti, qi, fx,
								fy, fz, acc);
		}
		px = act ? (double)(unsigned)qi.x * c.qd0 : 0.0;
		py = act ? (double)(unsigned)qi.y * c.qd1 : 0.0;
		pz = act ? (double)(unsigned)qi.z * c.qd2 : 0.0;
		return;
	}
	sepk_pos pi = {0.0, 0.0, 0.0, 0.0};
	if (act) {
		pi = s.pos[t];
		const int nbat = (cnt[t] + SEPK_PAD - 1) / SEPK_PAD;
		const size_t stride = (size_t)npad * SEPK_SUB;
		const int4 *lp = sepk_wave_list(nbr, t, sub);
		const unsigned ln = threadIdx.x & 63;
		const char *pb = (const char *)s.pos;
		// batch b + 1 in flight while batch b is computed, as above
		int4 jb = sepk_at(lp, ln);
		for (int b = 0; b < nbat; b++) {
			const int j[SEPK_BATCH] = {jb.x, jb.y, jb.z, jb.w};
			double px[SEPK_BATCH], py[SEPK_BATCH], pz[SEPK_BATCH];
			signed char tj[SEPK_BATCH];
#pragma unroll
			for (int u = 0; u < SEPK_BATCH; u++) {
				const sepk_pos &r = sepk_rec(pb, j[u]);
				px[u] = r.x;
				py[u] = r.y;
				pz[u] = r.z;
				if (TYPED)
					tj[u] = s.type[(unsigned)j[u]];
			}
			// the wave's last batch reloads itself (a cache hit)
			if (__ballot(b + 1 < nbat))
				lp += stride;
			jb = sepk_at(lp, ln);
#pragma unroll
			for (int u = 0; u < SEPK_BATCH; u++) {
				if (TYPED && !((ti == c.t0 && tj[u] == c.t1) ||
					       (ti == c.t1 && tj[u] == c.t0)))
					continue;
				double kx, ky, kz;
				const double dx = sepk_image<FAST>(pi.x - px[u], c.L0, c.iL0, kx);
				const double dy = sepk_image<FAST>(pi.y - py[u], c.L1, c.iL1, ky);
				const double dz = sepk_image<FAST>(pi.z - pz[u], c.L2, c.iL2, kz);
				// r^2 in the reference's order
				const double r2 = dx * dx + dy * dy + dz * dz;
				if (!(r2 < c.cf2))
					continue;
				const double q = c.sig2 * sepk_recip(r2);
				const double q3 = q * q * q;
				const double ft = fma(c.A, q3, c.nB) * q3 * q;
				const double e = fma(fma(c.C, q3, c.nD), q3, c.ushift);
				sepk_pair_accumulate(ft, e, dx, dy, dz, kx, ky, kz, c.L0, c.L1, c.L2,
						     fx, fy, fz, acc);
			}
		}
	}
	px = pi.x;
	py = pi.y;
	pz = pi.z;
}


template <bool TYPED, bool MIXED, bool OVERWRITE, bool FAST>
__global__ __launch_bounds__(SEPK_BLOCK) void k_lj(
	sepk_state s, const int *__restrict__ nbr, const int *__restrict__ cnt,
	long n, long npad, sepk_lj c, double *partial, long rows)
{
	const long lb = sepk_xcd_block();
	const long t = lb * (SEPK_BLOCK / SEPK_SUB) + threadIdx.x / SEPK_SUB;
	const int sub = threadIdx.x % SEPK_SUB;
	const bool frozen = *s.err != 0;
	double fx = 0.0, fy = 0.0, fz = 0.0;
	double acc[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
	bool act = t < n;
	signed char ti = 0;
	if (act && TYPED) {
		ti = s.type[t];
		act = ti == c.t0 || ti == c.t1;
	}
	double px = 0.0, py = 0.0, pz = 0.0;
	sepk_lj_pairs<TYPED, MIXED, FAST>(s, nbr, cnt, npad, c, t, sub, act, ti, fx, fy, fz, acc,
					   px, py, pz);
	sepk_pair_epilogue<OVERWRITE>(t, sub, n, npad, act, fx, fy, fz, px, py, pz, acc, s.f,
				      partial, lb, rows, frozen);
}

typedef void (*sepk_lj_kernel)(sepk_state, const int *, const int *, long, long,
			       sepk_lj, double *, long);

// qpos from pos for every slot (sepk_quant), after a position or charge
// upload or a change of box.
__global__ void k_quantize(sepk_state s, long npad, double q0, double q1, double q2)
{
	const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
	if (t < npad)
		s.qpos[t] = sepk_quant(s.pos[t], q0, q1, q2);
}

int sepk_fresh_qpos(sepdev *d, const double *L)
{
	if (!d->qpos_stale && d->qL[0] == L[0] && d->qL[1] == L[1] && d->qL[2] == L[2])
		return 0;
	k_quantize<<<sepk_blocks(d->npad), SEPK_BLOCK, 0, d->st>>>(
		d->s[0], d->npad, SEPK_QSCALE / L[0], SEPK_QSCALE / L[1], SEPK_QSCALE / L[2]);
	SEPK_LAUNCH_CHECK();
	for (int k = 0; k < 3; k++)
		d->qL[k] = L[k];
	d->qpos_stale = 0;
	return 0;
}

template <bool T, bool M, bool O>
static sepk_lj_kernel pick_lj3(bool fast)
{
	return fast ? k_lj<T, M, O, true> : k_lj<T, M, O, false>;
}

template <bool T, bool M>
static sepk_lj_kernel pick_lj(bool over, bool fast)
{
	return over ? pick_lj3<T, M, true>(fast) : pick_lj3<T, M, false>(fast);
}

// The fast image is exact for listed pairs when half the box exceeds the
// list cutoff plus the skin with room to spare (see sepk_wrap_fast and
// sepk_image).
static bool fast_image_ok(const sepdev *d, const double *L)
{
	if (!d->list_built)
		return false;
	// listed pairs start within the list cutoff and each atom moves at
	// most half the skin before a rebuild; twice the cutoff bounds both
	const double reach = 2.0 * sqrt(d->grid.rlist2);
	for (int k = 0; k < 3; k++)
		if (!(0.5 * L[k] > 1.05 * reach))
			return false;
	return true;
}

// One pair-force launch and its finishing task.
static int launch_lj(sepdev *d, const sepk_lj &c, int typed, int mixed, bool fast, int ret_slot,
		     int epot_assign)
{
	// first: claiming a region may launch a recorded pair call, which
	// consumes the pending f = 0
	int rc, region;
	if ((rc = sepk_term_region(d, &region)) || (rc = sepk_fork_point(d)))
		return rc;
	// owed bonded gathers go to f first (the sums keep their order)
	if ((rc = sepk_flush_gathers(d)))
		return rc;
	const bool over = d->f_zero_pending != 0;
	sepk_lj_kernel k;
	if (typed)
		k = mixed ? pick_lj<true, true>(over, fast) : pick_lj<true, false>(over, fast);
	else
		k = mixed ? pick_lj<false, true>(over, fast) : pick_lj<false, false>(over, fast);
	if ((rc = sepk_timer_begin(d, &d->t_pair)))
		return rc;
	const unsigned nb = sepk_blocks_xcd(d->n * SEPK_SUB);
	double *part = sepk_region(d, region);
	k<<<nb, SEPK_BLOCK, 0, d->st>>>(d->s[0], d->nbr, d->nbr_count, d->n, d->npad, c, part,
					  d->region_rows);
	SEPK_LAUNCH_CHECK();
	d->f_zero_pending = 0;
	if ((rc = sepk_timer_end(d, &d->t_pair)))
		return rc;
	if (!d->last_lj)
		d->last_lj = malloc(sizeof(sepk_lj));
	memcpy(d->last_lj, &c, sizeof c);
	d->last_lj_kernel = (const void *)(typed ? (mixed ? pick_lj<true, true>(true, fast)
							  : pick_lj<true, false>(true, fast))
					       : (mixed ? pick_lj<false, true>(true, fast)
							: pick_lj<false, false>(true, fast)));
	d->last_fused = 0;
	sepk_task f;
	memset(&f, 0, sizeof f);
	f.mode = SEPK_FIN_PAIR;
	f.region = region;
	f.nblk = (int)nb;
	f.nv = 7;
	f.epot_assign = epot_assign;
	sepk_task_ret(d, f, ret_slot);
	return sepk_queue_task(d, f);
}

extern "C" int sepdev_lj(sepdev *d, const sepdev_lj_args *a, int ret_slot)
{
	if (!d->list_built)
		return sepk_fail(SEP_GPU_ESTATE, "pair forces before a neighbour list was built");
	if (ret_slot < 0 || ret_slot >= d->nret)
		return sepk_fail(SEP_GPU_EARG, "ret slot %d", ret_slot);
	sepk_lj c;
	c.cf2 = a->cf2;
	c.A = a->eps48;
	c.nB = -(a->eps48 * a->awh);
	c.C = a->eps4;
	c.nD = -(a->eps4 * a->aw);
	c.sig2 = a->sig2;
	c.ushift = a->ushift;
	c.L0 = a->L[0];
	c.L1 = a->L[1];
	c.L2 = a->L[2];
	c.iL0 = 1.0 / a->L[0];
	c.iL1 = 1.0 / a->L[1];
	c.iL2 = 1.0 / a->L[2];
	c.qd0 = a->L[0] / SEPK_QSCALE;
	c.qd1 = a->L[1] / SEPK_QSCALE;
	c.qd2 = a->L[2] / SEPK_QSCALE;
	{
		// |dx~ - dx| <= one step per axis, so |r2~ - r2| <= q (2 sqrt(3) rc + 3 q)
		const double q = fmax(c.qd0, fmax(c.qd1, c.qd2));
		c.band = q * (4.0 * sqrt(a->cf2) + 4.0 * q) + 1e-12 * a->cf2;
		c.cf2lo = a->cf2 - c.band;
		c.cf2hi = a->cf2 + c.band;
	}
	c.Af = (float)c.A;
	c.nBf = (float)c.nB;
	c.Cf = (float)c.C;
	c.nDf = (float)c.nD;
	c.sig2f = (float)a->sig2;
	c.ushiftf = (float)a->ushift;
	c.t0 = a->t0;
	c.t1 = a->t1;
	int rc = sepk_flush_nh(d);
	if (rc || (a->mixed && (rc = sepk_fresh_qpos(d, a->L))))
		return rc;
	const bool over = d->f_zero_pending != 0;
	const bool fast = fast_image_ok(d, a->L);
	if (d->fuse_armed && !a->typed && over && !d->fused_pending) {
		// recorded: the step's leapfrog launches it fused with itself
		d->fused_pending = 1;
		d->fused_lj = c;
		d->fused_mixed = a->mixed;
		d->fused_fast = fast;
		d->fused_ret = ret_slot;
		d->fused_epot_assign = a->epot_assign;
		return 0;
	}
	if (d->pc_armed && !d->pc_pending && !d->fused_pending) {
		// recorded: a Coulomb call right after launches both terms
		d->pc_pending = 1;
		d->pc_lj = c;
		d->pc_mixed = a->mixed;
		d->pc_typed = a->typed;
		d->pc_fast = fast;
		d->pc_ret = ret_slot;
		d->pc_epot_assign = a->epot_assign;
		return 0;
	}
	return launch_lj(d, c, a->typed, a->mixed, fast, ret_slot, a->epot_assign);
}

// Launches a recorded pair call on its own (something other than the
// step's leapfrog needs its forces or its rows).
int sepk_flush_pair(sepdev *d)
{
	if (d->pc_pending) {
		d->pc_pending = 0;
		return launch_lj(d, d->pc_lj, d->pc_typed, d->pc_mixed, d->pc_fast != 0, d->pc_ret,
				 d->pc_epot_assign);
	}
	if (!d->fused_pending)
		return 0;
	d->fused_pending = 0;
	return launch_lj(d, d->fused_lj, 0, d->fused_mixed, d->fused_fast, d->fused_ret,
			 d->fused_epot_assign);
}

extern "C" int sepdev_fuse_step(sepdev *d, int on)
{
	d->fuse_armed = on != 0;
	return on ? 0 : sepk_flush_pair(d);
}

extern "C" int sepdev_fuse_pair_coulomb(sepdev *d, int on)
{
	d->pc_armed = on != 0;
	return on ? 0 : sepk_flush_pair(d);
}


// ---- shifted-force Coulomb (source/sepcoulomb.c:96-160) ---------------------

struct sepk_coul {
	double cf, cf2, icf, icf2;
	double L0, L1, L2, iL0, iL1, iL2;
	double qd0, qd1, qd2; // quantization step per axis (mixed form)
	float cff, icff, icf2f;
};

// Force factor and energy of a pair of charge product qq at squared distance r2
// (source/sepcoulomb.c:130-140): qq (1/r2 - 1/rc^2) / r and
// qq (1/r + (r - rc)/rc^2 - 1/rc).  r, 1/r, 1/r2 and the last division come
// from one hardware reciprocal square root (2^-24), a coupled Newton step and a
// residual correction each, which leaves every one of them at the rounding of
// the operation it stands for (against long double, r from 1e-6 to the cutoff
// 2.5, u = 2^-53: the force within 2.7 u |qq| (1/r^2 + 1/rc^2), where operations
// each at their own rounding may leave 9; the energy within a third of what they
// may); a square root and three divisions took three times the instructions, most
// of the FP64 walk's (a step of 96000 atoms of water: 251 -> 211 us).
__device__ __forceinline__ void sepk_coul_pair(const sepk_coul &c, double qq, double r2, double &ft,
					       double &e)
{
	const double y = __builtin_amdgcn_rsq(r2);
	double h = 0.5 * y, r = r2 * y;
	const double d = fma(-r, h, 0.5);
	r = fma(r, d, r);
	h = fma(h, d, h);
	r = fma(fma(-r, r, r2), h, r);
	double ri = 2.0 * h;
	ri = fma(ri, fma(-r, ri, 1.0), ri);
	double ri2 = ri * ri;
	ri2 = fma(ri2, fma(-r2, ri2, 1.0), ri2);
	const double a = qq * (ri2 - c.icf2);
	ft = a * ri;
	ft = fma(fma(-r, ft, a), ri, ft);
	// charges in one place: the energy stays infinite
	const bool zero = r2 == 0.0;
	e = qq * ((zero ? __builtin_inf() : ri) + ((zero ? 0.0 : r) - c.cf) * c.icf2 - c.icf);
}

// The mixed form of the pair loop below: positions and charges from the
// 16-byte quantized records (integer minimum image, charge as FP32 in w),
// r^2 and the cutoff test in FP64 from the exact integer differences, the
// pair force and energy in FP32 (hardware reciprocal square root, factored
// forms of the shifted-force terms), sums in FP64.  The charge test is the reference's |q| < DBL_EPSILON; the phantom's
// NaN charge fails it too.
__device__ __forceinline__ void sepk_coul_pairs_mixed(
	const sepk_state &s, const int *__restrict__ nbr, const int *__restrict__ cnt,
	long npad, const sepk_coul &c, long t, int sub, int4 qi, double &fx, double &fy,
	double &fz, double (&acc)[7])
{
	const float qif = __int_as_float(qi.w);
	const float epsf = (float)DBL_EPSILON;
	const int nbat = (cnt[t] + SEPK_PAD - 1) / SEPK_PAD;
	const size_t stride = (size_t)npad * SEPK_SUB;
	const int4 *lp = sepk_lane_list(nbr, t, sub);
	for (int b = 0; b < nbat; b++, lp += stride) {
		const int4 jb = *lp;
		const int j[SEPK_BATCH] = {jb.x, jb.y, jb.z, jb.w};
		int4 qj[SEPK_BATCH];
#pragma unroll
		for (int u = 0; u < SEPK_BATCH; u++)
			qj[u] = sepk_at(s.qpos, (unsigned)j[u]);
#pragma unroll
		for (int u = 0; u < SEPK_BATCH; u++) {
			const float qjf = __int_as_float(qj[u].w);
			if (!(fabsf(qjf) >= epsf))
				continue;
			const unsigned ux = (unsigned)qi.x, vx = (unsigned)qj[u].x;
			const unsigned uy = (unsigned)qi.y, vy = (unsigned)qj[u].y;
			const unsigned uz = (unsigned)qi.z, vz = (unsigned)qj[u].z;
			const int ix = (int)(ux - vx), iy = (int)(uy - vy), iz = (int)(uz - vz);
			const double dx = (double)ix * c.qd0;
			const double dy = (double)iy * c.qd1;
			const double dz = (double)iz * c.qd2;
			const double r2 = dx * dx + dy * dy + dz * dz;
			if (!(r2 < c.cf2))
				continue;
			// 1/r^2 - 1/rc^2 = (rc - r)(rc + r) / (r^2 rc^2) and
			// 1/r - 1/rc + (r - rc)/rc^2 = (rc - r)^2 / (r rc^2): the
			// reference's expressions without their cancellation near
			// the cutoff, which FP32 would carry into the energy sum
			const float r2f = (float)r2;
			const float ri = __builtin_amdgcn_rsqf(r2f);
			const float rf = r2f * ri;
			const float qq = qjf * qif;
			const float dc = c.cff - rf;
			const float qs = qq * c.icf2f * ri;
			const double ft = (double)(qs * (dc * (c.cff + rf)) * (ri * ri));
			const double e = (double)(qs * (dc * dc));
			fx = fma(ft, dx, fx);
			fy = fma(ft, dy, fy);
			fz = fma(ft, dz, fz);
			acc[0] += e;
			const bool bx = (ux < vx) != (ix < 0), by = (uy < vy) != (iy < 0),
				   bz = (uz < vz) != (iz < 0);
			if (bx | by | bz) {
				const double kx = bx ? (ix < 0 ? 1.0 : -1.0) : 0.0;
				const double ky = by ? (iy < 0 ? 1.0 : -1.0) : 0.0;
				const double kz = bz ? (iz < 0 ? 1.0 : -1.0) : 0.0;
				sepk_pair_cross(ft, dx, dy, dz, kx, ky, kz, c.L0, c.L1, c.L2, acc);
			}
		}
	}
}

template <bool OVERWRITE, bool FAST, bool MIXED>
__global__ __launch_bounds__(SEPK_BLOCK) void k_coulomb(
	sepk_state s, const int *__restrict__ nbr, const int *__restrict__ cnt,
	long n, long npad, sepk_coul c, double *partial, long rows)
{
	const long lb = sepk_xcd_block();
	const long t = lb * (SEPK_BLOCK / SEPK_SUB) + threadIdx.x / SEPK_SUB;
	const int sub = threadIdx.x % SEPK_SUB;
	const bool frozen = *s.err != 0;
	double fx = 0.0, fy = 0.0, fz = 0.0;
	double acc[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
	bool act = t < n;
	sepk_pos pi = {0.0, 0.0, 0.0, 0.0};
	if (act) {
		pi = s.pos[t];
		act = !(fabs(pi.q) < DBL_EPSILON);
	}
	if (MIXED) {
		int4 qi = make_int4(0, 0, 0, SEPK_QPHANTOM);
		if (act) {
			qi = s.qpos[t];
			sepk_coul_pairs_mixed(s, nbr, cnt, npad, c, t, sub, qi, fx, fy, fz, acc);
		}
		// the stress identity on the quantized positions
		const double px = act ? (double)(unsigned)qi.x * c.qd0 : 0.0;
		const double py = act ? (double)(unsigned)qi.y * c.qd1 : 0.0;
		const double pz = act ? (double)(unsigned)qi.z * c.qd2 : 0.0;
		sepk_pair_epilogue<OVERWRITE>(t, sub, n, npad, act, fx, fy, fz, px, py, pz, acc,
					      s.f, partial, lb, rows, frozen);
		return;
	}
	if (act) {
		const int nbat = (cnt[t] + SEPK_PAD - 1) / SEPK_PAD;
		const size_t stride = (size_t)npad * SEPK_SUB;
		const int4 *lp = sepk_lane_list(nbr, t, sub);
		const char *pb = (const char *)s.pos;
		for (int b = 0; b < nbat; b++, lp += stride) {
			const int4 jb = *lp;
			const int j[SEPK_BATCH] = {jb.x, jb.y, jb.z, jb.w};
			sepk_pos pj[SEPK_BATCH];
#pragma unroll
			for (int u = 0; u < SEPK_BATCH; u++)
				pj[u] = sepk_rec(pb, j[u]);
#pragma unroll
			for (int u = 0; u < SEPK_BATCH; u++) {
				// the phantom (charge 0) is skipped here
				if (fabs(pj[u].q) < DBL_EPSILON)
					continue;
				double kx, ky, kz;
				const double dx = sepk_image<FAST>(pi.x - pj[u].x, c.L0, c.iL0, kx);
				const double dy = sepk_image<FAST>(pi.y - pj[u].y, c.L1, c.iL1, ky);
				const double dz = sepk_image<FAST>(pi.z - pj[u].z, c.L2, c.iL2, kz);
				const double r2 = dx * dx + dy * dy + dz * dz;
				if (!(r2 < c.cf2))
					continue;
				double ft, e;
				sepk_coul_pair(c, pj[u].q * pi.q, r2, ft, e);
				sepk_pair_accumulate(ft, e, dx, dy, dz, kx, ky, kz, c.L0, c.L1, c.L2,
						     fx, fy, fz, acc);
			}
		}
	}
	sepk_pair_epilogue<OVERWRITE>(t, sub, n, npad, act, fx, fy, fz, pi.x, pi.y, pi.z, acc,
				      s.f, partial, lb, rows, frozen);
}

// ---- wide walks ------------------------------------------------------------------
//
// Four lanes an atom leave a small system waiting: each lane goes through its
// quarter of the list batch by batch, a gather's latency and a batch's
// arithmetic after the other, on a chip that is mostly empty.  A wide walk gives
// an atom 16 lanes, four for each of its four lanes: lane (g, sub) evaluates the
// batches g, g + 4, ... of lane sub, four of them at a time, with the gathers of
// the next four in flight.  The sums stay those of the walk by four lanes, bit
// for bit: a lane leaves its pairs' force factors, energies and separations in
// LDS, and the four lanes of one sub then each go through all four batches' pairs
// in list order for their own column -- the three force components and the
// energy, and two of the crossing stress each for three of them.  A pair left
// out stands there with factor, energy and separation zero, which add nothing.
// A wave holds 4 atoms and exchanges within itself; a workgroup, 16 atoms: its
// first wave takes their sums over as one wave of the kernel by four lanes does,
// and its row is that wave's (sepk_task::wide).
//
// An array is 32 bytes longer than its values, so that what the lanes of different
// g read from different arrays lies in different banks.
#define SEPK_WIDE_LEN (SEPK_BATCH * 64 + 4)
template <int NT>
struct sepk_wide_wave {
	double fe[NT][2][SEPK_WIDE_LEN]; // force factor, energy
	double d[3][SEPK_WIDE_LEN];
	unsigned cross[64]; // image count, two's complement in two bits an axis, a byte an entry
};

// per term: fx, fy, fz, e and the six crossing columns, by lane of the kernel by
// four lanes; then what else its lanes carry
template <int NT>
union sepk_wide_lds {
	sepk_wide_wave<NT> w[SEPK_BLOCK / 64];
	struct {
		double col[NT][10][64];
		int band[64];
	} r;
};

// one lane's evaluated batch
template <int NT>
struct sepk_wide_batch {
	double ft[NT][SEPK_BATCH], e[NT][SEPK_BATCH], d[3][SEPK_BATCH];
	unsigned cross;
};

// a lane's columns: its force component (or the energy) and crossing columns
template <int NT>
struct sepk_wide_acc {
	double m[NT], x0[NT], x1[NT];
};

__device__ __forceinline__ unsigned sepk_cross_code(double kx, double ky, double kz)
{
	return ((int)kx & 3) | ((int)ky & 3) << 2 | ((int)kz & 3) << 4;
}

__device__ __forceinline__ void sepk_wave_lds_fence()
{
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
}

// The four batches' pairs of an atom's sub, in list order, into a lane's columns;
// CROSS: some pair of the wave crosses the box.  Lanes g = 0, 1, 2 take the
// crossing columns xx, xy | xz, yy | yz, zz: separation along axes sa, g, image
// along ia, ib; a pair that does not cross has image 0 and adds nothing.
template <bool CROSS, int NT>
__device__ __forceinline__ void sepk_wide_columns(const sepk_wide_wave<NT> &w, double L0, double L1,
						  double L2, sepk_wide_acc<NT> &acc)
{
	const int ln = threadIdx.x & 63, g = (ln >> 2) & 3;
	const int first = ln & ~12; // lane (0, sub) of the atom
	const bool comp = g < 3;
	const double *pd = w.d[comp ? g : 0] + first;
	const double *ps = w.d[g == 2 ? 1 : 0] + first;
	const int ia = g == 0 ? 0 : 4, ib = g < 2 ? 2 : 4; // bits of the image axes
	const double La = g == 0 ? L0 : L2, Lb = g < 2 ? L1 : L2;
	const double *pa[NT];
#pragma unroll
	for (int k = 0; k < NT; k++)
		pa[k] = w.fe[k][comp ? 0 : 1] + first;
#pragma unroll
	for (int q = 0; q < 4; q++) {
		const unsigned code = CROSS ? w.cross[first + 4 * q] : 0u;
#pragma unroll
		for (int u = 0; u < SEPK_BATCH; u++) {
			const int i = u * 64 + 4 * q;
			const double d = comp ? pd[i] : 1.0;
			double a[NT];
#pragma unroll
			for (int k = 0; k < NT; k++) {
				a[k] = pa[k][i];
				acc.m[k] = fma(a[k], d, acc.m[k]);
			}
			if (CROSS) {
				const double ka = La * (double)((int)(code << (30 - 8 * u - ia)) >> 30);
				const double kb = Lb * (double)((int)(code << (30 - 8 * u - ib)) >> 30);
				const double da = ps[i];
#pragma unroll
				for (int k = 0; k < NT; k++) {
					acc.x0[k] = fma(-a[k] * da, ka, acc.x0[k]);
					acc.x1[k] = fma(-a[k] * d, kb, acc.x1[k]);
				}
			}
		}
	}
}

// Adds the wave's evaluated batches to the lanes' columns.
template <int NT>
__device__ __forceinline__ void sepk_wide_add(sepk_wide_wave<NT> &w, const sepk_wide_batch<NT> &b,
					      double L0, double L1, double L2,
					      sepk_wide_acc<NT> &acc)
{
	const int ln = threadIdx.x & 63;
#pragma unroll
	for (int u = 0; u < SEPK_BATCH; u++) {
#pragma unroll
		for (int k = 0; k < NT; k++) {
			w.fe[k][0][u * 64 + ln] = b.ft[k][u];
			w.fe[k][1][u * 64 + ln] = b.e[k][u];
		}
#pragma unroll
		for (int k = 0; k < 3; k++)
			w.d[k][u * 64 + ln] = b.d[k][u];
	}
	w.cross[ln] = b.cross;
	sepk_wave_lds_fence();
	if (__ballot(b.cross != 0))
		sepk_wide_columns<true>(w, L0, L1, L2, acc);
	else
		sepk_wide_columns<false>(w, L0, L1, L2, acc);
	sepk_wave_lds_fence(); // read before the next batches replace it
}

// Hands the block's columns to its first wave, lane (16 atoms) x 4 as in the
// kernel by four lanes: f and acc (energy, crossing stress) of each term, and
// band.  The other waves return false; they are done.
template <int NT>
__device__ __forceinline__ bool sepk_wide_hand_over(sepk_wide_lds<NT> &lds,
						    const sepk_wide_acc<NT> &w, bool &band,
						    double (&f)[NT][3], double (&acc)[NT][7])
{
	const int g = (threadIdx.x >> 2) & 3;
	const int at = (threadIdx.x >> 4) * 4 + (threadIdx.x & 3);
	__syncthreads(); // the walks are over
	if (threadIdx.x < 64)
		lds.r.band[threadIdx.x] = 0;
#pragma unroll
	for (int k = 0; k < NT; k++) {
		lds.r.col[k][g][at] = w.m[k];
		if (g < 3) {
			lds.r.col[k][4 + 2 * g][at] = w.x0[k];
			lds.r.col[k][5 + 2 * g][at] = w.x1[k];
		}
	}
	__syncthreads();
	if (band)
		lds.r.band[at] = 1; // any of the four lanes: the same value
	__syncthreads();
	if (threadIdx.x >= 64)
		return false;
	band = lds.r.band[threadIdx.x] != 0;
#pragma unroll
	for (int k = 0; k < NT; k++) {
#pragma unroll
		for (int i = 0; i < 3; i++)
			f[k][i] = lds.r.col[k][i][threadIdx.x];
#pragma unroll
		for (int i = 0; i < 7; i++)
			acc[k][i] = lds.r.col[k][3 + i][threadIdx.x];
	}
	return true;
}

// The batches of atom t's lane (g, sub): fetch(j, rec) gathers a batch's records,
// eval(rec, batch) evaluates it.  The records of the next batch and the indices
// of the one after it are under way while one is evaluated.
template <int NT, class REC, class FETCH, class EVAL>
__device__ __forceinline__ void sepk_wide_walk(sepk_wide_wave<NT> &w, const int *__restrict__ nbr,
					       const int *__restrict__ cnt, long npad, int maxbat,
					       long t, bool act, double L0, double L1, double L2,
					       FETCH fetch, EVAL eval, sepk_wide_acc<NT> &acc)
{
	const int g = (threadIdx.x >> 2) & 3, sub = threadIdx.x & 3;
	const size_t stride = (size_t)npad * SEPK_SUB;
	const int4 *lp = sepk_lane_list(nbr, act ? t : 0, sub);
	// the first indices go out with the count: the allocation holds them,
	// whatever the list's length
	int4 j0 = make_int4(0, 0, 0, 0), j1 = j0;
	if (act && g < maxbat)
		j0 = lp[g * stride];
	if (act && g + 4 < maxbat)
		j1 = lp[(g + 4) * stride];
	const int nbat = act ? (cnt[t] + SEPK_PAD - 1) / SEPK_PAD : 0;
	REC now[SEPK_BATCH], next[SEPK_BATCH];
	if (g < nbat)
		fetch(j0, now);
	for (int b = g; __ballot(b - g < nbat); b += 4) {
		if (b + 4 < nbat)
			fetch(j1, next);
		if (b + 8 < nbat)
			j1 = lp[(b + 8) * stride];
		sepk_wide_batch<NT> v;
		v.cross = 0;
#pragma unroll
		for (int u = 0; u < SEPK_BATCH; u++) {
#pragma unroll
			for (int k = 0; k < NT; k++)
				v.ft[k][u] = v.e[k][u] = 0.0;
#pragma unroll
			for (int k = 0; k < 3; k++)
				v.d[k][u] = 0.0;
		}
		if (b < nbat)
			eval(now, v);
		sepk_wide_add(w, v, L0, L1, L2, acc);
#pragma unroll
		for (int u = 0; u < SEPK_BATCH; u++)
			now[u] = next[u];
	}
}

template <int NT>
__device__ __forceinline__ sepk_wide_acc<NT> sepk_wide_zero()
{
	sepk_wide_acc<NT> a;
#pragma unroll
	for (int k = 0; k < NT; k++)
		a.m[k] = a.x0[k] = a.x1[k] = 0.0;
	return a;
}

// The walk of k_lj_coul by wide walk: true in the block's first wave, whose lane
// then holds what the lane of k_lj_coul holds for atom 16 lb + lane / 4, lane
// sub = lane % 4.
template <bool TYPED, bool MIXED, bool FAST>
__device__ __forceinline__ bool sepk_lj_coul_pairs_wide(
	sepk_wide_lds<2> &lds, const sepk_state &s, const int *__restrict__ nbr,
	const int *__restrict__ cnt, long n, long npad, int maxbat, const sepk_lj &c,
	const sepk_coul &cc, long lb, double (&f)[2][3], double (&acc)[2][7], bool &band)
{
	const long t = lb * (SEPK_BLOCK / 16) + threadIdx.x / 16;
	const bool act = t < n;
	sepk_wide_wave<2> &w = lds.w[threadIdx.x >> 6];
	sepk_wide_acc<2> wa = sepk_wide_zero<2>();
	band = false;
	const signed char ti = TYPED && act ? s.type[t] : 0;
	const bool act_l = act && (!TYPED || ti == c.t0 || ti == c.t1);
	const sepk_pos pi = act ? s.pos[t] : sepk_pos{0.0, 0.0, 0.0, 0.0};
	const bool act_c = act && !(fabs(pi.q) < DBL_EPSILON);
	const bool walks = act_l || act_c;
	const auto typed = [&](signed char tj) {
		return !TYPED || (ti == c.t0 && tj == c.t1) || (ti == c.t1 && tj == c.t0);
	};
	if (MIXED) {
		struct rec {
			int4 q;
			signed char t;
		};
		const int4 qi = walks ? s.qpos[t] : make_int4(0, 0, 0, SEPK_QPHANTOM);
		const float qif = __int_as_float(qi.w);
		const float epsf = (float)DBL_EPSILON;
		sepk_wide_walk<2, rec>(
			w, nbr, cnt, npad, maxbat, t, walks, c.L0, c.L1, c.L2,
			[&](const int4 &jb, rec (&r)[SEPK_BATCH]) {
				const int j[SEPK_BATCH] = {jb.x, jb.y, jb.z, jb.w};
#pragma unroll
				for (int u = 0; u < SEPK_BATCH; u++) {
					r[u].q = sepk_at(s.qpos, (unsigned)j[u]);
					r[u].t = TYPED ? s.type[(unsigned)j[u]] : 0;
				}
			},
			[&](const rec (&r)[SEPK_BATCH], sepk_wide_batch<2> &v) {
#pragma unroll
				for (int u = 0; u < SEPK_BATCH; u++) {
					const unsigned ux = (unsigned)qi.x, vx = (unsigned)r[u].q.x;
					const unsigned uy = (unsigned)qi.y, vy = (unsigned)r[u].q.y;
					const unsigned uz = (unsigned)qi.z, vz = (unsigned)r[u].q.z;
					const int ix = (int)(ux - vx), iy = (int)(uy - vy),
						  iz = (int)(uz - vz);
					const double dx = (double)ix * c.qd0;
					const double dy = (double)iy * c.qd1;
					const double dz = (double)iz * c.qd2;
					const double r2 = dx * dx + dy * dy + dz * dz;
					const bool lj = act_l && typed(r[u].t) && r[u].q.w != SEPK_QPHANTOM;
					if (lj && !(r2 < c.cf2lo))
						band |= r2 < c.cf2hi;
					const bool in_l = lj && r2 < c.cf2lo;
					if (in_l) {
						const float q = c.sig2f * __builtin_amdgcn_rcpf((float)r2);
						const float q3 = q * q * q;
						v.ft[0][u] = (double)(fmaf(c.Af, q3, c.nBf) * q3 * q);
						v.e[0][u] = (double)fmaf(fmaf(c.Cf, q3, c.nDf), q3, c.ushiftf);
					}
					const float qjf = __int_as_float(r[u].q.w);
					const bool in_c = act_c && fabsf(qjf) >= epsf && r2 < cc.cf2;
					// most listed pairs are inside: evaluated without a
					// branch, the four entries' chains overlap
					const float r2f = (float)r2;
					const float ri = __builtin_amdgcn_rsqf(r2f);
					const float rf = r2f * ri;
					const float qq = qjf * qif;
					const float dc = cc.cff - rf;
					const float qs = qq * cc.icf2f * ri;
					v.ft[1][u] = in_c ? (double)(qs * (dc * (cc.cff + rf)) * (ri * ri)) : 0.0;
					v.e[1][u] = in_c ? (double)(qs * (dc * dc)) : 0.0;
					v.d[0][u] = dx;
					v.d[1][u] = dy;
					v.d[2][u] = dz;
					if (in_l || in_c) {
						const bool bx = (ux < vx) != (ix < 0), by = (uy < vy) != (iy < 0),
							   bz = (uz < vz) != (iz < 0);
						v.cross |= ((bx ? (ix < 0 ? 1u : 3u) : 0u) |
							    (by ? (iy < 0 ? 4u : 12u) : 0u) |
							    (bz ? (iz < 0 ? 16u : 48u) : 0u))
							   << (8 * u);
					}
				}
			},
			wa);
	} else {
		struct rec {
			sepk_pos p;
			signed char t;
		};
		const char *pb = (const char *)s.pos;
		sepk_wide_walk<2, rec>(
			w, nbr, cnt, npad, maxbat, t, walks, c.L0, c.L1, c.L2,
			[&](const int4 &jb, rec (&r)[SEPK_BATCH]) {
				const int j[SEPK_BATCH] = {jb.x, jb.y, jb.z, jb.w};
#pragma unroll
				for (int u = 0; u < SEPK_BATCH; u++) {
					r[u].p = sepk_rec(pb, j[u]);
					r[u].t = TYPED ? s.type[(unsigned)j[u]] : 0;
				}
			},
			[&](const rec (&r)[SEPK_BATCH], sepk_wide_batch<2> &v) {
#pragma unroll
				for (int u = 0; u < SEPK_BATCH; u++) {
					const sepk_pos &p = r[u].p;
					double kx, ky, kz;
					const double dx = sepk_image<FAST>(pi.x - p.x, c.L0, c.iL0, kx);
					const double dy = sepk_image<FAST>(pi.y - p.y, c.L1, c.iL1, ky);
					const double dz = sepk_image<FAST>(pi.z - p.z, c.L2, c.iL2, kz);
					const double r2 = dx * dx + dy * dy + dz * dz;
					const bool in_l = act_l && typed(r[u].t) && r2 < c.cf2;
					if (in_l) {
						const double q = c.sig2 * sepk_recip(r2);
						const double q3 = q * q * q;
						v.ft[0][u] = fma(c.A, q3, c.nB) * q3 * q;
						v.e[0][u] = fma(fma(c.C, q3, c.nD), q3, c.ushift);
					}
					const bool in_c = act_c && !(fabs(p.q) < DBL_EPSILON) && r2 < cc.cf2;
					// most listed pairs are inside: evaluated without a
					// branch, the four entries' chains overlap
					double ft, e;
					sepk_coul_pair(cc, p.q * pi.q, in_c ? r2 : 1.0, ft, e);
					v.ft[1][u] = in_c ? ft : 0.0;
					v.e[1][u] = in_c ? e : 0.0;
					if (in_l || in_c) {
						v.d[0][u] = dx;
						v.d[1][u] = dy;
						v.d[2][u] = dz;
						v.cross |= sepk_cross_code(kx, ky, kz) << (8 * u);
					}
				}
			},
			wa);
	}
	return sepk_wide_hand_over<2>(lds, wa, band, f, acc);
}

// The end of k_lj_coul, from each lane's sums of the two terms: the force as the
// two calls would leave it, and the block's (WIDE: the wave's) row of each term.
template <bool OVERWRITE, bool MIXED, bool WIDE>
__device__ __forceinline__ void sepk_lj_coul_finish(
	const sepk_state &s, long n, long npad, const sepk_lj &c, long t, int sub, bool act_l,
	bool act_c, bool frozen, const sepk_pos &pi, const int4 &qi, double (&fl)[3],
	double (&fc)[3], double (&al)[7], double (&ac)[7], double *part_lj, double *part_c,
	long row, long rows)
{
	// the two epilogues of sepk_pair_epilogue, the second adding to the first
#pragma unroll
	for (int k = 0; k < 3; k++) {
		fl[k] = sepk_atom_sum(fl[k]);
		fc[k] = sepk_atom_sum(fc[k]);
	}
	if (t < n && sub == 0 && !frozen) {
		for (int k = 0; k < 3; k++) {
			double v = OVERWRITE ? fl[k] : s.f[k * npad + t];
			if (!OVERWRITE && act_l)
				v += fl[k];
			if (act_c)
				v += fc[k];
			s.f[k * npad + t] = v;
		}
	}
	// the stress identity's positions: quantized (mixed) or FP64
	const double px = MIXED ? (double)(unsigned)qi.x * c.qd0 : pi.x;
	const double py = MIXED ? (double)(unsigned)qi.y * c.qd1 : pi.y;
	const double pz = MIXED ? (double)(unsigned)qi.z * c.qd2 : pi.z;
	if (act_l && sub == 0) {
		const double gx = 2.0 * fl[0], gy = 2.0 * fl[1], gz = 2.0 * fl[2];
		al[1] = fma(gx, px, al[1]);
		al[2] = fma(gx, py, al[2]);
		al[3] = fma(gx, pz, al[3]);
		al[4] = fma(gy, py, al[4]);
		al[5] = fma(gy, pz, al[5]);
		al[6] = fma(gz, pz, al[6]);
	}
	if (act_c && sub == 0) {
		const double gx = 2.0 * fc[0], gy = 2.0 * fc[1], gz = 2.0 * fc[2];
		ac[1] = fma(gx, px, ac[1]);
		ac[2] = fma(gx, py, ac[2]);
		ac[3] = fma(gx, pz, ac[3]);
		ac[4] = fma(gy, py, ac[4]);
		ac[5] = fma(gy, pz, ac[5]);
		ac[6] = fma(gz, pz, ac[6]);
	}
	double v[14];
#pragma unroll
	for (int k = 0; k < 7; k++) {
		v[k] = al[k];
		v[7 + k] = ac[k];
	}
	const auto out = [=](int i, double r) {
		(i < 7 ? part_lj : part_c)[(size_t)(i < 7 ? i : i - 7) * rows + row] = r;
	};
	if constexpr (WIDE)
		sepk_wave_reduce<false>(v, 0.0, out);
	else
		sepk_block_reduce<false>(v, 0.0, out);
}

// A pair call (LJ, typed or not) and the shifted-force Coulomb call right
// after it, in either form, in one walk of the list: one gather of each
// neighbour's record serves both terms.  Each term keeps its own force sum,
// energy, crossing stress and partial rows, accumulated entry by entry in
// the order of its own kernel (k_lj, k_coulomb), and the atom's force is
// written as the two calls would leave it: the LJ sum (over or added to f),
// then the Coulomb sum added.  The results are those of the two launches,
// bit for bit.
template <bool TYPED, bool OVERWRITE, bool MIXED, bool FAST>
__global__ __launch_bounds__(SEPK_BLOCK) void k_lj_coul(
	sepk_state s, const int *__restrict__ nbr, const int *__restrict__ cnt, long n,
	long npad, sepk_lj c, sepk_coul cc, double *part_lj, double *part_c, long rows)
{
	const long lb = sepk_xcd_block();
	const long t = lb * (SEPK_BLOCK / SEPK_SUB) + threadIdx.x / SEPK_SUB;
	const int sub = threadIdx.x % SEPK_SUB;
	const bool frozen = *s.err != 0;
	double fl[3] = {0.0, 0.0, 0.0}, fc[3] = {0.0, 0.0, 0.0};
	double al[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
	double ac[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
	bool act_l = t < n, act_c = t < n;
	signed char ti = 0;
	if (act_l && TYPED) {
		ti = s.type[t];
		act_l = ti == c.t0 || ti == c.t1;
	}
	sepk_pos pi = {0.0, 0.0, 0.0, 0.0};
	if (act_l || act_c)
		pi = s.pos[t];
	if (act_c)
		act_c = !(fabs(pi.q) < DBL_EPSILON);
	int4 qi = make_int4(0, 0, 0, SEPK_QPHANTOM);
	if (!MIXED && (act_l || act_c)) {
		// the FP64 loops of sepk_lj_pairs and k_coulomb on 32-byte records
		const int nbat = (cnt[t] + SEPK_PAD - 1) / SEPK_PAD;
		const size_t stride = (size_t)npad * SEPK_SUB;
		const int4 *lp = sepk_wave_list(nbr, t, sub);
		const unsigned ln = threadIdx.x & 63;
		const char *pb = (const char *)s.pos;
		// batch b + 1 in flight while batch b is computed, as above
		int4 jb = sepk_at(lp, ln);
		for (int b = 0; b < nbat; b++) {
			const int j[SEPK_BATCH] = {jb.x, jb.y, jb.z, jb.w};
			sepk_pos pj[SEPK_BATCH];
			signed char tj[SEPK_BATCH];
#pragma unroll
			for (int u = 0; u < SEPK_BATCH; u++) {
				pj[u] = sepk_rec(pb, j[u]);
				if (TYPED)
					tj[u] = s.type[(unsigned)j[u]];
			}
			// the wave's last batch reloads itself (a cache hit)
			if (__ballot(b + 1 < nbat))
				lp += stride;
			jb = sepk_at(lp, ln);
#pragma unroll
			for (int u = 0; u < SEPK_BATCH; u++) {
				double kx, ky, kz;
				const double dx = sepk_image<FAST>(pi.x - pj[u].x, c.L0, c.iL0, kx);
				const double dy = sepk_image<FAST>(pi.y - pj[u].y, c.L1, c.iL1, ky);
				const double dz = sepk_image<FAST>(pi.z - pj[u].z, c.L2, c.iL2, kz);
				const double r2 = dx * dx + dy * dy + dz * dz;
				const bool tl = !TYPED || (ti == c.t0 && tj[u] == c.t1) ||
						(ti == c.t1 && tj[u] == c.t0);
				if (act_l && tl && r2 < c.cf2) {
					const double q = c.sig2 * sepk_recip(r2);
					const double q3 = q * q * q;
					const double ft = fma(c.A, q3, c.nB) * q3 * q;
					const double e = fma(fma(c.C, q3, c.nD), q3, c.ushift);
					sepk_pair_accumulate(ft, e, dx, dy, dz, kx, ky, kz, c.L0, c.L1, c.L2,
							     fl[0], fl[1], fl[2], al);
				}
				if (act_c && !(fabs(pj[u].q) < DBL_EPSILON) && r2 < cc.cf2) {
					double ft, e;
					sepk_coul_pair(cc, pj[u].q * pi.q, r2, ft, e);
					sepk_pair_accumulate(ft, e, dx, dy, dz, kx, ky, kz, cc.L0, cc.L1,
							     cc.L2, fc[0], fc[1], fc[2], ac);
				}
			}
		}
	}
	if (MIXED && (act_l || act_c)) {
		qi = s.qpos[t];
		const float qif = __int_as_float(qi.w);
		const float epsf = (float)DBL_EPSILON;
		const int nbat = (cnt[t] + SEPK_PAD - 1) / SEPK_PAD;
		const size_t stride = (size_t)npad * SEPK_SUB;
		const int4 *lp = sepk_wave_list(nbr, t, sub);
		const unsigned ln = threadIdx.x & 63;
		bool band = false;
		int4 jb = sepk_at(lp, ln); // batch b + 1 in flight, as above
		for (int b = 0; b < nbat; b++) {
			const int j[SEPK_BATCH] = {jb.x, jb.y, jb.z, jb.w};
			int4 qj[SEPK_BATCH];
			signed char tj[SEPK_BATCH];
#pragma unroll
			for (int u = 0; u < SEPK_BATCH; u++) {
				qj[u] = sepk_at(s.qpos, (unsigned)j[u]);
				if (TYPED)
					tj[u] = s.type[(unsigned)j[u]];
			}
			// the wave's last batch reloads itself (a cache hit)
			if (__ballot(b + 1 < nbat))
				lp += stride;
			jb = sepk_at(lp, ln);
#pragma unroll
			for (int u = 0; u < SEPK_BATCH; u++) {
				const unsigned ux = (unsigned)qi.x, vx = (unsigned)qj[u].x;
				const unsigned uy = (unsigned)qi.y, vy = (unsigned)qj[u].y;
				const unsigned uz = (unsigned)qi.z, vz = (unsigned)qj[u].z;
				const int ix = (int)(ux - vx), iy = (int)(uy - vy), iz = (int)(uz - vz);
				const double dx = (double)ix * c.qd0;
				const double dy = (double)iy * c.qd1;
				const double dz = (double)iz * c.qd2;
				const double r2 = dx * dx + dy * dy + dz * dz;
				const bool bx = (ux < vx) != (ix < 0), by = (uy < vy) != (iy < 0),
					   bz = (uz < vz) != (iz < 0);
				const double kx = bx ? (ix < 0 ? 1.0 : -1.0) : 0.0;
				const double ky = by ? (iy < 0 ? 1.0 : -1.0) : 0.0;
				const double kz = bz ? (iz < 0 ? 1.0 : -1.0) : 0.0;
				// the LJ term as in sepk_lj_pairs, pairs near the cutoff
				// left to sepk_lj_mixed_band after the loop
				const bool tl = !TYPED || (ti == c.t0 && tj[u] == c.t1) ||
						(ti == c.t1 && tj[u] == c.t0);
				const bool lj = act_l && tl && qj[u].w != SEPK_QPHANTOM;
				if (lj && !(r2 < c.cf2lo))
					band |= r2 < c.cf2hi;
				if (lj && r2 < c.cf2lo) {
					const float q = c.sig2f * __builtin_amdgcn_rcpf((float)r2);
					const float q3 = q * q * q;
					const double ft = (double)(fmaf(c.Af, q3, c.nBf) * q3 * q);
					const double e = (double)fmaf(fmaf(c.Cf, q3, c.nDf), q3, c.ushiftf);
					fl[0] = fma(ft, dx, fl[0]);
					fl[1] = fma(ft, dy, fl[1]);
					fl[2] = fma(ft, dz, fl[2]);
					al[0] += e;
					if (bx | by | bz)
						sepk_pair_cross(ft, dx, dy, dz, kx, ky, kz, c.L0, c.L1, c.L2, al);
				}
				// the Coulomb term as in sepk_coul_pairs_mixed
				const float qjf = __int_as_float(qj[u].w);
				if (act_c && fabsf(qjf) >= epsf && r2 < cc.cf2) {
					const float r2f = (float)r2;
					const float ri = __builtin_amdgcn_rsqf(r2f);
					const float rf = r2f * ri;
					const float qq = qjf * qif;
					const float dc = cc.cff - rf;
					const float qs = qq * cc.icf2f * ri;
					const double ft = (double)(qs * (dc * (cc.cff + rf)) * (ri * ri));
					const double e = (double)(qs * (dc * dc));
					fc[0] = fma(ft, dx, fc[0]);
					fc[1] = fma(ft, dy, fc[1]);
					fc[2] = fma(ft, dz, fc[2]);
					ac[0] += e;
					if (bx | by | bz)
						sepk_pair_cross(ft, dx, dy, dz, kx, ky, kz, cc.L0, cc.L1, cc.L2, ac);
				}
			}
		}
		if (band)
			sepk_lj_mixed_band<TYPED, FAST>(s, nbr, cnt, npad, c, t, sub, ti, qi, fl[0],
							fl[1], fl[2], al);
	}
	sepk_lj_coul_finish<OVERWRITE, MIXED, false>(s, n, npad, c, t, sub, act_l, act_c, frozen, pi, qi,
						     fl, fc, al, ac, part_lj, part_c, lb, rows);
}

// k_lj_coul by wide walk (maxbat: batches a list's allocation holds), for the
// systems that sepk_wide chooses.  The walk by four lanes is a chain of 26 batches
// in 0.4 wavefronts a SIMD at 6000 atoms of water; this one is 7 rounds in 1.5.
// What bounds it is the exchange through LDS.
template <bool TYPED, bool OVERWRITE, bool MIXED, bool FAST>
__global__ __launch_bounds__(SEPK_BLOCK) void k_lj_coul_wide(
	sepk_state s, const int *__restrict__ nbr, const int *__restrict__ cnt, long n,
	long npad, int maxbat, sepk_lj c, sepk_coul cc, double *part_lj, double *part_c, long rows)
{
	__shared__ sepk_wide_lds<2> lds;
	const long lb = sepk_xcd_block();
	const bool frozen = *s.err != 0;
	double f[2][3], acc[2][7];
	bool band;
	if (!sepk_lj_coul_pairs_wide<TYPED, MIXED, FAST>(lds, s, nbr, cnt, n, npad, maxbat, c, cc, lb, f,
							 acc, band))
		return;
	const long t = lb * (SEPK_BLOCK / 16) + threadIdx.x / SEPK_SUB;
	const int sub = threadIdx.x % SEPK_SUB;
	bool act_l = t < n, act_c = t < n;
	signed char ti = 0;
	if (act_l && TYPED) {
		ti = s.type[t];
		act_l = ti == c.t0 || ti == c.t1;
	}
	sepk_pos pi = {0.0, 0.0, 0.0, 0.0};
	if (t < n)
		pi = s.pos[t];
	if (act_c)
		act_c = !(fabs(pi.q) < DBL_EPSILON);
	int4 qi = make_int4(0, 0, 0, SEPK_QPHANTOM);
	if (MIXED && (act_l || act_c)) {
		qi = s.qpos[t];
		if (band)
			sepk_lj_mixed_band<TYPED, FAST>(s, nbr, cnt, npad, c, t, sub, ti, qi, f[0][0],
							f[0][1], f[0][2], acc[0]);
	}
	sepk_lj_coul_finish<OVERWRITE, MIXED, true>(s, n, npad, c, t, sub, act_l, act_c, frozen, pi, qi,
						    f[0], f[1], acc[0], acc[1], part_lj, part_c, lb,
						    rows);
}

// Whether 16 lanes an atom take the walk.  Its workgroups (59 KB of LDS, two a CU)
// stop being resident all at once at SEPK_WIDE_ATOMS; and a short list leaves most
// of an atom's lanes without a batch, while there are four times the waves.  How
// long the lists are the host knows from their allocation, twice the expected mean
// and 64.  Per step, four lanes -> 16 (us, FP64; mixed within 1 of it), by mean
// list length:
//   9 (room 96)     1000 atoms 16.3 -> 18.1, 8192 17.4 -> 20.9:       never
//   30 (128)        1000 18.9 -> 18.3, 3000 19.9 -> 18.7, 5000 20.3 -> 20.4, 8192 20.3 -> 21.2
//   72 (224)        1000 22.5 -> 20.8, 3000 22.7 -> 21.1, 5000 22.7 -> 23.9, 8192 23.0 -> 24.7
//                                                                     up to half the atoms
//   121 (320)       1000 27.6 -> 22.7, 5000 27.1 -> 25.9, 8192 27.0 -> 26.5
//   water, 413      3000 79 -> 48, 6000 86 -> 63, 8000 84 -> 62; past the line 9000 85 -> 76
//                   (mixed 78 -> 77), 16000 90 -> 97
static bool sepk_wide(const sepdev *d)
{
	return d->n <= (d->cap >= 256 ? SEPK_WIDE_ATOMS : d->cap >= 128 ? SEPK_WIDE_ATOMS / 2 : 0);
}

// The recorded pair call and this Coulomb call as one k_lj_coul launch,
// each with its own term region and finishing task, queued in call order.
static int launch_lj_coul(sepdev *d, const sepk_coul &cc, int ret_slot)
{
	d->pc_pending = 0;
	int rc;
	// two distinct free term regions (the queue is finished first if not)
	int r1 = -1, r2 = -1;
	for (int r = SEPK_R_PAIR; r < SEPK_R_PAIR + SEPK_NTERM && r2 < 0; r++) {
		bool held = false;
		for (int i = 0; i < d->npending; i++)
			held = held || d->pending[i].region == r;
		if (!held) {
			if (r1 < 0)
				r1 = r;
			else
				r2 = r;
		}
	}
	if (r2 < 0) {
		d->fork_ready = 0;
		if ((rc = sepk_flush_tasks(d)))
			return rc;
		r1 = SEPK_R_PAIR;
		r2 = SEPK_R_PAIR + 1;
	}
	if ((rc = sepk_fork_point(d)) || (rc = sepk_flush_gathers(d)))
		return rc;
	const bool over = d->f_zero_pending != 0;
#define SEPK_LJ_COUL(K)                                                                          \
	{{{{K<false, false, false, false>, K<false, false, false, true>},                        \
	   {K<false, false, true, false>, K<false, false, true, true>}},                         \
	  {{K<false, true, false, false>, K<false, true, false, true>},                          \
	   {K<false, true, true, false>, K<false, true, true, true>}}},                          \
	 {{{K<true, false, false, false>, K<true, false, false, true>},                          \
	   {K<true, false, true, false>, K<true, false, true, true>}},                           \
	  {{K<true, true, false, false>, K<true, true, false, true>},                            \
	   {K<true, true, true, false>, K<true, true, true, true>}}}}
	typedef void (*kfn)(sepk_state, const int *, const int *, long, long, sepk_lj, sepk_coul,
			    double *, double *, long);
	typedef void (*wfn)(sepk_state, const int *, const int *, long, long, int, sepk_lj,
			    sepk_coul, double *, double *, long);
	static const kfn table[2][2][2][2] = SEPK_LJ_COUL(k_lj_coul);
	static const wfn wtable[2][2][2][2] = SEPK_LJ_COUL(k_lj_coul_wide);
#undef SEPK_LJ_COUL
	const bool wide = sepk_wide(d);
	const int kt = d->pc_typed ? 1 : 0, ko = over ? 1 : 0, km = d->pc_mixed ? 1 : 0,
		  kf = d->pc_fast ? 1 : 0;
	const unsigned nb = sepk_blocks_xcd(d->n * SEPK_SUB);
	if (wide)
		wtable[kt][ko][km][kf]<<<4 * nb, SEPK_BLOCK, 0, d->st>>>(
			d->s[0], d->nbr, d->nbr_count, d->n, d->npad, d->cap / SEPK_PAD, d->pc_lj, cc,
			sepk_region(d, r1), sepk_region(d, r2), d->region_rows);
	else
		table[kt][ko][km][kf]<<<nb, SEPK_BLOCK, 0, d->st>>>(
			d->s[0], d->nbr, d->nbr_count, d->n, d->npad, d->pc_lj, cc,
			sepk_region(d, r1), sepk_region(d, r2), d->region_rows);
	SEPK_LAUNCH_CHECK();
	d->f_zero_pending = 0;
	d->last_fused = 0;
	sepk_task f;
	memset(&f, 0, sizeof f);
	f.mode = SEPK_FIN_PAIR;
	f.region = r1;
	f.nblk = (int)nb;
	f.nv = 7;
	f.wide = wide;
	f.epot_assign = d->pc_epot_assign;
	sepk_task_ret(d, f, d->pc_ret);
	if ((rc = sepk_queue_task(d, f)))
		return rc;
	memset(&f, 0, sizeof f);
	f.mode = SEPK_FIN_PAIR;
	f.region = r2;
	f.nblk = (int)nb;
	f.nv = 7;
	f.wide = wide;
	f.also_ecoul = 1;
	sepk_task_ret(d, f, ret_slot);
	return sepk_queue_task(d, f);
}

extern "C" int sepdev_coulomb(sepdev *d, const sepdev_coul_args *a, int ret_slot)
{
	if (!d->list_built)
		return sepk_fail(SEP_GPU_ESTATE, "Coulomb forces before a neighbour list was built");
	if (ret_slot < 0 || ret_slot >= d->nret)
		return sepk_fail(SEP_GPU_EARG, "ret slot %d", ret_slot);
	sepk_coul c = {a->cf, a->cf2, a->icf, a->icf2, a->L[0], a->L[1], a->L[2],
		       1.0 / a->L[0], 1.0 / a->L[1], 1.0 / a->L[2],
		       a->L[0] / SEPK_QSCALE, a->L[1] / SEPK_QSCALE, a->L[2] / SEPK_QSCALE,
		       (float)a->cf, (float)a->icf, (float)a->icf2};
	int rc = sepk_flush_nh(d);
	if (rc || (a->mixed && (rc = sepk_fresh_qpos(d, a->L))))
		return rc;
	// the recorded pair call joins this one when both read the same
	// records with the same image rule
	if (d->pc_pending && (a->mixed != 0) == (d->pc_mixed != 0) &&
	    (a->mixed || (fast_image_ok(d, a->L) ? 1 : 0) == (d->pc_fast ? 1 : 0)))
		return launch_lj_coul(d, c, ret_slot);
	int region;
	if ((rc = sepk_term_region(d, &region)) || (rc = sepk_fork_point(d)) ||
	    (rc = sepk_flush_gathers(d)))
		return rc;
	const bool over = d->f_zero_pending != 0;
	const bool fast = fast_image_ok(d, a->L);
	auto k = a->mixed ? (over ? k_coulomb<true, false, true> : k_coulomb<false, false, true>)
		 : over   ? (fast ? k_coulomb<true, true, false> : k_coulomb<true, false, false>)
			  : (fast ? k_coulomb<false, true, false> : k_coulomb<false, false, false>);
	const unsigned nb = sepk_blocks_xcd(d->n * SEPK_SUB);
	k<<<nb, SEPK_BLOCK, 0, d->st>>>(d->s[0], d->nbr, d->nbr_count, d->n, d->npad, c,
					  sepk_region(d, region), d->region_rows);
	SEPK_LAUNCH_CHECK();
	d->f_zero_pending = 0;
	sepk_task f;
	memset(&f, 0, sizeof f);
	f.mode = SEPK_FIN_PAIR;
	f.region = region;
	f.nblk = (int)nb;
	f.nv = 7;
	f.also_ecoul = 1;
	sepk_task_ret(d, f, ret_slot);
	return sepk_queue_task(d, f);
}

// ---- Nose-Hoover (source/sepintgr.c:149-168) ---------------------------------
//
// When the sum of m v^2 of the current velocities is known (the previous
// leapfrog computed it) the call is only recorded and the next leapfrog
// applies f -= alpha m v itself; otherwise: sum kernel, finisher, apply.

// Sum of m v^2 over the atoms, with the leapfrog's blocks (SEPK_SUB lanes
// per atom, lane 0 working, XCD-remapped block index) and its order of
// terms, so that it is the same bits as the sum a leapfrog leaves in
// sys->sumv2 for the same velocities.
__global__ __launch_bounds__(SEPK_BLOCK) void k_nh_sum(sepk_state s, long n, long npad,
							double *partial, long rows)
{
	if (*s.err)
		return; // the finisher applies nothing either
	const long lb = sepk_xcd_block();
	const long t = lb * (SEPK_BLOCK / SEPK_SUB) + threadIdx.x / SEPK_SUB;
	double acc[1] = {0.0};
	if (t < n && threadIdx.x % SEPK_SUB == 0) {
		const double m = s.m[t];
		const double vx = s.v[t], vy = s.v[npad + t], vz = s.v[2 * npad + t];
		acc[0] = (vx * vx * m + vy * vy * m) + vz * vz * m;
	}
	sepk_block_partial(acc, partial, lb, rows);
}

__global__ void k_nh_apply(sepk_state s, long n, long npad, const double *alpha)
{
	const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= n || *s.err)
		return;
	const double al = *alpha;
	const double m = s.m[t];
	for (int k = 0; k < 3; k++)
		s.f[k * npad + t] -= al * m * s.v[k * npad + t];
}

extern "C" int sepdev_nosehoover(sepdev *d, double Td, double tau, double dt,
				 int alpha_slot)
{
	if (alpha_slot < 0 || alpha_slot >= d->nscal)
		return sepk_fail(SEP_GPU_EARG, "alpha slot %d", alpha_slot);
	int rc = sepk_flush_nh(d);
	if (rc)
		return rc;
	if (d->sumv2_valid) {
		d->nh_pending = 1;
		d->nh_slot = alpha_slot;
		d->nh_Td = Td;
		d->nh_dt_tau2 = dt / (tau * tau);
		return 0;
	}
	if ((rc = sepk_materialize_forces(d)))
		return rc;
	const unsigned nb = sepk_blocks_xcd(d->n * SEPK_SUB);
	if ((rc = sepk_flush_tasks(d)))
		return rc;
	k_nh_sum<<<nb, SEPK_BLOCK, 0, d->st>>>(d->s[0], d->n, d->npad,
						sepk_region(d, SEPK_R_MISC), d->region_rows);
	SEPK_LAUNCH_CHECK();
	sepk_task f;
	memset(&f, 0, sizeof f);
	f.mode = SEPK_FIN_NH;
	f.region = SEPK_R_MISC;
	f.nblk = (int)nb;
	f.nv = 1;
	f.alpha = d->scal + alpha_slot;
	f.Td = Td;
	f.dt_tau2 = dt / (tau * tau);
	f.npart = (double)d->n;
	if ((rc = sepk_queue_task(d, f)) || (rc = sepk_flush_tasks(d)))
		return rc;
	d->sumv2_valid = 1;
	k_nh_apply<<<sepk_blocks(d->n), SEPK_BLOCK, 0, d->st>>>(d->s[0], d->n, d->npad,
								 d->scal + alpha_slot);
	SEPK_LAUNCH_CHECK();
	return 0;
}

// ---- leapfrog (source/sepintgr.c:18-88) ---------------------------------------
//
// Per atom: optional fused Nose-Hoover force term, a = f/m, v += a dt,
// x += v dt, wrap once per axis counting crossings, squared displacement
// from xn.  Row: {ekin sum, kin_P (6), max d2, sum m v_new^2}.

// Output arrays of the per-atom integrator step: the state's own arrays,
// except the positions of a fused step (the spare buffer, while other atoms
// still gather the old ones) and a timing run's scratch.
struct sepk_lfout {
	double *v, *f, *a, *xn;
	int *cn, *cr;
	sepk_pos *pos;
	int4 *qpos;
};

// sep_nosehoover's force term and sep_leapfrog for atom t
// (source/sepintgr.c:149-168, :42-88) from its force before the thermostat
// term, spread over lanes 0..2 of the atom's SEPK_SUB lanes, one axis each
// (lane k is given component k of the force as Fk).  Lane 0 gathers the
// other axes' values by DPP moves and forms the sums in axis order.  acc:
// m vh^2 summed, the six m vh (x) vh components, d^2 and m v^2.  Every lane
// of the wave calls it.
__device__ __forceinline__ void sepk_lf_atom_lanes(const sepk_state &s, const sepk_lfout &o,
						   long t, long npad, int sub, bool act, double F0,
						   double F1, double F2, double dt, double L0,
						   double L1, double L2, int nh, double al,
						   int pending, double qs0, double qs1, double qs2,
						   double (&acc)[9])
{
	double x = 0.0, v = 0.0, vh = 0.0, dr = 0.0, m = 0.0, q = 0.0;
	if (act && sub < 3) {
		const int k = sub;
		const sepk_pos p = s.pos[t];
		q = p.q;
		x = k == 0 ? p.x : (k == 1 ? p.y : p.z);
		const double L = k == 0 ? L0 : (k == 1 ? L1 : L2);
		const double Fk = k == 0 ? F0 : (k == 1 ? F1 : F2);
		m = s.m[t];
		const long i = k * npad + t;
		double xn = s.xn[i];
		int cn = s.cn[i];
		if (pending) {
			xn = x;
			cn = 0;
			o.xn[i] = xn;
		}
		v = s.v[i];
		double f = Fk;
		if (nh)
			f -= al * m * v;
		const double a = f / m;
		v += a * dt;
		x += v * dt;
		vh = v - 0.5 * a * dt;
		int cr = s.cr[i];
		if (x > L) {
			x -= L;
			cn++;
			cr++;
		} else if (x < 0.0) {
			x += L;
			cn--;
			cr--;
		}
		dr = (x + cn * L) - xn;
		o.f[i] = f;
		o.a[i] = a;
		o.v[i] = v;
		o.cn[i] = cn;
		o.cr[i] = cr;
	}
	const double x1 = sepk_dpp<SEPK_DPP_LANE1>(x), x2 = sepk_dpp<SEPK_DPP_LANE2>(x);
	const double v1 = sepk_dpp<SEPK_DPP_LANE1>(v), v2 = sepk_dpp<SEPK_DPP_LANE2>(v);
	const double h1 = sepk_dpp<SEPK_DPP_LANE1>(vh), h2 = sepk_dpp<SEPK_DPP_LANE2>(vh);
	const double r1 = sepk_dpp<SEPK_DPP_LANE1>(dr), r2 = sepk_dpp<SEPK_DPP_LANE2>(dr);
	if (act && sub == 0) {
		acc[0] = (vh * vh * m + h1 * h1 * m) + h2 * h2 * m;
		acc[8] = (v * v * m + v1 * v1 * m) + v2 * v2 * m;
		acc[1] = vh * vh * m;
		acc[2] = vh * h1 * m;
		acc[3] = vh * h2 * m;
		acc[4] = h1 * h1 * m;
		acc[5] = h1 * h2 * m;
		acc[6] = h2 * h2 * m;
		acc[7] = (dr * dr + r1 * r1) + r2 * r2;
		const sepk_pos p = {x, x1, x2, q};
		o.pos[t] = p;
		o.qpos[t] = sepk_quant(p, qs0, qs1, qs2);
	}
}

// The leapfrog on its own.  Its atoms map onto blocks exactly as the pair
// kernels' (SEPK_SUB lanes per atom, lane 0 working, XCD-remapped block
// index), so that its rows -- and hence every reduced sum -- are the same
// bits as those of the fused step kernel.
__global__ __launch_bounds__(SEPK_BLOCK) void k_leapfrog(
	sepk_state s, long n, long npad, double dt, double L0, double L1, double L2,
	const sepdev_sys *sys, int nh, const double *alpha, double Td, double dt_tau2,
	double *partial, long rows, double qs0, double qs1, double qs2, sepk_gpend gp)
{
	if (sys->error)
		return; // positions are updated in place: nothing to copy
	const long lb = sepk_xcd_block();
	const long t = lb * (SEPK_BLOCK / SEPK_SUB) + threadIdx.x / SEPK_SUB;
	const int sub = threadIdx.x % SEPK_SUB;
	double acc[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
	const int pending = sys->xn_pending;
	double al = 0.0;
	if (nh)
		al = sepk_nh_alpha(*alpha, sys->sumv2, (double)n, Td, dt_tau2);
	// one axis a lane, as in the fused step kernel (sepk_lf_atom_lanes), so
	// the two give the same bits; lane k needs only force component k, to
	// which it adds the owed bonded gathers as k_bonded_gather would
	const bool act = t < n;
	double Fk = 0.0;
	if (act && sub < 3) {
		Fk = gp.over ? 0.0 : s.f[sub * npad + t];
		if (gp.n) {
			const int o = s.orig[t];
			for (int q = 0; q < gp.n; q++)
				for (int e = gp.g[q].off[o]; e < gp.g[q].off[o + 1]; e++)
					Fk += gp.g[q].contrib[3 * (long)gp.g[q].idx[e] + sub];
		}
	}
	const sepk_lfout o = {s.v, s.f, s.a, s.xn, s.cn, s.cr, s.pos, s.qpos};
	sepk_lf_atom_lanes(s, o, t, npad, sub, act, Fk, Fk, Fk, dt, L0, L1, L2, nh, al, pending,
			   qs0, qs1, qs2, acc);
	const double v[8] = {acc[0], acc[1], acc[2], acc[3], acc[4], acc[5], acc[6], acc[8]};
	sepk_block_reduce<true>(v, acc[7], [=](int i, double r) {
		partial[(size_t)sepk_lf_col(i) * rows + lb] = r;
	});
}

// Pair forces, Nose-Hoover and leapfrog in one launch (a step whose only
// calls are one overwriting pair call, sep_nosehoover and sep_leapfrog):
// the pair loop and its rows as in k_lj, then the atom's integrator step
// from its summed force, with the new positions to o.pos / o.qpos.
template <bool MIXED, bool FAST>
__global__ __launch_bounds__(SEPK_BLOCK) __attribute__((amdgpu_waves_per_eu(MIXED ? 7 : FAST ? 6 : 5))) void k_lj_step(
	sepk_state s, const int *__restrict__ nbr, const int *__restrict__ cnt, long n,
	long npad, sepk_lj c, const sepdev_sys *sys, int nh, const double *alpha, double Td,
	double dt_tau2, double dt, double qs0, double qs1, double qs2, sepk_lfout o,
	double *ppart, double *lpart, long rows)
{
	const long lb = sepk_xcd_block();
	const long t = lb * (SEPK_BLOCK / SEPK_SUB) + threadIdx.x / SEPK_SUB;
	const int sub = threadIdx.x % SEPK_SUB;
	const bool act = t < n;
	if (sys->error) {
		// a step after a device error changes nothing: the positions go
		// through to the other buffer unchanged (the whole grid returns)
		if (act && sub == 0) {
			o.pos[t] = s.pos[t];
			o.qpos[t] = s.qpos[t];
		}
		return;
	}
	double fx = 0.0, fy = 0.0, fz = 0.0;
	double acc[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
	double px = 0.0, py = 0.0, pz = 0.0;
	sepk_lj_pairs<false, MIXED, FAST>(s, nbr, cnt, npad, c, t, sub, act, 0, fx, fy, fz, acc,
					   px, py, pz);
	fx = sepk_atom_sum(fx);
	fy = sepk_atom_sum(fy);
	fz = sepk_atom_sum(fz);
	double lf[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
	const int pending = sys->xn_pending;
	double al = 0.0;
	if (nh)
		al = sepk_nh_alpha(*alpha, sys->sumv2, (double)n, Td, dt_tau2);
	if (act && sub == 0) {
		// the stress identity's per-atom term, as sepk_pair_epilogue adds it
		const double gx = 2.0 * fx, gy = 2.0 * fy, gz = 2.0 * fz;
		acc[1] = fma(gx, px, acc[1]);
		acc[2] = fma(gx, py, acc[2]);
		acc[3] = fma(gx, pz, acc[3]);
		acc[4] = fma(gy, py, acc[4]);
		acc[5] = fma(gy, pz, acc[5]);
		acc[6] = fma(gz, pz, acc[6]);
	}
	sepk_lf_atom_lanes(s, o, t, npad, sub, act, fx, fy, fz, dt, c.L0, c.L1, c.L2, nh, al,
			   pending, qs0, qs1, qs2, lf);
	double v[15];
#pragma unroll
	for (int k = 0; k < 7; k++) {
		v[k] = acc[k];
		v[7 + k] = lf[k];
	}
	v[14] = lf[8];
	sepk_block_reduce<true>(v, lf[7], [=](int i, double r) {
		(i < 7 ? ppart : lpart)[(size_t)(i < 7 ? i : sepk_lf_col(i - 7)) * rows + lb] = r;
	});
}

// The leapfrog's finishing task (after the step's pair task, if fused).
static int queue_lf_task(sepdev *d, int nh, double *alpha, unsigned nb, double dt, double skin,
			 int ret_slot)
{
	sepk_task f;
	memset(&f, 0, sizeof f);
	f.mode = SEPK_FIN_LF;
	f.region = SEPK_R_LF;
	f.nblk = (int)nb;
	f.nv = 9;
	f.maxmask = 1u << 7;
	f.nh_fused = nh;
	f.alpha = alpha;
	f.Td = d->nh_Td;
	f.dt_tau2 = d->nh_dt_tau2;
	f.npart = (double)d->n;
	f.reset_max = d->max_reset_pending;
	d->max_reset_pending = 0;
	f.skin = skin;
	f.dt = dt;
	sepk_task_ret(d, f, ret_slot);
	if (d->ring) {
		f.ring = d->ring;
		f.ring_cap = d->ring_cap;
		f.ring_n = d->ring_n;
	}
	// one finisher launch for the whole step: any queued build and pair
	// results, then the leapfrog's
	int rc;
	if ((rc = sepk_queue_task(d, f)) || (rc = sepk_flush_tasks(d)))
		return rc;
	d->sumv2_valid = 1;
	return 0;
}

static void launch_step_kernel(sepdev *d, const sepk_lj &c, int mixed, bool fast, int nh,
			       const double *alpha, double dt, const double *L,
			       const sepk_lfout &o, unsigned nb)
{
	auto k = mixed ? (fast ? k_lj_step<true, true> : k_lj_step<true, false>)
		       : (fast ? k_lj_step<false, true> : k_lj_step<false, false>);
	k<<<nb, SEPK_BLOCK, 0, d->st>>>(d->s[0], d->nbr, d->nbr_count, d->n, d->npad, c, d->sys,
					  nh, alpha, d->nh_Td, d->nh_dt_tau2, dt,
					  SEPK_QSCALE / L[0], SEPK_QSCALE / L[1], SEPK_QSCALE / L[2], o,
					  sepk_region(d, SEPK_R_PAIR), sepk_region(d, SEPK_R_LF),
					  d->region_rows);
}

// The recorded pair call, the pending Nose-Hoover call and this leapfrog
// in one launch.
static int sepdev_fused_step(sepdev *d, double dt, double skin, const double *L, int ret_slot)
{
	d->fused_pending = 0;
	int rc;
	if ((rc = sepk_claim_region(d, SEPK_R_PAIR)) || (rc = sepk_claim_region(d, SEPK_R_LF)))
		return rc;
	const int nh = d->nh_pending;
	d->nh_pending = 0;
	double *alpha = nh ? d->scal + d->nh_slot : d->scal;
	const unsigned nb = sepk_blocks_xcd(d->n * SEPK_SUB);
	const sepk_state &s = d->s[0];
	const sepk_lfout o = {s.v, s.f, s.a, s.xn, s.cn, s.cr, d->pos_alt, d->qpos_alt};
	launch_step_kernel(d, d->fused_lj, d->fused_mixed, d->fused_fast != 0, nh, alpha, dt, L, o,
			   nb);
	SEPK_LAUNCH_CHECK();
	d->f_zero_pending = 0;
	// the new positions are current from here on
	sepk_pos *p = d->s[0].pos;
	d->s[0].pos = d->pos_alt;
	d->pos_alt = p;
	int4 *q = d->s[0].qpos;
	d->s[0].qpos = d->qpos_alt;
	d->qpos_alt = q;
	for (int k = 0; k < 3; k++) {
		d->qL[k] = L[k];
		d->fused_L[k] = L[k];
	}
	d->qpos_stale = 0;
	d->last_fused = 1;
	d->fused_nh = nh;
	d->fused_alpha = alpha;
	d->fused_dt = dt;
	sepk_task f;
	memset(&f, 0, sizeof f);
	f.mode = SEPK_FIN_PAIR;
	f.region = SEPK_R_PAIR;
	f.nblk = (int)nb;
	f.nv = 7;
	f.epot_assign = d->fused_epot_assign;
	sepk_task_ret(d, f, d->fused_ret);
	if ((rc = sepk_queue_task(d, f)))
		return rc;
	return queue_lf_task(d, nh, alpha, nb, dt, skin, ret_slot);
}

extern "C" int sepdev_leapfrog(sepdev *d, double dt, double skin, const double *L,
			       int ret_slot)
{
	if (ret_slot < 0 || ret_slot >= d->nret)
		return sepk_fail(SEP_GPU_EARG, "ret slot %d", ret_slot);
	d->fork_ready = 0; // the atoms move
	if (d->fused_pending)
		return sepdev_fused_step(d, dt, skin, L, ret_slot);
	// a recorded pair call goes first (it applies any owed gathers before
	// itself); the gathers owed after it are folded into the kernel
	int rc = sepk_flush_pair(d);
	if (rc)
		return rc;
	sepk_gpend gp;
	gp.n = d->ngpend;
	gp.over = d->gpend_over;
	for (int q = 0; q < gp.n; q++)
		gp.g[q] = d->gpend[q];
	d->ngpend = 0;
	d->gpend_over = 0;
	if ((rc = sepk_materialize_forces(d)))
		return rc;
	if ((rc = sepk_claim_region(d, SEPK_R_LF)))
		return rc;
	const int nh = d->nh_pending;
	d->nh_pending = 0;
	const unsigned nb = sepk_blocks_xcd(d->n * SEPK_SUB);
	double *alpha = nh ? d->scal + d->nh_slot : d->scal;
	k_leapfrog<<<nb, SEPK_BLOCK, 0, d->st>>>(d->s[0], d->n, d->npad, dt, L[0], L[1], L[2],
						  d->sys, nh, alpha, d->nh_Td, d->nh_dt_tau2,
						  sepk_region(d, SEPK_R_LF), d->region_rows,
						  SEPK_QSCALE / L[0], SEPK_QSCALE / L[1],
						  SEPK_QSCALE / L[2], gp);
	SEPK_LAUNCH_CHECK();
	for (int k = 0; k < 3; k++)
		d->qL[k] = L[k];
	d->qpos_stale = 0;
	return queue_lf_task(d, nh, alpha, nb, dt, skin, ret_slot);
}

// ---- list extraction ------------------------------------------------------------

// Half list (entries j > o, original numbering) of every atom o, written
// straight into pinned host memory as packed rows: a workgroup takes 64 atoms
// in original order, a wave an atom; it counts the atoms' entries, takes room
// for all of them at once and walks the lists again to write them.  Only
// entries that exist cross the link, and nothing is allocated for the call.
// Bound by the link and the host's copies out of it.  One thread per atom into
// rows of the list's capacity, all of them copied to memory allocated for the
// call, made a synchronised rebuild and its forces take 794 us at 8000 atoms
// (300 us now) and 10.5 ms at 32000 (1.0 ms).
// A workgroup that finds no room sets its offset to -1 and runs again in the
// next pass, which has its counts.
#define SEPK_HALF_ATOMS 64
// entries an atom the pinned buffer holds on average (a full list of 128), and
// entries it holds at most (256 MiB; or one workgroup's, where those are more)
#define SEPK_HALF_MEAN 64
#define SEPK_HALF_MOST (64L * 1024 * 1024)
__global__ __launch_bounds__(SEPK_BLOCK) void
k_half_list(const int *orig, const int *iperm, const int *nbr, const int *cnt, long n, long npad,
	    int *counts, long *off, int *rows, unsigned long long room,
	    unsigned long long *cursor, int again)
{
	const long o0 = (long)blockIdx.x * SEPK_HALF_ATOMS;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	__shared__ int len[SEPK_HALF_ATOMS];
	__shared__ long first;
	if (again && off[blockIdx.x] != -1)
		return;
	for (int a = wave; a < SEPK_HALF_ATOMS; a += SEPK_BLOCK / 64) {
		int c = 0;
		if (again) {
			c = o0 + a < n ? counts[o0 + a] : 0;
		} else if (o0 + a < n) {
			const int o = (int)(o0 + a), t = iperm[o], m = cnt[t];
			for (int k = 0; k < m; k += 64) {
				const int hit = k + lane < m &&
						orig[nbr[sepk_entry(k + lane, t, npad)]] > o;
				c += __popcll(__ballot(hit));
			}
		}
		if (lane == 0) {
			len[a] = c;
			if (!again && o0 + a < n)
				counts[o0 + a] = c;
		}
	}
	__syncthreads();
	if (wave == 0) {
		const int own = len[lane];
		int end = own;
		for (int s = 1; s < 64; s <<= 1) {
			const int up = __shfl_up(end, s);
			end += lane >= s ? up : 0;
		}
		len[lane] = end - own;
		if (lane == 63) {
			const unsigned long long at =
				atomicAdd(cursor, (unsigned long long)end);
			first = at + end <= room ? (long)at : -1;
			off[blockIdx.x] = first;
		}
	}
	__syncthreads();
	if (first < 0)
		return;
	for (int a = wave; a < SEPK_HALF_ATOMS && o0 + a < n; a += SEPK_BLOCK / 64) {
		const int o = (int)(o0 + a), t = iperm[o], m = cnt[t];
		int *row = rows + first + len[a];
		for (int k = 0; k < m; k += 64) {
			int oj = -1;
			if (k + lane < m)
				oj = orig[nbr[sepk_entry(k + lane, t, npad)]];
			const unsigned long long hits = __ballot(oj > o);
			if (oj > o)
				row[__popcll(hits & ((1ull << lane) - 1))] = oj;
			row += __popcll(hits);
		}
	}
}

extern "C" int sepdev_half_pass(sepdev *d, int again, sepdev_half *h)
{
	if (!d->list_built)
		return sepk_fail(SEP_GPU_ESTATE, "no neighbour list");
	if (d->capturing)
		return sepk_fail(SEP_GPU_ESTATE, "transfer during graph capture");
	int rc = sepk_flush_tasks(d);
	if (rc)
		return rc;
	const long nblk = (d->n + SEPK_HALF_ATOMS - 1) / SEPK_HALF_ATOMS;
	// any one workgroup's rows fit
	size_t room = (size_t)d->npad * SEPK_HALF_MEAN;
	if (room > SEPK_HALF_MOST)
		room = SEPK_HALF_MOST;
	if (room < (size_t)SEPK_HALF_ATOMS * d->cap)
		room = (size_t)SEPK_HALF_ATOMS * d->cap;
	if (room > d->half_room) {
		if (d->half)
			(void)hipHostFree(d->half);
		d->half = nullptr;
		d->half_room = 0;
		SEPK_CHECK(hipHostMalloc((void **)&d->half,
					 nblk * sizeof(long) + (d->npad + room) * sizeof(int),
					 hipHostMallocDefault));
		d->half_room = room;
	}
	long *off = (long *)d->half;
	int *counts = (int *)(off + nblk);
	int *rows = counts + d->npad;
	const unsigned long long zero = 0;
	if ((rc = sepk_store_words(d, d->half_cursor, &zero, sizeof zero)))
		return rc;
	k_half_list<<<(unsigned)nblk, SEPK_BLOCK, 0, d->st>>>(
		d->s[0].orig, d->iperm, d->nbr, d->nbr_count, d->n, d->npad, counts, off, rows,
		d->half_room, d->half_cursor, again);
	SEPK_LAUNCH_CHECK();
	SEPK_CHECK(hipStreamSynchronize(d->st));
	h->nblk = nblk;
	h->atoms = SEPK_HALF_ATOMS;
	h->off = off;
	h->counts = counts;
	h->rows = rows;
	return 0;
}

extern "C" int sepdev_list_stats(sepdev *d, double *mean_full, int *max_full)
{
	if (!d->list_built)
		return sepk_fail(SEP_GPU_ESTATE, "no neighbour list");
	int *h = (int *)malloc(d->n * sizeof(int));
	SEPK_CHECK(hipMemcpyAsync(h, d->nbr_count, d->n * sizeof(int), hipMemcpyDeviceToHost, d->st));
	SEPK_CHECK(hipStreamSynchronize(d->st));
	double s = 0.0;
	int mx = 0;
	for (long i = 0; i < d->n; i++) {
		s += h[i];
		if (h[i] > mx)
			mx = h[i];
	}
	free(h);
	*mean_full = s / (double)d->n;
	*max_full = mx;
	return 0;
}

extern "C" int sepdev_time_pair(sepdev *d, int reps, double *ms_per_launch)
{
	if ((!d->last_lj && !d->last_fused) || !d->list_built)
		return sepk_fail(SEP_GPU_ESTATE, "no pair-force launch to time");
	if (reps < 1 || d->capturing)
		return sepk_fail(SEP_GPU_EARG, "time_pair: reps %d%s", reps,
				 d->capturing ? " during capture" : "");
	// owed bonded gathers go to f before the timed launches replace it
	int rc = sepk_flush_nh(d);
	if (rc || (rc = sepk_flush_gathers(d)) || (rc = sepk_flush_tasks(d)))
		return rc;
	sepk_lj c;
	memcpy(&c, d->last_fused ? (const void *)&d->fused_lj : d->last_lj, sizeof c);
	const sepk_lj_kernel k = (sepk_lj_kernel)d->last_lj_kernel;
	const unsigned nb = sepk_blocks_xcd(d->n * SEPK_SUB);
	double *part = sepk_region(d, SEPK_R_PAIR);
	// a fused step kernel is timed with its integrator outputs sent to
	// scratch, so that back-to-back launches see the same state
	sepk_lfout dry;
	memset(&dry, 0, sizeof dry);
	if (d->last_fused) {
		const size_t np = (size_t)d->npad;
		if (!d->tscratch)
			SEPK_CHECK(hipMalloc(&d->tscratch, 21 * np * sizeof(double)));
		double *b = d->tscratch;
		dry.v = b;
		dry.f = b + 3 * np;
		dry.a = b + 6 * np;
		dry.xn = b + 9 * np;
		dry.cn = (int *)(b + 12 * np);
		dry.cr = (int *)(b + 12 * np) + 3 * np;
		dry.pos = (sepk_pos *)(b + 15 * np);
		dry.qpos = (int4 *)(b + 19 * np);
	}
	hipEvent_t e0, e1;
	SEPK_CHECK(hipEventCreate(&e0));
	SEPK_CHECK(hipEventCreate(&e1));
	hipError_t err = hipEventRecord(e0, d->st);
	for (int r = 0; r < reps && err == hipSuccess; r++) {
		if (d->last_fused)
			launch_step_kernel(d, c, d->fused_mixed, d->fused_fast != 0, d->fused_nh,
					   d->fused_alpha, d->fused_dt, d->fused_L, dry, nb);
		else
			k<<<nb, SEPK_BLOCK, 0, d->st>>>(d->s[0], d->nbr, d->nbr_count, d->n,
							  d->npad, c, part, d->region_rows);
		err = hipGetLastError();
	}
	if (err == hipSuccess)
		err = hipEventRecord(e1, d->st);
	if (err == hipSuccess)
		err = hipEventSynchronize(e1);
	float ms = 0.0f;
	if (err == hipSuccess)
		err = hipEventElapsedTime(&ms, e0, e1);
	(void)hipEventDestroy(e0);
	(void)hipEventDestroy(e1);
	if (err != hipSuccess)
		return sepk_fail(SEP_GPU_EDEVICE, "time_pair: %s", hipGetErrorString(err));
	d->f_zero_pending = 0;
	*ms_per_launch = ms / reps;
	return 0;
}
