// sepdev_core.hip -- device state lifetime, host<->device transfers in the
// caller's atom order, return/scalar slots, timing and graph capture.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "sepdev_impl.h"

// ---- errors ---------------------------------------------------------------

static char g_msg[512];
static int g_code;

int sepk_fail(int code, const char *fmt, ...)
{
	va_list ap;
	va_start(ap, fmt);
	vsnprintf(g_msg, sizeof g_msg, fmt, ap);
	va_end(ap);
	g_code = code;
	return code;
}

extern "C" const char *sepdev_error_message(void) { return g_msg; }
extern "C" int sepdev_last_code(void) { return g_code; }
extern "C" void sepdev_clear_error(void)
{
	g_code = 0;
	g_msg[0] = '\0';
}

// ---- allocation -------------------------------------------------------------

template <class T>
static int dalloc(T **p, size_t count)
{
	*p = nullptr;
	if (count == 0)
		count = 1;
	SEPK_CHECK(hipMalloc((void **)p, count * sizeof(T)));
	return 0;
}

static int alloc_state(sepk_state *s, long npad)
{
	memset(s, 0, sizeof *s);
	int rc = 0;
	rc |= dalloc(&s->pos, npad);
	rc |= dalloc(&s->qpos, npad);
	rc |= dalloc(&s->v, 3 * npad);
	rc |= dalloc(&s->f, 3 * npad);
	rc |= dalloc(&s->a, 3 * npad);
	rc |= dalloc(&s->xn, 3 * npad);
	rc |= dalloc(&s->cn, 3 * npad);
	rc |= dalloc(&s->cr, 3 * npad);
	rc |= dalloc(&s->m, npad);
	rc |= dalloc(&s->type, npad);
	rc |= dalloc(&s->mol, npad);
	rc |= dalloc(&s->orig, npad);
	return rc;
}

static void free_state(sepk_state *s)
{
	void *ptrs[] = {s->pos, s->qpos, s->v, s->f, s->a, s->xn, s->cn, s->cr,
			s->m, s->type, s->mol, s->orig, s->partners};
	for (void *p : ptrs)
		if (p)
			(void)hipFree(p);
	memset(s, 0, sizeof *s);
}

__global__ void k_init_identity(sepk_state s, int *iperm, long n, long npad)
{
	long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= npad)
		return;
	s.orig[t] = t < n ? (int)t : -1;
	if (t < n)
		iperm[t] = (int)t;
	// slots past the last atom are phantoms: lists are padded with the
	// first of them, and a NaN position fails every cutoff test
	const double nan = __builtin_nan("");
	s.pos[t] = t < n ? sepk_pos{0.0, 0.0, 0.0, 0.0} : sepk_pos{nan, nan, nan, 0.0};
	s.qpos[t] = make_int4(0, 0, 0, t < n ? 0 : SEPK_QPHANTOM);
	s.m[t] = 1.0;
	s.type[t] = t < n ? 'A' : 0;
	s.mol[t] = -1;
	for (int c = 0; c < 3; c++) {
		s.v[c * npad + t] = 0.0;
		s.f[c * npad + t] = 0.0;
		s.a[c * npad + t] = 0.0;
		s.xn[c * npad + t] = 0.0;
		s.cn[c * npad + t] = 0;
		s.cr[c * npad + t] = 0;
	}
}

// The fused step's second position buffer: phantoms as in k_init_identity.
__global__ void k_init_alt(sepk_pos *pos, int4 *qpos, long n, long npad)
{
	const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= npad)
		return;
	const double nan = __builtin_nan("");
	pos[t] = t < n ? sepk_pos{0.0, 0.0, 0.0, 0.0} : sepk_pos{nan, nan, nan, 0.0};
	qpos[t] = make_int4(0, 0, 0, t < n ? 0 : SEPK_QPHANTOM);
}

extern "C" sepdev *sepdev_create(long npart, int *err)
{
	*err = 0;
	if (npart <= 0 || npart > SEPDEV_MAXN) {
		*err = sepk_fail(SEP_GPU_EARG, "sepdev_create: npart = %ld (1 to %ld)", npart,
				 (long)SEPDEV_MAXN);
		return nullptr;
	}
	sepdev *d = (sepdev *)calloc(1, sizeof(sepdev));
	d->n = npart;
	if (hipGetDevice(&d->device) != hipSuccess)
		d->device = 0;
	// at least one slot past the last atom: the phantom that pads lists
	d->npad = (npart + 1 + 63) / 64 * 64;
	d->qpos_stale = 1;
	int rc = 0;
	if (hipStreamCreateWithFlags(&d->st, hipStreamNonBlocking) != hipSuccess) {
		*err = sepk_fail(SEP_GPU_EDEVICE, "hipStreamCreate failed");
		free(d);
		return nullptr;
	}
	rc |= alloc_state(&d->s[0], d->npad);
	rc |= alloc_state(&d->s[1], d->npad);
	rc |= dalloc(&d->pos_alt, d->npad);
	rc |= dalloc(&d->qpos_alt, d->npad);
	rc |= dalloc(&d->iperm, d->npad);
	rc |= dalloc(&d->cellid_old, d->npad);
	rc |= dalloc(&d->order_tmp, d->npad);
	rc |= dalloc(&d->cell_slot, d->npad);
	rc |= dalloc(&d->nbr_count, d->npad);
	{
		// rows per region: the widest launch is a list kernel (SEPK_SUB
		// lanes per atom, XCD-padded) or a bonded kernel over up to 20
		// terms per atom
		long rows = d->npad * SEPK_SUB / SEPK_BLOCK + 2 * SEPK_NXCD;
		const long brows = d->npad * 20 / SEPK_BLOCK + 8;
		if (brows > rows)
			rows = brows;
		// a wide walk's row per 16 atoms
		const long wrows = d->npad / 16 + 8 * SEPK_NXCD;
		if (d->npad <= SEPK_WIDE_ATOMS + 64 && wrows > rows)
			rows = wrows;
		d->region_rows = rows;
		d->region_words = rows * SEPK_MAXNV;
		d->partials_words = d->region_words * SEPK_NREGION;
	}
	rc |= dalloc(&d->partials, d->partials_words);
	rc |= dalloc(&d->fin_l2, (size_t)SEPK_MAXTASK * SEPK_MAXNV * SEPK_FIN_BLOCKS);
	rc |= dalloc(&d->sys, 1);
	rc |= dalloc(&d->half_cursor, 1);
	d->ret_cap = 16;
	rc |= dalloc(&d->ret, (size_t)d->ret_cap * SEPDEV_RET_WORDS);
	d->ret_zero = (unsigned char *)calloc(d->ret_cap, 1);
	d->scal_cap = 16;
	rc |= dalloc(&d->scal, d->scal_cap);
	if (hipHostMalloc(&d->hstage,
			  SEPK_HEAD_BYTES + (size_t)d->npad * SEPK_REC_WORDS * sizeof(int),
			  hipHostMallocDefault) != hipSuccess)
		rc |= sepk_fail(SEP_GPU_EDEVICE, "hipHostMalloc staging failed");
	d->hrec = (char *)d->hstage + SEPK_HEAD_BYTES;
	for (hipEvent_t &ev : d->chunk_ev)
		if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess)
			rc |= sepk_fail(SEP_GPU_EDEVICE, "hipEventCreate failed");
	if (rc) {
		*err = rc;
		sepdev_destroy(d);
		return nullptr;
	}
	d->s[0].err = d->s[1].err = &d->sys->error;
	// list lengths start at zero so that a pair kernel that runs before any
	// build reads no list entries
	(void)hipMemsetAsync(d->nbr_count, 0, d->npad * sizeof(int), d->st);
	(void)hipMemsetAsync(d->sys, 0, sizeof(sepdev_sys), d->st);
	(void)hipMemsetAsync(d->ret, 0, (size_t)d->ret_cap * SEPDEV_RET_WORDS * sizeof(double), d->st);
	for (int b = 0; b < 2; b++) {
		k_init_identity<<<sepk_blocks(d->npad), SEPK_BLOCK, 0, d->st>>>(d->s[b], d->iperm, d->n, d->npad);
	}
	k_init_alt<<<sepk_blocks(d->npad), SEPK_BLOCK, 0, d->st>>>(d->pos_alt, d->qpos_alt, d->n,
								    d->npad);
	if (hipStreamSynchronize(d->st) != hipSuccess) {
		*err = sepk_fail(SEP_GPU_EDEVICE, "device init failed");
		sepdev_destroy(d);
		return nullptr;
	}
	return d;
}

extern "C" void sepdev_destroy(sepdev *d)
{
	if (!d)
		return;
	if (d->st)
		(void)hipStreamSynchronize(d->st);
	sepdev_graph_drop(d);
	free_state(&d->s[0]);
	free_state(&d->s[1]);
	void *ptrs[] = {d->iperm, d->cell_count, d->cell_start,
			d->cellid_old, d->order_tmp, d->cell_slot,
			d->nbr, d->nbr_count, d->partials, d->fin_l2, d->ring, d->ring_n, d->ret,
			d->scal, d->sys, d->half_cursor, d->blist, d->alist, d->dlist,
			d->bcontrib, d->acontrib, d->dcontrib, d->bcsr_off,
			d->bcsr_idx, d->acsr_off, d->acsr_idx, d->dcsr_off,
			d->dcsr_idx, d->blen, d->aval, d->dval};
	for (void *p : ptrs)
		if (p)
			(void)hipFree(p);
	if (d->hstage)
		(void)hipHostFree(d->hstage);
	if (d->half)
		(void)hipHostFree(d->half);
	for (hipEvent_t ev : d->chunk_ev)
		if (ev)
			(void)hipEventDestroy(ev);
	free(d->ret_zero);
	free(d->last_lj);
	(void)hipFree(d->pos_alt);
	(void)hipFree(d->qpos_alt);
	(void)hipFree(d->tscratch);
	void *adj[] = {d->adj_g, d->adj_x, d->adj_out, d->adj_part};
	for (void *p : adj)
		if (p)
			(void)hipFree(p);
	if (d->timing) {
		for (int i = 0; i < 64; i++) {
			(void)hipEventDestroy(d->t_pair.beg[i]);
			(void)hipEventDestroy(d->t_pair.end[i]);
		}
	}
	if (d->side) {
		(void)hipStreamSynchronize(d->side);
		(void)hipEventDestroy(d->fork_ev);
		(void)hipEventDestroy(d->join_ev);
		(void)hipStreamDestroy(d->side);
	}
	if (d->st)
		(void)hipStreamDestroy(d->st);
	free(d);
}

// ---- transfers ----------------------------------------------------------------

// Atoms cross the host link as records: the 4-byte words of the chosen
// fields of one atom, side by side, atoms in original order, in pinned host
// memory that the kernels read and write themselves.  One call of the API
// moves all of its fields with one launch and the host layer packs or unpacks
// an atom's fields in one visit.  With a launch, a copy through a staging
// array and a pass over the atoms per field, a resident system took 0.19, 0.53,
// 9.8 and 18.6 ms to synchronise at 1000, 27000, 256000 and 500000 atoms; it
// takes 0.07, 0.25, 1.6 and 3.0 ms (4.4 and 9.0 ms where one host thread
// unpacks).
// Consecutive lanes take consecutive words, so the link sees whole 64-byte
// accesses whatever order the device keeps the atoms in.
struct sepk_rec {
	int nw;                     // words per record
	int byte;                   // the word that is a single byte on the device, or -1
	int stride[SEPK_REC_WORDS]; // words (bytes for `byte`) between two atoms
	char *base[SEPK_REC_WORDS]; // the word of device atom 0
};

#define SEPK_REC_ATOMS 64 // atoms per workgroup

static void rec_add(sepk_rec &r, void *base, int words, int stride)
{
	for (int h = 0; h < words; h++) {
		r.stride[r.nw] = stride;
		r.base[r.nw++] = (char *)base + 4 * h;
	}
}

// x, y, z blocks of npad elements of `words` words
static void rec_add3(sepk_rec &r, void *blocks, long npad, int words)
{
	for (int k = 0; k < 3; k++)
		rec_add(r, (char *)blocks + (size_t)k * npad * words * 4, words, words);
}

// The record of a field mask; the order is the one sepdev.h states.
static sepk_rec rec_of(const sepdev *d, unsigned mask)
{
	sepk_rec r;
	r.nw = 0;
	r.byte = -1;
	const sepk_state &s = d->s[0];
	if (mask & SEPDEV_X)
		rec_add(r, s.pos, 6, sizeof(sepk_pos) / 4);
	if (mask & SEPDEV_V)
		rec_add3(r, s.v, d->npad, 2);
	if (mask & SEPDEV_F)
		rec_add3(r, s.f, d->npad, 2);
	if (mask & SEPDEV_A)
		rec_add3(r, s.a, d->npad, 2);
	if (mask & SEPDEV_XN)
		rec_add3(r, s.xn, d->npad, 2);
	if (mask & SEPDEV_SCALARS) {
		rec_add(r, s.m, 2, 2);
		rec_add(r, &s.pos->q, 2, sizeof(sepk_pos) / 4);
	}
	if (mask & SEPDEV_CROSS_NB)
		rec_add3(r, s.cn, d->npad, 1);
	if (mask & SEPDEV_CROSS)
		rec_add3(r, s.cr, d->npad, 1);
	if (mask & SEPDEV_SCALARS) {
		rec_add(r, s.mol, 1, 1);
		r.byte = r.nw;
		rec_add(r, s.type, 1, 1);
	}
	return r;
}

// records [o0, n) of the host buffer -> device fields
__global__ void k_scatter_records(sepk_rec r, const int *rec, const int *iperm, long n)
{
	const long o0 = (long)blockIdx.x * SEPK_REC_ATOMS;
	for (int j = threadIdx.x; j < SEPK_REC_ATOMS * r.nw; j += SEPK_BLOCK) {
		const int a = j / r.nw, w = j - a * r.nw;
		if (o0 + a >= n)
			return;
		const int v = rec[(size_t)o0 * r.nw + j];
		const size_t t = (size_t)iperm[o0 + a] * r.stride[w];
		if (w == r.byte)
			((signed char *)r.base[w])[t] = (signed char)v;
		else
			((int *)r.base[w])[t] = v;
	}
}

// device fields -> records [o0, o1) of the host buffer
__global__ void k_gather_records(sepk_rec r, int *rec, const int *iperm, long o0, long o1)
{
	const long b0 = o0 + (long)blockIdx.x * SEPK_REC_ATOMS;
	for (int j = threadIdx.x; j < SEPK_REC_ATOMS * r.nw; j += SEPK_BLOCK) {
		const int a = j / r.nw, w = j - a * r.nw;
		if (b0 + a >= o1)
			return;
		rec[(size_t)b0 * r.nw + j] =
			((const int *)r.base[w])[(size_t)iperm[b0 + a] * r.stride[w]];
	}
}

static unsigned rec_blocks(long atoms)
{
	return (unsigned)((atoms + SEPK_REC_ATOMS - 1) / SEPK_REC_ATOMS);
}

static int scatter_records(sepdev *d, const sepk_rec &r)
{
	k_scatter_records<<<rec_blocks(d->n), SEPK_BLOCK, 0, d->st>>>(r, (const int *)d->hrec,
								      d->iperm, d->n);
	SEPK_LAUNCH_CHECK();
	return 0;
}

__global__ void k_zero_blocks(double *p, long count)
{
	long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
	if (t < count)
		p[t] = 0.0;
}

// A few words between the host and the device: the kernel writes pinned
// memory, or carries the words in its arguments, where a copy of its own would
// go through the copy queue and, on the way in, have to be waited for.
#define SEPK_SMALL_WORDS 64
struct sepk_words {
	int w[SEPK_SMALL_WORDS];
};

__global__ void k_fetch_words(int *dst, const int *src, int n)
{
	if ((int)threadIdx.x < n)
		dst[threadIdx.x] = src[threadIdx.x];
}

__global__ void k_store_words(int *dst, sepk_words w, int n)
{
	if ((int)threadIdx.x < n)
		dst[threadIdx.x] = w.w[threadIdx.x];
}

static int fetch_words(sepdev *d, void *dst, const void *src, size_t bytes)
{
	if (d->capturing)
		return sepk_fail(SEP_GPU_ESTATE, "transfer during graph capture");
	if (bytes > sizeof(sepk_words) || bytes % 4)
		return sepk_fail(SEP_GPU_EARG, "fetch of %zu bytes", bytes);
	k_fetch_words<<<1, SEPK_SMALL_WORDS, 0, d->st>>>((int *)d->hstage, (const int *)src,
							 (int)(bytes / 4));
	SEPK_LAUNCH_CHECK();
	SEPK_CHECK(hipStreamSynchronize(d->st));
	memcpy(dst, d->hstage, bytes);
	return 0;
}

int sepk_store_words(sepdev *d, void *dst, const void *src, size_t bytes)
{
	if (d->capturing)
		return sepk_fail(SEP_GPU_ESTATE, "transfer during graph capture");
	if (bytes > sizeof(sepk_words) || bytes % 4)
		return sepk_fail(SEP_GPU_EARG, "store of %zu bytes", bytes);
	sepk_words w;
	memset(&w, 0, sizeof w);
	memcpy(&w, src, bytes);
	k_store_words<<<1, SEPK_SMALL_WORDS, 0, d->st>>>((int *)dst, w, (int)(bytes / 4));
	SEPK_LAUNCH_CHECK();
	return 0;
}

extern "C" int sepdev_record_bytes(unsigned mask)
{
	int w = 0;
	for (unsigned f = SEPDEV_X; f <= SEPDEV_XN; f <<= 1)
		w += mask & f ? 6 : 0;
	w += mask & SEPDEV_SCALARS ? 6 : 0;
	w += mask & SEPDEV_CROSS_NB ? 3 : 0;
	w += mask & SEPDEV_CROSS ? 3 : 0;
	return 4 * w;
}

extern "C" int sepdev_put_open(sepdev *d, char **rec)
{
	if (d->capturing)
		return sepk_fail(SEP_GPU_ESTATE, "transfer during graph capture");
	// owed bonded gathers belong to the forces before this upload
	int rc = sepk_flush_nh(d);
	if (rc || (rc = sepk_flush_gathers(d)))
		return rc;
	// the buffer may still feed an earlier launch
	SEPK_CHECK(hipStreamSynchronize(d->st));
	*rec = d->hrec;
	return 0;
}

extern "C" int sepdev_put_close(sepdev *d, unsigned mask)
{
	if (mask & (SEPDEV_V | SEPDEV_SCALARS))
		d->sumv2_valid = 0;
	if (mask & (SEPDEV_X | SEPDEV_SCALARS))
		d->qpos_stale = 1; // requantized by the next mixed pair call
	if (mask & SEPDEV_F)
		d->f_zero_pending = 0;
	return scatter_records(d, rec_of(d, mask));
}

extern "C" int sepdev_get_settle(sepdev *d, unsigned mask)
{
	if (d->capturing)
		return sepk_fail(SEP_GPU_ESTATE, "transfer during graph capture");
	int rc = sepk_flush_nh(d);
	if (!rc && (mask & SEPDEV_F))
		rc = sepk_materialize_forces(d);
	return rc;
}

extern "C" int sepdev_get_open(sepdev *d, unsigned mask, const char **rec, int *nchunk)
{
	int rc = sepdev_get_settle(d, mask);
	if (rc)
		return rc;
	long nc = (d->n + SEPK_CHUNK_ATOMS - 1) / SEPK_CHUNK_ATOMS;
	if (nc > SEPK_CHUNKS)
		nc = SEPK_CHUNKS;
	d->chunk = (((d->n + nc - 1) / nc) + 63) / 64 * 64;
	const sepk_rec r = rec_of(d, mask);
	int k = 0;
	for (long o = 0; o < d->n; o += d->chunk, k++) {
		const long o1 = o + d->chunk < d->n ? o + d->chunk : d->n;
		k_gather_records<<<rec_blocks(o1 - o), SEPK_BLOCK, 0, d->st>>>(
			r, (int *)d->hrec, d->iperm, o, o1);
		SEPK_LAUNCH_CHECK();
		if (d->n > d->chunk)
			SEPK_CHECK(hipEventRecord(d->chunk_ev[k], d->st));
	}
	*rec = d->hrec;
	*nchunk = k;
	return 0;
}

extern "C" int sepdev_get_chunk(sepdev *d, int k, long *i0, long *i1)
{
	*i0 = k * d->chunk;
	*i1 = *i0 + d->chunk < d->n ? *i0 + d->chunk : d->n;
	return d->n > d->chunk ? (int)hipEventSynchronize(d->chunk_ev[k])
			       : (int)hipStreamSynchronize(d->st);
}

extern "C" int sepdev_get_failed(int code)
{
	return sepk_fail(SEP_GPU_EDEVICE, "download: %s", hipGetErrorString((hipError_t)code));
}

// A host 3n array in original order into / out of any 3 x npad device block
// in device order (adjoint inputs and outputs).
int sepk_put_vec_to(sepdev *d, double *dst, const double *src3n)
{
	// the buffer may still feed an earlier launch
	SEPK_CHECK(hipStreamSynchronize(d->st));
	memcpy(d->hrec, src3n, (size_t)d->n * 3 * sizeof(double));
	sepk_rec r;
	r.nw = 0;
	r.byte = -1;
	rec_add3(r, dst, d->npad, 2);
	return scatter_records(d, r);
}

int sepk_get_vec_from(sepdev *d, double *dst3n, const double *src)
{
	sepk_rec r;
	r.nw = 0;
	r.byte = -1;
	rec_add3(r, (void *)src, d->npad, 2);
	k_gather_records<<<rec_blocks(d->n), SEPK_BLOCK, 0, d->st>>>(r, (int *)d->hrec, d->iperm, 0,
								     d->n);
	SEPK_LAUNCH_CHECK();
	SEPK_CHECK(hipStreamSynchronize(d->st));
	memcpy(dst3n, d->hrec, (size_t)d->n * 3 * sizeof(double));
	return 0;
}

extern "C" int sepdev_put_partners(sepdev *d, const int *partners40n)
{
	for (int b = 0; b < 2; b++)
		if (!d->s[b].partners) {
			int rc = dalloc(&d->s[b].partners, (size_t)40 * d->npad);
			if (rc)
				return rc;
		}
	if (d->capturing)
		return sepk_fail(SEP_GPU_ESTATE, "transfer during graph capture");
	SEPK_CHECK(hipStreamSynchronize(d->st));
	memcpy(d->hrec, partners40n, (size_t)d->n * 40 * sizeof(int));
	sepk_rec r;
	r.nw = 0;
	r.byte = -1;
	for (int k = 0; k < 40; k++)
		rec_add(r, d->s[0].partners + (size_t)k * d->npad, 1, 1);
	return scatter_records(d, r);
}

extern "C" int sepdev_put_sys(sepdev *d, const sepdev_sys *s)
{
	// the host record replaces everything, including the cached sum m v^2
	d->max_reset_pending = 0;
	d->sumv2_valid = 0;
	return sepk_store_words(d, d->sys, s, sizeof *s);
}

extern "C" int sepdev_get_sys(sepdev *d, sepdev_sys *s)
{
	int rc = sepk_flush_tasks(d);
	if (rc)
		return rc;
	rc = fetch_words(d, s, d->sys, sizeof *s);
	if (!rc && d->max_reset_pending)
		s->max_dist2 = 0.0;
	return rc;
}

// ---- slots --------------------------------------------------------------------

extern "C" int sepdev_ret_alloc(sepdev *d)
{
	if (d->nret == d->ret_cap) {
		double *nr;
		int rc = dalloc(&nr, (size_t)2 * d->ret_cap * SEPDEV_RET_WORDS);
		if (rc)
			return -1;
		SEPK_CHECK(hipMemsetAsync(nr, 0, (size_t)2 * d->ret_cap * SEPDEV_RET_WORDS * sizeof(double), d->st));
		SEPK_CHECK(hipMemcpyAsync(nr, d->ret, (size_t)d->ret_cap * SEPDEV_RET_WORDS * sizeof(double), hipMemcpyDeviceToDevice, d->st));
		SEPK_CHECK(hipStreamSynchronize(d->st));
		(void)hipFree(d->ret);
		d->ret = nr;
		d->ret_zero = (unsigned char *)realloc(d->ret_zero, 2 * d->ret_cap);
		memset(d->ret_zero + d->ret_cap, 0, d->ret_cap);
		d->ret_cap *= 2;
	}
	return d->nret++;
}

extern "C" int sepdev_ret_zero(sepdev *d, int slot)
{
	if (slot < 0 || slot >= d->nret)
		return sepk_fail(SEP_GPU_EARG, "ret slot %d", slot);
	// owed to the next kernel that writes the slot (it zeroes it first)
	d->ret_zero[slot] = 1;
	return 0;
}

extern "C" int sepdev_ret_get(sepdev *d, int slot, double *words)
{
	if (slot < 0 || slot >= d->nret)
		return sepk_fail(SEP_GPU_EARG, "ret slot %d", slot);
	int rc = sepk_flush_tasks(d);
	if (rc)
		return rc;
	if (d->ret_zero[slot]) {
		// a fill kernel rather than a memset node, so it may sit in a graph
		k_zero_blocks<<<1, 64, 0, d->st>>>(d->ret + (size_t)slot * SEPDEV_RET_WORDS,
						   SEPDEV_RET_WORDS);
		SEPK_LAUNCH_CHECK();
		d->ret_zero[slot] = 0;
	}
	return fetch_words(d, words, d->ret + (size_t)slot * SEPDEV_RET_WORDS,
			   SEPDEV_RET_WORDS * sizeof(double));
}

extern "C" int sepdev_ret_put(sepdev *d, int slot, const double *words)
{
	if (slot < 0 || slot >= d->nret)
		return sepk_fail(SEP_GPU_EARG, "ret slot %d", slot);
	d->ret_zero[slot] = 0;
	return sepk_store_words(d, d->ret + (size_t)slot * SEPDEV_RET_WORDS, words,
			   SEPDEV_RET_WORDS * sizeof(double));
}

extern "C" int sepdev_scalar_alloc(sepdev *d, double init)
{
	if (d->nscal == d->scal_cap) {
		double *ns;
		if (dalloc(&ns, (size_t)2 * d->scal_cap))
			return -1;
		SEPK_CHECK(hipMemcpyAsync(ns, d->scal, (size_t)d->scal_cap * sizeof(double), hipMemcpyDeviceToDevice, d->st));
		SEPK_CHECK(hipStreamSynchronize(d->st));
		(void)hipFree(d->scal);
		d->scal = ns;
		d->scal_cap *= 2;
	}
	int slot = d->nscal++;
	if (sepdev_scalar_put(d, slot, init))
		return -1;
	return slot;
}

extern "C" int sepdev_scalar_get(sepdev *d, int slot, double *v)
{
	int rc = sepk_flush_nh(d);
	if (rc || (rc = sepk_flush_tasks(d)))
		return rc;
	return fetch_words(d, v, d->scal + slot, sizeof(double));
}

extern "C" int sepdev_scalar_put(sepdev *d, int slot, double v)
{
	return sepk_store_words(d, d->scal + slot, &v, sizeof(double));
}

// ---- misc -----------------------------------------------------------------------

extern "C" int sepdev_synchronize(sepdev *d)
{
	int rc = sepk_flush_tasks(d);
	if (rc)
		return rc;
	SEPK_CHECK(hipStreamSynchronize(d->st));
	return 0;
}

extern "C" int sepdev_timing(sepdev *d, int on)
{
	if (on && !d->timing) {
		for (int i = 0; i < 64; i++) {
			SEPK_CHECK(hipEventCreate(&d->t_pair.beg[i]));
			SEPK_CHECK(hipEventCreate(&d->t_pair.end[i]));
		}
		d->t_pair.used = 0;
		d->t_pair.ms = 0.0;
		d->t_pair.count = 0;
		d->timing = 1;
	} else if (!on && d->timing) {
		SEPK_CHECK(hipStreamSynchronize(d->st));
		for (int i = 0; i < 64; i++) {
			(void)hipEventDestroy(d->t_pair.beg[i]);
			(void)hipEventDestroy(d->t_pair.end[i]);
		}
		d->timing = 0;
	}
	return 0;
}

// Folds recorded event pairs into the running total.
static int timer_flush(sepk_timer *t)
{
	for (int i = 0; i < t->used; i++) {
		SEPK_CHECK(hipEventSynchronize(t->end[i]));
		float ms = 0.0f;
		SEPK_CHECK(hipEventElapsedTime(&ms, t->beg[i], t->end[i]));
		t->ms += ms;
		t->count++;
	}
	t->used = 0;
	return 0;
}

int sepk_timer_begin(sepdev *d, sepk_timer *t)
{
	if (!d->timing || d->capturing)
		return 0;
	if (t->used == 64) {
		int rc = timer_flush(t);
		if (rc)
			return rc;
	}
	SEPK_CHECK(hipEventRecord(t->beg[t->used], d->st));
	return 0;
}

int sepk_timer_end(sepdev *d, sepk_timer *t)
{
	if (!d->timing || d->capturing)
		return 0;
	SEPK_CHECK(hipEventRecord(t->end[t->used], d->st));
	t->used++;
	return 0;
}

extern "C" int sepdev_timing_reset(sepdev *d)
{
	if (!d->timing)
		return 0;
	int rc = timer_flush(&d->t_pair);
	d->t_pair.ms = 0.0;
	d->t_pair.count = 0;
	return rc;
}

extern "C" int sepdev_timing_get(sepdev *d, const char *name, double *ms, long *count)
{
	if (!d->timing)
		return sepk_fail(SEP_GPU_ESTATE, "timing not enabled");
	if (strcmp(name, "pair") != 0)
		return sepk_fail(SEP_GPU_EARG, "unknown timer '%s'", name);
	int rc = timer_flush(&d->t_pair);
	*ms = d->t_pair.ms;
	*count = d->t_pair.count;
	return rc;
}

extern "C" int sepdev_graph_begin(sepdev *d, int slot)
{
	if (slot < 0 || slot > 1)
		return sepk_fail(SEP_GPU_EARG, "graph slot %d", slot);
	// gathers owed before the capture are applied now, not in every replay
	int rc = sepk_flush_gathers(d);
	if (rc)
		return rc;
	if (slot == 0)
		sepdev_graph_drop(d);
	else if (d->exec[1] || d->graph[1])
		return sepk_fail(SEP_GPU_ESTATE, "graph slot 1 in use");
	SEPK_CHECK(hipStreamBeginCapture(d->st, hipStreamCaptureModeRelaxed));
	d->capturing = 1;
	return 0;
}

extern "C" int sepdev_capturing(sepdev *d) { return d->capturing; }

extern "C" int sepdev_graph_end(sepdev *d, int slot)
{
	// the captured step must leave nothing queued for the host side
	int rc = sepk_flush_gathers(d);
	if (!rc)
		rc = sepk_flush_tasks(d);
	d->capturing = 0;
	if (rc) {
		hipGraph_t g = nullptr;
		if (hipStreamEndCapture(d->st, &g) == hipSuccess && g)
			(void)hipGraphDestroy(g);
		return rc;
	}
	SEPK_CHECK(hipStreamEndCapture(d->st, &d->graph[slot & 1]));
	SEPK_CHECK(hipGraphInstantiate(&d->exec[slot & 1], d->graph[slot & 1], nullptr, nullptr, 0));
	return 0;
}

extern "C" int sepdev_graph_launch(sepdev *d, int slot, long times)
{
	if (slot < 0 || slot > 1 || !d->exec[slot])
		return sepk_fail(SEP_GPU_ESTATE, "no graph in slot %d", slot);
	for (long i = 0; i < times; i++)
		SEPK_CHECK(hipGraphLaunch(d->exec[slot], d->st));
	return 0;
}

extern "C" int sepdev_graph_drop(sepdev *d)
{
	// the replays of the last run may still be queued on the stream: the
	// executable graphs go only after they are done
	if (d->exec[0] || d->exec[1])
		(void)hipStreamSynchronize(d->st);
	for (int k = 0; k < 2; k++) {
		if (d->exec[k])
			(void)hipGraphExecDestroy(d->exec[k]);
		if (d->graph[k])
			(void)hipGraphDestroy(d->graph[k]);
		d->exec[k] = nullptr;
		d->graph[k] = nullptr;
	}
	return 0;
}

// ---- device checkpoint ---------------------------------------------------
//
// The state a resident run carries from one step to the next, as it stands
// between steps: every per-atom array in device order (with the order
// itself), the neighbour list, the system scalars and the host-side facts
// the next step's kernels depend on (list geometry, whether sum m v^2 of
// the current velocities is known, the box of the quantized positions).
// Read back into a device of the same size, the run continues bit for bit.

#define SEPK_CKPT_MAGIC "SEPGPUC1"

struct sepk_ckpt_head {
	char magic[8];
	long n, npad;
	int lcap, cap, cap_limit, list_built;
	int has_partners, sumv2_valid, qpos_stale, pad_;
	double qL[3];
	sepdev_grid grid;
	sepdev_sys sys;
};

static int ckpt_io(FILE *f, void *host, size_t bytes, int writing)
{
	const size_t done = writing ? fwrite(host, 1, bytes, f) : fread(host, 1, bytes, f);
	if (done != bytes)
		return sepk_fail(SEP_GPU_EARG, "checkpoint: short %s (%zu of %zu bytes)",
				 writing ? "write" : "read", done, bytes);
	return 0;
}

// One device array through a host buffer, in either direction.
static int ckpt_array(sepdev *d, FILE *f, void *dev, size_t bytes, void *buf, int writing)
{
	int rc;
	if (writing) {
		SEPK_CHECK(hipMemcpy(buf, dev, bytes, hipMemcpyDeviceToHost));
		return ckpt_io(f, buf, bytes, 1);
	}
	if ((rc = ckpt_io(f, buf, bytes, 0)))
		return rc;
	SEPK_CHECK(hipMemcpy(dev, buf, bytes, hipMemcpyHostToDevice));
	return 0;
}

static int ckpt_arrays(sepdev *d, FILE *f, const sepk_ckpt_head &h, int writing)
{
	const size_t np = (size_t)d->npad;
	const size_t list_ints = (size_t)h.lcap * SEPK_SUB * np;
	size_t most = np * 40 * sizeof(int);
	if (h.list_built && list_ints * sizeof(int) > most)
		most = list_ints * sizeof(int);
	void *buf = malloc(most);
	if (!buf)
		return sepk_fail(SEP_GPU_EHOST, "checkpoint: out of host memory");
	sepk_state &s = d->s[0];
	struct {
		void *p;
		size_t bytes;
	} parts[] = {
		{s.pos, np * sizeof(sepk_pos)}, {s.qpos, np * sizeof(int4)},
		{s.v, 3 * np * sizeof(double)}, {s.f, 3 * np * sizeof(double)},
		{s.a, 3 * np * sizeof(double)}, {s.xn, 3 * np * sizeof(double)},
		{s.cn, 3 * np * sizeof(int)},   {s.cr, 3 * np * sizeof(int)},
		{s.m, np * sizeof(double)},     {s.type, np},
		{s.mol, np * sizeof(int)},      {s.orig, np * sizeof(int)},
		{d->iperm, np * sizeof(int)},   {d->nbr_count, np * sizeof(int)},
	};
	int rc = 0;
	for (auto &p : parts)
		if ((rc = ckpt_array(d, f, p.p, p.bytes, buf, writing)))
			break;
	if (!rc && h.has_partners)
		rc = ckpt_array(d, f, s.partners, np * 40 * sizeof(int), buf, writing);
	if (!rc && h.list_built)
		rc = ckpt_array(d, f, d->nbr, list_ints * sizeof(int), buf, writing);
	free(buf);
	return rc;
}

extern "C" int sepdev_checkpoint_write(sepdev *d, void *file)
{
	FILE *f = (FILE *)file;
	if (d->capturing)
		return sepk_fail(SEP_GPU_ESTATE, "checkpoint during a graph capture");
	// the step's deferred work is done: the recorded calls, the finisher
	int rc = sepk_flush_pair(d);
	if (rc || (rc = sepk_flush_nh(d)) || (rc = sepk_materialize_forces(d)) ||
	    (rc = sepk_flush_tasks(d)))
		return rc;
	sepk_ckpt_head h;
	memset(&h, 0, sizeof h);
	memcpy(h.magic, SEPK_CKPT_MAGIC, 8);
	h.n = d->n;
	h.npad = d->npad;
	h.list_built = d->list_built && d->nbr;
	h.lcap = h.list_built ? d->lcap : 0;
	h.cap = h.list_built ? d->cap : 0;
	h.cap_limit = d->cap_limit;
	h.has_partners = d->s[0].partners != nullptr;
	h.sumv2_valid = d->sumv2_valid;
	h.qpos_stale = d->qpos_stale;
	for (int k = 0; k < 3; k++)
		h.qL[k] = d->qL[k];
	h.grid = d->grid;
	if ((rc = sepdev_get_sys(d, &h.sys)))
		return rc;
	SEPK_CHECK(hipStreamSynchronize(d->st));
	if ((rc = ckpt_io(f, &h, sizeof h, 1)))
		return rc;
	return ckpt_arrays(d, f, h, 1);
}

extern "C" int sepdev_checkpoint_read(sepdev *d, void *file)
{
	FILE *f = (FILE *)file;
	if (d->capturing)
		return sepk_fail(SEP_GPU_ESTATE, "restore during a graph capture");
	sepk_ckpt_head h;
	int rc = ckpt_io(f, &h, sizeof h, 0);
	if (rc)
		return rc;
	if (memcmp(h.magic, SEPK_CKPT_MAGIC, 8) != 0)
		return sepk_fail(SEP_GPU_EARG, "not a device checkpoint of this library");
	if (h.n != d->n || h.npad != d->npad)
		return sepk_fail(SEP_GPU_EARG, "checkpoint of %ld atoms, system of %ld", h.n, d->n);
	if ((rc = sepk_flush_pair(d)) || (rc = sepk_flush_nh(d)) || (rc = sepk_flush_tasks(d)))
		return rc;
	SEPK_CHECK(hipStreamSynchronize(d->st));
	if (h.list_built && (rc = sepdev_reserve_list(d, h.cap)))
		return rc;
	// a new list's lengths are cleared on the stream, which the copies below
	// do not wait for
	SEPK_CHECK(hipStreamSynchronize(d->st));
	if (h.has_partners && !d->s[0].partners) {
		for (int b = 0; b < 2; b++)
			if ((rc = dalloc(&d->s[b].partners, (size_t)40 * d->npad)))
				return rc;
	}
	if ((rc = ckpt_arrays(d, f, h, 0)))
		return rc;
	if ((rc = sepdev_put_sys(d, &h.sys)))
		return rc;
	SEPK_CHECK(hipStreamSynchronize(d->st));
	// the host side of the device state
	d->list_built = h.list_built;
	if (h.list_built) {
		d->cap = h.cap;
		d->grid = h.grid;
	}
	d->cap_limit = h.cap_limit;
	d->sumv2_valid = h.sumv2_valid;
	d->qpos_stale = h.qpos_stale;
	for (int k = 0; k < 3; k++)
		d->qL[k] = h.qL[k];
	d->f_zero_pending = 0;
	d->ngpend = 0; // owed gathers were for the forces just replaced
	d->gpend_over = 0;
	d->max_reset_pending = 0;
	d->nh_pending = 0;
	d->fork_ready = 0;
	return 0;
}
