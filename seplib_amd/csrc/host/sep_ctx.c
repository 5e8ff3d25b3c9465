/*
 * sep_ctx.c -- registry of atom arrays, their device contexts, error state,
 * AoS <-> device marshalling, return-value slots and cell grids.
 */
#include <math.h>
#include <pthread.h>
#include <signal.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "sephost.h"

/* ---- errors ----------------------------------------------------------- */

static int g_code;
static char g_msg[512];

int seph_fail(int code, const char *fmt, ...)
{
	va_list ap;
	va_start(ap, fmt);
	vsnprintf(g_msg, sizeof g_msg, fmt, ap);
	va_end(ap);
	g_code = code;
	return code;
}

int seph_dev_fail(int rc)
{
	if (rc == 0)
		return 0;
	g_code = rc;
	snprintf(g_msg, sizeof g_msg, "%s", sepdev_error_message());
	return rc;
}

int sep_gpu_last_error(void) { return g_code; }
const char *sep_gpu_last_error_message(void) { return g_msg; }
void sep_gpu_clear_error(void)
{
	g_code = 0;
	g_msg[0] = '\0';
	sepdev_clear_error();
}

/* ---- registry --------------------------------------------------------- */

typedef struct {
	seppart *atoms;
	long n;
	int nneighb;
	seph_ctx *ctx;
} seph_entry;

static seph_entry *g_reg;
static int g_nreg, g_capreg;

static seph_entry *find_entry(const seppart *atoms)
{
	for (int i = 0; i < g_nreg; i++)
		if (g_reg[i].atoms == atoms)
			return &g_reg[i];
	return NULL;
}

void seph_register(seppart *atoms, long n, int nneighb)
{
	seph_entry *e = find_entry(atoms);
	if (!e) {
		if (g_nreg == g_capreg) {
			g_capreg = g_capreg ? 2 * g_capreg : 16;
			g_reg = realloc(g_reg, sizeof(seph_entry) * (size_t)g_capreg);
		}
		e = &g_reg[g_nreg++];
		e->ctx = NULL;
	}
	e->atoms = atoms;
	e->n = n;
	e->nneighb = nneighb;
}

static void free_ctx(seph_ctx *c)
{
	if (!c)
		return;
	sepdev_destroy(c->dev);
	free(c->i3);
	free(c);
}

void seph_set_nneighb(seppart *atoms, int nneighb)
{
	seph_entry *e = find_entry(atoms);
	if (!e)
		return;
	e->nneighb = nneighb;
	if (e->ctx)
		e->ctx->nneighb = nneighb;
}

void seph_unregister(seppart *atoms)
{
	for (int i = 0; i < g_nreg; i++)
		if (g_reg[i].atoms == atoms) {
			free_ctx(g_reg[i].ctx);
			g_reg[i] = g_reg[--g_nreg];
			return;
		}
}

seph_ctx *seph_find(const seppart *atoms)
{
	seph_entry *e = find_entry(atoms);
	return e ? e->ctx : NULL;
}

/* Visits every context, for calls that only see a sepret pointer. */
int seph_each_ctx(int (*fn)(seph_ctx *, void *), void *arg)
{
	for (int i = 0; i < g_nreg; i++)
		if (g_reg[i].ctx) {
			int rc = fn(g_reg[i].ctx, arg);
			if (rc)
				return rc;
		}
	return 0;
}

seph_ctx *seph_ctx_for(seppart *atoms, const sepsys *sys)
{
	if (!atoms || !sys) {
		seph_fail(SEP_GPU_EARG, "null atoms or system pointer");
		return NULL;
	}
	seph_entry *e = find_entry(atoms);
	if (!e) {
		/* an array the library did not allocate: no list capacity known */
		seph_register(atoms, sys->npart, 0);
		e = find_entry(atoms);
	}
	if (e->n != sys->npart) {
		seph_fail(SEP_GPU_EARG, "sys->npart (%ld) differs from the %ld atoms allocated",
			  sys->npart, e->n);
		return NULL;
	}
	if (e->ctx)
		return e->ctx;
	seph_ctx *c = calloc(1, sizeof(seph_ctx));
	int err = 0;
	c->atoms = atoms;
	c->n = e->n;
	c->nneighb = e->nneighb;
	c->dev = sepdev_create(c->n, &err);
	if (!c->dev) {
		seph_dev_fail(err ? err : SEP_GPU_EDEVICE);
		free(c);
		return NULL;
	}
	c->ret_scratch = sepdev_ret_alloc(c->dev);
	c->alpha_scratch = sepdev_scalar_alloc(c->dev, 0.0);
	if (c->ret_scratch < 0 || c->alpha_scratch < 0) {
		seph_dev_fail(SEP_GPU_EDEVICE);
		free_ctx(c);
		return NULL;
	}
	e->ctx = c;
	return c;
}

/* ---- marshalling ------------------------------------------------------ */

/* Runs jobs 0 .. njobs-1, on SEPH_WORKERS threads when they handle many
 * atoms in all: the atom array (568 bytes an atom) is more than one core
 * streams while its records cross the link (sep_gpu_sync of 256000 atoms 4.1 ms
 * by one thread, 1.6 by four, of 50000 0.55 -> 0.34; sep_gpu_upload of 32768
 * 350 -> 218 us).  A program of synchronised calls goes through the array six
 * times a step, and what its one core holds of it after a call is spread over
 * four cores by threads: there the line is SEPH_CALL_ATOMS (a step of
 * sep_force_pairs, sep_nosehoover and sep_leapfrog, one thread -> four: 32768 atoms
 * 1.08 -> 1.80 ms, 40000 1.41 -> 1.83, 49152 2.05 -> 2.20, 55000 2.55 -> 2.26, 65000
 * 3.80 -> 2.80, 100000 6.5 -> 4.1). */
#define SEPH_WORKERS 4
#define SEPH_THREAD_ATOMS 32768
#define SEPH_CALL_ATOMS 49152

typedef struct {
	int njobs, next, rc;
	int (*job)(void *arg, int k);
	void *arg;
} job_queue;

static void *run_queue(void *p)
{
	job_queue *q = p;
	for (int k; (k = __atomic_fetch_add(&q->next, 1, __ATOMIC_RELAXED)) < q->njobs;) {
		const int rc = q->job(q->arg, k);
		if (rc)
			__atomic_store_n(&q->rc, rc, __ATOMIC_RELAXED);
	}
	return NULL;
}

int seph_run_jobs(int njobs, long atoms, int (*job)(void *arg, int k), void *arg)
{
	job_queue q = {njobs, 0, 0, job, arg};
	pthread_t th[SEPH_WORKERS];
	int nth = 0;
	if (atoms >= SEPH_THREAD_ATOMS) {
		/* the program's signals stay with its own threads: a helper takes
		 * none but those its own instructions raise */
		sigset_t block, mask;
		sigfillset(&block);
		sigdelset(&block, SIGSEGV);
		sigdelset(&block, SIGBUS);
		sigdelset(&block, SIGFPE);
		sigdelset(&block, SIGILL);
		pthread_sigmask(SIG_BLOCK, &block, &mask);
		while (nth < SEPH_WORKERS - 1 && nth < njobs - 1 &&
		       pthread_create(&th[nth], NULL, run_queue, &q) == 0)
			nth++;
		pthread_sigmask(SIG_SETMASK, &mask, NULL);
	}
	run_queue(&q);
	for (int i = 0; i < nth; i++)
		pthread_join(th[i], NULL);
	return q.rc;
}

/* One atom's fields to and from its record (the order is sepdev.h's). */
#define FIELD_OUT(flag, src)                                             \
	if (mask & (flag)) {                                             \
		memcpy(r, (src), sizeof(src));                           \
		r += sizeof(src);                                        \
	}
#define FIELD_IN(flag, dst)                                              \
	if (mask & (flag)) {                                             \
		memcpy((dst), r, sizeof(dst));                           \
		r += sizeof(dst);                                        \
	}

typedef struct {
	seph_ctx *c;
	unsigned mask;
	char *rec;
	int xn_pending;
	char type0;  /* uploads: the first atom's type */
	int mixed;   /* uploads: some atom's type differs from it */
	long per;
} xfer;

static int pack_job(void *arg, int k)
{
	xfer *t = arg;
	const unsigned mask = t->mask;
	const long i0 = k * t->per, i1 = i0 + t->per < t->c->n ? i0 + t->per : t->c->n;
	char *r = t->rec + (size_t)i0 * sepdev_record_bytes(mask);
	int mixed = 0;
	for (long i = i0; i < i1; i++) {
		const seppart *p = &t->c->atoms[i];
		FIELD_OUT(SEPDEV_X, p->x)
		FIELD_OUT(SEPDEV_V, p->v)
		FIELD_OUT(SEPDEV_F, p->f)
		FIELD_OUT(SEPDEV_A, p->a)
		FIELD_OUT(SEPDEV_XN, p->xn)
		if (mask & SEPDEV_SCALARS) {
			const double mz[2] = {p->m, p->z};
			memcpy(r, mz, sizeof mz);
			r += sizeof mz;
			mixed |= p->type != t->type0;
		}
		FIELD_OUT(SEPDEV_CROSS_NB, p->cross_neighb)
		FIELD_OUT(SEPDEV_CROSS, p->crossings)
		if (mask & SEPDEV_SCALARS) {
			const int mt[2] = {p->molindex, (signed char)p->type};
			memcpy(r, mt, sizeof mt);
			r += sizeof mt;
		}
	}
	if (mixed)
		__atomic_store_n(&t->mixed, 1, __ATOMIC_RELAXED);
	return 0;
}

/* The atoms that decide whether a call's transfers start threads. */
static long call_atoms(const seph_ctx *c) { return c->n >= SEPH_CALL_ATOMS ? c->n : 0; }

static int put_fields(seph_ctx *c, unsigned mask, long atoms)
{
	xfer t = {c, mask, NULL, 0, c->atoms[0].type, 0, 0};
	int rc = seph_dev_fail(sepdev_put_open(c->dev, &t.rec));
	if (rc)
		return rc;
	const int jobs = atoms >= SEPH_THREAD_ATOMS ? 4 * SEPH_WORKERS : 1;
	t.per = (c->n + jobs - 1) / jobs;
	seph_run_jobs(jobs, atoms, pack_job, &t);
	if (mask & SEPDEV_SCALARS) {
		c->uniform_type = t.mixed ? 0 : t.type0;
		c->uniform_type_valid = 1;
	}
	return seph_dev_fail(sepdev_put_close(c->dev, mask));
}

int seph_put(seph_ctx *c, unsigned mask) { return put_fields(c, mask, call_atoms(c)); }

int seph_put_noalloc(seph_ctx *c, unsigned mask) { return put_fields(c, mask, 0); }

static int unpack_job(void *arg, int k)
{
	xfer *t = arg;
	const unsigned mask = t->mask;
	long i0, i1;
	const int rc = sepdev_get_chunk(t->c->dev, k, &i0, &i1);
	if (rc)
		return rc;
	const char *r = t->rec + (size_t)i0 * sepdev_record_bytes(mask);
	for (long i = i0; i < i1; i++) {
		seppart *p = &t->c->atoms[i];
		FIELD_IN(SEPDEV_X, p->x)
		FIELD_IN(SEPDEV_V, p->v)
		FIELD_IN(SEPDEV_F, p->f)
		FIELD_IN(SEPDEV_A, p->a)
		FIELD_IN(SEPDEV_XN, p->xn)
		FIELD_IN(SEPDEV_CROSS_NB, p->cross_neighb)
		FIELD_IN(SEPDEV_CROSS, p->crossings)
		if (t->xn_pending) {
			/* the reference resets xn and cross_neighb right after the
			 * leapfrog that raised the flag (source/sepintgr.c:72-84) */
			memcpy(p->xn, p->x, sizeof p->xn);
			memset(p->cross_neighb, 0, sizeof p->cross_neighb);
		}
	}
	return 0;
}

static int get_fields(seph_ctx *c, unsigned mask, long atoms, int xn_pending)
{
	const char *rec;
	int nchunk;
	int rc = seph_dev_fail(sepdev_get_open(c->dev, mask, &rec, &nchunk));
	if (rc)
		return rc;
	xfer t = {c, mask, (char *)rec, xn_pending, 0, 0, 0};
	rc = seph_run_jobs(nchunk, atoms, unpack_job, &t);
	return rc ? seph_dev_fail(sepdev_get_failed(rc)) : 0;
}

int seph_get(seph_ctx *c, unsigned mask)
{
	return get_fields(c, mask, call_atoms(c), 0);
}

int seph_put_partners(seph_ctx *c)
{
	if (!c->i3 && !(c->i3 = malloc(sizeof(int) * 40 * (size_t)c->n)))
		return seph_fail(SEP_GPU_EHOST, "out of host memory");
	for (long i = 0; i < c->n; i++) {
		int *p = c->i3 + 40 * i;
		memcpy(p, c->atoms[i].bond, sizeof(int) * SEP_BOND);
		memcpy(p + 10, c->atoms[i].angle, sizeof(int) * SEP_ANGLE);
		memcpy(p + 20, c->atoms[i].dihed, sizeof(int) * SEP_DIHED);
	}
	int rc = seph_dev_fail(sepdev_put_partners(c->dev, c->i3));
	if (rc == 0)
		c->partners_on_device = 1;
	return rc;
}

int seph_put_topology(seph_ctx *c, const sepsys *sys)
{
	const sepmolinfo *m = sys->molptr;
	if (!m)
		return 0;
	const unsigned nb = m->flag_bonds == 1 ? m->num_bonds : 0;
	const unsigned na = m->flag_angles == 1 ? m->num_angles : 0;
	const unsigned nd = m->flag_dihedrals == 1 ? m->num_dihedrals : 0;
	if (c->topo_b == m->blist && c->topo_a == m->alist && c->topo_d == m->dlist &&
	    c->topo_nb == nb && c->topo_na == na && c->topo_nd == nd)
		return 0;
	int rc = seph_dev_fail(sepdev_put_topology(c->dev, m->blist, (int)nb, m->alist, (int)na,
						   m->dlist, (int)nd));
	if (rc)
		return rc;
	c->topo_b = m->blist;
	c->topo_a = m->alist;
	c->topo_d = m->dlist;
	c->topo_nb = nb;
	c->topo_na = na;
	c->topo_nd = nd;
	return 0;
}

static int any_partners(const seph_ctx *c)
{
	for (long i = 0; i < c->n; i++)
		if (c->atoms[i].bond[0] != -1 || c->atoms[i].angle[0] != -1 ||
		    c->atoms[i].dihed[0] != -1)
			return 1;
	return 0;
}

static void sys_to_dev(const sepsys *sys, sepdev_sys *ds)
{
	memset(ds, 0, sizeof *ds);
	ds->max_dist2 = sys->max_dist2;
	ds->tnow = sys->tnow;
	ds->neighb_flag = sys->neighb_flag;
	ds->nupdate_neighb = sys->nupdate_neighb;
}

int seph_put_all(seph_ctx *c, const sepsys *sys)
{
	int rc;
	if ((rc = seph_put_atoms(c)))
		return rc;
	if (any_partners(c) && (rc = seph_put_partners(c)))
		return rc;
	if ((rc = seph_put_topology(c, sys)))
		return rc;
	sepdev_sys ds;
	sys_to_dev(sys, &ds);
	return seph_dev_fail(sepdev_put_sys(c->dev, &ds));
}

static void ret_pack(const sepret *r, double *w)
{
	memset(w, 0, sizeof(double) * SEPDEV_RET_WORDS);
	w[SEPDEV_RET_EPOT] = r->epot;
	w[SEPDEV_RET_ECOUL] = r->ecoul;
	w[SEPDEV_RET_EKIN] = r->ekin;
	for (int a = 0; a < 3; a++)
		for (int b = 0; b < 3; b++) {
			w[SEPDEV_RET_POTP + 3 * a + b] = r->pot_P[a][b];
			w[SEPDEV_RET_KINP + 3 * a + b] = r->kin_P[a][b];
			w[SEPDEV_RET_BONDP + 3 * a + b] = r->pot_P_bond[a][b];
		}
}

void seph_ret_unpack(sepret *r, const double *w)
{
	r->epot = w[SEPDEV_RET_EPOT];
	r->ecoul = w[SEPDEV_RET_ECOUL];
	r->ekin = w[SEPDEV_RET_EKIN];
	for (int a = 0; a < 3; a++)
		for (int b = 0; b < 3; b++) {
			r->pot_P[a][b] = w[SEPDEV_RET_POTP + 3 * a + b];
			r->kin_P[a][b] = w[SEPDEV_RET_KINP + 3 * a + b];
			r->pot_P_bond[a][b] = w[SEPDEV_RET_BONDP + 3 * a + b];
		}
}

/* The per-atom state of a resident system back into the AoS; ds gets the
 * device's system scalars. */
static int get_atoms(seph_ctx *c, sepdev_sys *ds)
{
	const unsigned mask = SEPDEV_X | SEPDEV_V | SEPDEV_F | SEPDEV_A | SEPDEV_XN |
			      SEPDEV_CROSS_NB | SEPDEV_CROSS;
	int rc;
	if ((rc = seph_dev_fail(sepdev_get_settle(c->dev, mask))) ||
	    (rc = seph_dev_fail(sepdev_get_sys(c->dev, ds))))
		return rc;
	return get_fields(c, mask, c->n, ds->xn_pending != 0);
}

int seph_get_atoms(seph_ctx *c)
{
	sepdev_sys ds;
	return get_atoms(c, &ds);
}

int seph_put_atoms(seph_ctx *c)
{
	const int rc = put_fields(c, SEPDEV_X | SEPDEV_V | SEPDEV_F | SEPDEV_A | SEPDEV_XN |
					   SEPDEV_SCALARS | SEPDEV_CROSS_NB | SEPDEV_CROSS, c->n);
	/* a resident system looks its types up at the first call that needs them */
	c->uniform_type_valid = 0;
	return rc;
}

int seph_get_all(seph_ctx *c, sepsys *sys)
{
	int rc;
	sepdev_sys ds;
	if ((rc = get_atoms(c, &ds)))
		return rc;
	sys->max_dist2 = ds.max_dist2;
	sys->tnow = ds.tnow;
	sys->neighb_flag = ds.neighb_flag;
	sys->nupdate_neighb = ds.nupdate_neighb;
	for (int b = 0; b < c->nrets; b++) {
		double w[SEPDEV_RET_WORDS];
		if ((rc = seph_dev_fail(sepdev_ret_get(c->dev, c->rets[b].slot, w))))
			return rc;
		seph_ret_unpack((sepret *)c->rets[b].host, w);
	}
	for (int b = 0; b < c->nalphas; b++)
		if ((rc = seph_dev_fail(sepdev_scalar_get(c->dev, c->alphas[b].slot,
							  (double *)c->alphas[b].host))))
			return rc;
	if (sys->molptr && c->topo_nb + c->topo_na + c->topo_nd > 0) {
		sepmolinfo *m = sys->molptr;
		rc = seph_dev_fail(sepdev_get_bonded_values(
			c->dev, c->topo_nb ? m->blengths : NULL, c->topo_na ? m->angles : NULL,
			c->topo_nd ? m->dihedrals : NULL));
		if (rc)
			return rc;
	}
	return seph_check_device_error(c);
}

int seph_check_device_error(seph_ctx *c)
{
	sepdev_sys ds;
	int rc = seph_dev_fail(sepdev_get_sys(c->dev, &ds));
	if (rc)
		return rc;
	if (ds.error) {
		const int code = ds.error;
		ds.error = 0;
		sepdev_put_sys(c->dev, &ds);
		if (code == SEP_GPU_ENEIGHB)
			return seph_fail(code, "neighbour list capacity exceeded on the device (largest list %d)",
					 ds.max_full);
		if (code == SEP_GPU_ECELL)
			return seph_fail(code, "an atom position maps outside the cell grid (x < 0, x >= L or not finite)");
		return seph_fail(code, "device error %d", code);
	}
	return 0;
}

/* ---- slots ------------------------------------------------------------ */

int seph_ret_slot(seph_ctx *c, sepret *ret)
{
	for (int b = 0; b < c->nrets; b++)
		if (c->rets[b].host == ret)
			return c->rets[b].slot;
	if (c->nrets == SEPH_MAX_BIND) {
		seph_fail(SEP_GPU_EARG, "too many sepret structures bound to one system");
		return -1;
	}
	const int slot = sepdev_ret_alloc(c->dev);
	if (slot < 0) {
		seph_dev_fail(SEP_GPU_EDEVICE);
		return -1;
	}
	double w[SEPDEV_RET_WORDS];
	ret_pack(ret, w);
	if (seph_dev_fail(sepdev_ret_put(c->dev, slot, w)))
		return -1;
	c->rets[c->nrets].host = ret;
	c->rets[c->nrets].slot = slot;
	c->nrets++;
	return slot;
}

int seph_alpha_slot(seph_ctx *c, double *alpha)
{
	for (int b = 0; b < c->nalphas; b++)
		if (c->alphas[b].host == alpha)
			return c->alphas[b].slot;
	if (c->nalphas == SEPH_MAX_BIND) {
		seph_fail(SEP_GPU_EARG, "too many thermostat states bound to one system");
		return -1;
	}
	const int slot = sepdev_scalar_alloc(c->dev, *alpha);
	if (slot < 0) {
		seph_dev_fail(SEP_GPU_EDEVICE);
		return -1;
	}
	c->alphas[c->nalphas].host = alpha;
	c->alphas[c->nalphas].slot = slot;
	c->nalphas++;
	return slot;
}

void seph_ret_merge(sepret *ret, const double *w, int epot_assign, int bond_stress)
{
	if (epot_assign)
		ret->epot = w[SEPDEV_RET_EPOT];
	else
		ret->epot += w[SEPDEV_RET_EPOT];
	ret->ecoul += w[SEPDEV_RET_ECOUL];
	ret->ekin += w[SEPDEV_RET_EKIN];
	for (int a = 0; a < 3; a++)
		for (int b = 0; b < 3; b++) {
			ret->pot_P[a][b] += w[SEPDEV_RET_POTP + 3 * a + b];
			ret->kin_P[a][b] += w[SEPDEV_RET_KINP + 3 * a + b];
			if (bond_stress)
				ret->pot_P_bond[a][b] += w[SEPDEV_RET_BONDP + 3 * a + b];
		}
}

/* ---- grids ------------------------------------------------------------ */

/* The reference's 14-offset half-shell stencil (source/sepprfrc.c:424-426),
 * one (x, y, z) row per offset, in the reference's order. */
static const int HALF_SHELL[14][3] = {
	{0, 0, 0},  {1, 0, 0},  {1, 1, 0},  {0, 1, 0},  {-1, 1, 0},
	{0, 0, 1},  {1, 0, 1},  {1, 1, 1},  {0, 1, 1},  {-1, 1, 1},
	{-1, 0, 1}, {-1, -1, 1}, {0, -1, 1}, {1, -1, 1}};

void seph_grid_reference(const sepsys *sys, unsigned opt, sepdev_grid *g)
{
	memset(g, 0, sizeof *g);
	for (int k = 0; k < 3; k++) {
		g->n[k] = sys->nsubbox[k];
		g->l[k] = sys->lsubbox[k];
		g->L[k] = sys->length[k];
	}
	g->ref_index = 1;
	const double rl = sys->cf + sys->skin;
	g->rlist2 = rl * rl;
	g->opt = (int)opt;
	g->bonded_all = 1;
	int o = 0;
	if (g->n[0] >= 3 && g->n[1] >= 3 && g->n[2] >= 3) {
		/* No half-shell offset wraps onto its own cell and every
		 * (offset, -offset) pair reaches two distinct cells, so the
		 * reference's pairs seen from both ends are exactly the 27-cell
		 * stencil with j != i in the home cell.  Visit it in ascending
		 * (z, y, x) order: lists then come out in cell order. */
		for (int dz = -1; dz <= 1; dz++)
			for (int dy = -1; dy <= 1; dy++)
				for (int dx = -1; dx <= 1; dx++) {
					g->off[o][0] = dx;
					g->off[o][1] = dy;
					g->off[o][2] = dz;
					g->off[o++][3] = SEPDEV_RULE_NE;
				}
		g->noff = o;
		g->shift_ok = g->n[0] >= 5 && g->n[1] >= 5 && g->n[2] >= 5;
		return;
	}
	/* Fewer than three cells on some axis: offsets can alias.  Offset 0 in
	 * both directions = every other atom of the home cell; each further
	 * half-shell offset forward (j > i when it wraps onto the home cell)
	 * and backward (j < i), reproducing the reference's duplicates. */
	g->off[o][0] = g->off[o][1] = g->off[o][2] = 0;
	g->off[o++][3] = SEPDEV_RULE_NE;
	for (int s = 1; s < 14; s++) {
		for (int k = 0; k < 3; k++)
			g->off[o][k] = HALF_SHELL[s][k];
		g->off[o++][3] = SEPDEV_RULE_GT;
		for (int k = 0; k < 3; k++)
			g->off[o][k] = -HALF_SHELL[s][k];
		g->off[o++][3] = SEPDEV_RULE_LT;
	}
	g->noff = o;
}

void seph_grid_own(const sepsys *sys, double rlist, unsigned opt, int bonded_rule,
		   sepdev_grid *g)
{
	memset(g, 0, sizeof *g);
	int span[3];
	for (int k = 0; k < 3; k++) {
		int n = (int)(sys->length[k] / (rlist * (1.0 + 1e-9)));
		if (n < 3)
			n = 1;
		g->n[k] = n;
		g->l[k] = sys->length[k] / n;
		g->L[k] = sys->length[k];
		span[k] = n >= 3 ? 1 : 0;
	}
	g->ref_index = 0;
	g->rlist2 = rlist * rlist;
	g->opt = (int)opt;
	g->bonded_all = bonded_rule;
	g->shift_ok = g->n[0] >= 5 && g->n[1] >= 5 && g->n[2] >= 5;
	int o = 0;
	for (int dz = -span[2]; dz <= span[2]; dz++)
		for (int dy = -span[1]; dy <= span[1]; dy++)
			for (int dx = -span[0]; dx <= span[0]; dx++) {
				g->off[o][0] = dx;
				g->off[o][1] = dy;
				g->off[o][2] = dz;
				g->off[o++][3] = SEPDEV_RULE_NE;
			}
	g->noff = o;
}

/* ---- list build ------------------------------------------------------- */

typedef struct {
	sepdev_half h;
	long n;
	void (*row)(void *arg, long i, const int *entries, int count);
	void *arg;
	int missing;
} half_walk;

#define HALF_JOB 32 /* blocks a job */

static int half_job(void *arg, int k)
{
	half_walk *w = arg;
	for (long b = (long)k * HALF_JOB; b < (k + 1L) * HALF_JOB && b < w->h.nblk; b++) {
		if (w->h.off[b] < 0) {
			if (w->h.off[b] == -1)
				__atomic_store_n(&w->missing, 1, __ATOMIC_RELAXED);
			continue;
		}
		const int *e = w->h.rows + w->h.off[b];
		for (long i = b * w->h.atoms; i < (b + 1) * w->h.atoms && i < w->n; i++) {
			w->row(w->arg, i, e, w->h.counts[i]);
			e += w->h.counts[i];
		}
		w->h.off[b] = -2; /* done: another pass leaves it alone */
	}
	return 0;
}

int seph_half_lists(seph_ctx *c, int (*begin)(void *arg, const int *counts),
		    void (*row)(void *arg, long i, const int *entries, int count), void *arg)
{
	half_walk w = {.n = c->n, .row = row, .arg = arg};
	int rc = seph_dev_fail(sepdev_half_pass(c->dev, 0, &w.h));
	if (rc || (rc = begin(arg, w.h.counts)))
		return rc;
	for (;;) {
		w.missing = 0;
		/* rows take longer than records: a pair call that rebuilds, one thread
		 * -> four, 8192 atoms 277 -> 287 us, 16000 419 -> 402, 24000 539 -> 518,
		 * 32767 759 -> 654 */
		seph_run_jobs((int)((w.h.nblk + HALF_JOB - 1) / HALF_JOB), 2 * c->n, half_job, &w);
		if (!w.missing)
			return 0;
		if ((rc = seph_dev_fail(sepdev_half_pass(c->dev, 1, &w.h))))
			return rc;
	}
}

static int rows_fit(void *arg, const int *counts)
{
	const seph_ctx *c = arg;
	int maxc = 0;
	for (long i = 0; i < c->n; i++)
		if (counts[i] > maxc)
			maxc = counts[i];
	return maxc < c->nneighb ? 0 : seph_fail(SEP_GPU_ENEIGHB,
						 "Too many neighbours (%d >= capacity %d)", maxc,
						 c->nneighb);
}

static void write_row(void *arg, long i, const int *entries, int count)
{
	int *row = ((seph_ctx *)arg)->atoms[i].neighb;
	memcpy(row, entries, sizeof(int) * (size_t)count);
	row[count] = -1;
}

/* Writes the device list into atoms[i].neighb as a -1 terminated half list
 * (entries j > i, original numbering). */
static int write_half_lists(seph_ctx *c)
{
	return c->nneighb <= 0 ? 0 : seph_half_lists(c, rows_fit, write_row, c);
}

/* After a build that overflowed the list (SEP_GPU_ENEIGHB, longest list
 * max_full): grow the list and clear the error, or, where the longest list
 * exceeds the bound set by sep_gpu_list_limit, report the overflow. */
int seph_grow_list(seph_ctx *c, sepdev_sys *ds)
{
	if (c->list_limit > 0 && ds->max_full > c->list_limit) {
		ds->error = 0;
		sepdev_put_sys(c->dev, ds);
		return seph_fail(SEP_GPU_ENEIGHB,
				 "Too many neighbours: a list of %d entries exceeds the limit of %d",
				 ds->max_full, c->list_limit);
	}
	ds->error = 0;
	int rc = seph_dev_fail(sepdev_put_sys(c->dev, ds));
	if (!rc)
		rc = seph_dev_fail(sepdev_reserve_list(c->dev, ds->max_full + ds->max_full / 4 + 32));
	return rc;
}

int seph_build(seph_ctx *c, sepsys *sys, const sepdev_grid *g, int conditional)
{
	(void)sys;
	int rc = seph_dev_fail(sepdev_build_list(c->dev, g, conditional));
	if (rc || conditional)
		return rc;
	/* synchronised: check overflow and grow once */
	sepdev_sys ds;
	if ((rc = seph_dev_fail(sepdev_get_sys(c->dev, &ds))))
		return rc;
	if (ds.error == SEP_GPU_ENEIGHB) {
		if ((rc = seph_grow_list(c, &ds)))
			return rc;
		if ((rc = seph_dev_fail(sepdev_build_list(c->dev, g, 0))))
			return rc;
	}
	if ((rc = seph_check_device_error(c)))
		return rc;
	return write_half_lists(c);
}

static int grid_checked(const seph_ctx *c, const sepdev_grid *g)
{
	for (int i = 0; i < c->nchecked && i < SEPH_CHECKED; i++) {
		const seph_grid_key *k = &c->checked[i];
		if (k->n[0] == g->n[0] && k->n[1] == g->n[1] && k->n[2] == g->n[2] &&
		    k->opt == g->opt && k->rlist2 == g->rlist2)
			return 1;
	}
	return 0;
}

int seph_build_resident(seph_ctx *c, const sepdev_grid *g, int conditional)
{
	int rc = seph_dev_fail(sepdev_build_list(c->dev, g, conditional));
	/* a capture cannot hold the host check below (a stream
	 * synchronisation); an overflow there freezes the run, and sep_gpu_run
	 * reports it after the replay */
	if (rc || grid_checked(c, g) || sepdev_capturing(c->dev))
		return rc;
	/* first build of this grid: the initial capacity comes from the mean
	 * density, which grids of fewer than 3 cells per axis (whose stencil
	 * lists pairs more than once) or dense clusters can exceed; confirm
	 * it here, once, instead of letting SEP_GPU_ENEIGHB surface later */
	sepdev_sys ds;
	if ((rc = seph_dev_fail(sepdev_get_sys(c->dev, &ds))))
		return rc;
	if (ds.error == SEP_GPU_ENEIGHB) {
		if ((rc = seph_grow_list(c, &ds)) ||
		    (rc = seph_dev_fail(sepdev_build_list(c->dev, g, 0))))
			return rc;
	}
	if ((rc = seph_check_device_error(c)))
		return rc;
	seph_grid_key *k = &c->checked[c->nchecked % SEPH_CHECKED];
	for (int a = 0; a < 3; a++)
		k->n[a] = g->n[a];
	k->opt = g->opt;
	k->rlist2 = g->rlist2;
	c->nchecked++;
	return 0;
}

int seph_identify_potential(double (*fun)(double, char))
{
	if (fun == sep_lj)
		return SEPH_POT_LJ;
	if (fun == sep_lj_shift)
		return SEPH_POT_LJ_SHIFT;
	if (fun == sep_wca)
		return SEPH_POT_WCA;
	return SEPH_POT_NONE;
}
