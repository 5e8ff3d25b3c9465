/* sep_gpu_lj_adjoint_noalloc's host side, at an atom count whose other
 * uploads are packed by several threads: no allocation and no thread between
 * its entry and its return, and the records it packs hold the atoms' x, mass,
 * charge, molecule and type.  Linked with the library's host sources and
 * -Wl,--wrap for the counted functions (tests/test_host_layer.py); the device
 * calls it makes are defined here. */
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include "sephost.h"

#define N 40000L
#define REC (6 + 4 + 2) /* ints: x, mass and charge, molecule and type */

static int counting, counted;

void *__real_malloc(size_t n);
void *__real_calloc(size_t n, size_t m);
void *__real_realloc(void *p, size_t n);
int __real_pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x);

void *__wrap_malloc(size_t n) { counted += counting; return __real_malloc(n); }
void *__wrap_calloc(size_t n, size_t m) { counted += counting; return __real_calloc(n, m); }
void *__wrap_realloc(void *p, size_t n) { counted += counting; return __real_realloc(p, n); }
int __wrap_pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x)
{
	counted += counting;
	return __real_pthread_create(t, a, f, x);
}

static int device;
static int records[N * REC];
static unsigned sent;

sepdev *sepdev_create(long n, int *err) { *err = n == N ? 0 : SEP_GPU_EARG; return (sepdev *)&device; }
void sepdev_destroy(sepdev *d) { (void)d; }
int sepdev_ret_alloc(sepdev *d) { (void)d; return 0; }
int sepdev_scalar_alloc(sepdev *d, double v) { (void)d; (void)v; return 0; }
int sepdev_record_bytes(unsigned mask) { return mask == (SEPDEV_X | SEPDEV_SCALARS) ? 4 * REC : 0; }
int sepdev_put_open(sepdev *d, char **rec) { (void)d; *rec = (char *)records; return 0; }
int sepdev_put_close(sepdev *d, unsigned mask) { (void)d; sent = mask; return 0; }
int sepdev_lj_adjoint_noalloc(sepdev *d, const sepdev_ljtab_args *a, const double *g, double *dx,
			      double *dt)
{
	(void)d, (void)a, (void)g, (void)dx, (void)dt;
	return 0;
}

int main(void)
{
	seppart *p = sep_init(N, 1);
	sepsys sys;
	memset(&sys, 0, sizeof sys);
	sys.npart = N;
	for (long i = 0; i < N; i++) {
		for (int k = 0; k < 3; k++)
			p[i].x[k] = 0.5 * (double)i + k;
		p[i].m = 1.0 + (double)i;
		p[i].z = -(double)i;
		p[i].molindex = (int)(i / 3);
		p[i].type = i % 7 ? 'A' : 'B';
	}
	if (!seph_ctx_for(p, &sys))
		return 2;
	const double prm[4] = {2.5, 1.0, 1.0, 1.0};
	static double g[3 * N], dx[3 * N], dt[2];
	counting = 1;
	const int rc = sep_gpu_lj_adjoint_noalloc(p, &sys, 1, "A", prm, g, dx, dt);
	counting = 0;
	int bad = rc != 0 || sent != (SEPDEV_X | SEPDEV_SCALARS);
	for (long i = 0; i < N; i++) {
		double d[5];
		memcpy(d, records + i * REC, sizeof d);
		for (int k = 0; k < 3; k++)
			bad += d[k] != p[i].x[k];
		bad += d[3] != p[i].m || d[4] != p[i].z;
		bad += records[i * REC + 10] != p[i].molindex || records[i * REC + 11] != p[i].type;
	}
	printf("bad %d counted %d\n", bad, counted);
	return bad || counted;
}
