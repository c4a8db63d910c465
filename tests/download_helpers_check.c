/* CPU check of the staged downloads' helper threads against the stand-ins of
 * hip_memory_shim.c, which this program's own symbols put in place of the runtime's
 * (and, for new threads that get no CPU, of pthread_create).  Prints "ok". */
#include "hip_memory_shim.c"

#include <stdio.h>
#include <time.h>

#include "../include/mglc_lbm.h"

#define CHECK(x) \
    do { \
        if (!(x)) { \
            printf("line %d: %s\n", __LINE__, #x); \
            exit(1); \
        } \
    } while (0)

static double now(void) {
    struct timespec t;
    clock_gettime(CLOCK_MONOTONIC, &t);
    return t.tv_sec + 1e-9 * t.tv_nsec;
}

struct box {
    lbm_ctx *ctx;
    size_t n;
    double *in, *out;
    int bad;
};

static struct box make(int nx, int ny, int nz, double seed) {
    lbm_params p;
    memset(&p, 0, sizeof p);
    p.nx = nx, p.ny = ny, p.nz = nz, p.tau = 0.6, p.rho0 = 1.0, p.thermal_axis = 1;
    struct box b = {NULL, (size_t)nx * ny * nz, NULL, NULL, 0};
    b.in = malloc(sizeof(double) * 4 * b.n);
    b.out = malloc(sizeof(double) * 4 * b.n);
    for (size_t i = 0; i < 4 * b.n; ++i) b.in[i] = seed + (double)i;
    CHECK(lbm_create(&p, &b.ctx) == LBM_OK);
    CHECK(lbm_load_fields(b.ctx, b.in, b.in + b.n, b.in + 2 * b.n, b.in + 3 * b.n, NULL) == LBM_OK);
    return b;
}

static void *read_back(void *arg) {
    struct box *b = arg;
    for (int k = 0; k < 6; ++k) {
        memset(b->out, 0, sizeof(double) * 4 * b->n);
        if (lbm_download_macro(b->ctx, b->out, b->out + b->n, b->out + 2 * b->n, b->out + 3 * b->n) != LBM_OK) b->bad = 1;
        if (memcmp(b->in, b->out, sizeof(double) * 4 * b->n)) b->bad = 1;
    }
    return NULL;
}

static void drop(struct box *b) {
    CHECK(!b->bad && lbm_destroy(b->ctx) == LBM_OK);
    free(b->in);
    free(b->out);
}

int main(void) {
    for (int late_ms = 0; late_ms <= 1500; late_ms += 1500) {  /* helpers at once, then far too late */
        struct box b = make(130, 90, 75, 1.0);
        const int before = shim_threads_started();
        shim_set_thread_delay(late_ms);
        const double t = now();
        read_back(&b);
        const double took = now() - t;
        shim_set_thread_delay(0);
        if (late_ms) CHECK(shim_threads_started() > before && took < 1.0);
        drop(&b);
        if (late_ms) CHECK(now() - t >= 1.4);  /* the last context to go waited for them */
    }
    struct box a = make(130, 90, 75, 2.0), b = make(81, 80, 83, 3.0);  /* two threads, one staging memory */
    pthread_t t[2];
    CHECK(!pthread_create(&t[0], NULL, read_back, &a) && !pthread_create(&t[1], NULL, read_back, &b));
    for (int k = 0; k < 2; ++k) pthread_join(t[k], NULL);
    drop(&a);
    drop(&b);
    CHECK(shim_in_use() == 0);
    puts("ok");
    return 0;
}
