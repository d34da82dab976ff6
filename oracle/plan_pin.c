/* plan_pin.c — the library's host side of the batched products (matmat.c,
 * int8.c) compiled for the CPU with its launches and allocations recorded
 * instead of made (tests/test_gemm_plan.py). Test infrastructure only.
 *
 * SPDX-License-Identifier: MIT */
#include <string.h>

#include "../mynah-slm_amd/csrc/matmat.c"
#include "../mynah-slm_amd/csrc/int8.c"

typedef struct {
    char kernel[48];
    uint32_t gx, gy, gz, block;
    uint64_t y;                 /* floats from y's start */
    uint32_t tokens, slots;     /* GEMM and fold launches; slots: the fold's */
    uint32_t has_part;
} plan_rec;

static plan_rec *recs;
static int n_recs, max_recs, fail_allocs, n_allocs, n_frees;
static uint64_t alloc_bytes;
static mynah_device dev;
static float *const y_base = (float *)((uintptr_t)1 << 40);
static char *const part_base = (char *)((uintptr_t)1 << 41);

void mynah_set_error(const char *fmt, ...) { (void)fmt; }
mynah_device *mynah_dev(void) { return &dev; }
hipStream_t mynah_stream_or_default(mynah_device *d, void *stream) {
    (void)d;
    return (hipStream_t)stream;
}

int mynah_geometry(int type, size_t rows, size_t cols, size_t *row_bytes) {
    static const size_t unit[15] = {[MYNAH_Q4_0] = 18, [MYNAH_Q8_0] = 34, [MYNAH_Q4_K] = 144,
                                    [MYNAH_Q5_K] = 176, [MYNAH_Q6_K] = 210};
    const size_t elems = type == MYNAH_Q4_0 || type == MYNAH_Q8_0 ? 32 : 256;
    if (rows == 0 || cols == 0 || cols % elems) return -1;
    *row_bytes = cols / elems * unit[type];
    return 0;
}

int mynah_q40_launch(mynah_device *d, const void *w, size_t rows, size_t cols, const float *x,
                     float *y, size_t tokens, const float *res, hipStream_t stream) {
    (void)d, (void)w, (void)rows, (void)cols, (void)x, (void)y, (void)tokens, (void)res;
    (void)stream;
    return 0;
}

int mynah_launch3(mynah_device *d, int kernel, unsigned gx, unsigned gy, unsigned gz,
                  unsigned block, size_t shmem, hipStream_t stream, void **args) {
    static const char *const names[] = {
#define X(id, name) name,
        MYNAH_KERNEL_LIST(X)
#undef X
    };
    (void)d, (void)shmem, (void)stream;
    if (n_recs == max_recs) return -1;
    plan_rec *r = &recs[n_recs++];
    memset(r, 0, sizeof *r);
    strncpy(r->kernel, names[kernel], sizeof r->kernel - 1);
    r->gx = gx;
    r->gy = gy;
    r->gz = gz;
    r->block = block;
    if (kernel == MYNAH_K_GEMM_FOLD) {
        r->y = (uint64_t)(*(float **)args[2] - y_base);
        r->tokens = *(uint32_t *)args[4];
        r->slots = *(uint32_t *)args[5];
        r->has_part = *(char **)args[0] == part_base;
    } else if (strstr(r->kernel, "mfma") != NULL || strstr(r->kernel, "few") != NULL) {
        r->y = (uint64_t)(*(float **)args[2] - y_base);
        r->tokens = *(uint32_t *)args[5];
        r->has_part = *(char **)args[8] == part_base;
    }
    return 0;
}

int mynah_launch(mynah_device *d, int kernel, unsigned gx, unsigned gy, unsigned block,
                 size_t shmem, hipStream_t stream, void **args) {
    return mynah_launch3(d, kernel, gx, gy, 1, block, shmem, stream, args);
}

hipError_t hipMallocAsync(void **p, size_t bytes, hipStream_t stream) {
    (void)stream;
    n_allocs++;
    if (fail_allocs) return hipErrorOutOfMemory;
    alloc_bytes = bytes;
    *p = part_base;
    return hipSuccess;
}
hipError_t hipFreeAsync(void *p, hipStream_t stream) {
    (void)stream;
    n_frees++;
    return (char *)p == part_base ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) {
    (void)e;
    return "";
}

/* lane: 0 the batched order, 1 the matvec order, 2 the int8 lane's product.
 * The launches into out (at most max of them): their number, or -1. */
int orc_plan(int lane, int type, uint64_t rows, uint64_t cols, uint64_t tokens, int cus, int fail,
             plan_rec *out, int max, uint64_t *bytes, int *allocs, int *frees) {
    const void *w = (const void *)((uintptr_t)1 << 42);
    const float *x = (const float *)((uintptr_t)1 << 43);
    recs = out;
    max_recs = max;
    n_recs = n_allocs = n_frees = 0;
    alloc_bytes = 0;
    fail_allocs = fail;
    dev.cus = cus;
    const int rc = lane == 0 ? mynah_matmat_launch(&dev, type, w, rows, cols, x, y_base, tokens, 1, NULL)
                   : lane == 1
                       ? mynah_matmat_mv_launch(&dev, type, w, rows, cols, x, y_base, tokens, NULL, NULL)
                       : mynah_int8_product(&dev, type, w, rows, cols, x, y_base, tokens, NULL);
    *bytes = alloc_bytes;
    *allocs = n_allocs;
    *frees = n_frees;
    return rc == 0 ? n_recs : -1;
}
