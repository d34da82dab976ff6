/* matmat.c — batched Y[tokens][rows] = X[tokens][cols] · W^T.
 *
 * Replaces ingot_matmat (third_party/ingot/src/generic.c:107-124) and the
 * per-type batched kernels (kernels.c:1742-1751, 2597-2606, 2627-2648). Exact f32 for
 * every width unless the int8 lane is on (int8.c), like the reference's exact
 * path: the tiled kernel of
 * gemm_exact.hip keeps the batched reference's own summation order (natural
 * weight order per 256-value unit, kernels.c:1017-1039 and 2635-2648), so
 * every output is bit-identical to ingot's exact matmat. tokens == 1 is the
 * matvec, as in the reference (kernels.c:1726); the callers route it.
 *
 * SPDX-License-Identifier: MIT */
#include "kernels_hip.h"
#include "runtime_internal.h"

#include <stdlib.h>

static long env_long(const char *name, long dflt) {
    const char *e = getenv(name);
    return (e != NULL && e[0] != '\0') ? strtol(e, NULL, 10) : dflt;
}

/* How an exact GEMM runs: kw waves share each 16-row group of a 64 x 64 tile
 * and hand its running totals on, unit by unit, inside the workgroup; nz
 * splits of the super-blocks (gridDim.z) whose later unit sums go through
 * memory and are folded in order afterwards (mynah_gemm_fold). */
typedef struct {
    uint32_t kw, nz;
    double ns;      /* estimated */
} gemm_split;

/* Partial sums of a split launch, per output: the first split's running total
 * and one sum per unit of the later splits (0: nothing goes through memory). */
static uint32_t gemm_slots(uint32_t units, uint32_t nz) {
    return nz > 1 ? units - units / nz + 1u : 0u;
}

/* What a split's memory costs a call on its own: it is allocated in stream
 * order, but the pool keeps none of it over a synchronisation, and the call
 * after one pays about 20 us for up to 64 MiB of it and 40 - 85 for more (a
 * process's first, or a larger one than any before, 100 - 500). Up to one tile
 * per CU a split fills the chip and gains more. Past it the gain must cover most
 * of this, the line between runs of calls and calls on their own (2560 x 2048
 * Q4_K, 1,020 tokens, split without this: 209 us in a run of calls but 305 each
 * on its own, against 228 and 239 unsplit), and the memory stays below a
 * thousandth of the card's. */
#define GEMM_PAST_BYTES ((uint64_t)256 << 20)

static double gemm_past_ns(uint64_t bytes) {
    return bytes <= ((uint64_t)64 << 20) ? 15000.0 : 30000.0;
}

/* Nanoseconds per column step and SIMD with w waves on it, measured on MI355X
 * (Q4_K 512 .. 9728 rows x 2048 / 2560 columns, 512 and 2047 tokens), by kw
 * (1, 2, 4) and w. The bound is 28.7 at 2 or 4 waves, 34 at 3, 43.7 at 1;
 * waves that share row groups keep in step through two barriers more per
 * unit, so kw > 1 costs where a launch has waves enough without it
 * (9728 x 2560, 2047 tokens: 1600 us with kw 1, 1647 with 2, 1946 with 4) and
 * pays where it has not (2048 x 2048, 512 tokens: 111, 90 and 86 us). */
static const double gemm_step_ns[3][5] = {{0.0, 54.0, 37.8, 37.3, 33.0},
                                          {0.0, 0.0, 44.0, 0.0, 36.0},
                                          {0.0, 0.0, 0.0, 0.0, 41.0}};

/* The (kw, nz) of least estimated time. A CU holds 16 waves of these kernels,
 * 4 / kw workgroups; a launch runs in rounds of resident workgroups, each
 * round's length set by its longest split (in rounds of kw units) and the
 * waves per SIMD it leaves; a split costs the fold's traffic (each unit sum
 * past the first split written and read, about 4.5 TB/s) and its launch.
 * cap: most splits. unit_steps: MFMAs of a super-block and wave (256, or 64 a
 * 16-token group in the kernels for few tokens). past: the whole product has
 * more than one tile per CU, so a split must also gain gemm_past_ns and keep to
 * GEMM_PAST_BYTES of memory. */
static gemm_split gemm_plan(uint64_t tiles, uint32_t units, uint64_t outputs, uint32_t cus,
                            uint32_t max_kw, uint32_t cap, double unit_steps, int past) {
    gemm_split best = {1, 1, 0.0};
    for (uint32_t kw = 1, i = 0; kw <= max_kw && kw <= units; kw *= 2u, i++) {
        const uint64_t slots = (uint64_t)cus * (4u / kw);
        for (uint32_t nz = 1; nz <= cap && nz <= units; nz++) {
            if (nz > 1 && tiles * (nz - 1u) >= slots) break;
            const uint64_t bytes = 4u * outputs * gemm_slots(units, nz);
            if (past && bytes > GEMM_PAST_BYTES) continue;
            const uint32_t per = (units + nz - 1u) / nz;
            const double steps = unit_steps * (double)((per + kw - 1u) / kw);
            uint64_t left = tiles * nz;
            const uint64_t full = left / slots;
            double ns = (double)full * steps * 4.0 * gemm_step_ns[i][4];
            left -= full * slots;
            if (left > 0) {
                const uint32_t w = kw * (uint32_t)((left + cus - 1u) / cus);
                ns += steps * (double)w * gemm_step_ns[i][w];
            }
            if (nz > 1)
                ns += 4000.0 + 2.0 * (double)bytes / 4500.0 + (past ? gemm_past_ns(bytes) : 0.0);
            if (best.ns == 0.0 || ns < best.ns) {
                best.ns = ns;
                best.kw = kw;
                best.nz = nz;
            }
        }
    }
    return best;
}

/* Up to 32 tokens a tile's empty 16-token groups are not computed: four columns
 * of one group an MFMA, where the full tile has one column of four groups.
 * 9728 x 2560 Q4_K, full tile -> few: 2 tokens 64 -> 27 us, 16 67 -> 30, 32
 * 69 -> 45 (MYNAH_GEMM_FEW=0: always the full tile). The groups, or 0. */
static uint32_t gemm_few(size_t tokens) {
    return tokens <= 32 && env_long("MYNAH_GEMM_FEW", 1) ? (uint32_t)(tokens + 15) / 16 : 0u;
}

/* split: 0 keeps nz at 1; past: as gemm_plan's. */
static gemm_split gemm_split_of(const mynah_device *d, int type, int ord, size_t rows, size_t cols,
                                size_t tokens, int split, int past) {
    const uint32_t few = gemm_few(tokens);
    const uint64_t tiles = (uint64_t)((rows + 63) / 64) * ((tokens + 63) / 64);
    const double steps = few ? 64.0 * few : 256.0;
    const uint32_t units = (uint32_t)(cols / 256);
    /* The Q8_0 matvec order has no unit sums to split by. */
    const int whole = ord == 1 && type == MYNAH_Q8_0;
    const long cap = whole || !split ? 1 : env_long("MYNAH_GEMM_SPLIT", 64);
    return gemm_plan(tiles, units, (uint64_t)rows * tokens, (uint32_t)d->cus,
                     few || whole ? 1u : 4u, cap > 1 ? (uint32_t)cap : 1u, steps, past);
}

/* The exact GEMM with its products on MFMA (gemm_mfma.hip): the default;
 * MYNAH_GEMM_MFMA=0 runs the VALU kernels of gemm_exact.hip instead (same
 * bits). MYNAH_GEMM_SPLIT=0 never splits over gridDim.z, N at most N ways;
 * MYNAH_GEMM_KW=1|2|4 forces kw. */
static int gemm_mfma_part(mynah_device *d, int type, int ord, const void *w, size_t rows,
                          size_t cols, size_t rb, const float *x, float *y, size_t tokens,
                          const float *res, gemm_split p, float *part, hipStream_t stream) {
    /* Q6_K sums in one order either way. */
    static const int kid[2][4] = {
        {MYNAH_K_Q4K_GEMM_MFMA1, MYNAH_K_Q5K_GEMM_MFMA1, MYNAH_K_Q6K_GEMM_MFMA1,
         MYNAH_K_Q80_GEMM_MFMA1},
        {MYNAH_K_Q4K_GEMM_MV_MFMA1, MYNAH_K_Q5K_GEMM_MV_MFMA1, MYNAH_K_Q6K_GEMM_MFMA1,
         MYNAH_K_Q80_GEMM_MV_MFMA1}};
    static const int fid[2][4] = {
        {MYNAH_K_Q4K_GEMM_FEW16, MYNAH_K_Q5K_GEMM_FEW16, MYNAH_K_Q6K_GEMM_FEW16,
         MYNAH_K_Q80_GEMM_FEW16},
        {MYNAH_K_Q4K_GEMM_MV_FEW16, MYNAH_K_Q5K_GEMM_MV_FEW16, MYNAH_K_Q6K_GEMM_FEW16,
         MYNAH_K_Q80_GEMM_MV_FEW16}};
    const int ti = type == MYNAH_Q4_K ? 0 : type == MYNAH_Q5_K ? 1 : type == MYNAH_Q6_K ? 2 : 3;
    const uint32_t units = (uint32_t)(cols / 256);
    const unsigned gx = (unsigned)((rows + 63) / 64), gy = (unsigned)((tokens + 63) / 64);
    const uint32_t few = gemm_few(tokens);
    const uint32_t nz = p.nz;
    const int kernel = few ? fid[ord][ti] + (int)few - 1
                           : kid[ord][ti] + (p.kw == 4 ? 2 : p.kw == 2 ? 1 : 0);
    const unsigned block = 256u * p.kw;
    uint32_t r32 = (uint32_t)rows, c32 = (uint32_t)cols, t32 = (uint32_t)tokens,
             rb32 = (uint32_t)rb;
    void *args[] = {&w, &x, &y, &r32, &c32, &t32, &rb32, &res, &part};
    int rc = mynah_launch3(d, kernel, gx, gy, nz, block, 0, stream, args);
    if (rc == 0 && nz > 1) {
        uint32_t slots = gemm_slots(units, nz);
        void *fargs[] = {&part, &res, &y, &r32, &t32, &slots};
        rc = mynah_launch(d, MYNAH_K_GEMM_FOLD, (unsigned)((rows * tokens + 255) / 256), 1, 256, 0,
                          stream, fargs);
    }
    return rc;
}

/* A last tile of at most 32 tokens costs a full one: where the estimates say
 * so (8 us for the launches more), the tokens before it and these run as two
 * products, one after the other in one workspace, the second in the kernels
 * for few tokens. Every output is the same sum either way. 9728 x 2560 Q4_K, 65
 * tokens: 145 -> 97 us; 201: 246 -> 216; 2560 x 9728 Q6_K, 201: 263 -> 232;
 * 6144 x 2048 Q4_K, 130: 105 -> 90. Not for the Q8_0 matvec order, which cannot
 * split the second product (4096 x 2048, 270 tokens: 166 -> 169).
 *
 * Without the memory for a split's sums the product runs unsplit. */
static int gemm_mfma_launch(mynah_device *d, int type, int ord, const void *w, size_t rows,
                            size_t cols, size_t rb, const float *x, float *y, size_t tokens,
                            const float *res, hipStream_t stream) {
    const long kw = env_long("MYNAH_GEMM_KW", 0);
    const int whole = ord == 1 && type == MYNAH_Q8_0;
    const uint32_t units = (uint32_t)(cols / 256);
    const int past = (uint64_t)((rows + 63) / 64) * ((tokens + 63) / 64) > (uint64_t)d->cus;
    int split = 1;
    size_t head, last, bytes;
    gemm_split ph, pl;
    float *part;
    for (;; split = 0) {
        head = tokens;
        last = tokens % 64;
        ph = gemm_split_of(d, type, ord, rows, cols, tokens, split, past);
        pl = (gemm_split){1, 1, 0.0};
        if (!whole && last > 0 && last < tokens && gemm_few(last)) {
            const gemm_split a =
                gemm_split_of(d, type, ord, rows, cols, tokens - last, split, past);
            pl = gemm_split_of(d, type, ord, rows, cols, last, split, past);
            if (a.ns + pl.ns + 8000.0 < ph.ns) {
                head = tokens - last;
                ph = a;
            }
        }
        if (!whole && !gemm_few(head) && (kw == 1 || kw == 2 || kw == 4)) ph.kw = (uint32_t)kw;
        size_t n = gemm_slots(units, ph.nz) * (rows * head);
        if (head < tokens && gemm_slots(units, pl.nz) * (rows * last) > n)
            n = gemm_slots(units, pl.nz) * (rows * last);
        bytes = n * sizeof(float);
        part = NULL;
        if (bytes == 0 || hipMallocAsync((void **)&part, bytes, stream) == hipSuccess) break;
        (void)hipGetLastError();
    }
    int rc = gemm_mfma_part(d, type, ord, w, rows, cols, rb, x, y, head, res, ph, part, stream);
    if (rc == 0 && head < tokens)
        rc = gemm_mfma_part(d, type, ord, w, rows, cols, rb, x + head * cols, y + head * rows, last,
                            res ? res + head * rows : NULL, pl, part, stream);
    const hipError_t e = bytes ? hipFreeAsync(part, stream) : hipSuccess;
    if (rc == 0 && e != hipSuccess) {
        mynah_set_error("hipFreeAsync(split-K partials): %s", hipGetErrorString(e));
        return -1;
    }
    return rc;
}

/* The MFMA kernels address a tile's 64 rows of x in 32 bits: longer rows take
 * the VALU kernels. */
static int gemm_mfma_on(size_t cols) {
    const char *env = getenv("MYNAH_GEMM_MFMA");
    return (env == NULL || env[0] != '0') && cols < ((size_t)1 << 24);
}

int mynah_matmat_launch(mynah_device *d, int type, const void *w, size_t rows, size_t cols,
                        const float *x, float *y, size_t tokens, int exact, hipStream_t stream) {
    size_t rb;
    if (mynah_geometry(type, rows, cols, &rb) != 0) return -1;
    /* The batched Q4_K and Q5_K products take the int8 lane when it is on,
     * exactly where the reference's do (kernels.c:1723-1751, 2573-2595;
     * tokens >= 2). */
    if (!exact && (type == MYNAH_Q4_K || type == MYNAH_Q5_K) && tokens >= 2 &&
        mynah_int8_mode() != MYNAH_INT8_OFF)
        return mynah_int8_product(d, type, w, rows, cols, x, y, tokens, stream);
    /* Q4_0 has no batched kernel in the reference: its generic path runs the
     * matvec's chain per token (generic.c:76-93), and so does this one. */
    if (type == MYNAH_Q4_0) return mynah_q40_launch(d, w, rows, cols, x, y, tokens, NULL, stream);
    /* The reference's batched core works in 256-wide units for every type
     * and refuses anything else (kernels.c:1087-1088, 2641-2648). */
    if (cols % 256 != 0) {
        mynah_set_error("batched matmat needs cols to be a multiple of 256");
        return -1;
    }
    if (tokens == 0 || tokens > 0xffffffffu || rb > 0xffffffffu) {
        mynah_set_error("bad token count");
        return -1;
    }
    if (((uintptr_t)x & 15u) != 0 || mynah_w_misaligned(type, w)) {
        mynah_set_error("misaligned operand for the batched GEMM");
        return -1;
    }
    if (gemm_mfma_on(cols))
        return gemm_mfma_launch(d, type, 0, w, rows, cols, rb, x, y, tokens, NULL, stream);
    const int k = type == MYNAH_Q4_K   ? MYNAH_K_Q4K_GEMM
                  : type == MYNAH_Q5_K ? MYNAH_K_Q5K_GEMM
                  : type == MYNAH_Q6_K ? MYNAH_K_Q6K_GEMM
                                       : MYNAH_K_Q80_GEMM;
    uint32_t r32 = (uint32_t)rows, c32 = (uint32_t)cols, t32 = (uint32_t)tokens, rb32 = (uint32_t)rb;
    void *args[] = {&w, &x, &y, &r32, &c32, &t32, &rb32};
    return mynah_launch(d, k, (unsigned)((rows + 63) / 64), (unsigned)((tokens + 63) / 64), 256, 0,
                        stream, args);
}

int mynah_matmat_mv_launch(mynah_device *d, int type, const void *w, size_t rows, size_t cols,
                           const float *x, float *y, size_t tokens, const float *res,
                           hipStream_t stream) {
    size_t rb;
    if (mynah_geometry(type, rows, cols, &rb) != 0) return -1;
    /* Q4_0's matvec and batched product share one order (a single running
     * sum per output, kernels.c:2467-2484, generic.c:76-93): the batched
     * chains are the matvec-order GEMM. */
    if (type == MYNAH_Q4_0) {
        if (tokens == 0 || tokens > 0xffffffffu) {
            mynah_set_error("matvec-order GEMM needs 1 <= tokens < 2^32");
            return -1;
        }
        return mynah_q40_launch(d, w, rows, cols, x, y, tokens, res, stream);
    }
    if (cols % 256 != 0 || tokens == 0 || tokens > 0xffffffffu || rb > 0xffffffffu) {
        mynah_set_error("matvec-order GEMM needs cols %% 256 == 0 and 1 <= tokens < 2^32");
        return -1;
    }
    if (((uintptr_t)x & 15u) != 0 || mynah_w_misaligned(type, w)) {
        mynah_set_error("misaligned operand for the matvec-order GEMM");
        return -1;
    }
    if (gemm_mfma_on(cols))
        return gemm_mfma_launch(d, type, 1, w, rows, cols, rb, x, y, tokens, res, stream);
    const int k = type == MYNAH_Q4_K   ? MYNAH_K_Q4K_GEMM_MV
                  : type == MYNAH_Q5_K ? MYNAH_K_Q5K_GEMM_MV
                  : type == MYNAH_Q6_K ? MYNAH_K_Q6K_GEMM_MV
                                       : MYNAH_K_Q80_GEMM_MV;
    uint32_t r32 = (uint32_t)rows, c32 = (uint32_t)cols, t32 = (uint32_t)tokens, rb32 = (uint32_t)rb;
    void *args[] = {&w, &x, &y, &r32, &c32, &t32, &rb32, &res};
    return mynah_launch(d, k, (unsigned)((rows + 63) / 64), (unsigned)((tokens + 63) / 64), 256, 0,
                        stream, args);
}
