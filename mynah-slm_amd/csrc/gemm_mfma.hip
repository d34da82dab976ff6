// gemm_mfma.hip — the exact batched GEMM with its products on the matrix
// cores and only the ordered sums on the VALU.
//
// Same outputs, bit for bit, as gemm_exact.hip in both of its orders (the
// reference's batched order, third_party/ingot/src/kernels.c:1017-1039,
// 1053-1104, 2635-2648, and the matvec order of kernels.c:94-115, 319-337,
// 2525-2551): each super-block sum starts from 0 and takes the products
// w[i] * x[i] one at a time in that order, and the row total takes the
// super-block sums in order.
//
// Products: v_mfma_f32_16x16x1_4b_f32 with a zero accumulator forms the
// 4 x 16 x 16 outer products a_i * b_j of one column step; each is
// round(a_i * b_j) + 0, the bits of v_mul_f32 except that a -0 product
// comes out +0 (checked on gfx950 over 4.2 million operand pairs of this
// instruction and 8.4 million of its 32 x 32 sibling: normal, subnormal,
// zero, infinite and NaN operands, every one equal or a zero of the other
// sign). A zero's sign cannot reach a sum here: a running sum
// starts at +0 and x + (+0) == x + (-0) for every x except -0, which a sum
// that starts at +0 never holds (only -0 + -0 gives -0). Each product is then
// added to its running sum with its own v_add_f32 (no contraction), in
// column order — the same roundings as the VALU kernel, at one VALU
// instruction per product instead of two. The instruction's accumulate form
// (D = A B + C) cannot carry the sums: on gfx950 it rounds once, like fma
// (equal to fmaf on 16.8 million single and chained cases, and unlike a
// multiply then an add on a third of them), where the reference rounds the
// product and the sum separately.
//
// Tiling: a workgroup of 256 threads owns 64 rows x 64 tokens; wave w the rows
// 16 w .. 16 w + 15 and all 64 tokens. Per column step k lane l feeds B =
// x[token l][k] and A = w[row l % 16][k]; the MFMA's four blocks are the four
// 16-token groups against the same 16 rows, whose A block is broadcast to all
// of them (cbsz = 2), so one register holds A for four columns: block abid of
// it (lanes 16 abid .. + 15) serves its own column. A lane therefore decodes
// only 16 of a 64-value stage's weights of its row, in registers, and no
// weight passes through LDS: lane quarter q = l / 16 owns the values 8 q ..
// 8 q + 7 of each of the stage's two 32-value halves, the same 8 quant bytes
// in every format. Lane l then holds, in register 4 b + e, the product of row
// 4 (l / 16) + e and token 16 b + l % 16.
//
// Weight values: v_fma_mix_f32 reads a 16-bit half of a register as an f16
// operand; a code q < 1024 alone in a half is the f16 subnormal q 2^-24, so
// fma(D 2^24, half, C) = round(D q + C) with no conversion (D 2^24 is exact:
// D < 2^23).
//
// x goes through LDS, copied straight from global memory one stage ahead
// into the other of two buffers (16 KiB each; 16-byte chunk c of token t sits
// at chunk c ^ (t % 16) of the token's 256 bytes, so the 16 lanes of one read
// phase hit 16 different bank groups), one barrier per stage.
//
// What bounds it: issue. An MFMA of this shape takes 32 cycles of its SIMD
// (13.5 ns) and does not overlap f32 adds, its own wave's or another's; 16 adds
// of registers take 15 ns where two waves alternate (a wave alone issues one
// instruction every 4 cycles, and waves share two ports, so an odd number of
// them leaves one idle part of the time; any scalar-register operand doubles
// an add). Per column step and SIMD, measured: 43.7 ns with 1 wave, 29.3 with
// 2, 34.0 with 3, 28.8 with 4 (73 TFLOP/s). The kernel reaches 33.0 with four
// waves (9728 x 2560 Q4_K, 2047 tokens, 1651 -> 1600 us against the form that
// decoded weights into LDS for all four waves; 6144 x 2048, 512 tokens, 242 ->
// 229 us; 2560 x 9728 Q6_K, 201 tokens, 294 -> 261 us).
//
// Launches too small to give every SIMD four waves share a tile among more of
// them, in two ways (the host plans both). KW = 2 or 4 waves per row group: the
// template below. Split K (gridDim.z > 1): workgroup z takes the units
// [z U / Z, (z + 1) U / Z); z = 0 stores the running row total of its units
// (from 0, in order) to part[0][token][row], every other z stores each unit's sum to
// part[u][token][row]; mynah_gemm_fold then continues the total from slot 0
// over the later units in order (and adds res), the row total the single
// launch would give. Not for the Q8_0 matvec order, whose row total takes
// every 32-value block sum.
//
// SPDX-License-Identifier: MIT
#include "common.hip.h"

#define GF_ROWS 64
#define GF_TOK 64

typedef float gm_f2 __attribute__((ext_vector_type(2)));
typedef float gf_f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void gf_lds_void;

#define GF_TWO24 16777216.0f
#define GF_TWO20 1048576.0f

MYNAH_DEV float gf_lo(uint32_t v) { return f16_to_f32(v); }
MYNAH_DEV float gf_hi(uint32_t v) { return f16_to_f32(v >> 16); }

// Codes of the eight bytes (w0, w1) as weights: v[j] = round(D byte_j + C),
// the bytes already masked to their codes; ds = D 2^24.
MYNAH_DEV void gf_bytes(uint32_t w0, uint32_t w1, float ds, float c, float *v) {
#pragma clang fp contract(off)
    const uint32_t w[2] = {w0, w1};
#pragma unroll
    for (int m = 0; m < 2; m++) {
        const uint32_t e = w[m] & 0x00ff00ffu, o = (w[m] >> 8) & 0x00ff00ffu;
        v[4 * m] = __builtin_fmaf(ds, gf_lo(e), c);
        v[4 * m + 1] = __builtin_fmaf(ds, gf_lo(o), c);
        v[4 * m + 2] = __builtin_fmaf(ds, gf_hi(e), c);
        v[4 * m + 3] = __builtin_fmaf(ds, gf_hi(o), c);
    }
}

// Two dwords from any address (the kernels run in unaligned-access mode).
MYNAH_DEV uint2 gf_load8(const uint8_t *p) {
    uint2 v;
    __builtin_memcpy(&v, p, sizeof v);
    return v;
}

// Each holder keeps what lane quarter q needs of one super-block of its row
// and decodes stage ST (values 64 ST .. + 63) into v: v[j] = value 8 q + j of
// the stage's first 32, v[8 + j] of its second.
struct GfQ4K {
    static constexpr uint32_t UB = 144u;
    uint4 hdr;
    uint2 qs[4];
    __device__ __forceinline__ void load(const uint8_t *blk, uint32_t q) {
        hdr = *(const uint4 *)blk;
#pragma unroll
        for (int g = 0; g < 4; g++) qs[g] = *(const uint2 *)(blk + 16u + 32u * g + 8u * q);
    }
    template <int ST> __device__ __forceinline__ void decode(uint32_t, float *v) const {
#pragma clang fp contract(off)
        const float d = f16_to_f32(hdr.x), dmin = f16_to_f32(hdr.x >> 16);
        float sa, ma, sb, mb;
        q4k_sm<2 * ST>(hdr.y, hdr.z, hdr.w, sa, ma);
        q4k_sm<2 * ST + 1>(hdr.y, hdr.z, hdr.w, sb, mb);
        // The high nibbles stay in place: 16 q 2^-24 against D 2^20.
        const float da = (d * sa) * GF_TWO24, db = (d * sb) * GF_TWO20;
        const float na = -(dmin * ma), nb = -(dmin * mb);
        const uint32_t w[2] = {qs[ST].x, qs[ST].y};
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const uint32_t w8 = w[m] >> 8;
            const uint32_t a = w[m] & 0x000f000fu, b = w[m] & 0x00f000f0u;
            const uint32_t c = w8 & 0x000f000fu, e = w8 & 0x00f000f0u;
            v[4 * m] = __builtin_fmaf(da, gf_lo(a), na);
            v[4 * m + 1] = __builtin_fmaf(da, gf_lo(c), na);
            v[4 * m + 2] = __builtin_fmaf(da, gf_hi(a), na);
            v[4 * m + 3] = __builtin_fmaf(da, gf_hi(c), na);
            v[8 + 4 * m] = __builtin_fmaf(db, gf_lo(b), nb);
            v[8 + 4 * m + 1] = __builtin_fmaf(db, gf_lo(e), nb);
            v[8 + 4 * m + 2] = __builtin_fmaf(db, gf_hi(b), nb);
            v[8 + 4 * m + 3] = __builtin_fmaf(db, gf_hi(e), nb);
        }
    }
};

struct GfQ5K {
    static constexpr uint32_t UB = 176u;
    uint4 hdr;
    uint2 qh, qs[4];
    __device__ __forceinline__ void load(const uint8_t *blk, uint32_t q) {
        hdr = *(const uint4 *)blk;
        qh = *(const uint2 *)(blk + 16u + 8u * q);
#pragma unroll
        for (int g = 0; g < 4; g++) qs[g] = *(const uint2 *)(blk + 48u + 32u * g + 8u * q);
    }
    template <int ST> __device__ __forceinline__ void decode(uint32_t, float *v) const {
#pragma clang fp contract(off)
        const float d = f16_to_f32(hdr.x), dmin = f16_to_f32(hdr.x >> 16);
        float sa, ma, sb, mb;
        q4k_sm<2 * ST>(hdr.y, hdr.z, hdr.w, sa, ma);
        q4k_sm<2 * ST + 1>(hdr.y, hdr.z, hdr.w, sb, mb);
        uint32_t l0, h0, l1, h1;
        q5k_quants<ST>(qs[ST].x, qh.x, l0, h0);
        q5k_quants<ST>(qs[ST].y, qh.y, l1, h1);
        gf_bytes(l0, l1, (d * sa) * GF_TWO24, -(dmin * ma), v);
        gf_bytes(h0, h1, (d * sb) * GF_TWO24, -(dmin * mb), v + 8);
    }
};

// Q6_K stage ST = (h, i) = (ST / 2, ST % 2): the weights 128 h + 32 k + l for
// k = 2 i, 2 i + 1; l = 8 q .. 8 q + 7 lies in the 16-value half q / 2 of its
// sub-block pair, whose scale is byte 8 h + 2 k + q / 2.
struct GfQ6K {
    static constexpr uint32_t UB = 210u;
    uint2 ql[2][2], qh[2];
    uint4 sc;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *blk, uint32_t q) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            ql[h][0] = gf_load8(blk + 64u * h + 8u * q);
            ql[h][1] = gf_load8(blk + 64u * h + 32u + 8u * q);
            qh[h] = gf_load8(blk + 128u + 32u * h + 8u * q);
        }
        __builtin_memcpy(&sc, blk + 192u, sizeof sc);
        d = *(const uint16_t *)(blk + 208u);
    }
    template <int ST> __device__ __forceinline__ void decode(uint32_t q, float *v) const {
#pragma clang fp contract(off)
        constexpr int h = ST / 2, i = ST % 2;
        // Scale bytes 8 h + 4 i + 2 t + q / 2, t = 0, 1.
        const uint32_t word = i ? (h ? sc.w : sc.y) : (h ? sc.z : sc.x);
        const uint32_t sw = word >> (8u * (q >> 1));
        const float df = f16_to_f32(d);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const float ds = df * (float)(int)(int8_t)(sw >> (16 * t));
            constexpr int K0 = 2 * i;
            const int k = K0 + t;
            uint32_t w[2];
#pragma unroll
            for (int m = 0; m < 2; m++) {
                const uint32_t l = m ? ql[h][t].y : ql[h][t].x, hq = m ? qh[h].y : qh[h].x;
                const uint32_t hb = k < 2 ? hq << (4 - 2 * k) : hq >> (2 * k - 4);
                w[m] = ((i ? l >> 4 : l) & 0x0f0f0f0fu) | (hb & 0x30303030u);
            }
            gf_bytes(w[0], w[1], ds * GF_TWO24, -32.0f * ds, v + 8 * t);
        }
    }
};

// Q8_0: a 256-value unit is eight 34-byte blocks, a stage two of them.
struct GfQ80 {
    static constexpr uint32_t UB = 272u;
    uint2 qs[8];
    uint16_t d[8];
    __device__ __forceinline__ void load(const uint8_t *blk, uint32_t q) {
#pragma unroll
        for (int b = 0; b < 8; b++) {
            d[b] = *(const uint16_t *)(blk + 34u * b);
            qs[b] = gf_load8(blk + 34u * b + 2u + 8u * q);
        }
    }
    template <int ST> __device__ __forceinline__ void decode(uint32_t, float *v) const {
#pragma clang fp contract(off)
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const float df = f16_to_f32(d[2 * ST + t]);
            gf_bytes(qs[2 * ST + t].x ^ 0x80808080u, qs[2 * ST + t].y ^ 0x80808080u,
                     df * GF_TWO24, -128.0f * df, v + 8 * t);
        }
    }
};

// Stage copy of x: 1 KiB per instruction, four tokens of 64 values each;
// wave w copies tokens 16 w .. 16 w + 15. Lane l of copy k lands on token
// t = 16 w + 4 k + l / 16, chunk l % 16, so it reads chunk (l % 16) ^ (t % 16).
// xo: the lane's four offsets from the tile's first token (bytes; buffer
// loads, so that a stage is one scalar offset and no 64-bit addresses live).
MYNAH_DEV void gf_stage_x(float *buf, __amdgpu_buffer_rsrc_t xr, const uint32_t (&xo)[4],
                          uint32_t stage, uint32_t wave) {
#pragma unroll
    for (uint32_t k = 0; k < 4; k++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            xr, (gf_lds_void *)(buf + 1024u * wave + 256u * k), 16, xo[k], 256u * stage, 0, 0);
}

// A wave's 16 rows x 64 tokens into out[token][row] (+ res): register 4 b + e
// of lane l is row 4 (l / 16) + e, token 16 b + l % 16; the four rows of a
// block go out together where they all exist.
MYNAH_DEV void gf_store(float *out, const gf_f32x16 v, const float *res, uint32_t rows,
                        uint32_t tokens, uint32_t row0, uint32_t tok0, uint32_t lane) {
#pragma clang fp contract(off)
    const uint32_t row = row0 + 4u * (lane >> 4);
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const uint32_t t = tok0 + 16u * b + (lane & 15u);
        if (t >= tokens || row >= rows) continue;
        const size_t o = (size_t)t * rows + row;
        if (row + 3u < rows) {
            float f[4] = {v[4 * b], v[4 * b + 1], v[4 * b + 2], v[4 * b + 3]};
            if (res) {
                float rv[4];
                __builtin_memcpy(rv, res + o, sizeof rv);
#pragma unroll
                for (int e = 0; e < 4; e++) f[e] = rv[e] + f[e];
            }
            __builtin_memcpy(out + o, f, sizeof f);
        } else {
            for (uint32_t e = 0; e < 4u && row + e < rows; e++) {
                const float f = e == 0 ? v[4 * b] : e == 1 ? v[4 * b + 1] : v[4 * b + 2];
                out[o + e] = res ? res[o + e] + f : f;
            }
        }
    }
}

// The products and sums of one stage: A of column col in register v[8 (col /
// 32) + col % 8], block (col / 8) % 4; x chunk c of the lane's token at byte
// xa ^ 16 c of xs. Columns go in the summation order: natural, or (MIXED, the
// Q4_K / Q5_K matvec order) low and high halves alternating. FOLD32: every
// 32 columns' sum joins acc on its own (the Q8_0 matvec order).
template <bool MIXED, bool FOLD32>
MYNAH_DEV void gf_stage(gf_f32x16 &s, gf_f32x16 &acc, const float *v, const uint8_t *xs,
                        uint32_t xa) {
#pragma clang fp contract(off)
    const gf_f32x16 zero = {};
    // x of steps 4 i .. 4 i + 3: chunk i, or (MIXED) the halves' values 2 i and
    // 2 i + 1, low, high, low, high.
    auto fetch = [&](int i) __attribute__((always_inline)) {
        if constexpr (!MIXED) {
            return *(const gm_f4 *)(xs + (xa ^ (16u * (uint32_t)i)));
        } else {
            const uint8_t *p = xs + (xa ^ (16u * (uint32_t)(i >> 1))) + 8u * (uint32_t)(i & 1);
            const gm_f2 lo = *(const gm_f2 *)p;
            const gm_f2 hi = *(const gm_f2 *)(xs + (xa ^ (16u * (uint32_t)(i >> 1) + 128u)) +
                                              8u * (uint32_t)(i & 1));
            return gm_f4{lo.x, hi.x, lo.y, hi.y};
        }
    };
    auto product = [&](const float b, int i) __attribute__((always_inline)) {
        const int col = MIXED ? 32 * (i & 1) + (i >> 1) : i;
        const float a = v[8 * (col / 32) + col % 8];
        switch ((col / 8) % 4) {
        case 0: return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, zero, 2, 0, 0);
        case 1: return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, zero, 2, 1, 0);
        case 2: return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, zero, 2, 2, 0);
        default: return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, zero, 2, 3, 0);
        }
    };
    gm_f4 xc = fetch(0), xn = fetch(1);
    gf_f32x16 pc = product(xc.x, 0);
#pragma unroll
    for (int i = 0; i < 64; i += 4) {
        const float b[4] = {xc.y, xc.z, xc.w, xn.x};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            gf_f32x16 pn = pc;
            if (i + c + 1 < 64) pn = product(b[c], i + c + 1);
            // The next column's MFMA stays ahead of this column's adds.
            __builtin_amdgcn_sched_barrier(0);
            s = s + pc;
            __builtin_amdgcn_sched_barrier(0);
            pc = pn;
        }
        if (FOLD32 && (i & 31) == 28) {
            acc = acc + s;
            s = zero;
        }
        xc = xn;
        if (i + 8 < 64) xn = fetch(i / 4 + 2);
    }
}

// Four registers of the four lane quarters transposed: r[i] of quarter j
// becomes r[j] of quarter i.
MYNAH_DEV void gf_transpose(float &r0, float &r1, float &r2, float &r3) {
    uint32_t a = __float_as_uint(r0), b = __float_as_uint(r1), c = __float_as_uint(r2),
             d = __float_as_uint(r3);
    const auto ac = __builtin_amdgcn_permlane32_swap(a, c, false, false);
    const auto bd = __builtin_amdgcn_permlane32_swap(b, d, false, false);
    const auto ab = __builtin_amdgcn_permlane16_swap(ac[0], bd[0], false, false);
    const auto cd = __builtin_amdgcn_permlane16_swap(ac[1], bd[1], false, false);
    r0 = __uint_as_float(ab[0]);
    r1 = __uint_as_float(ab[1]);
    r2 = __uint_as_float(cd[0]);
    r3 = __uint_as_float(cd[1]);
}

// gf_stage for a tile whose tokens fill only G of its four 16-token groups:
// the MFMA's four blocks are four consecutive columns of one group instead of
// one column of four groups, so a stage takes 16 G MFMAs and their adds where
// gf_stage takes 64 whatever the tokens. 9728 x 2560 Q4_K, 16 tokens: 67 -> 30
// us; 2560 x 9728 Q6_K, 70 -> 33; 4096 x 2560 Q5_K, 32 tokens: 39.6 -> 28. Its
// own kernels: beside gf_stage in one kernel it spills. Block b (lane quarter b) of product (m, g) is step 4 m + b of the
// summation order; its register 4 b + e joins s[4 g + e], b = 0 .. 3 in order.
// The weights come decoded with a quarter's own eight columns (see load); one
// 4 x 4 transpose of registers and quarters per 16 of them puts each step's
// weight in its quarter.
template <bool MIXED, bool FOLD32, int G>
MYNAH_DEV void gf_stage_few(gf_f32x16 &s, gf_f32x16 &acc, float *v, const uint8_t *xs,
                            uint32_t buf, uint32_t lane) {
#pragma clang fp contract(off)
    const gf_f32x16 zero = {};
    const uint32_t t = lane & 15u, q = lane >> 4;
    // Step 4 m + b: natural, column 4 m + b = value 8 Q + J of a half, Q = m / 2
    // % 4, J = 4 (m % 2) + b; MIXED, value 2 m + b / 2 of half b % 2, Q = m / 4,
    // J = 2 (m % 4) + b / 2. a[m]: this quarter's step of product m.
    float a[16];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if constexpr (MIXED) {
            gf_transpose(v[2 * k], v[8 + 2 * k], v[2 * k + 1], v[8 + 2 * k + 1]);
            a[k] = v[2 * k];
            a[4 + k] = v[8 + 2 * k];
            a[8 + k] = v[2 * k + 1];
            a[12 + k] = v[8 + 2 * k + 1];
        } else {
            gf_transpose(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
#pragma unroll
            for (int Q = 0; Q < 4; Q++) a[8 * (k / 2) + 2 * Q + k % 2] = v[4 * k + Q];
        }
    }
    // x of product (m, g): the same step of token 16 g + t.
    auto fetch = [&](int i) __attribute__((always_inline)) {
        const uint32_t m = (uint32_t)(i / G), g = (uint32_t)(i % G);
        const uint32_t c = MIXED ? 8u * (q & 1u) + (m >> 1) : m;
        const uint32_t e = MIXED ? 2u * (m & 1u) + (q >> 1) : q;
        return *(const float *)(xs + buf + 4096u * g + 256u * t + 16u * (c ^ t) + 4u * e);
    };
    auto product = [&](const float b, int i) __attribute__((always_inline)) {
        return __builtin_amdgcn_mfma_f32_16x16x1f32(a[i / G], b, zero, 0, 0, 0);
    };
    constexpr int N = 16 * G, AHEAD = FOLD32 && G == 1 ? 2 : MIXED && G == 2 ? 3 : 4;
    float xb[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) xb[i] = fetch(i);
    gf_f32x16 pc = product(xb[0], 0);
#pragma unroll
    for (int i = 0; i < N; i++) {
        gf_f32x16 pn = pc;
        if (i + AHEAD < N) xb[i % AHEAD] = fetch(i + AHEAD);
        if (i + 1 < N) pn = product(xb[(i + 1) % AHEAD], i + 1);
        __builtin_amdgcn_sched_barrier(0);
        const int g = i % G;
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) s[4 * g + e] = s[4 * g + e] + pc[4 * b + e];
        __builtin_amdgcn_sched_barrier(0);
        if (FOLD32 && (i / G) % 8 == 7) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                acc[4 * g + e] = acc[4 * g + e] + s[4 * g + e];
                s[4 * g + e] = 0.0f;
            }
        }
        pc = pn;
    }
}

// KW: the waves of a workgroup that share a row group, each taking every
// KW-th super-block (the z-th split's units u0 + KW round + kz); the running
// row total passes from one to the next through LDS after every round, in
// unit order. KW = 1 keeps it in registers. G: the tile's 16-token groups (4,
// or fewer where the whole launch has no more tokens).
template <class Raw, int ORD, int FMT, uint32_t KW, int G = 4>
MYNAH_DEV void gemm_mfma(const uint8_t *__restrict__ w, const float *__restrict__ x, float *y,
                         uint32_t rows, uint32_t cols, uint32_t tokens, uint32_t row_bytes,
                         const float *res, float *__restrict__ part) {
#pragma clang fp contract(off)
    constexpr bool FOLD32 = ORD == 1 && FMT == 8;
    static_assert(KW == 1 || !FOLD32, "the Q8_0 matvec order has no unit sums to hand on");
    __shared__ __attribute__((aligned(16))) float xl[KW][2][GF_TOK * 64];
    __shared__ __attribute__((aligned(16))) gm_f4 hand[KW > 1 ? 4 : 1][4][64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wv & 3u, kz = wv >> 2;
    const uint32_t row0 = blockIdx.x * GF_ROWS + 16u * wave, tok0 = blockIdx.y * GF_TOK;
    const uint32_t units = cols / 256u;
    const uint32_t nz = gridDim.z, z = blockIdx.z;
    const uint32_t u0 = units * z / nz, u1 = units * (z + 1u) / nz;
    const bool split = nz > 1u;
    const uint32_t q = lane >> 4, r16 = lane & 15u;
    const uint32_t wr = row0 + r16 < rows ? row0 + r16 : rows - 1u;
    const uint8_t *blk = w + (size_t)wr * row_bytes + (size_t)Raw::UB * (u0 + kz);
    const uint32_t tmax = tokens - 1u - tok0;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(x + (size_t)tok0 * cols + 256u * u0), 0, 0xffffffffu, 0x00020000);
    uint32_t xo[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
        const uint32_t t = 16u * wave + 4u * k + q;
        xo[k] = (t < tmax ? t : tmax) * cols * 4u + 16u * (r16 ^ (t & 15u));
    }
    // Chunk c of this lane's token: byte xa ^ 16 c of the buffers, the buffer
    // toggled by bit 14 each stage (a value the loop carries, so that no
    // address made from it is kept in a register across the loop). stage
    // counts 64-value stages from u0.
    uint32_t xa = lane * 256u + 16u * r16, stage = 4u * kz;
    const gf_f32x16 zero = {};
    gf_f32x16 acc = zero, s = zero;
    Raw raw;
    if (u0 + kz < u1) {
        if (wave < (uint32_t)G) gf_stage_x(xl[kz][0], xr, xo, stage, wave);
        raw.load(blk, q);
    }
    for (uint32_t ub = u0; ub < u1; ub += KW) {
        const uint32_t u = ub + kz;
        const bool active = KW == 1 || u < u1;          // wave-uniform
        const bool more = u + KW < u1;
        s = zero;
#pragma nounroll
        for (uint32_t st = 0; st < 4u; st++) {
            // This stage's x (copied a stage ago) is in for every wave, and
            // every wave is done with the other buffer.
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (active) {
                stage += st == 3u ? 4u * KW - 3u : 1u;
                if (wave < (uint32_t)G && (st < 3u || more)) gf_stage_x(xl[kz][(st + 1u) & 1u], xr, xo, stage, wave);
                float v[16];
                if (st == 0) raw.template decode<0>(q, v);
                else if (st == 1) raw.template decode<1>(q, v);
                else if (st == 2) raw.template decode<2>(q, v);
                else raw.template decode<3>(q, v);
                if (st == 3u) {
                    blk += (size_t)Raw::UB * KW;
                    if (more) raw.load(blk, q);
                }
                constexpr bool MIXED = ORD == 1 && (FMT == 12 || FMT == 13);
                if constexpr (G == 4)
                    gf_stage<MIXED, FOLD32>(s, acc, v, (const uint8_t *)xl[kz], xa);
                else
                    gf_stage_few<MIXED, FOLD32, G>(s, acc, v, (const uint8_t *)xl[kz],
                                                   xa & (4u * 64u * GF_TOK), lane);
                xa ^= 4u * 64u * GF_TOK;
            }
        }
        if (FOLD32) continue;
        if (split && z > 0u) {
            // Unit u's sums, for the in-order fold: slot 1 + its place past
            // the first split's units.
            if (active)
                gf_store(part + (size_t)(u - units / nz + 1u) * tokens * rows, s, nullptr, rows,
                         tokens, row0, tok0, (xa >> 8) & 63u);
        } else if (KW == 1) {
            acc = acc + s;
        } else {
#pragma nounroll
            for (uint32_t k = 0; k < KW; k++) {
                if (k == kz && active) {
                    gf_f32x16 t = zero;
                    if (u > u0) {
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const gm_f4 h = hand[wave][i][lane];
#pragma unroll
                            for (int e = 0; e < 4; e++) t[4 * i + e] = h[e];
                        }
                    }
                    t = t + s;
                    if (u + 1u < u1) {
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            hand[wave][i][lane] =
                                gm_f4{t[4 * i], t[4 * i + 1], t[4 * i + 2], t[4 * i + 3]};
                    } else {
                        // The split's last unit. The first split's total
                        // starts the row total: slot 0 of the partials.
                        gf_store(split ? part : y, t, split ? nullptr : res, rows, tokens, row0,
                                 tok0, (xa >> 8) & 63u);
                    }
                }
                if (k + 1u < KW) __syncthreads();
            }
        }
    }
    if (KW > 1 || (split && z > 0u)) return;
    gf_store(split ? part : y, acc, split ? nullptr : res, rows, tokens, row0, tok0, lane);
}

// Grid (ceil(rows / 64), ceil(tokens / 64), Z), block 256 KW; cols % 256 == 0;
// 256 cols < 2^32; x 16-byte aligned; Q4_K / Q5_K rows 16-byte aligned, Q6_K /
// Q8_0 2-byte aligned. ORD 0 = the batched order, 1 = the matvec order; res
// (may be NULL or alias y) is added when Z == 1; part: Z > 1 only.
#define GEMM_MFMA_ENTRY(name, RAW, ORD, FMT, KW)                                              \
    extern "C" __global__ void __launch_bounds__(256 * KW, 4)                                  \
        name(const uint8_t *__restrict__ w, const float *__restrict__ x, float *y,             \
             uint32_t rows, uint32_t cols, uint32_t tokens, uint32_t row_bytes,                \
             const float *res, float *part) {                                                  \
        gemm_mfma<RAW, ORD, FMT, KW>(w, x, y, rows, cols, tokens, row_bytes, res, part);       \
    }
#define GEMM_MFMA_ENTRIES(name, RAW, ORD, FMT)                                                \
    GEMM_MFMA_ENTRY(name##1, RAW, ORD, FMT, 1)                                                 \
    GEMM_MFMA_ENTRY(name##2, RAW, ORD, FMT, 2)                                                 \
    GEMM_MFMA_ENTRY(name##4, RAW, ORD, FMT, 4)

GEMM_MFMA_ENTRIES(mynah_q4k_gemm_exact_mfma, GfQ4K, 0, 12)
GEMM_MFMA_ENTRIES(mynah_q5k_gemm_exact_mfma, GfQ5K, 0, 13)
GEMM_MFMA_ENTRIES(mynah_q6k_gemm_exact_mfma, GfQ6K, 0, 14)
GEMM_MFMA_ENTRIES(mynah_q80_gemm_exact_mfma, GfQ80, 0, 8)
GEMM_MFMA_ENTRIES(mynah_q4k_gemm_mv_mfma, GfQ4K, 1, 12)
GEMM_MFMA_ENTRIES(mynah_q5k_gemm_mv_mfma, GfQ5K, 1, 13)
GEMM_MFMA_ENTRY(mynah_q80_gemm_mv_mfma1, GfQ80, 1, 8, 1)

// At most 16 G tokens: grid (ceil(rows / 64), 1, Z), block 256. Four waves a
// SIMD like the full tile's, which the host's plan counts on: left at 129 - 132
// registers, four of them held three (17 - 32 tokens: 6874 x 8448 Q4_K, matvec
// order 110 -> 95 us, 10434 x 4096 Q5_K 88 -> 78, 7229 x 8448 Q6_K 115 -> 100).
// x is read fewer steps ahead where the registers would not hold it; the Q6_K
// form for 32 tokens spills one.
#define GEMM_FEW_ENTRY(name, RAW, ORD, FMT, G)                                                \
    extern "C" __global__ void __launch_bounds__(256, 4)                                       \
        name(const uint8_t *__restrict__ w, const float *__restrict__ x, float *y,             \
             uint32_t rows, uint32_t cols, uint32_t tokens, uint32_t row_bytes,                \
             const float *res, float *part) {                                                  \
        gemm_mfma<RAW, ORD, FMT, 1, G>(w, x, y, rows, cols, tokens, row_bytes, res, part);     \
    }
#define GEMM_FEW_ENTRIES(name, RAW, ORD, FMT)                                                 \
    GEMM_FEW_ENTRY(name##16, RAW, ORD, FMT, 1)                                                 \
    GEMM_FEW_ENTRY(name##32, RAW, ORD, FMT, 2)
GEMM_FEW_ENTRIES(mynah_q4k_gemm_exact_few, GfQ4K, 0, 12)
GEMM_FEW_ENTRIES(mynah_q5k_gemm_exact_few, GfQ5K, 0, 13)
GEMM_FEW_ENTRIES(mynah_q6k_gemm_exact_few, GfQ6K, 0, 14)
GEMM_FEW_ENTRIES(mynah_q80_gemm_exact_few, GfQ80, 0, 8)
GEMM_FEW_ENTRIES(mynah_q4k_gemm_mv_few, GfQ4K, 1, 12)
GEMM_FEW_ENTRIES(mynah_q5k_gemm_mv_few, GfQ5K, 1, 13)
GEMM_FEW_ENTRIES(mynah_q80_gemm_mv_few, GfQ80, 1, 8)

// The in-order fold of split-K unit sums: y[t][r] = (res[t][r] +) the row
// total continued from part[0][t][r] (the first split's running total) over
// part[i][t][r], i = 1 .. slots - 1 (the later units' sums) in order — the row
// total of the reference's order. One thread per output, consecutive rows
// consecutive threads; the loads go out four at a time.
extern "C" __global__ void __launch_bounds__(256)
mynah_gemm_fold(const float *__restrict__ part, const float *res, float *y, uint32_t rows,
                uint32_t tokens, uint32_t slots) {
#pragma clang fp contract(off)
    const uint64_t n = (uint64_t)rows * tokens;
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float acc = part[i];
    uint32_t u = 1u;
    for (; u + 4u <= slots; u += 4u) {
        float v[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) v[k] = part[(size_t)(u + k) * n + i];
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) acc = acc + v[k];
    }
    for (; u < slots; u++) acc = acc + part[(size_t)u * n + i];
    y[i] = res ? res[i] + acc : acc;
}

// Test hook for the product claim at the top of this file (no reference
// counterpart). Per workgroup (one wave): 64 values of a and of b, lane l
// feeding A and B of block l / 16 at row / column l % 16, and 1024 of c.
// prod = the instruction with a zero accumulator, acc = the same with c as
// the accumulator; mul and fused = the VALU's a * b and fmaf(a, b, c) of the
// same operand pairs. Every output is in the instruction's layout: lane l,
// register r holds block r / 4, row 4 (l / 16) + r % 4, column l % 16, at
// index 1024 blockIdx + 16 l + r.
extern "C" __global__ void __launch_bounds__(64)
mynah_mfma_probe(const float *__restrict__ a, const float *__restrict__ b,
                 const float *__restrict__ c, float *__restrict__ prod,
                 float *__restrict__ acc, float *__restrict__ mul, float *__restrict__ fused) {
#pragma clang fp contract(off)
    const uint32_t l = threadIdx.x;
    const size_t base = 64u * (size_t)blockIdx.x, out = 16u * (base + l);
    const gf_f32x16 zero = {};
    gf_f32x16 cv;
#pragma unroll
    for (int r = 0; r < 16; r++) cv[r] = c[out + r];
    const gf_f32x16 p = __builtin_amdgcn_mfma_f32_16x16x1f32(a[base + l], b[base + l], zero, 0, 0, 0);
    const gf_f32x16 q = __builtin_amdgcn_mfma_f32_16x16x1f32(a[base + l], b[base + l], cv, 0, 0, 0);
#pragma unroll
    for (uint32_t r = 0; r < 16; r++) {
        const uint32_t blk = r / 4u, row = 4u * (l / 16u) + r % 4u, col = l % 16u;
        const float x = a[base + 16u * blk + row], y = b[base + 16u * blk + col];
        prod[out + r] = p[r];
        acc[out + r] = q[r];
        mul[out + r] = x * y;
        fused[out + r] = __builtin_fmaf(x, y, cv[r]);
    }
}
