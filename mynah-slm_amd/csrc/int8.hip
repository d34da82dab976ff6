// int8.hip — the int8 activation lane of Q4_K products: the activation
// quantiser, the int8 matvec and the batched int8 GEMM on the matrix cores.
//
// The reference computes this lane in an AVX2 + FMA build of ingot
// (third_party/ingot/src/kernels.c:636-788 for the matvec, 1120-1751 for the
// batched form). Its arithmetic, which these kernels keep:
//   * quantiser (kernels.c:675-708): per 256-value super-block of a token,
//     amax = max |x|; scale = amax / 127, q = round-half-even(x * (127 / amax))
//     as int8; the eight sums of q over 32-value sub-blocks (all zero when
//     amax is 0);
//   * integer dots: Q4_K quants (0..15) times q over each 32-value sub-block,
//     exact in int32 whatever the order;
//   * matvec epilogue (kernels.c:712-739): per super-block
//     total = 0; per group g: total += d*sc*dot - dmin*m*sum for the low then
//     the high sub-block (products and sums separately rounded); the block's
//     value total * scale, summed over the row's super-blocks in order from 0;
//   * batched epilogue (kernels.c:1495-1581): per super-block and
//     (row, token), with scale_j = d*sc_j, offset_j = dmin*m_j:
//     total = fma(dot_j, scale_j, total); total = fma(-sum_j, offset_j, total)
//     for j = 0..7, for the tokens of a token tile that fall in whole groups
//     of four; the tile's last (count % 4) tokens take
//     total += scale_j*dot_j - offset_j*sum_j; then acc += total * scale,
//     super-block after super-block. The token tile is
//     clamp(4 MiB / (4 cols), 32, 128) rounded down to even (kernels.c:893-920).
// So every output is bit-identical to that build of the reference.
//
// Quantised activations live in HBM as xq[token][cols] int8,
// xs[token][cols / 256] f32 and xsum[token][cols / 32] int32.
//
// SPDX-License-Identifier: MIT
#include "common.hip.h"
#include "scratch.h"

typedef int i32x4 __attribute__((ext_vector_type(4)));

// The workspace of the allocation-free int8 product: one fixed array per
// device (each GPU that loads the code object holds its own copy until the
// process ends). The host resolves its device address by name when it loads
// the code object and passes that address to the kernels below as their xq /
// xs / xsum operands; nothing reads it before the quantiser has written it.
// No kernel names it (they take its address as an argument), so `used`
// keeps it in the code object's symbol table; the braces make this a
// definition with C linkage (a bare `extern "C"` would only declare it).
extern "C" {
__device__ __attribute__((aligned(256), used, visibility("default")))
unsigned char mynah_scratch[MYNAH_SCRATCH_BYTES];
}

// The (scale, min) pair of sub-block j from the 12 scale bytes s0..s2
// (kernels.c:83-92, scale_min), selects only.
MYNAH_DEV void q4k_scale_min(uint32_t s0, uint32_t s1, uint32_t s2, uint32_t j, uint32_t *sc,
                             uint32_t *m) {
    auto byte = [&](uint32_t k) -> uint32_t {
        const uint32_t wd = k < 4u ? s0 : (k < 8u ? s1 : s2);
        return (wd >> (8u * (k & 3u))) & 0xffu;
    };
    if (j < 4u) {
        *sc = byte(j) & 63u;
        *m = byte(j + 4u) & 63u;
    } else {
        *sc = (byte(j + 4u) & 15u) | ((byte(j - 4u) >> 6) << 4);
        *m = (byte(j + 4u) >> 4) | ((byte(j) >> 6) << 4);
    }
}

// ── quantiser ───────────────────────────────────────────────────────────
// One wave per (token, super-block); lane l holds values 4l..4l+3, so the
// lanes 8s..8s+7 hold sub-block s.
extern "C" __global__ __launch_bounds__(256) void mynah_q8_quantize(
    const float *__restrict__ x, int8_t *__restrict__ xq, float *__restrict__ xs,
    int32_t *__restrict__ xsum, uint32_t n_units, uint32_t nb, uint32_t cols) {
#pragma clang fp contract(off)
    const uint32_t u = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (u >= n_units) return;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t t = u / nb, b = u - t * nb;
    const size_t off = (size_t)t * cols + 256u * b + 4u * lane;
    const float4 v = *(const float4 *)(x + off);
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    for (int m = 32; m >= 1; m >>= 1) amax = fmaxf(amax, __shfl_xor(amax, m, 64));
    uint32_t packed = 0u;
    int32_t s = 0;
    float scale = 0.0f;
    if (amax > 0.0f) {
        scale = amax / 127.0f;
        const float inv = 127.0f / amax;
        const int32_t q0 = (int32_t)__builtin_rintf(v.x * inv);
        const int32_t q1 = (int32_t)__builtin_rintf(v.y * inv);
        const int32_t q2 = (int32_t)__builtin_rintf(v.z * inv);
        const int32_t q3 = (int32_t)__builtin_rintf(v.w * inv);
        s = q0 + q1 + q2 + q3;
        // |q| <= 127 here (|x| <= amax), so the saturating packs are identities.
        packed = ((uint32_t)q0 & 0xffu) | (((uint32_t)q1 & 0xffu) << 8) |
                 (((uint32_t)q2 & 0xffu) << 16) | ((uint32_t)q3 << 24);
    }
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    s += __shfl_xor(s, 4, 64);
    *(uint32_t *)(xq + off) = packed;
    if ((lane & 7u) == 0u) xsum[(size_t)u * 8u + (lane >> 3)] = s;
    if (lane == 0u) xs[u] = scale;
}

// ── int8 matvec (tokens == 1) ───────────────────────────────────────────
// One thread per (row, super-block): a workgroup owns `rpw` whole rows
// (rpw * nb <= 256 when nb <= 256), computes every block value into LDS, and
// one thread per row sums its row's values in order.
MYNAH_DEV float q4k_block_int8(const uint8_t *__restrict__ blk, const int8_t *__restrict__ q,
                               float xscale, const int32_t *__restrict__ sums) {
#pragma clang fp contract(off)
    const uint4 hdr = *(const uint4 *)blk;
    uint4 qs[8];
#pragma unroll
    for (int k = 0; k < 8; k++) qs[k] = ((const uint4 *)(blk + 16))[k];
    uint4 xv[16];
#pragma unroll
    for (int k = 0; k < 16; k++) xv[k] = ((const uint4 *)q)[k];
    const int4 s0 = ((const int4 *)sums)[0], s1 = ((const int4 *)sums)[1];
    const int32_t sm[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
    const float d = f16_to_f32(hdr.x), dmin = f16_to_f32(hdr.x >> 16);
    float total = 0.0f;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        // Group g: quant bytes 32g..32g+31 = qs[2g], qs[2g+1]; the low nibbles
        // are sub-block 2g, the high ones 2g+1.
        const uint32_t wq[8] = {qs[2 * g].x,     qs[2 * g].y,     qs[2 * g].z,     qs[2 * g].w,
                                qs[2 * g + 1].x, qs[2 * g + 1].y, qs[2 * g + 1].z, qs[2 * g + 1].w};
        const uint4 xl0 = xv[4 * g], xl1 = xv[4 * g + 1], xh0 = xv[4 * g + 2], xh1 = xv[4 * g + 3];
        const uint32_t wl[8] = {xl0.x, xl0.y, xl0.z, xl0.w, xl1.x, xl1.y, xl1.z, xl1.w};
        const uint32_t wh[8] = {xh0.x, xh0.y, xh0.z, xh0.w, xh1.x, xh1.y, xh1.z, xh1.w};
        int32_t dl = 0, dh = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            dl = __builtin_amdgcn_sdot4((int)(wq[k] & 0x0f0f0f0fu), (int)wl[k], dl, false);
            dh = __builtin_amdgcn_sdot4((int)((wq[k] >> 4) & 0x0f0f0f0fu), (int)wh[k], dh, false);
        }
        uint32_t sl, ml, sh, mh;
        q4k_scale_min(hdr.y, hdr.z, hdr.w, 2u * g, &sl, &ml);
        q4k_scale_min(hdr.y, hdr.z, hdr.w, 2u * g + 1u, &sh, &mh);
        total += d * (float)sl * (float)dl - dmin * (float)ml * (float)sm[2 * g];
        total += d * (float)sh * (float)dh - dmin * (float)mh * (float)sm[2 * g + 1];
    }
    return total * xscale;
}

extern "C" __global__ __launch_bounds__(256) void mynah_q4k_gemv_int8(
    const uint8_t *__restrict__ w, const int8_t *__restrict__ xq, const float *__restrict__ xs,
    const int32_t *__restrict__ xsum, float *__restrict__ y, uint32_t rows, uint32_t nb,
    uint32_t rpw) {
#pragma clang fp contract(off)
    extern __shared__ float blockv[];   // rpw * nb values
    const uint32_t r0 = blockIdx.x * rpw;
    const uint32_t nrows = rows - r0 < rpw ? rows - r0 : rpw;
    const uint32_t n = nrows * nb;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
        const uint32_t rr = i / nb, b = i - rr * nb;
        const uint8_t *blk = w + ((size_t)(r0 + rr) * nb + b) * 144u;
        blockv[i] = q4k_block_int8(blk, xq + 256u * b, xs[b], xsum + 8u * b);
    }
    __syncthreads();
    for (uint32_t rr = threadIdx.x; rr < nrows; rr += blockDim.x) {
        float s = 0.0f;
        for (uint32_t b = 0; b < nb; b++) s += blockv[rr * nb + b];
        y[r0 + rr] = s;
    }
}

// ── batched int8 GEMM (tokens >= 2) ─────────────────────────────────────
// A workgroup is WR x WT waves, each owning GI_TR 16-row tiles and GI_TT
// 16-token tiles.
// Per super-block and sub-block j, one v_mfma_i32_16x16x32_i8 per tile gives
// the tile's integer dots, tokens as A and rows as B: lane l feeds token
// (l % 16) and row (l % 16) with the 8 positions 8 (l / 16) .. + 7 of the
// sub-block, and receives the dots of tokens 4 (l / 16) + e, e = 0..3, for row
// l % 16. So a lane's scale and offset of a sub-block are one pair per row
// tile, and its tokens' sums one float4 per token tile, shared by all its
// tiles. Sub-blocks 2g and 2g+1 are the low and high nibbles of the same 8
// quant bytes: one 8-byte read per group.
// The accumulator starts at the bits of 1.5 * 2^23, whose unit is 1: the
// integer result, read as a float, is 1.5 * 2^23 + dot (|dot| < 2^17), and one
// subtraction gives the dot as an exact float. On gfx950 that subtraction (two
// operands, a literal) issues at twice the rate of a conversion.
// Operands go through LDS: per super-block the workgroup copies its rows'
// quant bytes (Q5_K: qh and qs) and its tokens' activations and scales
// straight from global memory into LDS (global_load_lds_dwordx4 / _dword: no
// registers, nothing for the compiler to move), double buffered, the next
// super-block's copy in flight while the current one is summed; the rows'
// (scale_j, -offset_j) and the tokens' sums as floats are computed into LDS
// from block headers and sums held in registers a super-block ahead. One
// barrier per super-block.
// What bounds it: issue. Per tile (256 outputs) and sub-block an i8 MFMA (7.0
// ns of its SIMD), 4 subtractions and 8 v_fmac (1.04 each) do not overlap: 19.5
// ns. The 128 x 128 tile alone has the four tiles a wave that a rank-one MFMA
// takes (13.5 ns for 16 v_fmac): 18.8. The tile the host picks for 6144 x 2048,
// 512 tokens is 96 x 128 (three a wave) and for 4096 x 2560, 130 tokens 32 x 32
// (one): 15 and 3.2 us by these, against calls of 38 and 28 (31 of them the
// first's kernel). In that they are 9.4 of 17.2 million VALU instructions; unpacking, staging and
// addresses are the others, about 9 us, and the rest waits for copies and the
// barrier of each super-block. Measured on MI355X with the
// quantiser, the form before (64 x 64 tiles, activations as the MFMA's columns,
// a conversion per dot) and this: 9728 x 2560 Q4_K, 2047 tokens 347 -> 245 us;
// 6144 x 2048, 512 tokens 57 -> 38 us; 4096 x 2560 Q5_K, 130 tokens 45 -> 28 us.
// Q5_K (FMT 13, kernels.c:1155-1185 q5_k_quants): the same tiles, the quant
// bytes at block offset 48 instead of 16, and each lane also holds the 8 qh
// bytes of its 8 positions: bit j of qh[i] is the fifth bit (+16) of weight
// i of sub-block j.
typedef __attribute__((address_space(3))) void gi_lds_void;

// One super-block's operands in LDS. A row's 128 quant bytes and a token's 256
// activations lie contiguous, 16-byte chunk c at place c ^ (row / 2 % 8) or c ^
// (token % 16), so that both the copies' global reads (whole rows) and the
// operand reads (16 rows or tokens, one chunk) meet no conflict.
template <int FMT, int ROWS, int TOK> struct GiBuf {
    uint8_t q[ROWS * 128];
    int8_t x[TOK * 256];
    uint8_t qh[FMT == 13 ? ROWS * 32 : 16];
    float sc[8 * ROWS];              // scale_j of row r at ROWS j + r
    float no[8 * ROWS];              // -offset_j
    float fsum[8 * TOK];             // sum_j of token t at TOK j + t
    float xs[TOK];
};

// The copies of a workgroup of NW waves: instruction n (1 KiB: 64 lanes x 16
// bytes) is wave n % NW's; per lane its byte offset from the tile's first row
// or token, the super-block a scalar offset. Rows and tokens past the ends
// read the last one (their results are not stored).
template <int FMT, int ROWS, int TOK, int NW> struct GiCopy {
    static constexpr int NQ = ROWS / 8, NX = TOK / 4, NH = FMT == 13 ? ROWS / 32 : 0;
    static constexpr int PQ = (NQ + NW - 1) / NW, PX = (NX + NW - 1) / NW;
    uint32_t qo[PQ], xo[PX], ho, so;
    __amdgpu_buffer_rsrc_t rq, rx, rs;
    __device__ __forceinline__ void init(const uint8_t *w, const int8_t *xq, const float *xs,
                                         uint32_t R0, uint32_t T0, uint32_t rows, uint32_t tokens,
                                         uint32_t cols, uint32_t nb, uint32_t rb, uint32_t wave,
                                         uint32_t lane) {
        const uint32_t rmax = rows - 1u - R0, tmax = tokens - 1u - T0;
#pragma unroll
        for (int k = 0; k < PQ; k++) {
            const uint32_t r = 8u * (NW * k + wave) + (lane >> 3), p = lane & 7u;
            qo[k] = (r < rmax ? r : rmax) * rb + 16u * (p ^ ((r >> 1) & 7u)) +
                    (FMT == 13 ? 48u : 16u);
        }
#pragma unroll
        for (int k = 0; k < PX; k++) {
            const uint32_t t = 4u * (NW * k + wave) + (lane >> 4), p = lane & 15u;
            xo[k] = (t < tmax ? t : tmax) * cols + 16u * (p ^ (t & 15u));
        }
        const uint32_t hr = 32u * wave + (lane >> 1), st = 64u * wave + lane;
        ho = (hr < rmax ? hr : rmax) * rb + 16u * (lane & 1u) + 16u;
        so = (st < tmax ? st : tmax) * nb * 4u;
        rq = __builtin_amdgcn_make_buffer_rsrc((void *)(w + (size_t)R0 * rb), 0, 0xffffffffu,
                                               0x00020000);
        rx = __builtin_amdgcn_make_buffer_rsrc((void *)(xq + (size_t)T0 * cols), 0, 0xffffffffu,
                                               0x00020000);
        rs = __builtin_amdgcn_make_buffer_rsrc((void *)(xs + (size_t)T0 * nb), 0, 0xffffffffu,
                                               0x00020000);
    }
    __device__ __forceinline__ void copy(GiBuf<FMT, ROWS, TOK> &buf, uint32_t b,
                                         uint32_t wave) const {
        constexpr uint32_t UB = FMT == 13 ? 176u : 144u;
#pragma unroll
        for (int k = 0; k < PQ; k++)
            if (NW * k + wave < (uint32_t)NQ)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rq, (gi_lds_void *)(buf.q + 1024u * (NW * k + wave)), 16, qo[k], UB * b, 0, 0);
#pragma unroll
        for (int k = 0; k < PX; k++)
            if (NW * k + wave < (uint32_t)NX)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rx, (gi_lds_void *)(buf.x + 1024u * (NW * k + wave)), 16, xo[k], 256u * b, 0,
                    0);
        if (FMT == 13 && wave < (uint32_t)NH)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rq, (gi_lds_void *)(buf.qh + 1024u * wave), 16, ho, UB * b, 0, 0);
        if (64u * wave < (uint32_t)TOK) {
            if (TOK % 64 == 0 || (threadIdx.x & 63u) < (uint32_t)TOK)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rs, (gi_lds_void *)(buf.xs + 64u * wave), 4, so, 4u * b, 0, 0);
        }
    }
};

// Scale and -offset of sub-blocks hj, hj + 1 of the staged row, into LDS.
template <int ROWS>
MYNAH_DEV void gi_stage(float *sc, float *no, const uint4 hdr, uint32_t hj, uint32_t row) {
#pragma clang fp contract(off)
    const float d = f16_to_f32(hdr.x), dmin = f16_to_f32(hdr.x >> 16);
    float s0, m0, s1, m1;
    q4k_sm_rt(hdr.y, hdr.z, hdr.w, hj, s0, m0);
    q4k_sm_rt(hdr.y, hdr.z, hdr.w, hj + 1u, s1, m1);
    sc[hj * ROWS + row] = d * s0;
    sc[(hj + 1u) * ROWS + row] = d * s1;
    no[hj * ROWS + row] = -(dmin * m0);
    no[(hj + 1u) * ROWS + row] = -(dmin * m1);
}

// Four of a token's eight sums as floats (exact: |sum| <= 32 * 127), into LDS
// by sub-block.
template <int TOK>
MYNAH_DEV void gi_stage_sums(float *fsum, const int4 v, uint32_t half, uint32_t tok) {
    float *p = fsum + 4u * half * TOK + tok;
    p[0] = (float)v.x;
    p[TOK] = (float)v.y;
    p[2 * TOK] = (float)v.z;
    p[3 * TOK] = (float)v.w;
}

// The bits of 1.5 * 2^23.
#define GI_MAGIC 0x4b400000

typedef float gi_f32x16 __attribute__((ext_vector_type(16)));

// One super-block's dots and epilogue from the LDS buffer, for the wave whose
// rows start at r0 and tokens at t0 of the tile. Tile n = GI_TT i + k of the
// wave is rows 16 i .. + 15, tokens 16 k .. + 15; lane l holds of it row l % 16
// and tokens 4 (l / 16) + e, in element 4 (n % 4) + e of tot[n / 4]. Over j =
// 0..7 in order tot = fma(xsum_j, -offset_j, fma(dot_j, scale_j, tot)), then
// acc += tot * xs. The second fma of four tiles is one MFMA: the outer product
// of 16 sums and 16 offsets per block, accumulated with fmaf's one rounding
// (13.7 ns against 16 v_fmac's 23.5); tiles past the last whole four take
// v_fmac. MIXED: some lane has a token outside the groups of four, which takes
// the plain form total += scale * dot - offset * sum (fma_path bit 4 k + e: the
// token's groups-of-four form).
template <int FMT, bool MIXED, int GI_TR, int GI_TT, int ROWS, int TOK>
MYNAH_DEV void gi_block(gi_f32x16 (&acc)[(GI_TR * GI_TT + 3) / 4],
                        const GiBuf<FMT, ROWS, TOK> &buf, uint32_t r0, uint32_t t0,
                        uint32_t lane, uint32_t fma_path) {
#pragma clang fp contract(off)
    constexpr int NT = GI_TR * GI_TT, NG = (NT + 3) / 4, NM = MIXED ? 0 : NT / 4;
    const uint32_t lm = lane & 15u, lk = lane >> 4;
    // Lane l reads the 8 bytes at position 8 (l / 16) of a 32-byte group:
    // chunk 2 g + (l / 16) / 2 of its row / token, half (l / 16) % 2.
    const uint32_t ck = lk >> 1, hb = 8u * (lk & 1u), sq = lm >> 1, sx = lm;
    const uint8_t *qrow = buf.q + 128u * (r0 + lm) + hb;
    const int8_t *xrow = buf.x + 256u * (t0 + lm) + hb;
    const float *srow = buf.sc + r0 + lm, *nrow = buf.no + r0 + lm;
    const float *frow = buf.fsum + t0 + 4u * lk;
    // Operands of the rank-one MFMA m: lane l feeds its block l / 16's tile.
    const float *mf[NM > 0 ? NM : 1], *mn[NM > 0 ? NM : 1];
#pragma unroll
    for (int m = 0; m < NM; m++) {
        const uint32_t n = 4u * m + lk;
        mf[m] = buf.fsum + t0 + 16u * (n % GI_TT) + lm;
        mn[m] = buf.no + r0 + 16u * (n / GI_TT) + lm;
    }
    uint2 qh[GI_TR];
    if (FMT == 13) {
#pragma unroll
        for (int i = 0; i < GI_TR; i++)
            qh[i] = *(const uint2 *)(buf.qh + 32u * (r0 + lm + 16u * i) + 8u * lk);
    }
    const i32x4 magic = {GI_MAGIC, GI_MAGIC, GI_MAGIC, GI_MAGIC};
    const gi_f32x16 zero = {};
    gi_f32x16 tot[NG];
#pragma unroll
    for (int m = 0; m < NG; m++) tot[m] = zero;
    // Two sub-blocks (a group of quant bytes) per round of the loop, which
    // stays rolled, so no more than one group's dots are ever live.
#pragma unroll 1
    for (uint32_t g = 0; g < 4u; g++) {
        uint2 qa[GI_TR];
#pragma unroll
        for (int i = 0; i < GI_TR; i++)
            qa[i] = *(const uint2 *)(qrow + 2048u * i + 16u * ((2u * g + ck) ^ sq));
        i32x4 dt[2][NT];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            long xb[GI_TT];
#pragma unroll
            for (int k = 0; k < GI_TT; k++)
                xb[k] = *(const long *)(xrow + 4096u * k + 16u * ((4u * g + 2u * h + ck) ^ sx));
#pragma unroll
            for (int i = 0; i < GI_TR; i++) {
                uint2 v = qa[i];
                if (h) v = make_uint2(v.x >> 4, v.y >> 4);
                v = make_uint2(v.x & 0x0f0f0f0fu, v.y & 0x0f0f0f0fu);
                if (FMT == 13) {
                    const uint32_t j = 2u * g + h;
                    v.x |= ((qh[i].x >> j) & 0x01010101u) << 4;
                    v.y |= ((qh[i].y >> j) & 0x01010101u) << 4;
                }
                const long q = (long)(((unsigned long long)v.y << 32) | v.x);
#pragma unroll
                for (int k = 0; k < GI_TT; k++)
                    dt[h][GI_TT * i + k] =
                        __builtin_amdgcn_mfma_i32_16x16x32_i8(xb[k], q, magic, 0, 0, 0);
            }
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t j = 2u * g + h;
            float sc[GI_TR], no[GI_TR];
            float4 fs[GI_TT];
#pragma unroll
            for (int i = 0; i < GI_TR; i++) {
                sc[i] = srow[j * ROWS + 16u * i];
                if (GI_TT * (i + 1) > 4 * NM) no[i] = nrow[j * ROWS + 16u * i];
            }
            if (NT > 4 * NM) {
#pragma unroll
                for (int k = 0; k < GI_TT; k++)
                    fs[k] = *(const float4 *)(frow + j * TOK + 16u * k);
            }
#pragma unroll
            for (int n = 0; n < NT; n++) {
                const int i = n / GI_TT, k = n % GI_TT;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float dv = __int_as_float(dt[h][n][e]) - 12582912.0f;
                    const float t = tot[n / 4][4 * (n % 4) + e];
                    float f = __builtin_fmaf(dv, sc[i], t);
                    if (n >= 4 * NM) {
                        const float xsv = e == 0   ? fs[k].x
                                          : e == 1 ? fs[k].y
                                          : e == 2 ? fs[k].z
                                                   : fs[k].w;
                        f = __builtin_fmaf(xsv, no[i], f);
                        if (MIXED) {
                            const float p = t + (sc[i] * dv + no[i] * xsv);
                            f = (fma_path >> (4 * k + e)) & 1u ? f : p;
                        }
                    }
                    tot[n / 4][4 * (n % 4) + e] = f;
                }
            }
#pragma unroll
            for (int m = 0; m < NM; m++)
                tot[m] = __builtin_amdgcn_mfma_f32_16x16x1f32(mf[m][j * TOK], mn[m][j * ROWS],
                                                              tot[m], 0, 0, 0);
        }
    }
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const float4 x4 = *(const float4 *)(buf.xs + t0 + 16u * (n % GI_TT) + 4u * lk);
        const float xsv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
        for (int e = 0; e < 4; e++)
            acc[n / 4][4 * (n % 4) + e] =
                acc[n / 4][4 * (n % 4) + e] + tot[n / 4][4 * (n % 4) + e] * xsv[e];
    }
}

// WR x WT waves; ROWS = 16 GI_TR WR, TOK = 16 GI_TT WT.
template <int FMT, int WR, int WT, int GI_TR, int GI_TT>
MYNAH_DEV void gemm_int8(const uint8_t *__restrict__ w, const int8_t *__restrict__ xq,
                         const float *__restrict__ xs, const int32_t *__restrict__ xsum,
                         float *__restrict__ y, uint32_t rows, uint32_t cols, uint32_t tokens,
                         uint32_t nb, uint32_t tile) {
    constexpr int ROWS = 16 * GI_TR * WR, TOK = 16 * GI_TT * WT, NW = WR * WT;
    static_assert(4 * ROWS <= 64 * NW && 2 * TOK <= 64 * NW && ROWS % 32 == 0 && TOK % 4 == 0,
                  "staging roles");
    constexpr uint32_t UB = FMT == 13 ? 176u : 144u;
    __shared__ __attribute__((aligned(16))) GiBuf<FMT, ROWS, TOK> buf[2];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r0 = 16u * GI_TR * (wave % WR), t0 = 16u * GI_TT * (wave / WR);
    const uint32_t R0 = blockIdx.x * ROWS, T0 = blockIdx.y * TOK;
    const uint32_t rb = nb * UB;
    const uint32_t lm = lane & 15u, lk = lane >> 4;

    // Bit 4 k + e: token T0 + t0 + 16 k + 4 lk + e falls in a whole group of
    // four of its token tile.
    uint32_t fma_path = 0u;
#pragma unroll
    for (uint32_t k = 0; k < GI_TT; k++)
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) {
            const uint32_t t = T0 + t0 + 16u * k + 4u * lk + e;
            const uint32_t tc = t < tokens ? t : tokens - 1u;
            const uint32_t tb = tc - tc % tile;
            const uint32_t cnt = tokens - tb < tile ? tokens - tb : tile;
            fma_path |= (tc - tb < (cnt & ~3u) ? 1u : 0u) << (4u * k + e);
        }
    const bool mixed = !__all(fma_path == (1u << (4 * GI_TT)) - 1u);
    // Scale staging: thread tid owns row tid / 4 of the workgroup, sub-blocks
    // 2 (tid % 4) and 2 (tid % 4) + 1; sum staging: token tid / 2, sub-blocks
    // 4 (tid % 2) .. + 3 (threads beyond stage none).
    const uint32_t srow = tid >> 2, hj = 2u * (tid & 3u);
    const bool stager = srow < ROWS, summer = tid < 2u * TOK;
    uint32_t hr = R0 + (stager ? srow : 0u), st = T0 + (summer ? tid >> 1 : 0u);
    hr = hr < rows ? hr : rows - 1u;
    st = st < tokens ? st : tokens - 1u;
    const uint8_t *hrow = w + (size_t)hr * rb;
    const int4 *sumrow = (const int4 *)(xsum + (size_t)st * nb * 8u) + (tid & 1u);

    constexpr int NG = (GI_TR * GI_TT + 3) / 4;
    const gi_f32x16 zero = {};
    gi_f32x16 acc[NG];
#pragma unroll
    for (int m = 0; m < NG; m++) acc[m] = zero;

    GiCopy<FMT, ROWS, TOK, NW> cp;
    cp.init(w, xq, xs, R0, T0, rows, tokens, cols, nb, rb, wave, lane);
    cp.copy(buf[0], 0u, wave);
    uint4 hdr = *(const uint4 *)hrow;
    int4 sums = sumrow[0];
    __builtin_amdgcn_s_waitcnt(0);
    if (stager) gi_stage<ROWS>(buf[0].sc, buf[0].no, hdr, hj, srow);
    if (summer) gi_stage_sums<TOK>(buf[0].fsum, sums, tid & 1u, tid >> 1);
    __syncthreads();
    for (uint32_t b = 0; b < nb; b++) {
        const uint32_t c = b & 1u;
        const bool more = b + 1u < nb;
        if (more) {
            hdr = *(const uint4 *)(hrow + (size_t)(b + 1u) * UB);
            sums = sumrow[2u * (b + 1u)];
            cp.copy(buf[c ^ 1u], b + 1u, wave);
        }
        if (mixed)
            gi_block<FMT, true, GI_TR, GI_TT, ROWS, TOK>(acc, buf[c], r0, t0, lane, fma_path);
        else
            gi_block<FMT, false, GI_TR, GI_TT, ROWS, TOK>(acc, buf[c], r0, t0, lane, fma_path);
        if (more) {
            __builtin_amdgcn_s_waitcnt(0);
            if (stager) gi_stage<ROWS>(buf[c ^ 1u].sc, buf[c ^ 1u].no, hdr, hj, srow);
            if (summer) gi_stage_sums<TOK>(buf[c ^ 1u].fsum, sums, tid & 1u, tid >> 1);
        }
        __syncthreads();
    }

#pragma unroll
    for (int k = 0; k < GI_TT; k++)
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) {
            const uint32_t t = T0 + t0 + 16u * k + 4u * lk + e;
            if (t >= tokens) continue;
            float *yo = y + (size_t)t * rows;
#pragma unroll
            for (int i = 0; i < GI_TR; i++) {
                const uint32_t r = R0 + r0 + 16u * i + lm;
                if (r < rows) yo[r] = acc[(GI_TT * i + k) / 4][4 * ((GI_TT * i + k) % 4) + e];
            }
        }
}

// ROWSxTOK: the workgroup's tile, of 16 waves (four per SIMD) where it is
// large. The tiles the host chooses among, by rows and tokens (int8.c). At four
// waves a SIMD the 128 x 128 tile spills one register (Q4_K) and four (Q5_K).
#define GEMM_INT8(NAME, FMT, WR, WT, TR, TT, TILE)                                           \
    extern "C" __global__ __launch_bounds__(64 * WR * WT, WR * WT == 16 ? 4 : 2) void        \
        NAME##_##TILE(const uint8_t *__restrict__ w, const int8_t *__restrict__ xq,          \
                      const float *__restrict__ xs, const int32_t *__restrict__ xsum,        \
                      float *__restrict__ y, uint32_t rows, uint32_t cols, uint32_t tokens,  \
                      uint32_t nb, uint32_t tile) {                                          \
        gemm_int8<FMT, WR, WT, TR, TT>(w, xq, xs, xsum, y, rows, cols, tokens, nb, tile);    \
    }
#define GEMM_INT8_TILES(NAME, FMT)                                                           \
    GEMM_INT8(NAME, FMT, 2, 2, 1, 1, 32x32)                                                  \
    GEMM_INT8(NAME, FMT, 4, 2, 1, 2, 64x64)                                                  \
    GEMM_INT8(NAME, FMT, 2, 8, 3, 1, 96x128)                                                 \
    GEMM_INT8(NAME, FMT, 4, 4, 2, 2, 128x128)
GEMM_INT8_TILES(mynah_q4k_gemm_int8, 12)
GEMM_INT8_TILES(mynah_q5k_gemm_int8, 13)
