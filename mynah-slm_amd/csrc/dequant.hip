// dequant.hip — matrix dequantisation bit-identical to the reference.
//
// SPDX-License-Identifier: MIT
#include "common.hip.h"

// ── bit-exact dequantisation ────────────────────────────────────────────────
// Same operation order as the reference decoders, so every value is the
// identical f32 (kernels.c:117-136 Q4_K, 1812-1833 Q5_K, 2176-2199 Q6_K,
// 2518-2523 Q8_0, 2353-2360 Q4_0).
//
// HBM-bound: 4 bytes written for every 0.6 - 1.1 read. Rows are whole blocks,
// one after the other, so the matrix is one run of blocks and values: a
// thread decodes four consecutive values (one quant dword, and the dword of
// fifth or upper bits) and stores them as one float4, so a wave's store is 1
// KiB in a row, and takes DQ_STEP such quads, a workgroup apart, with every
// load ahead of the first decode. (One thread per 32 values stored 128 bytes
// apart within a wave: 9728 x 2560 Q6_K took 46.2 us, 2.6 TB/s.)
#define DQ_STEP 4

// Four bytes of any alignment (the kernels run in unaligned-access mode).
MYNAH_DEV uint32_t dq_u32(const uint8_t *p) {
    uint32_t v;
    __builtin_memcpy(&v, p, sizeof v);
    return v;
}

// Holders: load what quad i (values 4 i .. + 3 of the matrix) needs, then
// decode it.
struct DqQ4K {
    uint4 hdr;
    uint32_t q;
    __device__ __forceinline__ void load(const uint8_t *w, uint64_t i) {
        const uint32_t v = (uint32_t)(i & 63u);               // quad of the super-block
        const uint8_t *blk = w + (i >> 6) * 144u;
        __builtin_memcpy(&hdr, blk, sizeof hdr);
        q = dq_u32(blk + 16u + 32u * (v >> 4) + 4u * (v & 7u));
    }
    __device__ __forceinline__ float4 decode(uint64_t i) const {
#pragma clang fp contract(off)
        const uint32_t j = (uint32_t)(i & 63u) >> 3;          // sub-block
        float sc, m;
        q4k_sm_rt(hdr.y, hdr.z, hdr.w, j, sc, m);
        const float dd = f16_to_f32(hdr.x) * sc, mm = f16_to_f32(hdr.x >> 16) * m;
        const uint32_t n = (j & 1u ? q >> 4 : q) & 0x0f0f0f0fu;
        return make_float4(dd * byte_f(n, 0) - mm, dd * byte_f(n, 1) - mm,
                           dd * byte_f(n, 2) - mm, dd * byte_f(n, 3) - mm);
    }
};

struct DqQ5K {
    uint4 hdr;
    uint32_t q, h;
    __device__ __forceinline__ void load(const uint8_t *w, uint64_t i) {
        const uint32_t v = (uint32_t)(i & 63u);
        const uint8_t *blk = w + (i >> 6) * 176u;
        __builtin_memcpy(&hdr, blk, sizeof hdr);
        h = dq_u32(blk + 16u + 4u * (v & 7u));
        q = dq_u32(blk + 48u + 32u * (v >> 4) + 4u * (v & 7u));
    }
    __device__ __forceinline__ float4 decode(uint64_t i) const {
#pragma clang fp contract(off)
        const uint32_t j = (uint32_t)(i & 63u) >> 3;
        float sc, m;
        q4k_sm_rt(hdr.y, hdr.z, hdr.w, j, sc, m);
        const float dd = f16_to_f32(hdr.x) * sc, mm = f16_to_f32(hdr.x >> 16) * m;
        const uint32_t n = ((j & 1u ? q >> 4 : q) & 0x0f0f0f0fu) | (((h >> j) & 0x01010101u) << 4);
        return make_float4(dd * byte_f(n, 0) - mm, dd * byte_f(n, 1) - mm,
                           dd * byte_f(n, 2) - mm, dd * byte_f(n, 3) - mm);
    }
};

struct DqQ6K {
    uint32_t ql, qh, sd;              // sd: the int8 scale (low byte), d (high 16)
    __device__ __forceinline__ void load(const uint8_t *w, uint64_t i) {
        // Value 128 h + 32 k + l: quads 32 h + 8 k + l / 4.
        const uint32_t v = (uint32_t)(i & 63u), h = v >> 5, k = (v >> 3) & 3u, l = 4u * (v & 7u);
        const uint8_t *blk = w + (i >> 6) * 210u;
        ql = dq_u32(blk + 64u * h + 32u * (k & 1u) + l);
        qh = dq_u32(blk + 128u + 32u * h + l);
        uint16_t d;
        __builtin_memcpy(&d, blk + 208u, sizeof d);
        sd = (uint32_t)blk[192u + 8u * h + 2u * k + (l >> 4)] | ((uint32_t)d << 16);
    }
    __device__ __forceinline__ float4 decode(uint64_t i) const {
#pragma clang fp contract(off)
        const uint32_t k = (uint32_t)(i & 31u) >> 3;
        const float ds = f16_to_f32(sd >> 16) * (float)(int)(int8_t)(sd & 0xffu);
        const uint32_t n = ((k < 2u ? ql : ql >> 4) & 0x0f0f0f0fu) |
                           (((qh >> (2u * k)) & 0x03030303u) << 4);
        return make_float4(ds * (byte_f(n, 0) - 32.0f), ds * (byte_f(n, 1) - 32.0f),
                           ds * (byte_f(n, 2) - 32.0f), ds * (byte_f(n, 3) - 32.0f));
    }
};

struct DqQ80 {
    uint32_t q;
    uint16_t d;
    __device__ __forceinline__ void load(const uint8_t *w, uint64_t i) {
        const uint8_t *blk = w + (i >> 3) * 34u;
        __builtin_memcpy(&d, blk, sizeof d);
        q = dq_u32(blk + 2u + 4u * (uint32_t)(i & 7u));
    }
    __device__ __forceinline__ float4 decode(uint64_t) const {
#pragma clang fp contract(off)
        const float df = f16_to_f32(d);
        return make_float4((float)(int8_t)q * df, (float)(int8_t)(q >> 8) * df,
                           (float)(int8_t)(q >> 16) * df, (float)(int8_t)(q >> 24) * df);
    }
};

struct DqQ40 {
    uint32_t q;
    uint16_t d;
    __device__ __forceinline__ void load(const uint8_t *w, uint64_t i) {
        const uint8_t *blk = w + (i >> 3) * 18u;
        __builtin_memcpy(&d, blk, sizeof d);
        q = dq_u32(blk + 2u + 4u * (uint32_t)(i & 3u));
    }
    __device__ __forceinline__ float4 decode(uint64_t i) const {
#pragma clang fp contract(off)
        const float df = f16_to_f32(d);
        const uint32_t n = (i & 4u ? q >> 4 : q) & 0x0f0f0f0fu;
        return make_float4(df * (byte_f(n, 0) - 8.0f), df * (byte_f(n, 1) - 8.0f),
                           df * (byte_f(n, 2) - 8.0f), df * (byte_f(n, 3) - 8.0f));
    }
};

template <class Dq>
MYNAH_DEV void dequant_body(const uint8_t *__restrict__ w, float *__restrict__ y, uint64_t quads) {
    const uint64_t i0 = (uint64_t)blockIdx.x * (256u * DQ_STEP) + threadIdx.x;
    Dq q[DQ_STEP];
#pragma unroll
    for (uint32_t k = 0; k < DQ_STEP; k++) {
        const uint64_t i = i0 + 256u * k;
        q[k].load(w, i < quads ? i : quads - 1u);
    }
#pragma unroll
    for (uint32_t k = 0; k < DQ_STEP; k++) {
        const uint64_t i = i0 + 256u * k;
        const float4 v = q[k].decode(i);
        if (i < quads) __builtin_memcpy(y + 4u * i, &v, sizeof v);
    }
}

// quads = rows * cols / 4; grid ceil(quads / (256 DQ_STEP)).
extern "C" __global__ void __launch_bounds__(256)
mynah_dequant(const uint8_t *__restrict__ w, float *__restrict__ y, uint32_t type,
              uint64_t quads) {
    if (type == 12u) dequant_body<DqQ4K>(w, y, quads);
    else if (type == 13u) dequant_body<DqQ5K>(w, y, quads);
    else if (type == 2u) dequant_body<DqQ40>(w, y, quads);
    else if (type == 14u) dequant_body<DqQ6K>(w, y, quads);
    else dequant_body<DqQ80>(w, y, quads);
}
