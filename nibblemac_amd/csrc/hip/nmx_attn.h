/* Shared by the attention kernels (nmx_glue.hip: steps and verify passes; nmx_attnc.hip: prefill
 * chunks): the launch arguments and the KV cache formats. Not part of the ABI. */
#ifndef NMX_ATTN_H
#define NMX_ATTN_H

#include "nmx_internal.h"

struct nmx_attn_dev {
    int n, nh, nkv, hd, rot, max_ctx;
    float *q;            /* [n][nh][2 hd]: query | gate per head */
    const float *k_in, *v_in; /* [n][nkv hd] */
    const float *q_norm, *k_norm;
    float eps, scale;
    const float *rcos, *rsin;  /* [max_ctx][rot/2] */
    void *kc, *vc;       /* KV caches of the launch's format (nmx_kv_bytes each) */
    const int32_t *pos;  /* device: position of token 0 is *pos + pos_off */
    int pos_off;
    float *o;            /* [n][nh hd] */
    int8_t *aq;
    float *ad, *afs;
    int an;              /* rows of the A8 output's block-major layout */
};

/* ---- KV cache formats (engine/src/forward_kv.c:28-188): row R = g max_ctx + p of a cache
 * holds hd values as fp32, binary16, or int8 with an fp32 scale in a [nkv][max_ctx] array
 * after the rows. */
enum { KV_F32 = 0, KV_F16 = 1, KV_I8 = 2 };

/* binary16 bits of x rounded to nearest even, subnormals kept (v_cvt_f16_f32); a NaN becomes
 * the quiet NaN with x's sign and top 10 payload bits (forward_kv.c:28-48 f32_to_f16) */
__device__ __forceinline__ uint32_t kv_half_bits(float x) {
    const uint32_t u = __float_as_uint(x);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x7fffffu))
        return ((u >> 16) & 0x8000u) | 0x7e00u | ((u & 0x7fffffu) >> 13);
    const _Float16 h = (_Float16)x;
    unsigned short b;
    __builtin_memcpy(&b, &h, 2);
    return b;
}

__device__ __forceinline__ float kv_half_value(uint32_t bits16) { /* exact widening */
    const unsigned short b = (unsigned short)bits16;
    _Float16 h;
    __builtin_memcpy(&h, &b, 2);
    return (float)h;
}

/* the int8 code of x at inv = 127 / amax (or 0): round half even, clamped to +-127, NaN to 0
 * (forward_kv.c:101-124) */
__device__ __forceinline__ uint32_t kv_i8_code(float x, float inv) {
    const float y = rintf(x * inv);
    const int q = y > 127.0f ? 127 : y < -127.0f ? -127 : y == y ? (int)y : 0;
    return (uint32_t)(uint8_t)(int8_t)q;
}

/* fp32 values of columns col .. col + 3 of cache row R (col % 4 == 0) */
template <int KVT>
__device__ __forceinline__ float4 kv_load4(const void *cache, size_t R, int hd, int col,
                                           const float *scales) {
    if constexpr (KVT == KV_F32) {
        return *(const float4 *)((const float *)cache + R * hd + col);
    } else if constexpr (KVT == KV_F16) {
        const uint2 h = *(const uint2 *)((const unsigned short *)cache + R * hd + col);
        return make_float4(kv_half_value(h.x), kv_half_value(h.x >> 16), kv_half_value(h.y),
                           kv_half_value(h.y >> 16));
    } else {
        const uint32_t w = *(const uint32_t *)((const int8_t *)cache + R * hd + col);
        const float sc = scales[R];
        return make_float4((float)(int8_t)w * sc, (float)(int8_t)(w >> 8) * sc,
                           (float)(int8_t)(w >> 16) * sc, (float)(int8_t)(w >> 24) * sc);
    }
}

template <int KVT>
__device__ __forceinline__ const float *kv_scales(const void *cache, const nmx_attn_dev &a) {
    return KVT == KV_I8 ? (const float *)((const int8_t *)cache + (size_t)a.nkv * a.max_ctx * a.hd)
                        : nullptr;
}

/* Scores, softmax and P.V of a prefill chunk (nmx_attnc.hip), on the queries and caches that
 * attn_prep_k left; sc: [n][nh][max_ctx] workspace (it ends holding the softmax weights).
 * hd a multiple of 64 up to 512. */
int nmx_attn_chunk(nmx_ctx *ctx, const nmx_attn_dev &a, int kv_dtype, float *sc);
/* Softmax and P.V of a few rows over the scores sc, for caches whose score rows do not fit in LDS. */
int nmx_attn_long(nmx_ctx *ctx, const nmx_attn_dev &a, int kv_dtype, const float *sc);

/* acc += x[0] + ... + x[n-1] in order, x contiguous in LDS and 16-byte aligned: the terms
 * arrive four per ds_read_b128 with immediate offsets, two sets of 32 taking turns (the next
 * set requested before the current one is added), so the chain's wave issues about 0.3 other
 * instructions per dependent add (pv_chain, strided, about 1.3). */
__device__ __forceinline__ float pv_chain4(float acc, const float *x, int n) {
    auto fetch = [&](float4 (&b)[8], int r0) {
#pragma unroll
        for (int u = 0; u < 8; u++) b[u] = *(const float4 *)(x + r0 + 4 * u);
    };
    auto add = [&](const float4 (&b)[8]) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
            acc = acc + b[u].x;
            acc = acc + b[u].y;
            acc = acc + b[u].z;
            acc = acc + b[u].w;
        }
    };
    int r = 0;
    if (n >= 32) {
        float4 ba[8], bb[8];
        fetch(ba, 0);
        for (; r + 64 <= n; r += 64) {
            __builtin_amdgcn_sched_barrier(0);
            fetch(bb, r + 32);
            __builtin_amdgcn_sched_barrier(0);
            add(ba);
            __builtin_amdgcn_sched_barrier(0);
            fetch(ba, r + 96 <= n ? r + 64 : r); /* clamped: not used past n */
            __builtin_amdgcn_sched_barrier(0);
            add(bb);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (r + 32 <= n) { /* ba holds terms r .. r + 31 */
            add(ba);
            r += 32;
        }
    }
    for (; r + 4 <= n; r += 4) {
        const float4 v = *(const float4 *)(x + r);
        acc = acc + v.x;
        acc = acc + v.y;
        acc = acc + v.z;
        acc = acc + v.w;
    }
    for (; r < n; r++) acc = acc + x[r];
    return acc;
}

#endif
