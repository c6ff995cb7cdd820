/* Attention of a prefill chunk (more than 8 tokens) for gfx950: scores, softmax, P.V
 * (engine/src/forward_kv.c:281-303, forward_attn.c:171-181, forward_ops.c:265-382), after
 * attn_prep_k stored the chunk's K / V rows and normed its queries. Every sum is the ordered
 * chain of the step kernels (nmx_glue.hip), so the results equal theirs bit for bit; what differs
 * is the split. A step has few chains, so there a chain runs on products that other waves prepare
 * and K / V rows are re-read per token. A chunk has n x heads rows over the same K / V rows, so
 * here a lane runs whole chains in registers, the K / V tile is staged once for the rows of a
 * workgroup, and the operand that is the same for the 64 lanes (a query element, a softmax
 * weight) is held 16 to a 16-lane row and broadcast by the multiply's DPP modifier (through the
 * scalar cache instead, every wave streaming its own row misses it: scores 53 us, P.V 126 us at
 * the first size below). Rows r of KV group g: token r / rep, head g rep + r % rep.
 * Bound: VALU, a product (4.2 clocks of a SIMD with DPP) and an add (2.2) per (row, position,
 * dim): 64 tokens x 8 heads x 4032 positions x 256 dims take 21 us of all SIMDs for the scores
 * and as much for P.V; what is above that is the wait for a tile when few waves share a SIMD. */
#include "nmx_internal.h"
#include "nmx_attn.h"
#include "nmx_math.h"
#include "nmx_a8.h"
#include "nmx_lanes.h"

namespace {

using Attn = nmx_attn_dev;

/* lane L of every 16-lane row, to the whole row: an operand modifier of the multiply (DPP
 * row_newbcast), so an operand held 16 to a row costs no instruction to broadcast */
template <int L>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(nmx_dpp<0x150 + L>(__float_as_int(v)));
}

/* x[L] = bcast(w, L) * v[L] for L = 0..15 */
template <int L = 0>
__device__ __forceinline__ void mul16(float (&x)[16], float w, const float (&v)[16]) {
    if constexpr (L < 16) {
        x[L] = row_bcast<L>(w) * v[L];
        mul16<L + 1>(x, w, v);
    }
}

/* c[L] += bcast(w, L) * v[L] for L = 0..15, the product and the sum rounded separately */
template <int L = 0>
__device__ __forceinline__ void acc16(float (&c)[16], float w, const float (&v)[16]) {
    if constexpr (L < 16) {
        c[L] = c[L] + row_bcast<L>(w) * v[L];
        acc16<L + 1>(c, w, v);
    }
}

constexpr int SC_P = 64;     /* positions per scores workgroup: one per lane */
constexpr int SC_ROWS = 32;  /* rows per scores workgroup: 8 waves x 4 */
constexpr int PV_P = 128;    /* positions per P.V tile */
constexpr int PV_D = 64;     /* output dims per P.V workgroup: one per lane */
constexpr int PV_W = 8;      /* rows per P.V workgroup: one per wave */
constexpr int SM_SEG = 4096; /* positions per softmax segment in LDS */
constexpr int SM_S4 = SM_SEG / 4 + 4; /* row stride of a segment's four partial sums */

/* Scores. Lane = position; a wave takes 4 rows at a time, whose query elements it holds 16 to a row
 * of lanes and broadcasts in the multiply, and keeps the 16 interleaved partial sums of each in
 * registers: per 16 elements 4 LDS reads of the position's key (shared by the 4 rows) feed 128 VALU
 * instructions. Tile rows are hd + 4 floats apart, so 16 lanes' 16-byte reads cover the banks once.
 * 64 tokens at 4000 positions, int8 cache: 45.5 us (attn_score_k, one token x 32 positions per
 * workgroup and so a key tile per token: 96.7); a 45-token prompt 18.6 us, a 2000-token fp32 prompt
 * in slices of 256 tokens 67.5 us each on average. A query element is requested one step of 16 dims
 * ahead only, which few waves per SIMD do not hide. */
template <int KVT>
__global__ __launch_bounds__(512) void attn_scc_k(Attn a, float *__restrict__ sc) {
    extern __shared__ float4 smem4[];
    float *ks = (float *)smem4; /* [SC_P][hd + 4] */
    const int hd = a.hd, rep = a.nh / a.nkv, rs = hd + 4, f4 = hd >> 2;
    const int g = blockIdx.z, p0 = blockIdx.x * SC_P, r0 = blockIdx.y * SC_ROWS;
    const int nrows = a.n * rep, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pos = *a.pos + a.pos_off;
    const int rl = (r0 + SC_ROWS < nrows ? r0 + SC_ROWS : nrows) - 1;
    const int npw = pos + rl / rep + 1; /* positions of the workgroup's last token */
    if (p0 >= npw) return;
    const int rows = npw - p0 < SC_P ? npw - p0 : SC_P;
    const size_t R0 = (size_t)g * a.max_ctx + p0;
    const float *ksc = kv_scales<KVT>(a.kc, a);
    for (int f0 = 0; f0 < rows * f4; f0 += 8 * 512) {
        float4 b[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int f = f0 + u * 512 + (int)threadIdx.x;
            b[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (f < rows * f4) b[u] = kv_load4<KVT>(a.kc, R0 + f / f4, hd, 4 * (f % f4), ksc);
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int f = f0 + u * 512 + (int)threadIdx.x;
            if (f < rows * f4) *(float4 *)(ks + (f / f4) * rs + 4 * (f % f4)) = b[u];
        }
    }
    __syncthreads();
    const int rb = r0 + 4 * w;
    if (rb >= nrows) return; /* uniform per wave, as every bound on rows here */
    const int rlast = rb + 3 < nrows ? rb + 3 : nrows - 1;
    if (p0 >= pos + rlast / rep + 1) return;
    const float *kr = ks + lane * rs; /* lanes past the tile's rows read rows left unwritten */
    float c[4][16], qv[4];
    const float *q[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int r = rb + j < nrows ? rb + j : nrows - 1, t = r / rep;
        q[j] = a.q + ((size_t)t * a.nh + g * rep + (r - t * rep)) * 2 * hd + (lane & 15);
        qv[j] = q[j][0];
#pragma unroll
        for (int l = 0; l < 16; l++) c[j][l] = 0.0f;
    }
    for (int i = 0; i < hd; i += 16) {
        float k[16], qn[4];
#pragma unroll
        for (int j = 0; j < 4; j++) qn[j] = q[j][i + 16]; /* the last step reads the gate's: unused */
#pragma unroll
        for (int l = 0; l < 16; l += 4) {
            const float4 x = *(const float4 *)(kr + i + l);
            k[l] = x.x, k[l + 1] = x.y, k[l + 2] = x.z, k[l + 3] = x.w;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc16(c[j], qv[j], k);
            qv[j] = qn[j];
        }
    }
    const int p = p0 + lane;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int r = rb + j, t = r / rep;
        if (r >= nrows) break;
        float h[4];
#pragma unroll
        for (int l = 0; l < 4; l++)
            h[l] = (c[j][4 * l] + c[j][4 * l + 1]) + (c[j][4 * l + 2] + c[j][4 * l + 3]);
        const float s = (h[0] + h[1]) + (h[2] + h[3]);
        if (p < pos + t + 1)
            sc[((size_t)t * a.nh + g * rep + (r - t * rep)) * a.max_ctx + p] = (s + 0.0f) * a.scale;
    }
}

/* Softmax weights in place, one workgroup per (head, token): max, e_p = exp(s_p - max), the four
 * interleaved partial sums and the tail in order, w_p = e_p * (1 / sum). A segment's exponentials
 * sit in LDS one partial sum after the other (16-byte chain reads); wave 0 adds a segment while
 * the other waves form the next one's, so a long row costs its chain, np / 4 dependent adds. 512
 * threads with 8 reads in flight each: 11.5 us for 512 rows of 4000 positions (256 threads with one
 * read each: 16.4 us). */
constexpr int SM_T = 512;

__global__ __launch_bounds__(SM_T) void attn_sm_k(Attn a, float *__restrict__ sc) {
    __shared__ __align__(16) float seg[2][4 * SM_S4 + 4];
    __shared__ float red[8];
    const int tid = threadIdx.x, h = blockIdx.x, t = blockIdx.y;
    const int np = *a.pos + a.pos_off + t + 1;
    float *row = sc + ((size_t)t * a.nh + h) * a.max_ctx;
    /* f(i, row[i]) for i = i0, i0 + step, .. < end, 8 reads in flight */
    auto sweep = [&](int i0, int step, int end, auto f) {
        for (int i = i0; i < end; i += 8 * step) {
            float x[8];
#pragma unroll
            for (int u = 0; u < 8; u++) x[u] = row[i + u * step < end ? i + u * step : end - 1];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (i + u * step < end) f(i + u * step, x[u]);
        }
    };
    float mx = -INFINITY;
    sweep(tid, SM_T, np, [&](int, float x) { mx = fmaxf(mx, x); });
    mx = nmx_max_f32_wave(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = red[0];
#pragma unroll
    for (int u = 1; u < SM_T / 64; u++) mx = fmaxf(mx, red[u]);
    const bool many = np > SM_SEG; /* the exponentials of a long row wait in the row itself */
    /* position s0 + i of a segment: partial sum i % 4, its term i / 4 */
    auto exps = [&](int s0, float *dst, int i0, int step) {
        sweep(s0 + i0, step, np - s0 < SM_SEG ? np : s0 + SM_SEG, [&](int p, float x) {
            const float e = nmx_expf_cephes(x - mx);
            dst[(p & 3) * SM_S4 + ((p - s0) >> 2)] = e;
            if (many) row[p] = e;
        });
    };
    exps(0, seg[0], tid, SM_T);
    __syncthreads();
    const int q4 = np & ~3; /* positions in whole quads */
    float chain = 0.0f;     /* lane l < 4: partial sum l; lane 4: the tail */
    for (int s0 = 0, s = 0; s0 < np; s0 += SM_SEG, s ^= 1) {
        if (tid < 5) {
            const int full = q4 - s0 < SM_SEG ? q4 - s0 : SM_SEG;
            if (tid < 4) chain = pv_chain4(chain, seg[s] + tid * SM_S4, full >> 2);
            else
                for (int i = full; i < SM_SEG && s0 + i < np; i++)
                    chain = chain + seg[s][(i & 3) * SM_S4 + (i >> 2)];
        } else if (tid >= 64 && s0 + SM_SEG < np) {
            exps(s0 + SM_SEG, seg[s ^ 1], tid - 64, SM_T - 64);
        }
        __syncthreads();
    }
    if (tid < 5) red[tid] = chain;
    __syncthreads();
    const float inv = 1.0f / (((red[0] + red[1]) + (red[2] + red[3])) + red[4]);
    if (many) {
        sweep(tid, SM_T, np, [&](int p, float e) { row[p] = e * inv; });
    } else {
        for (int p = tid; p < np; p += SM_T) row[p] = seg[0][(p & 3) * SM_S4 + (p >> 2)] * inv;
    }
}

/* P.V, the output gate and A8. Lane = output dim, wave = row: a lane's chain is o = o + w_p v_p[d]
 * over its row's positions, w_p held 16 to a row of lanes and broadcast in the multiply, v_p[d] from
 * the tile that the 8 rows of the workgroup share. 64 tokens x 8 heads fill 256 workgroups of 8 waves,
 * two waves per SIMD, which is what a SIMD needs to issue every cycle; a wave of two rows would halve
 * the LDS reads and the waves (54 against 52 us). Consecutive workgroups take different (dims, group)
 * slices, so a slice of V stays in one XCD's L2. 64 tokens at 4000 positions, int8 cache: 69.7 us (99
 * with weights and values requested one 64-position tile ahead); a 2000-token fp32 prompt in slices
 * of 256 tokens 52 us each on average. With attn_sm_k that replaces attn_pv_k (32 dims x 1 token per
 * workgroup, every product through LDS to one chain wave): 934 us at the first size. */
template <int KVT>
__global__ __launch_bounds__(512) void attn_pvc_k(const float *__restrict__ wts, Attn a) {
    constexpr int F4 = PV_D / 4, PER = PV_P * F4 / 512;
    __shared__ __align__(16) float vt[2][PV_P * PV_D];
    const int hd = a.hd, rep = a.nh / a.nkv, S = (hd / PV_D) * a.nkv, tid = threadIdx.x;
    const int sl = blockIdx.x % S, d0 = (sl % (hd / PV_D)) * PV_D, g = sl / (hd / PV_D);
    const int r0 = (int)(blockIdx.x / S) * PV_W, nrows = a.n * rep, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool live = r0 + w < nrows;
    const int r = live ? r0 + w : nrows - 1, t = r / rep, h = g * rep + (r - t * rep);
    const int pos = *a.pos + a.pos_off;
    const int rl = (r0 + PV_W < nrows ? r0 + PV_W : nrows) - 1;
    const int npw = pos + rl / rep + 1;     /* positions of the workgroup's last token */
    const int np = live ? pos + t + 1 : 0;  /* of the wave's (0: none, its loads read weight 0) */
    const size_t R0 = (size_t)g * a.max_ctx;
    const float *vsc = kv_scales<KVT>(a.vc, a);
    const int d = d0 + lane;
    const float gate = a.q[((size_t)t * a.nh + h) * 2 * hd + hd + d];
    const float *wr = wts + ((size_t)t * a.nh + h) * a.max_ctx;
    /* the next tile's values and the weights of the two next tiles (16 to each 16-lane row),
     * requested a tile's arithmetic ahead: the weights were written by other XCDs, so their first
     * reads miss this XCD's L2. Addresses are clamped, not masked: a load in a branch would make
     * every wait wait for all loads in flight. */
    constexpr int WB = PV_P / 16;
    float4 nb[PER];
    float wt[WB], wn[WB];
    auto fetch_v = [&](int base) {
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int f = u * 512 + tid, p = base + f / F4;
            nb[u] = kv_load4<KVT>(a.vc, R0 + (p < npw ? p : npw - 1), hd, d0 + 4 * (f % F4), vsc);
        }
    };
    auto fetch_w = [&](float (&x)[WB], int base) {
#pragma unroll
        for (int u = 0; u < WB; u++) {
            const int p = base + 16 * u + (lane & 15);
            x[u] = wr[p < np ? p : 0];
        }
    };
    fetch_w(wt, 0);
    fetch_v(0);
    fetch_w(wn, PV_P);
    float o = 0.0f;
    for (int base = 0, b = 0; base < npw; base += PV_P, b ^= 1) {
        float wc[WB];
#pragma unroll
        for (int u = 0; u < PER; u++) *(float4 *)(vt[b] + 4 * (u * 512 + tid)) = nb[u];
#pragma unroll
        for (int u = 0; u < WB; u++) wc[u] = wt[u], wt[u] = wn[u];
        fetch_v(base + PV_P);
        fetch_w(wn, base + 2 * PV_P);
        /* one barrier per tile: a wave stores tile i + 2 into the buffer of tile i only after
         * the barrier of tile i + 1, which every wave reaches past its reads of tile i */
        __syncthreads();
        const float *v = vt[b] + lane;
        const int m = np - base;
        float x[16], y[2][16];
        auto read = [&](int u) {
#pragma unroll
            for (int l = 0; l < 16; l++) y[u & 1][l] = v[(16 * u + l) * PV_D];
        };
        if (m >= PV_P) { /* batches of 16, the next one's values read before this one's adds */
            read(0);
#pragma unroll
            for (int u = 0; u < WB; u++) {
                mul16(x, wc[u], y[u & 1]);
                if (u + 1 < WB) read(u + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int l = 0; l < 16; l++) o = o + x[l];
            }
        } else { /* the row's last positions; the products past them are dropped */
#pragma unroll
            for (int u = 0; u < WB; u++) {
                if (16 * u >= m) break; /* uniform per wave */
                read(u);
                mul16(x, wc[u], y[u & 1]);
#pragma unroll
                for (int l = 0; l < 16; l++) o = 16 * u + l < m ? o + x[l] : o;
            }
        }
    }
    if (!live) return; /* whole waves */
    o = o * nmx_sigmoid(gate);
    const int col = h * hd + d;
    a.o[(size_t)t * a.nh * hd + col] = o;
    if (a.aq) {
        const size_t u = (size_t)(col >> 5) * a.an + t;
        nmx_a8_store(o, a.aq + u * 32, a.ad + u, a.afs + u);
    }
}

/* Softmax and P.V of a few rows in caches past 8192 positions (steps and verify passes): workgroup =
 * (32 dims, head, token). Each forms its row's max and sum itself (attn_sm_k's steps; the 8 workgroups
 * of a row run them side by side, and a separate launch would cost a short context 2 us), then wave
 * 0's lanes run the P.V chains, one per dim. The chain, one dependent add per position fed from LDS,
 * bounds it (8.2 clocks a step in tiles of 256, 68 us for 20000 positions; on registers 4.25), so
 * everything else runs beside it: waves 1-4 store tile i + 1's products
 * w_p v_p[d] in LDS, one row per dim, while wave 0 adds tile i, and have tile i + 2's values and scores
 * in flight. One token at 20000 positions, binary16 cache: 130 us (one kernel that stored each tile
 * between two runs of the chains: 429 us). Up to PL_SHORT positions a row is one pass.
 * 5 rows of 8 heads are 320 workgroups and 8 rows 512, two to a CU, whose 10 waves fit its SIMDs only
 * at 128 registers; at 140 (tiles of 440 positions in the short pass) the second one waited for the
 * first: 6.6 against 4.4 us for 5 rows at 40 positions, 23.6 against 14.8 us for 8 at 1000. Whole
 * layers of 1 token at 50, 5 at 40, 5 at 900, 8 at 300 and 8 at 3000 positions: 34.2, 41.5, 49.9, 51.9
 * and 78.5 us (34.8, 42.2, 58.2, 54.5 and 109.6 with the kernel that alternated). */
constexpr int PL_P = 256;        /* positions per tile */
constexpr int PL_D = 32;         /* output dims per workgroup: one A8 block */
constexpr int PL_RS = PL_P + 4;  /* row stride: 16-byte aligned, 4 words apart modulo 64 banks */
/* Positions up to which a row is one pass without the pipeline. us of the kernel at 1, 5 and 8 rows,
 * one pass against pipeline: 300 positions 6.8, 6.9, 7.2 against 7.6, 8.9, 9.3; 600: 9.8, 10.6, 10.7
 * against 9.8, 11.6, 12.0; 1000: 13.4, 14.6, 14.7 against 12.1, 14.1, 14.5. */
constexpr int PL_SHORT = 768;
constexpr int PS_P = 240;        /* positions per tile there: 6 values per thread, none left over */
constexpr int PL_LDS = 2 * PL_D * PL_RS * 4;

template <int KVT>
__global__ __launch_bounds__(320) __attribute__((amdgpu_waves_per_eu(4))) void attn_pvl_k(
    const float *__restrict__ sc, Attn a) {
    constexpr int F4 = PL_D / 4, PER = PL_P * F4 / 256, T = 320;
    /* the softmax's two segments, then the two tiles of products: PL_LDS bytes, dynamic, as the
     * compiler would count two workgroups per CU and not keep to the registers of four waves */
    extern __shared__ float4 smem4[];
    float *buf = (float *)smem4;
    static_assert(4 * SM_S4 <= PL_D * PL_RS, "a segment fits in a tile's place");
    __shared__ float red[8];
    const int hd = a.hd, rep = a.nh / a.nkv, S = (hd / PL_D) * a.nkv, tid = threadIdx.x;
    const int sl = blockIdx.x % S, k = blockIdx.x / S; /* a slice of V to one XCD, as attn_pvc_k */
    const int d0 = (sl % (hd / PL_D)) * PL_D, g = sl / (hd / PL_D);
    const int h = g * rep + k % rep, t = k / rep;
    const int np = *a.pos + a.pos_off + t + 1, ntile = (np + PL_P - 1) / PL_P;
    const size_t R0 = (size_t)g * a.max_ctx;
    const float *vsc = kv_scales<KVT>(a.vc, a);
    const float *row = sc + ((size_t)t * a.nh + h) * a.max_ctx;
    const float gate = tid < PL_D ? a.q[((size_t)t * a.nh + h) * 2 * hd + hd + d0 + tid] : 0.0f;
    auto finish = [&](float o) { /* lanes tid < PL_D */
        o = o * nmx_sigmoid(gate);
        const int col = h * hd + d0 + tid;
        a.o[(size_t)t * a.nh * hd + col] = o;
        if (a.aq) {
            const size_t u = (size_t)(col >> 5) * a.an + t;
            nmx_a8_store(o, a.aq + u * 32, a.ad + u, a.afs + u);
        }
    };
    if (np <= PL_SHORT) { /* uniform: the whole workgroup */
        /* the exponentials in LDS, one partial sum after the other; the first PS_P positions' values
         * requested at entry, every thread's products stored, then the chains */
        constexpr int S4 = PL_SHORT / 4 + 4, RS = PS_P + 4, PSR = PS_P * F4 / T;
        static_assert(PS_P * F4 % T == 0 && 4 * S4 + PL_D * RS <= 2 * PL_D * PL_RS, "fits in the tiles' place");
        float *e = buf, *vt = buf + 4 * S4;
        float4 v[PSR];
        auto values = [&](int base, int rows) {
#pragma unroll
            for (int u = 0; u < PSR; u++) { /* clamped, and whole sweeps of the threads left out */
                if (u * T >= rows * F4) break;
                const int f = u * T + tid, r = f / F4 < rows ? f / F4 : rows - 1;
                v[u] = kv_load4<KVT>(a.vc, R0 + base + r, hd, d0 + 4 * (f % F4), vsc);
            }
        };
        int rows = np < PS_P ? np : PS_P;
        float x[(PL_SHORT + T - 1) / T], mx = -INFINITY;
#pragma unroll
        for (int u = 0; u < (PL_SHORT + T - 1) / T; u++)
            if (u * T + tid < np) x[u] = row[u * T + tid];
        values(0, rows);
#pragma unroll
        for (int u = 0; u < (PL_SHORT + T - 1) / T; u++)
            if (u * T + tid < np) mx = fmaxf(mx, x[u]);
        mx = nmx_max_f32_wave(mx);
        if ((tid & 63) == 0) red[tid >> 6] = mx;
        __syncthreads();
        mx = red[0];
#pragma unroll
        for (int u = 1; u < T / 64; u++) mx = fmaxf(mx, red[u]);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < (PL_SHORT + T - 1) / T; u++) {
            const int p = u * T + tid;
            if (p < np) e[(p & 3) * S4 + (p >> 2)] = nmx_expf_cephes(x[u] - mx);
        }
        __syncthreads();
        if (tid < 4) {
            red[tid] = pv_chain4(0.0f, e + tid * S4, np >> 2);
        } else if (tid == 4) {
            float tl = 0.0f;
            for (int p = np & ~3; p < np; p++) tl = tl + e[(p & 3) * S4 + (p >> 2)];
            red[4] = tl;
        }
        __syncthreads();
        const float inv = 1.0f / (((red[0] + red[1]) + (red[2] + red[3])) + red[4]);
        float o = 0.0f;
        for (int base = 0; base < np; base += PS_P) {
#pragma unroll
            for (int u = 0; u < PSR; u++) {
                if (u * T >= rows * F4) break;
                const int f = u * T + tid, r = f / F4, p = base + r < np ? base + r : np - 1;
                float *y = vt + 4 * (f % F4) * RS + r; /* past the rows: stored, never added */
                const float w = e[(p & 3) * S4 + (p >> 2)] * inv;
                y[0] = w * v[u].x;
                y[RS] = w * v[u].y;
                y[2 * RS] = w * v[u].z;
                y[3 * RS] = w * v[u].w;
            }
            const int next = base + PS_P, nrows = np - next < PS_P ? np - next : PS_P;
            if (next < np) values(next, nrows);
            __syncthreads();
            if (tid < PL_D) o = pv_chain4(o, vt + tid * RS, rows);
            __syncthreads();
            rows = nrows;
        }
        if (tid < PL_D) finish(o);
        return;
    }
    /* waves 1-4: 8 lanes to a position; the first tile's values requested before the softmax */
    const int f0 = tid >= 64 ? tid - 64 : 0, c4 = f0 % F4, r0 = f0 / F4;
    float4 v[PER];
    float x[PER];
    auto fetch = [&](int i) { /* clamped: positions past the row are stored and never added */
#pragma unroll
        for (int u = 0; u < PER; u++) {
            int p = i * PL_P + u * (256 / F4) + r0;
            p = p < np ? p : np - 1;
            v[u] = kv_load4<KVT>(a.vc, R0 + p, hd, d0 + 4 * c4, vsc);
            x[u] = row[p];
        }
    };
    fetch(0);
    /* f(i, row[i]) for i = i0, i0 + step, .. < end, 8 reads in flight */
    auto sweep = [&](int i0, int step, int end, auto f) {
        for (int i = i0; i < end; i += 8 * step) {
            float y[8];
#pragma unroll
            for (int u = 0; u < 8; u++) y[u] = row[i + u * step < end ? i + u * step : end - 1];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (i + u * step < end) f(i + u * step, y[u]);
        }
    };
    float mx = -INFINITY;
    sweep(tid, T, np, [&](int, float y) { mx = fmaxf(mx, y); });
    mx = nmx_max_f32_wave(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = red[0];
#pragma unroll
    for (int u = 1; u < T / 64; u++) mx = fmaxf(mx, red[u]);
    auto exps = [&](int s0, float *dst, int i0, int step) {
        sweep(s0 + i0, step, np - s0 < SM_SEG ? np : s0 + SM_SEG, [&](int p, float y) {
            dst[(p & 3) * SM_S4 + ((p - s0) >> 2)] = nmx_expf_cephes(y - mx);
        });
    };
    exps(0, buf, tid, T);
    __syncthreads();
    const int q4 = np & ~3; /* positions in whole quads */
    float chain = 0.0f;     /* lane l < 4: partial sum l; lane 4: the tail */
    for (int s0 = 0, s = 0; s0 < np; s0 += SM_SEG, s ^= 1) {
        float *seg = buf + s * PL_D * PL_RS;
        if (tid < 5) {
            const int full = q4 - s0 < SM_SEG ? q4 - s0 : SM_SEG;
            if (tid < 4) chain = pv_chain4(chain, seg + tid * SM_S4, full >> 2);
            else
                for (int i = full; i < SM_SEG && s0 + i < np; i++)
                    chain = chain + seg[(i & 3) * SM_S4 + (i >> 2)];
        } else if (tid >= 64 && s0 + SM_SEG < np) {
            exps(s0 + SM_SEG, buf + (s ^ 1) * PL_D * PL_RS, tid - 64, T - 64);
        }
        __syncthreads();
    }
    if (tid < 5) red[tid] = chain;
    __syncthreads();
    const float inv = 1.0f / (((red[0] + red[1]) + (red[2] + red[3])) + red[4]);

    if (tid >= 64) {
        for (int i = 0; i < ntile; i++) {
            float *q = buf + (i & 1) * PL_D * PL_RS + 4 * c4 * PL_RS + r0;
#pragma unroll
            for (int u = 0; u < PER; u++) {
                float *y = q + u * (256 / F4);
                const float w = nmx_expf_cephes(x[u] - mx) * inv;
                y[0] = w * v[u].x;
                y[PL_RS] = w * v[u].y;
                y[2 * PL_RS] = w * v[u].z;
                y[3 * PL_RS] = w * v[u].w;
            }
            fetch(i + 1);
            __syncthreads(); /* tile i stored; tile i - 1 added */
        }
        return;
    }
    float o = 0.0f;
    for (int i = 0; i < ntile; i++) {
        __syncthreads();
        const int rows = np - i * PL_P < PL_P ? np - i * PL_P : PL_P;
        if (tid < PL_D) o = pv_chain4(o, buf + (i & 1) * PL_D * PL_RS + tid * PL_RS, rows);
    }
    if (tid < PL_D) finish(o);
}

template <int KVT>
int launch_chunk(nmx_ctx *ctx, const Attn &a, float *sc) {
    const int rows = a.n * (a.nh / a.nkv);
    const size_t lds = (size_t)SC_P * (a.hd + 4) * 4;
    static std::atomic<uint64_t> lds_set;
    if (nmx_dyn_lds(ctx, (const void *)attn_scc_k<KVT>, SC_P * (512 + 4) * 4, lds_set)) return -1;
    const dim3 sgrid((unsigned)((a.max_ctx + SC_P - 1) / SC_P),
                     (unsigned)((rows + SC_ROWS - 1) / SC_ROWS), (unsigned)a.nkv);
    attn_scc_k<KVT><<<sgrid, 512, lds, ctx->stream>>>(a, sc);
    NMX_LAUNCHED(ctx, "attn_scc");
    attn_sm_k<<<dim3((unsigned)a.nh, (unsigned)a.n), SM_T, 0, ctx->stream>>>(a, sc);
    NMX_LAUNCHED(ctx, "attn_sm");
    const unsigned pg = (unsigned)((a.hd / PV_D) * a.nkv * ((rows + PV_W - 1) / PV_W));
    attn_pvc_k<KVT><<<pg, 512, 0, ctx->stream>>>(sc, a);
    NMX_LAUNCHED(ctx, "attn_pvc");
    return 0;
}

template <int KVT>
int launch_long(nmx_ctx *ctx, const Attn &a, const float *sc) {
    static std::atomic<uint64_t> lds_set;
    if (nmx_dyn_lds(ctx, (const void *)attn_pvl_k<KVT>, PL_LDS, lds_set)) return -1;
    attn_pvl_k<KVT><<<(unsigned)((a.hd / PL_D) * a.nh * a.n), 320, PL_LDS, ctx->stream>>>(sc, a);
    NMX_LAUNCHED(ctx, "attn_pvl");
    return 0;
}

} // namespace

int nmx_attn_long(nmx_ctx *ctx, const nmx_attn_dev &a, int kv_dtype, const float *sc) {
    if (kv_dtype == KV_F16) return launch_long<KV_F16>(ctx, a, sc);
    if (kv_dtype == KV_I8) return launch_long<KV_I8>(ctx, a, sc);
    return launch_long<KV_F32>(ctx, a, sc);
}

int nmx_attn_chunk(nmx_ctx *ctx, const nmx_attn_dev &a, int kv_dtype, float *sc) {
    if (kv_dtype == KV_F16) return launch_chunk<KV_F16>(ctx, a, sc);
    if (kv_dtype == KV_I8) return launch_chunk<KV_I8>(ctx, a, sc);
    return launch_chunk<KV_F32>(ctx, a, sc);
}
