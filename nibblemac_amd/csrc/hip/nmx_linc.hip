/* The Gated DeltaNet mixer over a prefill chunk (more than 8 tokens, no rollback log) for gfx950:
 * conv + SiLU + L2 norms + gates with the tokens in parallel, then the recurrence. The arithmetic
 * is that of nmx_lin_pre and nmx_lin_rule (engine/src/forward_lin.c:36-67, matvec_ref.c:114-136),
 * operation for operation; the gated norm after it is nmx_lin_post's kernel.
 *
 * The recurrence is one chain per value column: per token kv = sum of 128 keys in order, then
 * delta, then the state, which the next token's kv needs. A dependent add on registers takes 4.25
 * clocks (1.78 ns), 5.16 on average with a hand-over to the next lane every 8, so the adds of a token
 * are 0.28 us; it takes 0.40 (the slope from 256 to 512 tokens), the rest being the products, the
 * broadcast of kv, delta, the state's update and the operands' reads. Three things are moved out of
 * that chain's way:
 *   - o_t = sum of S_t q_t is a chain of its own, but nothing waits for it: other waves run it,
 *     on a copy of the state that they advance from the published deltas. There the 16 lanes of a
 *     column work on 16 consecutive tokens at once (lane c on token tau - c, its partial sum passed
 *     to lane c + 1 at the next step), so every add of a step belongs to a sum.
 *   - 16 lanes share a column's keys (8 each at dk = 128), so the multiplies and the state update
 *     are 32 instructions per token instead of the 128 of 4 lanes (lin_rule_k, lin_mix_k).
 *   - 8 columns per workgroup of 4 waves (two on the kv chains, two on o): one wave per SIMD, 256
 *     workgroups at 16 heads x 128 columns, where lin_mix_k's one workgroup per head left 240 CUs
 *     idle and put two chain waves on each SIMD.
 * 64 tokens, 16 heads x 128 x 128: 34.3 us, 512 tokens 215 us (lin_mix_k, conv and gated norm
 * included: 97-100 us for 64, 1.45 us per token). */
#include "nmx_internal.h"
#include "nmx_linc.h"
#include "nmx_lanes.h"
#include "nmx_math.h"

namespace {

constexpr int PC_TB = 8; /* tokens per workgroup of the conv kernel */

/* Conv + SiLU (+ L2 norm of q and k heads) of dk channels x PC_TB tokens, or, for the last
 * blockIdx.x, the gates of PC_TB tokens. Rows before the chunk come from the conv state, which is
 * only read here (lin_rulec_k writes the chunk's last rows into it): blocks of tokens run in any
 * order. lin_pre_k walks the tokens in one workgroup per channel group. */
__global__ __launch_bounds__(256) void lin_prec_k(nmx_lin_pre_args a) {
    extern __shared__ float sq[]; /* [PC_TB][dk] squares */
    __shared__ float red[4 * PC_TB];
    const int tid = threadIdx.x, t0 = blockIdx.y * PC_TB;
    const int nb = a.n - t0 < PC_TB ? a.n - t0 : PC_TB;
    if (blockIdx.x == gridDim.x - 1) {
        for (int u = tid; u < nb * a.heads; u += blockDim.x) {
            const int t = t0 + u / a.heads, h = u % a.heads;
            const float b = a.b_in[(size_t)t * a.g_stride + h];
            const float av = a.a_in[(size_t)t * a.g_stride + h];
            a.beta[t * a.heads + h] = 1.0f / (1.0f + nmx_gate_expf(-b));
            const float A = a.A ? a.A[h] : -nmx_gate_expf(a.A_log[h]);
            float sp = av + a.dt_bias[h];
            sp = sp > 20.0f ? sp : nmx_gate_log1pf(nmx_gate_expf(sp));
            a.decay[t * a.heads + h] = nmx_gate_expf(A * sp);
        }
        return;
    }
    const int ch = blockIdx.x * a.dk + tid;
    const bool live = tid < a.dk && ch < a.C;
    const int cc = live ? ch : 0;
    float x[PC_TB + 3], w[4], y[PC_TB];
#pragma unroll
    for (int r = 0; r < 4; r++) w[r] = a.conv_w[(size_t)cc * 4 + r];
#pragma unroll
    for (int r = 0; r < PC_TB + 3; r++) { /* rows t0 - 3 .. of [state | raw] */
        int t = t0 - 3 + r;
        t = t < a.n ? t : a.n - 1;
        x[r] = t < 0 ? a.state[(size_t)(t + 3) * a.C + cc] : a.raw[(size_t)t * a.raw_stride + cc];
    }
#pragma unroll
    for (int u = 0; u < PC_TB; u++) {
        float acc = w[0] * x[u];
        acc = acc + w[1] * x[u + 1];
        acc = acc + w[2] * x[u + 2];
        acc = acc + w[3] * x[u + 3];
        y[u] = nmx_silu(acc);
    }
    if ((int)blockIdx.x * a.dk < 2 * a.kd) { /* a q or k head */
        const float scale = (int)blockIdx.x * a.dk < a.kd ? a.qscale : 1.0f;
#pragma unroll
        for (int u = 0; u < PC_TB; u++)
            if (tid < a.dk) sq[u * a.dk + tid] = live ? y[u] * y[u] : 0.0f;
        __syncthreads();
        if (tid < 4 * PC_TB) { /* 4 interleaved partial sums per token */
            const float *v = sq + (tid >> 2) * a.dk + (tid & 3);
            const int m4 = a.dk >> 2;
            float c = 0.0f;
            for (int m = 0; m < m4; m += 8) {
                float b[8];
#pragma unroll
                for (int k = 0; k < 8; k++) b[k] = v[4 * (m + k)];
#pragma unroll
                for (int k = 0; k < 8; k++) c = c + b[k];
            }
            red[tid] = c;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < PC_TB; u++) {
            const float ss = ((red[4 * u] + red[4 * u + 1]) + (red[4 * u + 2] + red[4 * u + 3])) + 0.0f;
            const float r = 1.0f / sqrtf(ss + a.l2eps);
            y[u] = (y[u] * r) * scale;
        }
    }
#pragma unroll
    for (int u = 0; u < PC_TB; u++)
        if (u < nb && live) a.out[(size_t)(t0 + u) * a.C + ch] = y[u];
}

/* Tokens run in batches of TB (one barrier, one staged batch each). The o chains end a batch and 15
 * steps after the kv chains, which restart their operand reads at every batch: batches of 8 for
 * chunks of up to RC_SHORT tokens, where the end counts, of 16 above. us in batches of 8 and of 16:
 * 64 tokens 34.3 and 37.4, 192 86.2 and 87.6, 256 111.9 and 113.0, 320 138.1 and 137.9, 512 216.0 and
 * 214.7. */
constexpr int RC_SHORT = 256;
constexpr int RC_JW = 8;   /* value columns per workgroup */
constexpr int RC_TOK = 64; /* tokens in LDS: a batch being staged, one in the kv chains, those of the
                            * last 15 steps in the o chains */

/* LDS row stride of a token's keys: 16 lanes reading their keys of 16 consecutive tokens are
 * 4 (mod 64) words apart, so their 16-byte reads cover the banks once */
constexpr int rc_row(int dk) { return dk + (dk == 128 ? 4 : dk == 64 ? 8 : 12); }

template <int KP>
__device__ __forceinline__ void load_keys(float (&x)[KP], const float *p) {
#pragma unroll
    for (int r = 0; r < KP; r += 4) {
        const float4 v = *(const float4 *)(p + r);
        x[r] = v.x, x[r + 1] = v.y, x[r + 2] = v.z, x[r + 3] = v.w;
    }
}

/* the previous lane's value within a row of 16 (0 in lane 0) */
__device__ __forceinline__ float from_prev(float v) {
    return __int_as_float(nmx_dpp<0x111>(__float_as_int(v))); /* row_shr:1 */
}

/* KP keys per lane (dk = 16 KP). Waves 0, 1: kv chains of columns 4 w .. 4 w + 3; waves 2, 3: o
 * chains of the same columns, and the staging of every batch. Iteration i: batch i in the kv
 * chains, the steps of batch i - 1 in the o chains (reaching back 15 tokens),
 * batch i + 1 staged. */
template <int KP, int RC_TB>
__global__ __launch_bounds__(256) void lin_rulec_k(nmx_lin_args a, const float *__restrict__ raw,
                                                   int raw_stride, float *__restrict__ conv, int C) {
    constexpr int DK = 16 * KP, ROW = rc_row(DK), RC_RING = RC_TOK / RC_TB;
    constexpr int RC_LAG = 1 + (15 + RC_TB - 1) / RC_TB; /* batches from the kv chains' end to the o's */
    extern __shared__ __align__(16) float sm[];
    float *sk = sm, *sq = sk + RC_TOK * ROW;          /* [RC_TOK][ROW] */
    float *sv = sq + RC_TOK * ROW, *sdel = sv + RC_TOK * RC_JW; /* [RC_TOK][RC_JW] */
    float *sdec = sdel + RC_TOK * RC_JW, *sbet = sdec + RC_TOK;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, part = lane & 15;
    const int h = blockIdx.x, j0 = blockIdx.y * RC_JW, jl = 4 * (wave & 1) + (lane >> 4), j = j0 + jl;
    const int n = a.n, heads = a.heads, dv = a.dv, kh = h / a.rep, kd = (heads / a.rep) * DK;
    const int nbat = (n + RC_TB - 1) / RC_TB;
    const bool kvw = wave < 2;

    float *Sp = a.S + state_lane(h, j, part >> 2, DK, dv);
    const int SS = state_slot(j, dv), k0 = (part & 3) * (KP / 4);
    float s[KP];
#pragma unroll
    for (int r = 0; r < KP; r += 4) {
        const float4 x = *(const float4 *)(Sp + (k0 + (r >> 2)) * SS);
        s[r] = x.x, s[r + 1] = x.y, s[r + 2] = x.z, s[r + 3] = x.w;
    }
    int keep = a.keep;
    if (a.keep_dev) {
        const int kd_ = *a.keep_dev;
        keep = kd_ < keep ? kd_ : keep;
    }
    for (int u = 0; u < keep; u++) { /* pending rows (matvec_ref.c:169-188 arithmetic) */
        const float *row = a.pend + ((size_t)u * heads + h) * (DK + dv + 1);
        const float pdec = row[DK + dv], pdel = row[DK + j];
        float kk[KP];
#pragma unroll
        for (int r = 0; r < KP; r++) kk[r] = row[part * KP + r];
#pragma unroll
        for (int r = 0; r < KP; r++) {
            s[r] = s[r] * pdec;
            s[r] = s[r] + kk[r] * pdel;
        }
    }

    /* staging by waves 2, 3 (thread x of 128): q and k rows as float4, v, gates */
    constexpr int F4 = DK / 4, PER = RC_TB * F4 / 128;
    const int x0 = tid - 128;
    float4 fq[PER], fk[PER];
    float fv = 0.0f, fg = 0.0f;
    auto request = [&](int b) {
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const int x = e * 128 + x0;
            int t = b * RC_TB + x / F4;
            t = t < n ? t : n - 1;
            const float *row = a.qkv + (size_t)t * a.qkv_stride + kh * DK + 4 * (x % F4);
            fq[e] = *(const float4 *)row;
            fk[e] = *(const float4 *)(row + kd);
        }
        const int xv = x0 % (RC_TB * RC_JW); /* RC_TB tokens x 8 columns */
        int t = b * RC_TB + xv / RC_JW;
        t = t < n ? t : n - 1;
        fv = a.qkv[(size_t)t * a.qkv_stride + 2 * kd + h * dv + j0 + xv % RC_JW];
        int tg = b * RC_TB + x0 % RC_TB;
        tg = tg < n ? tg : n - 1;
        fg = (x0 < RC_TB ? a.decay : a.beta)[(size_t)tg * heads + h];
    };
    auto stage = [&](int b) {
        const int s0 = (b % RC_RING) * RC_TB;
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const int x = e * 128 + x0, o = (s0 + x / F4) * ROW + 4 * (x % F4);
            *(float4 *)(sq + o) = fq[e];
            *(float4 *)(sk + o) = fk[e];
        }
        if (x0 < RC_TB * RC_JW) sv[s0 * RC_JW + x0] = fv;
        if (x0 < RC_TB) sdec[s0 + x0] = fg;
        else if (x0 < 2 * RC_TB) sbet[s0 + x0 - RC_TB] = fg;
    };
    if (!kvw) {
        request(0);
        stage(0);
    }
    __syncthreads();
    float acc = 0.0f;
    for (int i = 0; i < nbat + RC_LAG; i++) {
        if (kvw) {
            if (i < nbat) {
                const int tn = n - i * RC_TB < RC_TB ? n - i * RC_TB : RC_TB;
                const int s0 = (i % RC_RING) * RC_TB;
                const float *kr = sk + s0 * ROW + part * KP;
                float k[KP], v = sv[s0 * RC_JW + jl], dec = sdec[s0], bet = sbet[s0];
                load_keys(k, kr);
                for (int u = 0; u < tn; u++) {
                    /* the next token's operands, ahead of this one's chain (past the batch: the
                     * next slot's, unused; the ring's last slot reads the first) */
                    const int sn = (s0 + u + 1) & (RC_TOK - 1);
                    float kn[KP];
                    load_keys(kn, sk + sn * ROW + part * KP);
                    const float vn = sv[sn * RC_JW + jl], decn = sdec[sn], betn = sbet[sn];
                    float p[KP];
#pragma unroll
                    for (int r = 0; r < KP; r++) {
                        s[r] = s[r] * dec;
                        p[r] = s[r] * k[r];
                    }
                    /* lane c adds its keys at step c, to the sum that lane c - 1 left */
                    float kv = 0.0f;
#pragma unroll
                    for (int c = 0; c < 16; c++) {
                        kv = from_prev(kv);
#pragma unroll
                        for (int r = 0; r < KP; r++) kv = kv + p[r];
                    }
                    kv = __int_as_float(nmx_dpp<0x15F>(__float_as_int(kv))); /* row_newbcast:15 */
                    const float del = (v - kv) * bet;
                    sdel[(s0 + u) * RC_JW + jl] = del; /* the same value from 16 lanes */
#pragma unroll
                    for (int r = 0; r < KP; r++) {
                        s[r] = s[r] + k[r] * del;
                        k[r] = kn[r];
                    }
                    v = vn, dec = decn, bet = betn;
                }
            }
        } else {
            if (i + 1 < nbat) request(i + 1);
            if (i > 0) {
                const int tau0 = (i - 1) * RC_TB;
                float k[KP], q[KP], dec, del;
                auto operands = [&](int u) { /* of step u; outside the chunk some slot's, unused */
                    const int sl = (tau0 + u - part) & (RC_TOK - 1);
                    load_keys(k, sk + sl * ROW + part * KP);
                    load_keys(q, sq + sl * ROW + part * KP);
                    dec = sdec[sl], del = sdel[sl * RC_JW + jl];
                };
                operands(0);
#pragma unroll
                for (int u = 0; u < RC_TB; u++) {
                    const int t = tau0 + u - part;
                    acc = from_prev(acc);
                    float kc[KP], qc[KP];
                    const float dc = dec, ec = del;
#pragma unroll
                    for (int r = 0; r < KP; r++) kc[r] = k[r], qc[r] = q[r];
                    if (u + 1 < RC_TB) operands(u + 1);
                    if (t >= 0 && t < n) {
#pragma unroll
                        for (int r = 0; r < KP; r++) {
                            s[r] = s[r] * dc;
                            s[r] = s[r] + kc[r] * ec;
                            acc = acc + s[r] * qc[r];
                        }
                        if (part == 15) a.o[(size_t)t * a.o_stride + h * dv + j] = acc;
                    }
                }
            } else if (conv) { /* the chunk's last rows are the next conv state (lin_prec_k has read
                                * the old one) */
                const int nth = gridDim.x * gridDim.y * 128;
                for (int x = (blockIdx.y * gridDim.x + blockIdx.x) * 128 + x0; x < 3 * C; x += nth) {
                    const int r = x / C, c = x - r * C;
                    conv[x] = raw[(size_t)(n - 3 + r) * raw_stride + c];
                }
            }
            if (i + 1 < nbat) stage(i + 1);
        }
        __syncthreads();
    }
    if (kvw) {
#pragma unroll
        for (int r = 0; r < KP; r += 4)
            *(float4 *)(Sp + (k0 + (r >> 2)) * SS) = make_float4(s[r], s[r + 1], s[r + 2], s[r + 3]);
    }
}

template <int KP, int TB>
int launch_rulec(nmx_ctx *ctx, const nmx_lin_args &a, const float *raw, int raw_stride, float *conv,
                 int C) {
    const size_t lds = (2 * (size_t)RC_TOK * rc_row(16 * KP) + 2 * RC_TOK * RC_JW + 2 * RC_TOK) * 4;
    static std::atomic<uint64_t> lds_set;
    if (nmx_dyn_lds(ctx, (const void *)lin_rulec_k<KP, TB>, lds, lds_set)) return -1;
    const dim3 grid((unsigned)a.heads, (unsigned)(a.dv / RC_JW));
    lin_rulec_k<KP, TB><<<grid, 256, lds, ctx->stream>>>(a, raw, raw_stride, conv, C);
    NMX_LAUNCHED(ctx, "lin_rulec");
    return 0;
}

template <int TB>
int dispatch_tb(nmx_ctx *ctx, const nmx_lin_args &a, const float *raw, int raw_stride, float *conv, int C) {
    if (a.dk == 64) return launch_rulec<4, TB>(ctx, a, raw, raw_stride, conv, C);
    if (a.dk == 128) return launch_rulec<8, TB>(ctx, a, raw, raw_stride, conv, C);
    return launch_rulec<16, TB>(ctx, a, raw, raw_stride, conv, C);
}

int dispatch(nmx_ctx *ctx, const nmx_lin_args &a, const float *raw, int raw_stride, float *conv, int C) {
    return a.n <= RC_SHORT ? dispatch_tb<8>(ctx, a, raw, raw_stride, conv, C)
                           : dispatch_tb<16>(ctx, a, raw, raw_stride, conv, C);
}

} // namespace

/* More than 8 tokens without a log: below that the pipeline's fill (15 steps, one staged batch)
 * and, in the mixer, two more launches cost more than the chains save; a log's rows are written by
 * the verify kernels only. Whole groups of columns and float4 rows. */
bool nmx_lin_rulec_ok(const nmx_lin_args &a) {
    return a.n > 8 && !a.log && (a.dk == 64 || a.dk == 128 || a.dk == 256) && a.dv % RC_JW == 0 &&
           a.qkv_stride % 4 == 0 && ((uintptr_t)a.qkv & 15) == 0 && ((uintptr_t)a.S & 15) == 0;
}

int nmx_lin_rulec(nmx_ctx *ctx, const nmx_lin_args &a) {
    return dispatch(ctx, a, nullptr, 0, nullptr, 0);
}

int nmx_lin_mixc(nmx_ctx *ctx, const nmx_lin_pre_args &p, const nmx_lin_args &a) {
    const int groups = (p.C + p.dk - 1) / p.dk;
    const dim3 grid((unsigned)(groups + 1), (unsigned)((p.n + PC_TB - 1) / PC_TB));
    const unsigned threads = p.dk < 64 ? 64 : (unsigned)p.dk;
    lin_prec_k<<<grid, threads, (size_t)PC_TB * p.dk * 4, ctx->stream>>>(p);
    NMX_LAUNCHED(ctx, "lin_prec");
    return dispatch(ctx, a, p.raw, p.raw_stride, p.state, p.C);
}
