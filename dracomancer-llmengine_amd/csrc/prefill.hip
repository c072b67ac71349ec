// prefill.hip -- chunked prefill of the llama family (gfx950): the T tokens
// of a chunk go through each layer together, with the weight products on the
// f16-MFMA GEMM (gemmh.hip) and these row-parallel kernels around them:
//
//   k_pf_embed          X[t] = embedding row ids[t]
//   k_pf_rms            Xn[t] = RMSNorm(X[t]) * w            (src/m6_engine.c:31-37)
//   k_pf_add_rms        X[t] += Y[t], then the RMSNorm of the sum
//   k_pf_rope_append    rope on Q[t] and K[t] at position pos0 + t, K/V rows
//                       appended at cache row row0 + t       (src/m6_engine.c:456-481)
//   k_pf_attn, k_pf_merge
//                       causal attention: token t attends cache rows
//                       [0, row0 + t]                        (src/m6_engine.c:482-505)
//   k_pf_add            X += Y (residual)
//
// The result equals running the tokens one by one through m6_forward_token
// up to fp32 rounding (summation orders differ; the softmax is the split
// online form, exact in exact arithmetic).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "dev_common.h"
#include "embed_dev.h"
#include "formats.h"
#include "prefill.h"

namespace {

__global__ __launch_bounds__(256) void k_pf_embed(const uint8_t* __restrict__ base, DracoLayout L,
                                                  const int* __restrict__ ids, float* __restrict__ X) {
    const int t = blockIdx.y, p = blockIdx.x * 256 + threadIdx.x;
    if (p < L.n_in) X[(size_t)t * L.n_in + p] = embed_value(base, L, ids[t], p);
}

// one block of 256 threads per token row; x held in registers (h <= 256 * PF_RMS_PT)
constexpr int PF_RMS_PT = PF_H_MAX / 256;
__global__ __launch_bounds__(256) void k_pf_rms(const float* __restrict__ X, const float* __restrict__ w,
                                                float* __restrict__ Xn, int h, float eps) {
    __shared__ float red[4];
    const float* x = X + (size_t)blockIdx.x * h;
    float* o = Xn + (size_t)blockIdx.x * h;
    // every load (the row and its norm weights, clamped index) before the
    // first wait; a null weight re-reads the row
    const float* wp = w ? w : x;
    float v[PF_RMS_PT], wv[PF_RMS_PT];
#pragma unroll
    for (int k = 0; k < PF_RMS_PT; k++) {
        const int i = threadIdx.x + 256 * k, ic = i < h ? i : h - 1;
        v[k] = x[ic];
        wv[k] = wp[ic];
    }
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < PF_RMS_PT; k++) {
        if (threadIdx.x + 256 * k >= h) v[k] = 0.f;
        s = fmaf(v[k], v[k], s);
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    lds_barrier();
    const float tot = (red[0] + red[1]) + (red[2] + red[3]);
    const float inv = 1.f / sqrtf(tot / (float)h + eps);
#pragma unroll
    for (int k = 0; k < PF_RMS_PT; k++) {
        const int i = threadIdx.x + 256 * k;
        if (i < h) o[i] = w ? v[k] * inv * wv[k] : v[k] * inv;
    }
}

// X[t] += Y[t] (the residual), then Xn[t] = (X[t] * inv_rms) * w: one block
// per token row, the sum held in registers between the two steps
__global__ __launch_bounds__(256) void k_pf_add_rms(float* __restrict__ X, const float* __restrict__ Y,
                                                    const float* __restrict__ w, float* __restrict__ Xn, int h,
                                                    float eps) {
    __shared__ float red[4];
    float* x = X + (size_t)blockIdx.x * h;
    const float* y = Y + (size_t)blockIdx.x * h;
    float* o = Xn + (size_t)blockIdx.x * h;
    // every load (row, residual, norm weights; clamped index) before the
    // first wait and the first store; a null weight re-reads the row
    const float* wp = w ? w : x;
    float v[PF_RMS_PT], yv[PF_RMS_PT], wv[PF_RMS_PT];
#pragma unroll
    for (int k = 0; k < PF_RMS_PT; k++) {
        const int i = threadIdx.x + 256 * k, ic = i < h ? i : h - 1;
        v[k] = x[ic];
        yv[k] = y[ic];
        wv[k] = wp[ic];
    }
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < PF_RMS_PT; k++) {
        const int i = threadIdx.x + 256 * k;
        v[k] = i < h ? v[k] + yv[k] : 0.f;
        if (i < h) x[i] = v[k];
        s = fmaf(v[k], v[k], s);
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    lds_barrier();
    const float tot = (red[0] + red[1]) + (red[2] + red[3]);
    const float inv = 1.f / sqrtf(tot / (float)h + eps);
#pragma unroll
    for (int k = 0; k < PF_RMS_PT; k++) {
        const int i = threadIdx.x + 256 * k;
        if (i < h) o[i] = w ? v[k] * inv * wv[k] : v[k] * inv;
    }
}

// Q [T][NH*HD] rotated in place; K [T][KD] rotated into kc row row0 + t; V
// [T][KD] copied into vc row row0 + t.  One thread per even index of a pair
// (pairs (2i, 2i+1) of a head, the GGML "normal" rope, src/m6_engine.c:134-143).
__global__ __launch_bounds__(256) void k_pf_rope_append(float* __restrict__ Q, const float* __restrict__ K,
                                                        const float* __restrict__ V, float* __restrict__ kc,
                                                        float* __restrict__ vc, const float* __restrict__ tab,
                                                        int pos0, int row0, int NH, int NKV, int HD, int rot) {
    const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
    const int QD = NH * HD, KD = NKV * HD, half = rot / 2;
    const float* ang = tab + (size_t)(pos0 + t) * half * 2;
    if (i < QD) {
        const int d = i % HD;
        float* q = Q + (size_t)t * QD;
        if (d < rot && (d & 1) == 0) {
            const float c = ang[d], s = ang[d + 1];
            const float a = q[i], b = q[i + 1];
            q[i] = a * c - b * s;
            q[i + 1] = a * s + b * c;
        }
    } else if (i < QD + KD) {
        const int j = i - QD, d = j % HD;
        const float* k = K + (size_t)t * KD;
        float* dst = kc + (size_t)(row0 + t) * KD;
        if (d < rot) {
            if ((d & 1) == 0) {
                const float c = ang[d], s = ang[d + 1];
                const float a = k[j], b = k[j + 1];
                dst[j] = a * c - b * s;
                dst[j + 1] = a * s + b * c;
            }
        } else {
            dst[j] = k[j];
        }
    } else if (i < QD + 2 * KD) {
        const int j = i - QD - KD;
        vc[(size_t)(row0 + t) * KD + j] = V[(size_t)t * KD + j];
    }
}

// Causal attention of a chunk on the fp32 matrix instructions (16x16x4),
// split over the key rows: products and sums stay fp32, as a VALU dot's.
// Wave (16 queries of one q head) x tiles of 32 keys:
//   S^T = K Q^T   A = K rows (LDS), B = the queries (registers); lane (n, u) =
//                 (lane & 15, lane >> 4) gets keys 4u .. 4u+3 of query n
//   O^T += V^T P^T  the lane's scores are already the B operand of the step
//                 whose four keys are 4u + r, so P never leaves its registers;
//                 A row n of dim tile dt is dim 64 dg + 4 n + dt: one 16-byte
//                 LDS read feeds four products, and a lane's outputs come out
//                 as float4
// with the online softmax per 32 keys (a query's keys lie in four lanes: one
// max over them a tile, the sum only at the end).  A block is `hg` q heads of
// one kv head (a group's waves share the staged rows) x blockDim / 64 / hg
// query tiles; blockIdx.x = kv head * head groups + group.  K and V tiles are
// double-buffered in LDS, rows padded by 4 floats (conflict-free for both
// reads).  Writes the unnormalised (o[HD], m, l) of (head, query, split) for
// the merge kernel (pf_part_row).
//
// Bound by the matrix instructions' issue on whole chunks (HD products of 32
// cycles per 32 keys and wave).  Per launch, average over a prompt: 256-token
// chunks of 32 heads of 64 up to 960 keys 51 -> 19.3 us, 75 tokens at 275
// keys 36 -> 8.3; 191 tokens of 32 heads of 128 634 -> 16; 256-token chunks of
// 16 heads of 256 up to 2000 keys 107 -> 60 (a VALU lane per query, whose q
// and o of 128 dims spilled, before).
constexpr int PF_QT = 16, PF_KT = 32;
constexpr int PF_WAVES = 2048;  // waves a launch splits the keys for (launch_attn)
typedef float v4f __attribute__((ext_vector_type(4)));

template <int HD>
__global__ __launch_bounds__(512) void k_pf_attn(const float* __restrict__ Q, const float* __restrict__ kc,
                                                 const float* __restrict__ vc, float* __restrict__ part, int row0,
                                                 int T, int NH, int NKV, int nspl, int hg, float scale) {
    static_assert(pf_part_row(HD) % 4 == 0, "16-byte aligned rows of partials");
    constexpr int RS = HD + 4, NL = HD / 32;  // LDS row, float4 of a tile per thread of a 256-thread block
    extern __shared__ __align__(16) float sm[];  // [2][K 32 rows, V 32 rows][RS]
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, n = lane & 15, u = lane >> 4, NT = blockDim.x;
    const int rep = NH / NKV, ngrp = (rep + hg - 1) / hg, qw = (NT >> 6) / hg;
    const int g = blockIdx.x / ngrp, j = (blockIdx.x % ngrp) * hg + w % hg, qt = blockIdx.y * qw + w / hg;
    const int h = g * rep + min(j, rep - 1), KD = NKV * HD, QD = NH * HD;
    const int t = qt * PF_QT + n, qrow = row0 + t;
    const bool live = t < T && j < rep;
    const int kend = row0 + min(T, ((int)blockIdx.y + 1) * qw * PF_QT);
    const int chunk = ((kend + nspl - 1) / nspl + PF_KT - 1) / PF_KT * PF_KT;
    const int k0 = min(kend, (int)blockIdx.z * chunk), k1 = min(kend, k0 + chunk);
    // this wave's queries end here (a wave without any computes nothing)
    const int wend = j < rep && qt * PF_QT < T ? row0 + min(T, (qt + 1) * PF_QT) : 0;
    float4 q[HD / 16];
    const int tq = min(t, T - 1);  // a query past the chunk reads the last row and is discarded
#pragma unroll
    for (int i = 0; i < HD / 16; i++) q[i] = ld4(Q + (size_t)tq * QD + h * HD + 16 * i + 4 * u);
    float4 rg[NL];
    auto fetch = [&](const float* __restrict__ src, int kb) {  // rows past the split repeat its last one (masked)
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int e = min(tid + i * NT, PF_KT * HD / 4 - 1), r = e / (HD / 4), c = 4 * (e % (HD / 4));
            rg[i] = ld4(src + (size_t)min(kb + r, k1 - 1) * KD + g * HD + c);
        }
    };
    auto stash = [&](float* dst) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int e = tid + i * NT, r = e / (HD / 4), c = 4 * (e % (HD / 4));
            if (e < PF_KT * HD / 4) *reinterpret_cast<float4*>(dst + r * RS + c) = rg[i];
        }
    };
    v4f o[HD / 16];
#pragma unroll
    for (int i = 0; i < HD / 16; i++) o[i] = (v4f){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    if (k0 < k1) {
        fetch(kc, k0);
        stash(sm);
        fetch(vc, k0);
        stash(sm + PF_KT * RS);
    }
    // the queries have arrived before the loop (a wait for them inside would
    // also wait for the next tile)
#pragma unroll
    for (int i = 0; i < HD / 16; i++) asm volatile("" : "+v"(q[i].x), "+v"(q[i].y), "+v"(q[i].z), "+v"(q[i].w));
    lds_barrier();
    int b = 0;
    for (int kb = k0; kb < k1; kb += PF_KT, b ^= 1) {
        const bool more = kb + PF_KT < k1;
        // the next tile's K arrives during the scores, its V during P V (one
        // set of registers); the other buffer was last read before the barrier
        if (more) fetch(kc, kb + PF_KT);
        const float* Ks = sm + b * 2 * PF_KT * RS;
        const float* Vs = Ks + PF_KT * RS;
        float* const next = sm + (b ^ 1) * 2 * PF_KT * RS;
        v4f sc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        if (kb < wend) {
#pragma unroll
            for (int i = 0; i < HD / 16; i++) {
                const float4 ka = ld4(Ks + n * RS + 16 * i + 4 * u), kz = ld4(Ks + (16 + n) * RS + 16 * i + 4 * u);
                sc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.x, q[i].x, sc[0], 0, 0, 0);
                sc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kz.x, q[i].x, sc[1], 0, 0, 0);
                sc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.y, q[i].y, sc[0], 0, 0, 0);
                sc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kz.y, q[i].y, sc[1], 0, 0, 0);
                sc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.z, q[i].z, sc[0], 0, 0, 0);
                sc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kz.z, q[i].z, sc[1], 0, 0, 0);
                sc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.w, q[i].w, sc[0], 0, 0, 0);
                sc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kz.w, q[i].w, sc[1], 0, 0, 0);
            }
        }
        if (more) {
            stash(next);
            fetch(vc, kb + PF_KT);
        }
        if (kb < wend) {
            float cm = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int key = kb + 16 * kt + 4 * u + r;
                    sc[kt][r] = live && key <= qrow && key < k1 ? sc[kt][r] * scale : -INFINITY;
                    cm = fmaxf(cm, sc[kt][r]);
                }
            const float mn = fmaxf(m, rows_reduce(cm, OpMax{}));
            const float corr = m > -INFINITY ? expf(m - mn) : 0.f;
            l *= corr;
#pragma unroll
            for (int i = 0; i < HD / 16; i++) o[i] *= corr;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float p = sc[kt][r] > -INFINITY ? expf(sc[kt][r] - mn) : 0.f;
                    l += p;
                    const float* vr = Vs + (16 * kt + 4 * u + r) * RS + 4 * n;
#pragma unroll
                    for (int dg = 0; dg < HD / 64; dg++) {
                        const float4 v = ld4(vr + 64 * dg);
                        o[4 * dg] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.x, p, o[4 * dg], 0, 0, 0);
                        o[4 * dg + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.y, p, o[4 * dg + 1], 0, 0, 0);
                        o[4 * dg + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.z, p, o[4 * dg + 2], 0, 0, 0);
                        o[4 * dg + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.w, p, o[4 * dg + 3], 0, 0, 0);
                    }
                }
            m = mn;
        }
        if (more) {
            stash(next + PF_KT * RS);
            lds_barrier();
        }
    }
    l = rows_sum(l);
    if (!live) return;
    float* pp = part + (((size_t)h * T + t) * nspl + blockIdx.z) * pf_part_row(HD);
#pragma unroll
    for (int dg = 0; dg < HD / 64; dg++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            *reinterpret_cast<float4*>(pp + 64 * dg + 16 * u + 4 * r) =
                make_float4(o[4 * dg][r], o[4 * dg + 1][r], o[4 * dg + 2][r], o[4 * dg + 3][r]);
    if (u == 0) {
        pp[HD] = m;
        pp[HD + 1] = l;
    }
}

// The split merge of four dims of one (query, head): M = max_s m_s, then
// num / den with den = sum_s l_s e^(m_s - M), num = sum_s o_s e^(m_s - M) in
// split order.  Loads go in batches of 8 splits, all of a batch requested
// together (clamped split index; the merge skips the clamped ones), instead of
// one dependent round trip per split.
__device__ __forceinline__ float4 pf_merge4(const float* __restrict__ pp, int HD, int nspl, int d) {
    constexpr int MB = 8;
    float M = -INFINITY;
    float4 num = make_float4(0.f, 0.f, 0.f, 0.f);
    float den = 0.f;
    float2 ml[MB];
    float4 ov[MB];
    auto load = [&](int s0) {
#pragma unroll
        for (int k = 0; k < MB; k++) {
            const float* q = pp + (size_t)min(s0 + k, nspl - 1) * pf_part_row(HD);
            ml[k] = *reinterpret_cast<const float2*>(q + HD);
            ov[k] = ld4(q + d);
        }
    };
    auto add = [&](int s0) {
#pragma unroll
        for (int k = 0; k < MB; k++) {
            if (s0 + k >= nspl || ml[k].x == -INFINITY) continue;
            const float e = expf(ml[k].x - M);
            den = fmaf(ml[k].y, e, den);
            num.x = fmaf(ov[k].x, e, num.x);
            num.y = fmaf(ov[k].y, e, num.y);
            num.z = fmaf(ov[k].z, e, num.z);
            num.w = fmaf(ov[k].w, e, num.w);
        }
    };
    load(0);  // the only batch of up to 8 splits: one round trip
#pragma unroll
    for (int k = 0; k < MB; k++) M = fmaxf(M, ml[k].x);
    for (int s = MB; s < nspl; s++) M = fmaxf(M, pp[(size_t)s * pf_part_row(HD) + HD]);
    add(0);
    for (int s0 = MB; s0 < nspl; s0 += MB) {
        load(s0);
        add(s0);
    }
    return make_float4(num.x / den, num.y / den, num.z / den, num.w / den);
}

// out[t][h*HD + d] = sum_s o_s[d] e^(m_s - M) / sum_s l_s e^(m_s - M); a
// thread per four dims (a block per (token, head) of HD threads made
// 8192 one-wave blocks of a chunk: 9.7 us, now 5.2).  gate (nullable): the qwen35 output
// gate, O *= sigmoid(gate row t, h*g_head + d) (the reference's attn *
// sigmoid(q gate half), src/qwen35_prefill.py:164-166 / src/m6_layer.c:497).
__global__ __launch_bounds__(256) void k_pf_merge(const float* __restrict__ part, float* __restrict__ O, int T,
                                                  int NH, int HD, int nspl, const float* __restrict__ gate,
                                                  int g_row, int g_head) {
    const int i = blockIdx.x * 256 + threadIdx.x, nd = HD / 4;
    if (i >= T * NH * nd) return;
    const int d = 4 * (i % nd), h = i / nd % NH, t = i / nd / NH;
    const float* pp = part + ((size_t)h * T + t) * nspl * pf_part_row(HD);
    float4 gv;
    if (gate) gv = ld4(gate + (size_t)t * g_row + (size_t)h * g_head + d);
    float4 v = pf_merge4(pp, HD, nspl, d);
    if (gate) {
        v.x *= 1.f / (1.f + expf(-gv.x));
        v.y *= 1.f / (1.f + expf(-gv.y));
        v.z *= 1.f / (1.f + expf(-gv.z));
        v.w *= 1.f / (1.f + expf(-gv.w));
    }
    *reinterpret_cast<float4*>(O + (size_t)t * NH * HD + h * HD + d) = v;
}

// GDN gates of a chunk (src/qwen35_prefill.py:118-123): for token t and V
// head e, B = sigmoid(Xn[t] . bw[e]) and G = exp(softplus(Xn[t] . aw[e] +
// dt[e]) * a[e]); bw / aw stored [n_vh][H].  Block (t, e), 256 threads.
__global__ __launch_bounds__(256) void k_pf_gdn_gates(const float* __restrict__ Xn, int H,
                                                      const float* __restrict__ bw, const float* __restrict__ aw,
                                                      const float* __restrict__ dt, const float* __restrict__ sa,
                                                      float* __restrict__ B, float* __restrict__ G, int n_vh) {
    __shared__ float red[2][4];
    const int t = blockIdx.x, e = blockIdx.y, tid = threadIdx.x;
    const float* x = Xn + (size_t)t * H;
    float sb = 0.f, sa_ = 0.f;
    for (int i = tid * 4; i < H; i += 1024) {
        const float4 xv = ld4(x + i), bv = ld4(bw + (size_t)e * H + i), av = ld4(aw + (size_t)e * H + i);
        sb = fmaf(xv.x, bv.x, sb); sb = fmaf(xv.y, bv.y, sb); sb = fmaf(xv.z, bv.z, sb); sb = fmaf(xv.w, bv.w, sb);
        sa_ = fmaf(xv.x, av.x, sa_); sa_ = fmaf(xv.y, av.y, sa_); sa_ = fmaf(xv.z, av.z, sa_); sa_ = fmaf(xv.w, av.w, sa_);
    }
    sb = wave_sum(sb);
    sa_ = wave_sum(sa_);
    if ((tid & 63) == 0) {
        red[0][tid >> 6] = sb;
        red[1][tid >> 6] = sa_;
    }
    __syncthreads();
    if (tid == 0) {
        const float b = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
        const float a = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]) + dt[e];
        const float sp = a > 0.f ? a + log1pf(expf(-a)) : log1pf(expf(a));  // softplus, src/m6_layer.c:253
        B[(size_t)t * n_vh + e] = 1.f / (1.f + expf(-b));
        G[(size_t)t * n_vh + e] = expf(sp * sa[e]);
    }
}

__global__ __launch_bounds__(256) void k_pf_add(float* __restrict__ X, const float* __restrict__ Y, size_t n) {
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) X[i] += Y[i];
}

}  // namespace

int pf_attn_nsplit(int row0, int T) {
    // about 64 key rows per split at the tile holding the chunk's last query
    const int n = (row0 + T + 63) / 64;
    return n < 1 ? 1 : (n > 64 ? 64 : n);
}

// Enough for every chunk of up to T tokens: launch_attn's splits are at most
// nspl, and at most PF_WAVES / waves rounded up, with at least NH * T / 16 waves.
size_t pf_part_floats(int NH, int T, int HD, int nspl) {
    return std::min((size_t)NH * T * nspl, (size_t)PF_QT * PF_WAVES + (size_t)NH * T) * pf_part_row(HD);
}

int pf_embed(const uint8_t* base, const DracoLayout& L, const int* ids, int T, float* X, hipStream_t st) {
    if (T < 1) return -1;
    hipLaunchKernelGGL(k_pf_embed, dim3((L.n_in + 255) / 256, T), dim3(256), 0, st, base, L, ids, X);
    return 0;
}

int pf_rms(const float* X, const float* w, float* Xn, int T, int h, float eps, hipStream_t st) {
    if (T < 1 || h > PF_H_MAX) return -1;
    hipLaunchKernelGGL(k_pf_rms, dim3(T), dim3(256), 0, st, X, w, Xn, h, eps);
    return 0;
}

int pf_add_rms(float* X, const float* Y, const float* w, float* Xn, int T, int h, float eps, hipStream_t st) {
    if (T < 1 || h > PF_H_MAX) return -1;
    hipLaunchKernelGGL(k_pf_add_rms, dim3(T), dim3(256), 0, st, X, Y, w, Xn, h, eps);
    return 0;
}

int pf_rope_append(float* Q, const float* K, const float* V, float* kc, float* vc, const float* tab, int pos0,
                   int row0, int T, int NH, int NKV, int HD, int rot, hipStream_t st) {
    if (T < 1 || (rot & 1) || rot > HD) return -1;
    const int n = NH * HD + 2 * NKV * HD;
    hipLaunchKernelGGL(k_pf_rope_append, dim3((n + 255) / 256, T), dim3(256), 0, st, Q, K, V, kc, vc, tab, pos0,
                       row0, NH, NKV, HD, rot);
    return 0;
}

namespace {

// The attention launch of a chunk.  Blocks of 4 to 8 waves: a kv head's q
// heads (up to 8), and two or four query tiles where the group has fewer than
// four.  The key rows are split until about PF_WAVES waves run (never finer
// than pf_attn_nsplit): a split costs a row of partials per query that the
// merge reads again.  1024 / 2048 / 4096 waves: 22.3 / 19.3 / 18.9 us at head
// dim 64 (chunks of a 960-token prompt), 92 / 60 / 76 at 256 (2000 tokens).
template <int HD>
int launch_attn(const float* Q, const float* kc, const float* vc, float* part, int row0, int T, int NH, int NKV,
                float scale, hipStream_t st, int* nsplit) {
    const int rep = NH / NKV, hg = rep < 8 ? rep : 8, qw = hg >= 4 ? 1 : (hg == 1 ? 4 : 2), ngrp = (rep + hg - 1) / hg;
    const int qb = (T + PF_QT * qw - 1) / (PF_QT * qw), waves = NKV * ngrp * qb * hg * qw;
    const int nspl = std::min(pf_attn_nsplit(row0, T), (PF_WAVES + waves - 1) / waves);
    constexpr int lds = sizeof(float) * 2 * 2 * PF_KT * (HD + 4);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pf_attn<HD>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return -1;
    hipLaunchKernelGGL(k_pf_attn<HD>, dim3(NKV * ngrp, qb, nspl), dim3(64 * hg * qw), lds, st, Q, kc, vc, part, row0,
                       T, NH, NKV, nspl, hg, scale);
    *nsplit = nspl;
    return 0;
}

}  // namespace

int pf_attention(const float* Q, const float* kc, const float* vc, float* part, float* O, int row0, int T, int NH,
                 int NKV, int HD, float scale, hipStream_t st) {
    if (T < 1 || !pf_attention_ok(NH, NKV, HD)) return -1;
    int nspl = 1;
    const int rc = HD == 64 ? launch_attn<64>(Q, kc, vc, part, row0, T, NH, NKV, scale, st, &nspl)
                            : launch_attn<128>(Q, kc, vc, part, row0, T, NH, NKV, scale, st, &nspl);
    if (rc) return rc;
    hipLaunchKernelGGL(k_pf_merge, dim3((T * NH * (HD / 4) + 255) / 256), dim3(256), 0, st, part, O, T, NH, HD, nspl,
                       (const float*)nullptr, 0, 0);
    return 0;
}

int pf_attention256(const float* Q, const float* kc, const float* vc, float* part, float* O, int row0, int T, int NH,
                    int NKV, float scale, const float* gate, int g_row, int g_head, hipStream_t st) {
    if (T < 1 || NKV < 1 || NH % NKV || NH / NKV > 16 || !gate) return -1;
    int nspl = 1;
    if (launch_attn<256>(Q, kc, vc, part, row0, T, NH, NKV, scale, st, &nspl)) return -1;
    hipLaunchKernelGGL(k_pf_merge, dim3((T * NH * 64 + 255) / 256), dim3(256), 0, st, part, O, T, NH, 256, nspl, gate,
                       g_row, g_head);
    return 0;
}

int pf_gdn_gates(const float* Xn, int T, int H, const float* bw, const float* aw, const float* dt, const float* sa,
                 float* B, float* G, int n_vh, hipStream_t st) {
    if (T < 1 || H % 4 || n_vh < 1) return -1;
    hipLaunchKernelGGL(k_pf_gdn_gates, dim3(T, n_vh), dim3(256), 0, st, Xn, H, bw, aw, dt, sa, B, G, n_vh);
    return 0;
}

int pf_add(float* X, const float* Y, size_t n, hipStream_t st) {
    const size_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(k_pf_add, dim3(blocks < 2048 ? (unsigned)blocks : 2048u), dim3(256), 0, st, X, Y, n);
    return 0;
}
