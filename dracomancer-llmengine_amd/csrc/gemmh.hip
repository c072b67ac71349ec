// gemmh.hip -- chunked-prefill GEMM on f16 MFMA (gfx950): Y[t][n] = x_t . W_n
// for Q4_K, Q5_K, Q6_K and Q8_0 weights in their device layouts (formats.h).
//
// Exactness.  The weights enter the MFMA as f16 integers: Q4_K sc*(q-8) (at
// most 63*8), Q5_K sc*(q-16) (63*16), Q8_0 q, all exact; Q6_K sc*(q-32) (|.| <= 4096)
// as its f16 rounding plus the rest (-1, 0 or 1).  Per (token, 256-value
// super-block) the activations are scaled by 2^-e (e = ilogb(max|x|) - 14, so
// |x'| < 2^15) and split into two f16 (hi = f16(x'), lo = f16(x' - hi)): 23 of
// an fp32 value's 24 bits, x' - hi - lo at most 2^-23 |x'|, or 2^-25 where lo is
// an f16 subnormal (values below 2^-16 of the super-block's largest: 2^-39 of
// that one).  The product left out (Q6_K's lo * rest) is below 2^-22 of the
// value's.  f16 x f16 products are exact; the MFMA adds them to fp32 with their
// low bits rounded down (tile_mma, Q8_0).
// Per super-block and row, with 2^e the token's scale:
//   Q4_K, Q5_K: y += 2^e * (d * (sum_k (sc*(q-z))_k x'_k + 32 * z * sum_sb sc_sb S'_sb)
//                           - 32 * dmin * sum_sb m_sb S'_sb), z = 8 or 16,
//         with S'_sb = 2^-5 * (sum of the sub-block's x'), the sums over
//         sub-blocks themselves on the MFMA (K = 8 sub-blocks, hi/lo);
//   Q6_K: y += 2^e * d * sum (sc*(q-32)) x';
//   Q8_0: y += 2^e * sum_blocks d_block * (sum q x').
// The hi and the lo products accumulate apart: the lo sums are 2^-11 of the
// hi ones, so their roundings vanish and the hi chain is half as long.  (In one
// MFMA the lo products lose their low bits to the hi ones', always downwards:
// the min and centre sums formed so left a mean error of -3e-8.)
// Relative error against 64 bits at 256 tokens: Q4_K 1.15e-7 (2048-wide rows;
// 2.3e-7 in one chain, not centred), Q5_K 1.17e-7 (its GEMV 1.27e-7), Q6_K
// 1.28e-7 (1.56e-7 with scales split in two), Q8_0 9.7e-8 (2560-wide; its GEMV
// 1.26e-7, whose fp32 x keeps the 24th bit and values of any range).
//
// Operand order.  v_mfma_f32_32x32x16_f16: A lane l = row (token) l%32,
// K 8*(l/32)..+7; B lane l = column (weight row) l%32, same K; C lane l =
// column l%32, rows 8*(i/4) + 4*(l/32) + i%4.  The K order inside a
// super-block is the one the tile layout hands each lane: K-step s (0..15),
// lane half u supplies the 8 values 16*G + 8*(s&1) + i of group
// G = 8*(s>>3) + 2*((s>>1)&3) + u -- for Q4_K the low (s>>1 even) or high
// nibbles of quant vector (r = s>>3, gh = (s>>2)&1), for Q6_K fragment
// (s>>1)&3 of lane slot s>>3, for Q8_0 half u of block s>>1.  k_gemmh_x
// writes the activations in the same order, so one activation buffer serves
// every format.
//
// The kernel (k_gemmr).  A block is 8 waves on one 32-token tile: NSB
// super-block slots x 8 / NSB row streams.  A wave holds its super-block's
// activation operands, hi and lo of 16 K-steps, in 128 VGPRs and runs the
// block's row tiles past them; a tile's weight registers refill with the next
// tile's bytes as they fall free; the slots' sums meet in LDS.  So
// activations are read once per block and pass instead of once per row tile,
// no wave waits for another inside a tile, and there is no K split over
// blocks with partials in memory unless rows are long (plan).  What bounds it:
// issue -- about 307 VALU and 36 MFMA instructions a (row tile, super-block) for
// Q4_K, which overlap only in part (a step of two waves takes 5.4k cycles, 2.3k
// of MFMA and 2.5k of VALU); a 32-token tile re-forms the weights that the next
// one forms too.  Against the kernel it replaced (activations staged in LDS
// super-block by super-block, K split over the grid and a reduce launch), us a
// product incl. reduce: T=256 2048x2048 Q4_K 15.7 -> 10.6, 8192x2048 31.6 -> 29.2;
// T=64 8192x2048 17.3 -> 11.5; Q6_K T=256 512x2048 12.4 -> 7.6, 2048x8192 50.9 ->
// 41.0, T=31 2048x8192 17.9 -> 12.3.  The two MFMAs of the centre term and its
// shifts cost Q4_K some 6%: it is slower than that kernel in launches of many
// tokens and rows (8192x2048 from 448 tokens on, 52 against 49 us) and on
// 768-wide rows of 8192 (T=256 17.9 against 15.1: three of four slots busy).
// Against GEMVs, whole host calls at 24 tokens: Q8_0 960x960 146 -> 46, Q5_K
// 2048x2048 159 -> 60.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "dev_common.h"
#include "formats.h"
#include "gemm.h"

namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int XH_A = 16 * 2 * 64 * 16;          // A operands of one super-block (bytes)
constexpr int XH_M = 2 * 64 * 16;               // min-term A operands
constexpr int XH_SB = XH_A + XH_M + 32 * 4;     // + 32 token scales = 34944 B per (token tile, super-block)

// ------------------------------------------------------------ activations --
// Block (b, tt), 256 threads: thread (m = tid/8, sb = tid%8) owns the 32
// values of sub-block sb of token 32*tt + m in super-block b; with `rows` the
// token's values are row rows[token] of X (negative: zeros), else its own row.
// Within each 8 the order is 0 2 1 3 4 6 5 7: the weights' bytes 0, 2 and 1, 3
// of a dword are formed as pairs.  Rows whose
// length is not a multiple of 256 (Q8_0) are padded with zeros.  An infinite
// value keeps its sign in hi with lo = 0 and a NaN stays NaN, so that token's
// results are not finite and the others' are untouched.  A Q8_0 row meets it as
// the fp32 dot would (inf * 0 = NaN included); Q4_K, Q5_K and Q6_K give NaN where
// the dot is infinite (their infinite min, centre and rest terms cancel).
__device__ __forceinline__ constexpr int kord(int i) { return (i & 4) + ((i & 1) << 1) + ((i >> 1) & 1); }
__global__ __launch_bounds__(256) void k_gemmh_x(const float* __restrict__ X, int T, int n_in,
                                                 const int* __restrict__ rows, uint8_t* __restrict__ xh) {
    const int b = blockIdx.x, tt = blockIdx.y, tid = threadIdx.x;
    const int m = tid >> 3, sb = tid & 7, t = 32 * tt + m, nb = (n_in + 255) >> 8;
    float v[32];
    if (rows && rows[32 * tt] < 0) return;  // a tile without tokens (they fill tiles from the front)
    const int row = t < T ? (rows ? rows[t] : t) : -1;
    const bool live = row >= 0 && b * 256 + 32 * sb < n_in;  // whole 32-value blocks (n_in % 32 == 0)
    const float* src = X + (size_t)max(row, 0) * n_in + (size_t)b * 256 + 32 * sb;
#pragma unroll
    for (int i = 0; i < 32; i += 4) {
        const float4 q = live ? ld4(src + i) : make_float4(0.f, 0.f, 0.f, 0.f);
        v[i] = q.x; v[i + 1] = q.y; v[i + 2] = q.z; v[i + 3] = q.w;
    }
    float am = 0.f;
#pragma unroll
    for (int i = 0; i < 32; i++) am = fmaxf(am, fabsf(v[i]));
    am = group_max<8>(am);  // the token's 8 threads are consecutive lanes
    const int e = am > 0.f ? min(max(ilogbf(am) - 14, -100), 113) : 0;
    const float sdown = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);  // 2^-e (e in [-100, 113])
    uint8_t* base = xh + ((size_t)tt * nb + b) * XH_SB;
    float ssum[4];  // the sub-block's sum, pairwise: the min terms multiply its rounding
#pragma unroll
    for (int gg = 0; gg < 2; gg++) {           // the two 16-value groups of this sub-block
        const int G = 2 * sb + gg, u = G & 1;
        const int lane = m + 32 * u;
#pragma unroll
        for (int bh = 0; bh < 2; bh++) {
            const int s = 8 * (G >> 3) + 2 * ((G >> 1) & 3) + bh;
            v8h hi, lo;
            float xv[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float xs = v[16 * gg + 8 * bh + kord(i)] * sdown;
                xv[i] = xs;
                const _Float16 h = (_Float16)xs;
                hi[i] = h;
                lo[i] = fabsf(xs) < INFINITY ? (_Float16)(xs - (float)h) : (_Float16)0.f;
            }
            ssum[2 * gg + bh] = ((xv[0] + xv[1]) + (xv[2] + xv[3])) + ((xv[4] + xv[5]) + (xv[6] + xv[7]));
            *reinterpret_cast<v8h*>(base + ((size_t)(2 * s) * 64 + lane) * 16) = hi;
            *reinterpret_cast<v8h*>(base + ((size_t)(2 * s + 1) * 64 + lane) * 16) = lo;
        }
    }
    // min-term operand: lane m (u = 0) holds S'_sb for sb = 0..7 in its 8 K slots
    // (the same order); lanes m + 32 (u = 1) hold zeros
    const float s5 = ((ssum[0] + ssum[1]) + (ssum[2] + ssum[3])) * 0.03125f;
    const _Float16 sh = (_Float16)s5;
    const _Float16 sl = fabsf(s5) < INFINITY ? (_Float16)(s5 - (float)sh) : (_Float16)0.f;
    _Float16* mh = reinterpret_cast<_Float16*>(base + XH_A);
    _Float16* ml = reinterpret_cast<_Float16*>(base + XH_A + 64 * 16);
    const int so = kord(sb);  // its own inverse
    mh[m * 8 + so] = sh;
    ml[m * 8 + so] = sl;
    mh[(m + 32) * 8 + so] = (_Float16)0.f;
    ml[(m + 32) * 8 + so] = (_Float16)0.f;
    if (sb == 0) reinterpret_cast<float*>(base + XH_A + XH_M)[m] = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
}

// ------------------------------------------------------------------ GEMM --
__device__ __forceinline__ v8h pack8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(v8h, (v4u32){a, b, c, d});
}
__device__ __forceinline__ v8h lds8(const uint8_t* p) { return *reinterpret_cast<const v8h*>(p); }
__device__ __forceinline__ v2h h2(uint32_t w) { return __builtin_bit_cast(v2h, w); }
__device__ __forceinline__ uint32_t u2(v2h h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ v2h splat(float v) { return (v2h){(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ v16f mfma16(v8h a, v8h b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
// (w & m) | k: with k = 0x64006400 the f16 pair (1024 + byte 0, 1024 + byte 2)
// of w & m.  The constant is held in a VGPR (magic_k): v_and_or_b32 takes one scalar operand, and with two constants the
// compiler uses two instructions (445 -> 365 VALU a tile).
__device__ __forceinline__ uint32_t magic(uint32_t w, uint32_t m, uint32_t k) { return (w & m) | k; }
__device__ __forceinline__ uint32_t magic_k() {
    uint32_t k = 0x64006400u;
    asm volatile("" : "+v"(k));
    return k;
}
// (byte 0, byte 2) and (byte 1, byte 3) of w as f16 pairs, plus 1024
__device__ __forceinline__ void pairs(uint32_t w, uint32_t mk, v2h& a, v2h& b) {
    a = h2(magic(w, 0x00FF00FFu, mk));
    b = h2(magic(w >> 8, 0x00FF00FFu, mk));
}

// One wave's raw weights of a (32-row tile, super-block), lane (n, u): row n
// of the tile, lane half u.  FM 1 = Q4_K, 2 = Q6_K, 3 = Q8_0, 4 = Q5_K.
template <int FM>
struct WFrag;
template <>
struct WFrag<1> {  // quant vectors (r, gh) = (v>>1, v&1), the row header
    uint4 qv[4], h;
};
template <>
struct WFrag<4> {  // the Q4_K ones, then the 16 fifth-bit bytes of half u
    uint4 qv[4], h, qh;
};
template <>
struct WFrag<2> {  // ql A, ql B, qh and 4 scales of lane slots g2 = 0, 1; d
    uint4 qa[2], qb[2], qh[2];
    uint32_t sc4[2];
    uint32_t d;
};
template <>
struct WFrag<3> {  // the 16 quants of (block k, half u) of the 8 blocks, and the blocks' f16 scales
    uint4 q[8];
    uint32_t d[8];
    int live;  // blocks that the row has from this super-block on
};

// Super-block b of 32-row tile t through a buffer descriptor: one wave-uniform
// base, the lane's offset fixed for the whole kernel (wlane), so walking tiles
// forms no per-lane address.  Reads past the matrix return zero (the rows
// after n_out).
template <int FM>
__device__ __forceinline__ int wlane(const DracoLayout& L, int n, int u) {
    constexpr int IB = FM == 1 ? DRACO_Q4T_ITEM : FM == 2 ? DRACO_Q6T_ITEM : DRACO_Q5T_ITEM;
    if constexpr (FM == 3) return n * L.nb * 32 + 16 * u;
    else return (n >> 4) * L.nb * IB + 16 * ((n & 15) + 16 * u);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const uint8_t* base, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), (short)0,
                                             (int)(bytes > 0x7FFFFFFFu ? 0x7FFFFFFFu : (uint32_t)bytes), 0x00020000);
}
__device__ __forceinline__ uint4 buf4(__amdgpu_buffer_rsrc_t r, int off) {
    const v4u32 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return make_uint4(v.x, v.y, v.z, v.w);
}
template <int FM>
struct WPtr {
    __amdgpu_buffer_rsrc_t r, rd;  // rd: Q8_0 scales
    int vo, n, u, live;
    __device__ __forceinline__ WPtr(const uint8_t* W, const DracoLayout& L, int t, int b, int vo_, int n_, int u_)
        : vo(vo_), n(n_), u(u_) {
        if constexpr (FM == 3) {
            const size_t e = (size_t)32 * t * L.nb + 8 * b, all = (size_t)L.n_out * L.nb;  // in blocks
            r = rsrc(W + L.off[0] + e * 32, e < all ? (all - e) * 32 : 0);
            rd = rsrc(W + L.off[1] + e * 2, e < all ? (all - e) * 2 : 0);
            live = L.nb - 8 * b;
        } else {
            constexpr size_t IB = FM == 1 ? DRACO_Q4T_ITEM : FM == 2 ? DRACO_Q6T_ITEM : DRACO_Q5T_ITEM;
            const size_t e = (size_t)2 * t * L.nb + b, all = (size_t)L.ntiles * L.nb;
            r = rsrc(W + e * IB, e < all ? (all - e) * IB : 0);
        }
    }
    // the pieces of WFrag<FM>, each loaded on its own so that a tile's
    // registers refill with the next tile's bytes as they fall free
    __device__ __forceinline__ void hdr(WFrag<FM>& f) const {
        if constexpr (FM == 1 || FM == 4) f.h = buf4(r, vo + 2048 - 256 * u);
        if constexpr (FM == 4) f.qh = buf4(r, vo + 2304);
        if constexpr (FM == 2) {
            const int j4 = 4 * ((n & 15) + 16 * u);  // this lane's slot, in 4-byte units
#pragma unroll
            for (int g2 = 0; g2 < 2; g2++)
                f.sc4[g2] = __builtin_amdgcn_raw_buffer_load_b32(r, vo - 3 * j4 + 3072 + 128 * g2, 0, 0);
            f.d = __builtin_amdgcn_raw_buffer_load_b16(r, vo - 4 * j4 + 3328 + 2 * (n & 15), 0, 0);
        }
        if constexpr (FM == 3) {
            const int vd = (vo - 16 * u) >> 4;
#pragma unroll
            for (int k = 0; k < 8; k++) f.d[k] = __builtin_amdgcn_raw_buffer_load_b16(rd, vd + 2 * k, 0, 0);
            f.live = live;
        }
    }
    // the quants of K-steps [4v, 4v + 4) (Q4_K, Q5_K, Q8_0) or, for even v, [4v, 4v + 8) (Q6_K)
    __device__ __forceinline__ void quants(WFrag<FM>& f, int v) const {
        if constexpr (FM == 1 || FM == 4) f.qv[v] = buf4(r, vo + (v >> 1) * 1024 + 512 * (v & 1));
        if constexpr (FM == 2) {
            if ((v & 1) == 0) {
                f.qa[v >> 1] = buf4(r, vo + 512 * (v >> 1));
                f.qb[v >> 1] = buf4(r, vo + 1024 + 512 * (v >> 1));
                f.qh[v >> 1] = buf4(r, vo + 2048 + 512 * (v >> 1));
            }
        }
        if constexpr (FM == 3) {
#pragma unroll
            for (int k = 2 * v; k < 2 * v + 2; k++) f.q[k] = buf4(r, vo + 32 * k);
        }
    }
};

// A (row tile, super-block)'s contribution before the token scales, o[i] per C
// element: hi / lo the wave's activation operands, mm its min-term operands
// (LDS, hi then lo, 1 KB each), nx the tile that follows.  The next K-step's
// weights are formed between this one's MFMAs (without the group barriers the
// compiler puts them all before: 53.6 -> 49.0 us at T=256 16384x2048), and the
// barrier per K-step keeps the live registers within two waves a SIMD.
template <int FM>
__device__ __forceinline__ void tile_mma(WFrag<FM>& f, const WPtr<FM>& nx, const v8h (&hi)[16], const v8h (&lo)[16],
                                         const uint8_t* mm, int lane, float (&o)[16]) {
    const uint32_t mk = magic_k();
    if constexpr (FM == 1 || FM == 4) {
        // 6-bit scales and mins (src/m5_kern_scalar.c:39-46), bytes of sub-blocks 0..3 and 4..7.
        // The quant sits at bits 4.. of its half: (1024 + 16 q) (c / 16) - (64 + z) c = (q - z) c with z = 8
        // (Q4_K) or 16 (Q5_K), and z sum_sb sc_sb S_sb joins beside the min term: centred, the weights' sum
        // is not twice the size of what the min term leaves of it
        constexpr float Z = FM == 4 ? 16.f : 8.f;
        const uint4 h = f.h;
        uint4 qh = {};
        if constexpr (FM == 4) qh = f.qh;
        const uint32_t sb[2] = {h.y & 0x3F3F3F3Fu, (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u)};
        const uint32_t mb[2] = {h.z & 0x3F3F3F3Fu, ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u)};
        const float dd = h2f((uint16_t)(h.x & 0xFFFF)), dm = -32.f * h2f((uint16_t)(h.x >> 16));
        v2h cc[4], oo[4];  // of sub-blocks (0, 2), (1, 3), (4, 6), (5, 7)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            v2h a, b;
            pairs(sb[q], mk, a, b);
            a = a - splat(1024.f);
            b = b - splat(1024.f);
            cc[2 * q] = a * splat(0.0625f);
            oo[2 * q] = a * splat(-64.f - Z);
            cc[2 * q + 1] = b * splat(0.0625f);
            oo[2 * q + 1] = b * splat(-64.f - Z);
        }
        nx.hdr(f);
        auto bfrag = [&](int s) {  // the weights of K-step s
            const int k = s >> 1, bh = s & 1, nib = k & 1;
            const uint4 qv = f.qv[s >> 2];
            const v2h cp = cc[2 * (k >> 2) + nib], op = oo[2 * (k >> 2) + nib];
            const v2h c = (k & 2) ? (v2h){cp.y, cp.y} : (v2h){cp.x, cp.x};
            const v2h of = (k & 2) ? (v2h){op.y, op.y} : (v2h){op.x, op.x};
            uint32_t p[4];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                uint32_t w = q ? (bh ? qv.w : qv.y) : (bh ? qv.z : qv.x);
                if constexpr (FM == 1) w ^= 0x80808080u;  // stored XOR 0x80
                uint32_t a = magic(nib ? w : w << 4, 0x00F000F0u, mk);
                uint32_t b = magic(nib ? w >> 8 : w >> 4, 0x00F000F0u, mk);
                if constexpr (FM == 4) {  // the fifth bit (value 32k + i: bit k of qh[i]) at bit 8
                    const uint32_t H = q ? (bh ? qh.w : qh.y) : (bh ? qh.z : qh.x);
                    a = magic(H << (8 - k), 0x01000100u, a);
                    b = magic(H >> k, 0x01000100u, b);
                }
                p[2 * q] = u2(__builtin_elementwise_fma(h2(a), c, of));
                p[2 * q + 1] = u2(__builtin_elementwise_fma(h2(b), c, of));
            }
            return pack8(p[0], p[1], p[2], p[3]);
        };
        v16f P = {}, Q = {};
        v8h B = bfrag(0), Bn = B;
#pragma unroll
        for (int s = 0; s < 16; s++) {
            __builtin_amdgcn_sched_barrier(0);
            if (s < 15) Bn = bfrag(s + 1);
            P = mfma16(hi[s], B, P);
            Q = mfma16(lo[s], B, Q);
            if ((s & 3) == 2) nx.quants(f, s >> 2);
#pragma unroll
            for (int g = 0; g < 2; g++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // one MFMA, then up to six VALU
                __builtin_amdgcn_sched_group_barrier(0x2, 6, 0);
            }
            B = Bn;
        }
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t keep = lane < 32 ? ~0u : 0u;  // min term: lanes (n, 1) hold zeros
        uint32_t bm[4];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            v2h a, b;
            pairs(mb[q], mk, a, b);
            bm[2 * q] = u2(a - splat(1024.f)) & keep;
            bm[2 * q + 1] = u2(b - splat(1024.f)) & keep;
        }
        const v8h Bm = pack8(bm[0], bm[1], bm[2], bm[3]);
        const v8h mh = lds8(mm + lane * 16), ml = lds8(mm + 1024 + lane * 16);
        const v16f M = mfma16(mh, Bm, mfma16(ml, Bm, (v16f){}));
        // 32 z sum_sb sc_sb S'_sb onto the small lo sums (cc holds sc / 16)
        uint32_t bs[4];
#pragma unroll
        for (int q = 0; q < 4; q++) bs[q] = u2(cc[q] * splat(512.f * Z)) & keep;
        const v8h Bs = pack8(bs[0], bs[1], bs[2], bs[3]);
        Q = mfma16(mh, Bs, mfma16(ml, Bs, Q));
#pragma unroll
        for (int i = 0; i < 16; i++) o[i] = fmaf(dd, P[i], fmaf(dm, M[i], dd * Q[i]));
    } else if constexpr (FM == 2) {
        const float dd = h2f((uint16_t)f.d);
        v2h c[2][2];
#pragma unroll
        for (int g = 0; g < 2; g++) {
            pairs(f.sc4[g] ^ 0x80808080u, mk, c[g][0], c[g][1]);
            c[g][0] = c[g][0] - splat(1152.f);
            c[g][1] = c[g][1] - splat(1152.f);
        }
        nx.hdr(f);
        auto bfrag = [&](int s, v8h& B, v8h& R) {  // rounding and rest of K-step s
            const int g = s >> 3, r6 = (s >> 1) & 3, bh = s & 1;
            const v2h cp = c[g][r6 & 1], cc = (r6 & 2) ? (v2h){cp.y, cp.y} : (v2h){cp.x, cp.x};
            const uint4 A4 = f.qa[g], B4 = f.qb[g], H4 = f.qh[g];
            uint32_t b[4], r[4];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const uint32_t av = bh ? (k ? A4.w : A4.z) : (k ? A4.y : A4.x);
                const uint32_t bv = bh ? (k ? B4.w : B4.z) : (k ? B4.y : B4.x);
                const uint32_t hv = bh ? (k ? H4.w : H4.z) : (k ? H4.y : H4.x);
                // the GGUF 6-bit map of src/m5_kern_scalar.c:115-142 (as the GEMV's dot_q6)
                uint32_t w;
                if (r6 == 0) w = (av & 0x0F0F0F0Fu) | ((hv << 4) & 0x30303030u);
                else if (r6 == 1) w = (bv & 0x0F0F0F0Fu) | ((hv << 2) & 0x30303030u);
                else if (r6 == 2) w = ((av >> 4) & 0x0F0F0F0Fu) | (hv & 0x30303030u);
                else w = ((bv >> 4) & 0x0F0F0F0Fu) | ((hv >> 2) & 0x30303030u);
                v2h q2[2];
                pairs(w, mk, q2[0], q2[1]);
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const v2h q = q2[e] - splat(1056.f), v = q * cc;
                    b[2 * k + e] = u2(v);
                    r[2 * k + e] = u2(__builtin_elementwise_fma(q, cc, -v));
                }
            }
            B = pack8(b[0], b[1], b[2], b[3]);
            R = pack8(r[0], r[1], r[2], r[3]);
        };
        v16f P = {}, Q = {};
        v8h B, R, Bn, Rn;
        bfrag(0, B, R);
        Bn = B;
        Rn = R;
#pragma unroll
        for (int s = 0; s < 16; s++) {
            __builtin_amdgcn_sched_barrier(0);
            if (s < 15) bfrag(s + 1, Bn, Rn);
            P = mfma16(hi[s], B, P);
            Q = mfma16(lo[s], B, Q);
            Q = mfma16(hi[s], R, Q);
            if ((s & 7) == 6) nx.quants(f, 2 * (s >> 3));
#pragma unroll
            for (int g = 0; g < 3; g++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);
            }
            B = Bn;
            R = Rn;
        }
#pragma unroll
        for (int i = 0; i < 16; i++) o[i] = fmaf(dd, P[i], dd * Q[i]);
    } else {
        // K-steps 2k, 2k + 1 are the row's block k: its scale multiplies the
        // block's dot (MFMAs from a zero accumulator), so d*q needs no
        // rounding.  Blocks past the row's end read the next row's quants
        // against activations that are zero, with a zero scale.
        // The odd blocks' quants enter negated, and their scale too: the MFMA
        // rounds the products' low bits down, not to nearest, so every block's
        // dot is off in the same direction.  Block sums of one sign left a mean
        // error of 3e-8 of the result's rms at 960-wide rows (5e-8 at 2560), the
        // same for every token: what averages over tokens (the attention)
        // kept it while its own size fell.  With the signs alternating it is
        // below 1e-9.
        uint32_t dk[4];
        const int lv = f.live;
#pragma unroll
        for (int k = 0; k < 4; k++) dk[k] = f.d[2 * k] | (f.d[2 * k + 1] << 16);
#pragma unroll
        for (int i = 0; i < 16; i++) o[i] = 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            __builtin_amdgcn_sched_barrier(0);
            v16f S = {};
            const uint4 q = f.q[k];
#pragma unroll
            for (int bh = 0; bh < 2; bh++) {
                const int s = 2 * k + bh;
                uint32_t p[4];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    v2h a, b;  // bytes XOR 0x80 read 128 + q
                    pairs((e ? (bh ? q.w : q.y) : (bh ? q.z : q.x)) ^ 0x80808080u, mk, a, b);
                    p[2 * e] = u2(k & 1 ? splat(1152.f) - a : a - splat(1152.f));
                    p[2 * e + 1] = u2(k & 1 ? splat(1152.f) - b : b - splat(1152.f));
                }
                const v8h B = pack8(p[0], p[1], p[2], p[3]);
                S = mfma16(lo[s], B, S);
                S = mfma16(hi[s], B, S);
            }
            __builtin_amdgcn_sched_barrier(0);
            const float d = k < lv ? h2f((uint16_t)(dk[k >> 1] >> (16 * (k & 1)))) : 0.f;
#pragma unroll
            for (int i = 0; i < 16; i++) o[i] = fmaf(k & 1 ? -d : d, S[i], o[i]);
            if (k & 1) nx.quants(f, k >> 1);
            if (k == 3) nx.hdr(f);  // (not from the start: its 8 registers are not there)
        }
    }
}

constexpr int GR_NR = 2;  // row tiles (or gate / up pairs' halves) per reduction step
constexpr size_t PART_MAX = (size_t)1 << 25;  // floats of partial sums that a launch takes at most (128 MB)

// The steps of one block on one matrix (PAIR: on two of the same shape and
// format, tile r of both, with the SwiGLU of the pair as the result).
template <int FM, int NSB, bool PAIR>
__device__ __forceinline__ void gemmr_body(const GemmHArgs& a, const GemmHSeg& sg, const uint8_t* W1, const uint8_t* W0,
                                           int tt, int t_live, int r0, int z, uint8_t* sm) {
    constexpr int RS = 8 / NSB;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, u = lane >> 5;
    const int slot = w % NSB, rs = w / NSB;
    const DracoLayout& L = sg.L;
    const int nb = (a.n_in + 255) >> 8, rts = (L.n_out + 31) >> 5;
    const int tiles = min(a.rpb, (rts - r0 + RS - 1) / RS);  // row tiles of the longest stream
    const int units = PAIR ? 2 * tiles : tiles;
    float* red = reinterpret_cast<float*>(sm);                     // [2][8][GR_NR][1024]
    uint8_t* mm = sm + 2 * 8 * GR_NR * 4096 + w * (2048 + 128);    // per wave: min operands, token scales
    v8h hi[16], lo[16];
    auto load_a = [&](int b) {
        const __amdgpu_buffer_rsrc_t r = rsrc(a.xh + ((size_t)tt * nb + b) * XH_SB, XH_SB);
        const v4u32 m0 = __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, XH_A, 0);
        const v4u32 m1 = __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, XH_A + 1024, 0);
        const uint32_t ts = __builtin_amdgcn_raw_buffer_load_b32(r, 4 * (lane & 31), XH_A + XH_M, 0);
#pragma unroll
        for (int s = 0; s < 16; s++) {
            hi[s] = __builtin_bit_cast(v8h, __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, (2 * s) * 1024, 0));
            lo[s] = __builtin_bit_cast(v8h, __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, (2 * s + 1) * 1024, 0));
        }
        *reinterpret_cast<v4u32*>(mm + lane * 16) = m0;
        *reinterpret_cast<v4u32*>(mm + 1024 + lane * 16) = m1;
        if (lane < 32) reinterpret_cast<uint32_t*>(mm + 2048)[lane] = ts;
    };
    // this block's passes of the row: split z of ksp
    const int passes = min(a.pps, (nb + NSB - 1) / NSB - z * a.pps), sb0 = slot + z * a.pps * NSB;
    float* const out = PAIR || a.ksp == 1 ? sg.Y : a.part + (size_t)z * a.T * sg.ldy;
    const int vo = wlane<FM>(L, n, u);
    // unit i of the block: row tile r0 + (i or i / 2) * RS + rs of matrix 0 (or 1 for the odd units of a pair)
    auto ptr = [&](int i, int b) {
        i = min(i, units - 1);
        return WPtr<FM>(PAIR && (i & 1) ? W1 : W0, L, r0 + (PAIR ? i >> 1 : i) * RS + rs, min(b, nb - 1), vo, n, u);
    };
    load_a(min(sb0, nb - 1));
    WFrag<FM> f;
    {
        const WPtr<FM> q = ptr(0, sb0);
        q.hdr(f);
#pragma unroll
        for (int v = 0; v < 4; v++) q.quants(f, v);
    }
    for (int st = 0; st < units; st += GR_NR) {
        float* rd = red + (size_t)((st / GR_NR) & 1) * 8 * GR_NR * 1024;
        float* own = rd + (size_t)w * GR_NR * 1024 + lane;
        const int nr = min(GR_NR, units - st);
        for (int ps = 0; ps < passes; ps++) {
            const int b = sb0 + ps * NSB;
            if (b >= nb) {  // a slot past the row's end (uniform per wave)
                if (ps == 0)
                    for (int e = 0; e < 16 * nr; e++) own[e * 64] = 0.f;
                continue;
            }
            if (passes > 1 && (st | ps)) load_a(b);
            // the pass whose weights follow this one's (this slot's last pass may be short)
            const int nps = ps + 1 < passes && b + NSB < nb ? ps + 1 : 0;
            for (int r = 0; r < nr; r++) {
                const WPtr<FM> nx = r + 1 < nr ? ptr(st + r + 1, b) : ptr(nps ? st : st + GR_NR, sb0 + nps * NSB);
                float o[16];
                tile_mma<FM>(f, nx, hi, lo, mm, lane, o);
                float* y = own + r * 1024;
                const float* ts = reinterpret_cast<const float*>(mm + 2048) + 4 * u;
                if (ps) {  // uniform; a pass at a time, so that no sum is held across tiles
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int e = 8 * (i >> 2) + (i & 3);
                        y[i * 64] = fmaf(o[i], ts[e], y[i * 64]);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 16; i++) y[i * 64] = o[i] * ts[8 * (i >> 2) + (i & 3)];
                }
            }
        }
        lds_barrier();
        // the slots' sums, pairwise: stream rs's elements over its NSB waves
        auto total = [&](int r, int i) {
            float v[NSB];
#pragma unroll
            for (int k = 0; k < NSB; k++) v[k] = rd[(size_t)((rs * NSB + k) * GR_NR + r) * 1024 + i * 64 + lane];
#pragma unroll
            for (int h = NSB / 2; h; h >>= 1)
#pragma unroll
                for (int k = 0; k < h; k++) v[k] += v[k + h];
            return v[0];
        };
        for (int e = slot; e < 16 * (PAIR ? 1 : nr); e += NSB) {
            const int i = e & 15, r = e >> 4;
            float s = total(r, i);
            if (PAIR) s = (s / (1.f + expf(-s))) * total(1, i);
            const int row = 32 * (r0 + (PAIR ? st >> 1 : st + r) * RS + rs) + n;
            const int tl = 8 * (i >> 2) + 4 * u + (i & 3);
            if (row < L.n_out && tl < t_live) out[(size_t)(32 * tt + tl) * sg.ldy + row] = s;
        }
    }
}

// An XCD (blocks x, x + 8, ...) runs the token tiles of one row group (of one
// split of its rows) one after the other, so a group's weights come from HBM
// once per XCD; in grouped launches the row groups of one tile, whose
// activations stay in that XCD's L2 (the experts' weights are read once anyway).
// gemmh_place spreads what does not divide by eight: with every row group whole
// on one XCD, launches of fewer than 8 groups (more than 1024 tokens) left the
// other XCDs idle and those of 9 put a second round of blocks on one (Q4_K: T=288
// 8192x2048 61.6 -> 35.4 us, T=4096 2048x2048 362 -> 118).
// F0 / F1: the formats that the launch's matrices have.
template <int F0, int F1, int NSB, bool PAIR>
__global__ __launch_bounds__(512) void k_gemmr(const GemmHArgs a) {
    extern __shared__ __align__(16) uint8_t sm[];
    const int ntt = a.groups ? a.max_tiles : (a.T + 31) >> 5;
    int maj, mnr;
    if (!gemmh_place(a.groups ? ntt : a.ksp * a.n_rg, a.groups ? a.n_rg : ntt, blockIdx.x, maj, mnr)) return;
    const int tt = a.groups ? maj : mnr, z = !PAIR && a.ksp > 1 ? maj / a.n_rg : 0;  // (grouped: ksp 1)
    const int rg = a.groups ? mnr : maj - z * a.n_rg;
    const int s = a.nseg > 1 && rg >= a.seg[1].rg0 ? (a.nseg > 2 && rg >= a.seg[2].rg0 ? 2 : 1) : 0;
    const GemmHSeg& sg = a.seg[s];
    const uint8_t *W0 = sg.W, *W1 = PAIR ? a.seg[1].W : nullptr;
    int live = a.T - 32 * tt;
    if (a.groups) {  // token tile tt belongs to one expert (negative: past the last tile)
        const int e = a.groups[tt];
        if (e < 0) return;
        W0 = sg.bases[e];
        if (PAIR) W1 = a.seg[1].bases[e];
        live = 32;
    }
    const int r0 = (rg - sg.rg0) * a.rpb * (8 / NSB);
    if (F0 == F1 || sg.fm == F0) gemmr_body<F0, NSB, PAIR>(a, sg, W1, W0, tt, live, r0, z, sm);
    else gemmr_body<F1, NSB, PAIR>(a, sg, W1, W0, tt, live, r0, z, sm);
}

// Y = the sum of the ksp partial products, in their order
__global__ __launch_bounds__(256) void k_gemmr_sum(const float* __restrict__ part, float* __restrict__ Y, size_t n,
                                                   int ksp) {
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        float s = part[i];
        for (int z = 1; z < ksp; z++) s += part[z * n + i];
        Y[i] = s;
    }
}
__global__ __launch_bounds__(256) void k_gemmr_sum4(const float4* __restrict__ part, float4* __restrict__ Y, size_t n,
                                                    int ksp) {
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        float4 s = part[i];
        for (int z = 1; z < ksp; z++) {
            const float4 v = part[z * n + i];
            s.x += v.x;
            s.y += v.y;
            s.z += v.z;
            s.w += v.w;
        }
        Y[i] = s;
    }
}

constexpr size_t GR_LDS = 2 * 8 * GR_NR * 4096 + 8 * (2048 + 128);

int fm_of(int code) {
    switch (code) {
    case DRACO_Q4_K: return 1;
    case DRACO_Q6_K: return 2;
    case DRACO_Q8_0: return 3;
    case DRACO_Q5_K: return 4;
    default: return 0;
    }
}

template <int F0, int F1, int NSB, bool PAIR>
void launch_r(const GemmHArgs& a, unsigned grid, hipStream_t st) {
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemmr<F0, F1, NSB, PAIR>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)GR_LDS);
        attr = true;
    }
    hipLaunchKernelGGL((k_gemmr<F0, F1, NSB, PAIR>), dim3(grid), dim3(512), GR_LDS, st, a);
}

template <int NSB>
void pick(const GemmHArgs& a, int f0, int f1, unsigned grid, hipStream_t st) {
    if (a.pair) {
        switch (f0) {
        case 1: launch_r<1, 1, NSB, true>(a, grid, st); return;
        case 2: launch_r<2, 2, NSB, true>(a, grid, st); return;
        case 3: launch_r<3, 3, NSB, true>(a, grid, st); return;
        default: launch_r<4, 4, NSB, true>(a, grid, st); return;
        }
    }
    if (f0 == f1) {
        switch (f0) {
        case 1: launch_r<1, 1, NSB, false>(a, grid, st); return;
        case 2: launch_r<2, 2, NSB, false>(a, grid, st); return;
        case 3: launch_r<3, 3, NSB, false>(a, grid, st); return;
        default: launch_r<4, 4, NSB, false>(a, grid, st); return;
        }
    }
    if (f0 == 1) launch_r<1, 2, NSB, false>(a, grid, st);
    else launch_r<4, 2, NSB, false>(a, grid, st);
}

}  // namespace

size_t draco_gemmh_x_bytes(int T, int n_in) { return (size_t)((T + 31) / 32) * ((n_in + 255) / 256) * XH_SB + 256; }

bool draco_gemmh_serves(int code) { return fm_of(code) != 0; }

unsigned draco_gemmh_blocks(int M, int m) {
    const GemmHMap g = gemmh_map(M, m);
    return 8u * (unsigned)(g.full + g.rem);
}
int draco_gemmh_place(int M, int m, int block) {
    int maj, mnr;
    return gemmh_place(M, m, block, maj, mnr) ? maj * m + mnr : -1;
}

// The formats one launch can mix: Q4_K or Q5_K with Q6_K (a Q4_K_M / Q5_K_M layer's q, k and v).
bool draco_gemmh_mixes(int c0, int c1) {
    return c0 == c1 || ((c0 == DRACO_Q4_K || c0 == DRACO_Q5_K) && c1 == DRACO_Q6_K) ||
           ((c1 == DRACO_Q4_K || c1 == DRACO_Q5_K) && c0 == DRACO_Q6_K);
}

int draco_gemmh_x_launch(const float* X, int T, int n_in, uint8_t* buf, hipStream_t st, const int* rows) {
    if (T < 1 || n_in < 32 || n_in % 32) return -1;
    hipLaunchKernelGGL(k_gemmh_x, dim3((n_in + 255) / 256, (T + 31) / 32), dim3(256), 0, st, X, T, n_in, rows, buf);
    return 0;
}

namespace {

// What a launch does per block: NSB super-block slots, rpb row tiles per
// stream, the row's passes (of NSB super-blocks) in ksp blocks of pps each.
struct Plan {
    int NSB, rpb, ksp, pps;
};

// Row tiles per block: as few as leave at most one block per CU (256).  With
// up to 512: T=256 2048x2048 10.6 -> 13.4 us, 12288x2048 at T=64 14.7 -> 19.9 (at
// T=128 23.3 -> 26.7).  Four super-block slots (two row streams) where rows have
// at most four super-blocks and there are row tiles enough for both streams:
// Q8_0 960x960 at T=31 7.5 us with eight slots, half of them idle, 8.9 with four;
// 5120x960 at T=31 7.7 / 9.2, at T=75 (480 tiles) 9.9 / 9.6.
//
// Rows of several passes load a block's activations again for every two row
// tiles and pass.  A single matrix may have its passes in ksp blocks instead,
// whose partial sums a second launch adds: where that is less work by the
// costs below (us), measured at 8 waves a block.  In blocks of whole rows / as
// split, incl. the operand launch: Q6_K 2048x8192 at T=16 25.4 / 16.2, 64 28.7 /
// 22.5, 160 43.1 / 39.4 (at 128 32.5 / 31.6 and 192 44.5 / 44.5: not split, the
// second launch costs a chain of eager launches more than that); 512x4096 at T=16
// 15.7 / 12.9; Q4_K 4096x14336 at T=16 37.0 / 24.5, 160 96.8 / 80.2.
Plan plan(const GemmHArgs& a, bool may_split) {
    const int ntt = a.groups ? a.max_tiles : (a.T + 31) / 32, nb = (a.n_in + 255) / 256;
    const int walk = a.pair ? 1 : a.nseg;  // matrices whose rows the blocks walk
    int rts = 0;
    for (int s = 0; s < walk; s++) rts += (a.seg[s].L.n_out + 31) / 32;
    Plan p;
    p.NSB = nb <= 4 && rts * ntt >= 1024 ? 4 : 8;
    const int RS = 8 / p.NSB, passes = (nb + p.NSB - 1) / p.NSB;
    auto rpb_of = [&](int ksp) {
        // (at least the row tiles over the streams of 256 blocks)
        for (int rpb = std::max(1, (int)((long long)rts * ntt * ksp / (256 * RS)));; rpb++) {
            int rg = 0;
            for (int s = 0; s < walk; s++) rg += ((a.seg[s].L.n_out + 31) / 32 + rpb * RS - 1) / (rpb * RS);
            if ((long long)rg * ntt * ksp <= 256 || rpb >= rts) return rpb;
        }
    };
    p.rpb = rpb_of(1);
    p.ksp = 1;
    p.pps = passes;
    if (!may_split || passes == 1) return p;
    constexpr double STEP = 2.2, LOAD = 1.8, SUM = 3.0;  // a tile's pass, an activation load, the second launch
    auto cost = [&](const Plan& q) {
        const double n = (double)a.T * a.seg[0].L.n_out;
        return q.rpb * q.pps * STEP + (q.pps > 1 ? (q.rpb + GR_NR - 1) / GR_NR * q.pps : 1) * LOAD +
               (q.ksp > 1 ? SUM + q.ksp * n * 8 / 5e6 : 0.);
    };
    Plan best = p;
    for (int pps = passes - 1; pps >= 1; pps--) {
        Plan q = p;
        q.pps = pps;
        q.ksp = (passes + pps - 1) / pps;
        q.rpb = rpb_of(q.ksp);
        if (q.ksp * ntt <= 256 && (size_t)q.ksp * a.T * a.seg[0].L.n_out <= PART_MAX && cost(q) < cost(best)) best = q;
    }
    // (blocks of several row tiles: up to 2 us less by these costs is a tie)
    return cost(best) + (best.rpb > 2 ? 2.2 : 0.) < cost(p) ? best : p;
}
bool splits(const GemmHArgs& a) { return a.nseg == 1 && !a.pair && !a.groups && a.seg[0].ldy == a.seg[0].L.n_out; }

}  // namespace

void draco_gemmh_plan(int n_out, int n_in, int T, int* out) {
    GemmHArgs a = {};
    a.nseg = 1;
    a.n_in = n_in;
    a.T = T;
    a.seg[0].L.n_out = a.seg[0].ldy = n_out;
    const Plan p = plan(a, true);
    out[0] = p.NSB;
    out[1] = p.rpb;
    out[2] = p.ksp;
    out[3] = p.pps;
}

size_t draco_gemmh_part_floats(const GemmHArgs& a) {
    if (!splits(a)) return 0;
    const Plan p = plan(a, true);
    return p.ksp > 1 ? (size_t)p.ksp * a.T * a.seg[0].L.n_out : 0;
}

int draco_gemmh_launch(GemmHArgs& a, hipStream_t st) {
    if (a.nseg < 1 || a.nseg > 3 || a.T < 1 || a.n_in < 32 || a.n_in % 32 || !a.xh) return -1;
    if (a.groups && (a.max_tiles < 1 || a.nseg != (a.pair ? 2 : 1))) return -1;
    int f0 = 0, f1 = 0;
    for (int s = 0; s < a.nseg; s++) {
        GemmHSeg& g = a.seg[s];
        g.fm = fm_of(g.L.code);
        if (!g.fm || g.L.n_in != a.n_in || (a.groups ? !g.bases : !g.W) || (!g.Y && !(a.pair && s))) return -1;
        if (s && !draco_gemmh_mixes(a.seg[0].L.code, g.L.code)) return -1;
        // F0 is the Q4_K / Q5_K one of a mix
        if (s == 0) f0 = f1 = g.fm;
        else if (g.fm != f0 && g.fm != f1) (g.fm == 2 ? f1 : f0) = g.fm;
    }
    if (a.pair && (a.nseg != 2 || f0 != f1 || a.seg[0].L.n_out != a.seg[1].L.n_out)) return -1;
    const Plan p = plan(a, a.part && splits(a));
    const int ntt = a.groups ? a.max_tiles : (a.T + 31) / 32, walk = a.pair ? 1 : a.nseg, RS = 8 / p.NSB;
    a.rpb = p.rpb;
    a.ksp = p.ksp;
    a.pps = p.pps;
    a.n_rg = 0;
    for (int s = 0; s < walk; s++) {
        a.seg[s].rg0 = a.n_rg;
        a.n_rg += ((a.seg[s].L.n_out + 31) / 32 + p.rpb * RS - 1) / (p.rpb * RS);
    }
    if (a.pair) a.nseg = 1;  // (the second matrix is read through its base)
    const unsigned grid = draco_gemmh_blocks(a.groups ? ntt : a.ksp * a.n_rg, a.groups ? a.n_rg : ntt);
    if (p.NSB == 4) pick<4>(a, f0, f1, grid, st);
    else pick<8>(a, f0, f1, grid, st);
    if (p.ksp > 1) {
        const size_t n = (size_t)a.T * a.seg[0].L.n_out;
        const bool v4 = n % 4 == 0 && (uintptr_t)a.seg[0].Y % 16 == 0 && (uintptr_t)a.part % 16 == 0;
        const size_t m = v4 ? n / 4 : n;
        const unsigned blocks = (unsigned)std::min<size_t>((m + 255) / 256, 4096);
        if (v4)
            hipLaunchKernelGGL(k_gemmr_sum4, dim3(blocks), dim3(256), 0, st, (const float4*)a.part, (float4*)a.seg[0].Y, m,
                               p.ksp);
        else
            hipLaunchKernelGGL(k_gemmr_sum, dim3(blocks), dim3(256), 0, st, a.part, a.seg[0].Y, m, p.ksp);
    }
    return 0;
}
