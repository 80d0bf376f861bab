// Gemma-2 text encoder (the stage before the denoiser: src/gemma_encoder.cpp,
// which runs llama.cpp's Gemma-2 graph in embeddings mode) on one MI355X,
// and its C ABI.
//
// Per layer, with T tokens (rows), hidden H, nh query heads and nkv kv heads
// of dimension d, FFN width F:
//   a16  = rmsnorm(x) * attn_norm                        gemma_norm_kernel
//   qkv  = a16 [Wq; Wk; Wv]^T                            one MFMA GEMM, fp32 out
//   q16, k16 = rope(q) * query_scale, rope(k); V^T       gemma_qkv_kernel
//   o16_h = softmax(mask(softcap(q16_h k16_kv(h)^T))) V_kv(h)
//                                                        gemma_attention_kernel, all sequences and heads;
//                                                        d other than 64, 128, 256: attention_by_products
//   x   += rmsnorm(o16 Wo^T) * post_attention_norm       split-K GEMM + gemma_norm_kernel
//   a16  = rmsnorm(x) * ffn_norm
//   g16  = gelu_tanh(a16 Wgate^T) * (a16 Wup^T)        one GEMM, gate / up rows
//                                                        interleaved, gated in its epilogue
//   x   += rmsnorm(g16 Wdown^T) * post_ffw_norm          split-K GEMM + gemma_norm_kernel
// Each post-norm residual add and the pre-norm after it are one launch.
// The layers of one encode run as one cached graph per sequence-length list.
// out = rmsnorm(x) * output_norm.  Activations are token-major; GEMM operands
// fp16 with fp32 accumulation; the residual stream, norms, softmax and RoPE
// in fp32.  RMSNorm weights are taken as stored in the GGUF (1 + w).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "../../include/sana_dit.h"
#include "gguf.h"
#include "hip_common.h"
#include "host_util.h"
#include "kernels.h"
#include "soft_math.h"

using sana::half_t;
using namespace sana_host;

#define SANA_LDS(p) ((__attribute__((address_space(3))) void *)(p))

namespace {

unsigned blocks_for(int64_t n, int per = 256) { return (unsigned)((n + per - 1) / per); }

// x32[t][c] = embed[token[t]][c] * scale (token ids checked on the host).
__global__ void gemma_embed_kernel(const int32_t * __restrict__ tok, const f16 * __restrict__ emb,
                                   float * __restrict__ x, int T, int H, float scale) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)T * H) return;
    const int t = (int)(i / H), c = (int)(i - (int64_t)t * H);
    x[i] = (float)emb[(int64_t)tok[t] * H + c] * scale;
}

// One workgroup of 256 threads per row of C (<= 1024 * NC4) channels:
// v = y / sqrt(mean(y^2) + eps) * w, y the fixed-order sum of PARTS split-K
// partials part_stride floats apart; the sum of squares is reduced over the
// four waves through LDS.  MODE 0: out16 = fp16(v); 1: x += v (post-norm
// residual, out32 = x); 2: out32 = v; 3: x += v as mode 1, then the next
// pre-norm of the new row, out16 = fp16(x / sqrt(mean(x^2) + eps) * w2), with
// the same summation order as a separate mode-0 launch on x.
// Every load of the row (partials, residual, weights) is requested before the
// first sum, without branches (columns past C read the last one and count as
// zero): one memory latency instead of four in a row (23 rows of 2304, four
// partials, modes 1 and 3: 7.4 -> 4.75 us; 738 rows, two partials: 9.87 -> 8.6).
template <int NC4, int MODE, int PARTS>
__global__ __launch_bounds__(256) void gemma_norm_kernel(const float * __restrict__ y, int64_t part_stride, int C,
                                                         const float * __restrict__ w, float eps,
                                                         f16 * __restrict__ out16, float * __restrict__ out32,
                                                         const float * __restrict__ w2) {
    __shared__ float wsum[8];
    const int row = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63;
    const int n4 = C >> 2;
    float4 v[NC4], u[PARTS][NC4], g[NC4], g2[MODE == 3 ? NC4 : 1], x[MODE == 1 || MODE == 3 ? NC4 : 1];
#pragma unroll
    for (int i = 0; i < NC4; ++i) {
        const int c4 = min(tid + 256 * i, n4 - 1);
#pragma unroll
        for (int z = 0; z < PARTS; ++z)
            u[z][i] = reinterpret_cast<const float4 *>(y + z * part_stride + (int64_t)row * C)[c4];
        if constexpr (MODE == 1 || MODE == 3) x[i] = reinterpret_cast<const float4 *>(out32 + (int64_t)row * C)[c4];
        g[i] = reinterpret_cast<const float4 *>(w)[c4];
        if constexpr (MODE == 3) g2[i] = reinterpret_cast<const float4 *>(w2)[c4];
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NC4; ++i) {
        v[i] = u[0][i];
#pragma unroll
        for (int z = 1; z < PARTS; ++z)
            v[i] = make_float4(v[i].x + u[z][i].x, v[i].y + u[z][i].y, v[i].z + u[z][i].z, v[i].w + u[z][i].w);
        if (tid + 256 * i >= n4) v[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        ss += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
    }
    ss = wave_sum(ss);
    if (lane == 0) wsum[tid >> 6] = ss;
    __syncthreads();
    const float tot = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
    const float inv = 1.0f / sqrtf(tot / (float)C + eps);
    float ss2 = 0.0f;
#pragma unroll
    for (int i = 0; i < NC4; ++i) {
        const int c4 = tid + 256 * i;
        if (c4 >= n4) continue;
        float o[4] = {v[i].x * inv * g[i].x, v[i].y * inv * g[i].y, v[i].z * inv * g[i].z, v[i].w * inv * g[i].w};
        if constexpr (MODE == 0) {
            f16x4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = (f16)o[e];
            *reinterpret_cast<f16x4 *>(out16 + (int64_t)row * C + 4 * c4) = h;
        } else {
            float4 * xr = reinterpret_cast<float4 *>(out32 + (int64_t)row * C) + c4;
            if constexpr (MODE == 1 || MODE == 3) {
                const float4 xn = make_float4(x[i].x + o[0], x[i].y + o[1], x[i].z + o[2], x[i].w + o[3]);
                *xr = xn;
                v[i] = xn;  // the new residual row, for mode 3's second norm
                ss2 += (xn.x * xn.x + xn.y * xn.y) + (xn.z * xn.z + xn.w * xn.w);
            } else {
                *xr = make_float4(o[0], o[1], o[2], o[3]);
            }
        }
    }
    if constexpr (MODE == 3) {
        ss2 = wave_sum(ss2);
        if (lane == 0) wsum[4 + (tid >> 6)] = ss2;
        __syncthreads();
        const float tot2 = (wsum[4] + wsum[5]) + (wsum[6] + wsum[7]);
        const float inv2 = 1.0f / sqrtf(tot2 / (float)C + eps);
#pragma unroll
        for (int i = 0; i < NC4; ++i) {
            const int c4 = tid + 256 * i;
            if (c4 >= n4) continue;
            f16x4 h;
            h[0] = (f16)(v[i].x * inv2 * g2[i].x);
            h[1] = (f16)(v[i].y * inv2 * g2[i].y);
            h[2] = (f16)(v[i].z * inv2 * g2[i].z);
            h[3] = (f16)(v[i].w * inv2 * g2[i].w);
            *reinterpret_cast<f16x4 *>(out16 + (int64_t)row * C + 4 * c4) = h;
        }
    }
}

// s_waitcnt with only the vector-memory (or only the LDS) counter constrained;
// the scheduler moves no memory operation across.
template <int N>
__device__ inline void wait_vmcnt() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
}
__device__ inline void wait_lgkmcnt0() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
    __builtin_amdgcn_sched_barrier(0);
}

// The sequences of one encode as the kernels see them (sana_gemma_encode_pair
// has two): rows [row0, row0 + T) of the token-major buffers.
struct GemmaSeqs {
    int n;
    int row0[2], T[2], Tp[2];
    int64_t vt_off[2];
};

// qkv32 [M][(nh + 2 nkv) d] -> q16 [M][nh d] = rope(q) * qscale, k16 [M][nkv d]
// = rope(k), vt16 [nkv][d][Tp] per sequence = V^T (tokens T..Tp-1 zero; `perm`:
// within each 16 tokens in the order 0-3, 8-11, 4-7, 12-15, which
// gemma_attention_kernel reads).  NeoX
// RoPE: pair (i, i + d/2) of a head rotated by t * theta^(-2i/d), t the position
// in its sequence.  The first rope_blocks workgroups take one (row, rotation
// pair) per thread for four heads (one powf and sincosf instead of one per
// head); the others transpose a 64 x 64 (token, channel) tile of V through
// LDS, so both sides move whole lines (read along the tokens, each lane touched
// a line of its own).  438 + 300 rows of 4096: 2 x 8.6 -> 6.5 us, one launch.
__global__ __launch_bounds__(256) void gemma_qkv_kernel(const float * __restrict__ qkv, GemmaSeqs sq, int M, int nh,
                                                        int nkv, int d, float theta, float qscale,
                                                        int rope_blocks, int perm, f16 * __restrict__ q16,
                                                        f16 * __restrict__ k16, f16 * __restrict__ vt16) {
    const int half = d / 2, ld = (nh + 2 * nkv) * d;
    const int tid = threadIdx.x;
    if ((int)blockIdx.x < rope_blocks) {
        // (row, group of 4 heads, pair)
        const int64_t i = (int64_t)blockIdx.x * 256 + tid;
        const int groups = (nh + nkv + 3) / 4;
        if (i >= (int64_t)M * groups * half) return;
        const int rg = (int)(i / half), p = (int)(i - (int64_t)rg * half);
        const int row = rg / groups, h0 = (rg - row * groups) * 4;
        const int t = row - (sq.n > 1 && row >= sq.row0[1] ? sq.row0[1] : 0);
        const float inv = powf(theta, -2.0f * (float)p / (float)d);
        float sn, cs;
        sincosf((float)t * inv, &sn, &cs);
        const float * src = qkv + (int64_t)row * ld + p;
        float a[4], b[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int head = min(h0 + e, nh + nkv - 1);
            a[e] = src[head * d];
            b[e] = src[head * d + half];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int head = h0 + e;  // heads 0..nh-1 are q, then k
            if (head >= nh + nkv) break;
            const float oa = a[e] * cs - b[e] * sn, ob = b[e] * cs + a[e] * sn;
            f16 * dst = head < nh ? q16 + ((int64_t)row * nh + head) * d : k16 + ((int64_t)row * nkv + head - nh) * d;
            const float sc = head < nh ? qscale : 1.0f;
            dst[p] = (f16)(oa * sc);
            dst[p + half] = (f16)(ob * sc);
        }
        return;
    }
    __shared__ f16 tile[64][72];
    const int ctiles = nkv * d / 64;
    int b = (int)blockIdx.x - rope_blocks, si = 0;
    if (b >= sq.Tp[0] / 64 * ctiles) {
        b -= sq.Tp[0] / 64 * ctiles;
        si = 1;
    }
    const int t0 = b / ctiles * 64, c0 = b % ctiles * 64, T = sq.T[si], Tp = sq.Tp[si];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int item = tid + 256 * k, t = item >> 4, c = (item & 15) * 4;
        const int tt = min(t0 + t, T - 1);
        const float4 v = *reinterpret_cast<const float4 *>(qkv + (int64_t)(sq.row0[si] + tt) * ld + (nh + nkv) * d +
                                                           c0 + c);
        const bool ok = t0 + t < T;
        const int u = perm ? (t & ~12) | (t & 4) << 1 | (t & 8) >> 1 : t;
        tile[c][u] = ok ? (f16)v.x : (f16)0.0f;
        tile[c + 1][u] = ok ? (f16)v.y : (f16)0.0f;
        tile[c + 2][u] = ok ? (f16)v.z : (f16)0.0f;
        tile[c + 3][u] = ok ? (f16)v.w : (f16)0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int item = tid + 256 * k, c = item >> 3, t = (item & 7) * 8;
        *reinterpret_cast<f16x8 *>(vt16 + sq.vt_off[si] + (int64_t)(c0 + c) * Tp + t0 + t) =
            *reinterpret_cast<const f16x8 *>(&tile[c][t]);
    }
}

// Causal soft-capped attention with a sliding window, one pass (online
// softmax), for all sequences and heads in one launch: head dims D of 64, 128
// and 256 (others take attention_by_products: the score product, the softmax
// and the P.V product, 56 us for 438 + 300 tokens of 8 heads of 256).
// s = cap * tanh(q.k / cap) over keys j <= t (and j > t - window when
// window > 0).
//
// A workgroup takes 32 queries of one head; its four waves take every fourth
// block of 32 keys each, with a running max, sum and output of their own, which
// are merged through LDS at the end: no barrier in the loop.  Each wave stages
// its K block (32 x D) and V^T block (D x 32) in LDS of its own by direct
// global -> LDS DMA, whole rows at a time (fragments read straight from global
// memory touch 32 lines per instruction: 30 us for 438 + 300 tokens against
// 23.9; 23 tokens 8.3 us).  The next block's K is requested when this one's
// fragments are in registers, its V^T when this one's products are done.  What
// bounds it is the chain of one wave's key blocks (up to 4 here): the
// accumulators, q and K take the registers of one wave per SIMD, so nothing
// hides a block's LDS reads and exponentials.  These keep the accuracy of expf and
// tanhf (soft_math.h) and of a division by the cap; while every |score| of a wave's
// block is below the cap, tanh is its polynomial alone.
// S^T = K Q^T (K rows as the first MFMA operand, q in registers), so a lane
// holds 16 keys of one query, exactly what it feeds back as the P^T operand of
// O^T = V^T P^T: the contraction takes key 16 s + 8 (e / 4) + 4 (lane / 32) + e %
// 4 as element e of step s, the order in which gemma_qkv_kernel stores V^T
// within each 16 keys, so nothing crosses lanes.
// LDS rows: 16-byte chunk c of K row r at slot c ^ (r & 15) (D 64: c ^ ((r >> 1)
// & 7)), of V^T row r at c ^ ((r >> 2) & 3): 16 consecutive rows at one chunk meet
// 16 distinct bank groups.
template <int D>
__global__ __launch_bounds__(256, 1) void gemma_attention_kernel(const f16 * __restrict__ q16,
                                                                 const f16 * __restrict__ k16,
                                                                 const f16 * __restrict__ vt16, GemmaSeqs sq,
                                                                 int nh, int nkv, float cap, int window,
                                                                 f16 * __restrict__ o16) {
    const float inv_cap = 1.0f / cap;
    constexpr int KS = D / 16, DT = D / 32;  // 16-deep steps over d, 32-row tiles of O^T
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    float4 * part = reinterpret_cast<float4 *>(lds);                      // [wave][DT][4][64]
    float * stat = reinterpret_cast<float *>(lds + 4 * DT * 4 * 64 * 16);  // [wave][max, sum][32]
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ql = lane & 31, hf = lane >> 5;
    const int h = blockIdx.y, kvh = h / (nh / nkv);
    const int nb0 = (sq.T[0] + 31) / 32;
    const int si = (int)blockIdx.x >= nb0 ? 1 : 0;
    // the longest rows first
    const int nb = (sq.T[si] + 31) / 32, qb = nb - 1 - ((int)blockIdx.x - (si ? nb0 : 0));
    const int T = sq.T[si], Tp = sq.Tp[si];
    const int64_t row0 = sq.row0[si];
    const int q0 = qb * 32, tq = min(q0 + ql, T - 1);
    const f16 * qr = q16 + ((row0 + tq) * nh + h) * D + 8 * hf;
    f16x8 qf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const f16x8 *>(qr + 16 * s);
    const f16 * vb = vt16 + sq.vt_off[si] + (int64_t)kvh * D * Tp;
    const f16 * kbase = k16 + (row0 * nkv + kvh) * D;
    const int kb_first = window > 0 ? max(0, q0 - window + 1) / 32 : 0, kb_last = min(q0 + 31, T - 1) / 32;
    constexpr int CPR = D / 8;  // 16-byte chunks of a K row
    unsigned char * kl = lds + w * (2 * D * 64), * vl = kl + D * 64;
    auto ksw = [](int r) { return D == 64 ? (r >> 1) & 7 : r & 15; };
    // (blocks past the last: the last again, never used)
    auto load_k = [&](int kb) {
        const int k0 = min(kb, kb_last) * 32;
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            const int n = i * 64 + lane, r = n / CPR, c = (n % CPR) ^ ksw(r);
            __builtin_amdgcn_global_load_lds(
                static_cast<const void *>(kbase + ((unsigned)min(k0 + r, T - 1) * (unsigned)(nkv * D) + c * 8)),
                SANA_LDS(kl + i * 1024), 16, 0, 0);
        }
    };
    auto load_v = [&](int kb) {
        const int k0 = min(kb, kb_last) * 32;
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            const int n = i * 64 + lane, r = n / 4, c = (n % 4) ^ ((r >> 2) & 3);
            __builtin_amdgcn_global_load_lds(static_cast<const void *>(vb + ((unsigned)(r * Tp) + k0 + c * 8)),
                                             SANA_LDS(vl + i * 1024), 16, 0, 0);
        }
    };
    load_k(kb_first + w);
    load_v(kb_first + w);
    f32x16 o[DT];
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[j][e] = 0.0f;
    float mx = -INFINITY, sum = 0.0f;
    for (int kb = kb_first + w; kb <= kb_last; kb += 4) {
        const int k0 = kb * 32;
        f16x8 kf[KS];
        wait_vmcnt<KS>();  // K has landed, V^T may be in flight
#pragma unroll
        for (int s = 0; s < KS; ++s)
            kf[s] = *reinterpret_cast<const f16x8 *>(kl + ql * (D * 2) + (((2 * s + hf) ^ ksw(ql)) << 4));
        wait_lgkmcnt0();
        load_k(kb + 4);
        f32x16 sc, sd;  // even and odd steps: two MFMA chains
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[e] = sd[e] = 0.0f;
#pragma unroll
        for (int s = 0; s < KS; s += 2) {
            sc = mfma_32x32x16(kf[s], qf[s], sc);
            sd = mfma_32x32x16(kf[s + 1], qf[s + 1], sd);
        }
        // lane: query q0 + ql, keys k0 + 8 (e / 4) + 4 hf + e % 4
        float um = 0.0f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            // score / cap to its last bit: a quotient by the rounded 1 / cap (far past
            // tanh's range cut off, so that no inf - inf arises) and its correction
            const float x = sc[e] + sd[e], u = __builtin_amdgcn_fmed3f(x * inv_cap, -64.0f, 64.0f);
            sc[e] = fmaf(fmaf(-u, cap, x), inv_cap, u);
            um = fmaxf(um, fabsf(sc[e]));
        }
        if (__any(um >= 1.0f)) {
#pragma unroll
            for (int e = 0; e < 16; ++e) sc[e] = cap * sana::soft_tanh(sc[e]);
        } else {  // the same without the other branch of tanh
#pragma unroll
            for (int e = 0; e < 16; ++e) sc[e] = cap * sana::soft_tanh_below_1(sc[e]);
        }
        float bm = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int j = k0 + 8 * (e >> 2) + 4 * hf + (e & 3), t = q0 + ql;
            const bool in = j <= t && j < T && (window <= 0 || j > t - window);
            sc[e] = in ? sc[e] : -INFINITY;
            bm = fmaxf(bm, sc[e]);
        }
        bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
        const float mn = fmaxf(mx, bm);
        // a query without a key so far keeps sums of zero
        const float m0 = mn == -INFINITY ? 0.0f : mn, f = expf(mx - m0);
        float bs = 0.0f;
        f16x8 pf[2];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float p = expf(sc[e] - m0);
            bs += p;
            pf[e >> 3][e & 7] = (f16)p;
        }
        bs += __shfl_xor(bs, 32, 64);
        sum = sum * f + bs;
        mx = mn;
        if (!__all(f == 1.0f)) {  // a new maximum somewhere
#pragma unroll
            for (int j = 0; j < DT; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[j][e] *= f;
        }
        wait_vmcnt<KS>();  // V^T has landed, the next K may be in flight
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                const int r = j * 32 + ql;
                const f16x8 v =
                    *reinterpret_cast<const f16x8 *>(vl + r * 64 + (((2 * s + hf) ^ ((r >> 2) & 3)) << 4));
                o[j] = mfma_32x32x16(v, pf[s], o[j]);
            }
        wait_lgkmcnt0();
        load_v(kb + 4);
    }
    wait_vmcnt<0>();
    const int64_t qrow = ((row0 + q0 + ql) * nh + h) * (int64_t)D;
    auto store4 = [&](int i, const float4 & a, float rs) {  // 4 consecutive d: 32 (i / 4) + 8 (i % 4) + 4 hf
        f16x4 hv;
        hv[0] = (f16)(a.x * rs);
        hv[1] = (f16)(a.y * rs);
        hv[2] = (f16)(a.z * rs);
        hv[3] = (f16)(a.w * rs);
        *reinterpret_cast<f16x4 *>(o16 + qrow + 32 * (i >> 2) + 8 * (i & 3) + 4 * hf) = hv;
    };
    // waves that had keys; alone, the first one stores
    const int nw = min(4, kb_last - kb_first + 1);
    if (nw == 1) {
        if (w > 0 || q0 + ql >= T) return;
        const float rs = 1.0f / sum;
#pragma unroll
        for (int i = 0; i < DT * 4; ++i) {
            const f32x16 & t = o[i >> 2];
            store4(i, make_float4(t[4 * (i & 3)], t[4 * (i & 3) + 1], t[4 * (i & 3) + 2], t[4 * (i & 3) + 3]), rs);
        }
        return;
    }
    // merge the waves: common max, scaled sums and outputs
    if (hf == 0) {
        stat[w * 64 + ql] = mx;
        stat[w * 64 + 32 + ql] = sum;
    }
    __syncthreads();  // also: every wave is done with its K and V^T
    float gm = -INFINITY, gs = 0.0f;
    for (int v = 0; v < nw; ++v) gm = fmaxf(gm, stat[v * 64 + ql]);
    for (int v = 0; v < nw; ++v) {
        const float m = stat[v * 64 + ql];
        gs += m == -INFINITY ? 0.0f : stat[v * 64 + 32 + ql] * expf(m - gm);
    }
    if (w < nw) {
        const float f = mx == -INFINITY ? 0.0f : expf(mx - gm);
#pragma unroll
        for (int j = 0; j < DT; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                part[((w * DT + j) * 4 + q) * 64 + lane] =
                    make_float4(o[j][4 * q] * f, o[j][4 * q + 1] * f, o[j][4 * q + 2] * f, o[j][4 * q + 3] * f);
    }
    __syncthreads();
    if (q0 + ql >= T) return;
    const float rs = 1.0f / gs;
    for (int i = w; i < DT * 4; i += 4) {
        float4 a = part[i * 64 + lane];
        for (int v = 1; v < nw; ++v) {
            const float4 b = part[(v * DT * 4 + i) * 64 + lane];
            a = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
        }
        store4(i, a, rs);
    }
}

template <int D>
hipError_t launch_gemma_attention(const f16 * q, const f16 * k, const f16 * vt, const GemmaSeqs & sq, int nh, int nkv,
                                  float cap, int window, f16 * o, hipStream_t s) {
    constexpr int lds = 4 * (D / 32) * 4 * 64 * 16 + 4 * 64 * 4;
    static const bool ok = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemma_attention_kernel<D>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
    (void)ok;
    int blocks = 0;
    for (int i = 0; i < sq.n; ++i) blocks += (sq.T[i] + 31) / 32;
    hipLaunchKernelGGL((gemma_attention_kernel<D>), dim3((unsigned)blocks, (unsigned)nh), dim3(256), lds, s, q, k, vt,
                       sq, nh, nkv, cap, window, o);
    return hipGetLastError();
}

// Rows (head, t) of S [nh][T][Tp]: s = cap * tanh(S / cap) over keys j <= t
// (and j > t - window when window > 0), softmax in fp32 -> P fp16 [nh][T][Tp]
// with zeros for the masked and padding keys.  One wave per row; lane keeps
// keys lane + 64 k (k < NJ, Tp <= 64 NJ) in registers, so each soft-capped
// score and its exponential are computed once.
template <int NJ>
__global__ __launch_bounds__(256) void gemma_softmax_kernel(const float * __restrict__ S, f16 * __restrict__ P,
                                                            int nh, int T, int Tp, float cap, int window) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= nh * T) return;
    const int t = row % T;
    const int j0 = window > 0 ? max(0, t - window + 1) : 0;
    const float * sr = S + (int64_t)row * Tp;
    f16 * pr = P + (int64_t)row * Tp;
    float v[NJ];
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < NJ; ++k) {
        const int j = lane + 64 * k;
        v[k] = (j >= j0 && j <= t) ? cap * tanhf(sr[j] / cap) : -INFINITY;
        mx = fmaxf(mx, v[k]);
    }
    mx = wave_max(mx);
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < NJ; ++k) {
        v[k] = v[k] == -INFINITY ? 0.0f : expf(v[k] - mx);
        sum += v[k];
    }
    sum = wave_sum(sum);
    const float rs = 1.0f / sum;
#pragma unroll
    for (int k = 0; k < NJ; ++k) {
        const int j = lane + 64 * k;
        if (j < Tp) pr[j] = (f16)(v[k] * rs);
    }
}

struct LayerDev {
    DevMem wqkv, wo, wgu, wdown;          // fp16, [out][in]; wgu rows gate_0, up_0, gate_1, up_1, ...
    DevMem n_attn, n_post_attn, n_ffn, n_post_ffw;  // fp32
};

}  // namespace

struct sana_gemma {
    sana_gemma_config cfg{};
    int64_t Dq = 0, Dkv = 0;
    std::vector<std::unique_ptr<LayerDev>> layers;
    DevMem emb16, out_norm;
    std::map<std::string, bool> loaded;
    std::vector<std::string> required;
    hipStream_t stream = nullptr;
    // workspace: rows of all sequences of one encode, and the per-sequence
    // attention buffers (V^T, scores, probabilities) back to back
    int64_t ws_M = 0, ws_vt = 0, ws_att = 0;
    DevMem tok, x32, y32, a16, qkv32, q16, k16, vt16, s32, p16, o16, g16, out32;
    // the encoder's kernels as one graph per sequence-length list (workspace
    // and weight pointers are baked in: dropped when either is reallocated)
    std::map<std::vector<int64_t>, hipGraphExec_t> graphs;
    ~sana_gemma() {
        for (auto & kv : graphs) (void)hipGraphExecDestroy(kv.second);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace {

void drop_graphs(sana_gemma * g) {
    for (auto & kv : g->graphs) (void)hipGraphExecDestroy(kv.second);
    g->graphs.clear();
}

void upload_bytes(DevMem & d, const void * src, size_t bytes) {
    d.ensure(bytes, false);
    copy_to_device(d.p, src, bytes, "upload gemma weight");
}

// fp32 -> fp16 operand rows; a value fp16 cannot hold fails with
// SANA_ERR_FORMAT naming the tensor.
void upload_f16_rows(DevMem & d, const float * src, size_t n, size_t total, size_t offset, const std::string & tensor) {
    if (!d.p) d.ensure(total * 2, false);
    std::vector<_Float16> h(n);
    for (size_t i = 0; i < n; ++i) h[i] = to_f16_checked(src[i], tensor, i);
    copy_to_device(static_cast<_Float16 *>(d.p) + offset, h.data(), n * 2, "upload gemma weight");
}

// Rows r of src ([n_rows][width] fp32) to rows 2 r + parity of d ([2 n_rows][width] fp16).
void upload_f16_rows_interleaved(DevMem & d, const float * src, size_t n_rows, size_t width, int parity,
                                 const std::string & tensor) {
    if (!d.p) d.ensure(2 * n_rows * width * 2, false);
    std::vector<_Float16> h(n_rows * width);
    for (size_t i = 0; i < h.size(); ++i) h[i] = to_f16_checked(src[i], tensor, i);
    hip_check(hipMemcpy2D(static_cast<_Float16 *>(d.p) + parity * width, 2 * width * 2, h.data(), width * 2,
                          width * 2, n_rows, hipMemcpyHostToDevice),
              "upload gemma weight");
    // a pageable copy may return before the data lands: h must outlive it, and
    // the encoder's non-blocking stream is not ordered after the null stream
    hip_check(hipStreamSynchronize(nullptr), "upload gemma weight");
}

void expect(const std::string & name, const int64_t * shape, int ndim, std::vector<int64_t> want) {
    bool ok = ndim == (int)want.size();
    for (int i = 0; ok && i < ndim; ++i) ok = shape[i] == want[i];
    if (!ok) {
        std::string got, exp;
        for (int i = 0; i < ndim; ++i) got += (i ? "," : "") + std::to_string(shape[i]);
        for (size_t i = 0; i < want.size(); ++i) exp += (i ? "," : "") + std::to_string(want[i]);
        throw_err(SANA_ERR_SHAPE, "gemma weight " + name + " has shape [" + got + "], expected [" + exp + "]");
    }
}

std::vector<std::string> required_names(const sana_gemma * g) {
    std::vector<std::string> r = {"token_embd.weight", "output_norm.weight"};
    for (int64_t l = 0; l < g->cfg.layers; ++l)
        for (const char * s : {"attn_norm", "attn_q", "attn_k", "attn_v", "attn_output", "post_attention_norm",
                               "ffn_norm", "ffn_gate", "ffn_up", "ffn_down", "post_ffw_norm"})
            r.push_back("blk." + std::to_string(l) + "." + s + ".weight");
    return r;
}

void set_weight(sana_gemma * g, const std::string & n, const float * d, const int64_t * sh, int nd) {
    drop_graphs(g);
    const sana_gemma_config & c = g->cfg;
    const int64_t H = c.hidden, F = c.ffn, Dq = g->Dq, Dkv = g->Dkv;
    if (n == "token_embd.weight") {
        expect(n, sh, nd, {c.vocab, H});
        upload_f16_rows(g->emb16, d, (size_t)(c.vocab * H), (size_t)(c.vocab * H), 0, n);
    } else if (n == "output_norm.weight") {
        expect(n, sh, nd, {H});
        upload_bytes(g->out_norm, d, (size_t)H * 4);
    } else {
        const std::string pre = "blk.";
        const size_t dot = n.find('.', pre.size());
        if (n.compare(0, pre.size(), pre) != 0 || dot == std::string::npos)
            throw_err(SANA_ERR_INVALID_ARGUMENT, "unknown gemma weight " + n);
        const int64_t l = std::stoll(n.substr(pre.size(), dot - pre.size()));
        if (l < 0 || l >= c.layers) throw_err(SANA_ERR_INVALID_ARGUMENT, "gemma layer index out of range: " + n);
        const std::string s = n.substr(dot + 1);
        LayerDev & L = *g->layers[l];
        const size_t qkv_rows = (size_t)(Dq + 2 * Dkv);
        if (s == "attn_q.weight") {
            expect(n, sh, nd, {Dq, H});
            upload_f16_rows(L.wqkv, d, (size_t)(Dq * H), qkv_rows * H, 0, n);
        } else if (s == "attn_k.weight") {
            expect(n, sh, nd, {Dkv, H});
            upload_f16_rows(L.wqkv, d, (size_t)(Dkv * H), qkv_rows * H, (size_t)(Dq * H), n);
        } else if (s == "attn_v.weight") {
            expect(n, sh, nd, {Dkv, H});
            upload_f16_rows(L.wqkv, d, (size_t)(Dkv * H), qkv_rows * H, (size_t)((Dq + Dkv) * H), n);
        } else if (s == "attn_output.weight") {
            expect(n, sh, nd, {H, Dq});
            upload_f16_rows(L.wo, d, (size_t)(H * Dq), (size_t)(H * Dq), 0, n);
        } else if (s == "ffn_gate.weight") {
            expect(n, sh, nd, {F, H});
            upload_f16_rows_interleaved(L.wgu, d, (size_t)F, (size_t)H, 0, n);
        } else if (s == "ffn_up.weight") {
            expect(n, sh, nd, {F, H});
            upload_f16_rows_interleaved(L.wgu, d, (size_t)F, (size_t)H, 1, n);
        } else if (s == "ffn_down.weight") {
            expect(n, sh, nd, {H, F});
            upload_f16_rows(L.wdown, d, (size_t)(H * F), (size_t)(H * F), 0, n);
        } else {
            DevMem * dst = s == "attn_norm.weight"             ? &L.n_attn
                           : s == "post_attention_norm.weight" ? &L.n_post_attn
                           : s == "ffn_norm.weight"            ? &L.n_ffn
                           : s == "post_ffw_norm.weight"       ? &L.n_post_ffw
                                                               : nullptr;
            if (!dst) throw_err(SANA_ERR_INVALID_ARGUMENT, "unknown gemma weight " + n);
            expect(n, sh, nd, {H});
            upload_bytes(*dst, d, (size_t)H * 4);
        }
    }
    g->loaded[n] = true;
}

void check_ready(const sana_gemma * g) {
    for (const std::string & n : g->required)
        if (!g->loaded.count(n)) throw_err(SANA_ERR_STATE, "gemma weight not set: " + n);
}

// One sequence of an encode: its rows [row0, row0 + T) of the token-major
// buffers and its offsets into the per-sequence attention buffers.
struct Seq {
    int64_t row0, T, Tp, vt_off, att_off;
};

std::vector<Seq> layout(const sana_gemma * g, const std::vector<int64_t> & lens) {
    std::vector<Seq> q;
    int64_t row = 0, vt = 0, att = 0;
    for (int64_t T : lens) {
        const int64_t Tp = round_up(T, 64);
        q.push_back({row, T, Tp, vt, att});
        row += T;
        vt += g->Dkv * Tp;
        att += g->cfg.heads * T * Tp;
    }
    return q;
}

bool one_pass_attention(const sana_gemma_config & c) {
    // (32-bit offsets into the K rows: up to 8192 tokens; a soft cap whose
    // reciprocal and quotients are normal numbers)
    return (c.head_dim == 64 || c.head_dim == 128 || c.head_dim == 256) && c.kv_heads * c.head_dim <= 65536 &&
           c.attn_softcap >= 1e-20f && c.attn_softcap <= 1e20f;
}

void ensure_workspace(sana_gemma * g, const std::vector<Seq> & q) {
    const Seq & e = q.back();
    const int64_t M = e.row0 + e.T, vt = e.vt_off + g->Dkv * e.Tp, att = e.att_off + g->cfg.heads * e.T * e.Tp;
    if (M <= g->ws_M && vt <= g->ws_vt && att <= g->ws_att) return;
    drop_graphs(g);
    const sana_gemma_config & c = g->cfg;
    const int64_t H = c.hidden;
    g->ws_M = std::max(g->ws_M, M);
    g->ws_vt = std::max(g->ws_vt, vt);
    g->ws_att = std::max(g->ws_att, att);
    const size_t R = (size_t)g->ws_M;
    g->tok.ensure(R * 4, false);
    g->x32.ensure(R * H * 4, false);
    g->y32.ensure(R * H * 4 * 4, false);  // up to four split-K partials
    g->a16.ensure(R * H * 2, false);
    g->qkv32.ensure(R * (g->Dq + 2 * g->Dkv) * 4, false);
    g->q16.ensure(R * g->Dq * 2, false);
    g->k16.ensure(R * g->Dkv * 2, false);
    g->vt16.ensure((size_t)g->ws_vt * 2, false);
    if (!one_pass_attention(c)) {
        g->s32.ensure((size_t)g->ws_att * 4, false);
        g->p16.ensure((size_t)g->ws_att * 2, false);
    }
    g->o16.ensure(R * g->Dq * 2, false);
    g->g16.ensure(R * c.ffn * 2, false);
    g->out32.ensure(R * H * 4, false);
}

void gemm(const half_t * A, int64_t lda, const half_t * W, int64_t ldw, int64_t M, int64_t N, int64_t K,
          half_t * o16, int64_t ldo16, float * o32, int64_t ldo32, hipStream_t s, int act = sana::kActNone,
          int runs = 1) {
    sana::GemmParams p;
    p.act = act;
    // a row's sums must not depend on the rows encoded with it
    p.order_rows = -1;
    p.k_runs = runs;
    p.A = A;
    p.lda = lda;
    p.W = W;
    p.ldw = ldw;
    p.M = (int)M;
    p.N = (int)N;
    p.K = (int)K;
    p.out16 = o16;
    p.ldo16 = ldo16;
    p.out32 = o32;
    p.ldo32 = ldo32;
    launch_check(sana::gemm(p, s), "gemma gemm");
}

// `batch` products in one launch: product z reads A + z * sa and W + (z / wdiv) * sw,
// writes o16 + z * so16 / o32 + z * so32.
void gemm_batched(const half_t * A, int64_t lda, int64_t sa, const half_t * W, int64_t ldw, int64_t sw, int wdiv,
                  int64_t M, int64_t N, int64_t K, half_t * o16, int64_t ldo16, int64_t so16, float * o32,
                  int64_t ldo32, int64_t so32, int batch, hipStream_t s, int runs = 1) {
    sana::GemmParams p;
    p.order_rows = -1;
    p.k_runs = runs;
    p.A = A;
    p.lda = lda;
    p.W = W;
    p.ldw = ldw;
    p.M = (int)M;
    p.N = (int)N;
    p.K = (int)K;
    p.out16 = o16;
    p.ldo16 = ldo16;
    p.out32 = o32;
    p.ldo32 = ldo32;
    p.batch = batch;
    p.batch_w_div = wdiv;
    p.batch_a = sa;
    p.batch_w = sw;
    p.batch_o16 = so16;
    p.batch_o32 = so32;
    launch_check(sana::gemm(p, s), "gemma batched gemm");
}

template <int MODE, int PARTS>
void norm_as(const float * y, int64_t M, int64_t C, const float * w, float eps, f16 * o16, float * o32,
             const float * w2, hipStream_t s) {
    const dim3 grid((unsigned)M), blk(256);
#define SANA_GEMMA_NORM(n4) \
    hipLaunchKernelGGL((gemma_norm_kernel<n4, MODE, PARTS>), grid, blk, 0, s, y, M * C, (int)C, w, eps, o16, o32, w2)
    if (C <= 1024) SANA_GEMMA_NORM(1);
    else if (C <= 2048) SANA_GEMMA_NORM(2);
    else if (C <= 3072) SANA_GEMMA_NORM(3);
    else SANA_GEMMA_NORM(4);
#undef SANA_GEMMA_NORM
    launch_check(hipGetLastError(), "gemma norm");
}

template <int MODE>
void norm(const sana_gemma * g, const float * y, int64_t M, const DevMem & w, half_t * o16, float * o32,
          hipStream_t s, int parts = 1, const DevMem * w2 = nullptr) {
    const int64_t C = g->cfg.hidden;
    f16 * h = reinterpret_cast<f16 *>(o16);
    const float * w2p = w2 ? w2->as<float>() : nullptr;
    if (parts == 1) norm_as<MODE, 1>(y, M, C, w.as<float>(), g->cfg.rms_eps, h, o32, w2p, s);
    else if (parts == 2) norm_as<MODE, 2>(y, M, C, w.as<float>(), g->cfg.rms_eps, h, o32, w2p, s);
    else norm_as<MODE, 4>(y, M, C, w.as<float>(), g->cfg.rms_eps, h, o32, w2p, s);
}

// Split-K factor of an M x H output with contraction K: the down and output
// projections have long K and few output tiles, so their K is cut into parts
// (multiples of 64) whose fp32 partials the following norm kernel sums in
// fixed order.  Four parts of at least 2048 (the 2B down projection: 66.6 ->
// 46.0 us for a 738-row prompt pair, 2 % slower for 438 + 300 rows encoded
// apart), else two of at least 512 (the output projection; 2B shapes encoded
// apart: 14.3 ms unsplit, 10.7 ms in two).  The factor depends on K only, so
// a row's sums do not depend on the other rows of the encode.
int split_k(int64_t K) {
    if (K % 256 == 0 && K / 4 >= 2048) return 4;
    return K % 128 == 0 && K / 2 >= 512 ? 2 : 1;
}

// Runs of k-tiles that a long contraction is summed in (GemmParams::k_runs):
// few-row encodes sum them side by side, where k in one sequence is a chain of
// K / 64 tile latencies.  Depends on K only, as split_k.
int k_runs(int64_t K) { return K >= 1024 ? 4 : 1; }

// Attention of other head dims: per sequence the scores of all heads as one
// batched product (head h uses K head h / grp), the softmax, and the batched
// P.V product.
void attention_by_products(sana_gemma * g, const std::vector<Seq> & seqs, int window, hipStream_t s) {
    const sana_gemma_config & c = g->cfg;
    const int64_t d = c.head_dim, nh = c.heads, Dq = g->Dq, Dkv = g->Dkv, grp = nh / c.kv_heads;
    for (const Seq & q : seqs) {
        const int64_t T = q.T, Tp = q.Tp;
        const half_t * q16 = g->q16.as<half_t>() + q.row0 * Dq;
        const half_t * k16 = g->k16.as<half_t>() + q.row0 * Dkv;
        const half_t * vt16 = g->vt16.as<half_t>() + q.vt_off;
        float * s32 = g->s32.as<float>() + q.att_off;
        half_t * p16 = g->p16.as<half_t>() + q.att_off;
        gemm_batched(q16, Dq, d, k16, Dkv, d, (int)grp, T, T, d, nullptr, 0, 0, s32, Tp, T * Tp, (int)nh, s);
        const dim3 sg((unsigned)((nh * T + 3) / 4)), sb(256);
        f16 * pp = reinterpret_cast<f16 *>(p16);
#define SANA_GEMMA_SOFTMAX(nj)                                                                                \
    hipLaunchKernelGGL((gemma_softmax_kernel<nj>), sg, sb, 0, s, s32, pp, (int)nh, (int)T, (int)Tp, c.attn_softcap, \
                       window)
        // Tp <= 64 NJ (token counts up to 8192: Tp <= 8192)
        if (Tp <= 512) SANA_GEMMA_SOFTMAX(8);
        else if (Tp <= 1024) SANA_GEMMA_SOFTMAX(16);
        else if (Tp <= 2048) SANA_GEMMA_SOFTMAX(32);
        else if (Tp <= 4096) SANA_GEMMA_SOFTMAX(64);
        else SANA_GEMMA_SOFTMAX(128);
#undef SANA_GEMMA_SOFTMAX
        launch_check(hipGetLastError(), "gemma softmax");
        gemm_batched(p16, Tp, T * Tp, vt16, Tp, d * Tp, (int)grp, T, d, Tp, g->o16.as<half_t>() + q.row0 * Dq, Dq, d,
                     nullptr, 0, 0, (int)nh, s);
    }
}

// decode_embeddings (src/gemma_encoder.cpp:95-152) on device token ids, for
// one or more independent sequences at once: their rows share every
// per-token kernel (norms, the projections, GeGLU), and RoPE and the one-pass
// attention take all sequences in one launch each, positions and keys kept to
// a row's own sequence (attention_by_products runs per sequence).  Each row's
// result is bit-identical to encoding its sequence alone: the per-row
// arithmetic and its order do not depend on the other rows.
void encode(sana_gemma * g, const std::vector<Seq> & seqs, hipStream_t s) {
    const sana_gemma_config & c = g->cfg;
    const int64_t H = c.hidden, F = c.ffn, d = c.head_dim, nh = c.heads, nkv = c.kv_heads;
    const int64_t Dq = g->Dq, Dkv = g->Dkv, Dqkv = Dq + 2 * Dkv;
    const int64_t M = seqs.back().row0 + seqs.back().T;
    hipLaunchKernelGGL(gemma_embed_kernel, dim3(blocks_for(M * H)), dim3(256), 0, s, g->tok.as<int32_t>(),
                       g->emb16.as<f16>(), g->x32.as<float>(), (int)M, (int)H, std::sqrt((float)H));
    launch_check(hipGetLastError(), "gemma embed");
    half_t * a16 = g->a16.as<half_t>();
    for (int64_t l = 0; l < c.layers; ++l) {
        LayerDev & L = *g->layers[l];
        // the pre-attention norm: layer 0 here, later layers in the previous
        // layer's last norm launch
        if (l == 0) norm<0>(g, g->x32.as<float>(), M, L.n_attn, a16, nullptr, s);
        gemm(a16, H, L.wqkv.as<half_t>(), H, M, Dqkv, H, nullptr, 0, g->qkv32.as<float>(), Dqkv, s, sana::kActNone,
             k_runs(H));
        const int window = (c.sliding_window > 0 && l % 2 == 0) ? (int)c.sliding_window : 0;
        GemmaSeqs sq{};
        sq.n = (int)seqs.size();
        int vblocks = 0;
        for (int i = 0; i < sq.n; ++i) {
            sq.row0[i] = (int)seqs[i].row0;
            sq.T[i] = (int)seqs[i].T;
            sq.Tp[i] = (int)seqs[i].Tp;
            sq.vt_off[i] = seqs[i].vt_off;
            vblocks += (int)(seqs[i].Tp / 64 * (nkv * d / 64));
        }
        const int rblocks = (int)blocks_for(M * ((nh + nkv + 3) / 4) * (d / 2));
        f16 * q16 = g->q16.as<f16>();
        f16 * k16 = g->k16.as<f16>();
        f16 * vt16 = g->vt16.as<f16>();
        f16 * o16 = g->o16.as<f16>();
        hipLaunchKernelGGL(gemma_qkv_kernel, dim3((unsigned)(rblocks + vblocks)), dim3(256), 0, s,
                           g->qkv32.as<float>(), sq, (int)M, (int)nh, (int)nkv, (int)d, c.rope_theta, c.query_scale,
                           rblocks, one_pass_attention(c) ? 1 : 0, q16, k16, vt16);
        launch_check(hipGetLastError(), "gemma qkv");
        hipError_t ae = hipSuccess;
        if (!one_pass_attention(c)) attention_by_products(g, seqs, window, s);
        else if (d == 64) ae = launch_gemma_attention<64>(q16, k16, vt16, sq, (int)nh, (int)nkv, c.attn_softcap, window, o16, s);
        else if (d == 128) ae = launch_gemma_attention<128>(q16, k16, vt16, sq, (int)nh, (int)nkv, c.attn_softcap, window, o16, s);
        else ae = launch_gemma_attention<256>(q16, k16, vt16, sq, (int)nh, (int)nkv, c.attn_softcap, window, o16, s);
        launch_check(ae, "gemma attention");
        const int so = split_k(Dq);
        gemm_batched(g->o16.as<half_t>(), Dq, Dq / so, L.wo.as<half_t>(), Dq, Dq / so, 1, M, H, Dq / so, nullptr, 0,
                     0, g->y32.as<float>(), H, M * H, so, s, k_runs(Dq / so));
        // x += post-attention norm of the projection, then the pre-FFN norm
        norm<3>(g, g->y32.as<float>(), M, L.n_post_attn, a16, g->x32.as<float>(), s, so, &L.n_ffn);
        gemm(a16, H, L.wgu.as<half_t>(), H, M, 2 * F, H, g->g16.as<half_t>(), F, nullptr, 0, s, sana::kActGeglu);
        const int sd = split_k(F);
        gemm_batched(g->g16.as<half_t>(), F, F / sd, L.wdown.as<half_t>(), F, F / sd, 1, M, H, F / sd, nullptr, 0, 0,
                     g->y32.as<float>(), H, M * H, sd, s, k_runs(F / sd));
        // x += post-FFN norm, then the next layer's pre-attention norm
        if (l + 1 < c.layers)
            norm<3>(g, g->y32.as<float>(), M, L.n_post_ffw, a16, g->x32.as<float>(), s, sd,
                    &g->layers[l + 1]->n_attn);
        else
            norm<1>(g, g->y32.as<float>(), M, L.n_post_ffw, nullptr, g->x32.as<float>(), s, sd);
    }
    norm<2>(g, g->x32.as<float>(), M, g->out_norm, nullptr, g->out32.as<float>(), s);
}

// Encodes the token sequences seqs[i] (host ids, lengths lens[i]) into
// hidden[i] (host, lens[i] x hidden floats) through the cached graph of
// this length list.
void run_encode(sana_gemma * g, const std::vector<const int32_t *> & toks, const std::vector<int64_t> & lens,
                const std::vector<float *> & hidden) {
    hip_check(hipSetDevice(g->cfg.device), "hipSetDevice");
    check_ready(g);
    int64_t total = 0;
    for (size_t i = 0; i < lens.size(); ++i) {
        const int64_t n = lens[i];
        if (n <= 0 || n > 8192) throw_err(SANA_ERR_INVALID_ARGUMENT, "gemma token count must be in [1, 8192]");
        for (int64_t j = 0; j < n; ++j)
            if (toks[i][j] < 0 || toks[i][j] >= g->cfg.vocab)
                throw_err(SANA_ERR_INVALID_ARGUMENT, "gemma token id out of range at position " + std::to_string(j) +
                                                         (lens.size() > 1 ? " of sequence " + std::to_string(i) : ""));
        total += n;
    }
    if (total > 16384) throw_err(SANA_ERR_INVALID_ARGUMENT, "gemma token count of one encode must be <= 16384");
    const std::vector<Seq> seqs = layout(g, lens);
    ensure_workspace(g, seqs);
    for (size_t i = 0; i < lens.size(); ++i)
        hip_check(hipMemcpyAsync(g->tok.as<int32_t>() + seqs[i].row0, toks[i], (size_t)lens[i] * 4,
                                 hipMemcpyHostToDevice, g->stream),
                  "upload tokens");
    auto it = g->graphs.find(lens);
    if (it == g->graphs.end()) {
        if (g->graphs.size() >= 8) drop_graphs(g);
        hipGraph_t graph = nullptr;
        hip_check(hipStreamBeginCapture(g->stream, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
        try {
            encode(g, seqs, g->stream);
        } catch (...) {
            (void)hipStreamEndCapture(g->stream, &graph);
            if (graph) (void)hipGraphDestroy(graph);
            throw;
        }
        hip_check(hipStreamEndCapture(g->stream, &graph), "hipStreamEndCapture");
        hipGraphExec_t exec = nullptr;
        const hipError_t r = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        hip_check(r, "hipGraphInstantiate");
        it = g->graphs.emplace(lens, exec).first;
    }
    hip_check(hipGraphLaunch(it->second, g->stream), "hipGraphLaunch");
    for (size_t i = 0; i < lens.size(); ++i)
        hip_check(hipMemcpyAsync(hidden[i], g->out32.as<float>() + seqs[i].row0 * g->cfg.hidden,
                                 (size_t)lens[i] * g->cfg.hidden * 4, hipMemcpyDeviceToHost, g->stream),
                  "download hidden");
    hip_check(hipStreamSynchronize(g->stream), "gemma encode");
}

void validate_config(const sana_gemma_config * c) {
    auto bad = [](const char * m) { throw_err(SANA_ERR_INVALID_ARGUMENT, m); };
    if (c->vocab <= 0 || c->layers <= 0 || c->heads <= 0 || c->kv_heads <= 0) bad("gemma sizes must be positive");
    if (c->heads % c->kv_heads) bad("gemma query heads must be a multiple of the kv heads");
    if (c->hidden <= 0 || c->hidden % 64 || c->hidden > 4096) bad("gemma hidden size must be a multiple of 64 up to 4096");
    if (c->head_dim <= 0 || c->head_dim % 64) bad("gemma head dim must be a multiple of 64");
    if (c->ffn <= 0 || c->ffn % 64) bad("gemma FFN width must be a multiple of 64");
    if (!(c->rms_eps > 0.0f) || !(c->rope_theta > 0.0f) || !(c->attn_softcap > 0.0f) || !(c->query_scale > 0.0f))
        bad("gemma eps, rope theta, soft-cap and query scale must be positive");
    if (c->sliding_window < 0) bad("gemma sliding window must be >= 0");
}

}  // namespace

extern "C" {

int sana_gemma_create(const sana_gemma_config * cfg, sana_gemma ** out) {
    if (!cfg || !out) return set_err(SANA_ERR_INVALID_ARGUMENT, "null argument");
    *out = nullptr;
    return guarded([&] {
        validate_config(cfg);
        int ndev = 0;
        hip_check(hipGetDeviceCount(&ndev), "hipGetDeviceCount");
        if (cfg->device < 0 || cfg->device >= ndev) throw_err(SANA_ERR_INVALID_ARGUMENT, "no such device");
        hip_check(hipSetDevice(cfg->device), "hipSetDevice");
        auto g = std::make_unique<sana_gemma>();
        g->cfg = *cfg;
        g->Dq = cfg->heads * cfg->head_dim;
        g->Dkv = cfg->kv_heads * cfg->head_dim;
        for (int64_t l = 0; l < cfg->layers; ++l) g->layers.push_back(std::make_unique<LayerDev>());
        g->required = required_names(g.get());
        hip_check(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking), "hipStreamCreate");
        *out = g.release();
    });
}

int sana_gemma_destroy(sana_gemma * g) {
    if (!g) return SANA_OK;
    (void)hipSetDevice(g->cfg.device);
    (void)hipDeviceSynchronize();
    delete g;
    return SANA_OK;
}

int sana_gemma_set_weight(sana_gemma * g, const char * name, const float * data, const int64_t * shape, int ndim) {
    if (!g || !name || !data || !shape) return set_err(SANA_ERR_INVALID_ARGUMENT, "null argument");
    return guarded([&] {
        hip_check(hipSetDevice(g->cfg.device), "hipSetDevice");
        set_weight(g, name, data, shape, ndim);
    });
}

int sana_gemma_check_weights(sana_gemma * g) {
    if (!g) return set_err(SANA_ERR_INVALID_ARGUMENT, "null argument");
    return guarded([&] { check_ready(g); });
}

int sana_gemma_load_gguf(sana_gemma * g, const char * path) {
    if (!g || !path) return set_err(SANA_ERR_INVALID_ARGUMENT, "null argument");
    return guarded([&] {
        using namespace sana::gguf;
        hip_check(hipSetDevice(g->cfg.device), "hipSetDevice");
        Index idx;
        try {
            idx = read_index(path);
        } catch (const std::exception & e) {
            throw_err(SANA_ERR_IO, e.what());
        }
        MappedFile f(path);
        std::map<std::string, const TensorInfo *> by;
        for (const auto & t : idx.tensors) by[t.name] = &t;
        std::vector<float> tmp;
        for (const std::string & n : g->required) {
            auto it = by.find(n);
            if (it == by.end()) throw_err(SANA_ERR_INVALID_ARGUMENT, "weight name not found in weight index: " + n);
            const TensorInfo & t = *it->second;
            size_t cnt = 1;
            for (int64_t dd : t.shape) cnt *= (size_t)dd;
            const float * src;
            if (t.type == kF32) {
                src = reinterpret_cast<const float *>(f.data() + t.offset);
            } else if (t.type == kF16 || t.type == kBF16) {
                tmp.resize(cnt);
                const uint16_t * h = reinterpret_cast<const uint16_t *>(f.data() + t.offset);
                for (size_t i = 0; i < cnt; ++i) {
                    if (t.type == kF16) {
                        _Float16 x;
                        std::memcpy(&x, h + i, 2);
                        tmp[i] = (float)x;
                    } else {
                        const uint32_t u = (uint32_t)h[i] << 16;
                        std::memcpy(&tmp[i], &u, 4);
                    }
                }
                src = tmp.data();
            } else {
                throw_err(SANA_ERR_FORMAT, "unsupported gguf tensor type for " + t.name);
            }
            set_weight(g, n, src, t.shape.data(), (int)t.shape.size());
        }
    });
}

int sana_gemma_encode(sana_gemma * g, const int32_t * tokens, int64_t n, float * hidden) {
    if (!g || !tokens || !hidden) return set_err(SANA_ERR_INVALID_ARGUMENT, "null argument");
    return guarded([&] { run_encode(g, {tokens}, {n}, {hidden}); });
}

int sana_gemma_encode_pair(sana_gemma * g, const int32_t * tokens_a, int64_t na, const int32_t * tokens_b,
                           int64_t nb, float * hidden_a, float * hidden_b) {
    if (!g || !tokens_a || !tokens_b || !hidden_a || !hidden_b)
        return set_err(SANA_ERR_INVALID_ARGUMENT, "null argument");
    return guarded([&] { run_encode(g, {tokens_a, tokens_b}, {na, nb}, {hidden_a, hidden_b}); });
}

}  // extern "C"
