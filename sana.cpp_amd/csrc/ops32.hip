// fp32 kernels behind the op-level API of the drop-in (the declarations of the
// reference's src/common_ops.h and src/transformer_ops.h): a batched GEMM on
// MFMA (v_mfma_f32_16x16x4f32: fp32 products, fp32 accumulation), row
// softmax with scale and key bias, SiLU / GELU-tanh, RMSNorm, k x k depthwise
// convolution, the GLU of the split channels, ReLU linear attention, and the
// head layout moves.  Every buffer is fp32 and in the reference's layouts.
// These serve API-level calls on host tensors; the DiT forward itself runs on
// the fused fp16-operand kernels of gemm.hip / attention.hip / ffn.hip / norm.hip.
#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>

#include "../../include/sana_dit.h"
#include "hip_common.h"

namespace sana {
void set_last_error(const std::string & m);
}

namespace {

using v4f = __attribute__((ext_vector_type(4))) float;

// v_mfma_f32_16x16x4f32: lane l holds row l % 16, k = l / 16 of either operand;
// D: column (second operand's row) l % 16, rows (first operand's) 4 (l / 16) + r.
__device__ inline v4f mfma_16x16x4(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct OpGemm {
    const float * A;
    const float * B;
    const float * bias;
    float * C;
    int64_t lda, ldb, ldc, sA, sB, sC;
    int M, N, K, bias_mode, accumulate;
};

constexpr int kTK = 32;

// C[z] (+)= A[z] . op(B[z]) (+ bias), A [M, K] row-major, op(B) = B [K, N] or
// (BT) B^T with B [N, K].  The bias is added after the products (bias_mode 1:
// per column, 2: per row).
//
// Bound: the fp32 matrix rate (256 flops per clock and CU), once the loads are
// out of its way: four waves (2 x 2) share a BM x BN tile; k-tiles of 32 go
// through registers (zero fill at the edges, any alignment) into one of two
// LDS buffers while the other is multiplied, one barrier per k-tile, and small
// tiles keep several workgroups on a CU.  k-contiguous operands lie in LDS as
// rows of 32 floats with 16-byte chunk c of row r at slot c ^ ((r >> 1) & 7)
// (conflict-free 16-byte reads of 16 rows); a lane's 16 bytes feed four MFMAs,
// so product j of a 16-deep step contracts k = 16 s + 4 g + j over the lane
// groups g.  B [K, N] lies as rows of BN + 4 floats, read four k rows apart
// (64 distinct banks).
//
// VA, VB: floats per global load of A and B, 4 where base, strides and extents
// are multiples of 4 elements (16 bytes), else 1.  VC, where the same holds for
// C's base and strides: the MFMA computes the transposed tile and a lane stores
// four consecutive columns of a row at once; else the tile itself, and a store
// covers 16 consecutive columns of four rows (16 products of 1023 x 1021 x 64 50.2 ->
// 34.8 us; as single elements of the transposed tile those were 16 bytes apart).
//
// Measured on MI355X: 2048 x 1152 x 1152 59 us (92 TFLOP/s); with the other
// kernels of this file the fp32 self-attention block (2 x 1024 tokens, four
// such products) went from 1326 to 284 us and the cross-attention block (2 x
// 256 tokens, 300 keys) from 785 to 136 us, against a 64 x 64 tile with
// single-buffered 16-deep k-tiles and two barriers each.
template <int BM, int BN, bool BT, int VA, int VB, bool VC>
__global__ __launch_bounds__(256) void gemm_f32_kernel(OpGemm p, int tiles_n) {
    constexpr int TM = BM / 32, TN = BN / 32;        // 16 x 16 tiles per wave
    constexpr int AF = BM * kTK / 256, BF = BN * kTK / 256;  // floats per thread and k-tile
    constexpr int A_SZ = BM * kTK, B_LD = BN + 4, B_SZ = BT ? BN * kTK : kTK * B_LD;
    __shared__ __attribute__((aligned(16))) float lds[2][A_SZ + B_SZ];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = (w >> 1) * (BM / 2), wn = (w & 1) * (BN / 2);
    const int lr = lane & 15, g = lane >> 4;
    // workgroup -> tile: each XCD (id % 8) takes a contiguous run of tiles
    // (column by column within a row panel), so A panels are shared in its L2
    const int nwg = gridDim.x, id = blockIdx.x, per = nwg / 8;
    const int order = id < per * 8 ? (id % 8) * per + id / 8 : id;
    const int m0 = (order / tiles_n) * BM, n0 = (order % tiles_n) * BN;
    const float * A = p.A + (int64_t)blockIdx.z * p.sA;
    const float * B = p.B + (int64_t)blockIdx.z * p.sB;
    float * C = p.C + (int64_t)blockIdx.z * p.sC;

    float ra[AF], rb[BF];
    // rows [r0, r0 + ROWS) x k [k0, k0 + 32) of a k-contiguous operand
    auto load_k = [&](const float * src, int64_t ld, int r0, int rows, int k0, float * reg, auto vec, auto count) {
        constexpr int V = decltype(vec)::value, CNT = decltype(count)::value / V;
#pragma unroll
        for (int i = 0; i < CNT; ++i) {
            const int item = tid + i * 256;
            const int r = r0 + item / (kTK / V), k = k0 + (item % (kTK / V)) * V;
            const bool ok = r < rows && k < p.K;
            const float * q = src + (int64_t)r * ld + k;
            if constexpr (V == 4) {
                const float4 v = ok ? *reinterpret_cast<const float4 *>(q) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                reg[4 * i] = v.x; reg[4 * i + 1] = v.y; reg[4 * i + 2] = v.z; reg[4 * i + 3] = v.w;
            } else {
                reg[i] = ok ? *q : 0.0f;
            }
        }
    };
    auto store_k = [&](float * dst, const float * reg, auto vec, auto count) {
        constexpr int V = decltype(vec)::value, CNT = decltype(count)::value / V;
#pragma unroll
        for (int i = 0; i < CNT; ++i) {
            const int item = tid + i * 256;
            const int r = item / (kTK / V), k = (item % (kTK / V)) * V;
            float * q = dst + r * kTK + (((k >> 2) ^ ((r >> 1) & 7)) << 2) + (k & 3);
            if constexpr (V == 4)
                *reinterpret_cast<float4 *>(q) = make_float4(reg[4 * i], reg[4 * i + 1], reg[4 * i + 2], reg[4 * i + 3]);
            else
                *q = reg[i];
        }
    };
    using AV = std::integral_constant<int, VA>;
    using BV = std::integral_constant<int, VB>;
    using AC = std::integral_constant<int, AF>;
    using BC = std::integral_constant<int, BF>;
    auto load = [&](int k0) {
        load_k(A, p.lda, m0, p.M, k0, ra, AV{}, AC{});
        if constexpr (BT) {
            load_k(B, p.ldb, n0, p.N, k0, rb, BV{}, BC{});
        } else {
#pragma unroll
            for (int i = 0; i < BF / VB; ++i) {
                const int item = tid + i * 256;
                const int k = k0 + item / (BN / VB), n = n0 + (item % (BN / VB)) * VB;
                const bool ok = k < p.K && n < p.N;
                const float * q = B + (int64_t)k * p.ldb + n;
                if constexpr (VB == 4) {
                    const float4 v = ok ? *reinterpret_cast<const float4 *>(q) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    rb[4 * i] = v.x; rb[4 * i + 1] = v.y; rb[4 * i + 2] = v.z; rb[4 * i + 3] = v.w;
                } else {
                    rb[i] = ok ? *q : 0.0f;
                }
            }
        }
    };
    auto store = [&](float * buf) {
        store_k(buf, ra, AV{}, AC{});
        if constexpr (BT) {
            store_k(buf + A_SZ, rb, BV{}, BC{});
        } else {
#pragma unroll
            for (int i = 0; i < BF / VB; ++i) {
                const int item = tid + i * 256;
                float * q = buf + A_SZ + (item / (BN / VB)) * B_LD + (item % (BN / VB)) * VB;
                if constexpr (VB == 4)
                    *reinterpret_cast<float4 *>(q) = make_float4(rb[4 * i], rb[4 * i + 1], rb[4 * i + 2], rb[4 * i + 3]);
                else
                    *q = rb[i];
            }
        }
    };

    // a lone 16 x 16 tile per wave alternates two accumulators (the MFMAs are a dependent chain otherwise)
    constexpr int NA = TM * TN == 1 ? 2 : 1;
    v4f acc[NA][TM][TN];
#pragma unroll
    for (int h = 0; h < NA; ++h)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[h][i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    // `steps` 16-deep steps of the k-tile in buf
    auto multiply = [&](const float * As, auto steps) {
        const float * Bs = As + A_SZ;
#pragma unroll
        for (int s = 0; s < decltype(steps)::value; ++s) {
            v4f a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int r = wm + i * 16 + lr;
                a[i] = *reinterpret_cast<const v4f *>(As + r * kTK + (((4 * s + g) ^ ((r >> 1) & 7)) << 2));
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int r = wn + j * 16 + lr;
                if constexpr (BT) {
                    b[j] = *reinterpret_cast<const v4f *>(Bs + r * kTK + (((4 * s + g) ^ ((r >> 1) & 7)) << 2));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) b[j][e] = Bs[(16 * s + 4 * g + e) * B_LD + r];
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        v4f & c = acc[e % NA][i][j];
                        c = VC ? mfma_16x16x4(b[j][e], a[i][e], c) : mfma_16x16x4(a[i][e], b[j][e], c);
                    }
        }
    };
    const int KT = (p.K + kTK - 1) / kTK;
    if (KT > 0) {
        load(0);
        store(lds[0]);
        __syncthreads();
    }
    for (int kt = 0; kt + 1 < KT; ++kt) {
        load((kt + 1) * kTK);
        __builtin_amdgcn_sched_barrier(0);  // (sunk between the MFMAs, the loads come up to 5 % later)
        multiply(lds[kt & 1], std::integral_constant<int, kTK / 16>{});
        store(lds[(kt + 1) & 1]);
        __syncthreads();
    }
    // the last k-tile; its upper half is skipped where it holds none of K
    if (KT > 0) {
        if (p.K - (KT - 1) * kTK > kTK / 2) multiply(lds[(KT - 1) & 1], std::integral_constant<int, kTK / 16>{});
        else multiply(lds[(KT - 1) & 1], std::integral_constant<int, kTK / 32>{});
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            v4f v = acc[0][i][j];
            if constexpr (NA == 2) v += acc[1][i][j];
            if constexpr (VC) {
                const int row = m0 + wm + i * 16 + lr, col = n0 + wn + j * 16 + 4 * g;
                if (row >= p.M || col >= p.N) continue;
                float * dst = C + (int64_t)row * p.ldc + col;
                const int nc = min(4, p.N - col);
                const float rbias = p.bias && p.bias_mode == 2 ? p.bias[row] : 0.0f;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (p.bias && e < nc) v[e] = (p.bias_mode == 2 ? rbias : p.bias[col + e]) + v[e];
                if (nc == 4) {
                    if (p.accumulate) v = *reinterpret_cast<const v4f *>(dst) + v;
                    *reinterpret_cast<v4f *>(dst) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (e < nc) dst[e] = p.accumulate ? dst[e] + v[e] : v[e];
                }
            } else {
                const int row = m0 + wm + i * 16 + 4 * g, col = n0 + wn + j * 16 + lr;
                if (col >= p.N) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (row + e >= p.M) continue;
                    if (p.bias) v[e] = p.bias[p.bias_mode == 2 ? row + e : col] + v[e];
                    float * dst = C + (int64_t)(row + e) * p.ldc + col;
                    *dst = p.accumulate ? *dst + v[e] : v[e];
                }
            }
        }
    }
}

template <int BM, int BN>
void launch_gemm_f32(const OpGemm & p, bool bt, bool va, bool vb, bool vc, unsigned batch, hipStream_t s) {
    const int tn = (p.N + BN - 1) / BN;
    const dim3 grid((unsigned)(((p.M + BM - 1) / BM) * tn), 1, batch), blk(256);
#define SANA_GEMM32(T, A, B)                                                                                  \
    do {                                                                                                      \
        if (vc) hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, T, A, B, true>), grid, blk, 0, s, p, tn);         \
        else hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, T, A, B, false>), grid, blk, 0, s, p, tn);           \
    } while (0)
    if (bt) {
        if (va && vb) SANA_GEMM32(true, 4, 4);
        else if (va) SANA_GEMM32(true, 4, 1);
        else if (vb) SANA_GEMM32(true, 1, 4);
        else SANA_GEMM32(true, 1, 1);
    } else {
        if (va && vb) SANA_GEMM32(false, 4, 4);
        else if (va) SANA_GEMM32(false, 4, 1);
        else if (vb) SANA_GEMM32(false, 1, 4);
        else SANA_GEMM32(false, 1, 1);
    }
#undef SANA_GEMM32
}

__global__ void unary_f32_kernel(const float * __restrict__ x, float * __restrict__ y, int64_t n, int op) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = x[i];
    y[i] = op == SANA_OP_SILU ? silu_f(v) : (op == SANA_OP_GELU_TANH ? gelu_tanh_f(v) : fmaxf(v, 0.0f));
}

// One wave per row: v = x * scale (+ bias[(row / bias_div) * cols + col]);
// y = exp(v - max) * (1 / sum exp(v - max)).  Rows of up to 64 NJ columns stay
// in registers, so x is read and y written once (three passes over y for
// longer rows, softmax_f32_long_kernel; same arithmetic in the same order).
template <int NJ>
__global__ __launch_bounds__(256) void softmax_f32_kernel(const float * x, float * y, int64_t rows, int cols,
                                                          float scale, const float * __restrict__ bias,
                                                          int64_t bias_div) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float * xr = x + row * cols;
    const float * br = bias ? bias + (row / bias_div) * cols : nullptr;
    float * yr = y + row * cols;
    float v[NJ], mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int c = lane + 64 * j;
        v[j] = c < cols ? xr[c] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int c = lane + 64 * j;
        if (c >= cols) continue;
        v[j] *= scale;
        if (br) v[j] += br[c];
        mx = fmaxf(mx, v[j]);
    }
    mx = wave_max(mx);
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        if (lane + 64 * j >= cols) continue;
        v[j] = expf(v[j] - mx);
        sum += v[j];
    }
    const float recip = 1.0f / wave_sum(sum);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int c = lane + 64 * j;
        if (c < cols) yr[c] = v[j] * recip;
    }
}

__global__ __launch_bounds__(256) void softmax_f32_long_kernel(const float * __restrict__ x, float * __restrict__ y,
                                                               int64_t rows, int cols, float scale,
                                                               const float * __restrict__ bias, int64_t bias_div) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float * xr = x + row * cols;
    const float * br = bias ? bias + (row / bias_div) * cols : nullptr;
    float * yr = y + row * cols;
    float mx = -INFINITY;
    for (int c = lane; c < cols; c += 64) {
        float v = xr[c] * scale;
        if (br) v += br[c];
        yr[c] = v;
        mx = fmaxf(mx, v);
    }
    mx = wave_max(mx);
    float sum = 0.0f;
    for (int c = lane; c < cols; c += 64) {
        const float e = expf(yr[c] - mx);
        yr[c] = e;
        sum += e;
    }
    const float recip = 1.0f / wave_sum(sum);
    for (int c = lane; c < cols; c += 64) yr[c] *= recip;
}

// One wave per row: y = x / sqrt(mean(x^2) + eps) (* w).
__global__ __launch_bounds__(256) void rms_norm_f32_kernel(const float * __restrict__ x, const float * __restrict__ w,
                                                           float * __restrict__ y, int64_t rows, int cols, float eps) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float * xr = x + row * cols;
    float * yr = y + row * cols;
    float ss = 0.0f;
    for (int c = lane; c < cols; c += 64) ss += xr[c] * xr[c];
    const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)cols + eps);
    for (int c = lane; c < cols; c += 64) {
        float v = xr[c] * inv;
        if (w) v *= w[c];
        yr[c] = v;
    }
}

// k x k depthwise convolution, zero padding k/2, NCHW; taps in (ky, kx)
// order, then the bias.  One thread per output element.
__global__ void dwconv_f32_kernel(const float * __restrict__ x, const float * __restrict__ w,
                                  const float * __restrict__ bias, float * __restrict__ y, int64_t planes, int C,
                                  int H, int W, int ks) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t HW = (int64_t)H * W;
    if (i >= planes * HW) return;
    const int64_t plane = i / HW;
    const int c = (int)(plane % C);
    const int yy = (int)((i % HW) / W), xx = (int)(i % W);
    const float * xp = x + plane * HW;
    const float * wc = w + (int64_t)c * ks * ks;
    const int pad = ks / 2;
    float sum = 0.0f;
    for (int ky = 0; ky < ks; ++ky) {
        const int iy = yy + ky - pad;
        if (iy < 0 || iy >= H) continue;
        for (int kx = 0; kx < ks; ++kx) {
            const int ix = xx + kx - pad;
            if (ix >= 0 && ix < W) sum += xp[(int64_t)iy * W + ix] * wc[ky * ks + kx];
        }
    }
    if (bias) sum += bias[c];
    y[i] = sum;
}

// y[b, c, s] = x[b, c, s] * silu(x[b, F + c, s]) for x [B, 2F, S].
__global__ void glu_f32_kernel(const float * __restrict__ x, float * __restrict__ y, int64_t B, int64_t F,
                               int64_t S) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B * F * S) return;
    const int64_t b = i / (F * S), r = i % (F * S);
    const float * xb = x + b * 2 * F * S;
    y[i] = xb[r] * silu_f(xb[F * S + r]);
}

// ReLU linear attention for head dims up to 80 (multiples of 4), on MFMA.
//
// State S[r][d] = sum_t v[t][r] relu(k[t][d]) and ksum[d] = sum_t relu(k[t][d])
// (row r = D) of one token chunk of one (batch, head).  Bound: the reads of k
// and v; one thread per state entry walking all tokens, which this replaces,
// was a serial chain of N dependent loads.  Operands go straight from global
// memory into MFMA fragments (four tokens per step: 64-byte runs), TT = 16-wide
// tiles per side; the four waves split the chunk's tokens (TS ways) and the
// state's row tiles (RS ways), and the TS partial states are added through LDS
// in a fixed order.  With several chunks each writes its partial to `dst` (the
// not yet written output serves as scratch) and linattn_reduce_f32_kernel adds
// them in chunk order.
template <int TT>
__global__ __launch_bounds__(256) void linattn_state_mfma_f32_kernel(const float * __restrict__ k,
                                                                     const float * __restrict__ v,
                                                                     float * __restrict__ dst, int N, int D,
                                                                     int chunk_tokens) {
    constexpr int RS = TT <= 2 ? 1 : 2, TS = 4 / RS, RT = (TT + RS - 1) / RS;
    constexpr int U = 4;  // token steps of 4 in flight
    __shared__ float part[(16 * TT + 1) * 16 * TT];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int lr = lane & 15, g = lane >> 4;
    const int rs = w % RS, ts = w / RS;
    const int64_t bh = blockIdx.y;
    const float * kb = k + bh * N * D;
    const float * vb = v + bh * N * D;
    const int c0 = blockIdx.x * chunk_tokens, c1 = min(N, c0 + chunk_tokens);
    const int per = ((c1 - c0 + TS - 1) / TS + 3) / 4 * 4;
    const int t0 = c0 + ts * per, t1 = min(c1, t0 + per);
    v4f acc[RT][TT];
    float ks[TT];
#pragma unroll
    for (int j = 0; j < TT; ++j) {
        ks[j] = 0.0f;
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (int t = t0; t < t1; t += 4 * U) {
        float vf[U][RT], kf[U][TT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int tt = t + 4 * u + g;
            const bool ok = tt < t1;
            const int64_t row = (int64_t)(ok ? tt : t0) * D;
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int r = (i * RS + rs) * 16 + lr;
                vf[u][i] = ok && r < D ? vb[row + r] : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < TT; ++j) {
                const int d = j * 16 + lr;
                kf[u][j] = ok && d < D ? fmaxf(kb[row + d], 0.0f) : 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < TT; ++j) {
                ks[j] += kf[u][j];
#pragma unroll
                for (int i = 0; i < RT; ++i) acc[i][j] = mfma_16x16x4(vf[u][i], kf[u][j], acc[i][j]);
            }
    }
#pragma unroll
    for (int j = 0; j < TT; ++j) {
        ks[j] += __shfl_xor(ks[j], 16, 64);
        ks[j] += __shfl_xor(ks[j], 32, 64);
    }
    // add the TS partials of each entry in token order: wave ts adds to what wave ts - 1 left
    float * out = dst + (bh * gridDim.x + blockIdx.x) * (int64_t)(D + 1) * D;
    for (int step = 0; step < TS; ++step) {
        if (step > 0) __syncthreads();
        if (ts != step) continue;
#pragma unroll
        for (int j = 0; j < TT; ++j) {
            const int d = j * 16 + lr;
            if (d >= D) continue;
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = (i * RS + rs) * 16 + 4 * g + e;
                    if (r >= D) continue;
                    const float x = step > 0 ? part[r * D + d] + acc[i][j][e] : acc[i][j][e];
                    if (step + 1 < TS) part[r * D + d] = x;
                    else out[r * D + d] = x;
                }
            if (g == 0 && rs == 0) {
                const float x = step > 0 ? part[D * D + d] + ks[j] : ks[j];
                if (step + 1 < TS) part[D * D + d] = x;
                else out[D * D + d] = x;
            }
        }
    }
}

// state[bh][e] = sum over chunks, in order, of the partial states.
__global__ __launch_bounds__(256) void linattn_reduce_f32_kernel(const float * __restrict__ part,
                                                                 float * __restrict__ state, int entries,
                                                                 int chunks) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t bh = blockIdx.y;
    if (e >= entries) return;
    const float * p = part + bh * chunks * (int64_t)entries + e;
    float s = p[0];
    for (int c = 1; c < chunks; ++c) s += p[(int64_t)c * entries];
    state[bh * entries + e] = s;
}

// out[t][r] = sum_d S[r][d] relu(q[t][d]) / (sum_d ksum[d] relu(q[t][d]) + 1e-15).
// One wave per 16-token group (GROUPS groups in a row), the state in registers
// as MFMA fragments; the denominator is the product's row D.  The MFMA
// computes the transposed tile, so a lane stores four consecutive channels of
// one token.  A group's q rows are read before any of its outputs is stored.
// KS = 16-deep steps over D, TR = 16-row tiles over D + 1.
template <int KS, int TR>
__global__ __launch_bounds__(256) void linattn_apply_mfma_f32_kernel(const float * q, const float * __restrict__ state,
                                                                     float * out, int Nq, int D, int groups) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int lr = lane & 15, g = lane >> 4;
    const int64_t bh = blockIdx.y;
    const float * S = state + bh * (int64_t)(D + 1) * D;
    v4f sf[KS][TR];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < TR; ++j) {
            const int r = j * 16 + lr, d = 16 * s + 4 * g;
            sf[s][j] = r <= D && d < D ? *reinterpret_cast<const v4f *>(S + r * D + d) : v4f{0.0f, 0.0f, 0.0f, 0.0f};
        }
    const int jd = D >> 4, gd = (D & 15) >> 2;  // tile and lane group of row D (D is a multiple of 4)
    for (int n = 0; n < groups; ++n) {
        const int t = ((blockIdx.x * 4 + w) * groups + n) * 16 + lr;
        if (t - lr >= Nq) break;
        const bool ok = t < Nq;
        const int64_t row = (bh * Nq + (ok ? t : Nq - 1)) * (int64_t)D;
        v4f qf[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int d = 16 * s + 4 * g;
            qf[s] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            if (d < D) qf[s] = *reinterpret_cast<const v4f *>(q + row + d);
        }
        v4f acc[TR];
#pragma unroll
        for (int j = 0; j < TR; ++j) acc[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = fmaxf(qf[s][e], 0.0f);
#pragma unroll
                for (int j = 0; j < TR; ++j) acc[j] = mfma_16x16x4(sf[s][j][e], x, acc[j]);
            }
        float den = 0.0f;
#pragma unroll
        for (int j = 0; j < TR; ++j)
            if (j == jd) den = acc[j][0];
        den = __shfl(den, gd * 16 + lr, 64) + 1e-15f;
        if (!ok) continue;
#pragma unroll
        for (int j = 0; j < TR; ++j) {
            const int r = j * 16 + 4 * g;
            if (r >= D) continue;
            v4f o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = acc[j][e] / den;
            *reinterpret_cast<v4f *>(out + row + r) = o;
        }
    }
}

bool ranges_overlap(const float * a, int64_t na, const float * b, int64_t nb) { return a < b + nb && b < a + na; }

// The MFMA pair (or triple, with chunked states) above; T = 16-wide tiles of D.
template <int T>
hipError_t launch_linattn_mfma(const float * q, const float * k, const float * v, float * out, int64_t BH, int64_t Nq,
                               int64_t Nk, int64_t D, float * state, hipStream_t s) {
    const int64_t entries = (D + 1) * D;
    // Chunks of at least 128 tokens, about two workgroups per CU over all
    // heads, as many as the output buffer holds partial states of; the partials
    // may not touch the inputs, so an output that shares memory with one keeps
    // a single chunk (1024 tokens, 72 heads of 32, 8 chunks:
    // state 12.0, reduction 4.9, apply 8.5 us).
    int64_t chunks = std::min((512 + BH - 1) / BH, Nk / 128);
    chunks = std::min(chunks, Nq * D / entries);
    if (ranges_overlap(out, BH * Nq * D, q, BH * Nq * D) || ranges_overlap(out, BH * Nq * D, k, BH * Nk * D) ||
        ranges_overlap(out, BH * Nq * D, v, BH * Nk * D))
        chunks = 1;
    chunks = std::max<int64_t>(chunks, 1);
    const int64_t per = std::max<int64_t>(((Nk + chunks - 1) / chunks + 15) / 16 * 16, 16);
    chunks = std::max<int64_t>((Nk + per - 1) / per, 1);
    hipLaunchKernelGGL((linattn_state_mfma_f32_kernel<T>), dim3((unsigned)chunks, (unsigned)BH), dim3(256), 0, s, k, v,
                       chunks > 1 ? out : state, (int)Nk, (int)D, (int)per);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (chunks > 1) {
        hipLaunchKernelGGL(linattn_reduce_f32_kernel, dim3((unsigned)((entries + 255) / 256), (unsigned)BH), dim3(256),
                           0, s, out, state, (int)entries, (int)chunks);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (Nq == 0) return hipSuccess;
    // groups of 16 tokens per wave: more while at least two workgroups per CU remain
    const int64_t g16 = (Nq + 15) / 16;
    int groups = 1;
    while (groups < 8 && (g16 + 8 * groups - 1) / (8 * groups) * BH >= 512) groups *= 2;
    const dim3 grid((unsigned)((g16 + 4 * groups - 1) / (4 * groups)), (unsigned)BH);
    if (D < 16 * T)  // row D falls into the last column tile's padding
        hipLaunchKernelGGL((linattn_apply_mfma_f32_kernel<T, T>), grid, dim3(256), 0, s, q, state, out, (int)Nq, (int)D,
                           groups);
    else
        hipLaunchKernelGGL((linattn_apply_mfma_f32_kernel<T, T + 1>), grid, dim3(256), 0, s, q, state, out, (int)Nq,
                           (int)D, groups);
    return hipGetLastError();
}

// Any head dim.
// Linear-attention state of one (batch*head, entry): entries r < D are
// S[r][d] = sum_t v[t][r] * relu(k[t][d]); entry r = D is ksum[d] =
// sum_t relu(k[t][d]).  Tokens are summed in order.  state: [BH][D + 1][D].
__global__ void linattn_state_f32_kernel(const float * __restrict__ k, const float * __restrict__ v,
                                         float * __restrict__ state, int N, int D) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t bh = blockIdx.y;
    if (e >= (D + 1) * D) return;
    const int r = e / D, d = e % D;
    const float * kb = k + bh * N * D;
    const float * vb = v + bh * N * D;
    float s = 0.0f;
    for (int t = 0; t < N; ++t) {
        const float kv = fmaxf(kb[(int64_t)t * D + d], 0.0f);
        s += (r < D ? vb[(int64_t)t * D + r] : 1.0f) * kv;
    }
    state[bh * (D + 1) * D + e] = s;
}

// out[t][r] = sum_d S[r][d] relu(q[t][d]) / (sum_d ksum[d] relu(q[t][d]) + 1e-15).
__global__ void linattn_apply_f32_kernel(const float * __restrict__ q, const float * __restrict__ state,
                                         float * __restrict__ out, int Nq, int D) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t bh = blockIdx.y;
    if (i >= (int64_t)Nq * D) return;
    const int t = (int)(i / D), r = (int)(i % D);
    const float * qr = q + (bh * Nq + t) * D;
    const float * S = state + bh * (D + 1) * D;
    float num = 0.0f, den = 0.0f;
    for (int d = 0; d < D; ++d) {
        const float qv = fmaxf(qr[d], 0.0f);
        num += S[r * D + d] * qv;
        den += S[D * D + d] * qv;
    }
    out[(bh * Nq + t) * D + r] = num / (den + 1e-15f);
}

// split = 1: y[b][h][t][d] = x[b][t][h*D + d]; split = 0: the inverse.  Head
// dims that are a multiple of 4, 16-byte aligned: 16 bytes per thread and
// 32-bit index arithmetic (a copy: bound by its 2 x 4 bytes per element; the
// element-wise 64-bit divisions below took most of the time): 9.4 MB in
// 5.7 us.
__global__ __launch_bounds__(256) void heads_f32_vec4_kernel(const float4 * __restrict__ x, float4 * __restrict__ y,
                                                             unsigned n4, unsigned N, unsigned H, unsigned D4,
                                                             int split) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    // i indexes the [B, N, H*D] layout
    const unsigned row = i / (H * D4), c = i - row * (H * D4);
    const unsigned h = c / D4, d = c - h * D4;
    const unsigned b = row / N, t = row - b * N;
    const unsigned j = ((b * H + h) * N + t) * D4 + d;
    if (split)
        y[j] = x[i];
    else
        y[i] = x[j];
}

// Any shape and alignment.
__global__ void heads_f32_kernel(const float * __restrict__ x, float * __restrict__ y, int64_t B, int64_t N,
                                 int64_t H, int64_t D, int split) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B * N * H * D) return;
    // i indexes the [B, N, H*D] layout
    const int64_t d = i % D, h = (i / D) % H, t = (i / (D * H)) % N, b = i / (D * H * N);
    const int64_t j = ((b * H + h) * N + t) * D + d;
    if (split)
        y[j] = x[i];
    else
        y[i] = x[j];
}

int fail(const char * what) {
    sana::set_last_error(what);
    return SANA_ERR_INVALID_ARGUMENT;
}

int launched(const char * what) {
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) return SANA_OK;
    sana::set_last_error(std::string(what) + ": " + hipGetErrorString(e));
    return SANA_ERR_HIP;
}

bool aligned16(const void * p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

unsigned blocks_for(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

extern "C" {

int sana_op_gemm_f32(const float * A, int64_t lda, int64_t strideA, const float * B, int64_t ldb, int64_t strideB,
                     int b_transposed, const float * bias, int bias_mode, float * C, int64_t ldc, int64_t strideC,
                     int64_t M, int64_t N, int64_t K, int64_t batch, int accumulate, void * stream) {
    if (!A || !B || !C) return fail("null operand");
    if (M <= 0 || N <= 0 || K < 0 || batch <= 0 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX ||
        batch > 65535)
        return fail("gemm dimensions out of range");
    if (lda < K || ldb < (b_transposed ? K : N) || ldc < N) return fail("gemm leading dimension too small");
    if (bias && bias_mode != 1 && bias_mode != 2) return fail("bias_mode must be 1 (per column) or 2 (per row)");
    if ((M + 63) / 64 > 65535) return fail("gemm M too large");
    OpGemm p{A, B, bias, C, lda, ldb, ldc, strideA, strideB, strideC, (int)M, (int)N, (int)K, bias_mode,
             accumulate ? 1 : 0};
    // 16-byte accesses: base, row stride, batch stride and the contiguous extent all multiples of 4 elements
    const bool va = aligned16(A) && lda % 4 == 0 && K % 4 == 0 && (batch == 1 || strideA % 4 == 0);
    const bool vb = aligned16(B) && ldb % 4 == 0 && (b_transposed ? K : N) % 4 == 0 && (batch == 1 || strideB % 4 == 0);
    const bool vc = aligned16(C) && ldc % 4 == 0 && (batch == 1 || strideC % 4 == 0);
    // The tile with the least modelled time: `fixed` + `round` per round of 256
    // workgroups, both measured at K = 1152 (us x 10; 64 to 4096 rows, 1152
    // columns, within 7 %).  Small tiles have the shorter k-step chain, large
    // ones fewer LDS reads per product.  32x32, 64x32 and 64x96, us: 400 rows 21.9,
    // 23.6, 42.1; 1024 rows 36.6, 39.6, 42.3; 2048 61.1, 60.2, 68.3; 4096 112, 102,
    // 96.6.  B [K, N] that is read float by float over few k-tiles waits for its
    // loads: there the middle tile, with twice the workgroups per CU, instead of
    // the largest (16 products of 1023 x 1021 x 40: 39.6 -> 35.7 us).
    struct {
        int64_t m, n, round, fixed;
    } const tiles[3] = {{64, 96, 266, 156}, {64, 32, 101, 115}, {32, 32, 59, 92}};
    int best = 0;
    int64_t best_cost = INT64_MAX;
    for (int i = 0; i < 3; ++i) {
        const int64_t t = ((M + tiles[i].m - 1) / tiles[i].m) * ((N + tiles[i].n - 1) / tiles[i].n) * batch;
        const int64_t cost = tiles[i].fixed + (t + 255) / 256 * tiles[i].round;
        if (i == 0 && !b_transposed && !vb && K <= 96) continue;
        if (t / batch < (1 << 24) && cost < best_cost) {  // a launch holds fewer than 2^32 threads per axis
            best = i;
            best_cost = cost;
        }
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool bt = b_transposed != 0;
    if (best == 0) launch_gemm_f32<64, 96>(p, bt, va, vb, vc, (unsigned)batch, s);
    else if (best == 1) launch_gemm_f32<64, 32>(p, bt, va, vb, vc, (unsigned)batch, s);
    else launch_gemm_f32<32, 32>(p, bt, va, vb, vc, (unsigned)batch, s);
    return launched("gemm_f32");
}

int sana_op_unary_f32(const float * x, float * y, int64_t n, int op, void * stream) {
    if (!x || !y || n < 0) return fail("bad unary arguments");
    if (op != SANA_OP_SILU && op != SANA_OP_GELU_TANH && op != SANA_OP_RELU) return fail("unknown unary op");
    if (n == 0) return SANA_OK;
    hipLaunchKernelGGL(unary_f32_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), x,
                       y, n, op);
    return launched("unary_f32");
}

int sana_op_softmax_f32(const float * x, float * y, int64_t rows, int64_t cols, float scale, const float * bias,
                        int64_t bias_div, void * stream) {
    if (!x || !y || rows < 0 || cols <= 0 || cols > INT32_MAX) return fail("bad softmax arguments");
    if (bias && bias_div <= 0) return fail("softmax bias_div must be positive");
    if (rows == 0) return SANA_OK;
    const dim3 grid(blocks_for(rows, 4)), blk(256);
    hipStream_t s = static_cast<hipStream_t>(stream);
#define SANA_SOFTMAX32(k) hipLaunchKernelGGL(k, grid, blk, 0, s, x, y, rows, (int)cols, scale, bias, bias_div)
    if (cols <= 128) SANA_SOFTMAX32(softmax_f32_kernel<2>);
    else if (cols <= 512) SANA_SOFTMAX32(softmax_f32_kernel<8>);
    else if (cols <= 2048) SANA_SOFTMAX32(softmax_f32_kernel<32>);
    else SANA_SOFTMAX32(softmax_f32_long_kernel);
#undef SANA_SOFTMAX32
    return launched("softmax_f32");
}

int sana_op_rms_norm_f32(const float * x, const float * w, float * y, int64_t rows, int64_t cols, float eps,
                         void * stream) {
    if (!x || !y || rows < 0 || cols <= 0 || cols > INT32_MAX) return fail("bad rms_norm arguments");
    if (rows == 0) return SANA_OK;
    hipLaunchKernelGGL(rms_norm_f32_kernel, dim3(blocks_for(rows, 4)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), x, w, y, rows, (int)cols, eps);
    return launched("rms_norm_f32");
}

int sana_op_dwconv_f32(const float * x, const float * w, const float * bias, float * y, int64_t B, int64_t C,
                       int64_t H, int64_t W, int64_t ksize, void * stream) {
    if (!x || !w || !y || B < 0 || C <= 0 || H <= 0 || W <= 0 || (ksize != 3 && ksize != 5) || C > INT32_MAX ||
        H > INT32_MAX || W > INT32_MAX)
        return fail("bad depthwise conv arguments");
    const int64_t n = B * C * H * W;
    if (n == 0) return SANA_OK;
    hipLaunchKernelGGL(dwconv_f32_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), x,
                       w, bias, y, B * C, (int)C, (int)H, (int)W, (int)ksize);
    return launched("dwconv_f32");
}

int sana_op_glu_f32(const float * x, float * y, int64_t B, int64_t F, int64_t S, void * stream) {
    if (!x || !y || B < 0 || F < 0 || S < 0) return fail("bad glu arguments");
    const int64_t n = B * F * S;
    if (n == 0) return SANA_OK;
    hipLaunchKernelGGL(glu_f32_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), x, y,
                       B, F, S);
    return launched("glu_f32");
}

int sana_op_linear_attention_f32(const float * q, const float * k, const float * v, float * out, int64_t BH,
                                 int64_t Nq, int64_t Nk, int64_t D, float * state, void * stream) {
    if (!q || !k || !v || !out || !state || BH < 0 || Nq < 0 || Nk < 0 || D <= 0 || D > 4096 || BH > 65535 ||
        Nq > INT32_MAX || Nk > INT32_MAX)
        return fail("bad linear attention arguments");
    if (BH == 0) return SANA_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // (up to four tokens the kernels below, one thread per entry, are the shorter
    // chain: 36 heads of 32 6.9 us against 8.4)
    if (D <= 80 && D % 4 == 0 && (Nq > 4 || Nk > 4) && aligned16(q) && aligned16(out) && aligned16(state)) {
        hipError_t e;
        switch ((D + 15) / 16) {
            case 1: e = launch_linattn_mfma<1>(q, k, v, out, BH, Nq, Nk, D, state, s); break;
            case 2: e = launch_linattn_mfma<2>(q, k, v, out, BH, Nq, Nk, D, state, s); break;
            case 3: e = launch_linattn_mfma<3>(q, k, v, out, BH, Nq, Nk, D, state, s); break;
            case 4: e = launch_linattn_mfma<4>(q, k, v, out, BH, Nq, Nk, D, state, s); break;
            default: e = launch_linattn_mfma<5>(q, k, v, out, BH, Nq, Nk, D, state, s); break;
        }
        if (e == hipSuccess) return SANA_OK;
        sana::set_last_error(std::string("linattn_f32: ") + hipGetErrorString(e));
        return SANA_ERR_HIP;
    }
    hipLaunchKernelGGL(linattn_state_f32_kernel, dim3(blocks_for((D + 1) * D, 256), (unsigned)BH), dim3(256), 0, s,
                       k, v, state, (int)Nk, (int)D);
    int rc = launched("linattn_state_f32");
    if (rc != SANA_OK || Nq == 0) return rc;
    hipLaunchKernelGGL(linattn_apply_f32_kernel, dim3(blocks_for(Nq * D, 256), (unsigned)BH), dim3(256), 0, s, q,
                       state, out, (int)Nq, (int)D);
    return launched("linattn_apply_f32");
}

int sana_op_heads_f32(const float * x, float * y, int64_t B, int64_t N, int64_t H, int64_t D, int split,
                      void * stream) {
    if (!x || !y || B < 0 || N < 0 || H <= 0 || D < 0) return fail("bad head layout arguments");
    const int64_t n = B * N * H * D;
    if (n == 0) return SANA_OK;
    if (D % 4 == 0 && n / 4 < ((int64_t)1 << 31) && N < ((int64_t)1 << 31) && aligned16(x) && aligned16(y)) {
        hipLaunchKernelGGL(heads_f32_vec4_kernel, dim3(blocks_for(n / 4, 256)), dim3(256), 0,
                           static_cast<hipStream_t>(stream), reinterpret_cast<const float4 *>(x),
                           reinterpret_cast<float4 *>(y), (unsigned)(n / 4), (unsigned)N, (unsigned)H,
                           (unsigned)(D / 4), split ? 1 : 0);
        return launched("heads_f32");
    }
    hipLaunchKernelGGL(heads_f32_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), x,
                       y, B, N, H, D, split ? 1 : 0);
    return launched("heads_f32");
}

}  // extern "C"
