// K1: MFMA GEMM for every dense projection of the DiT (QKV, attention output,
// cross-attention q/k/v/out, Mix-FFN inverted/point 1x1 convs, caption MLP).
//
// C[m, n] = sum_k A[m, k] * W[n, k], fp16 operands, fp32 accumulation on
// v_mfma_f32_32x32x16_f16.  A (activations, token-major) and W (weights,
// PyTorch [out, in] order) are both K-contiguous, so each MFMA lane's operand
// (8 consecutive k of one row) is a single 16-byte LDS read.
//
// Data movement (gfx950):
//   * HBM/L2 -> LDS with global_load_lds_dwordx4: each wave instruction moves
//     8 rows x 64 k (1 KB) straight into LDS without passing through VGPRs.
//   * A STAGES-deep ring of LDS k-tiles (BK = 64): when tile kt is done its
//     stage is refilled with tile kt+STAGES, so each load has STAGES-1 tiles
//     of MFMA work to land.  Completion is tracked with an explicit vmcnt
//     wait (the loads of later tiles stay outstanding) and one s_barrier per
//     k-tile, placed after the tile's last MFMAs are issued (schedule 2: before
//     the last quarter of them, which then covers the barrier and the next
//     tile's first LDS reads).
//   * LDS rows are 128 bytes; 16-byte chunk c of row r is stored in slot
//     c ^ ((r >> 1) & 7).  The DMA writes lane l to slot l & 7 of row l >> 3 of
//     its 8-row block, so lane l fetches the chunk that maps there.  gfx950's
//     LDS serves a 16-byte read 16 lanes (256 bytes, all 64 banks) per cycle;
//     an MFMA operand read of 16 consecutive rows at one chunk then hits 16
//     distinct 16-byte bank groups (row parity picks the half of the 256-byte
//     window, (r >> 1) & 7 the group within it): no bank conflicts.  The
//     slot c ^ (r & 7) conflicts two ways (rows r and r + 8 share a group).
//   * Epilogue staged through LDS: the MFMA computes the transposed tile, so
//     each lane holds runs of 4 consecutive columns of one row and writes
//     them to LDS as one 16-byte (fp32) or 8-byte (fp16) store; then every
//     thread moves 8 consecutive columns with 16-byte global accesses.
//     Outputs that are fp16 only are rounded in registers and staged as fp16
//     (one pass for every tile shape).
//
// The workgroup -> tile map is XCD-aware: gfx950 deals workgroups round-robin
// to 8 XCDs (each with its own L2), so workgroup id i goes to position
// (i % 8) * (T / 8) + i / 8 of a grouped tile order (8 row panels at a time,
// column by column): the tiles one XCD runs concurrently form a compact 2-D
// block whose A and W panels are shared through its L2.
//
// Fused epilogues (reference ops they replace):
//   store   : bias (+SiLU | +GELU-tanh), fp16 and/or fp32 out
//             (linear_3d_lastdim src/common_ops.cpp:177-209, silu src/tensor.cpp:551-555,
//              gelu_tanh src/transformer_ops.cpp:15-18)
//   residual: x += gate * (acc + bias), optional fp16 copy of the new x
//             (mul_inplace_broadcast_lastdim + add_inplace, src/tensor.cpp:101-160)
//   V^T     : transposed per-batch store of the cross-attention values.
#include <string>

#include "hip_common.h"
#include "kernels.h"

#define SANA_LDS(p) ((__attribute__((address_space(3))) void *)(p))

namespace sana {
namespace gemm_detail {

constexpr int kBK = 64;

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding:
// vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] << 14).
template <int N>
SANA_DEV void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// s_waitcnt lgkmcnt(0): every LDS read of this wave has returned.
SANA_DEV void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14)); }

// KG: k-groups of WM x WN waves.  Group g sums the g-th of KG runs of
// consecutive k-tiles through its own part of every stage, and the groups'
// sums are added in group order before the epilogue.
template <int BM, int BN, int WM, int WN, int STAGES, int KG = 1>
struct Cfg {
    static constexpr int GW = WM * WN;  // waves per k-group
    static constexpr int NW = GW * KG;
    static constexpr int NT = 64 * NW;
    static constexpr int WTM = BM / WM, WTN = BN / WN;
    static constexpr int TM = WTM / 32, TN = WTN / 32;
    static constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128;
    static constexpr int SUB_BYTES = A_BYTES + B_BYTES;  // one k-tile
    static constexpr int STAGE_BYTES = KG * SUB_BYTES;
    static constexpr int A_LOADS = BM / 8 / GW, B_LOADS = BN / 8 / GW;  // wave instructions per stage
    static constexpr int LOADS = A_LOADS + B_LOADS;
    static constexpr int CPAD = 4;                                      // fp32 epilogue row padding
    // The fp32 epilogue tile is staged in LDS: whole when it fits in the operand
    // ring or in 80 KB (two workgroups per CU), else one wave row (WTM rows) per pass.
    static constexpr int RING_BYTES = STAGES * STAGE_BYTES;
    static constexpr int EPI_ROWS =
        (BM * (BN + CPAD) * 4 <= (RING_BYTES > 80 * 1024 ? RING_BYTES : 80 * 1024)) ? BM : WTM;
    static constexpr int EPI_BYTES = EPI_ROWS * (BN + CPAD) * 4;
    static constexpr int EPI16_BYTES = BM * (BN + 8) * 2;  // the fp16 epilogue's tile, always whole
    static constexpr int EPI_MAX = EPI_BYTES > EPI16_BYTES ? EPI_BYTES : EPI16_BYTES;
    static constexpr int LDS_BYTES = RING_BYTES > EPI_MAX ? RING_BYTES : EPI_MAX;
    static constexpr int PART_BYTES = GW * TM * TN * 4096;  // one k-group's sums
    static_assert((KG - 1) * PART_BYTES <= LDS_BYTES, "k-group partial sums");
    static_assert(BM % (8 * GW) == 0 && BN % (8 * GW) == 0, "tile rows must split into 8-row wave loads");
    static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile must be a multiple of 32x32");
    static_assert(LOADS * STAGES < 64, "vmcnt range");
    static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

// Wait until at most `keep` stages (0 <= keep < STAGES) of this wave's loads are outstanding.
template <int LOADS, int STAGES>
SANA_DEV void wait_stages(int keep) {
    if constexpr (STAGES <= 1) {
        wait_vmcnt<0>();
    } else {
        if (keep >= STAGES - 1) wait_vmcnt<(STAGES - 1) * LOADS>();
        else wait_stages<LOADS, STAGES - 1>(keep);
    }
}

// CONV: 0 plain A rows; 1 implicit 3x3 conv over a zero-bordered NHWC input;
// 2 the same over the nearest-2x upsample of the input (GemmParams::conv).
template <int BM, int BN, int WM, int WN, int STAGES, int MODE, int SCHED, int ACT, int CONV = 0, int KG = 1,
          bool FOLD = false>
__global__ __launch_bounds__(64 * WM * WN * KG) void gemm_kernel(GemmParams p_in) {
    using G = Cfg<BM, BN, WM, WN, STAGES, KG>;
    static_assert((KG == 1 || SCHED == 1) && (!FOLD || (KG == 1 && SCHED != 2)), "schedule");
    // product blockIdx.y of a batched launch (plain stores only)
    GemmParams p = p_in;
    if constexpr (MODE == kGemmStore && CONV == 0) {
        const int z = blockIdx.y;
        p.A += z * p.batch_a;
        p.W += (z / p.batch_w_div) * p.batch_w;
        if (p.out16) p.out16 += z * p.batch_o16;
        if (p.out32) p.out32 += z * p.batch_o32;
    }
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    // Workgroup -> tile: XCD x (= id % 8) takes a contiguous range of tiles in
    // a grouped order (kGroup row panels, column by column), so the tiles an
    // XCD runs together form a compact block whose A and W panels stay in its L2.
    const int ntn = (p.N + BN - 1) / BN;
    const int ntm = (p.M + BM - 1) / BM;
    const int nwg = ntn * ntm;
    const int id = blockIdx.x;
    const int per = nwg / 8;
    const int order = (id < per * 8) ? (id % 8) * per + id / 8 : id;
    constexpr int kGroup = 8;
    const int gsz = kGroup * ntn;
    const int grp = order / gsz, gm = min(kGroup, ntm - grp * kGroup);
    const int within = order - grp * gsz;
    const int tm = grp * kGroup + within % gm, tn = within / gm;
    const int m0 = tm * BM, n0 = tn * BN;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wid = tid >> 6;
    const int kg = KG == 1 ? 0 : wid / G::GW, wi = KG == 1 ? wid : wid % G::GW;  // k-group, wave within it
    const int wm = wi / WN, wn = wi % WN;
    const int KT = p.K / kBK;
    const int NT_K = (KT + KG - 1) / KG;  // k-tiles per group

    // Per-lane global source of each wave load (row clamped into range; the
    // rows past M / N are computed but never stored).
    const int lrow = lane >> 3;
    // chunk fetched by this lane for 8-row block blk (rows 8 blk .. 8 blk + 7)
    auto lchunk = [&](int blk) { return (lane & 7) ^ ((4 * (blk & 1) + (lrow >> 1)) & 7); };
    const f16 * asrc[G::A_LOADS];
    const f16 * bsrc[G::B_LOADS];
    // conv: output pixel (image, y, x) of each A load row; asrc is the image's bordered input base
    int cy[CONV ? G::A_LOADS : 1], cx[CONV ? G::A_LOADS : 1];
#pragma unroll
    for (int i = 0; i < G::A_LOADS; ++i) {
        const int r = (wi + i * G::GW) * 8 + lrow;
        const int m = min(m0 + r, p.M - 1);
        if constexpr (CONV == 0) {
            asrc[i] = reinterpret_cast<const f16 *>(p.A) + (int64_t)m * p.lda + lchunk(wi + i * G::GW) * 8;
        } else {
            const int hw = p.conv_h * p.conv_w;
            const int img = m / hw, rem = m - img * hw;
            cy[i] = rem / p.conv_w;
            cx[i] = rem - cy[i] * p.conv_w;
            const int ih = CONV == 2 ? p.conv_h / 2 : p.conv_h, iw = CONV == 2 ? p.conv_w / 2 : p.conv_w;
            asrc[i] = reinterpret_cast<const f16 *>(p.A) + (int64_t)img * (ih + 2) * (iw + 2) * p.lda +
                      lchunk(wi + i * G::GW) * 8;
        }
    }
#pragma unroll
    for (int i = 0; i < G::B_LOADS; ++i) {
        const int r = (wi + i * G::GW) * 8 + lrow;
        bsrc[i] = reinterpret_cast<const f16 *>(p.W) + (int64_t)min(n0 + r, p.N - 1) * p.ldw + lchunk(wi + i * G::GW) * 8;
    }
    auto issue = [&](int kt, int st) {
        unsigned char * base = smem + st * G::STAGE_BYTES + kg * G::SUB_BYTES;
        // this group's k-tile (past the last one: the last again, never multiplied)
        if constexpr (KG > 1) kt = min(kg * NT_K + kt, KT - 1);
        const int k0 = kt * kBK;
        if constexpr (CONV == 0) {
#pragma unroll
            for (int i = 0; i < G::A_LOADS; ++i)
                __builtin_amdgcn_global_load_lds(static_cast<const void *>(asrc[i] + k0),
                                                 SANA_LDS(base + (wi + i * G::GW) * 1024), 16, 0, 0);
        } else {
            // k-tile kt = (tap, 64-channel chunk): one 128-byte run of the source pixel
            const int cpt = (int)(p.lda >> 6);
            const int tap = kt / cpt, c0 = (kt - tap * cpt) << 6;
            const int ky = tap / 3, kx = tap - 3 * ky;
#pragma unroll
            for (int i = 0; i < G::A_LOADS; ++i) {
                int sr, sc, wp;
                if constexpr (CONV == 1) {
                    // bordered input: output (y, x) at tap (ky, kx) reads (y + ky, x + kx)
                    sr = cy[i] + ky;
                    sc = cx[i] + kx;
                    wp = p.conv_w + 2;
                } else {
                    // upsampled coordinate u = y + ky - 1 in [-1, conv_h]: the border outside
                    const int u = cy[i] + ky - 1, v = cx[i] + kx - 1;
                    sr = u < 0 ? 0 : (u >= p.conv_h ? p.conv_h / 2 + 1 : (u >> 1) + 1);
                    sc = v < 0 ? 0 : (v >= p.conv_w ? p.conv_w / 2 + 1 : (v >> 1) + 1);
                    wp = p.conv_w / 2 + 2;
                }
                __builtin_amdgcn_global_load_lds(static_cast<const void *>(asrc[i] + ((int64_t)sr * wp + sc) * p.lda + c0),
                                                 SANA_LDS(base + (wi + i * G::GW) * 1024), 16, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < G::B_LOADS; ++i)
            __builtin_amdgcn_global_load_lds(static_cast<const void *>(bsrc[i] + k0), SANA_LDS(base + G::A_BYTES + (wi + i * G::GW) * 1024),
                                             16, 0, 0);
    };

    f32x16 acc[G::TM][G::TN];
#pragma unroll
    for (int i = 0; i < G::TM; ++i)
#pragma unroll
        for (int j = 0; j < G::TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // Operand read offsets within a stage: row R, chunk ch -> R*128 + ((ch ^ ((R >> 1) & 7)) << 4).
    const int arow0 = wm * G::WTM + (lane & 31);
    const int brow0 = wn * G::WTN + (lane & 31);
    const int khalf = lane >> 5;

    // Fragments of a whole k-tile (schedules 1 and 3) or of two MFMA k-steps (2).
    constexpr int NS = kBK / 16;               // MFMA k-steps per tile
    constexpr int NB = (SCHED == 1 || SCHED == 3) ? NS : 2;    // fragment buffers
    f16x8 af[NB][G::TM], bf[NB][G::TN];
    auto load_frags = [&](int stage, int s, int buf) {
        const unsigned char * sa = smem + stage * G::STAGE_BYTES + kg * G::SUB_BYTES;
        const unsigned char * sb = sa + G::A_BYTES;
        const int ch = 2 * s + khalf;
#pragma unroll
        for (int i = 0; i < G::TM; ++i) {
            const int R = arow0 + i * 32;
            af[buf][i] = *reinterpret_cast<const f16x8 *>(sa + R * 128 + ((ch ^ ((R >> 1) & 7)) << 4));
        }
#pragma unroll
        for (int j = 0; j < G::TN; ++j) {
            const int R = brow0 + j * 32;
            bf[buf][j] = *reinterpret_cast<const f16x8 *>(sb + R * 128 + ((ch ^ ((R >> 1) & 7)) << 4));
        }
    };
    // The MFMA computes the transposed tile, D^T = W_frag * A_frag^T, so that
    // lane l of wave tile (i, j) holds output row wm*WTM + i*32 + (l & 31) and,
    // in acc[i][j][4g .. 4g+3], the four consecutive columns
    // wn*WTN + j*32 + 8g + 4(l >> 5) + 0..3: the epilogue then writes 16-byte
    // (fp32) or 8-byte (fp16) row runs to LDS instead of single elements.
    auto mfmas = [&](int buf) {
#pragma unroll
        for (int i = 0; i < G::TM; ++i)
#pragma unroll
            for (int j = 0; j < G::TN; ++j) acc[i][j] = mfma_32x32x16(bf[buf][j], af[buf][i], acc[i][j]);
    };

    // FOLD: the sums of p.k_runs runs of consecutive k-tiles, added in run order --
    // the order of that many k-groups, so that kernels of either kind agree bit
    // for bit.
    f32x16 tot[FOLD ? G::TM : 1][FOLD ? G::TN : 1];
    if constexpr (FOLD) {
#pragma unroll
        for (int i = 0; i < G::TM; ++i)
#pragma unroll
            for (int j = 0; j < G::TN; ++j) tot[i][j] = acc[i][j];
    }
    const int run = FOLD ? (KT + p.k_runs - 1) / p.k_runs : KT;
    int run_left = run;  // k-tiles of the current run still to come
    auto fold = [&]() {
        if constexpr (FOLD) {
            if (--run_left) return;
            run_left = run;
#pragma unroll
            for (int i = 0; i < G::TM; ++i)
#pragma unroll
                for (int j = 0; j < G::TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        tot[i][j][r] += acc[i][j][r];
                        acc[i][j][r] = 0.0f;
                    }
        }
    };

    // Residual epilogue inputs (x rows and the gate), loaded before the main loop
    // so their latency hides behind it: single-pass epilogues with at most two
    // rows per thread (the 64 x 64 and 128 x 64 tiles), plain A.  The thread ->
    // (8-column chunk, rows) map is the epilogue's.
    constexpr int ECPR = BN / 8, ERSTEP = G::NT / ECPR, ERPT = (G::EPI_ROWS + ERSTEP - 1) / ERSTEP;
    constexpr bool kPrefetch = MODE == kGemmResidual && CONV == 0 && G::EPI_ROWS == BM && ERPT <= 2;
    float xpre[kPrefetch ? ERPT : 1][8], gpre[kPrefetch ? ERPT : 1][8], bpre[8];
    // The fp16 epilogue's bias, one column per lane and wave sub-tile (column
    // wn*WTN + j*32 + (lane & 31)); the epilogue hands each lane the values of
    // its 4-column runs with lane shuffles.  Loaded here, its latency hides
    // behind the main loop (loaded in the epilogue it cost 1-2 us per launch).
    constexpr bool kH16 = MODE == kGemmQKV || (MODE == kGemmStore && ACT != kActGeglu);
    float bcol[kH16 ? G::TN : 1];
    if constexpr (kH16) {
#pragma unroll
        for (int j = 0; j < G::TN; ++j) {
            const int c = n0 + wn * G::WTN + j * 32 + (lane & 31);
            bcol[j] = (p.bias && c < p.N) ? p.bias[c] : 0.0f;
        }
    }
    if constexpr (kPrefetch) {
        const int col = n0 + (tid % ECPR) * 8;
        const int nc = min(8, p.N - col);
        const bool act = nc > 0 && tid < ERSTEP * ECPR;
        // bias of the thread's 8 columns
#pragma unroll
        for (int e = 0; e < 8; ++e) bpre[e] = 0.0f;
        if (act && p.bias) {
            if (p.vec && nc == 8) {
                const float4 b0 = *reinterpret_cast<const float4 *>(p.bias + col);
                const float4 b1 = *reinterpret_cast<const float4 *>(p.bias + col + 4);
                bpre[0] = b0.x; bpre[1] = b0.y; bpre[2] = b0.z; bpre[3] = b0.w;
                bpre[4] = b1.x; bpre[5] = b1.y; bpre[6] = b1.z; bpre[7] = b1.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (e < nc) bpre[e] = p.bias[col + e];
            }
        }
#pragma unroll
        for (int k = 0; k < ERPT; ++k) {
            const int row = m0 + tid / ECPR + k * ERSTEP;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                xpre[k][e] = 0.0f;
                gpre[k][e] = 1.0f;
            }
            if (!act || row >= p.M) continue;
            const float * xr = p.out32 + (int64_t)row * p.ldo32 + col;
            const float * ga = p.gate_a ? p.gate_a + (int64_t)(row / p.rows_per_batch) * p.gate_stride + col : nullptr;
            if (p.vec && nc == 8) {
                const float4 x0 = *reinterpret_cast<const float4 *>(xr);
                const float4 x1 = *reinterpret_cast<const float4 *>(xr + 4);
                xpre[k][0] = x0.x; xpre[k][1] = x0.y; xpre[k][2] = x0.z; xpre[k][3] = x0.w;
                xpre[k][4] = x1.x; xpre[k][5] = x1.y; xpre[k][6] = x1.z; xpre[k][7] = x1.w;
                if (ga) {
                    const float4 g0 = *reinterpret_cast<const float4 *>(ga);
                    const float4 g1 = *reinterpret_cast<const float4 *>(ga + 4);
                    gpre[k][0] = g0.x; gpre[k][1] = g0.y; gpre[k][2] = g0.z; gpre[k][3] = g0.w;
                    gpre[k][4] = g1.x; gpre[k][5] = g1.y; gpre[k][6] = g1.z; gpre[k][7] = g1.w;
                    if (p.gate_t) {
                        const float4 t0 = *reinterpret_cast<const float4 *>(p.gate_t + col);
                        const float4 t1 = *reinterpret_cast<const float4 *>(p.gate_t + col + 4);
                        gpre[k][0] += t0.x; gpre[k][1] += t0.y; gpre[k][2] += t0.z; gpre[k][3] += t0.w;
                        gpre[k][4] += t1.x; gpre[k][5] += t1.y; gpre[k][6] += t1.z; gpre[k][7] += t1.w;
                    }
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if (e >= nc) continue;
                    xpre[k][e] = xr[e];
                    if (ga) gpre[k][e] = ga[e] + (p.gate_t ? p.gate_t[col + e] : 0.0f);
                }
            }
        }
    }

#pragma unroll
    for (int s = 0; s < STAGES; ++s)
        if (s < NT_K) issue(s, s);
    wait_stages<G::LOADS, STAGES>(min(STAGES - 1, NT_K - 1));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (SCHED == 3) {
        // Early stage release: all fragments of tile kt are read into registers,
        // a barrier confirms every wave is done with the stage, and the stage is
        // refilled with tile kt+STAGES before the tile's MFMAs run.  With two
        // stages, two tiles of DMA are in flight during the MFMAs instead of one,
        // which hides the longer latency of weights that come from HBM.
        for (int kt = 0; kt < NT_K; ++kt) {
            const int st = kt % STAGES;
            if (kt > 0) {
                __builtin_amdgcn_sched_barrier(0);
                wait_stages<G::LOADS, STAGES>(min(STAGES - 1, NT_K - 1 - kt));
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int s = 0; s < NS; ++s) load_frags(st, s, s);
            __builtin_amdgcn_sched_barrier(0);
            wait_lgkmcnt0();
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            if (kt + STAGES < NT_K) issue(kt + STAGES, st);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < NS; ++s) mfmas(s);
            fold();
        }
    } else if constexpr (SCHED == 1) {
        // every fragment of the tile is requested right after the barrier; the
        // MFMAs of step s wait only for the reads of steps <= s (in-order lgkmcnt)
        for (int kt = 0; kt < NT_K; ++kt) {
            const int st = kt % STAGES;
            if (KG == 1 || kg * NT_K + kt < KT) {
#pragma unroll
                for (int s = 0; s < NS; ++s) load_frags(st, s, s);
#pragma unroll
                for (int s = 0; s < NS; ++s) mfmas(s);
            }
            fold();
            if (kt + 1 < NT_K) {
                __builtin_amdgcn_sched_barrier(0);
                wait_stages<G::LOADS, STAGES>(min(STAGES - 2, NT_K - 2 - kt));
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                if (kt + STAGES < NT_K) issue(kt + STAGES, st);
            }
        }
    } else {
        // Operand fragments double-buffered in registers: the LDS reads of k-step
        // s+1 go out between the MFMAs of step s.  The tile boundary (wait for the
        // next tile's DMA, barrier, refill of the freed stage) comes before the last
        // step's MFMAs, whose fragments are in registers by then, and the next tile's
        // first fragments are requested there too: those MFMAs cover the barrier and
        // the reads, so one workgroup per CU can keep the matrix cores busy.
        constexpr int RD = G::TM + G::TN, MF = G::TM * G::TN;
        load_frags(0, 0, 0);
        for (int kt = 0; kt < NT_K; ++kt) {
            const int st = kt % STAGES;
#pragma unroll
            for (int s = 0; s < NS - 1; ++s) {
                load_frags(st, s + 1, (s + 1) & 1);
                mfmas(s & 1);
#pragma unroll
                for (int q = 0; q < RD; ++q) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                   // an LDS read of step s+1
                    __builtin_amdgcn_sched_group_barrier(0x008, (MF + RD - 1) / RD, 0);  // MFMAs of step s
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (kt + 1 < NT_K) {
                // this wave's reads of stage st have returned and its part of tile kt+1
                // has landed; after the barrier every wave's
                wait_lgkmcnt0();
                wait_stages<G::LOADS, STAGES>(min(STAGES - 2, NT_K - 2 - kt));
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                load_frags((kt + 1) % STAGES, 0, 0);
                if (kt + STAGES < NT_K) issue(kt + STAGES, st);
            }
            mfmas((NS - 1) & 1);
        }
    }

    if constexpr (FOLD) {  // the last run (all zeros where it was folded above)
#pragma unroll
        for (int i = 0; i < G::TM; ++i)
#pragma unroll
            for (int j = 0; j < G::TN; ++j) acc[i][j] += tot[i][j];
    }
    // groups 1.. hand their sums to group 0 through LDS, lane by lane; group 0
    // adds them in group order and runs the epilogue's staging
    if constexpr (KG > 1) {
        float4 * part = reinterpret_cast<float4 *>(smem);
        constexpr int PF4 = G::PART_BYTES / 16;
        __syncthreads();  // every wave is done reading the operand ring
        if (kg > 0) {
#pragma unroll
            for (int i = 0; i < G::TM; ++i)
#pragma unroll
                for (int j = 0; j < G::TN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        part[(kg - 1) * PF4 + ((wi * G::TM + i) * G::TN + j) * 256 + q * 64 + lane] = make_float4(
                            acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
        }
        __syncthreads();
        if (kg == 0) {
#pragma unroll
            for (int i = 0; i < G::TM; ++i)
#pragma unroll
                for (int j = 0; j < G::TN; ++j)
#pragma unroll
                    for (int h = 0; h < KG - 1; ++h)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const float4 v = part[h * PF4 + ((wi * G::TM + i) * G::TN + j) * 256 + q * 64 + lane];
                            acc[i][j][4 * q] += v.x;
                            acc[i][j][4 * q + 1] += v.y;
                            acc[i][j][4 * q + 2] += v.z;
                            acc[i][j][4 * q + 3] += v.w;
                        }
        }
    }

    // ------------------------------------------------------------ epilogue
    // fp16 output row of tile row `row`: plain, or inside the bordered grid of a conv output
    auto orow16 = [&](int row) -> int64_t {
        if constexpr (CONV != 0) {
            if (p.out16_pad) {
                const int hw = p.conv_h * p.conv_w;
                const int img = row / hw, rem = row - img * hw;
                const int y = rem / p.conv_w, x = rem - y * p.conv_w;
                return ((int64_t)img * (p.conv_h + 2) + y + 1) * (p.conv_w + 2) + x + 1;
            }
        }
        return row;
    };
    // fp16-only outputs (plain stores with no fp32 copy, and the q|k|v split):
    // bias, activation and the fp16 rounding are applied to the accumulators in
    // registers (the same operations, in the same order, as the fp32-staged
    // path below), the rounded tile is staged in LDS once as fp16 (8-byte row
    // runs, rows 16-byte aligned), and every thread then issues all of its
    // 16-byte LDS reads before its 16-byte global stores.  Against the fp32
    // staging this halves the LDS bytes, needs a single pass for every tile
    // shape, and keeps several stores in flight per thread.
    if constexpr (MODE == kGemmQKV || (MODE == kGemmStore && ACT != kActGeglu)) {
        if (p.vec && !p.out32) {
            constexpr int LDH = BN + 8;
            static_assert(BM * LDH * 2 <= G::LDS_BYTES, "fp16 epilogue tile");
            f16 * ht = reinterpret_cast<f16 *>(smem);
            __syncthreads();  // every wave is done reading the operand ring
            if (KG == 1 || kg == 0) {  // the k-group that holds the sums
#pragma unroll
            for (int j = 0; j < G::TN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int c = wn * G::WTN + j * 32 + 8 * g + 4 * (lane >> 5);
                    const int col = n0 + c;
                    float b4[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) b4[e] = __shfl(bcol[j], 8 * g + 4 * (lane >> 5) + e, 64);
                    // q and k sections are ReLU'd (a 4-column run never straddles
                    // a section: qkv_c is a multiple of 8)
                    const bool relu = MODE == kGemmQKV && col < 2 * p.qkv_c;
#pragma unroll
                    for (int i = 0; i < G::TM; ++i) {
                        const int row = wm * G::WTM + i * 32 + (lane & 31);
                        f16x4 h;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            float v = acc[i][j][4 * g + e] + b4[e];
                            if constexpr (ACT == kActSilu) v = silu_fast(v);
                            if constexpr (ACT == kActGelu) v = gelu_tanh_f(v);
                            if (relu) v = fmaxf(v, 0.0f);
                            h[e] = (f16)v;
                        }
                        *reinterpret_cast<f16x4 *>(ht + row * LDH + c) = h;
                    }
                }
            }
            __syncthreads();
            // row-major stores (the whole tile, or the q section of the split)
            constexpr int HCPR = BN / 8, CHUNKS = BM * HCPR;
            constexpr int PER = (CHUNKS + G::NT - 1) / G::NT;
            f16x8 hv[PER];
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                const int idx = tid + k * G::NT;
                if (CHUNKS % G::NT == 0 || idx < CHUNKS)
                    hv[k] = *reinterpret_cast<const f16x8 *>(ht + (idx / HCPR) * LDH + (idx % HCPR) * 8);
            }
            f16 * o16 = reinterpret_cast<f16 *>(p.out16);
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                const int idx = tid + k * G::NT;
                if (CHUNKS % G::NT != 0 && idx >= CHUNKS) continue;
                const int row = m0 + idx / HCPR, col = n0 + (idx % HCPR) * 8;
                if (row >= p.M || col >= p.N) continue;
                if constexpr (MODE == kGemmQKV) {
                    if (col >= p.qkv_c) continue;
                }
                f16 * dst = o16 + orow16(row) * p.ldo16 + col;
                if (col + 8 <= p.N) {
                    *reinterpret_cast<f16x8 *>(dst) = hv[k];
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (col + e < p.N) dst[e] = hv[k][e];
                }
            }
            if constexpr (MODE == kGemmQKV) {
                // k and v sections: items (column, 8-row octet), 32 consecutive
                // columns of one octet per 32 items; each item leaves as one
                // 16-byte token run of relu(K)^T or V^T.  Rows of an octet share
                // a batch (qkv_n % 8 == 0).
                constexpr int OCT = BM / 8;
                const int C3 = p.qkv_c;
                for (int item = tid; item < BN * OCT; item += G::NT) {
                    const int c32 = item % 32, rest = item / 32;
                    const int oct = rest % OCT, cl = (rest / OCT) * 32 + c32;
                    const int col = n0 + cl, row0 = m0 + oct * 8;
                    if (col >= p.N || row0 >= p.M || col < C3) continue;
                    const bool is_k = col < 2 * C3;
                    const int ch = col - (is_k ? C3 : 2 * C3);
                    f16x8 h;
#pragma unroll
                    for (int jj = 0; jj < 8; ++jj) h[jj] = ht[(oct * 8 + jj) * LDH + cl];
                    const int b = row0 / p.qkv_n, t0 = row0 - b * p.qkv_n;
                    f16 * dst = reinterpret_cast<f16 *>(is_k ? p.kt16 : p.vt16);
                    *reinterpret_cast<f16x8 *>(dst + ((int64_t)b * C3 + ch) * p.qkv_n + t0) = h;
                }
            }
            return;
        }
    }
    {
        float * ct = reinterpret_cast<float *>(smem);
        constexpr int LDC = BN + G::CPAD;
        constexpr int ER = G::EPI_ROWS;  // tile rows staged per pass
        // Each thread owns one 8-column chunk of the tile for all its rows, so
        // the bias is fetched once; rows step by NT / CPR (threads past the
        // last whole row of chunks stay idle).
        constexpr int CPR = BN / 8;
        static_assert(G::NT >= CPR, "epilogue chunk mapping");
        const int c8 = (tid % CPR) * 8;
        const int col = n0 + c8;
        const int nc = min(8, p.N - col);
        bool active = nc > 0 && tid < (G::NT / CPR) * CPR;
        if constexpr (MODE == kGemmQKV) active = active && col < p.qkv_c;  // k / v columns: item loop
        const bool vec8 = p.vec && nc == 8;
        float bv[8];
        if constexpr (kPrefetch) {
#pragma unroll
            for (int e = 0; e < 8; ++e) bv[e] = bpre[e];
        } else if (!active) {
#pragma unroll
            for (int e = 0; e < 8; ++e) bv[e] = 0.0f;
        } else if (MODE == kGemmVT) {  // bias per row, added below
#pragma unroll
            for (int e = 0; e < 8; ++e) bv[e] = 0.0f;
        } else if (p.bias && vec8) {
            const float4 b0 = *reinterpret_cast<const float4 *>(p.bias + col);
            const float4 b1 = *reinterpret_cast<const float4 *>(p.bias + col + 4);
            bv[0] = b0.x; bv[1] = b0.y; bv[2] = b0.z; bv[3] = b0.w;
            bv[4] = b1.x; bv[5] = b1.y; bv[6] = b1.z; bv[7] = b1.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) bv[e] = (p.bias && e < nc) ? p.bias[col + e] : 0.0f;
        }
        for (int pass = 0; pass < BM / ER; ++pass) {
            __syncthreads();  // the operand ring (pass 0) or the previous pass's rows are free
            if ((KG == 1 || kg == 0) && (ER == BM || wm == pass)) {
                // 16-byte row runs (rows are 16-byte aligned: LDC = BN + 4, BN a multiple of 8)
#pragma unroll
                for (int i = 0; i < G::TM; ++i)
#pragma unroll
                    for (int j = 0; j < G::TN; ++j) {
                        const int rr = (wm * G::WTM - pass * ER) + i * 32 + (lane & 31);
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const int c = wn * G::WTN + j * 32 + 8 * g + 4 * (lane >> 5);
                            *reinterpret_cast<float4 *>(&ct[rr * LDC + c]) =
                                make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
                        }
                    }
            }
            __syncthreads();
            if constexpr (MODE == kGemmQKV) {
                // k and v sections: items (column, 8-row octet).  32 consecutive
                // items take 32 consecutive columns of one octet and the next 32 the
                // same columns one octet further: rows 8 apart are 32 banks apart
                // (LDC = BN + 4), so a wave's fp32 LDS reads hit 64 distinct banks,
                // and each column's two octets leave as one 32-byte token run.  Rows
                // of an octet share a batch (qkv_n % 8 == 0).  The q section is
                // handled below as a plain store.
                constexpr int OCT = ER / 8;
                static_assert(BN % 32 == 0, "32-column item groups");
                const int C3 = p.qkv_c;
                for (int item = tid; item < BN * OCT; item += G::NT) {
                    const int c32 = item % 32, rest = item / 32;
                    const int oct = rest % OCT, cl = (rest / OCT) * 32 + c32;
                    const int col = n0 + cl, row0 = m0 + pass * ER + oct * 8;
                    if (col >= p.N || row0 >= p.M || col < C3) continue;
                    const bool is_k = col < 2 * C3;
                    const int ch = col - (is_k ? C3 : 2 * C3);
                    const float bcol = p.bias ? p.bias[col] : 0.0f;
                    f16x8 h;
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        float v = ct[(oct * 8 + j) * LDC + cl] + bcol;
                        if (is_k) v = fmaxf(v, 0.0f);
                        h[j] = (f16)v;
                    }
                    const int b = row0 / p.qkv_n, t0 = row0 - b * p.qkv_n;
                    f16 * dst = reinterpret_cast<f16 *>(is_k ? p.kt16 : p.vt16);
                    *reinterpret_cast<f16x8 *>(dst + ((int64_t)b * C3 + ch) * p.qkv_n + t0) = h;
                }
            }
            if constexpr (MODE == kGemmVT) {
                // element (m, n), m = blk * vt_rows + r, n = b * vt_cols + j, goes to
                // out16[((blk * vt_batch + b) * vt_rows + r) * vt_ld + j]; bias per row.
                // A chunk inside one batch's columns leaves as two 8-byte stores
                // (vt_cols need not be a multiple of 8, so j is a multiple of 4 at best).
                const int vb = col / p.vt_cols, vj = col - vb * p.vt_cols;
                const bool vec4 = p.vec && nc == 8 && vj + 8 <= p.vt_cols && (vj & 3) == 0 && (p.vt_ld & 3) == 0;
                f16 * o16 = reinterpret_cast<f16 *>(p.out16);
                if (active) {
                    for (int rr = tid / CPR; rr < ER; rr += G::NT / CPR) {
                        const int row = m0 + pass * ER + rr;
                        if (row >= p.M) break;
                        const int blk = row / p.vt_rows, r = row - blk * p.vt_rows;
                        const float bvr = p.bias ? p.bias[row] : 0.0f;
                        const float4 v0 = *reinterpret_cast<const float4 *>(&ct[rr * LDC + c8]);
                        const float4 v1 = *reinterpret_cast<const float4 *>(&ct[rr * LDC + c8 + 4]);
                        const float v[8] = {v0.x + bvr, v0.y + bvr, v0.z + bvr, v0.w + bvr,
                                            v1.x + bvr, v1.y + bvr, v1.z + bvr, v1.w + bvr};
                        if (vec4) {
                            f16 * dst = o16 + ((int64_t)(blk * p.vt_batch + vb) * p.vt_rows + r) * p.vt_ld + vj;
                            f16x4 h0, h1;
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                h0[e] = (f16)v[e];
                                h1[e] = (f16)v[4 + e];
                            }
                            *reinterpret_cast<f16x4 *>(dst) = h0;
                            *reinterpret_cast<f16x4 *>(dst + 4) = h1;
                        } else {
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                if (e >= nc) continue;
                                const int b = (col + e) / p.vt_cols, jj = col + e - b * p.vt_cols;
                                o16[((int64_t)(blk * p.vt_batch + b) * p.vt_rows + r) * p.vt_ld + jj] = (f16)v[e];
                            }
                        }
                    }
                }
            } else if (active && MODE != kGemmResidual) {
                for (int rr = tid / CPR; rr < ER; rr += G::NT / CPR) {
                    const int row = m0 + pass * ER + rr;
                    if (row >= p.M) break;
                    const float4 v0 = *reinterpret_cast<const float4 *>(&ct[rr * LDC + c8]);
                    const float4 v1 = *reinterpret_cast<const float4 *>(&ct[rr * LDC + c8 + 4]);
                    float v[8] = {v0.x + bv[0], v0.y + bv[1], v0.z + bv[2], v0.w + bv[3],
                                  v1.x + bv[4], v1.y + bv[5], v1.z + bv[6], v1.w + bv[7]};
                    if constexpr (MODE == kGemmStore && ACT == kActGeglu) {
                        // gate / up column pairs -> 4 gated outputs at column col / 2
                        f16x4 h;
#pragma unroll
                        for (int e = 0; e < 4; ++e) h[e] = (f16)(gelu_tanh_f(v[2 * e]) * v[2 * e + 1]);
                        f16 * o = reinterpret_cast<f16 *>(p.out16) + (int64_t)row * p.ldo16 + col / 2;
                        if (vec8) {
                            *reinterpret_cast<f16x4 *>(o) = h;
                        } else {
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                if (2 * e + 1 < nc) o[e] = h[e];
                        }
                    } else if constexpr (MODE == kGemmStore || MODE == kGemmQKV) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            if constexpr (ACT == kActSilu) v[e] = silu_fast(v[e]);
                            if constexpr (ACT == kActGelu) v[e] = gelu_tanh_f(v[e]);
                            if constexpr (MODE == kGemmQKV) v[e] = fmaxf(v[e], 0.0f);
                        }
                        if (vec8) {
                            if (p.out16) {
                                f16x8 h;
#pragma unroll
                                for (int e = 0; e < 8; ++e) h[e] = (f16)v[e];
                                *reinterpret_cast<f16x8 *>(reinterpret_cast<f16 *>(p.out16) + orow16(row) * p.ldo16 + col) = h;
                            }
                            if (p.out32) {
                                float * o = p.out32 + (int64_t)row * p.ldo32 + col;
                                *reinterpret_cast<float4 *>(o) = make_float4(v[0], v[1], v[2], v[3]);
                                *reinterpret_cast<float4 *>(o + 4) = make_float4(v[4], v[5], v[6], v[7]);
                            }
                        } else {
#pragma unroll
                            for (int e = 0; e < 8; ++e) {  // static indices: v stays in registers
                                if (e >= nc) continue;
                                if (p.out16) reinterpret_cast<f16 *>(p.out16)[orow16(row) * p.ldo16 + col + e] = (f16)v[e];
                                if (p.out32) p.out32[(int64_t)row * p.ldo32 + col + e] = v[e];
                            }
                        }
                    }
                }
            }
            if constexpr (MODE == kGemmResidual) {
                if (active) {
                    // x += gate * (acc + bias).  All of this
                    // thread's residual rows are loaded first (one batch of loads in
                    // flight), then updated and stored.
                    constexpr int RSTEP = G::NT / CPR;
                    constexpr int RPT = (ER + RSTEP - 1) / RSTEP;
                    const int rbase = tid / CPR;
                    float xin[RPT][8];
#pragma unroll
                    for (int k = 0; k < RPT; ++k) {
                        const int rr = rbase + k * RSTEP;
                        const int row = m0 + pass * ER + rr;
#pragma unroll
                        for (int e = 0; e < 8; ++e) xin[k][e] = 0.0f;
                        if constexpr (kPrefetch) {
#pragma unroll
                            for (int e = 0; e < 8; ++e) xin[k][e] = xpre[k][e];
                            continue;
                        }
                        if (rr >= ER || row >= p.M) continue;
                        bool gathered = false;
                        if constexpr (CONV == 2) {
                            if (p.up_src) {
                                // the residual starts as the pixel-shuffled channel-repeat
                                // shortcut of the low-resolution input
                                const int hw = p.conv_h * p.conv_w;
                                const int img = row / hw, rem = row - img * hw;
                                const int Y = rem / p.conv_w, X = rem - Y * p.conv_w;
                                const float * src =
                                    p.up_src + ((int64_t)(img * (p.conv_h / 2) + (Y >> 1)) * (p.conv_w / 2) + (X >> 1)) *
                                                   p.up_c;
                                const int q = 2 * (Y & 1) + (X & 1);
#pragma unroll
                                for (int e = 0; e < 8; ++e)
                                    if (e < nc) xin[k][e] = src[((col + e) * 4 + q) / p.up_rep];
                                gathered = true;
                            }
                        }
                        if (!gathered) {
                            const float * xr = p.out32 + (int64_t)row * p.ldo32 + col;
                            if (vec8) {
                                const float4 x0 = *reinterpret_cast<const float4 *>(xr);
                                const float4 x1 = *reinterpret_cast<const float4 *>(xr + 4);
                                xin[k][0] = x0.x; xin[k][1] = x0.y; xin[k][2] = x0.z; xin[k][3] = x0.w;
                                xin[k][4] = x1.x; xin[k][5] = x1.y; xin[k][6] = x1.z; xin[k][7] = x1.w;
                            } else {
#pragma unroll
                                for (int e = 0; e < 8; ++e)
                                    if (e < nc) xin[k][e] = xr[e];
                            }
                        }
                    }
#pragma unroll
                    for (int k = 0; k < RPT; ++k) {
                        const int rr = rbase + k * RSTEP;
                        const int row = m0 + pass * ER + rr;
                        if (rr >= ER || row >= p.M) continue;
                        const float4 v0 = *reinterpret_cast<const float4 *>(&ct[rr * LDC + c8]);
                        const float4 v1 = *reinterpret_cast<const float4 *>(&ct[rr * LDC + c8 + 4]);
                        float v[8] = {v0.x + bv[0], v0.y + bv[1], v0.z + bv[2], v0.w + bv[3],
                                      v1.x + bv[4], v1.y + bv[5], v1.z + bv[6], v1.w + bv[7]};
                        const int b = row / p.rows_per_batch;
                        float g[8];
                        if constexpr (kPrefetch) {
#pragma unroll
                            for (int e = 0; e < 8; ++e) g[e] = gpre[k][e];
                        } else if (p.gate_a && vec8) {
                            const float * ga = p.gate_a + (int64_t)b * p.gate_stride + col;
                            const float4 g0 = *reinterpret_cast<const float4 *>(ga);
                            const float4 g1 = *reinterpret_cast<const float4 *>(ga + 4);
                            g[0] = g0.x; g[1] = g0.y; g[2] = g0.z; g[3] = g0.w;
                            g[4] = g1.x; g[5] = g1.y; g[6] = g1.z; g[7] = g1.w;
                            if (p.gate_t) {
                                const float4 t0 = *reinterpret_cast<const float4 *>(p.gate_t + col);
                                const float4 t1 = *reinterpret_cast<const float4 *>(p.gate_t + col + 4);
                                g[0] += t0.x; g[1] += t0.y; g[2] += t0.z; g[3] += t0.w;
                                g[4] += t1.x; g[5] += t1.y; g[6] += t1.z; g[7] += t1.w;
                            }
                        } else {
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                g[e] = 1.0f;
                                if (p.gate_a && e < nc) {
                                    g[e] = p.gate_a[(int64_t)b * p.gate_stride + col + e];
                                    if (p.gate_t) g[e] += p.gate_t[col + e];
                                }
                            }
                        }
                        float x[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e) x[e] = xin[k][e] + g[e] * v[e];
                        float * xr = p.out32 + (int64_t)row * p.ldo32 + col;
                        if (vec8) {
                            *reinterpret_cast<float4 *>(xr) = make_float4(x[0], x[1], x[2], x[3]);
                            *reinterpret_cast<float4 *>(xr + 4) = make_float4(x[4], x[5], x[6], x[7]);
                            if (p.out16) {
                                f16x8 h;
#pragma unroll
                                for (int e = 0; e < 8; ++e) h[e] = (f16)x[e];
                                *reinterpret_cast<f16x8 *>(reinterpret_cast<f16 *>(p.out16) + orow16(row) * p.ldo16 + col) = h;
                            }
                        } else {
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                if (e >= nc) continue;
                                xr[e] = x[e];
                                if (p.out16) reinterpret_cast<f16 *>(p.out16)[orow16(row) * p.ldo16 + col + e] = (f16)x[e];
                            }
                        }
                    }
                }
            }
        }
    }
}

bool set_lds_limit(const void * k, size_t lds) {
    return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
}

template <int BM, int BN, int WM, int WN, int STAGES, int MODE, int SCHED, int ACT, int CONV = 0, int KG = 1,
          bool FOLD = false>
hipError_t launch_mode(const GemmParams & p, int tiles, hipStream_t s) {
    using G = Cfg<BM, BN, WM, WN, STAGES, KG>;
    static const bool attr = set_lds_limit(
        reinterpret_cast<const void *>(&gemm_kernel<BM, BN, WM, WN, STAGES, MODE, SCHED, ACT, CONV, KG, FOLD>), G::LDS_BYTES);
    (void)attr;
    static const std::string name = "gemm_kernel<" + std::to_string(BM) + ", " + std::to_string(BN) + ", " +
                                    std::to_string(WM) + ", " + std::to_string(WN) + ", " + std::to_string(STAGES) +
                                    ", " + std::to_string(MODE) + ", " + std::to_string(SCHED) + ", " +
                                    std::to_string(ACT) + ", " + std::to_string(CONV) + ", " +
                                    std::to_string(KG) + (FOLD ? ", true>" : ", false>");
    note_kernel(name.c_str());
    hipLaunchKernelGGL((gemm_kernel<BM, BN, WM, WN, STAGES, MODE, SCHED, ACT, CONV, KG, FOLD>), dim3(tiles, p.batch), dim3(G::NT),
                       G::LDS_BYTES, s, p);
    return hipGetLastError();
}

// Implicit 3x3 convolutions: plain stores (optionally SiLU) and residual updates.
template <int BM, int BN, int WM, int WN, int STAGES, int SCHED, int CONV>
hipError_t launch_conv_mode(const GemmParams & p, hipStream_t s) {
    const int tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
    if (p.mode == kGemmResidual)
        return launch_mode<BM, BN, WM, WN, STAGES, kGemmResidual, SCHED, kActNone, CONV>(p, tiles, s);
    if (p.act == kActSilu) return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActSilu, CONV>(p, tiles, s);
    return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActNone, CONV>(p, tiles, s);
}

template <int BM, int BN, int WM, int WN, int STAGES, int SCHED>
hipError_t launch_conv(const GemmParams & p, hipStream_t s) {
    if (p.conv == 2) return launch_conv_mode<BM, BN, WM, WN, STAGES, SCHED, 2>(p, s);
    return launch_conv_mode<BM, BN, WM, WN, STAGES, SCHED, 1>(p, s);
}

// Sums of several runs of k (GemmParams::k_runs): KG groups of waves, one run
// each, or (KG = 1) one group that folds its sums.  Stores, residual updates and
// the q|k|v split.
template <int BM, int BN, int WM, int WN, int STAGES, int SCHED, int KG>
hipError_t launch_runs(const GemmParams & p, hipStream_t s) {
    constexpr bool F = KG == 1;
    const int tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
    if (p.mode == kGemmResidual)
        return launch_mode<BM, BN, WM, WN, STAGES, kGemmResidual, SCHED, kActNone, 0, KG, F>(p, tiles, s);
    if (p.mode == kGemmQKV) return launch_mode<BM, BN, WM, WN, STAGES, kGemmQKV, SCHED, kActNone, 0, KG, F>(p, tiles, s);
    if (p.act == kActSilu) return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActSilu, 0, KG, F>(p, tiles, s);
    if (p.act == kActGelu) return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActGelu, 0, KG, F>(p, tiles, s);
    return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActNone, 0, KG, F>(p, tiles, s);
}

// The same for the 3x3 convolutions.
template <int BM, int BN, int WM, int WN, int STAGES, int SCHED, int CONV, int KG>
hipError_t launch_conv_runs_mode(const GemmParams & p, hipStream_t s) {
    constexpr bool F = KG == 1;
    const int tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
    if (p.mode == kGemmResidual)
        return launch_mode<BM, BN, WM, WN, STAGES, kGemmResidual, SCHED, kActNone, CONV, KG, F>(p, tiles, s);
    if (p.act == kActSilu) return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActSilu, CONV, KG, F>(p, tiles, s);
    return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActNone, CONV, KG, F>(p, tiles, s);
}

template <int BM, int BN, int WM, int WN, int STAGES, int SCHED, int KG>
hipError_t launch_conv_runs(const GemmParams & p, hipStream_t s) {
    if (p.conv == 2) return launch_conv_runs_mode<BM, BN, WM, WN, STAGES, SCHED, 2, KG>(p, s);
    return launch_conv_runs_mode<BM, BN, WM, WN, STAGES, SCHED, 1, KG>(p, s);
}

// 256 x 256 tiles (8 waves of 128 x 64, one workgroup per CU): stores and the q|k|v split.
hipError_t launch256(const GemmParams & p, hipStream_t s) {
    const int tiles = ((p.M + 255) / 256) * ((p.N + 255) / 256);
    if (p.mode == kGemmQKV) return launch_mode<256, 256, 2, 4, 2, kGemmQKV, 2, kActNone>(p, tiles, s);
    if (p.act == kActSilu) return launch_mode<256, 256, 2, 4, 2, kGemmStore, 2, kActSilu>(p, tiles, s);
    if (p.act == kActGelu) return launch_mode<256, 256, 2, 4, 2, kGemmStore, 2, kActGelu>(p, tiles, s);
    if (p.act == kActGeglu) return launch_mode<256, 256, 2, 4, 2, kGemmStore, 2, kActGeglu>(p, tiles, s);
    return launch_mode<256, 256, 2, 4, 2, kGemmStore, 2, kActNone>(p, tiles, s);
}

template <int BM, int BN, int WM, int WN, int STAGES, int SCHED>
hipError_t launch(const GemmParams & p, hipStream_t s) {
    const int tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
    if (p.mode == kGemmResidual) return launch_mode<BM, BN, WM, WN, STAGES, kGemmResidual, SCHED, kActNone>(p, tiles, s);
    if (p.mode == kGemmVT) return launch_mode<BM, BN, WM, WN, STAGES, kGemmVT, SCHED, kActNone>(p, tiles, s);
    if (p.mode == kGemmQKV) return launch_mode<BM, BN, WM, WN, STAGES, kGemmQKV, SCHED, kActNone>(p, tiles, s);
    if (p.act == kActSilu) return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActSilu>(p, tiles, s);
    if (p.act == kActGelu) return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActGelu>(p, tiles, s);
    if (p.act == kActGeglu) return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActGeglu>(p, tiles, s);
    return launch_mode<BM, BN, WM, WN, STAGES, kGemmStore, SCHED, kActNone>(p, tiles, s);
}

}  // namespace gemm_detail

using namespace gemm_detail;

hipError_t gemm(const GemmParams & p_in, hipStream_t s) {
    GemmParams p = p_in;
    if (p.M <= 0 || p.N <= 0 || p.K <= 0 || p.K % kBK != 0) return hipErrorInvalidValue;
    if (p.conv < 0 || p.conv > 2) return hipErrorInvalidValue;
    if (p.conv) {
        // implicit 3x3 conv: K = 9 taps x lda channels, M whole images of conv_h x conv_w
        if (p.conv_h <= 0 || p.conv_w <= 0 || p.lda <= 0 || p.lda % kBK || p.K != 9 * p.lda ||
            p.M % (p.conv_h * p.conv_w) || (p.mode != kGemmStore && p.mode != kGemmResidual) ||
            (p.conv == 2 && (p.conv_h % 2 || p.conv_w % 2)))
            return hipErrorInvalidValue;
    } else if (p.out16_pad || p.lda < p.K) {
        return hipErrorInvalidValue;
    }
    if (!p.A || !p.W || p.ldw < p.K || p.lda % 8 || p.ldw % 8) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(p.A) | reinterpret_cast<uintptr_t>(p.W)) & 15) return hipErrorInvalidValue;
    if (p.mode == kGemmResidual && !p.out32) return hipErrorInvalidValue;
    if (p.up_src && (p.conv != 2 || p.mode != kGemmResidual || p.up_c <= 0 || p.up_rep <= 0 ||
                     ((int64_t)p.N * 4 + p.up_rep - 1) / p.up_rep > p.up_c))
        return hipErrorInvalidValue;
    if (p.mode == kGemmVT && (!p.out16 || p.vt_rows <= 0 || p.vt_cols <= 0 || p.vt_batch <= 0 ||
                              p.vt_ld < p.vt_cols || p.N != p.vt_batch * p.vt_cols || p.M % p.vt_rows))
        return hipErrorInvalidValue;
    if (p.mode == kGemmStore && !p.out16 && !p.out32) return hipErrorInvalidValue;
    if (p.act < kActNone || p.act > kActGeglu) return hipErrorInvalidValue;
    if (p.act == kActGeglu && (p.mode != kGemmStore || p.conv || !p.out16 || p.out32 || p.N % 8 ||
                               p.ldo16 < p.N / 2 || p.batch != 1))
        return hipErrorInvalidValue;
    if (p.mode == kGemmQKV &&
        (!p.out16 || p.out32 || !p.kt16 || !p.vt16 || p.qkv_c <= 0 || p.qkv_c % 8 || p.N != 3 * p.qkv_c ||
         p.qkv_n <= 0 || p.qkv_n % 8 || p.M % p.qkv_n ||
         ((reinterpret_cast<uintptr_t>(p.kt16) | reinterpret_cast<uintptr_t>(p.vt16)) & 15)))
        return hipErrorInvalidValue;
    if (p.gate_a && p.rows_per_batch <= 0) return hipErrorInvalidValue;
    if (p.k_runs != 1 && (p.k_runs != 4 || p.mode != kGemmStore || p.conv || p.act != kActNone))
        return hipErrorInvalidValue;
    if (p.batch < 1 || p.batch > 65535 || p.batch_w_div < 1 ||
        (p.batch > 1 && (p.mode != kGemmStore || p.conv ||
                         ((p.batch_a | p.batch_w | p.batch_o16 | p.batch_o32) & 7) != 0)))
        return hipErrorInvalidValue;
    // 16-byte epilogue accesses need 8-element aligned rows and 16-byte aligned bases.
    bool vec = true;
    if (p.out16) vec = vec && p.ldo16 % 8 == 0 && (reinterpret_cast<uintptr_t>(p.out16) & 15) == 0;
    if (p.out32) vec = vec && p.ldo32 % 4 == 0 && (reinterpret_cast<uintptr_t>(p.out32) & 15) == 0;
    if (p.gate_a) vec = vec && p.gate_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(p.gate_a) & 15) == 0;
    if (p.gate_t) vec = vec && (reinterpret_cast<uintptr_t>(p.gate_t) & 15) == 0;
    if (p.bias) vec = vec && (reinterpret_cast<uintptr_t>(p.bias) & 15) == 0;
    p.vec = vec ? 1 : 0;
    const int64_t co = std::max(p.co, 1) * (int64_t)p.batch;
    // 32x64 tiles with four k-groups, one workgroup per CU: a few more than 256 still
    // fit a round where another launch shares the CUs, alone they take a second one
    auto one_round = [](int64_t launches) { return launches > 1 ? 288 : 256; };
    auto grid = [&](int bm, int bn) { return ((int64_t)p.M + bm - 1) / bm * ((p.N + bn - 1) / bn) * co; };
    // The order of the k sums follows from the rows that decide it alone
    // (GemmParams::order_rows), the tiles below from the launch's own rows.
    if (p.k_runs == 1 && p.order_rows >= 0 &&
        (p.conv || (p.K >= 512 && p.batch == 1 && p.mode != kGemmVT && p.act != kActGeglu))) {
        const int64_t rows = p.order_rows > 0 ? p.order_rows : p.M;
        const int64_t oco = p.order_co > 0 ? p.order_co : co;
        auto order = [&](int bm, int bn) { return (rows + bm - 1) / bm * ((p.N + bn - 1) / bn) * oco; };
        if (order(32, 64) <= one_round(oco) || (!p.conv && order(32, 32) <= 256)) p.k_runs = 4;
        else if (order(64, 64) <= (p.conv ? 320 : 256)) p.k_runs = 2;
    }
    // Rounds (in 1/64) of `slots` workgroups at a time that bm x bn tiles of all
    // rows take; launches that share the CUs fill each other's last round.
    auto rounds = [&](int bm, int bn, int64_t slots) {
        const int64_t t = ((int64_t)p.M + bm - 1) / bm * ((p.N + bn - 1) / bn) * co;
        return co > 1 ? std::max<int64_t>(64, t * 64 / slots) : (t + slots - 1) / slots * 64;
    };
    if (p.conv) {
        if (p.k_runs == 4 && grid(32, 64) <= one_round(co)) return launch_conv_runs<32, 64, 1, 2, 3, 1, 4>(p, s);
        if (p.k_runs == 4 && grid(64, 64) <= 256) return launch_conv_runs<64, 64, 2, 2, 2, 1, 4>(p, s);
        if (p.k_runs == 2 && grid(64, 64) <= 320) return launch_conv_runs<64, 64, 2, 2, 4, 1, 2>(p, s);
        if (p.k_runs > 1) {
            if (p.N > 64 && grid(128, 128) > 256) return launch_conv_runs<128, 128, 4, 2, 2, 1, 1>(p, s);
            if (grid(128, 64) >= 256) return launch_conv_runs<128, 64, 2, 2, 2, 3, 1>(p, s);
            return launch_conv_runs<64, 64, 2, 2, 3, 1, 1>(p, s);
        }
        if (p.N <= 64) return launch_conv<128, 64, 2, 2, 2, 3>(p, s);
        // A round of 256 workgroups of 256x256 takes 1.85 of a round of 512 of
        // 128x128 (us, before -> after: 512^2 x 256 conv1 364 -> 337, conv2 391 ->
        // 370; 256^2 x 512 340 -> 301, 348 -> 323; onto 512^2 x 256 820 -> 700).
        if (rounds(256, 256, 256) * 185 < rounds(128, 128, 512) * 100)
            return launch_conv<256, 256, 2, 4, 2, 2>(p, s);
        // (1024^2 x 128: conv1 433 -> 426, conv2 467 -> 460; the upsampling conv, whose
        // residual epilogue reads the shortcut, 944 -> 897 with 8 waves)
        if (p.conv == 2) return launch_conv<128, 128, 4, 2, 2, 2>(p, s);
        return launch_conv<128, 128, 2, 2, 2, 2>(p, s);
    }
    // Tile choice from sweeps on MI355X with cold weights (each GEMM's weights
    // come from HBM, as in the 28-block forward).  Every CU pulls at most
    // ~110 GB/s from L2, so larger tiles (fewer operand bytes per flop) win as
    // long as the grid still covers the 256 CUs:
    //  * grids of <= 160 128x128 tiles: shared with a concurrent launch (the
    //    two CFG branches), 64x64 tiles with three stages, early release for
    //    stores and the plain schedule for the residual GEMMs (1024 px forward
    //    5.055 -> 5.037 ms in one process);
    //    alone, 128x64 tiles with early stage release when that makes >= 256
    //    tiles, else 64x64 tiles (three stages and early release for K >= 2048:
    //    600-row caption projection, K = 2304: 20.3 -> 15.8 us);
    //  * grids of 161..256 128x128 tiles: 128x64 tiles with early release
    //    (738-row Gemma q|k|v 36.8 -> 31.3 us, its split output projection
    //    20.6 -> 17.2 us);
    //  * N a multiple of 192 and >= 768 128x192 tiles (1.5 rounds of the 512
    //    two-per-CU slots): 128x192, stores and residual alike (16384-row
    //    launches: 5-12 % faster than 128x128);
    //  * plain stores of N >= 3456 whose 128x192 grid fits one round of slots
    //    where the 128x128 grid does not: 128x192 (1024-row inverted FFN);
    //  * at most 5 row (or column) tiles of 128 against >= 128 of the other
    //    (the step's cross K 600 x 32256 and V^T 32256 x 600): 128x128 tiles
    //    of 8 waves (4 x 2, 32 x 64 per wave): 67.4 -> 60.0 us and 63.2 -> 60.8 us;
    //  * stores and the q|k|v split with more 128x128 tiles than slots: 256x256
    //    tiles where their rounds of 256 workgroups, 1.82 of a round of 512 of
    //    128x128 each (128x192: 1.41), come to less (us, before -> after: 738 x
    //    18432 x 2304 gate | up 90 -> 75; 4096 x 3456 x 1152 48.4 -> 42.5; 8192 x
    //    5760 x 1152 with SiLU 146 -> 140; 8192^3 945 -> 1105 TFLOP/s).  Their waves read
    //    half of the LDS bytes per product of 64 x 64 ones;
    //  * otherwise 128x128 tiles with two stages, two workgroups per CU.
    //  These use schedule 2 (against 1, 16384 rows: 128x192 stores and q|k|v 260 ->
    //  256 and 163 -> 156 us, K = 2880 residuals 138 -> 136.5; 128x128 q|k|v of two
    //  2048-row launches 45.2 -> 43.0), except
    //  - the at most 5 row tiles above;
    //  - 128x192 residual GEMMs with K <= 1152: 8 waves (4 x 2) and schedule 1 (72 us
    //    against 74);
    //  - two rounds of 128x128 q|k|v of which the second is less than half full, the
    //    same 8 waves and schedule 1, and 128x192 beside another launch with 1.5 to
    //    1.6 rounds, schedule 1 (steps of 36 x 36 and 40 x 40 tokens 7.23 -> 7.13 and
    //    7.70 -> 7.37 ms; from 14 row panels on, 41 x 41 tokens, schedule 2 is the
    //    faster one again).
    // (tile counts are scaled by the launches that share the CUs, p.co, and
    // by the products of a batched launch)
    // Grids of few tiles leave most CUs idle and each workgroup with a chain of
    // K / 64 tile latencies (0.44 us each); k-groups cut the chain and keep more
    // bytes in flight per CU.  The smallest tiles that still fit about one
    // workgroup per CU; graph chains, us per launch, before -> after (M x N x K):
    //  128 x 1152 x 1152 residual 11.5 -> 6.4, K = 2880 18.3 -> 9.6 (32x32, 4 groups);
    //  143 x 3072 x 1024 9.8 -> 6.3 (32x64, 4 groups); 512 x 1152 x 1152 store
    //  10.7 -> 7.8, residual K = 2880 19.1 -> 15.3 (64x64, 2 groups).  32x64 tiles
    //  stay to 288 of them only beside another launch: alone those are a second
    //  round (33 x 9000 x 1024, 282 of them 10.0 us with weights in the cache and
    //  11.8 without, 141 of 64x64 in 2 groups 6.9 and 7.8).  From 1.3
    //  workgroups per CU on (324 64x64 tiles) the gain is 3 % and falls to none.
    //  Where the rows that decide the order are fewer than the launch's (a batch
    //  of images sums as one image does), k-groups stay while the launch's own
    //  grid is that small; beyond it one group folds the runs on the tiles that
    //  the grid fills (k-groups of 32x32 tiles there read four times the operand
    //  bytes: 32 decodes of 8 x 8 latents 33.6 -> 29.2 ms, 8 of 16 x 16 29.6 -> 28.6).
    //  Sums that may not depend on M (the text encoder) take k_runs: 23 x 4096 x
    //  2304 15.2 -> 9.3, 23 x 2304 x 2304 15.2 -> 8.7; folding the same four runs
    //  in one group costs 738-row launches 0-2 %.  Its gate | up product keeps k
    //  in one sequence; up to 32 rows one-wave 32x32 tiles stream its weights from
    //  memory at 4.5 TB/s (27.0 -> 19.1 us; only there: a plain store whose weights
    //  are in the cache is slower on them, 32 x 18432 x 2304 18.9 -> 21.3).
    if (p.k_runs > 1) {
        if (p.k_runs == 4) {
            if (grid(32, 32) <= 256) return launch_runs<32, 32, 1, 1, 3, 1, 4>(p, s);
            if (p.order_rows < 0 && p.M > 32 && p.M <= 64 && grid(64, 32) <= 256)
                return launch_mode<64, 32, 2, 1, 3, kGemmStore, 1, kActNone, 0, 4>(
                    p, ((p.M + 63) / 64) * ((p.N + 31) / 32), s);
            if (grid(32, 64) <= (p.order_rows < 0 ? 256 : one_round(co))) return launch_runs<32, 64, 1, 2, 3, 1, 4>(p, s);
            if (grid(64, 64) <= 256) return launch_runs<64, 64, 2, 2, 2, 1, 4>(p, s);
        } else if (grid(64, 64) <= 256) {
            return launch_runs<64, 64, 2, 2, 4, 1, 2>(p, s);
        }
        if (p.N > 64 && grid(128, 128) > 256) return launch_runs<128, 128, 4, 2, 2, 1, 1>(p, s);
        // (as below, 64x64 tiles for few 128x128 ones beside other launches or products:
        // the four parts of the 184-row text-encoder down projection 30.9 -> 25 us)
        if (!(co >= 2 && grid(128, 128) <= 160) && grid(128, 64) >= 256)
            return launch_runs<128, 64, 2, 2, 2, 3, 1>(p, s);
        return launch_runs<64, 64, 2, 2, 3, 1, 1>(p, s);
    }
    if (p.M <= 32 && p.act == kActGeglu && p.N >= 8192) return launch<32, 32, 1, 1, 4, 1>(p, s);
    const int64_t tm128 = (p.M + 127) / 128;
    const int64_t t128 = tm128 * ((p.N + 127) / 128) * co;
    if (t128 <= 160) {
        if (co >= 2)
            return p.mode == kGemmResidual ? launch<64, 64, 2, 2, 3, 1>(p, s) : launch<64, 64, 2, 2, 3, 3>(p, s);
        if (tm128 * ((p.N + 63) / 64) >= 256) return launch<128, 64, 2, 2, 2, 3>(p, s);
        if (p.K >= 2048) return launch<64, 64, 2, 2, 3, 3>(p, s);
        return launch<64, 64, 2, 2, 2, 1>(p, s);
    }
    if (t128 <= 256 && tm128 * ((p.N + 63) / 64) * co >= 256) return launch<128, 64, 2, 2, 2, 3>(p, s);
    const int64_t tn128 = (p.N + 127) / 128;
    const int64_t t192 = p.N % 192 == 0 ? tm128 * (p.N / 192) * co : 0;
    constexpr int64_t kSlots = 512;
    const bool one_round192 = p.mode == kGemmStore && p.N >= 3456 && t192 > 0 && t192 <= kSlots && t128 > kSlots;
    if (t128 > kSlots && (p.mode == kGemmStore || p.mode == kGemmQKV)) {
        const int64_t c256 = rounds(256, 256, 256) * 182, c128 = rounds(128, 128, kSlots) * 100;
        if (c256 < c128 && (p.N % 192 || c256 < rounds(128, 192, kSlots) * 141)) return launch256(p, s);
    }
    if (!one_round192 && co == 1 && std::min(tm128, tn128) <= 5 && std::max(tm128, tn128) >= 128)
        return launch<128, 128, 4, 2, 2, 1>(p, s);
    if (t192 >= kSlots * 3 / 2 || one_round192) {
        if (p.mode == kGemmResidual && p.K <= 1152) return launch<128, 192, 4, 2, 2, 1>(p, s);
        if (co > 1 && t192 >= kSlots * 3 / 2 && t192 < kSlots * 8 / 5) return launch<128, 192, 2, 2, 2, 1>(p, s);
        return launch<128, 192, 2, 2, 2, 2>(p, s);
    }
    if (p.mode == kGemmQKV && t128 > kSlots && t128 < kSlots * 3 / 2) return launch<128, 128, 4, 2, 2, 1>(p, s);
    return launch<128, 128, 2, 2, 2, 2>(p, s);
}

}  // namespace sana
