/*
 * k_qgemm.hip - dequantize-on-use GEMM on gfx950 MFMA:  y[M,N] = x[M,K] W[N,K]^T (+ b)
 *
 * Replaces the reference's aria_linear_q8 / aria_linear_q4 (src/aria_quant.c:98-145,
 * 469-538) and its device path (k_dequant_q8/q4 into an fp16 scratch copy of W, then
 * cublasGemmEx, src/aria_cuda.cu:1009-1035). Here the packed weights never leave
 * their quantized layout in HBM: each workgroup fetches 32-wide K slices of its
 * weight rows still packed, unpacks them in registers, and writes fp16 into LDS for
 * the MFMA.
 *
 *   Q8 (per-row symmetric): the int8 values are exact in fp16; the row scale is
 *       applied once in the epilogue, y = acc * scale[n] (+ b[n]), the reference's
 *       order (src/aria_quant.c:141).
 *   Q4 (per-32-block asymmetric): a 32-wide slice is exactly one quantization block,
 *       so each row needs one [min, step] pair per slice; the weight is rebuilt as
 *       min + nib*step in fp32 (the reference's dequant value, src/aria_cuda.cu:825-835)
 *       and rounded to fp16.
 *   F16: fp16 weights (the unquantized projections of the DiT, e.g. ca_to_kv).
 * Activations are fp32 (rounded to fp16 when staged) or already fp16 (emitted by the
 * fused norm kernels). Accumulation is fp32 in the MFMA accumulators. Error budget vs
 * the reference's fp32 dequantized GEMM: activation (and Q4 weight) rounding to fp16,
 * ~2^-11 relative per product, a few 1e-4 of max|y|.
 *
 * Tiling: 256 threads = 4 waves in a WGM x WGN grid; each wave owns FM x FN blocks of
 * 32x32 computed with v_mfma_f32_32x32x16_f16 as W x^T (two MFMAs per 32-wide K slice),
 * so a lane's accumulators hold 4 consecutive n of one m. Workgroup tiles run from
 * 64x64 to 192x128 / 128x256 (m x n), picked per shape (pick_tiles).
 * Pipeline: a ring of three register stages holds raw (still packed) slices; the
 * global loads of slice k+3 are issued while slice k is multiplied out of LDS, so each
 * load has two slice-times to land; a slice is unpacked to fp16 only when it is stored
 * to the LDS double buffer (one barrier per slice). Loads past the M / N edge re-read the
 * last row, so the steady-state loop has no branches around its loads.
 * Epilogue: each wave stages 32 x 32*FN fp32 results at a time through LDS and writes
 * whole row segments (16 B per lane, coalesced), applying the Q8 scale, bias and GELU.
 * Operand layout of the 32x32x16 MFMA: lane l supplies row (l % 32) and the 8
 * consecutive k at 8*(l / 32); accumulator register r of lane l holds row
 * 8*(r/4) + 4*(l/32) + r%4, column l % 32.
 *
 * Shapes with K % 32 != 0, N % 4 != 0 or unaligned operands take a SIMT fp32 kernel with
 * the same dequant values (k_qgemm_simt).
 */
#include "qgemm_dev.h"

#define BK 32          /* k per slice */
#define LDS_STRIDE 32  /* halves per LDS row: 64 B, 4 chunks of 8 k */

/* LDS tiles are unpadded [rows][32] halves; chunk c of row r sits at position
 * c ^ ((r >> 2) & 3). The producers write one 16 B chunk per lane, four lanes per row
 * (the order that keeps their global loads coalesced), and the MFMA fragment reads take
 * 32 rows x 2 chunks per instruction: with this swizzle neither pattern has bank
 * conflicts on gfx950 (64 banks, 16 lanes per cycle for 16 B accesses). */
__device__ __forceinline__ int lds_off(int row, int chunk) { return row * LDS_STRIDE + ((chunk ^ ((row >> 2) & 3)) << 3); }
/* producer slot c -> (row, chunk), row-major */
__device__ __forceinline__ int slot_row(int c) { return c >> 2; }
__device__ __forceinline__ int slot_chunk(int c) { return c & 3; }

/* ---- tile configuration: a 2-D grid of WGM x WGN waves, each owning FM x FN 32x32
 * blocks (FM along the activation rows m, FN along the weight rows n) ---- */
template <int FM_, int FN_, int WGM_, int WGN_>
struct Cfg {
    static constexpr int FM = FM_, FN = FN_, WGM = WGM_, WGN = WGN_;
    static constexpr int BM = 32 * FM * WGM, BN = 32 * FN * WGN, NT = 64 * WGM * WGN;
    /* workgroups per CU the register allocation must allow (two waves per SIMD, except
     * the 128-accumulator 128x256 tile, which runs one) */
    static constexpr int MINB = FM * FN >= 8 ? 1 : 2;
    /* epilogue staging: per wave 32 rows x 32*FN fp32, rows padded by 16 B */
    static constexpr int EPI_STRIDE = 32 * FN * 4 + 16;
    static constexpr int TILE_BYTES = 2 * (BM + BN) * LDS_STRIDE * 2, EPI_BYTES = 4 * 32 * EPI_STRIDE;
    static constexpr int LDS_BYTES = TILE_BYTES > EPI_BYTES ? TILE_BYTES : EPI_BYTES;
};

/* per-thread staging of one BK slice in its global encoding; every chunk is 8 k of one
 * row: activations 16 B fp16 or 32 B fp32, weights 8 B int8 (Q8), 4 B nibbles + the
 * block's [min, step] (Q4), 16 B fp16 */
template <class C, int WT, bool AF16>
struct Stage {
    static constexpr int CH = C::BM * (BK / 8), XI = (CH + C::NT - 1) / C::NT, XW = AF16 ? 4 : 8;
    static constexpr int WCH = C::BN * (BK / 8), WI = (WCH + C::NT - 1) / C::NT;
    static constexpr int WW = (WT == ARIA_WQ8) ? 2 : (WT == ARIA_WQ4) ? 3 : 4;
    static_assert(C::BM % 32 == 0 && C::BN % 32 == 0, "tiles are whole MFMA blocks");
    uint32_t x[XI][XW];
    uint32_t w[WI][WW];
};

template <class C, int WT, bool AF16>
struct Tile {
    using S = Stage<C, WT, AF16>;
    const QArgs &q;
    int tid, m0, n0;
    uint16_t *Xs, *Ws;   /* [2][rows * LDS_STRIDE] */

    /* rows past the edge re-read the last row: their products land only in output rows
     * or columns the epilogue never stores, and the branch-free loads keep the vmcnt
     * accounting exact so the prefetch stays in flight */
    __device__ __forceinline__ void load(S &s, int kt) const {
        const int k0 = kt * BK;
#pragma unroll
        for (int i = 0; i < S::XI; i++) {
            const int c = tid + i * C::NT;
            if (S::CH % C::NT != 0 && c >= S::CH) break;
            const int m = min(m0 + slot_row(c), q.M - 1), k = k0 + 8 * slot_chunk(c);
            if (AF16) {
                const uint4 u = *reinterpret_cast<const uint4 *>((const uint16_t *)q.x + (size_t)m * q.K + k);
                s.x[i][0] = u.x; s.x[i][1] = u.y; s.x[i][2] = u.z; s.x[i][3] = u.w;
            } else {
                const uint4 *p = reinterpret_cast<const uint4 *>((const float *)q.x + (size_t)m * q.K + k);
                const uint4 u0 = p[0], u1 = p[1];
                s.x[i][0] = u0.x; s.x[i][1] = u0.y; s.x[i][2] = u0.z; s.x[i][3] = u0.w;
                s.x[i][4] = u1.x; s.x[i][5] = u1.y; s.x[i][6] = u1.z; s.x[i][7] = u1.w;
            }
        }
#pragma unroll
        for (int i = 0; i < S::WI; i++) {
            const int c = tid + i * C::NT;
            if (S::WCH % C::NT != 0 && c >= S::WCH) break;
            const int n = min(n0 + slot_row(c), q.N - 1), k = k0 + 8 * slot_chunk(c);
            if (WT == ARIA_WQ8) {
                const uint2 u = *reinterpret_cast<const uint2 *>((const int8_t *)q.q + (size_t)n * q.K + k);
                s.w[i][0] = u.x; s.w[i][1] = u.y;
            } else if (WT == ARIA_WQ4) {
                s.w[i][0] = *reinterpret_cast<const uint32_t *>((const uint8_t *)q.q + (size_t)n * (q.K >> 1) + (k >> 1));
                const uint2 pr = *reinterpret_cast<const uint2 *>(q.scale + ((size_t)n * q.nblk + (k >> 5)) * 2);
                s.w[i][1] = pr.x; s.w[i][2] = pr.y;
            } else {
                const uint4 u = *reinterpret_cast<const uint4 *>((const uint16_t *)q.q + (size_t)n * q.K + k);
                s.w[i][0] = u.x; s.w[i][1] = u.y; s.w[i][2] = u.z; s.w[i][3] = u.w;
            }
        }
    }

    /* unpack to fp16 and write the slice into LDS buffer buf */
    __device__ __forceinline__ void store(const S &s, int buf) const {
        uint16_t *X = Xs + buf * (C::BM * LDS_STRIDE), *W = Ws + buf * (C::BN * LDS_STRIDE);
#pragma unroll
        for (int i = 0; i < S::XI; i++) {
            const int c = tid + i * C::NT;
            if (S::CH % C::NT != 0 && c >= S::CH) break;
            uint4 o;
            if (AF16) {
                o = make_uint4(s.x[i][0], s.x[i][1], s.x[i][2], s.x[i][3]);
            } else {
                const float *f = reinterpret_cast<const float *>(s.x[i]);
                o = make_uint4(pack2h(f[0], f[1]), pack2h(f[2], f[3]), pack2h(f[4], f[5]), pack2h(f[6], f[7]));
            }
            *reinterpret_cast<uint4 *>(&X[lds_off(slot_row(c), slot_chunk(c))]) = o;
        }
#pragma unroll
        for (int i = 0; i < S::WI; i++) {
            const int c = tid + i * C::NT;
            if (S::WCH % C::NT != 0 && c >= S::WCH) break;
            uint4 o;
            if (WT == ARIA_WQ8) {
                q8x4_to_h(s.w[i][0], o.x, o.y);
                q8x4_to_h(s.w[i][1], o.z, o.w);
            } else if (WT == ARIA_WQ4) {
                /* w = min + nib * step in fp32 (the reference's dequant value), rounded to
                 * fp16; even k in the low nibble */
                const float mn = __builtin_bit_cast(float, s.w[i][1]), st = __builtin_bit_cast(float, s.w[i][2]);
                const uint32_t lo = s.w[i][0] & 0x0F0F0F0Fu, hi = (s.w[i][0] >> 4) & 0x0F0F0F0Fu;
                uint32_t h[4];
#pragma unroll
                for (int e = 0; e < 4; e++)
                    h[e] = pack2h(__builtin_fmaf((float)((lo >> (8 * e)) & 0xFF), st, mn),
                                  __builtin_fmaf((float)((hi >> (8 * e)) & 0xFF), st, mn));
                o = make_uint4(h[0], h[1], h[2], h[3]);
            } else {
                o = make_uint4(s.w[i][0], s.w[i][1], s.w[i][2], s.w[i][3]);
            }
            *reinterpret_cast<uint4 *>(&W[lds_off(slot_row(c), slot_chunk(c))]) = o;
        }
    }
};

template <class C, int WT, bool AF16>
__global__ __launch_bounds__(C::NT, C::MINB) void k_qgemm_mfma(QArgs a, int NTN, int T) {
    using TL = Tile<C, WT, AF16>;
    using S = typename TL::S;
    constexpr int FM = C::FM, FN = C::FN, BM = C::BM, BN = C::BN;
    __shared__ __attribute__((aligned(16))) uint16_t lds[C::LDS_BYTES / 2];
    uint16_t *Xs = lds, *Ws = lds + 2 * BM * LDS_STRIDE;

    const int t = xcd_tile(blockIdx.x, T);
    if (t >= T) return;                     /* uniform per workgroup */
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / C::WGN, wn = wave % C::WGN;
    const TL tl{a, tid, (t / NTN) * BM, (t % NTN) * BN, Xs, Ws};
    const int KT = a.K / BK;

    /* acc[i][j]: the 32x32 block (weight rows j, activation rows i), computed as
     * W x^T so a lane holds 4 consecutive n of one m */
    f32x16_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    const int lrow = lane & 31, lh = lane >> 5;
    auto compute = [&](int buf) {
        const uint16_t *X = Xs + buf * (BM * LDS_STRIDE), *W = Ws + buf * (BN * LDS_STRIDE);
#pragma unroll
        for (int ks = 0; ks < BK / 16; ks++) {
            half8_t xf[FM], wf[FN];
#pragma unroll
            for (int j = 0; j < FN; j++)
                wf[j] = *reinterpret_cast<const half8_t *>(&W[lds_off(wn * 32 * FN + j * 32 + lrow, 2 * ks + lh)]);
#pragma unroll
            for (int i = 0; i < FM; i++)
                xf[i] = *reinterpret_cast<const half8_t *>(&X[lds_off(wm * 32 * FM + i * 32 + lrow, 2 * ks + lh)]);
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[j], xf[i], acc[i][j], 0, 0, 0);
        }
    };

    /* ring of three register stages: at slice kt, stage (kt+1)%3 holds slice kt+1 and
     * stage kt%3 receives slice kt+3. Steady-state steps store and load unconditionally
     * (no path without the loads, so the compiler's vmcnt waits stay exact); the last
     * few steps run the guarded form. */
    S s0, s1, s2;
    tl.load(s0, 0);
    if (KT > 1) tl.load(s1, 1);
    if (KT > 2) tl.load(s2, 2);
    tl.store(s0, 0);
    __syncthreads();
    auto full = [&](int kt, S &nxt, S &fill) {
        compute(kt & 1);
        tl.store(nxt, (kt + 1) & 1);
        tl.load(fill, kt + 3);
        __syncthreads();
    };
    auto step = [&](int kt, S &nxt, S &fill) {
        compute(kt & 1);
        if (kt + 1 < KT) tl.store(nxt, (kt + 1) & 1);
        if (kt + 3 < KT) tl.load(fill, kt + 3);
        __syncthreads();
    };
    int kt = 0;
    for (; kt + 6 <= KT; kt += 3) {
        full(kt, s1, s0);
        full(kt + 1, s2, s1);
        full(kt + 2, s0, s2);
    }
    for (; kt + 3 <= KT; kt += 3) {
        step(kt, s1, s0);
        step(kt + 1, s2, s1);
        step(kt + 2, s0, s2);
    }
    if (kt < KT) step(kt, s1, s0);
    if (kt + 1 < KT) step(kt + 1, s2, s1);

    /* the last slice's barrier has released the tile buffers */
    float *E = reinterpret_cast<float *>(lds) + wave * (32 * C::EPI_STRIDE / 4);
    epilogue<FM, FN, WT, EPI_ANY>(a, acc, E, lane, tl.m0 + wm * 32 * FM, tl.n0 + wn * 32 * FN);
}

/* ---- SIMT fallback: any K, any alignment; fp32 FMA on the dequantized values ---- */
template <int WT>
__device__ __forceinline__ float deq_w(const QArgs &a, int n, int k) {
    if (WT == ARIA_WQ8) return (float)((const int8_t *)a.q)[(size_t)n * a.K + k];
    if (WT == ARIA_WQ4) {
        const size_t rb = (size_t)(a.K + 1) / 2;
        const uint8_t byte = ((const uint8_t *)a.q)[(size_t)n * rb + (k >> 1)];
        const int nib = (k & 1) ? (byte >> 4) : (byte & 0x0F);
        const size_t si = ((size_t)n * a.nblk + k / 32) * 2;
        return a.scale[si] + (float)nib * a.scale[si + 1];
    }
    return (float)__builtin_bit_cast(_Float16, ((const uint16_t *)a.q)[(size_t)n * a.K + k]);
}

template <int WT, bool AF16>
__global__ __launch_bounds__(256) void k_qgemm_simt(QArgs a) {
    __shared__ float As[16][64 + 4];
    __shared__ float Bs[16][64 + 4];
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    const int tid = threadIdx.x, tr = tid / 16, tc = tid % 16;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < a.K; k0 += 16) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int idx = tid + e * 256, r = idx / 16, kk = idx % 16;
            const int gm = m0 + r, gn = n0 + r, gk = k0 + kk;
            float av = 0.0f, bv = 0.0f;
            if (gm < a.M && gk < a.K)
                av = AF16 ? (float)__builtin_bit_cast(_Float16, ((const uint16_t *)a.x)[(size_t)gm * a.K + gk])
                          : ((const float *)a.x)[(size_t)gm * a.K + gk];
            if (gn < a.N && gk < a.K) bv = deq_w<WT>(a, gn, gk);
            As[kk][r] = av;
            Bs[kk][r] = bv;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; kk++)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = __builtin_fmaf(As[kk][tr * 4 + i], Bs[kk][tc * 4 + j], acc[i][j]);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int m = m0 + tr * 4 + i;
        if (m >= a.M) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int n = n0 + tc * 4 + j;
            if (n >= a.N) continue;
            float v = acc[i][j];
            if (WT == ARIA_WQ8) v = v * a.scale[n];
            if (a.bias) v = v + a.bias[n];
            if (a.gelu) v = gelu_tanh_f(v);
            if (a.y_f16) ((uint16_t *)a.y)[(size_t)m * a.N + n] = f2h_bits(v);
            else ((float *)a.y)[(size_t)m * a.N + n] = v;
        }
    }
}

template <class C, int WT, bool AF16>
static void launch_cfg(const QArgs &a, hipStream_t s) {
    const int MT = (a.M + C::BM - 1) / C::BM, NTN = (a.N + C::BN - 1) / C::BN, T = MT * NTN;
    const int grid = ((T + 7) / 8) * 8;
    hipLaunchKernelGGL((k_qgemm_mfma<C, WT, AF16>), dim3(grid), dim3(C::NT), 0, s, a, NTN, T);
}

/* workgroup tiles (activation rows x weight rows), index = the `tiles` argument - 1 */
using C1 = Cfg<3, 2, 2, 2>;   /* 192 x 128 */
using C2 = Cfg<2, 2, 2, 2>;   /* 128 x 128 */
using C3 = Cfg<3, 2, 1, 4>;   /*  96 x 256 */
using C4 = Cfg<3, 1, 1, 4>;   /*  96 x 128 */
using C5 = Cfg<2, 4, 2, 2>;   /* 128 x 256 */
using C6 = Cfg<1, 2, 2, 2>;   /*  64 x 128 */
using C7 = Cfg<2, 1, 2, 2>;   /* 128 x  64 */
using C8 = Cfg<1, 1, 2, 2>;   /*  64 x  64 */
#define NCFG 8
static const int cfg_bm[NCFG] = {192, 128, 96, 96, 128, 64, 128, 64};
static const int cfg_bn[NCFG] = {128, 128, 256, 128, 256, 128, 64, 64};
static const int cfg_fn[NCFG] = {2, 2, 2, 1, 4, 2, 1, 1};   /* 32x32 blocks per wave along n */

/* Tile shape from the shape (measured on MI355X at the DiT's shapes): the largest tile
 * that still gives every CU about two workgroups wins (per-tile efficiency grows with
 * the tile, but a tile count near the CU count leaves CUs idle at the tail); when none
 * does, the one with the most tiles. Order of preference: 192x128, 128x128, 64x128 /
 * 128x64, 64x64. HEADS epilogues need a 64-column head inside one wave (FN >= 2). */
static int pick_tiles(int M, int N, bool heads) {
    static const int order[5] = {0, 1, 5, 6, 7};
    int most = -1;
    long most_t = -1;
    for (int k = 0; k < 5; k++) {
        const int i = order[k];
        if (heads && cfg_fn[i] < 2) continue;   /* a head's 64 columns must sit in one wave */
        const long T = (long)((M + cfg_bm[i] - 1) / cfg_bm[i]) * ((N + cfg_bn[i] - 1) / cfg_bn[i]);
        if (T >= 384) return i;
        if (T > most_t) { most_t = T; most = i; }
    }
    return most;
}

/* Weights-in-registers kernel pick (Q8/Q4, fp16 activations, K % 64 == 0): BM = 32 * FM
 * rows by 256 weight rows per workgroup, FM = 1..4. Cost model fitted to MI355X sweeps of
 * the DiT's GEMMs (M = 2592; N/K = 3072/1024, 1024/1024, 4096/1024, 1024/4096,
 * 8192/1024): rounds of workgroups over 256 CUs (two resident per CU for FM <= 2) times
 * the per-workgroup time, which grows with FM and with the workgroups sharing a CU,
 * scaled by a per-FM efficiency (LDS and L1 traffic per MFMA fall with FM; FM = 4 runs one
 * wave per SIMD and hides less latency). */
static int pick_wr(int M, int N, int K) {
    (void)K;
    static const float eff[5] = {0.0f, 1.6f, 1.25f, 1.1f, 1.35f};
    int best = 2;
    float best_c = 1e30f;
    for (int fm = 1; fm <= 4; fm++) {
        const long T = (long)((M + 32 * fm - 1) / (32 * fm)) * ((N + 255) / 256);
        const int occ = fm <= 2 ? 2 : 1;
        const long rounds = (T + 256L * occ - 1) / (256L * occ);
        const long share = T >= 256 * occ ? occ : (T + 255) / 256;   /* workgroups per CU at once */
        const float c = (float)(rounds * fm * (share < 1 ? 1 : share)) * eff[fm];
        if (c < best_c) { best_c = c; best = fm; }
    }
    return best;
}

/* ---- which kernel and tile: a launch costs about c0 + n (c1 + ck K / 1024) + co M N / 10^6 us, n = the
 * tiles on the busiest of the 256 CUs (co, the output's bytes, only in the second set below). The constants are least-squares fits per configuration to a sweep of
 * M = 40 .. 2592 over the DiT's projections (N / K = 1024 / 1024, 3072 / 1024, 4096 / 1024,
 * 8192 / 1024, 1024 / 4096), each launch alone in a replayed graph over six operand sets; rms
 * error 5-9 %. A candidate displaces the configuration that M = 2592 takes only where it is
 * predicted 8 % faster. Over the sweep the picks run 1.64x (Q8, Q4), 1.24x (fp16), 1.52x (int8),
 * HEADS 1.6-1.9x faster than those configurations in the geometric mean and are within 1-2 % of
 * the fastest of each shape on average (fp16 4 %). Down to two rows of tiles the small tiles of
 * k_qgemm_ks.hip win because they give every CU work; from about M = 860 (N = 8192) to 1420
 * (N = 1024) on, the large tiles' fewer bytes per product do. (fp16 outside HEADS has no fit for
 * the 96 x 64 and the two-per-CU 64 x 64 K-split tiles: of 308 shapes, the decoder's among them, 20 would
 * run 3-20 % faster on one of them than on their pick, none of the decoder's from M = 1836 on.) */
struct TileCost { int pick, bm, bn; float c0, c1, ck, co; };
static const TileCost cost_q8[] = {{GEMM_KS, 32, 32, 1.0f, 1.6f, 1.4f}, {GEMM_KS + 1, 32, 64, 1.2f, 1.7f, 2.0f},
    {GEMM_KS + 2, 64, 64, 1.3f, 3.2f, 2.6f}, {GEMM_KS + 3, 96, 64, 2.0f, 3.9f, 3.2f}, {GEMM_KS + 4, 64, 64, 2.9f, 0.6f, 3.4f},
    {0, 96, 128, 2.5f, 3.4f, 5.5f}, {1, 128, 128, 3.2f, 3.8f, 6.5f}, {4, 224, 128, 8.7f, 6.4f, 6.4f},
    {5, 96, 128, -0.5f, 7.1f, 4.9f}, {7, 192, 256, -4.8f, 14.9f, 14.9f}};
static const TileCost cost_q4[] = {{GEMM_KS, 32, 32, 0.9f, 1.5f, 1.8f}, {GEMM_KS + 1, 32, 64, 1.1f, 1.7f, 2.7f},
    {GEMM_KS + 2, 64, 64, 1.5f, 3.3f, 3.1f}, {GEMM_KS + 3, 96, 64, 1.8f, 3.6f, 4.0f}, {GEMM_KS + 4, 64, 64, 3.4f, 0.0f, 4.6f},
    {0, 96, 128, 3.0f, 2.7f, 7.0f}, {1, 128, 128, 3.2f, 3.4f, 7.9f}, {4, 224, 128, 7.9f, 7.1f, 7.1f},
    {5, 96, 128, -0.3f, 6.9f, 6.3f}, {7, 192, 256, -6.2f, 16.3f, 16.3f}};
static const TileCost cost_f16[] = {{GEMM_KS, 32, 32, 1.1f, 1.6f, 1.5f}, {GEMM_KS + 1, 32, 64, 1.3f, 1.9f, 2.1f},
    {GEMM_KS + 2, 64, 64, 1.3f, 3.0f, 2.8f}, {0, 64, 128, 1.6f, 2.4f, 5.4f}, {1, 96, 128, 4.1f, 0.7f, 8.6f},
    {2, 128, 128, 5.0f, 1.0f, 9.9f}, {3, 160, 128, 6.1f, 0.7f, 11.2f}, {4, 192, 128, 6.8f, 1.6f, 12.0f}};
static const TileCost cost_i8[] = {{GEMM_KS, 32, 32, 1.0f, 1.6f, 0.8f}, {GEMM_KS + 1, 32, 64, 0.9f, 2.2f, 1.1f},
    {GEMM_KS + 2, 64, 64, 0.9f, 3.4f, 1.4f}, {GEMM_KS + 3, 96, 64, 1.4f, 4.1f, 1.9f}, {0, 64, 128, 2.0f, 3.1f, 2.2f},
    {2, 128, 128, 6.0f, 0.2f, 4.9f}, {3, 192, 128, 7.5f, 2.3f, 5.7f}, {4, 96, 128, -0.2f, 6.1f, 3.4f},
    {6, 192, 256, -6.7f, 12.3f, 12.3f}};
/* The same away from that sweep, M > 2592 or K < 512, fitted to K = 64 .. 8192 (M > 2592) and 64 .. 768, N = 64 ..
 * 16384, M up to 12000 (rms error 4-12 %): many tiles of few products are bound by their output, and the
 * constants above took 64 x 64 K-split tiles for them (Q4, M = 8192, K = 128, N = 16384: 117 us as
 * 224 x 128 tiles, 237 so; int8, M = 8192, K = 1024, N = 8192: 138 us as 192 x 128 tiles, 151 as 128 x
 * 128). A candidate has to be predicted 6 % faster; the picks are within 1-2 % of the fastest on average
 * and at most 6 % behind the configuration they displace, 11 % over shapes that were not fitted. Two
 * K-split tiles stay out above M = 2592: 96 x 64 (Q8, M = 5184, K = 1024, N = 256 10.2 -> 12.1 us), and
 * HEADS on any at K < 512 (int8, M = 3000, K = 256, N = 768 8.7 -> 10.5). */
static const TileCost far_q8[] = {{GEMM_KS, 32, 32, 1.59f, 0.99f, 1.62f, 1.09f}, {GEMM_KS + 1, 32, 64, 1.65f, 1.23f, 2.08f, 0.80f},
    {GEMM_KS + 2, 64, 64, 1.61f, 1.72f, 3.97f, 0.61f}, {GEMM_KS + 3, 96, 64, 1.44f, 2.37f, 5.61f, 0.49f},
    {GEMM_KS + 4, 64, 64, 2.78f, 0.29f, 3.99f, 0.61f}, {0, 96, 128, 4.07f, 0.00f, 6.06f, 0.69f}, {1, 128, 128, 4.64f, 0.00f, 7.60f, 0.65f},
    {4, 224, 128, 6.30f, 0.00f, 11.54f, 0.62f}, {5, 96, 128, 2.33f, 1.60f, 6.63f, 0.82f}, {7, 192, 256, 3.36f, 2.25f, 16.72f, 0.63f}};
static const TileCost far_q4[] = {{GEMM_KS, 32, 32, 1.68f, 0.97f, 1.79f, 1.36f}, {GEMM_KS + 1, 32, 64, 1.69f, 1.28f, 2.53f, 0.83f},
    {GEMM_KS + 2, 64, 64, 1.64f, 1.83f, 4.34f, 0.60f}, {GEMM_KS + 3, 96, 64, 1.43f, 2.39f, 5.98f, 0.45f},
    {GEMM_KS + 4, 64, 64, 2.84f, 0.26f, 4.86f, 0.58f}, {0, 96, 128, 3.91f, 0.00f, 7.52f, 0.61f}, {1, 128, 128, 4.32f, 0.00f, 8.90f, 0.59f},
    {4, 224, 128, 5.84f, 0.00f, 12.78f, 0.58f}, {5, 96, 128, 2.37f, 1.38f, 8.16f, 0.77f}, {7, 192, 256, 3.38f, 1.83f, 18.52f, 0.63f}};
static const TileCost far_i8[] = {{GEMM_KS, 32, 32, 1.55f, 1.01f, 0.88f, 1.32f}, {GEMM_KS + 1, 32, 64, 1.67f, 1.22f, 1.18f, 1.03f},
    {GEMM_KS + 2, 64, 64, 1.74f, 1.80f, 2.04f, 0.83f}, {GEMM_KS + 3, 96, 64, 1.78f, 2.20f, 2.94f, 0.75f},
    {0, 64, 128, 3.04f, 0.33f, 2.84f, 0.64f}, {2, 128, 128, 4.52f, 0.00f, 4.31f, 0.69f}, {3, 192, 128, 5.72f, 0.00f, 5.56f, 0.63f},
    {4, 96, 128, 1.87f, 1.91f, 4.07f, 0.74f}, {6, 192, 256, 2.30f, 3.37f, 9.28f, 0.55f}};
/* HEADS (64 columns in one wave; timed at K = 1024 only, N = 1024 and 3072) */
static const TileCost cost_q8_heads[] = {{GEMM_KS + 1, 32, 64, 1.1f, 2.4f, 2.0f}, {GEMM_KS + 3, 96, 64, 2.0f, 5.4f, 3.2f},
    {GEMM_KS + 4, 64, 64, 3.5f, 1.2f, 3.4f}, {6, 64, 256, 1.0f, 8.0f, 6.2f}, {8, 64, 512, 7.7f, 6.0f, 9.4f}};
static const TileCost cost_f16_heads[] = {{GEMM_KS + 1, 32, 64, 1.4f, 2.4f, 2.1f}, {GEMM_KS + 2, 64, 64, 1.3f, 4.1f, 2.8f},
    {GEMM_KS + 3, 96, 64, 1.7f, 5.2f, 3.6f}, {GEMM_KS + 4, 64, 64, 3.5f, 1.4f, 3.6f}};
static const TileCost cost_i8_heads[] = {{GEMM_KS + 1, 32, 64, 0.8f, 2.7f, 1.1f}, {GEMM_KS + 2, 64, 64, 0.9f, 4.3f, 1.4f},
    {GEMM_KS + 3, 96, 64, 1.8f, 5.1f, 1.9f}, {GEMM_KS + 4, 64, 64, 3.4f, 1.5f, 1.9f}, {1, 64, 256, 12.3f, 0.9f, 2.2f},
    {5, 64, 256, 3.0f, 6.2f, 4.0f}};

int qgemm_pick(int wt, bool heads, int M, int N, int K, int cur) {
    struct Table { const TileCost *t; int n; };
#define TBL(x) Table{x, (int)(sizeof x / sizeof x[0])}
    const bool far = !heads && wt != ARIA_WF16 && (M > 2592 || K < 512);
    const Table tb = far ? (wt == ARIA_WI8 ? TBL(far_i8) : wt == ARIA_WQ4 ? TBL(far_q4) : TBL(far_q8))
                   : wt == ARIA_WI8 ? (heads ? TBL(cost_i8_heads) : TBL(cost_i8))
                   : wt == ARIA_WF16 ? (heads ? TBL(cost_f16_heads) : TBL(cost_f16))
                   : heads ? TBL(cost_q8_heads) : wt == ARIA_WQ4 ? TBL(cost_q4) : TBL(cost_q8);
#undef TBL
    const float k = (float)K / 1024.0f;
    auto us = [&](const TileCost &c) {
        const long T = (long)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
        return c.c0 + (float)((T + 255) / 256) * (c.c1 + c.ck * k) + c.co * ((float)M * (float)N * 1e-6f);
    };
    /* fp16 HEADS runs on the LDS-operand kernel otherwise: K = 1024 13.4 us at N = 1024 up to M = 1836, 14 ->
     * 31 us at N = 3072 from M = 600 to 2592; K = 2048, N = 2048 20.4 us at M = 432, 32.4 at M = 1836 */
    float cur_us = wt == ARIA_WF16 && heads ? 3.4f + k * (8.6f + 2.5e-6f * (float)M * (float)N) : 1e30f;
    for (int i = 0; i < tb.n; i++)
        if (tb.t[i].pick == cur) cur_us = us(tb.t[i]);
    int best = cur;
    float best_us = (far ? 0.94f : 0.92f) * cur_us;
    const int steps = K / (wt == ARIA_WI8 ? 128 : 64);
    for (int i = 0; i < tb.n; i++) {
        const TileCost &c = tb.t[i];
        /* only the K-split kernel and the large-tile configurations whose K is unsplit or even */
        const bool split = c.pick < GEMM_KS && (wt == ARIA_WI8 ? c.pick == 4 || c.pick == 5 : wt != ARIA_WF16 && (c.pick == 5 || c.pick == 6));
        if ((split && steps % 2) || (wt == ARIA_WF16 && c.pick < GEMM_KS) || (M > 2592 && (heads ? c.pick >= GEMM_KS && K < 512 : far && c.pick == GEMM_KS + 3))) continue;
        const float t = us(c);
        if (t < best_us) { best_us = t; best = c.pick; }
    }
    return best;
}

static bool qgemm_aligned(const QArgs &a, int wt) {
    return a.K % BK == 0 && a.N % 4 == 0 && ((uintptr_t)a.x & 15u) == 0 && ((uintptr_t)a.q & 15u) == 0 &&
           ((uintptr_t)a.y & 15u) == 0 && (a.bias == nullptr || ((uintptr_t)a.bias & 15u) == 0) &&
           (wt != ARIA_WQ8 || ((uintptr_t)a.scale & 15u) == 0) && (wt != ARIA_WQ4 || ((uintptr_t)a.scale & 7u) == 0);
}

/* the output and the activations (xb bytes each) share memory */
static bool qgemm_overlaps(const QArgs &a, int xb) {
    const uintptr_t x0 = (uintptr_t)a.x, y0 = (uintptr_t)a.y;
    return x0 < y0 + (size_t)a.M * a.N * (a.y_f16 ? 2 : 4) && y0 < x0 + (size_t)a.M * a.K * xb;
}

/* fp32 activations straight into the K-split kernel: its configuration (the first of 32 x 32, 32 x 64
 * and 64 x 64 whose tiles fit one round of the 256 CUs), or -1. It reads twice the activation bytes
 * per tile, and saves the staging pass (a launch of 3 us and one more dependent kernel) or, where
 * there is none, the 128 x 128 tiles of the LDS-operand kernel (few workgroups, each a serial chain
 * of K / 32 slices). Measured in us, fp16 weights, (M, K, N), staged / LDS-operand / direct:
 * (172, 1024, 1024) 6.9 / 16.7 / 4.9; (1024, 1024, 1024) 11.5 / 17.4 / 10.2; (256, 1024, 3072)
 * 10.2 / 17.3 / 9.0; (108, 256, 1024) 5.3 / 7.4 / 3.2; (1292, 1024, 256) 9.4 / 17.1 / 7.4. Past one
 * round it loses ((344, 1024, 3072) 12.6 / 17.3 / 14.8), and so it does on long chains: at K = 4096
 * (172, 4096, 1024) 11.4 / 49.0 / 11.9, so the line is drawn at twice the K that gains 2 us.
 * An output that overlaps the activations keeps the staging pass: its copy is what lets one
 * workgroup store rows that another has yet to read. */
static int qgemm_f32_pick(const QArgs &a, int wt) {
    if (a.K % 64 || a.K > 2048 || !qgemm_aligned(a, wt) || (wt == ARIA_WQ4 && ((uintptr_t)a.scale & 15u))) return -1;
    if (qgemm_overlaps(a, 4)) return -1;
    const long long m32 = (a.M + 31) / 32, m64 = (a.M + 63) / 64, n32 = (a.N + 31) / 32, n64 = (a.N + 63) / 64;
    return m32 * n32 <= 256 ? 0 : m32 * n64 <= 256 ? 1 : m64 * n64 <= 256 ? 2 : -1;
}

extern "C" int aria_k_qgemm_f32_direct(const void *y, int y_f16, const void *x, int wtype, const void *q, const float *scale,
                                       const float *bias, int M, int K, int N) {
    QArgs a;
    memset(&a, 0, sizeof a);
    a.y = (void *)y; a.y_f16 = y_f16; a.x = x; a.q = q; a.scale = scale; a.bias = bias; a.M = M; a.K = K; a.N = N;
    return qgemm_f32_pick(a, wtype) >= 0;
}

/* The kernel for fp16 activations with no tile asked for: a k_qgemm_big.hip configuration, GEMM_KS + a
 * k_qgemm_ks.hip one, or -1 (the kernels below). The k_qgemm_big.hip configurations at M = 2592, from
 * which qgemm_pick starts: N <= 1024 without HEADS (96 x 128
 * tiles, two workgroups per CU), HEADS with N <= 3072 (the qkv projection: 64 x 512 in
 * 8-wave workgroups, one per CU), other N <= 3072 without HEADS (128 x 128, two per CU), N = 4096
 * (192 x 256 in 8-wave workgroups, one per CU) and wider (224 x 128); N <= 1024 with an
 * even number of K-tiles in 96 x 128
 * tiles of 8 waves, the two halves of K on their own pipelines (216 tiles at M = 2592
 * leave 40 CUs idle; the split doubles the waves on the busy ones), and HEADS with N <=
 * 1024 (ca_q) likewise in 64 x 256 tiles (164 tiles: one workgroup per busy CU, so the
 * split's second half is what gives those CUs two waves per SIMD; 15.6 -> 15.2 us);
 * HEADS wider than 3072 stays on the weights-in-registers kernel. fp16 weights: qgemm_big_f16_pick's,
 * and for HEADS, which needs 64 columns per wave, the LDS-operand kernel where qgemm_pick finds none.
 * An output over the activations (fp16, in place: K = N) keeps them: up to N = 128 a tile has whole
 * rows there, read to the end before the first is stored, where one of several narrower tiles would
 * store what the next has yet to read. */
static int qgemm_route(const QArgs &a, int wt) {
    if (a.K % 64 || (a.gelu && a.epi.mode != ARIA_EPI_STORE) || (wt == ARIA_WQ4 && ((uintptr_t)a.scale & 15u))) return -1;
    const bool heads = a.epi.mode == ARIA_EPI_HEADS, even = (a.K / 64) % 2 == 0;
    const int cur = wt == ARIA_WF16 ? (heads ? -1 : qgemm_big_f16_pick(a.M, a.N))
                  : heads ? (a.N <= 1024 && even ? 6 : a.N <= 3072 ? 8 : -1)
                  : a.N <= 1024 ? (even ? 5 : 0) : a.N <= 3072 ? 1 : a.N <= 4096 ? 7 : 4;
    if (cur < 0 && wt != ARIA_WF16) return -1;
    if (a.epi.mode == ARIA_EPI_STORE && qgemm_overlaps(a, 2)) return cur;
    return qgemm_pick(wt, heads, a.M, a.N, a.K, cur);
}

extern "C" int aria_k_qgemm_route(const void *y, int y_f16, const void *x, int wtype, const void *q, const float *scale,
                                  const float *bias, int M, int K, int N) {
    QArgs a;
    memset(&a, 0, sizeof a);
    a.y = (void *)y; a.y_f16 = y_f16; a.x = x; a.q = q; a.scale = scale; a.bias = bias; a.M = M; a.K = K; a.N = N;
    a.epi.mode = ARIA_EPI_STORE;
    return qgemm_aligned(a, wtype) ? qgemm_route(a, wtype) : -1;
}

template <int WT, bool AF16>
static hipError_t launch_q(const QArgs &a, int tiles, hipStream_t s) {
    if (!qgemm_aligned(a, WT)) {
        if (a.epi.mode != ARIA_EPI_STORE) return hipErrorInvalidValue;   /* fused epilogues need the MFMA path */
        dim3 grid((a.N + 63) / 64, (a.M + 63) / 64);
        hipLaunchKernelGGL((k_qgemm_simt<WT, AF16>), grid, dim3(256), 0, s, a);
        return hipGetLastError();
    }
    if constexpr (!AF16) {   /* fp32 activations: the K-split kernel where it takes them as they are, else (no
                              * fp16 staging buffer, or none used: the step's io projections) 128 x 128 tiles */
        if (a.epi.mode == ARIA_EPI_HEADS) return hipErrorInvalidValue;
        if (tiles >= GEMM_KS) return qgemm_ks_f32_launch(a, WT, tiles - GEMM_KS, s);
        const bool plain = !a.gelu && (a.epi.mode == ARIA_EPI_STORE || a.epi.mode == ARIA_EPI_ADD);
        const int c = tiles == 0 && plain ? qgemm_f32_pick(a, WT) : -1;
        if (c >= 0) return qgemm_ks_f32_launch(a, WT, c, s);
        launch_cfg<C2, WT, AF16>(a, s);
        return hipGetLastError();
    } else {
    if (tiles >= GEMM_KS) return qgemm_ks_launch(a, WT, tiles - GEMM_KS, s);   /* explicit: configuration tiles - GEMM_KS */
    if (tiles >= 13) return qgemm_big_launch(a, WT, tiles - 13, s);   /* likewise: k_qgemm_big.hip's tiles - 13 */
    if (tiles == 0) {
        const int c = qgemm_route(a, WT);
        if (c >= GEMM_KS) return qgemm_ks_launch(a, WT, c - GEMM_KS, s);
        if (c >= 0) return qgemm_big_launch(a, WT, c, s);
    }
    if constexpr (WT != ARIA_WF16) {
        /* weights-in-registers kernel: explicit tiles 9..12 (BM = 32 * (tiles - 8)), or the pick */
        int fm = (tiles > NCFG) ? tiles - NCFG : (tiles == 0 ? pick_wr(a.M, a.N, a.K) : 0);
        /* Q8 with N and K <= 1024 (the DiT's sa_out / ca_out): 64 x 64 LDS-operand tiles, 2.5
         * workgroups per CU, measured 8 % faster than the weights-in-registers pick */
        if (tiles == 0 && WT == ARIA_WQ8 && a.N <= 1024 && a.K <= 1024 && a.epi.mode != ARIA_EPI_HEADS) fm = 0;
        const bool wr_ok = a.K % 64 == 0 && (!a.gelu || a.epi.mode == ARIA_EPI_STORE);
        if (fm > 0 && wr_ok) return qgemm_wr_launch(a, WT, fm, s);
        if (tiles == 0 && fm == 0 && WT == ARIA_WQ8 && a.N <= 1024 && a.K <= 1024 && a.epi.mode != ARIA_EPI_HEADS) {
            launch_cfg<C8, WT, AF16>(a, s);
            return hipGetLastError();
        }
    }
    int c = (tiles >= 1 && tiles <= NCFG) ? tiles - 1 : pick_tiles(a.M, a.N, a.epi.mode == ARIA_EPI_HEADS);
    if (a.epi.mode == ARIA_EPI_HEADS && cfg_fn[c] < 2) c = pick_tiles(a.M, a.N, true);
    switch (c) {
        case 0: launch_cfg<C1, WT, AF16>(a, s); break;
        case 1: launch_cfg<C2, WT, AF16>(a, s); break;
        case 2: launch_cfg<C3, WT, AF16>(a, s); break;
        case 3: launch_cfg<C4, WT, AF16>(a, s); break;
        case 4: launch_cfg<C5, WT, AF16>(a, s); break;
        case 5: launch_cfg<C6, WT, AF16>(a, s); break;
        case 6: launch_cfg<C7, WT, AF16>(a, s); break;
        default: launch_cfg<C8, WT, AF16>(a, s); break;
    }
    return hipGetLastError();
    }
}

extern "C" hipError_t aria_k_qgemm_e(void *y, int y_f16, const void *x, int x_f16, int wtype, const void *q,
                                     const float *scale, const float *bias, int M, int K, int N, int tiles,
                                     int gelu, const aria_qgemm_epi *epi, hipStream_t s) {
    if (M <= 0 || N <= 0) return hipSuccess;
    QArgs a;
    a.y = y; a.x = x; a.q = q; a.scale = scale; a.bias = bias;
    a.M = M; a.K = K; a.N = N; a.y_f16 = y_f16; a.nblk = (K + 31) / 32; a.gelu = gelu;
    a.xscale = nullptr;
    if (epi) a.epi = *epi;
    else { memset(&a.epi, 0, sizeof a.epi); a.epi.mode = ARIA_EPI_STORE; }
    if (a.epi.mode == ARIA_EPI_HEADS) {
        if (N % 64 || a.epi.nsec < 1 || a.epi.nsec > 3 || a.epi.heads * 64 * a.epi.nsec != N ||
            a.epi.rows_per_batch <= 0 || (a.epi.rot && (a.epi.rot > 64 || (a.epi.rot & 7)))) return hipErrorInvalidValue;
        a.y = (void *)a.epi.dst[0];   /* alignment check only; y is not written */
    } else if (a.epi.mode == ARIA_EPI_GLU) {
        if (N % 4 || a.gelu) return hipErrorInvalidValue;
    } else if (a.epi.mode == ARIA_EPI_ADD_DYT) {   /* the decoder's fp16-weight GEMMs only */
        if (wtype != ARIA_WF16 || !x_f16 || y_f16 || a.gelu || a.epi.rows_per_batch <= 0 || !a.epi.dst[0] ||
            !a.epi.w[0] || !a.epi.w[1] || ((uintptr_t)a.epi.dst[0] & 7u) || ((uintptr_t)a.epi.w[0] & 15u) ||
            ((uintptr_t)a.epi.w[1] & 15u))
            return hipErrorInvalidValue;
    } else if (a.epi.mode == ARIA_EPI_DYT_ROPE) {   /* the decoder's to_qkv only */
        const aria_qgemm_epi &e = a.epi;
        const int rot = e.rot;
        bool ok = wtype == ARIA_WF16 && x_f16 && !y_f16 && !a.gelu && e.heads > 0 && N == 5 * 64 * e.heads &&
                  e.rows_per_batch > 0 && (rot == 0 || rot == 8 || rot == 16 || rot == 32);
        for (int i = 0; ok && i < 4; i++) ok = e.w[i] && ((uintptr_t)e.w[i] & 15u) == 0;
        if (ok && rot) ok = e.cos_t && e.sin_t && ((uintptr_t)e.cos_t & 15u) == 0 && ((uintptr_t)e.sin_t & 15u) == 0;
        if (!ok) return hipErrorInvalidValue;
    } else if (a.epi.mode > ARIA_EPI_DYT_ROPE || a.epi.mode < 0) {
        return hipErrorInvalidValue;
    } else if (a.epi.mode != ARIA_EPI_STORE) {
        if (y_f16 || a.epi.rows_per_batch <= 0) return hipErrorInvalidValue;
    }
    if (wtype == ARIA_WQ8) return x_f16 ? launch_q<ARIA_WQ8, true>(a, tiles, s) : launch_q<ARIA_WQ8, false>(a, tiles, s);
    if (wtype == ARIA_WQ4) return x_f16 ? launch_q<ARIA_WQ4, true>(a, tiles, s) : launch_q<ARIA_WQ4, false>(a, tiles, s);
    if (wtype == ARIA_WF16)
        return x_f16 ? launch_q<ARIA_WF16, true>(a, tiles, s) : launch_q<ARIA_WF16, false>(a, tiles, s);
    return hipErrorInvalidValue;
}

extern "C" hipError_t aria_k_qgemm_t(void *y, int y_f16, const void *x, int x_f16, int wtype, const void *q,
                                     const float *scale, const float *bias, int M, int K, int N, int tiles,
                                     int gelu, hipStream_t s) {
    return aria_k_qgemm_e(y, y_f16, x, x_f16, wtype, q, scale, bias, M, K, N, tiles, gelu, nullptr, s);
}

extern "C" hipError_t aria_k_qgemm(void *y, int y_f16, const void *x, int x_f16, int wtype, const void *q,
                                   const float *scale, const float *bias, int M, int K, int N, hipStream_t s) {
    return aria_k_qgemm_t(y, y_f16, x, x_f16, wtype, q, scale, bias, M, K, N, 0, 0, s);
}
