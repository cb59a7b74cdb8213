/*
 * k_dec.hip - the small-music autoencoder decoder's glue and attention on gfx950.
 *
 * Replaces the per-op CPU loops of the reference's taae_v2 decoder (src/aria_sa3_dec.c:
 * aria_sa3_same_decode and aria_unpatch_stereo, lines 47-116; src/aria_taae.c:
 * taae_block_forward, lines 93-162) around the GEMMs, which run on the dequant GEMM
 * kernels with fp16 weights:
 *   k_dec_in      softnorm inverse and transpose: latent [256, T] * std -> fp16 [T, 256]
 *   k_dec_expand  the 17-token groups: frame t's projected token, then 16 new_tokens
 *   k_dec_dyt     DynamicTanh norm tanh(alpha x) * gamma + beta -> fp16 GEMM operand
 *   k_dec_attn_mfma  one chunk-head of the differential self-attention, fused: the
 *                 difference of two softmax(q k^T / 8) over the chunk's 34 tokens, times v,
 *                 on the fp32 MFMA, merged fp16 (the q/k DynamicTanh norms and RoPE, 32
 *                 rotated dims, are the to_qkv GEMM's DYT_ROPE epilogue)
 *   k_dec_split   the k = 3 mapping convolution's input rows (the last 16 of each group), every
 *                 value split into three bf16 parts
 *   k_dec_map     the mapping convolution at fp32 precision on the bf16 MFMA (the reference
 *                 keeps it fp32), trimmed to T * 16 rows and unpatched to stereo in its stores
 * Arithmetic follows the reference's order (built with -ffp-contract=off). tanh: block 0's pre
 * norm (k_dec_dyt) uses the device library's tanhf; the other 11 block norms (the ADD_DYT
 * epilogue of to_out / ff_out) and the q/k norms (the DYT_ROPE epilogue of to_qkv) use
 * tanh_fast (exp + rcp, a few 1e-7 absolute, before the fp16 rounding of the GEMM operand);
 * the softmax exponential is v_exp_f32 (~1 ulp).
 */
#include "qgemm_dev.h"   /* dma16, wait_vm */

#define DEC_D 768
#define DEC_S 34
#define DEC_HD 64
#define DEC_QKV 3840

/* xt[t][c] = half(latent[c][t] * std): 64 x 4 tiles through LDS (coalesced on both sides) */
__global__ __launch_bounds__(256) void k_dec_in(uint16_t *xt, const float *lat, int T, float std) {
    __shared__ float tile[64][65];
    const int t0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int r = ty; r < 64; r += 4) {
        const int c = c0 + r, t = t0 + tx;
        tile[r][tx] = (t < T) ? lat[(size_t)c * T + t] * std : 0.0f;
    }
    __syncthreads();
    for (int r = ty; r < 64; r += 4) {
        const int t = t0 + r;
        if (t < T) xt[(size_t)t * 256 + c0 + tx] = f2h_bits(tile[tx][r]);
    }
}

/* seq[r] for r < Tp * 17: group t = r / 17, slot j = r % 17; slot 0 is x[t] (zeros for the
 * padding frame t >= T), slots 1..16 the learned new_tokens (src/aria_sa3_dec.c:69-77) */
__global__ __launch_bounds__(256) void k_dec_expand(float4 *seq, const float4 *x, const float4 *tok, int T, int Tp) {
    const size_t n = (size_t)Tp * 17 * (DEC_D / 4);
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const int r = (int)(i / (DEC_D / 4)), c = (int)(i % (DEC_D / 4));
        const int t = r / 17, j = r % 17;
        float4 v;
        if (j) v = tok[c];
        else v = (t < T) ? x[(size_t)t * (DEC_D / 4) + c] : make_float4(0.f, 0.f, 0.f, 0.f);
        seq[i] = v;
    }
}

/* y = half(tanhf(alpha * x) * g + b) over [rows, 768], as aria_dynamic_tanh
 * (src/aria_cpu.c:684-698) */
__global__ __launch_bounds__(256) void k_dec_dyt(uint2 *y, const float4 *x, float alpha, const float4 *g,
                                                 const float4 *b, size_t n4) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % (DEC_D / 4));
        const float4 v = x[i], gg = g[c], bb = b[c];
        float o0 = tanhf(alpha * v.x), o1 = tanhf(alpha * v.y), o2 = tanhf(alpha * v.z), o3 = tanhf(alpha * v.w);
        o0 = o0 * gg.x + bb.x; o1 = o1 * gg.y + bb.y; o2 = o2 * gg.z + bb.z; o3 = o3 * gg.w + bb.w;
        y[i] = make_uint2((uint32_t)f2h_bits(o0) | ((uint32_t)f2h_bits(o1) << 16),
                          (uint32_t)f2h_bits(o2) | ((uint32_t)f2h_bits(o3) << 16));
    }
}

struct DecAttnArgs {
    uint16_t *merged;           /* [nch * 34, 768] fp16 */
    const float *qkv;           /* [nch * 34, 3840]: q | k | v | qd | kd, q / k normed and rotated */
};

/* ---- the chunk attention on the fp32 MFMA (v_mfma_f32_16x16x4_f32) ----
 * One (chunk, head) per workgroup of three waves; wave w computes the 16 queries of block w of
 * the chunk's 34 tokens (padded to 48) for both pairs (q, k and qd, kd). The q / k sections of
 * qkv arrive DynamicTanh-normed and rotated (the to_qkv GEMM's DYT_ROPE epilogue).
 *   k, kd and v (34 rows of 256 B each) travel to LDS by LDS DMA first thing, in whole rows; the
 *     16-byte chunk c of LDS row R sits at slot c ^ (R % 16), so 16 lanes that read one chunk of
 *     16 rows, or one whole row, meet no bank twice
 *   S^T = k q^T (keys are the rows): lane l supplies key row l % 16 (A) and query l % 16 (B) at
 *     dims 16 j + 4 (l / 16) + e in step (j, e), so 16-byte reads feed four steps, and query l %
 *     16's scores of keys 16 b + 4 (l / 16) + v end up in the accumulators of its four lanes: the
 *     softmax is 9 values a lane and two lane swaps, and a probability is already where the second
 *     product wants it (k = l / 16, column l % 16), with no pass through LDS
 *   O = (P0 - P1) v, one product for the two pairs' difference: O^T = v^T D^T, step (b, v) over
 *     keys 16 b + 4 (l / 16) + v; output block j row m holds dim 4 m + j, so a lane's A operands
 *     of a step are one 16-byte read of v and its 16 outputs are dims 16 (l / 16) .. of one query
 *   keys 32 and 33 would fill two of 16 rows of a third block: their scores are summed on the VALU
 *     (each lane its 16 dims, then over the four lanes), and in the second product they share one
 *     step (lq 0 and 1)
 * Memory bounds it at T = 646: 168 MB of fp32 qkv and 17 MB of output are 38 us at the rate of a
 * large copy. One wave per (pair, query block) with k and P through LDS, two products and scattered
 * 16-byte loads took 69 us there (576 MFMAs a workgroup, 300 now) and 16.5 us at T = 108; this form
 * 44 and 12.3 (46.5 and 13.4 with a third key block on the MFMA). Relative error against float64 is
 * the fp16 output's, 2.07e-4 before and now.
 * fp32 operands, as the reference keeps this attention fp32. */
#define DA_WAVES 3
#define DA_ROWS (3 * DEC_S)                       /* k, kd, v */
#define DA_DMA ((DA_ROWS * 16 + 63) / 64)         /* transfers of 64 16-byte chunks */

typedef float f32x4_dec __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) float4 lds_f4_dec;

/* over the four lanes l % 16 + {0, 16, 32, 48} */
template <typename Op>
__device__ __forceinline__ float dec_quad(float v, Op op) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned a = r[0], b = r[1];
    const float w = op(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
    const unsigned u2 = __builtin_bit_cast(unsigned, w);
    const auto t = __builtin_amdgcn_permlane32_swap(u2, u2, false, false);
    const unsigned c = t[0], d = t[1];
    return op(__builtin_bit_cast(float, c), __builtin_bit_cast(float, d));
}

__global__ __launch_bounds__(64 * DA_WAVES) void k_dec_attn_mfma(DecAttnArgs a, int H) {
    __shared__ __attribute__((aligned(16))) float4 sm[DA_DMA * 64];
    const int ch = blockIdx.x / H, h = blockIdx.x % H;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int lr = lane & 15, lq = lane >> 4;
    const float *base = a.qkv + (size_t)ch * DEC_S * DEC_QKV + h * DEC_HD;

    /* transfer i fills slots 64 i ..; slots past the last row re-read it */
    for (int i = wave; i < DA_DMA; i += DA_WAVES) {
        const int p = 64 * i + lane, R = min(p >> 4, DA_ROWS - 1);
        const int sec = R >= 2 * DEC_S ? 2 : R >= DEC_S;
        const float *src = base + (size_t)(R - sec * DEC_S) * DEC_QKV + (sec == 2 ? 1536 : sec ? 3072 : 768);
        dma16(src + 4 * ((p ^ R) & 15), (uint32_t)(uintptr_t)(lds_f4_dec *)sm + 1024 * i);
    }
    /* the wave's query (rows past the chunk repeat the last one; they are not stored) */
    const int qrow = 16 * wave + lr;
    float4 qf[2][4];
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const float *row = base + (size_t)min(qrow, DEC_S - 1) * DEC_QKV + (p ? 2304 : 0) + 4 * lq;
#pragma unroll
        for (int j = 0; j < 4; j++) qf[p][j] = *reinterpret_cast<const float4 *>(row + 16 * j);
    }
    wait_vm<0>();
    __syncthreads();   /* k, kd and v in LDS */

    f32x4_dec sc[2][2];
    float st[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};   /* keys 32 and 33: this lane's dims */
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int b = 0; b < 2; b++) sc[p][b] = f32x4_dec{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float4 kf[2][2], kt[2][2];
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const int R = p * DEC_S + 16 * b + lr, Rt = p * DEC_S + 32 + b;
                kf[p][b] = sm[R * 16 + (((4 * j + lq) ^ R) & 15)];
                kt[p][b] = sm[Rt * 16 + (((4 * j + lq) ^ Rt) & 15)];
            }
#define DA_STEP(c)                                                                                            \
        _Pragma("unroll") for (int p = 0; p < 2; p++)                                                         \
            _Pragma("unroll") for (int b = 0; b < 2; b++)                                                     \
                st[p][b] = __builtin_fmaf(kt[p][b].c, qf[p][j].c, st[p][b]),                                  \
                sc[p][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[p][b].c, qf[p][j].c, sc[p][b], 0, 0, 0);
        DA_STEP(x) DA_STEP(y) DA_STEP(z) DA_STEP(w)
#undef DA_STEP
    }

    /* softmax over the 34 keys: eight in the accumulators, the last two as a ninth value of lq 0 and 1 */
    float D[9];
#pragma unroll
    for (int p = 0; p < 2; p++) {
        float x[9];
#pragma unroll
        for (int i = 0; i < 8; i++) { const float t = sc[p][i >> 2][i & 3]; x[i] = t * 0.125f; }
        const float t0 = dec_quad(st[p][0], OpSum()), t1 = dec_quad(st[p][1], OpSum());
        x[8] = lq < 2 ? (lq ? t1 : t0) * 0.125f : -INFINITY;
        float mx = x[0], sum = 0.0f;
#pragma unroll
        for (int i = 1; i < 9; i++) mx = fmaxf(mx, x[i]);
        mx = dec_quad(mx, OpMax());
#pragma unroll
        for (int i = 0; i < 9; i++) { x[i] = exp_fast(x[i] - mx); sum += x[i]; }
        sum = dec_quad(sum, OpSum());
        const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
#pragma unroll
        for (int i = 0; i < 9; i++) D[i] = p ? D[i] - x[i] * inv : x[i] * inv;
    }

    f32x4_dec oc[4];
#pragma unroll
    for (int j = 0; j < 4; j++) oc[j] = f32x4_dec{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 9; i++) {
        const int R = 2 * DEC_S + (i < 8 ? 16 * (i >> 2) + 4 * lq + (i & 3) : 32 + min(lq, 1));
        const float4 v = sm[R * 16 + ((lr ^ R) & 15)];
        oc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.x, D[i], oc[0], 0, 0, 0);
        oc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.y, D[i], oc[1], 0, 0, 0);
        oc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.z, D[i], oc[2], 0, 0, 0);
        oc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.w, D[i], oc[3], 0, 0, 0);
    }
    if (qrow < DEC_S) {
        uint4 *dst = reinterpret_cast<uint4 *>(a.merged + ((size_t)ch * DEC_S + qrow) * DEC_D + h * DEC_HD + 16 * lq);
        uint32_t w[8];
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
                /* a value that is not finite is NaN, as the difference of two such products is */
                const float o0 = oc[j][v], o1 = oc[j + 1][v];
                w[2 * v + j / 2] = (uint32_t)f2h_bits(o0 + (o0 - o0)) | ((uint32_t)f2h_bits(o1 + (o1 - o1)) << 16);
            }
        dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
        dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
    }
}

/* ---- the mapping convolution on the bf16 matrix cores, at fp32 precision ----
 * audio[n / 256][m * 256 + n % 256] = sum over taps j < 3, i < 768 of feat[m + j - 1][i] W[n][i][j]
 * + b[n], m < M = T * 16, n < 512 (src/aria_sa3_dec.c:85-116: the k = 3 convolution over the last
 * 16 rows of each 17-row group, the trim and aria_unpatch_stereo). Feature position p is seq row
 * (p / 16) * 17 + 1 + p % 16.
 * The reference keeps this product in fp32. The fp32 MFMA runs at a sixteenth of the bf16 rate
 * and bound it (at T = 646 234 us, and 31 for the im2col before it), so every fp32 operand is split
 * into three bf16 parts, x = x0 + x1 + x2, each the nearest one to what the parts before it left (the
 * method of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype for
 * Higher-Precision Computations", ARITH 2019): 24 bits in all, so the split is exact down to bf16's
 * last bit, 2^-133. x y is then the six products x_i y_j with i + j <= 2; as |x1| <= 2^-8 |x| and
 * |x2| <= 2^-17 |x|, the three left out are at most 2^-24 (1 + 2^-10) of x y, of either sign (parts cut
 * off instead of rounded leave out up to 2^-21, always with the product's sign). x0 y0 has an
 * accumulator of its own and the five small products another, which is added at the end, so the
 * large sum is rounded 144 times (once per MFMA) where the fp32 MFMA rounded it 1152 times.
 * A non-finite operand keeps its class: the parts after x0 are zero, and a sum whose large part is
 * not finite is that part alone (also one within 2^-7 of the largest float: x0 y0 can exceed x y).
 * Relative error against float64, T = 1 .. 646 and values scaled by 1e-4 .. 300: 2.0-2.9e-7 where the
 * fp32 MFMA had 6.1-8.6e-7; where one product makes up the sum, 1.0e-7 at most (4.7e-7 with parts cut
 * off). Time alone, the input pass (im2col before, the split now) + the product: T = 108 8 + 56 -> 4 +
 * 32 us, T = 300 16 + 124 -> 6 + 78, T = 646 31 + 234 -> 13 + 125.
 *
 * Layout: a row of 32-k blocks, 192 bytes each: the three parts of the block's 32 values, 64 bytes
 * a part. Features sit in rows 1 .. of xs (row 0 and the row past the end are the convolution's
 * zeros), 24 blocks = 4608 bytes a row, and W's k index is 768 j + i: an output row's 72 blocks
 * are then three consecutive feature rows, 13824 contiguous bytes, and the convolution is one
 * product over overlapping rows with nothing gathered. */
#define MAP_KB 72                   /* 32-k blocks of an output row (2304 k) */
#define MAP_BB 192                  /* bytes of a block: 3 parts x 32 bf16 */
#define MAP_XROW (24 * MAP_BB)      /* bytes of a feature row */
#define MAP_N 512

/* bf16 nearest to the finite value of these bits (ties to even) */
__device__ __forceinline__ uint32_t bf16_rn(uint32_t u) { return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16; }

/* the three bf16 parts of x, as bits; the remainders are exact in fp32 */
__device__ __forceinline__ void bf16x3(float x, uint32_t (&p)[3]) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    p[0] = u >> 16;
    p[1] = p[2] = 0;
    if ((u & 0x7F800000u) == 0x7F800000u) {
        if (u & 0x007FFFFFu) p[0] |= 0x0040u;   /* a NaN stays one without its low bits */
        return;
    }
    const uint32_t n = bf16_rn(u);
    if ((n & 0x7F80u) != 0x7F80u) p[0] = n;     /* a value that would round to infinity stays truncated */
    const float r = x - __builtin_bit_cast(float, p[0] << 16);
    p[1] = bf16_rn(__builtin_bit_cast(uint32_t, r));
    p[2] = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, p[1] << 16)) >> 16;
}

/* eight values -> a 16-byte chunk of each part */
__device__ __forceinline__ void bf16x3_store(uint8_t *d, const float (&f)[8]) {
    uint32_t w[3][4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        uint32_t a[3], b[3];
        bf16x3(f[2 * e], a);
        bf16x3(f[2 * e + 1], b);
#pragma unroll
        for (int p = 0; p < 3; p++) w[p][e] = a[p] | (b[p] << 16);
    }
#pragma unroll
    for (int p = 0; p < 3; p++) *reinterpret_cast<uint4 *>(d + 64 * p) = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
}

/* the split features, rows 0 .. Lt + 1: row r = feature position r - 1, zero outside [0, Lout) */
__global__ __launch_bounds__(256) void k_dec_split(uint8_t *xs, const float *seq, int Lt, int Lout) {
    const size_t n = (size_t)(Lt + 2) * (DEC_D / 8);
    for (size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x; idx < n; idx += (size_t)gridDim.x * 256) {
        const int r = (int)(idx / (DEC_D / 8)), c = (int)(idx % (DEC_D / 8)), t = r - 1;
        float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (t >= 0 && t < Lout) {
            const float4 *s = reinterpret_cast<const float4 *>(seq + (size_t)((t / 16) * 17 + 1 + t % 16) * DEC_D + 8 * c);
            const float4 u = s[0], v = s[1];
            f[0] = u.x; f[1] = u.y; f[2] = u.z; f[3] = u.w; f[4] = v.x; f[5] = v.y; f[6] = v.z; f[7] = v.w;
        }
        bf16x3_store(xs + (size_t)r * MAP_XROW + (c >> 2) * MAP_BB + (c & 3) * 16, f);
    }
}

/* the split weights [512][72 blocks] from the folded mapping weight [512][768][3] */
__global__ __launch_bounds__(256) void k_dec_split_w(uint8_t *ws, const float *W) {
    const int idx = blockIdx.x * 256 + threadIdx.x;   /* 512 x 288 chunks of eight k */
    if (idx >= MAP_N * 4 * MAP_KB) return;
    const int row = idx / (4 * MAP_KB), c = idx % (4 * MAP_KB), tap = c / 96, i0 = (c % 96) * 8;
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; e++) f[e] = W[(size_t)row * 3 * DEC_D + (size_t)(i0 + e) * 3 + tap];
    bf16x3_store(ws + ((size_t)row * MAP_KB + (c >> 2)) * MAP_BB + (c & 3) * 16, f);
}

typedef float f32x16_dec __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_dec __attribute__((ext_vector_type(8)));

/* A workgroup of KG groups of WM x WN waves, each wave FM x FN blocks of 32 x 32, owns 32 FM WM
 * rows by 32 FN WN columns; group g takes the k blocks g, g + KG, .. on stages of its own, and the groups'
 * sums meet in LDS in group order. A K step is one block: it moves by LDS DMA into one of NST
 * stages, NST - 1 steps ahead, and a barrier publishes it. Chunk c of part p of row r is stored at
 * 192 r + 64 p + 16 (c ^ ((r >> 2) & 3)): 16 lanes' fragment reads (16 rows, one chunk) touch
 * all 64 banks once; MFMA step s of lane half h takes chunk 2 h + s on both sides. */
template <int FM, int FN, int WM, int WN, int KG>
__global__ __launch_bounds__(64 * WM * WN * KG) void k_dec_map(float *audio, const uint8_t *xs, const uint8_t *ws,
                                                               const float *bias, int M) {
    constexpr int W = WM * WN, BM = 32 * FM * WM, BN = 32 * FN * WN, SB = (BM + BN) * MAP_BB;   /* bytes of a stage */
    constexpr int NST = 160 * 1024 / (KG * SB) > 3 ? 3 : 160 * 1024 / (KG * SB);
    constexpr int DM = (SB / 1024 + W - 1) / W;   /* transfers per wave and step (the last ones may repeat) */
    constexpr int KT = MAP_KB / KG;
    /* the next step's transfers go out one by one between the MFMAs: a wave that issues them all
     * at once waits at the full queue while its SIMD's matrix core idles (128 x 128 tiles: 81 -> 74
     * us a launch of one round). One block per wave has too few MFMAs to spread them over. */
    constexpr bool SPREAD = FM * FN > 1;
    static_assert(NST >= 2 && SB % 1024 == 0 && MAP_KB % KG == 0 && MAP_N % BN == 0, "whole transfers and steps");
    static_assert(KG == 1 || NST * SB >= 64 * W * FM * FN * 16 * 4, "a group's sums fit its stages");
    __shared__ __attribute__((aligned(16))) uint8_t smem[KG * NST * SB];
    const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x / (64 * W)));
    const int tid = threadIdx.x % (64 * W), wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wm = wave / WN, wn = wave % WN, lr = lane & 31, lh = lane >> 5;
    uint8_t *const own = smem + grp * (NST * SB);
    const uint32_t obase = (uint32_t)(uintptr_t)own;
    /* tiles in row order per XCD: the columns of one row panel share its features in one L2 */
    constexpr int NT = MAP_N / BN;
    const int T = (M + BM - 1) / BM * NT, t = xcd_tile(blockIdx.x, T);
    if (t >= T) return;                     /* uniform per workgroup, before any barrier */
    const int m0 = t / NT * BM, n0 = t % NT * BN;

    /* transfer i of this wave: 64 chunks of the stage, feature rows first, then weight rows; rows
     * past M re-read the last one */
    const uint8_t *src[DM];
#pragma unroll
    for (int i = 0; i < DM; i++) {
        const int q = 64 * min(W * i + wave, SB / 1024 - 1) + lane, r = q / 12, p = q % 12, c = (p & 12) | ((p & 3) ^ ((r >> 2) & 3));
        src[i] = r < BM ? xs + (size_t)min(m0 + r, M - 1) * MAP_XROW + 16 * c
                        : ws + (size_t)(n0 + r - BM) * (MAP_KB * MAP_BB) + 16 * c;
    }
    auto issue1 = [&](int i, int st, int kt) __attribute__((always_inline)) {
        dma16(src[i] + (size_t)(grp + KG * kt) * MAP_BB, obase + st * SB + 1024 * min(W * i + wave, SB / 1024 - 1));
    };
    auto issue = [&](int st, int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < DM; i++) issue1(i, st, kt);
    };
    auto barrier = []() __attribute__((always_inline)) {   /* every fragment read has returned; transfers stay in flight */
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    f32x16_dec hi[FM][FN], lo[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) hi[i][j][r] = lo[i][j][r] = 0.0f;

#pragma unroll
    for (int p = 0; p < NST - 1; p++) issue(p, p);
    wait_vm<(NST - 2) * DM>();
    barrier();
    int st = 0;
    for (int kt = 0; kt < KT; kt++) {
        const bool more = kt + NST - 1 < KT;
        const int nst = st == 0 ? NST - 1 : st - 1;
        if (!SPREAD && more) issue(nst, kt + NST - 1);
        const uint8_t *S = own + st * SB;
        bf16x8_dec x[2][3][FM], w[2][3][FN];   /* every read of the step is requested before its first MFMA */
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const int off = lr * MAP_BB + 16 * ((2 * lh + s) ^ ((lr >> 2) & 3));
#pragma unroll
            for (int p = 0; p < 3; p++) {
#pragma unroll
                for (int i = 0; i < FM; i++)
                    x[s][p][i] = *reinterpret_cast<const bf16x8_dec *>(S + (wm * 32 * FM + 32 * i) * MAP_BB + off + 64 * p);
#pragma unroll
                for (int j = 0; j < FN; j++)
                    w[s][p][j] = *reinterpret_cast<const bf16x8_dec *>(S + (BM + wn * 32 * FN + 32 * j) * MAP_BB + off + 64 * p);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int q = 0; q < 6; q++) {   /* in the order in which the operands arrive */
                constexpr int pw[6] = {0, 0, 1, 1, 0, 2}, px[6] = {0, 1, 0, 1, 2, 0};
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++) {
                        if (q == 0) hi[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[s][0][j], x[s][0][i], hi[i][j], 0, 0, 0);
                        else lo[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[s][pw[q]][j], x[s][px[q]][i], lo[i][j], 0, 0, 0);
                    }
                if constexpr (SPREAD) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 6 * s + q; i < DM; i += 12)
                        if (more) issue1(i, nst, kt + NST - 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        if (more) wait_vm<(NST - 2) * DM>();
        else wait_vm<0>();
        barrier();
        st = st + 1 == NST ? 0 : st + 1;
    }
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float h = hi[i][j][r];
                hi[i][j][r] = __builtin_isfinite(h) ? h + lo[i][j][r] : h;
            }
    if constexpr (KG == 2) {
        float *X = reinterpret_cast<float *>(smem + NST * SB) + tid;   /* the second group's stages, lane-major */
        if (grp == 1) {
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) X[((i * FN + j) * 16 + r) * 64 * W] = hi[i][j][r];
        }
        __syncthreads();
        if (grp == 1) return;
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) hi[i][j][r] = hi[i][j][r] + X[((i * FN + j) * 16 + r) * 64 * W];
    }
    /* accumulator r of lane l: n = 8 (r / 4) + 4 (l / 32) + r % 4, m = l % 32 (per block): 4
     * consecutive audio samples per 16-byte store */
#pragma unroll
    for (int i = 0; i < FM; i++) {
        const int m = m0 + wm * 32 * FM + i * 32 + lr;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int n = n0 + wn * 32 * FN + j * 32 + 8 * g + 4 * lh;
                const float4 b = *reinterpret_cast<const float4 *>(bias + n);
                *reinterpret_cast<float4 *>(audio + (size_t)(n >> 8) * M * 256 + (size_t)m * 256 + (n & 255)) =
                    make_float4(hi[i][j][4 * g] + b.x, hi[i][j][4 * g + 1] + b.y, hi[i][j][4 * g + 2] + b.z,
                                hi[i][j][4 * g + 3] + b.w);
            }
    }
}

static inline dim3 grid_for(size_t n) {
    size_t b = (n + 255) / 256;
    if (b > 8192) b = 8192;
    return dim3((unsigned)(b ? b : 1));
}

extern "C" hipError_t aria_k_dec_in(uint16_t *xt, const float *lat, int T, float std, hipStream_t s) {
    if (T <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dec_in, dim3((T + 63) / 64, 4), dim3(256), 0, s, xt, lat, T, std);
    return hipGetLastError();
}
extern "C" hipError_t aria_k_dec_expand(float *seq, const float *x, const float *tok, int T, int Tp, hipStream_t s) {
    hipLaunchKernelGGL(k_dec_expand, grid_for((size_t)Tp * 17 * (DEC_D / 4)), dim3(256), 0, s, (float4 *)seq,
                       (const float4 *)x, (const float4 *)tok, T, Tp);
    return hipGetLastError();
}
extern "C" hipError_t aria_k_dec_dyt(uint16_t *y, const float *x, float alpha, const float *g, const float *b,
                                     int rows, hipStream_t s) {
    const size_t n4 = (size_t)rows * (DEC_D / 4);
    hipLaunchKernelGGL(k_dec_dyt, grid_for(n4), dim3(256), 0, s, (uint2 *)y, (const float4 *)x, alpha,
                       (const float4 *)g, (const float4 *)b, n4);
    return hipGetLastError();
}
extern "C" hipError_t aria_k_dec_attn(uint16_t *merged, const float *qkv, int nch, hipStream_t s) {
    if (nch <= 0) return hipSuccess;
    DecAttnArgs a;
    a.merged = merged; a.qkv = qkv;
    hipLaunchKernelGGL(k_dec_attn_mfma, dim3(nch * 12), dim3(64 * DA_WAVES), 0, s, a, 12);
    return hipGetLastError();
}
extern "C" hipError_t aria_k_dec_split(void *xs, const float *seq, int Lt, int Lout, hipStream_t s) {
    hipLaunchKernelGGL(k_dec_split, grid_for((size_t)(Lt + 2) * (DEC_D / 8)), dim3(256), 0, s, (uint8_t *)xs, seq, Lt, Lout);
    return hipGetLastError();
}
extern "C" hipError_t aria_k_dec_split_w(void *ws, const float *W, hipStream_t s) {
    hipLaunchKernelGGL(k_dec_split_w, dim3(MAP_N * 4 * MAP_KB / 256), dim3(256), 0, s, (uint8_t *)ws, W);
    return hipGetLastError();
}
template <int FM, int FN, int WM, int WN, int KG>
static void launch_map(float *audio, const void *xs, const void *ws, const float *b, int M, hipStream_t s) {
    const int T = (M + 32 * FM * WM - 1) / (32 * FM * WM) * (MAP_N / (32 * FN * WN));
    hipLaunchKernelGGL((k_dec_map<FM, FN, WM, WN, KG>), dim3((T + 7) / 8 * 8), dim3(64 * WM * WN * KG), 0, s, audio,
                       (const uint8_t *)xs, (const uint8_t *)ws, b, M);
}
extern "C" hipError_t aria_k_dec_map(float *audio, const void *xs, const void *ws, const float *b, int M, int form,
                                     hipStream_t s) {
    if (M <= 0) return hipSuccess;
    if (form == 0) {
        /* the fewest us of the busiest CU: tiles of 64 x 64 with K over two wave groups take 30 us
         * (216 tiles at T = 108: 34 us), 128 x 128 80 us (T = 300: 81 us; the 64 x 64 form 92 us), 192 x
         * 128 122 us (T = 646, 216 tiles: 131 us; 128 x 128 in two rounds 170 us) */
        const int mt[3] = {(M + 63) / 64 * 8, (M + 127) / 128 * 4, (M + 191) / 192 * 4};
        const int us[3] = {30, 80, 122};
        int best = 1 << 30;
        for (int i = 0; i < 3; i++) {
            const int c = (mt[i] + 255) / 256 * us[i];
            if (c < best) { best = c; form = i + 1; }
        }
    }
    if (form == 1) launch_map<1, 1, 2, 2, 2>(audio, xs, ws, b, M, s);
    else if (form == 2) launch_map<2, 2, 2, 2, 1>(audio, xs, ws, b, M, s);
    else if (form == 3) launch_map<3, 2, 2, 2, 1>(audio, xs, ws, b, M, s);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
