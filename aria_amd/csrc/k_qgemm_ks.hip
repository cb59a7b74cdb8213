/*
 * k_qgemm_ks.hip - the GEMM for few output tiles (gfx950 MFMA): y[M,N] = x[M,K] W[N,K]^T (+ b)
 * for Q8 / Q4 / fp16 weights with fp16 activations and the W8A8 int8 form, with every fused
 * epilogue, K % 64 == 0 (int8: K % 128 == 0).
 * Replaces the same reference functions as k_qgemm.hip (aria_linear_q8 / aria_linear_q4,
 * src/aria_quant.c:98-145, 469-538; aria_linear_q8a8, src/aria_quant.c:253-345).
 *
 * A short sequence leaves the large-tile kernel (k_qgemm_big.hip) a handful of workgroups, each
 * walking the whole K range with a barrier per K-tile: the launch is one long latency chain on a
 * few CUs. Here a workgroup of KW waves owns one small tile of 32 FM x 32 FN outputs and the
 * waves split K between them: wave w takes the K-tiles w, w + KW, ... (RB bytes of each activation
 * row) on a pipeline of its own (NST stages of LDS that no other wave touches), so the main loop has
 * no barrier at all. While a wave waits for a K-tile, NST - 1 later ones are in flight; it reads the
 * tile into registers, sends for tile + NST into the same stage, and multiplies. NST is what fits the
 * LDS, up to four (KCfg): 2 or 3 in most configurations, 1 with fp16 or int8 weights in configuration
 * 1, whose next tile then travels only while the last one is multiplied. The partial sums then meet in
 * LDS once, each element added in wave order (a fixed order: the same bits every launch; int32
 * exactly), and every wave finalises its share of the rows with the fused epilogue.
 *
 * Operands travel HBM -> LDS by LDS DMA (global_load_lds_dwordx4) and come back as MFMA
 * fragments; Q8 and Q4 are unpacked in registers. A K-tile is RB = 128 (configuration 4: 64) bytes
 * of every activation row: KK = RB / 2 fp16, RB int8 or RB / 4 fp32 values, NK MFMA steps. Its 16-byte
 * chunk c holds k [8c, 8c + 8) (int8: [16c, 16c + 16); fp32: [4c, 4c + 4)); step s of lane half h takes
 * chunk NK h + s on both sides (fp32 activations: the two chunks of its eight k), so a lane's Q8
 * weights of a K-tile are 8 NK contiguous bytes and its Q4 weights 4 NK (all in one quantization block).
 *
 * Order of the tiles: an XCD's contiguous run goes down the rows of one weight panel first
 * (N-major), so a weight panel comes from HBM into one XCD's L2; the few activation rows are what
 * every XCD reads.
 */
#include "qgemm_dev.h"

namespace {

/* 16-byte chunk c of row r in a tile of 32-, 64- or 128-byte rows is stored at c ^ swz(r): 16
 * lanes' 16-byte fragment reads (16 rows, one chunk) then touch all 64 banks once */
template <int RB>
__device__ __forceinline__ int swz(int r) {
    return RB == 128 ? (r >> 1) & 7 : RB == 64 ? (r >> 2) & 3 : RB == 32 ? (r >> 3) & 1 : 0;
}

/* one K-tile of one wave in LDS (bytes): RB bytes of each activation row, and the weight rows'
 * share of the same k */
template <int WT, int FM, int FN, int RB, bool AF32>
struct KStage {
    static_assert(!AF32 || (WT != ARIA_WI8 && RB == 128), "fp32 activations: 32 k per K-tile");
    static constexpr bool WIDE = WT == ARIA_WI8 || WT == ARIA_WF16;
    static constexpr int KK = WT == ARIA_WI8 ? RB : AF32 ? RB / 4 : RB / 2;   /* k per K-tile */
    static constexpr int NK = KK / (WT == ARIA_WI8 ? 32 : 16);                /* MFMA steps per K-tile */
    static constexpr int WB = WT == ARIA_WF16 ? 2 * KK : WT == ARIA_WQ4 ? KK / 2 : KK;   /* bytes of a weight row */
    static constexpr int A = 32 * FM * RB;
    static constexpr int NQ = (32 * FN * WB + 1023) / 1024, NS = WT == ARIA_WQ4 ? (FN + 1) / 2 : 0;
    static constexpr int WQ = NQ * 1024, WS = NS * 1024;   /* WS: [min, step] pairs, 16 B per row */
    static constexpr int BYTES = A + WQ + WS;
    static constexpr int NA = A / 1024, DMA = NA + NQ + NS;   /* transfers of 1 KB */
};

template <int WT, int FM, int FN, int KW, int RB, bool AF32>
struct KCfg {
    using St = KStage<WT, FM, FN, RB, AF32>;
    static constexpr int ESTR = 32 * FN * 4 + 16;       /* partial-sum row stride (padded by 16 B) */
    static constexpr int PART = 32 * ESTR;              /* one wave's partial sums of a 32-row group */
    /* stages: as many (up to four) as the LDS share of PW workgroups per CU allows */
    static constexpr int PW = KW <= 4 && RB == 64 ? 2 : 1;
    static constexpr int FIT = 160 * 1024 / PW / (KW * St::BYTES);
    static constexpr int NST = FIT > 4 ? 4 : FIT;
    /* 32-row groups whose partial sums fit a wave's own stages: reduced in one round */
    static constexpr int G = FM * PART <= NST * St::BYTES ? FM : (FM % 2 == 0 && FM / 2 * PART <= NST * St::BYTES) ? FM / 2 : 1;
    static constexpr int REG = NST * St::BYTES > PART ? NST * St::BYTES : PART;   /* LDS of one wave */
    static_assert(NST >= 1, "a stage fits");
    static_assert(KW * REG <= 160 * 1024 / PW, "the LDS share of a workgroup");
    static_assert((NST - 1) * St::DMA < 64, "vmcnt");
    static_assert(FM % G == 0, "whole rounds");
};

/* the fused epilogue of NU row segments of this wave: unit u is 4 columns (nb ..) of row m[u],
 * v[u] the finished sums. The arithmetic and its order are those of epilogue() in qgemm_dev.h;
 * rr holds the residual rows of the read-modify-write modes, loaded by the caller. */
template <int FN, int NU, int WT, int MODE, bool GELU>
__device__ __forceinline__ void row_epilogue(const QArgs &a, float (&v)[NU][4], const int (&m)[NU], const bool (&on)[NU],
                                             const float4 (&rr)[NU], const float4 sc, const float4 bb, int nb, int lane) {
    const aria_qgemm_epi &e = a.epi;
    const bool col_ok = nb < a.N;
    const int nbc = col_ok ? nb : 0;
    const float scv[4] = {sc.x, sc.y, sc.z, sc.w}, bv[4] = {bb.x, bb.y, bb.z, bb.w};
    float xs[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) xs[u] = WT == ARIA_WI8 ? a.xscale[min(m[u], a.M - 1)] : 1.0f;
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (WT == ARIA_WI8) v[u][q] = v[u][q] * xs[u];
            if (WT == ARIA_WQ8 || WT == ARIA_WI8) v[u][q] = v[u][q] * scv[q];
            v[u][q] = v[u][q] + bv[q];
            if constexpr (GELU) v[u][q] = gelu_tanh_f(v[u][q]);
        }
    if constexpr (MODE == ARIA_EPI_STORE) {
#pragma unroll
        for (int u = 0; u < NU; u++) {
            if (!on[u] || m[u] >= a.M || !col_ok) continue;
            if (a.y_f16)
                *reinterpret_cast<uint2 *>((uint16_t *)a.y + (size_t)m[u] * a.N + nb) =
                    make_uint2(pack2h(v[u][0], v[u][1]), pack2h(v[u][2], v[u][3]));
            else
                *reinterpret_cast<float4 *>((float *)a.y + (size_t)m[u] * a.N + nb) =
                    make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
        }
    } else if constexpr (MODE == ARIA_EPI_GLU) {
#pragma unroll
        for (int u = 0; u < NU; u++) {
            if (!on[u] || m[u] >= a.M || !col_ok) continue;
            const float g0 = silu_f(v[u][1]) * v[u][0], g1 = silu_f(v[u][3]) * v[u][2];
            if (a.y_f16)
                *reinterpret_cast<uint32_t *>((uint16_t *)a.y + (size_t)m[u] * (a.N >> 1) + (nb >> 1)) = pack2h(g0, g1);
            else
                *reinterpret_cast<float2 *>((float *)a.y + (size_t)m[u] * (a.N >> 1) + (nb >> 1)) = make_float2(g0, g1);
        }
    } else if constexpr (MODE == ARIA_EPI_GATE_RES || MODE == ARIA_EPI_ADD || MODE == ARIA_EPI_ADD_DYT) {
        float4 g[NU];
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const int mc = min(m[u], a.M - 1);
            g[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if constexpr (MODE == ARIA_EPI_GATE_RES) {
                const int bt = mc / e.rows_per_batch;
                g[u] = *reinterpret_cast<const float4 *>(e.gate + (size_t)bt * e.gate_bs + nbc);
                if (e.gate2) {
                    const float4 ga = *reinterpret_cast<const float4 *>(e.gate2 + (size_t)bt * e.gate2_bs + nbc);
                    g[u] = make_float4(g[u].x + ga.x, g[u].y + ga.y, g[u].z + ga.z, g[u].w + ga.w);
                }
            } else if (MODE == ARIA_EPI_ADD && e.add2) {
                g[u] = *reinterpret_cast<const float4 *>(e.add2 + (size_t)mc * a.N + nbc);
            }
        }
        float4 dg = make_float4(0.f, 0.f, 0.f, 0.f), db = dg;
        if constexpr (MODE == ARIA_EPI_ADD_DYT) {
            dg = *reinterpret_cast<const float4 *>(e.w[0] + nbc);
            db = *reinterpret_cast<const float4 *>(e.w[1] + nbc);
        }
#pragma unroll
        for (int u = 0; u < NU; u++) {
            if (!on[u] || m[u] >= a.M || !col_ok) continue;
            float4 o;
            if constexpr (MODE == ARIA_EPI_GATE_RES) {
                o = make_float4(rr[u].x + v[u][0] * gate_sig_f(g[u].x), rr[u].y + v[u][1] * gate_sig_f(g[u].y),
                                rr[u].z + v[u][2] * gate_sig_f(g[u].z), rr[u].w + v[u][3] * gate_sig_f(g[u].w));
            } else {
                o = make_float4(rr[u].x + v[u][0], rr[u].y + v[u][1], rr[u].z + v[u][2], rr[u].w + v[u][3]);
                if (MODE == ARIA_EPI_ADD && e.add2) o = make_float4(o.x + g[u].x, o.y + g[u].y, o.z + g[u].z, o.w + g[u].w);
            }
            *reinterpret_cast<float4 *>((float *)a.y + (size_t)m[u] * a.N + nb) = o;
            if constexpr (MODE == ARIA_EPI_ADD_DYT) {
                const float al = e.eps;
                const float h0 = tanh_fast(al * o.x) * dg.x + db.x, h1 = tanh_fast(al * o.y) * dg.y + db.y;
                const float h2 = tanh_fast(al * o.z) * dg.z + db.z, h3 = tanh_fast(al * o.w) * dg.w + db.w;
                *reinterpret_cast<uint2 *>(e.dst[0] + (size_t)m[u] * a.N + nb) = make_uint2(pack2h(h0, h1), pack2h(h2, h3));
            }
        }
    } else {   /* HEADS, DYT_ROPE */
        const int S = e.rows_per_batch, rh = e.rot >> 1;
        int kind, d0;
        float4 gw = make_float4(1.0f, 1.0f, 1.0f, 1.0f), dbv = make_float4(0.f, 0.f, 0.f, 0.f);
        float dal = 0.0f;
        uint16_t *dsec = nullptr;
        int hh = 0;
        if constexpr (MODE == ARIA_EPI_HEADS) {
            const int secw = e.heads * 64, sec = min(nb / secw, e.nsec - 1);
            hh = (nb % secw) >> 6;
            kind = e.kind[sec];
            dsec = e.dst[sec];
            d0 = 4 * (lane & 15);
            if (kind != 2 && e.w[sec]) gw = *reinterpret_cast<const float4 *>(e.w[sec] + d0);
        } else {
            const int sec = nb / (e.heads * 64);
            d0 = nb & 63;
            kind = (!col_ok || sec == 2) ? 2 : (sec == 0 || sec == 3) ? 0 : 1;
            if (kind != 2) {
                gw = *reinterpret_cast<const float4 *>((kind == 0 ? e.w[0] : e.w[2]) + d0);
                dbv = *reinterpret_cast<const float4 *>((kind == 0 ? e.w[1] : e.w[3]) + d0);
                dal = kind == 0 ? e.eps : e.eps2;
            }
        }
        const bool rot = e.rot > 0 && (MODE == ARIA_EPI_DYT_ROPE || e.cos_t);
        const bool rope = kind != 2 && rot && d0 < e.rot, first = d0 < rh;
        const int i0 = first ? d0 : d0 - rh;
        float4 cs[NU], sn[NU];
        int sb[NU], sp[NU];
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const int mc = min(m[u], a.M - 1);
            sb[u] = mc / S;
            sp[u] = mc - sb[u] * S;
            cs[u] = sn[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (rope) {
                cs[u] = *reinterpret_cast<const float4 *>(e.cos_t + (size_t)sp[u] * rh + i0);
                sn[u] = *reinterpret_cast<const float4 *>(e.sin_t + (size_t)sp[u] * rh + i0);
            }
        }
        const float gv[4] = {gw.x, gw.y, gw.z, gw.w}, dv[4] = {dbv.x, dbv.y, dbv.z, dbv.w};
#pragma unroll
        for (int u = 0; u < NU; u++) {
            float *w4 = v[u];
            if constexpr (MODE == ARIA_EPI_HEADS) {   /* kind is uniform over a head's 16 lanes */
                float ss = (w4[0] * w4[0] + w4[1] * w4[1]) + (w4[2] * w4[2] + w4[3] * w4[3]);
                ss = grp_sum<16>(ss);
                const float inv = __builtin_amdgcn_rsqf(ss * (1.0f / 64) + e.eps);
                if (kind != 2) {
#pragma unroll
                    for (int q = 0; q < 4; q++) w4[q] = (w4[q] * inv) * gv[q];
                }
            } else if (kind != 2) {
#pragma unroll
                for (int q = 0; q < 4; q++) w4[q] = tanh_fast(dal * w4[q]) * gv[q] + dv[q];
            }
            if (rot) {   /* uniform over the grid: every lane takes part in the exchange */
                float p[4];
#pragma unroll
                for (int q = 0; q < 4; q++)
                    p[q] = MODE == ARIA_EPI_HEADS ? rope_partner(w4[q], lane, rh >> 2) : __shfl_xor(w4[q], rh >> 2);
                if (rope) {
                    const float cv[4] = {cs[u].x, cs[u].y, cs[u].z, cs[u].w};
                    const float sv[4] = {sn[u].x, sn[u].y, sn[u].z, sn[u].w};
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float c0 = w4[q] * cv[q], s1 = p[q] * sv[q];
                        w4[q] = first ? c0 - s1 : c0 + s1;
                    }
                }
            }
            if (!on[u] || m[u] >= a.M || !col_ok) continue;
            if constexpr (MODE == ARIA_EPI_HEADS)
                *reinterpret_cast<uint2 *>(dsec + (((size_t)sb[u] * e.heads + hh) * S + sp[u]) * 64 + d0) =
                    make_uint2(pack2h(w4[0], w4[1]), pack2h(w4[2], w4[3]));
            else
                *reinterpret_cast<float4 *>((float *)a.y + (size_t)m[u] * a.N + nb) = make_float4(w4[0], w4[1], w4[2], w4[3]);
        }
    }
}

}  // namespace

template <int WT, int FM, int FN, int KW, int RB, bool AF32>
__global__ __launch_bounds__(64 * KW) __attribute__((amdgpu_waves_per_eu(KW * KCfg<WT, FM, FN, KW, RB, AF32>::PW / 4))) void
k_qgemm_ks(QArgs a, int MT, int T) {
    using C = KCfg<WT, FM, FN, KW, RB, AF32>;
    using St = KStage<WT, FM, FN, RB, AF32>;
    constexpr int NST = C::NST, NK = St::NK, WB = St::WB;
    __shared__ __attribute__((aligned(16))) uint8_t smem[KW * C::REG];

    const int t = xcd_tile(blockIdx.x, T);
    if (t >= T) return;                     /* uniform per workgroup, before any barrier */
    const int m0 = (t % MT) * (32 * FM), n0 = (t / MT) * (32 * FN);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lrow = lane & 31, lh = lane >> 5;
    uint8_t *const own = smem + wave * C::REG;
    const uint32_t obase = (uint32_t)(uintptr_t)own;
    const int KT = a.K / St::KK;
    const int nt = (KT - wave + KW - 1) / KW;   /* this wave's K-tiles: wave, wave + KW, ... */
    uint32_t magic = 0x64006400u;               /* fp16 1024 in both halves, kept in a VGPR */
    asm volatile("" : "+v"(magic));

    /* per-lane sources of the transfers for K-tile 0. Rows past the edge re-read the last one:
     * their products land in rows or columns that are never stored */
    const uint8_t *xsrc[St::NA], *wsrc[St::NQ], *ssrc[St::NS ? St::NS : 1];
    constexpr int XB = WT == ARIA_WI8 ? 1 : AF32 ? 4 : 2;   /* bytes per activation */
    /* transfer i fills rows (1024 / row bytes) i ..: lane -> row and stored chunk */
#pragma unroll
    for (int i = 0; i < St::NA; i++) {
        const int r = (1024 / RB) * i + lane / (RB / 16), c = (lane % (RB / 16)) ^ swz<RB>(r);
        xsrc[i] = (const uint8_t *)a.x + (size_t)min(m0 + r, a.M - 1) * a.K * XB + 16 * c;
    }
#pragma unroll
    for (int i = 0; i < St::NQ; i++) {   /* (a transfer past the last row repeats the first ones) */
        const int r = ((1024 / WB) * i + lane / (WB / 16)) % (32 * FN), c = (lane % (WB / 16)) ^ swz<WB>(r);
        wsrc[i] = (const uint8_t *)a.q + (size_t)min(n0 + r, a.N - 1) * ((size_t)a.K * WB / St::KK) + 16 * c;
    }
    if constexpr (WT == ARIA_WQ4) {
#pragma unroll
        for (int i = 0; i < St::NS; i++)
            ssrc[i] = (const uint8_t *)(a.scale + (size_t)min(n0 + (64 * i + lane) % (32 * FN), a.N - 1) * a.nblk * 2);
    }
    auto issue = [&](int st, int kt) __attribute__((always_inline)) {
        const uint32_t b = obase + st * St::BYTES;
#pragma unroll
        for (int i = 0; i < St::NA; i++) dma16(xsrc[i] + (size_t)kt * RB, b + 1024 * i);
#pragma unroll
        for (int i = 0; i < St::NQ; i++) dma16(wsrc[i] + (size_t)kt * WB, b + St::A + 1024 * i);
        if constexpr (WT == ARIA_WQ4) {   /* the pairs of 64 k: this K-tile's, with 32 k also its neighbour's */
#pragma unroll
            for (int i = 0; i < St::NS; i++)
                dma16(ssrc[i] + (size_t)(St::KK == 32 ? kt >> 1 : kt) * 16, b + St::A + St::WQ + 1024 * i);
        }
    };

    using AccT = typename std::conditional<WT == ARIA_WI8, i32x16_t, f32x16_t>::type;
    using FragT = typename std::conditional<WT == ARIA_WI8, i32x4_t, half8_t>::type;
    using ET = typename std::conditional<WT == ARIA_WI8, int, float>::type;
    AccT acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0;

#pragma unroll
    for (int p = 0; p < NST; p++)
        if (p < nt) issue(p, wave + p * KW);

    /* fragment offsets: step s of lane half lh reads chunk NK lh + s of row lrow (fp32 activations:
     * the 32 bytes of its eight k, two chunks) */
    int aoff[NK * (AF32 ? 2 : 1)], woff[NK];
#pragma unroll
    for (int k = 0; k < NK * (AF32 ? 2 : 1); k++)
        aoff[k] = lrow * RB + 16 * (((AF32 ? 2 : 1) * NK * lh + k) ^ swz<RB>(lrow));
#pragma unroll
    for (int k = 0; k < NK; k++) woff[k] = lrow * WB + 16 * ((NK * lh + k) ^ swz<WB>(lrow));
    int st = 0;
    for (int i = 0; i < nt; i++) {
        /* this tile's transfers are the oldest in flight; up to NST - 1 tiles follow them */
        const int later = min(NST - 1, nt - 1 - i);
        static_for<NST>([&](auto R) __attribute__((always_inline)) {
            if (later == decltype(R)::value) wait_vm<decltype(R)::value * St::DMA>();
        });
        asm volatile("" ::: "memory");
        const uint8_t *S = own + st * St::BYTES;
        const int kt = wave + i * KW;
        FragT xf[NK][FM], wf[NK][FN];
        uint32_t qw[FN][2 * NK];   /* the lane's packed weights: Q8 8 NK bytes, Q4 4 NK and its pair */
        uint2 pr[FN];
#pragma unroll
        for (int k = 0; k < NK; k++)
#pragma unroll
            for (int m = 0; m < FM; m++) {
                if constexpr (AF32) {   /* rounded to fp16 as the staging pass rounds them */
                    const float4 u = *reinterpret_cast<const float4 *>(S + 32 * RB * m + aoff[2 * k]);
                    const float4 v = *reinterpret_cast<const float4 *>(S + 32 * RB * m + aoff[2 * k + 1]);
                    xf[k][m] = __builtin_bit_cast(FragT, make_uint4(pack2h(u.x, u.y), pack2h(u.z, u.w), pack2h(v.x, v.y), pack2h(v.z, v.w)));
                } else {
                    xf[k][m] = *reinterpret_cast<const FragT *>(S + 32 * RB * m + aoff[k]);
                }
            }
#pragma unroll
        for (int j = 0; j < FN; j++) {
            const int r = 32 * j + lrow;
            if constexpr (St::WIDE) {
#pragma unroll
                for (int k = 0; k < NK; k++) wf[k][j] = *reinterpret_cast<const FragT *>(S + St::A + 32 * WB * j + woff[k]);
            } else if constexpr (WT == ARIA_WQ8) {
#pragma unroll
                for (int k = 0; k < NK / 2; k++) {
                    const uint4 u = *reinterpret_cast<const uint4 *>(S + St::A + r * WB + 16 * ((NK / 2 * lh + k) ^ swz<WB>(r)));
                    qw[j][4 * k] = u.x; qw[j][4 * k + 1] = u.y; qw[j][4 * k + 2] = u.z; qw[j][4 * k + 3] = u.w;
                }
            } else {
                if constexpr (NK == 4) {
                    const uint4 u = *reinterpret_cast<const uint4 *>(S + St::A + r * WB + 16 * (lh ^ swz<WB>(r)));
                    qw[j][0] = u.x; qw[j][1] = u.y; qw[j][2] = u.z; qw[j][3] = u.w;
                } else {
                    const uint2 u = *reinterpret_cast<const uint2 *>(S + St::A + r * WB + 8 * lh);
                    qw[j][0] = u.x; qw[j][1] = u.y;
                }
                pr[j] = *reinterpret_cast<const uint2 *>(S + St::A + St::WQ + 16 * r + 8 * (St::KK == 32 ? kt & 1 : lh));
            }
        }
        /* every read of this stage has returned before its next transfers are issued */
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (i + NST < nt) issue(st, kt + NST * KW);
        if constexpr (WT == ARIA_WQ8) {
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int k = 0; k < NK; k++) {
                    uint32_t o[4];
                    q8x4_to_h(qw[j][2 * k], o[0], o[1]);
                    q8x4_to_h(qw[j][2 * k + 1], o[2], o[3]);
                    wf[k][j] = __builtin_bit_cast(FragT, make_uint4(o[0], o[1], o[2], o[3]));
                }
        } else if constexpr (WT == ARIA_WQ4) {
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const QOff f = q4_off(__builtin_bit_cast(float, pr[j].x), __builtin_bit_cast(float, pr[j].y));
#pragma unroll
                for (int k = 0; k < NK; k++) wf[k][j] = __builtin_bit_cast(FragT, q4x8_to_h(qw[j][k], magic, f));
            }
        }
#pragma unroll
        for (int k = 0; k < NK; k++)
#pragma unroll
            for (int m = 0; m < FM; m++)
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    if constexpr (WT == ARIA_WI8)
                        acc[m][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[k][j], xf[k][m], acc[m][j], 0, 0, 0);
                    else
                        acc[m][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[k][j], xf[k][m], acc[m][j], 0, 0, 0);
                }
        st = st + 1 == NST ? 0 : st + 1;
    }

    /* ---- reduction and epilogue, G 32-row groups per round ---- */
    constexpr int G = C::G, LPR = 8 * FN, RPI = 64 / LPR;         /* lanes per row, rows per 64 lanes */
    constexpr int SLOTS = 32 * G / RPI, NU = (SLOTS + KW - 1) / KW;
    const int ecol = (lane % LPR) * 4, nb = n0 + ecol;
    const bool col_ok = nb < a.N;
    const int nbc = col_ok ? nb : 0;
    float4 sc = make_float4(1.0f, 1.0f, 1.0f, 1.0f), bb = make_float4(-0.0f, -0.0f, -0.0f, -0.0f);
    if (WT == ARIA_WQ8 || WT == ARIA_WI8) sc = *reinterpret_cast<const float4 *>(a.scale + nbc);
    if (a.bias) bb = *reinterpret_cast<const float4 *>(a.bias + nbc);
    else if (WT == ARIA_WI8) bb = make_float4(0.0f, 0.0f, 0.0f, 0.0f);   /* the reference adds 0.0f */
    const int mode = a.epi.mode;
    const bool rmw = mode == ARIA_EPI_GATE_RES || mode == ARIA_EPI_ADD || mode == ARIA_EPI_ADD_DYT;
#pragma unroll
    for (int rd = 0; rd < FM / G; rd++) {
        int m[NU];
        bool on[NU];
        float4 rr[NU];
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const int slot = wave + KW * u;
            on[u] = slot < SLOTS;
            m[u] = m0 + rd * 32 * G + min(slot, SLOTS - 1) * RPI + lane / LPR;
            rr[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (rmw) rr[u] = *reinterpret_cast<const float4 *>((const float *)a.y + (size_t)min(m[u], a.M - 1) * a.N + nbc);
        }
        /* the wave's own stages are free (its reads have returned, its transfers have landed) */
#pragma unroll
        for (int i = 0; i < G; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    /* (the elements by value: __builtin_bit_cast of a vector's element in place
                     * takes the vector's first one) */
                    const ET c0 = acc[rd * G + i][j][4 * g], c1 = acc[rd * G + i][j][4 * g + 1];
                    const ET c2 = acc[rd * G + i][j][4 * g + 2], c3 = acc[rd * G + i][j][4 * g + 3];
                    *reinterpret_cast<uint4 *>(own + (32 * i + lrow) * C::ESTR + (j * 32 + 8 * g + 4 * lh) * 4) =
                        make_uint4(__builtin_bit_cast(uint32_t, c0), __builtin_bit_cast(uint32_t, c1),
                                   __builtin_bit_cast(uint32_t, c2), __builtin_bit_cast(uint32_t, c3));
                }
        __syncthreads();
        float v[NU][4];
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const uint8_t *p = smem + (m[u] - m0 - rd * 32 * G) * C::ESTR + ecol * 4;
            ET s4[4];
#pragma unroll
            for (int w = 0; w < KW; w++) {
                const uint4 x = *reinterpret_cast<const uint4 *>(p + w * C::REG);
                const ET e4[4] = {__builtin_bit_cast(ET, x.x), __builtin_bit_cast(ET, x.y), __builtin_bit_cast(ET, x.z),
                                  __builtin_bit_cast(ET, x.w)};
#pragma unroll
                for (int q = 0; q < 4; q++) s4[q] = w == 0 ? e4[q] : s4[q] + e4[q];
            }
#pragma unroll
            for (int q = 0; q < 4; q++) v[u][q] = (float)s4[q];
        }
        if (rd + 1 < FM / G) __syncthreads();   /* the sums are read before the next round's are written */
#define KS_EPI(MODE_, GELU_) row_epilogue<FN, NU, WT, MODE_, GELU_>(a, v, m, on, rr, sc, bb, nb, lane)
        switch (mode) {
            case ARIA_EPI_GATE_RES: KS_EPI(ARIA_EPI_GATE_RES, false); break;
            case ARIA_EPI_ADD: KS_EPI(ARIA_EPI_ADD, false); break;
            case ARIA_EPI_GLU: KS_EPI(ARIA_EPI_GLU, false); break;
            case ARIA_EPI_HEADS:
                if constexpr (FN == 2) KS_EPI(ARIA_EPI_HEADS, false);
                break;
            case ARIA_EPI_ADD_DYT:
                if constexpr (WT == ARIA_WF16) KS_EPI(ARIA_EPI_ADD_DYT, false);
                break;
            case ARIA_EPI_DYT_ROPE:
                if constexpr (WT == ARIA_WF16) KS_EPI(ARIA_EPI_DYT_ROPE, false);
                break;
            default:
                if (a.gelu) KS_EPI(ARIA_EPI_STORE, true);
                else KS_EPI(ARIA_EPI_STORE, false);
                break;
        }
#undef KS_EPI
    }
}

template <int WT, int FM, int FN, int KW, int RB, bool AF32 = false>
static void launch_ks(const QArgs &a, hipStream_t s) {
    const int MT = (a.M + 32 * FM - 1) / (32 * FM), T = MT * ((a.N + 32 * FN - 1) / (32 * FN));
    hipLaunchKernelGGL((k_qgemm_ks<WT, FM, FN, KW, RB, AF32>), dim3((T + 7) / 8 * 8), dim3(64 * KW), 0, s, a, MT, T);
}

/* the configurations compiled: 32-row blocks, 32-column blocks, waves, bytes of an activation row
 * per K-tile. One launch alone, Q8 weights, M = 172 (one 10 s sequence), against the large-tile
 * kernel's pick, us:
 *   N = 1024, K = 4096: 24.4 -> 8.4 (0)     N = 1024, K = 1024: 9.4 -> 3.9 (0)
 *   N = 3072, K = 1024: 12.8 -> 7.2 (4)     N = 8192, K = 1024: 18.5 -> 9.3 (3)
 * and at M = 710 (60 s) N = 1024, K = 4096: 24.9 -> 15.2 (2). What bounds it: a CU takes in
 * 60-75 KB/us (25-31 B/clk) whatever is in flight, so a launch costs about 3 us plus the bytes of
 * the tiles on its busiest CU at that rate. 128-byte K-tiles (whole cache lines) against 64-byte
 * ones: 9.8 -> 8.4 us Q8, 13.5 -> 9.7 us Q4 at N = 1024, K = 4096; 64-byte ones leave room for
 * two workgroups per CU of configuration 4, where each CU has two tiles or more. Sixteen waves per
 * workgroup (0-5 % slower), 128 x 64 tiles (no shape) and four waves of 32 x 32 tiles (no faster)
 * were measured and are not compiled. */
#define KS_CFGS(X) X(0, 1, 1, 8, 128) X(1, 1, 2, 8, 128) X(2, 2, 2, 4, 128) X(3, 3, 2, 4, 128) X(4, 2, 2, 4, 64)
static const int ks_fn[] = {1, 2, 2, 2, 2};
int qgemm_ks_ncfg() { return (int)(sizeof ks_fn / sizeof ks_fn[0]); }

template <int WT>
static hipError_t launch_ks_f32(const QArgs &a, int cfg, hipStream_t s) {
    if (cfg == 0) launch_ks<WT, 1, 1, 8, 128, true>(a, s);
    else if (cfg == 1) launch_ks<WT, 1, 2, 8, 128, true>(a, s);
    else if (cfg == 2) launch_ks<WT, 2, 2, 4, 128, true>(a, s);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t qgemm_ks_f32_launch(const QArgs &a, int wt, int cfg, hipStream_t s) {
    if (a.K % 64 || (a.gelu && a.epi.mode != ARIA_EPI_STORE) || (a.epi.mode != ARIA_EPI_STORE && a.epi.mode != ARIA_EPI_ADD) ||
        (wt == ARIA_WQ4 && ((uintptr_t)a.scale & 15u)))
        return hipErrorInvalidValue;
    if (wt == ARIA_WQ8) return launch_ks_f32<ARIA_WQ8>(a, cfg, s);
    if (wt == ARIA_WQ4) return launch_ks_f32<ARIA_WQ4>(a, cfg, s);
    if (wt == ARIA_WF16) return launch_ks_f32<ARIA_WF16>(a, cfg, s);
    return hipErrorInvalidValue;
}

hipError_t qgemm_ks_launch(const QArgs &a, int wt, int cfg, hipStream_t s) {
    if (a.K % (wt == ARIA_WI8 ? 128 : 64) || cfg < 0 || cfg >= qgemm_ks_ncfg() || (a.gelu && a.epi.mode != ARIA_EPI_STORE) ||
        (a.epi.mode == ARIA_EPI_HEADS && ks_fn[cfg] != 2) ||
        (wt != ARIA_WF16 && (a.epi.mode == ARIA_EPI_ADD_DYT || a.epi.mode == ARIA_EPI_DYT_ROPE)) ||
        (wt == ARIA_WQ4 && ((uintptr_t)a.scale & 15u)))   /* the Q4 pairs move 16 bytes at a time */
        return hipErrorInvalidValue;
#define KS_CASE(i, fm, fn, kw, rb)                                            \
    case i:                                                                   \
        if (wt == ARIA_WQ8) launch_ks<ARIA_WQ8, fm, fn, kw, rb>(a, s);        \
        else if (wt == ARIA_WQ4) launch_ks<ARIA_WQ4, fm, fn, kw, rb>(a, s);   \
        else if (wt == ARIA_WF16) launch_ks<ARIA_WF16, fm, fn, kw, rb>(a, s); \
        else if (wt == ARIA_WI8) launch_ks<ARIA_WI8, fm, fn, kw, rb>(a, s);   \
        else return hipErrorInvalidValue;                                     \
        break;
    switch (cfg) {
        KS_CFGS(KS_CASE)
        default: return hipErrorInvalidValue;
    }
#undef KS_CASE
    return hipGetLastError();
}
