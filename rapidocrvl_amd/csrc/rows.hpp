// rows.hpp — the layer matrices of a batched decode step (2 to 16 sequences,
// one activation row each) on the bf16 matrix cores.
//
// Every row of activations is handed from kernel to kernel as three bf16
// planes: hi = bf16(x), mid = bf16(x − hi), lo = bf16(x − hi − mid).  Eight
// significant bits each, so the three hold all 24 of an f32 and nothing of x is
// lost for 0 and 2^-103 ≤ |x| < 2^128 − 2^119: below, the last bits fall under
// bf16's smallest normal number, 2^-126; from there on bf16(x) is infinite and
// the row NaN.  The weight codes (|code| ≤ 127) are exact in bf16 too, so the
// products are exact and only the f32 accumulation rounds (digit planes: exact
// int32 sums over 22-bit operands; error against 64-bit sums level at 4 rows,
// 2.01e-6 → 2.05e-6, and 16, 5.77e-6 → 5.65e-6).  Unlike digit planes they
// need no scale, hence no pass over the whole row: the producer of a value (the
// step prologue, the attention merge, the epilogues below) writes its planes
// at once, already multiplied by the next RMSNorm's weight, and adds its square
// to the row's partial sums; the consumer applies fastRsqrt(Σx²/n + eps) to its
// row sums.  A layer is six launches (it was ten with a digitizing launch
// before each matrix).
//
// Bound: latency (launch, one round trip for weights and operands, the LDS sum),
// and at 16 rows a CU's L2 rate for the operand image.  Measured inside decode
// steps, kernel trace, µs (digitizing launch + small int8 GEMM before → now, two
// boxes): 16 rows Q4, 1,345 rows of context each: q|k|v 4.4 + 5.2 → 4.3–4.8,
// o_proj 4.7 + 9.0 → 5.0–5.5, gate/up 4.4 + 6.1 → 5.2–5.7, down 5.4 + 9.0 →
// 6.2–7.0; 4 rows Q6 (four-vector GEMV before): 7.9 → 4.0–4.4, 7.1 → 4.9–5.1,
// 9.1 → 5.1–5.5, 8.3 → 5.6–5.9.  The step prologue, which writes the first
// image, 4.4 → 5.5 at 4 rows.  A step of 16 requests of the whole 4-bit model
// 1.26 → 0.82 ms.
//
// Operand image of K columns: for stage u (128 columns), plane and MFMA j the
// 64 lanes' 16 bytes in lane order, lane (token n, group lg) holding columns
// 128u + 32lg + 8j .. +7 — the columns the weights' tile image gives the same
// lane group (k_tile_weight).  Up to kRowsPackMax rows the 16 MFMA columns are
// (row, plane) pairs instead, 3n + plane: a third of the MFMAs and loads.
#pragma once

#include "gemm.hpp"

namespace pocr {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kRowsThreads = 512;  // 8 waves: the K stages are dealt out to them
constexpr int kRowsWaves = kRowsThreads / 64;
constexpr int kRowsPackMax = 5;    // 3·5 = 15 of the 16 MFMA columns
constexpr int kRowsPitch = 20;     // floats per column of a wave's LDS block (16 rows, 16-byte aligned)

enum : int { R_PLAIN = 0, R_SWIGLU = 1, R_OPROJ = 2, R_DOWN = 3 };

struct RowsParams {
    const uint8_t *w[3];     // tile images: row segments (one matrix), or gate and up
    const float *scale[3];
    int seg_end[2];          // first rows of segments 1 and 2
    int rows;                // rows of the output (each matrix)
    int nst;                 // K / 128
    int ntok;
    const uint16_t *x;       // operand image of K columns
    const float *ssq;        // [nparts][16] partial Σx² of the normed input, or null
    int nparts;
    float eps;
    float *out;              // R_PLAIN: [ntok][rows]
    float *h;                // R_OPROJ, R_DOWN: residual rows [ntok][rows]
    float *vbuf;             // R_DOWN of the last layer: h + y, h untouched
    const float *norm_w;     // weight of the norm that reads this output next
    uint16_t *img;           // the output's operand image (R_PLAIN: none)
    float *ssq_out;          // [rows / 16][16]
    StepState *const *rst;   // R_OPROJ: row n's step state
    int quirk;
    int last;
};

// 32 weight codes of a lane and stage, as loaded
template <int QT>
struct RowsRaw {
    uint32_t d[ALds<QT>::chunks * ALds<QT>::bytes / 4];
};
template <int QT>
__device__ __forceinline__ RowsRaw<QT> rows_load_w(const uint8_t *block, int u, int lane) {
    using A = ALds<QT>;
    RowsRaw<QT> r;
#pragma unroll
    for (int c = 0; c < A::chunks; ++c) {
        const uint32_t *p = reinterpret_cast<const uint32_t *>(block + ((size_t)(u * A::chunks + c) * 64 + lane) * A::bytes);
        typedef unsigned u4v __attribute__((ext_vector_type(4)));
        if constexpr (A::bytes == 16) {
            const u4v v = __builtin_nontemporal_load(reinterpret_cast<const u4v *>(p));
#pragma unroll
            for (int i = 0; i < 4; ++i) r.d[4 * c + i] = v[i];
        } else {
#pragma unroll
            for (int i = 0; i < 3; ++i) r.d[3 * c + i] = __builtin_nontemporal_load(p + i);
        }
    }
    return r;
}

// codes 8j..8j+7 of the lane as the bf16 A operand: each is a small integer, so
// the upper half of its f32 is the bf16 itself
template <int QT>
__device__ __forceinline__ v8bf rows_codes(const RowsRaw<QT> &r, int j) {
    float f[8];
    if constexpr (QT == QT_Q4) {
        const uint32_t lo = r.d[j] & 0x0F0F0F0Fu, hi = (r.d[j] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            f[2 * b] = ubyte(lo, b) - 8.0f;
            f[2 * b + 1] = ubyte(hi, b) - 8.0f;
        }
    } else if constexpr (QT == QT_Q8) {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t u = r.d[2 * j + w] ^ 0x80808080u;
#pragma unroll
            for (int b = 0; b < 4; ++b) f[4 * w + b] = ubyte(u, b) - 128.0f;
        }
    } else {
        const uint32_t d0 = r.d[3 * (j >> 1)], d1 = r.d[3 * (j >> 1) + 1], d2 = r.d[3 * (j >> 1) + 2];
        const uint32_t a = (j & 1) ? (uint32_t)spread6(__builtin_amdgcn_alignbit(d2, d1, 16)) : (uint32_t)spread6(d0);
        const uint32_t b = (j & 1) ? (uint32_t)spread6(d2 >> 8) : (uint32_t)spread6(__builtin_amdgcn_alignbit(d1, d0, 24));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[i] = ubyte(a, i) - 32.0f;
            f[4 + i] = ubyte(b, i) - 32.0f;
        }
    }
    v4i v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        v[i] = (int)__builtin_amdgcn_perm(__float_as_uint(f[2 * i + 1]), __float_as_uint(f[2 * i]), 0x07060302u);
    return __builtin_bit_cast(v8bf, v);
}

// Workgroup: 16 rows (of each matrix) × TG activation rows from TG·blockIdx.y;
// wave w takes the K stages w, w + 8, … (NS of them requested at once: a wave
// waits on memory once for K ≤ 1024·NS) and the waves' sums meet in LDS.
// PACK: columns are (row, plane) pairs.
template <int QT, int EPI, int NS, bool PACK, int TG>
static __global__ void __launch_bounds__(kRowsThreads) k_rows(RowsParams p) {
    constexpr int NMAT = EPI == R_SWIGLU ? 2 : 1;
    constexpr int NP = PACK ? 1 : 3;  // MFMA column sets per 8 columns
    __shared__ __align__(16) float part[kRowsWaves][NMAT][16 * kRowsPitch];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int c = lane & 15, lg = lane >> 4;
    const int r0 = blockIdx.x * 16;
    const int n0 = PACK ? 0 : blockIdx.y * TG;
    asm volatile("" ::"s"(p.w[0]), "s"(p.w[1]), "s"(p.w[2]), "s"(p.scale[0]), "s"(p.scale[1]), "s"(p.scale[2]));
    asm volatile("" ::"s"(p.x), "s"(p.ssq), "s"(p.out), "s"(p.h), "s"(p.vbuf), "s"(p.norm_w), "s"(p.img), "s"(p.ssq_out));
    asm volatile("" ::"s"(p.seg_end[0]), "s"(p.seg_end[1]), "s"(p.rows), "s"(p.nst), "s"(p.ntok), "s"(p.nparts));

    // the matrices' 16-row blocks
    const uint8_t *wb[NMAT];
    const float *sb[NMAT];
    constexpr int block_stage = ALds<QT>::block_stage;
    if constexpr (NMAT == 2) {
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
            wb[mi] = p.w[mi] + (size_t)(r0 / 16) * p.nst * block_stage;
            sb[mi] = p.scale[mi] + r0;
        }
    } else {
        const int sg = r0 >= p.seg_end[1] ? 2 : (r0 >= p.seg_end[0] ? 1 : 0);
        const int start = sg == 2 ? p.seg_end[1] : (sg == 1 ? p.seg_end[0] : 0);
        wb[0] = (sg == 2 ? p.w[2] : (sg == 1 ? p.w[1] : p.w[0])) + (size_t)((r0 - start) / 16) * p.nst * block_stage;
        sb[0] = (sg == 2 ? p.scale[2] : (sg == 1 ? p.scale[1] : p.scale[0])) + (r0 - start);
    }

    // rows past ntok (their columns' results are never read) load nothing
    const bool live = PACK ? c < 3 * p.ntok : (c < TG && n0 + c < p.ntok);
    const uint16_t *xl = p.x + (size_t)(lane + (PACK ? 0 : n0)) * 8;
    v4f acc[NMAT][NP];
#pragma unroll
    for (int mi = 0; mi < NMAT; ++mi)
#pragma unroll
        for (int pl = 0; pl < NP; ++pl) acc[mi][pl] = v4f{0.f, 0.f, 0.f, 0.f};
    RowsRaw<QT> a[NS][NMAT];
    v4i b[NS][NP][4];
    auto request = [&](int u0) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int u = min(u0 + kRowsWaves * s, p.nst - 1);  // clamped: loaded, not used
#pragma unroll
            for (int pl = 0; pl < NP; ++pl)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    b[s][pl][j] = v4i{0, 0, 0, 0};
                    if (live)
                        b[s][pl][j] = *reinterpret_cast<const v4i *>(xl + (size_t)((u * NP + pl) * 4 + j) * 512);
                }
#pragma unroll
            for (int mi = 0; mi < NMAT; ++mi) a[s][mi] = rows_load_w<QT>(wb[mi], u, lane);
        }
    };
    request(wave);

    // epilogue operands of thread (row i, activation row n)
    const int i = t & 15, nl = (t >> 4) & 15, n = n0 + nl, r = r0 + i;
    const bool mine = t < 256 && nl < TG && n < p.ntok;
    const int nc = min(n, p.ntok - 1);
    float sc[NMAT], resid = 0.f, nw = 0.f, ss = 0.f;
    int clen = 0;
    if (t < 256) {
#pragma unroll
        for (int mi = 0; mi < NMAT; ++mi) sc[mi] = sb[mi][i];
        if constexpr (EPI == R_OPROJ || EPI == R_DOWN) {
            resid = p.h[(size_t)nc * p.rows + r];
            nw = p.norm_w[r];
        }
        if constexpr (EPI == R_OPROJ) clen = p.rst[nc]->clen;
        if constexpr (EPI == R_PLAIN || EPI == R_SWIGLU)
            for (int k = i; k < p.nparts; k += 16) ss += p.ssq[k * 16 + nc];
    }

    for (int u0 = wave;; u0 += kRowsWaves * NS) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (u0 + kRowsWaves * s >= p.nst) break;  // uniform
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int mi = 0; mi < NMAT; ++mi) {
                    const v8bf av = rows_codes<QT>(a[s][mi], j);
#pragma unroll
                    for (int pl = 0; pl < NP; ++pl)
                        acc[mi][pl] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            av, __builtin_bit_cast(v8bf, b[s][pl][j]), acc[mi][pl], 0, 0, 0);
                }
        }
        if (u0 + kRowsWaves * NS >= p.nst) break;  // uniform
        request(u0 + kRowsWaves * NS);
    }

    // waves' sums → LDS [column][row]; lane (c, lg) holds rows 4lg..4lg+3
#pragma unroll
    for (int mi = 0; mi < NMAT; ++mi) {
        v4f y = acc[mi][0];
        if constexpr (!PACK) y = (acc[mi][2] + acc[mi][1]) + y;  // smallest plane first
        *reinterpret_cast<v4f *>(&part[wave][mi][c * kRowsPitch + 4 * lg]) = y;
    }
    __syncthreads();
    if (t >= 256) return;
    float y[NMAT];
#pragma unroll
    for (int mi = 0; mi < NMAT; ++mi) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < kRowsWaves; ++w) {
            const float *q = part[w][mi];
            if constexpr (PACK) {
                const int cb = 3 * min(nl, kRowsPackMax - 1);
                v += (q[(cb + 2) * kRowsPitch + i] + q[(cb + 1) * kRowsPitch + i]) + q[cb * kRowsPitch + i];
            } else {
                v += q[nl * kRowsPitch + i];
            }
        }
        y[mi] = v;
    }
    if constexpr (EPI == R_PLAIN || EPI == R_SWIGLU) {
        // Σx² over the partial sums: 16 lanes of one activation row
        ss += xchg<XQ1>(ss);
        ss += xchg<XQ2>(ss);
        ss += xchg<XM8>(ss);
        ss += xchg<XM16>(ss);
        const float f = fast_rsqrt_ref(ss / (float)(p.nst * 128) + p.eps);
#pragma unroll
        for (int mi = 0; mi < NMAT; ++mi) y[mi] = y[mi] * f;
    }
#pragma unroll
    for (int mi = 0; mi < NMAT; ++mi) y[mi] = y[mi] * sc[mi];
    if constexpr (EPI == R_PLAIN) {
        if (mine) p.out[(size_t)n * p.rows + r] = y[0];
    } else if constexpr (EPI == R_SWIGLU) {
#pragma clang fp contract(off)
        const float g = silu_ref(y[0]) * y[NMAT - 1];
        if (mine) rows_put(p.img, PACK, n, r, g);
    } else {
#pragma clang fp contract(off)
        const float v = resid + y[0];
        if (EPI == R_DOWN && p.last) {
            if (mine) p.vbuf[(size_t)n * p.rows + r] = v;
            return;
        }
        // model.go:3895-3902, 4051-4057: Q4/Q6 rows keep the residual before
        // attention at cache length 0 and from 6 on
        if (mine && (EPI == R_DOWN || !(p.quirk && (clen == 0 || clen >= 6)))) p.h[(size_t)n * p.rows + r] = v;
        if (mine) rows_put(p.img, PACK, n, r, v * nw);
        float q = v * v;
        q += xchg<XQ1>(q);
        q += xchg<XQ2>(q);
        q += xchg<XM8>(q);
        q += xchg<XM16>(q);
        if (mine && i == 0) p.ssq_out[blockIdx.x * 16 + n] = q;
    }
}

}  // namespace pocr
