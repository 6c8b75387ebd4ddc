// k_enc.hip — Conformer encoder kernels other than the GEMMs: the relative-
// position attention core, the depthwise-conv/BN/SiLU stage of the conv
// module, and the convolutional subsampling front-end.
//
// Activations are position-major ([t][channel]) everywhere so the pointwise
// convolutions are plain GEMMs.
#include "ct_dev.h"
#include "ct_launch.h"
#include "../../include/model_types.h"
#include <stdio.h>
#include <stdlib.h>
#include <type_traits>

namespace {

// ---------------------------------------------------------------------------
// Relative-position attention core (backends/cpu/backend.c:262-296) on fp32
// MFMA (v_mfma_f32_16x16x4f32: exact fp32 products, fp32 sums).
// Workgroup = 16 query rows x one head, 4 waves.  S[q][k] = ((Q_q+u).K_k)*s +
// ((Q_q+v).P_{k+T-1-q})*s with s = 1/sqrt(160), softmax over k, then S V.
//   A: 16 x 16 score tiles over the keys (waves take tiles w, w+4, ...);
//   B: 16 x 16 tiles over the window of T+15 P rows the block needs; window
//      row j of query i is key j + i - 15, so each product lands on exactly
//      one score and is added there;
//   softmax per row in LDS; C: O = S V as 10 tiles of 16 head dimensions.
// MFMA lanes: A[i][k] from lane 16k + i, B[k][j] from lane 16k + j, result
// D[4(l/16) + r][l%16] in lane l.  Scores live in LDS, row stride ldS.
// Rows of Q, K, P, V must be 16-byte aligned (the launchers check).
// ---------------------------------------------------------------------------
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int RQ = 16;                // query rows per workgroup
constexpr int RKS = ENC_DK / 4;       // 40 MFMA K-steps over the head dimension

template <bool PACKED>
__global__ __launch_bounds__(256) void relpos_attn_kernel(float *O, const float *Q, const float *K,
                                                          const float *V, const float *P,
                                                          const uint16_t *pbu, const uint16_t *pbv,
                                                          int T_arg, int T_max, const int *seq_off,
                                                          const int *seq_T, const int *blk_seq,
                                                          const int *blk_q0, int ldS,
                                                          uint16_t *Oh, uint16_t *Ol) {
    extern __shared__ float S[];      // [RQ][ldS]
    // Dispatch order: workgroup L = x + y * gridDim.x runs on XCD L mod 8, so
    // L is taken as (block L / 8, head L mod 8): every block of head h runs on
    // XCD h, in block order, and a clip-head's consecutive query blocks share
    // that XCD's L2 for its K, P and V rows.
    const int lin = blockIdx.x + blockIdx.y * gridDim.x;
    const int bi = lin / ENC_H, h = lin % ENC_H;
    int T, q0;
    long off = 0;
    if (PACKED) {
        const int sq = blk_seq[bi];
        q0 = blk_q0[bi];
        T = seq_T[sq];
        off = seq_off[sq];
        P += (long)(T_max - T) * ENC_D;     // this clip's window of the T_max table
    } else {
        T = T_arg;
        q0 = bi * RQ;
    }
    Q += off * ENC_D; K += off * ENC_D; V += off * ENC_D;
    // the output goes to O, or split hi/lo to the planes Oh/Ol
    if (Oh) { Oh += off * ENC_D; Ol += off * ENC_D; }
    else O += off * ENC_D;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int nq = min(RQ, T - q0);
    const long hc = (long)h * ENC_DK;
    const float sc = 1.0f / sqrtf((float)ENC_DK);

    // The MFMA K index of step st = 4c + e in lane group lk is head dim
    // 16c + 4lk + e: a float4 load c of row li takes dims [16c, 16c + 16) of
    // the row across the 4 lane groups, one 64-byte segment.  (With a 160-
    // byte run per lane, each segment is requested by 4 successive loads and
    // the L1 does not keep it between them: twice the L1 -> L2 requests.)
    // A fragments of Q+u and Q+v: row li.
    float au[RKS], av[RKS];
    {
        const bool ok = li < nq;
        const float4 *qp = reinterpret_cast<const float4 *>(Q + (long)(q0 + li) * ENC_D + hc + 4 * lk);
#pragma unroll
        for (int c = 0; c < RKS / 4; c++) {
            const float4 x = ok ? qp[4 * c] : make_float4(0.f, 0.f, 0.f, 0.f);
            const float xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int st = 4 * c + e, d = 16 * c + 4 * lk + e;
                au[st] = xs[e] + bf2f(pbu[hc + d]);
                av[st] = xs[e] + bf2f(pbv[hc + d]);
            }
        }
    }
    // A: content scores
    const int nkt = (T + 15) / 16;
    for (int kt = w; kt < nkt; kt += 4) {
        const int key = kt * 16 + li;
        const bool ok = key < T;
        const float4 *kp = reinterpret_cast<const float4 *>(K + (long)key * ENC_D + hc + 4 * lk);
        float b[RKS];
#pragma unroll
        for (int c = 0; c < RKS / 4; c++) {
            const float4 x = ok ? kp[4 * c] : make_float4(0.f, 0.f, 0.f, 0.f);
            b[4 * c] = x.x; b[4 * c + 1] = x.y; b[4 * c + 2] = x.z; b[4 * c + 3] = x.w;
        }
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < RKS; st++) acc = mfma4(au[st], b[st], acc);
        if (ok) {
#pragma unroll
            for (int j = 0; j < 4; j++) S[(4 * lk + j) * ldS + key] = acc[j] * sc;
        }
    }
    __syncthreads();
    // B: position scores over window rows p = plo + win, win in [0, T+15)
    const int plo = T - 1 - (q0 + RQ - 1);
    const int nwt = (T + RQ - 1 + 15) / 16;
    for (int wt = w; wt < nwt; wt += 4) {
        const int win = wt * 16 + li, p = plo + win;
        const bool ok = win < T + RQ - 1 && p >= 0 && p <= 2 * T - 2;
        const float4 *pp = reinterpret_cast<const float4 *>(P + (long)p * ENC_D + hc + 4 * lk);
        float b[RKS];
#pragma unroll
        for (int c = 0; c < RKS / 4; c++) {
            const float4 x = ok ? pp[4 * c] : make_float4(0.f, 0.f, 0.f, 0.f);
            b[4 * c] = x.x; b[4 * c + 1] = x.y; b[4 * c + 2] = x.z; b[4 * c + 3] = x.w;
        }
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < RKS; st++) acc = mfma4(av[st], b[st], acc);
        // column li of the tile is window row win; query i = 4*lk + j reads
        // it as key win + i - 15
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int qi = 4 * lk + j, k = win + qi - (RQ - 1);
            if (ok && qi < nq && k >= 0 && k < T) S[qi * ldS + k] += acc[j] * sc;
        }
    }
    __syncthreads();
    // softmax per row (backends/cpu/backend.c:67-73)
    for (int qi = w; qi < nq; qi += 4) {
        float *row = S + qi * ldS;
        float mx = -INFINITY;
        for (int k = lane; k < T; k += 64) mx = fmaxf(mx, row[k]);
        mx = wave_max(mx);
        float sum = 0.0f;
        // e^(s - max) as 2^((s - max) log2 e) on the hardware exp2
        for (int k = lane; k < T; k += 64) {
            const float e = __builtin_amdgcn_exp2f((row[k] - mx) * 1.4426950408889634f);
            row[k] = e;
            sum += e;
        }
        sum = wave_sum(sum);
        for (int k = lane; k < T; k += 64) row[k] /= sum;
    }
    __syncthreads();
    // C: O = S V, 10 tiles of 16 dimensions, keys in steps of 4
    for (int dt = w; dt < ENC_DK / 16; dt += 4) {
        const int d = dt * 16 + li;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        const float *vp = V + hc + d;
        const float *sr = S + (li < nq ? li : 0) * ldS;
        int k0 = 0;
        for (; k0 + 32 <= T; k0 += 32) {
            float a[8], bv[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int k = k0 + 4 * u + lk;
                a[u] = sr[k];
                bv[u] = vp[(long)k * ENC_D];
            }
#pragma unroll
            for (int u = 0; u < 8; u++) acc = mfma4(a[u], bv[u], acc);
        }
        if (k0 < T) {
            // the last T - k0 < 32 keys: every load of the batch goes out before
            // the first MFMA (one round trip instead of one per step of 4
            // keys); the MFMAs are the same steps as one at a time
            float a[8], bv[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int k = k0 + 4 * u + lk;
                a[u] = k < T ? sr[k] : 0.0f;
                bv[u] = k < T ? vp[(long)k * ENC_D] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (k0 + 4 * u < T) acc = mfma4(a[u], bv[u], acc);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int qi = 4 * lk + j;
            if (qi >= nq) continue;
            const long o = (long)(q0 + qi) * ENC_D + hc + d;
            if (Oh) {
                uint16_t hh, ll;
                split_bf16(acc[j], hh, ll);
                Oh[o] = hh;
                Ol[o] = ll;
            } else {
                O[o] = acc[j];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Depthwise conv (k = 9, zero padding 4 inside the sequence) + inference
// BatchNorm + SiLU (backends/cpu/backend.c:312-334).
// ---------------------------------------------------------------------------
// One thread per 8 consecutive channels of DW_RB consecutive rows: the
// DW_RB + 8 input rows the taps reach are read once (16-byte pieces) and kept
// in registers.  The arithmetic per element is the scalar form's (taps in
// order, taps outside the row's sequence skipped, then BN and SiLU).  With few
// rows the launch is bound by one thread's instructions, so a thread takes a
// single row; with many, by the rows fetched again by their neighbours, so it
// takes 8.  us at 101 rows: 8 rows a thread 12.1, 4 8.4, 2 5.8, 1 4.7; at 1008
// 12.4, 9.4, 8.2, 7.8; at 2600 14.8, 14.4, 16.6, 18.1; at 13000 53, 54, 63, 72.
constexpr int DW_ROWS_FEW = 1600;
template <int DW_RB>
__global__ __launch_bounds__(256) void dwconv_bn_silu_kernel(float *out, uint16_t *out_hi, uint16_t *out_lo,
                                                             const float *in, int M, const int *row_start,
                                                             const int *row_len, const uint16_t *dww,
                                                             const uint16_t *dwb, const uint16_t *bnw,
                                                             const uint16_t *bnb, const uint16_t *bnm,
                                                             const uint16_t *bnv) {
    constexpr int G = ENC_D / 8, HALO = (ENC_CK - 1) / 2, NX = DW_RB + ENC_CK - 1;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int nrb = (M + DW_RB - 1) / DW_RB;
    if (i >= (long)nrb * G) return;
    const int r0 = (int)(i / G) * DW_RB, c0 = (int)(i % G) * 8;
    // input rows r0 - 4 .. r0 + DW_RB + 3 of these 8 channels (zero outside [0, M))
    float x[NX][8];
#pragma unroll
    for (int j = 0; j < NX; j++) {
        const int rr = r0 - HALO + j;
        if (rr >= 0 && rr < M) {
            const float4 *p = reinterpret_cast<const float4 *>(in + (long)rr * ENC_D + c0);
            const float4 x0 = p[0], x1 = p[1];
            x[j][0] = x0.x; x[j][1] = x0.y; x[j][2] = x0.z; x[j][3] = x0.w;
            x[j][4] = x1.x; x[j][5] = x1.y; x[j][6] = x1.z; x[j][7] = x1.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) x[j][e] = 0.0f;
        }
    }
    // taps of the 8 channels: dww[c][k] for c0 <= c < c0 + 8, 72 contiguous values
    uint16_t wk[8 * ENC_CK];
#pragma unroll
    for (int v = 0; v < ENC_CK; v++) {
        const u16x8 w8 = *reinterpret_cast<const u16x8 *>(dww + c0 * ENC_CK + 8 * v);
#pragma unroll
        for (int e = 0; e < 8; e++) wk[8 * v + e] = w8[e];
    }
    const u16x8 b8 = *reinterpret_cast<const u16x8 *>(dwb + c0);
    const u16x8 m8 = *reinterpret_cast<const u16x8 *>(bnm + c0), v8 = *reinterpret_cast<const u16x8 *>(bnv + c0);
    const u16x8 w8 = *reinterpret_cast<const u16x8 *>(bnw + c0), bb8 = *reinterpret_cast<const u16x8 *>(bnb + c0);
#pragma unroll
    for (int rb = 0; rb < DW_RB; rb++) {
        const int r = r0 + rb;
        if (r >= M) break;
        const int st = row_start ? row_start[r] : 0;       // this row's sequence: [st, st + T)
        const int T = row_len ? row_len[r] : M;
        const int t = r - st;
        float s[8];
#pragma unroll
        for (int e = 0; e < 8; e++) s[e] = bf2f(b8[e]);
#pragma unroll
        for (int k = 0; k < ENC_CK; k++) {
            const int ti = t - HALO + k;
            if (ti < 0 || ti >= T) continue;
            // input row st + ti = r - HALO + k is x[rb + k]
#pragma unroll
            for (int e = 0; e < 8; e++) s[e] += bf2f(wk[e * ENC_CK + k]) * x[rb + k][e];
        }
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float v = (s[e] - bf2f(m8[e])) / sqrtf(bf2f(v8[e]) + 1e-5f) * bf2f(w8[e]) + bf2f(bb8[e]);
            o[e] = v * sigmoid_hw(v);
        }
        const long oi = (long)r * ENC_D + c0;
        if (out_hi) {
            u16x8 h8, l8;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                uint16_t hh, ll;
                split_bf16(o[e], hh, ll);
                h8[e] = hh; l8[e] = ll;
            }
            *reinterpret_cast<u16x8 *>(out_hi + oi) = h8;
            *reinterpret_cast<u16x8 *>(out_lo + oi) = l8;
        } else {
            float4 *y = reinterpret_cast<float4 *>(out + oi);
            y[0] = make_float4(o[0], o[1], o[2], o[3]);
            y[1] = make_float4(o[4], o[5], o[6], o[7]);
        }
    }
}

// ---------------------------------------------------------------------------
// Subsampling (backends/cpu/backend.c:188-229).
// conv0: 3x3 stride 2 pad 1, 1 -> 256 channels, + ReLU, over the image
// img[t][m] = mel[m*stride + t]; output [T1][64][256].
// ---------------------------------------------------------------------------
__global__ void sub_conv0_kernel(float *out, const float *mel, int T_mel, int stride,
                                 const uint16_t *w, const uint16_t *b) {
    const int T1 = (T_mel + 1) / 2;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)T1 * 64 * SUB_CH) return;
    const int oc = (int)(i % SUB_CH);
    const int ow = (int)((i / SUB_CH) % 64);
    const int oh = (int)(i / (SUB_CH * 64));
    float s = bf2f(b[oc]);
#pragma unroll
    for (int kh = 0; kh < 3; kh++) {
        const int ih = oh * 2 - 1 + kh;
        if (ih < 0 || ih >= T_mel) continue;
#pragma unroll
        for (int kw = 0; kw < 3; kw++) {
            const int iw = ow * 2 - 1 + kw;
            if (iw < 0 || iw >= N_MELS) continue;
            s += mel[(long)iw * stride + ih] * bf2f(w[oc * 9 + kh * 3 + kw]);
        }
    }
    out[i] = s > 0.0f ? s : 0.0f;
}

// Depthwise 3x3 stride 2 pad 1 over [H][Wd][256] -> [(H+1)/2][(Wd+1)/2][256].
__global__ void sub_dwconv_kernel(float *out, const float *in, int H, int Wd,
                                  const uint16_t *w, const uint16_t *b) {
    const int Ho = (H + 1) / 2, Wo = (Wd + 1) / 2;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)Ho * Wo * SUB_CH) return;
    const int c = (int)(i % SUB_CH);
    const int ow = (int)((i / SUB_CH) % Wo);
    const int oh = (int)(i / ((long)SUB_CH * Wo));
    float s = bf2f(b[c]);
#pragma unroll
    for (int kh = 0; kh < 3; kh++) {
        const int ih = oh * 2 - 1 + kh;
        if (ih < 0 || ih >= H) continue;
#pragma unroll
        for (int kw = 0; kw < 3; kw++) {
            const int iw = ow * 2 - 1 + kw;
            if (iw < 0 || iw >= Wd) continue;
            s += in[((long)ih * Wd + iw) * SUB_CH + c] * bf2f(w[c * 9 + kh * 3 + kw]);
        }
    }
    out[i] = s;
}

// Request of packed row tau: the r with off[r] <= tau < off[r + 1] (off has
// n + 1 ascending entries, off[0] = 0).
__device__ __forceinline__ int packed_owner(const int *off, int n, int tau) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= tau) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// The first two subsampling stages fused, over several requests packed
// along time: conv 3x3 stride 2 (1 -> 256 channels, ReLU) then depthwise
// 3x3 stride 2, without storing the conv output.  Workgroup = one output row
// tau of the depthwise stage (request r, row oh = tau - o2[r]; without tables,
// one request of T_arg frames) and SUB_SEG of its 32 output columns, thread =
// channel c.  The 7 mel frames the row needs (4*oh - 3 .. 4*oh + 3) are staged
// in LDS frame-contiguous, zero outside the clip, so a thread fetches a bin's
// 7 frames as two 16-byte broadcasts.
// Going along the columns, a thread keeps the conv column its next output
// shares with this one and a mel bin: 6 conv values and 4 bins an output,
// where computing every tap's conv value takes 9 values and 81 LDS reads.  It
// is bound by its multiply-adds (63 an output and channel).  Every value is
// summed in the order of sub_conv0 then sub_dwconv (taps in order, those
// outside skipped, whatever their weights are), so the result is bit-identical
// to running the two stages (backends/cpu/backend.c:201-221).  The skips are
// tests of whole-workgroup conditions, made only in the outputs that have a
// tap outside: a clip's first and last rows and each row's first column.  The
// output is written split hi/lo for the pointwise GEMM that reads it.
// 24 clips (4134 rows) 199 -> 71 us; one clip of 10 s (251 rows) 9.7, where
// the two stages took 60.
constexpr int SUB_SEG = 8;                        // output columns of a workgroup
__global__ __launch_bounds__(256) void sub_conv0_dw_packed_kernel(uint16_t *out_hi, uint16_t *out_lo,
                                                                  const float *mel,
                                                                  const int *o1, const int *o2,
                                                                  const int *tmel, const int *moff, int n,
                                                                  int T_arg, int stride_arg,
                                                                  const uint16_t *w0, const uint16_t *b0,
                                                                  const uint16_t *wd, const uint16_t *bd) {
    constexpr int NB = 4 * SUB_SEG + 3;           // bins 4*ow0 - 3 .. 4*ow0 + 4*SUB_SEG - 1
    __shared__ float4 sm[NB][2];
    const int tau = blockIdx.x, c = threadIdx.x, ow0 = blockIdx.y * SUB_SEG;
    const int r = o2 ? packed_owner(o2, n, tau) : 0;
    const int oh = o2 ? tau - o2[r] : tau;
    const int T_mel = o2 ? tmel[r] : T_arg, H1 = o2 ? o1[r + 1] - o1[r] : (T_arg + 1) / 2;
    const long stride = o2 ? T_mel : stride_arg;
    const float *m = mel + (o2 ? moff[r] : 0);
    const int f0 = 4 * oh - 3;                    // first mel frame of the window
    for (int e = c; e < NB * 8; e += 256) {
        const int bin = 4 * ow0 - 3 + e / 8, f = f0 + e % 8;
        reinterpret_cast<float *>(sm)[e] =
            (e % 8 < 7 && bin >= 0 && bin < N_MELS && f >= 0 && f < T_mel) ? m[bin * stride + f] : 0.0f;
    }
    float k0[9], kd[9];
#pragma unroll
    for (int k = 0; k < 9; k++) { k0[k] = bf2f(w0[c * 9 + k]); kd[k] = bf2f(wd[c * 9 + k]); }
    const float bias0 = bf2f(b0[c]), biasd = bf2f(bd[c]);
    __syncthreads();
    struct Bin { float f[8]; };
    auto bin = [&](int i) {                       // bin 4*ow0 - 3 + i
        Bin b;
        const float4 x = sm[i][0], y = sm[i][1];
        b.f[0] = x.x; b.f[1] = x.y; b.f[2] = x.z; b.f[3] = x.w;
        b.f[4] = y.x; b.f[5] = y.y; b.f[6] = y.z; b.f[7] = y.w;
        return b;
    };
    // The three conv values of one column (rows 2*oh - 1 .. 2*oh + 1) from its
    // three bins.  edge: frames may lie outside the clip, and bin x0 where not in0.
    struct Col { float v[3]; };
    auto conv = [&](auto edge, const Bin &x0, const Bin &x1, const Bin &x2, bool in0) {
        constexpr bool E = decltype(edge)::value;
        Col q;
#pragma unroll
        for (int kh2 = 0; kh2 < 3; kh2++) {
            float x = bias0;
#pragma unroll
            for (int kh = 0; kh < 3; kh++) {
                const int f = 2 * kh2 + kh;
                if (E && (f0 + f < 0 || f0 + f >= T_mel)) continue;
                if (!E || in0) x += x0.f[f] * k0[kh * 3];
                x += x1.f[f] * k0[kh * 3 + 1];
                x += x2.f[f] * k0[kh * 3 + 2];
            }
            q.v[kh2] = x > 0.0f ? x : 0.0f;
        }
        return q;
    };
    using Edge = std::true_type;
    using Inner = std::false_type;
    const bool edge_rows = f0 < 0 || f0 + 7 > T_mel;      // the row has taps outside the clip
    Bin last = bin(2);                            // bin 4*ow - 1
    // conv column 2*ow - 1 (of column -1 nothing is used)
    Col left = edge_rows ? conv(Edge(), bin(0), bin(1), last, true) : conv(Inner(), bin(0), bin(1), last, true);
    const long orow = ((long)tau * 32 + ow0) * SUB_CH + c;
    auto output = [&](auto edge, int j) {
        constexpr bool E = decltype(edge)::value;
        const bool in0 = ow0 + j > 0;             // column 0 has no column and no bin to its left
        const Bin x1 = bin(4 * j + 3), x2 = bin(4 * j + 4), x3 = bin(4 * j + 5), x4 = bin(4 * j + 6);
        const Col mid = conv(edge, last, x1, x2, in0), right = conv(edge, x2, x3, x4, true);
        float acc = biasd;
#pragma unroll
        for (int kh2 = 0; kh2 < 3; kh2++) {
            const int ih1 = 2 * oh - 1 + kh2;
            if (E && (ih1 < 0 || ih1 >= H1)) continue;
            if (!E || in0) acc += left.v[kh2] * kd[kh2 * 3];
            acc += mid.v[kh2] * kd[kh2 * 3 + 1];
            acc += right.v[kh2] * kd[kh2 * 3 + 2];
        }
        uint16_t hh, ll;
        split_bf16(acc, hh, ll);
        out_hi[orow + (long)j * SUB_CH] = hh;
        out_lo[orow + (long)j * SUB_CH] = ll;
        left = right;
        last = x4;
    };
    int j = 0;
    for (const int je = edge_rows ? SUB_SEG : ow0 == 0 ? 1 : 0; j < je; j++) output(Edge(), j);
#pragma unroll 2
    for (; j < SUB_SEG; j++) output(Inner(), j);
}

// sub_dwconv_kernel over several requests, written split hi/lo for the
// pointwise GEMM: request r's input rows oin[r] .. oin[r + 1] of
// [sum H][Wd][256], output rows oout[r] .. oout[r + 1] of
// [sum (H+1)/2][(Wd+1)/2][256] (without tables, one request of H_arg rows).
// Workgroup = one output row and SUB_SEG of its columns, thread = channel: the
// 2*SUB_SEG + 1 input columns of the three rows all in flight at once, each
// read once; each sum is the scalar form's (taps in order, those outside
// skipped: whole-workgroup conditions).
// 24 clips (2071 rows) 91 -> 38 us.
__global__ __launch_bounds__(256) void sub_dw_split_packed_kernel(uint16_t *out_hi, uint16_t *out_lo,
                                                                  const float *in, const int *oin,
                                                                  const int *oout, int n, int H_arg, int Wd,
                                                                  const uint16_t *w, const uint16_t *b) {
    constexpr int NX = 2 * SUB_SEG + 1;
    const int Wo = (Wd + 1) / 2;
    const int tau = blockIdx.x, c = threadIdx.x, ow0 = blockIdx.y * SUB_SEG;
    const int r = oout ? packed_owner(oout, n, tau) : 0;
    const int oh = oout ? tau - oout[r] : tau, H = oout ? oin[r + 1] - oin[r] : H_arg;
    const float *x = in + (long)(oout ? oin[r] : 0) * Wd * SUB_CH + c;
    float v[3][NX];
#pragma unroll
    for (int kh = 0; kh < 3; kh++) {
        const int ih = oh * 2 - 1 + kh;
#pragma unroll
        for (int j = 0; j < NX; j++) {
            const int iw = 2 * ow0 - 1 + j;
            v[kh][j] = ih >= 0 && ih < H && iw >= 0 && iw < Wd ? x[((long)ih * Wd + iw) * SUB_CH] : 0.0f;
        }
    }
    float k[9];
#pragma unroll
    for (int j = 0; j < 9; j++) k[j] = bf2f(w[c * 9 + j]);
    const float bias = bf2f(b[c]);
#pragma unroll
    for (int j = 0; j < SUB_SEG; j++) {
        if (ow0 + j >= Wo) break;
        float s = bias;
#pragma unroll
        for (int kh = 0; kh < 3; kh++) {
            const int ih = oh * 2 - 1 + kh;
            if (ih < 0 || ih >= H) continue;
#pragma unroll
            for (int kw = 0; kw < 3; kw++) {
                const int iw = 2 * (ow0 + j) - 1 + kw;    // < 0 at kw 0, >= Wd at kw 2 alone
                if ((kw == 0 && iw < 0) || (kw == 2 && iw >= Wd)) continue;
                s += v[kh][2 * j + kw] * k[kh * 3 + kw];
            }
        }
        uint16_t hh, ll;
        split_bf16(s, hh, ll);
        const long o = ((long)tau * Wo + ow0 + j) * SUB_CH + c;
        out_hi[o] = hh;
        out_lo[o] = ll;
    }
}

// [T][16][256] -> [T][ch*16 + f] (backends/cpu/backend.c:222-226).
__global__ void sub_flatten_kernel(float *out, const float *in, int T) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)T * 16 * SUB_CH) return;
    const int f = (int)(i % 16);
    const int c = (int)((i / 16) % SUB_CH);
    const long t = i / (16 * SUB_CH);
    out[i] = in[(t * 16 + f) * SUB_CH + c];
}

// The same flatten, written as hi/lo bf16 planes for the pre-split GEMM.
__global__ void sub_flatten_split_kernel(uint16_t *hi, uint16_t *lo, const float *in, int T) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)T * 16 * SUB_CH) return;
    const int f = (int)(i % 16);
    const int c = (int)((i / 16) % SUB_CH);
    const long t = i / (16 * SUB_CH);
    uint16_t h, l;
    split_bf16(in[(t * 16 + f) * SUB_CH + c], h, l);
    hi[i] = h;
    lo[i] = l;
}

inline unsigned nblk(long n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// The 8-channel form reads every operand in 16-byte pieces.
static void dw_check(const float *out, const uint16_t *out_hi, const float *in, const uint16_t *dww,
                     const uint16_t *dwb, const uint16_t *bnw, const uint16_t *bnb,
                     const uint16_t *bnm, const uint16_t *bnv) {
    const uintptr_t a = (uintptr_t)out | (uintptr_t)out_hi | (uintptr_t)in | (uintptr_t)dww |
                        (uintptr_t)dwb | (uintptr_t)bnw | (uintptr_t)bnb | (uintptr_t)bnm | (uintptr_t)bnv;
    if (a & 15) {
        fprintf(stderr, "dwconv: activations and parameters must be 16-byte aligned\n");
        exit(1);
    }
}

static int relpos_qb(int) { return RQ; }

// Score rows of ldS floats: T rounded up to 16, plus 4 so that 16 rows x 4
// columns of a fragment read fall in distinct banks.
static int relpos_lds(int max_T, size_t *bytes) {
    const int ldS = (max_T + 15) / 16 * 16 + 4;
    *bytes = (size_t)RQ * ldS * sizeof(float);
    return ldS;
}

template <bool PACKED>
static void relpos_allow_lds(size_t bytes) {
    static size_t allowed = 64 * 1024;
    if (bytes <= allowed) return;
    if (hipFuncSetAttribute((const void *)relpos_attn_kernel<PACKED>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) {
        fprintf(stderr, "relpos_attn: cannot reserve %zu bytes of LDS\n", bytes);
        exit(1);
    }
    allowed = bytes;
}

extern "C" void ctk_relpos_attn(float *O, const float *Q, const float *K, const float *V,
                                const float *P, const uint16_t *pbu, const uint16_t *pbv,
                                int T, hipStream_t s) {
    if (T <= 0) return;
    if (T > 2048) {
        fprintf(stderr, "ctk_relpos_attn: T=%d exceeds the supported 2048 frames\n", T);
        exit(1);
    }
    if (((uintptr_t)Q | (uintptr_t)K | (uintptr_t)V | (uintptr_t)P) & 15) {
        fprintf(stderr, "ctk_relpos_attn: Q, K, V and P must be 16-byte aligned\n");
        exit(1);
    }
    size_t lds;
    const int ldS = relpos_lds(T, &lds);
    relpos_allow_lds<false>(lds);
    const dim3 grid((T + RQ - 1) / RQ, ENC_H);
    hipLaunchKernelGGL((relpos_attn_kernel<false>), grid, dim3(256), lds, s,
                       O, Q, K, V, P, pbu, pbv, T, T, nullptr, nullptr, nullptr, nullptr, ldS,
                       nullptr, nullptr);
}

extern "C" int ctk_relpos_plan(int *blk_seq, int *blk_q0, const int *seq_T, int n_seq) {
    int mx = 0;
    for (int i = 0; i < n_seq; i++) mx = seq_T[i] > mx ? seq_T[i] : mx;
    const int qb = relpos_qb(mx);
    int n = 0;
    for (int i = 0; i < n_seq; i++)
        for (int q0 = 0; q0 < seq_T[i]; q0 += qb) {
            if (blk_seq) { blk_seq[n] = i; blk_q0[n] = q0; }
            n++;
        }
    return n;
}

extern "C" void ctk_relpos_attn_packed(float *O, uint16_t *Oh, uint16_t *Ol, const float *Q,
                                       const float *K, const float *V, const float *P, int T_max,
                                       const uint16_t *pbu, const uint16_t *pbv, const int *seq_off,
                                       const int *seq_T, const int *blk_seq, const int *blk_q0,
                                       int n_blk, int max_T, hipStream_t s) {
    if (n_blk <= 0) return;
    if (max_T > 2048) {
        fprintf(stderr, "ctk_relpos_attn_packed: T=%d exceeds the supported 2048 frames\n", max_T);
        exit(1);
    }
    if (((uintptr_t)Q | (uintptr_t)K | (uintptr_t)V | (uintptr_t)P) & 15) {
        fprintf(stderr, "ctk_relpos_attn: Q, K, V and P must be 16-byte aligned\n");
        exit(1);
    }
    if (!O == !Oh || !Oh != !Ol) {
        fprintf(stderr, "ctk_relpos_attn_packed: give either O or both planes Oh, Ol\n");
        exit(1);
    }
    size_t lds;
    const int ldS = relpos_lds(max_T, &lds);
    relpos_allow_lds<true>(lds);
    const dim3 grid(n_blk, ENC_H);
    hipLaunchKernelGGL((relpos_attn_kernel<true>), grid, dim3(256), lds, s,
                       O, Q, K, V, P, pbu, pbv, 0, T_max, seq_off, seq_T, blk_seq, blk_q0, ldS, Oh, Ol);
}

static void launch_dwconv(float *out, uint16_t *out_hi, uint16_t *out_lo, const float *in, int M, const int *row_start,
                          const int *row_len, const uint16_t *dww, const uint16_t *dwb, const uint16_t *bnw,
                          const uint16_t *bnb, const uint16_t *bnm, const uint16_t *bnv, hipStream_t s) {
    if (M <= DW_ROWS_FEW)
        hipLaunchKernelGGL(dwconv_bn_silu_kernel<1>, dim3(nblk((long)M * (ENC_D / 8))), dim3(256), 0, s, out, out_hi,
                           out_lo, in, M, row_start, row_len, dww, dwb, bnw, bnb, bnm, bnv);
    else
        hipLaunchKernelGGL(dwconv_bn_silu_kernel<8>, dim3(nblk((long)((M + 7) / 8) * (ENC_D / 8))), dim3(256), 0, s, out,
                           out_hi, out_lo, in, M, row_start, row_len, dww, dwb, bnw, bnb, bnm, bnv);
}

extern "C" void ctk_dwconv_bn_silu(float *out, const float *in, int T, const uint16_t *dww,
                                   const uint16_t *dwb, const uint16_t *bnw, const uint16_t *bnb,
                                   const uint16_t *bnm, const uint16_t *bnv, hipStream_t s) {
    if (T <= 0) return;
    dw_check(out, nullptr, in, dww, dwb, bnw, bnb, bnm, bnv);
    launch_dwconv(out, nullptr, nullptr, in, T, nullptr, nullptr, dww, dwb, bnw, bnb, bnm, bnv, s);
}

extern "C" void ctk_dwconv_bn_silu_packed(uint16_t *out_hi, uint16_t *out_lo, const float *in, int M,
                                          const int *row_start, const int *row_len,
                                          const uint16_t *dww, const uint16_t *dwb,
                                          const uint16_t *bnw, const uint16_t *bnb,
                                          const uint16_t *bnm, const uint16_t *bnv, hipStream_t s) {
    if (M <= 0) return;
    dw_check(nullptr, out_hi, in, dww, dwb, bnw, bnb, bnm, bnv);
    if ((uintptr_t)out_lo & 15) { fprintf(stderr, "dwconv: outputs must be 16-byte aligned\n"); exit(1); }
    launch_dwconv(nullptr, out_hi, out_lo, in, M, row_start, row_len, dww, dwb, bnw, bnb, bnm, bnv, s);
}

extern "C" void ctk_sub_conv0(float *out, const float *mel, int T_mel, int stride,
                              const uint16_t *w, const uint16_t *b, hipStream_t s) {
    const long n = (long)((T_mel + 1) / 2) * 64 * SUB_CH;
    if (n <= 0) return;
    hipLaunchKernelGGL(sub_conv0_kernel, dim3(nblk(n)), dim3(256), 0, s, out, mel, T_mel, stride, w, b);
}

extern "C" void ctk_sub_dwconv(float *out, const float *in, int H, int Wd,
                               const uint16_t *w, const uint16_t *b, hipStream_t s) {
    const long n = (long)((H + 1) / 2) * ((Wd + 1) / 2) * SUB_CH;
    if (n <= 0) return;
    hipLaunchKernelGGL(sub_dwconv_kernel, dim3(nblk(n)), dim3(256), 0, s, out, in, H, Wd, w, b);
}

extern "C" void ctk_sub_conv0_dw_packed(uint16_t *out_hi, uint16_t *out_lo, const float *mel, const int *o1,
                                        const int *o2,
                                        const int *tmel, const int *moff, int n, int rows2,
                                        const uint16_t *w0, const uint16_t *b0, const uint16_t *wd,
                                        const uint16_t *bd, hipStream_t s) {
    if (rows2 <= 0 || n <= 0) return;
    hipLaunchKernelGGL(sub_conv0_dw_packed_kernel, dim3(rows2, 32 / SUB_SEG), dim3(256), 0, s, out_hi, out_lo, mel, o1,
                       o2, tmel, moff, n, 0, 0, w0, b0, wd, bd);
}

extern "C" void ctk_sub_conv0_dw(uint16_t *out_hi, uint16_t *out_lo, const float *mel, int T_mel, int stride,
                                 const uint16_t *w0, const uint16_t *b0, const uint16_t *wd, const uint16_t *bd,
                                 hipStream_t s) {
    const int rows2 = ((T_mel + 1) / 2 + 1) / 2;
    if (T_mel <= 0) return;
    hipLaunchKernelGGL(sub_conv0_dw_packed_kernel, dim3(rows2, 32 / SUB_SEG), dim3(256), 0, s, out_hi, out_lo, mel,
                       nullptr, nullptr, nullptr, nullptr, 1, T_mel, stride, w0, b0, wd, bd);
}

extern "C" void ctk_sub_dw_split_packed(uint16_t *out_hi, uint16_t *out_lo, const float *in, const int *oin,
                                        const int *oout, int n, int rows_out, int Wd, const uint16_t *w,
                                        const uint16_t *b, hipStream_t s) {
    if (rows_out <= 0 || n <= 0) return;
    hipLaunchKernelGGL(sub_dw_split_packed_kernel, dim3(rows_out, ((Wd + 1) / 2 + SUB_SEG - 1) / SUB_SEG), dim3(256), 0, s,
                       out_hi, out_lo, in, oin, oout, n, 0, Wd, w, b);
}

extern "C" void ctk_sub_dw_split(uint16_t *out_hi, uint16_t *out_lo, const float *in, int H, int Wd, const uint16_t *w,
                                 const uint16_t *b, hipStream_t s) {
    if (H <= 0) return;
    hipLaunchKernelGGL(sub_dw_split_packed_kernel, dim3((H + 1) / 2, ((Wd + 1) / 2 + SUB_SEG - 1) / SUB_SEG), dim3(256), 0,
                       s, out_hi, out_lo, in, nullptr, nullptr, 1, H, Wd, w, b);
}

extern "C" void ctk_sub_flatten_split(uint16_t *hi, uint16_t *lo, const float *in, int T, hipStream_t s) {
    const long n = (long)T * 16 * SUB_CH;
    if (n <= 0) return;
    hipLaunchKernelGGL(sub_flatten_split_kernel, dim3(nblk(n)), dim3(256), 0, s, hi, lo, in, T);
}

extern "C" void ctk_sub_flatten(float *out, const float *in, int T, hipStream_t s) {
    const long n = (long)T * 16 * SUB_CH;
    if (n <= 0) return;
    hipLaunchKernelGGL(sub_flatten_kernel, dim3(nblk(n)), dim3(256), 0, s, out, in, T);
}
