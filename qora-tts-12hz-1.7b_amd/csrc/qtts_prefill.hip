// qtts_prefill.hip — batched talker prefill for long prompts on the matrix
// cores (prefill_talker_raw_from, talker.rs:379-482).
//
// A prompt of M rows runs layer by layer (k_resid_norm first: the input rows
// normed and split): per layer
//   k_q4_gemm (parts)    [M x 2048] x [2048 x 4096] q|k|v    talker.rs:392-400
//   k_prefill_qkv_post   parts summed, QK-norm, RoPE,        talker.rs:402-425
//                        K/V append
//   k_prefill_attn_mx    causal attention over the cache,    talker.rs:427-458
//                        its rows split for the o-projection
//   k_q4_gemm (parts)    attn x o_proj                       talker.rs:460
//   k_resid_norm         x += parts; post-attention norm,    talker.rs:461-468
//                        the normed rows split
//   k_q4_gemm (swiglu)   silu(gate) * up, split              talker.rs:470-474
//   k_q4_gemm (parts)    h x down_proj                       talker.rs:475
//   k_resid_norm         x += parts; next layer's norm       talker.rs:476
// then k_final_rms on the last row (talker.rs:477-481).
//
// k_q4_gemm (qtts_gemm.hip) contracts on the f16 matrix cores with split
// operands, f32-accurate.  With QTTS_GEMM_F32=1, or in a layer with a weight
// whose scales leave the split's range, the GEMMs run on k_gemm_q4 below instead:
// f32 rows, v_mfma_f32_16x16x4_f32, the decode GEMV's tiled weights.

#include "qtts_device.h"
#include "qtts_kernels.h"
#include "qtts_devutil.h"
#include "qtts_mfma.h"

#include <algorithm>
#include <cmath>

namespace qtts {

// ---------------------------------------------------------------------------
// Q4 GEMM on the f32 matrix instructions: Y[M][n] (op)= A'[M][K] x W[K][n],
// with A' = A * inv[row] * gamma[k] when a norm is fused (the reference's
// x * inv_rms * gamma order) and W dequantised as (nibble - 8) * scale,
// exact in f32.
//
// Workgroup tile: 16*MB rows x 128 columns (four 32-column groups), K in
// chunks of 32 through double-buffered LDS; a weight with S k-slices runs S
// workgroups per tile, each writing its partial sums (GEMM_PART) for the
// consumer kernel to add in slice order.  All four waves cover every row
// of the tile; wave w owns the 16-column blocks c = (w&1) + 4*(w>>1) and
// c + 2, so for the gate|up weight (groups interleaved gate, up, gate, up)
// a lane holds gate and up of the same output column and the SwiGLU
// epilogue stays in registers.
//
// v_mfma_f32_16x16x4_f32 lane layout: A operand lane l = A[l%16][l/16],
// B operand B[l/16][l%16], result element i = D[4*(l/16)+i][l%16].  The
// contraction index of lane group q = l/16 at sub-step e is k = 4q + e of a
// 16-wide slice, so each lane reads its A row and B column as one 16-byte
// LDS load (As is [row][k], Bs is [column][k]).
// ---------------------------------------------------------------------------

constexpr int GN = MFMA_N, GK = MFMA_K, GLD = MFMA_LD;

enum GemmEpi : int { GEMM_STORE = 0, GEMM_PART = 1, GEMM_SWIGLU = 2, GEMM_BIAS = 3, GEMM_BIAS_SILU = 4 };

struct GemmA {
    const float *A;
    int lda;
    const float *inv;        // per-row 1/rms, or null
    const uint16_t *gamma;   // [K] f16, or null
    int M;
};

struct GemmOut {
    float *Y;
    int ldy, ncols;
    const float *bias;       // GEMM_BIAS*: [ncols]
    size_t slice_stride;     // GEMM_PART: floats between the slices' blocks
};

// word 3 of a raw buffer descriptor on this GPU family (untyped dword
// access, no swizzle, offsets checked against the record count in bytes)
constexpr int BUF_RSRC_W3 = 0x00020000;

template <int MB, int EPI, bool NORM>
__global__ void __launch_bounds__(256, 2)
k_gemm_q4(GemmA a, Q4Tiled w, GemmOut o, int tm, int S)
{
    constexpr int BM = 16 * MB;
    constexpr int NA = (BM * GK / 4 + 255) / 256;   // 16-byte A slots per thread
    __shared__ __attribute__((aligned(16))) float As[2][BM * GLD];
    __shared__ __attribute__((aligned(16))) float Bs[2][GN * GLD];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    // Workgroups are dealt round-robin to the 8 XCDs: give each XCD a
    // contiguous run of tiles (row blocks fastest) so the row blocks that
    // share a weight tile share that XCD's L2.
    const int nwg = gridDim.x, id = blockIdx.x;
    const int xcd = id & 7, qq = nwg >> 3, rem = nwg & 7;
    const int logical = xcd * qq + min(xcd, rem) + (id >> 3);
    const int mt = logical % tm, rest = logical / tm;
    const int sl = rest % S, nt = rest / S;
    const int m0 = mt * BM;
    const int nch = w.k / GK, c0 = sl * nch / S, c1 = (sl + 1) * nch / S;
    const TileShape ts = tile_shape(w.cfg);
    const int P = ts.T / ts.GB;
    const bool wave_groups = (ts.T / 64) % ts.GB == 0;

    // A staging: slot i = t + 256 j (clamped: spare threads repeat the last
    // slot) covers row i / 8, floats 4 (i % 8)..+4 of the chunk.  Rows past
    // M load row M-1 and stage zeros.
    uint32_t aoffg[NA];
    int aoff[NA], akk[NA];
    float amul[NA];
#pragma unroll
    for (int j = 0; j < NA; j++) {
        const int slot = min(t + 256 * j, BM * GK / 4 - 1);
        const int r = slot >> 3, m = m0 + r;
        aoffg[j] = (uint32_t)(min(m, a.M - 1) * a.lda + 4 * (slot & 7)) * 4u;
        aoff[j] = r * GLD + 4 * (slot & 7);
        akk[j] = 4 * (slot & 7);
        amul[j] = m < a.M ? (NORM ? a.inv[m] : 1.0f) : 0.0f;
    }
    // B staging: bytes 4*qw..+4 (8 columns) of row kr of groups 4*nt + gi
    // and + 2; groups past G stage zeros.  gi is the same across a wave: read
    // as a scalar, so the tile addresses below come from the scalar unit.
    const int kr = t & 31, qw = (t >> 5) & 3;
    const int gi = __builtin_amdgcn_readfirstlane(t >> 7);
    int gt[2], gct[2];
    bool gok[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int g = 4 * nt + gi + 2 * h;
        gok[h] = g < w.G;
        const int gc = min(g, w.G - 1);
        gct[h] = gc / ts.GB;
        gt[h] = gc - gct[h] * ts.GB;
    }
    // tile position of (pt, group): one group per wave when wave_groups,
    // else groups interleaved by thread -- one formula for both
    const int tA = wave_groups ? 1 : ts.GB, tB = wave_groups ? 64 : 1;
    // With P >= 32 (every tile but 8 groups x 128 threads) a chunk's 32 rows
    // lie in one tile row r0 and one 64-position block (pt0 is a multiple of
    // 32), so tt = ttu(k0) + kr * tA + gt * tB: a wave-uniform part per chunk
    // and this constant thread part.
    uint32_t thr_w[2], thr_s[2];   // byte offsets of the word and the scale from the chunk's base
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t tt = (uint32_t)(kr * tA + gt[h] * tB);
        thr_w[h] = tt * 16u + 4u * (uint32_t)qw;
        thr_s[h] = tt * (uint32_t)ts.R * 2u;
    }
    // A and the tiled weight are read through buffer descriptors: the
    // chunk's wave-uniform offset goes in a scalar register (soffset), the
    // thread's byte offset is a constant vector register, so a chunk's loads
    // need no per-chunk vector address arithmetic
    const __amdgpu_buffer_rsrc_t rsA =
        __builtin_amdgcn_make_buffer_rsrc((void *)a.A, (short)0, (int)((size_t)a.M * a.lda * 4), BUF_RSRC_W3);
    const __amdgpu_buffer_rsrc_t rsW =
        __builtin_amdgcn_make_buffer_rsrc((void *)w.data, (short)0, (int)((size_t)w.S * w.CT * w.tile_bytes), BUF_RSRC_W3);
    struct Fetch {
        f32x4 ra[NA];
        uint32_t rg[NA][2];
        uint32_t rb[2], rs[2];
    };
    auto fetch = [&](Fetch &f, int k0) {
#pragma unroll
        for (int j = 0; j < NA; j++) {
            f.ra[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsA, aoffg[j], k0 * 4, 0));
            if (NORM) {
                const uint2 gv = *(const uint2 *)(a.gamma + k0 + akk[j]);
                f.rg[j][0] = gv.x;
                f.rg[j][1] = gv.y;
            }
        }
        // k = k0 + kr: slice s, row r, position pt of the tiled layout; k0 is
        // a multiple of 32, so only P = 16 splits a chunk over rows
        const int s = k0 / w.KC, rr0 = k0 - s * w.KC, r0 = rr0 / P, pt0 = rr0 - r0 * P;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t word;
            uint16_t sc;
            if (P >= 32) {
                const int ttu = (pt0 >> 6) * 64 * ts.GB + (pt0 & 63) * tA;
                const int tb = (s * w.CT + gct[h]) * w.tile_bytes;
                word = __builtin_amdgcn_raw_buffer_load_b32(rsW, thr_w[h], tb + (r0 * ts.T + ttu) * 16, 0);
                sc = __builtin_amdgcn_raw_buffer_load_b16(rsW, thr_s[h], tb + ts.R * ts.T * 16 + (ttu * ts.R + r0) * 2, 0);
            } else {
                const uint8_t *tile = w.data + (size_t)(s * w.CT + gct[h]) * w.tile_bytes;
                const int ptk = pt0 + kr;
                const int r = r0 + (ptk >> 4), pt = ptk & 15;
                const int tt = (pt >> 6) * 64 * ts.GB + (pt & 63) * tA + gt[h] * tB;
                word = *(const uint32_t *)(tile + ((size_t)r * ts.T + tt) * 16 + 4 * qw);
                sc = *((const uint16_t *)(tile + (size_t)ts.R * ts.T * 16) + tt * ts.R + r);
            }
            f.rb[h] = gok[h] ? word : 0x88888888u;
            f.rs[h] = gok[h] ? (uint32_t)sc : 0u;
        }
    };
    auto stage = [&](const Fetch &f, int buf) {
#pragma unroll
        for (int j = 0; j < NA; j++) {
            f32x4 x = f.ra[j] * amul[j];
            if (NORM) {
                x.x *= h2f(f.rg[j][0] & 0xFFFFu);
                x.y *= h2f(f.rg[j][0] >> 16);
                x.z *= h2f(f.rg[j][1] & 0xFFFFu);
                x.w *= h2f(f.rg[j][1] >> 16);
            }
            *(f32x4 *)&As[buf][aoff[j]] = x;
        }
        // 8 columns 32*g + 8*qw + c, c = 0..7: byte c/2, low nibble even c
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float sc = h2f(f.rs[h]);
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const float v = (float)((int)((f.rb[h] >> (4 * c)) & 15u) - 8) * sc;
                Bs[buf][(32 * gi + 8 * qw + 64 * h + c) * GLD + kr] = v;
            }
        }
    };

    // compute roles: wave w owns 16-column blocks cb0 and cb0 + 2
    const int r16 = lane & 15, q = lane >> 4;
    const int cb0 = (wv & 1) + 4 * (wv >> 1);
    const int cb[2] = {cb0, cb0 + 2};
    f32x4 acc[MB][2];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    mfma_pipeline<Fetch>(
        c1 - c0, [&](Fetch &f, int c) { fetch(f, (c0 + c) * GK); }, stage,
        [&](int buf) { mfma_chunk<MB>(acc, As[buf], Bs[buf], cb, lane); });

    // epilogue: element e of acc[i][j] is row 16i + 4q + e of the tile,
    // column 128nt + 16(cb0 + 2j) + r16
    float *Y = o.Y + (EPI == GEMM_PART ? (size_t)sl * o.slice_stride : 0);
#pragma unroll
    for (int i = 0; i < MB; i++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int m = m0 + 16 * i + 4 * q + e;
            if (m >= a.M) continue;
            float *yr = Y + (size_t)m * o.ldy;
            if constexpr (EPI == GEMM_SWIGLU) {
                // groups (4nt, 4nt+1) and (4nt+2, 4nt+3) are (gate, up) pairs
                const int col = 32 * (2 * nt + (wv >> 1)) + 16 * (wv & 1) + r16;
                if (col < o.ncols) yr[col] = silu_f(acc[i][0][e]) * acc[i][1][e];
            } else {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int col = GN * nt + 16 * (cb0 + 2 * j) + r16;
                    if (col >= o.ncols) continue;
                    const float v = acc[i][j][e];
                    if (EPI == GEMM_BIAS) yr[col] = v + o.bias[col];
                    else if (EPI == GEMM_BIAS_SILU) yr[col] = silu_f(v + o.bias[col]);
                    else yr[col] = v;
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// q|k|v partial rows -> QK-norm (talker.rs:89-99), RoPE at start + row
// (rope.rs:79-92), q rows out, K (normed, roped) and V (raw) appended to the
// paged cache at the same position (talker.rs:419-425).  One wave per (row,
// head): heads 0..15 q, 16..23 k, 24..31 v; lane holds dims (l, l+64).
// ---------------------------------------------------------------------------

template <int NP>
__global__ void __launch_bounds__(256)
k_prefill_qkv_post(MmParts p, int M, int64_t start, const uint16_t *qn_g, const uint16_t *kn_g,
                   const float *rope_cos, const float *rope_sin, KvPaged kv, int layer, float *q, int ldq)
{
    const int lane = threadIdx.x & 63;
    const int m = blockIdx.x, hh = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (m >= M) return;
    const int64_t pos = start + m;
    const size_t at = (size_t)m * p.ld + hh * HEAD_DIM;
    const float x0 = sum_parts<NP>(p, at + lane), x1 = sum_parts<NP>(p, at + lane + 64);
    if (hh >= 24) {
        float *vp = kv_ptr(kv, layer, (int)pos, hh - 24, 1);
        vp[lane] = x0;
        vp[lane + 64] = x1;
        return;
    }
    const uint16_t *gam = hh < 16 ? qn_g : kn_g;
    const float ss = wave_sum_dpp(x0 * x0 + x1 * x1);
    const float inv = 1.0f / sqrtf(ss / 128.0f + 1e-6f);
    const float n0 = x0 * inv * h2f(gam[lane]), n1 = x1 * inv * h2f(gam[lane + 64]);
    const float cs = rope_cos[pos * 64 + lane], sn = rope_sin[pos * 64 + lane];
    const float r0 = n0 * cs - n1 * sn, r1 = n1 * cs + n0 * sn;
    float *out = hh < 16 ? q + (size_t)m * ldq + hh * HEAD_DIM : kv_ptr(kv, layer, (int)pos, hh - 16, 0);
    out[lane] = r0;
    out[lane + 64] = r1;
}

// ---------------------------------------------------------------------------
// Residual add of a projection's partial sums (x += parts: talker.rs:461,
// 474; p.n = 0: nothing to add) fused with the next RMSNorm (gemv.rs:445-454):
// 1/rms of the updated row, and with a gamma the normed row (x * inv) * gamma
// split for the GEMM, staged times 2^nshift.  One workgroup per row of at
// most 2048 columns, each thread's values in registers.
// ---------------------------------------------------------------------------

template <int NP>
__global__ void __launch_bounds__(256)
k_resid_norm(float *x, int H, MmParts p, float *inv_out, const uint16_t *gamma, int nshift, uint8_t *split, int kc)
{
    __shared__ float red[4];
    const int t = threadIdx.x, m = blockIdx.x;
    float *xr = x + (size_t)m * H;
    f32x4 v[2];
    uint2 g[2];
    float ss = 0.0f;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int j = 4 * t + 1024 * u;
        v[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        g[u] = uint2{0, 0};
        if (j >= H) continue;
        v[u] = ld4(xr + j);
        if (gamma) g[u] = *(const uint2 *)(gamma + j);
        if (p.n) {
            v[u] += sum_parts4<NP>(p, (size_t)m * p.ld + j);
            *(f32x4 *)(xr + j) = v[u];
        }
        ss = fmaf(v[u].x, v[u].x, ss);
        ss = fmaf(v[u].y, v[u].y, ss);
        ss = fmaf(v[u].z, v[u].z, ss);
        ss = fmaf(v[u].w, v[u].w, ss);
    }
    ss = wave_sum_dpp(ss);
    if ((t & 63) == 0) red[t >> 6] = ss;
    __syncthreads();
    const float inv = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)H + 1e-6f);
    if (inv_out && t == 0) inv_out[m] = inv;
    if (!split) return;
    const float mul = inv * __builtin_ldexpf(1.0f, nshift);
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int j = 4 * t + 1024 * u;
        if (j >= 64 * kc) continue;
        f32x4 y = v[u] * mul;
        y.x *= h2f(g[u].x & 0xFFFFu);
        y.y *= h2f(g[u].x >> 16);
        y.z *= h2f(g[u].y & 0xFFFFu);
        y.w *= h2f(g[u].y >> 16);
        uint32_t h0, l0, h1, l1;
        split_f16_pair<true>(y.x, y.y, h0, l0);
        split_f16_pair<true>(y.z, y.w, h1, l1);
        uint8_t *o = split + ((size_t)m * kc + (j >> 6)) * 256 + ((j >> 5) & 1) * 128 + (j & 31) * 2;
        *(uint2 *)o = uint2{h0, h1};
        *(uint2 *)(o + 64) = uint2{l0, l1};
    }
}

// ---------------------------------------------------------------------------
// Causal prefill attention (talker.rs:427-458): query row m (position
// start + m) attends to cached positions 0..start+m.  Workgroup (block of
// QB rows, kv head h) serves q heads 2h and 2h+1 of its rows -- 2*QB
// queries -- with one pass over the K/V pages they need and an online
// softmax across pages (the reference's softmax_raw over the whole row,
// regrouped).  Thread t keeps K row t/4 of the page (dims 32*(t%4)..+32)
// and V dims 4*(t%32)..+4 of page rows 8*(t/32)..+8 in registers, reused
// by every query of the block; the next page's K/V loads are issued before
// the current page's probabilities are formed.
// ---------------------------------------------------------------------------

template <int QB>
__global__ void __launch_bounds__(256)
k_prefill_attn(const float *q, int ldq, int M, int64_t start, KvPaged kv, int layer, float *out, int ldo)
{
    constexpr int NQ = 2 * QB;                    // query j: row j/2, head 2h + j%2
    __shared__ __attribute__((aligned(16))) float qs[NQ][HEAD_DIM];
    __shared__ float pr[NQ][KV_PAGE];
    __shared__ float wmax[4][NQ], wsum[4][NQ];
    __shared__ __attribute__((aligned(16))) float ored[4][NQ][HEAD_DIM];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int m0 = blockIdx.x * QB, h = blockIdx.y;
    const int nq = min(QB, M - m0);
    const int Lmax = (int)(start + m0 + nq);      // positions the block's last row attends
    const int C = (Lmax + KV_PAGE - 1) / KV_PAGE;
    const float scale = 1.0f / sqrtf(128.0f);
    const int tk = t >> 2, kq = t & 3;
    const int vd = (t & 31) * 4, vt0 = (t >> 5) * 8;
    for (int i = t; i < NQ * HEAD_DIM; i += 256) {
        const int j = i / HEAD_DIM, d = i - j * HEAD_DIM, r = j >> 1;
        qs[j][d] = r < nq ? q[(size_t)(m0 + r) * ldq + (2 * h + (j & 1)) * HEAD_DIM + d] : 0.0f;
    }
    float mrun[NQ], lrun[NQ];
    f32x4 acc[NQ];
#pragma unroll
    for (int j = 0; j < NQ; j++) {
        mrun[j] = -INFINITY;
        lrun[j] = 0.0f;
        acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    f32x4 kk[8], vv[8];
    {
        const float *Kp = kv_ptr(kv, layer, 0, h, 0), *Vp = kv_ptr(kv, layer, 0, h, 1);
#pragma unroll
        for (int i = 0; i < 8; i++) kk[i] = ld4(Kp + tk * HEAD_DIM + kq * 32 + 4 * i);
#pragma unroll
        for (int i = 0; i < 8; i++) vv[i] = ld4(Vp + (vt0 + i) * HEAD_DIM + vd);
    }
    __syncthreads();
    for (int c = 0; c < C; c++) {
        const int pos = c * KV_PAGE + tk;
        // scores of K row tk against every query of the block
        float sc[NQ];
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            float d = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const f32x4 qa = *(const f32x4 *)&qs[j][kq * 32 + 4 * i];
                const f32x4 k = kk[i];
                d = fmaf(qa.x, k.x, fmaf(qa.y, k.y, fmaf(qa.z, k.z, fmaf(qa.w, k.w, d))));
            }
            d += dpp_mov<0xB1>(d);
            d += dpp_mov<0x4E>(d);
            const bool valid = (j >> 1) < nq && pos <= (int)start + m0 + (j >> 1);
            sc[j] = valid ? d * scale : -INFINITY;
        }
        // this page's V rows stay in registers; the next page's K is free to load
        f32x4 vcur[8];
#pragma unroll
        for (int i = 0; i < 8; i++) vcur[i] = vv[i];
        if (c + 1 < C) {
            const float *Kp = kv_ptr(kv, layer, (c + 1) * KV_PAGE, h, 0), *Vp = kv_ptr(kv, layer, (c + 1) * KV_PAGE, h, 1);
#pragma unroll
            for (int i = 0; i < 8; i++) kk[i] = ld4(Kp + tk * HEAD_DIM + kq * 32 + 4 * i);
#pragma unroll
            for (int i = 0; i < 8; i++) vv[i] = ld4(Vp + (vt0 + i) * HEAD_DIM + vd);
        }
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            const float mw = wave_max_dpp(sc[j]);
            if (lane == 0) wmax[wv][j] = mw;
        }
        __syncthreads();
        float f[NQ];
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            const float pm = fmaxf(fmaxf(wmax[0][j], wmax[1][j]), fmaxf(wmax[2][j], wmax[3][j]));
            const float mn = fmaxf(mrun[j], pm);
            f[j] = mn == -INFINITY ? 0.0f : expf(mrun[j] - mn);   // 0 before the row's first position
            const float e = sc[j] == -INFINITY ? 0.0f : expf(sc[j] - mn);
            if (kq == 0) pr[j][tk] = e;
            const float lw = wave_sum_dpp(kq == 0 ? e : 0.0f);
            if (lane == 0) wsum[wv][j] = lw;
            mrun[j] = mn;
        }
        __syncthreads();
        // P.V over this thread's 8 rows and 4 dims (rows past the written
        // cache may hold anything and are skipped)
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            f32x4 a = acc[j] * f[j];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const bool ok = c * KV_PAGE + vt0 + i < Lmax;
                const float p = pr[j][vt0 + i];
                const f32x4 v = vcur[i];
                a.x = ok ? fmaf(p, v.x, a.x) : a.x; a.y = ok ? fmaf(p, v.y, a.y) : a.y;
                a.z = ok ? fmaf(p, v.z, a.z) : a.z; a.w = ok ? fmaf(p, v.w, a.w) : a.w;
            }
            acc[j] = a;
            lrun[j] = lrun[j] * f[j] + ((wsum[0][j] + wsum[1][j]) + (wsum[2][j] + wsum[3][j]));
        }
        __syncthreads();                             // wmax, wsum and pr are reused by the next page
    }
    // rows 8*(t/32): lanes l and l^32 of a wave hold the same dims
#pragma unroll
    for (int j = 0; j < NQ; j++) {
        f32x4 a = acc[j];
        a.x += __shfl_xor(a.x, 32); a.y += __shfl_xor(a.y, 32);
        a.z += __shfl_xor(a.z, 32); a.w += __shfl_xor(a.w, 32);
        if (lane < 32) *(f32x4 *)&ored[wv][j][vd] = a;
    }
    __syncthreads();
    for (int i = t; i < NQ * HEAD_DIM; i += 256) {
        const int j = i / HEAD_DIM, d = i - j * HEAD_DIM, r = j >> 1;
        if (r < nq) {
            const float o = (ored[0][j][d] + ored[1][j][d]) + (ored[2][j][d] + ored[3][j][d]);
            float l = 0.0f;
#pragma unroll
            for (int jj = 0; jj < NQ; jj++) l = jj == j ? lrun[jj] : l;
            out[(size_t)(m0 + r) * ldo + (2 * h + (j & 1)) * HEAD_DIM + d] = o / l;
        }
    }
}

// rows per workgroup: at 400 rows x 28 layers, 1 / 2 / 4 / 8 rows measured
// 75 / 62 / 76 / 140 us per layer (the per-page chain and the occupancy bind)
constexpr int PREFILL_ATTN_QB = 2;

// ---------------------------------------------------------------------------
// The same causal attention on the matrix cores.  Workgroup (block of 8
// rows, kv head h): 16 queries, query i = (row i/2, head 2h + i%2).  Wave w
// takes positions 16w..16w+15 of every 64-position page and keeps its own
// online softmax (max, sum, output) per query; the four waves are merged
// once at the end, in wave order.  Per page and wave:
//   S^T = K Q^T on v_mfma_f32_16x16x32_f16: A = the wave's 16 K rows, B = the
//        16 queries; lane l then holds query l%16 at positions 4(l/16)..+3,
//   which is the B operand of
//   O^T += V^T P^T on v_mfma_f32_16x16x16_f16 (A = V^T: dims 16t + l%16 at
//        the same 4 positions), so the probabilities never leave the lane
//        and the softmax statistics of a query stay in its lanes.
// Every product is split f16 (hi*hi + hi*lo + lo*hi, f32 accumulation), as
// in the GEMM.  Cache rows at or past the block's length may hold anything:
// their scores are replaced by -inf and their V values by 0 (selects).  A
// query's result depends only on its own row and position, not on the
// block it shares, so a prompt prefilled in pieces matches one prefilled
// whole bit for bit.
// ---------------------------------------------------------------------------

// (results straight into matrix instructions: the register form of the split)
__device__ __forceinline__ void split8(const f32x4 &a, const f32x4 &b, half8 &hi, half8 &lo)
{
    uint32_t h[4], l[4];
    split_f16_pair<true>(a.x, a.y, h[0], l[0]);
    split_f16_pair<true>(a.z, a.w, h[1], l[1]);
    split_f16_pair<true>(b.x, b.y, h[2], l[2]);
    split_f16_pair<true>(b.z, b.w, h[3], l[3]);
    hi = __builtin_bit_cast(half8, uint4{h[0], h[1], h[2], h[3]});
    lo = __builtin_bit_cast(half8, uint4{l[0], l[1], l[2], l[3]});
}

__device__ __forceinline__ void split4(float a, float b, float c, float d, half4 &hi, half4 &lo)
{
    uint32_t h[2], l[2];
    split_f16_pair<true>(a, b, h[0], l[0]);
    split_f16_pair<true>(c, d, h[1], l[1]);
    hi = __builtin_bit_cast(half4, uint2{h[0], h[1]});
    lo = __builtin_bit_cast(half4, uint2{l[0], l[1]});
}

// Split range: with SC, q, K and V are staged times 2^sq, 2^sk, 2^sv, static
// powers of two from the layer's bounds (the QK-norm gammas, the input norm
// and v_proj) for a layer whose bounds leave [2^-4, 2^14], so their f16
// halves neither overflow nor go subnormal; the scores are scaled back by
// 2^-(sq + sk), the output by 2^-sv (exact).  Layers within that band run
// without the scalings (SC false).
template <bool SC>
__global__ void __launch_bounds__(256)
k_prefill_attn_mx(const float *q, int ldq, int M, int64_t start, KvPaged kv, int layer, float *out, int ldo,
                  uint8_t *split, float *rsc, int ldr, int sq, int sk, int sv)
{
    constexpr int QR = 8;
    __shared__ float smax[4][16], ssum[4][16];
    __shared__ __attribute__((aligned(16))) float so[4][16][HEAD_DIM + 4];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, r16 = lane & 15, qd = lane >> 4;
    const int m0 = blockIdx.x * QR, h = blockIdx.y;
    const int nq = min(QR, M - m0);
    const int Lmax = (int)(start + m0 + nq);     // positions 0..Lmax-1 hold the block's keys
    const int C = (Lmax + KV_PAGE - 1) / KV_PAGE;
    const float scale = 1.0f / sqrtf(128.0f);
    // this lane's query: row r16/2 of the block, head 2h + r16%2
    const int qrow = r16 >> 1;
    const int qpos = (int)start + m0 + qrow;

    // Q as the B operand of S^T: dims 32c + 8qd..+7 of the lane's query
    half8 qh[4], ql[4];
    {
        const bool ok = qrow < nq;
        const float *qp = q + (size_t)(m0 + min(qrow, nq - 1)) * ldq + (2 * h + (r16 & 1)) * HEAD_DIM + 8 * qd;
        const float pq = __builtin_ldexpf(1.0f, sq);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            f32x4 a = ld4(qp + 32 * c), b = ld4(qp + 32 * c + 4);
            if constexpr (SC) {
                a *= pq;
                b *= pq;
            }
            const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
            split8(ok ? a : z, ok ? b : z, qh[c], ql[c]);
        }
    }
    const float pk = __builtin_ldexpf(1.0f, sk), pv = __builtin_ldexpf(1.0f, sv);
    const float uqk = __builtin_ldexpf(1.0f, -(sq + sk)), uv = __builtin_ldexpf(1.0f, -sv);
    // K rows p0 + r16 (dims 32c + 8qd..+7) and V rows p0 + 4qd + kk (dims
    // 16t + r16) of page c, p0 = 64c + 16w
    auto load_kv = [&](int c, f32x4 (&kr)[8], float (&vr)[32]) {
        const float *Kp = kv_ptr(kv, layer, c * KV_PAGE, h, 0) + (16 * wv + r16) * HEAD_DIM + 8 * qd;
        const float *Vp = kv_ptr(kv, layer, c * KV_PAGE, h, 1) + (16 * wv + 4 * qd) * HEAD_DIM + r16;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            kr[2 * i] = ld4(Kp + 32 * i);
            kr[2 * i + 1] = ld4(Kp + 32 * i + 4);
        }
#pragma unroll
        for (int tt = 0; tt < 8; tt++)
#pragma unroll
            for (int kk = 0; kk < 4; kk++) vr[tt * 4 + kk] = Vp[kk * HEAD_DIM + 16 * tt];
    };
    float mrun = -INFINITY, lrun = 0.0f;
    f32x4 o[8];
#pragma unroll
    for (int tt = 0; tt < 8; tt++) o[tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 kn[8];
    float vn[32];
    load_kv(0, kn, vn);
    for (int c = 0; c < C; c++) {
        f32x4 kr[8];
        float vr[32];
#pragma unroll
        for (int i = 0; i < 8; i++) kr[i] = kn[i];
#pragma unroll
        for (int i = 0; i < 32; i++) vr[i] = vn[i];
        if (c + 1 < C) load_kv(c + 1, kn, vn);
        const int p0 = c * KV_PAGE + 16 * wv;
        // scores S^T[position p0 + 4qd + e][query r16]
        f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            half8 kh, kl;
            if constexpr (SC)
                split8(kr[2 * i] * pk, kr[2 * i + 1] * pk, kh, kl);
            else
                split8(kr[2 * i], kr[2 * i + 1], kh, kl);
            s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl, qh[i], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, ql[i], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, qh[i], s, 0, 0, 0);
        }
        // causal mask, the wave's online softmax for query r16 (its four
        // lanes r16 + 16j combine by lane swaps, in a fixed order)
        float sc[4];
#pragma unroll
        for (int e = 0; e < 4; e++) sc[e] = p0 + 4 * qd + e <= qpos ? (SC ? s[e] * uqk : s[e]) * scale : -INFINITY;
        float mx = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(mrun, mx);
        const float alpha = mn == -INFINITY ? 1.0f : expf(mrun - mn);
        float p[4];
#pragma unroll
        for (int e = 0; e < 4; e++) p[e] = sc[e] == -INFINITY ? 0.0f : expf(sc[e] - mn);
        float ps = (p[0] + p[1]) + (p[2] + p[3]);
        ps += __shfl_xor(ps, 16);
        ps += __shfl_xor(ps, 32);
        lrun = lrun * alpha + ps;
        mrun = mn;
        half4 ph, pl;
        split4(p[0], p[1], p[2], p[3], ph, pl);
        // O^T[dim 16t + 4qd + e][query r16] += V^T P^T
#pragma unroll
        for (int tt = 0; tt < 8; tt++) {
            float v[4];
#pragma unroll
            for (int kk = 0; kk < 4; kk++) v[kk] = p0 + 4 * qd + kk < Lmax ? (SC ? vr[tt * 4 + kk] * pv : vr[tt * 4 + kk]) : 0.0f;
            half4 vh, vl;
            split4(v[0], v[1], v[2], v[3], vh, vl);
            f32x4 a = o[tt] * alpha;
            a = __builtin_amdgcn_mfma_f32_16x16x16f16(vl, ph, a, 0, 0, 0);
            a = __builtin_amdgcn_mfma_f32_16x16x16f16(vh, pl, a, 0, 0, 0);
            o[tt] = __builtin_amdgcn_mfma_f32_16x16x16f16(vh, ph, a, 0, 0, 0);
        }
    }
    // merge the waves: weights exp(m_w - max_w m_w), in wave order
    if (qd == 0) {
        smax[wv][r16] = mrun;
        ssum[wv][r16] = lrun;
    }
#pragma unroll
    for (int tt = 0; tt < 8; tt++) *(f32x4 *)&so[wv][r16][16 * tt + 4 * qd] = o[tt];
    __syncthreads();
    const int qi = t >> 4, d0 = 8 * (t & 15), row = qi >> 1;
    if (row < nq) {
        const float mm = fmaxf(fmaxf(smax[0][qi], smax[1][qi]), fmaxf(smax[2][qi], smax[3][qi]));
        float wgt[4], l = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            wgt[w] = smax[w][qi] == -INFINITY ? 0.0f : expf(smax[w][qi] - mm);
            l = fmaf(wgt[w], ssum[w][qi], l);
        }
        const float inv = 1.0f / l;
        const int col = (2 * h + (qi & 1)) * HEAD_DIM + d0;
        float mx = 0.0f;
        f32x4 v[2];
        // (the sums of P V times 2^sv, merged, divided by l, scaled back)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int w = 0; w < 4; w++) acc += wgt[w] * *(const f32x4 *)&so[w][qi][d0 + 4 * j];
            acc = SC ? (acc * inv) * uv : acc * inv;
            v[j] = acc;
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(acc.x), fabsf(acc.y)), fmaxf(fabsf(acc.z), fabsf(acc.w))));
        }
        if (!split) {
            float *op = out + (size_t)(m0 + row) * ldo + col;
            *(f32x4 *)op = v[0];
            *(f32x4 *)(op + 4) = v[1];
            return;
        }
        // the row's two heads (256 columns, one K segment of the
        // o-projection) staged by their largest |output|: the row's 32 lanes
        // are one half-wave
        mx = fmaxf(mx, __shfl_xor(mx, 1));
        mx = fmaxf(mx, __shfl_xor(mx, 2));
        mx = fmaxf(mx, __shfl_xor(mx, 4));
        mx = fmaxf(mx, __shfl_xor(mx, 8));
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        const int sh = range_shift(mx);
        const float p2 = __builtin_ldexpf(1.0f, sh);
        half8 hi, lo;
        split8(v[0] * p2, v[1] * p2, hi, lo);
        uint8_t *sp = split + (size_t)(m0 + row) * (16 * HEAD_DIM * 4) + (col >> 5) * 128 + (col & 31) * 2;
        *(half8 *)sp = hi;
        *(half8 *)(sp + 64) = lo;
        if ((t & 31) == 0) rsc[(size_t)h * ldr + m0 + row] = __builtin_ldexpf(1.0f, -sh);
    }
}

// the matrix-core attention unless QTTS_PREFILL_ATTN_VALU=1
static bool prefill_attn_mx()
{
    // read at every launch (a few hundred ns), so a caller or test can switch
    // paths between calls
    const char *v = getenv("QTTS_PREFILL_ATTN_VALU");
    return !(v && *v && *v != '0');
}

// final-normed hidden of one row (talker.rs:477-481)
__global__ void __launch_bounds__(256)
k_final_rms(const float *x, const uint16_t *gamma, int H, float *out)
{
    __shared__ float red[4];
    const int t = threadIdx.x, lane = t & 63;
    float s = 0.0f;
    for (int k = t; k < H; k += 256) s = fmaf(x[k], x[k], s);
    s = wave_sum_dpp(s);
    if (lane == 0) red[t >> 6] = s;
    __syncthreads();
    const float inv = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)H + 1e-6f);
    for (int k = t; k < H; k += 256) out[k] = x[k] * inv * h2f(gamma[k]);
}

// Synthetic rows for timing: x[i] uniform in [-1, 1) from a hash of (seed, i).
__global__ void k_fill_rows(float *x, int64_t n, uint32_t seed)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        uint32_t h = (uint32_t)i * 0x9E3779B1u ^ seed * 0x85EBCA77u;
        h ^= h >> 15;
        h *= 0x2C1B3C6Du;
        h ^= h >> 12;
        x[i] = (float)(h >> 8) * (1.0f / 8388608.0f) - 1.0f;
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

#define PCHK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) return e_; } while (0)

static bool gemm_shape_ok(const Q4Tiled &w, int K)
{
    return K == w.k && K % GK == 0 && K >= 2 * GK;   // two chunks at least per k-slice
}

// Rows per tile, 16 * MB: one tile when M <= 80; else MB in 3..5 with the
// least padding (larger MB on ties: each weight tile is dequantised once per
// row tile).
static int pick_mb(int M)
{
    if (M <= 80) return (M + 15) / 16;
    int best = 5, pad = 1 << 30;
    for (int mb = 5; mb >= 3; mb--) {
        const int p = (M + 16 * mb - 1) / (16 * mb) * 16 * mb;
        if (p < pad) {
            pad = p;
            best = mb;
        }
    }
    return best;
}

// k-slices of a weight for the prefill projections whose consumer adds
// partials (q|k|v, o, down): about 96 workgroups per row tile.  A function
// of the weight alone, so a row's sums do not depend on the prompt length
// (prefix + suffix prefill stays bit-identical to one full prefill).
static int part_slices(const Q4Tiled &w)
{
    const int tn = (w.G * 32 + GN - 1) / GN, nch = w.k / GK;
    int S = std::max(1, (96 + tn / 2) / tn);
    S = std::min(S, 8);
    while (S > 1 && nch / S < 8) S--;
    return S;
}

bool gemm_x3()
{
    // read at every launch (a few hundred ns), so a caller or test can switch
    // paths between calls
    const char *v = getenv("QTTS_GEMM_F32");
    return !(v && *v && *v != '0');
}

template <int MB, int EPI>
static hipError_t launch_gemm_mb(const GemmA &a, const Q4Tiled &w, const GemmOut &o, int S, hipStream_t s)
{
    const int tm = (a.M + 16 * MB - 1) / (16 * MB), tn = (w.G * 32 + GN - 1) / GN;
    const dim3 grid(tm * tn * S);
    if (a.inv)
        hipLaunchKernelGGL((k_gemm_q4<MB, EPI, true>), grid, dim3(256), 0, s, a, w, o, tm, S);
    else
        hipLaunchKernelGGL((k_gemm_q4<MB, EPI, false>), grid, dim3(256), 0, s, a, w, o, tm, S);
    return hipGetLastError();
}

template <int EPI>
static hipError_t launch_gemm(const GemmA &a, const Q4Tiled &w, const GemmOut &o, int S, hipStream_t s)
{
    if (!gemm_shape_ok(w, w.k) || a.M < 1 || a.lda % 4 || S < 1 || S > w.k / (2 * GK)) return hipErrorInvalidValue;
    if (EPI == GEMM_SWIGLU && (!w.interleave || w.G % 4)) return hipErrorInvalidValue;
    if ((EPI == GEMM_BIAS || EPI == GEMM_BIAS_SILU) && !o.bias) return hipErrorInvalidValue;
    if (EPI != GEMM_PART && S != 1) return hipErrorInvalidValue;
    if (!a.inv != !a.gamma) return hipErrorInvalidValue;   // a fused norm has both
    switch (pick_mb(a.M)) {
    case 1: return launch_gemm_mb<1, EPI>(a, w, o, S, s);
    case 2: return launch_gemm_mb<2, EPI>(a, w, o, S, s);
    case 3: return launch_gemm_mb<3, EPI>(a, w, o, S, s);
    case 4: return launch_gemm_mb<4, EPI>(a, w, o, S, s);
    default: return launch_gemm_mb<5, EPI>(a, w, o, S, s);
    }
}

bool gemm_supported(const Q4Tiled &w)
{
    return gemm_shape_ok(w, w.k);
}

// Rows of any magnitude (gemm_q4 takes any finite input, gemv.rs:349-412).
// ws: the split path's workspace (enqueue_mm_rows).
hipError_t enqueue_gemm_rows(const Q4Tiled &w, const Q4Frag &f, const float *X, int rows, float *Y, int ldy, float *ws,
                             size_t ws_floats, hipStream_t s)
{
    if (gemm_x3() && f.data && ws_floats >= (size_t)f.kc * 64 + (f.kc + 3) / 4)
        return enqueue_mm_rows(f, X, w.k, rows, nullptr, false, Y, ldy, ws, ws_floats, s);
    return launch_gemm<GEMM_STORE>(GemmA{X, w.k, nullptr, nullptr, rows}, w,
                                   GemmOut{Y, ldy, std::min(ldy, w.G * 32), nullptr, 0}, 1, s);
}

// Y = X W + bias, optionally through SiLU (the text projection's fc1 / fc2,
// talker.rs:105-116, over a batch of rows).
hipError_t enqueue_gemm_bias(const Q4Tiled &w, const Q4Frag &f, const float *X, int rows, const float *bias, bool silu,
                             float *Y, int ldy, float *ws, size_t ws_floats, hipStream_t s)
{
    if (gemm_x3() && f.data && w.n % 32 == 0)
        return enqueue_mm_rows(f, X, w.k, rows, bias, silu, Y, ldy, ws, ws_floats, s);
    const GemmA a{X, w.k, nullptr, nullptr, rows};
    const GemmOut o{Y, ldy, std::min(ldy, w.n), bias, 0};
    return silu ? launch_gemm<GEMM_BIAS_SILU>(a, w, o, 1, s) : launch_gemm<GEMM_BIAS>(a, w, o, 1, s);
}

bool prefill_supported(const TalkerDev &m)
{
    if (m.n_heads != 16 || m.n_kv_heads != 8 || m.hidden % GK) return false;
    for (int l = 0; l < m.n_layers; l++) {
        const LayerDev &L = m.layers[l];
        if (!gemm_shape_ok(L.qkv, m.hidden) || !gemm_shape_ok(L.o, 16 * HEAD_DIM) ||
            !gemm_shape_ok(L.gate_up, m.hidden) || !gemm_shape_ok(L.down, m.inter) || !L.gate_up.interleave ||
            L.gate_up.G % 4 || L.qkv.G * 32 < 32 * HEAD_DIM || L.gate_up.G * 16 < m.inter ||
            L.o.G * 32 < m.hidden || L.down.G * 32 < m.hidden)
            return false;
    }
    return true;
}

// Column slots of the factors of a split GEMM input (PrefillWs.rsc): 8 for
// the o-projection's (one per kv head), one per 64 columns for the down
// projection's.
int64_t prefill_rsc_slots(const TalkerDev &m) { return std::max<int64_t>(8, (m.inter + 63) / 64); }

// The staging power of two of rows normed with this gamma (f16 bit
// patterns, on the host): |x * inv * gamma| <= sqrt(n) * max|gamma|, since
// |x_k| * inv <= sqrt(n); the shift takes that bound into [2^13, 2^14].
// Largest finite |value| of n f16 bit patterns (inf / NaN skipped: they
// give no finite bound and propagate as in f32).
double f16_max_abs(const uint16_t *h, int n)
{
    double g = 0.0;
    for (int k = 0; k < n; k++) {
        const uint16_t a = h[k] & 0x7FFFu;
        if (a >= 0x7C00u) continue;
        const int e = a >> 10, f = a & 0x3FF;
        g = std::max(g, e ? std::ldexp(1024.0 + f, e - 25) : std::ldexp((double)f, -24));
    }
    return g;
}

// The power of two that takes a bound on |values| into [2^13, 2^14].
int bound_shift(double bound)
{
    if (!(bound > 0.0) || !std::isfinite(bound)) return 0;
    return std::max(-100, std::min(100, 14 - (int)std::ceil(std::log2(bound))));
}

// The attention's staging shifts: none while the bound lies in [2^-4, 2^14]
// (the values' f16 halves then neither overflow nor lose precision against
// the bound), else the shift that takes it into [2^13, 2^14].
int attn_shift(double bound)
{
    if (bound >= 0x1p-4 && bound <= 0x1p14) return 0;
    return bound_shift(bound);
}

int norm_shift(const uint16_t *gamma_host, int n)
{
    return bound_shift(std::sqrt((double)n) * f16_max_abs(gamma_host, n));
}

static bool layer_has_frags(const LayerDev &L)
{
    return L.qkv_f.data && L.o_f.data && L.gate_up_f.data && L.down_f.data;
}

// Whether a layer takes the split GEMM: all four matrices, since each hands
// its successor rows in the form that one reads.  A layer with a matrix
// outside the split's range (a scale of 4096 or more) runs on the f32
// instructions, the others as before.
static bool split_layer(const TalkerDev &m, int l)
{
    return gemm_x3() && layer_has_frags(m.layers[l]);
}

int prefill_split_layers(const TalkerDev &m)
{
    int n = 0;
    for (int l = 0; l < m.n_layers; l++) n += split_layer(m, l);
    return n;
}

// Floats of partial sums the prompt's projections need at up to `rows` rows.
int64_t prefill_part_floats(const TalkerDev &m, int rows)
{
    int64_t f = 0;
    for (int l = 0; l < m.n_layers; l++) {
        const LayerDev &L = m.layers[l];
        for (const Q4Tiled *w : {&L.qkv, &L.o, &L.down}) f = std::max<int64_t>(f, (int64_t)rows * part_slices(*w) * w->G * 32);
        if (!layer_has_frags(L)) continue;
        // a small batch may cut K finer than a large one
        for (int r : {rows, std::min(64, rows), std::min(16, rows)}) {
            f = std::max<int64_t>(f, (int64_t)mm_part_floats(L.qkv_f, r));
            f = std::max<int64_t>(f, (int64_t)mm_part_floats(L.o_f, r));
            f = std::max<int64_t>(f, (int64_t)mm_part_floats(L.down_f, r));
            f = std::max<int64_t>(f, (int64_t)mm_swiglu_part_floats(L.gate_up_f, r));
        }
    }
    return f;
}

hipError_t enqueue_fill_rows(float *x, int64_t n, uint32_t seed, hipStream_t s)
{
    hipLaunchKernelGGL(k_fill_rows, dim3(1024), dim3(256), 0, s, x, n, seed);
    return hipGetLastError();
}

template <int NP>
struct ResidNorm {
    static hipError_t go(float *x, int H, int M, const MmParts &p, float *inv, const uint16_t *gamma, int nshift,
                         uint8_t *split, hipStream_t s)
    {
        hipLaunchKernelGGL(k_resid_norm<NP>, dim3(M), dim3(256), 0, s, x, H, p, inv, gamma, nshift, split, (H + 63) / 64);
        return hipGetLastError();
    }
};

template <int NP>
struct QkvPost {
    static hipError_t go(const TalkerDev &m, const LayerDev &L, const PrefillWs &pw, const MmParts &p, int M, int64_t start,
                         int l, hipStream_t s)
    {
        hipLaunchKernelGGL(k_prefill_qkv_post<NP>, dim3(M, 8), dim3(256), 0, s, p, M, start, L.q_norm, L.k_norm, m.rope_cos,
                           m.rope_sin, m.kv, l, pw.q, 16 * HEAD_DIM);
        return hipGetLastError();
    }
};

// The prefill's gate|up GEMM of layer l alone (pw.xs rows; on the f32 path
// pw.x rows and pw.inv).
hipError_t enqueue_gemm_gateup(const TalkerDev &m, const PrefillWs &pw, int l, int M, hipStream_t s)
{
    const LayerDev &L = m.layers[l];
    if (split_layer(m, l)) {
        const int kc = (m.hidden + 63) / 64;
        return enqueue_mm_swiglu(RowsSplit{(const uint8_t *)pw.xs, kc, M, nullptr, 0, __builtin_ldexpf(1.0f, -L.post_shift)},
                                 L.gate_up_f, pw.part, (uint8_t *)pw.h, (m.inter + 63) / 64, pw.rsc, s);
    }
    return launch_gemm<GEMM_SWIGLU>(GemmA{pw.x, m.hidden, pw.inv, L.post_norm, M}, L.gate_up,
                                    GemmOut{pw.h, m.inter, m.inter, nullptr, 0}, 1, s);
}

// What enqueue_gemm_gateup reads, from pw.x: the rows normed and split (for
// layer l's staging), or their 1/rms.
hipError_t enqueue_gateup_input(const TalkerDev &m, const PrefillWs &pw, int l, int M, hipStream_t s)
{
    const bool sp = split_layer(m, l);
    return ResidNorm<1>::go(pw.x, m.hidden, M, MmParts{}, pw.inv, sp ? m.layers[l].post_norm : nullptr,
                            m.layers[l].post_shift, sp ? (uint8_t *)pw.xs : nullptr, s);
}

// A projection of the f32 path into k-slice partials: slice s of row m at
// part[s * M * ld + m * ld], ld = the weight's padded width.
static hipError_t gemm_parts(const GemmA &a, const Q4Tiled &w, const PrefillWs &pw, MmParts *p, hipStream_t s)
{
    const int S = part_slices(w), ld = w.G * 32;
    *p = MmParts{pw.part, ld, (size_t)a.M * ld, S, 1};
    return launch_gemm<GEMM_PART>(a, w, GemmOut{pw.part, ld, ld, nullptr, p->stride}, S, s);
}

// Rows pw.x[0..M) at positions start..start+M-1 through every layer; the
// last row's final-normed hidden goes to hidden_out.  Positions
// start..start+M-1 must be backed by the page table.
hipError_t enqueue_talker_prefill(const TalkerDev &m, const PrefillWs &pw, int M, int64_t start, float *hidden_out,
                                  hipStream_t s)
{
    if (M < 1 || M > pw.cap_rows || m.hidden > 2048) return hipErrorInvalidValue;
    const int H = m.hidden, A = 16 * HEAD_DIM, kh = (H + 63) / 64, ki = (m.inter + 63) / 64;
    uint8_t *const xs = (uint8_t *)pw.xs;
    MmParts p{};
    // x += parts, then the rows the next GEMM takes: normed and split, or
    // their 1/rms for the f32 instructions
    const auto resid = [&](bool split, const uint16_t *gamma, int shift) {
        return by_parts<ResidNorm>(p.n, pw.x, H, M, p, pw.inv, split ? gamma : nullptr, shift, split ? xs : nullptr, s);
    };
    PCHK(resid(split_layer(m, 0), m.layers[0].input_norm, m.layers[0].in_shift));
    for (int l = 0; l < m.n_layers; l++) {
        const LayerDev &L = m.layers[l];
        const bool sp = split_layer(m, l);
        // q|k|v, QK-norm + RoPE + KV append, attention
        if (sp)
            PCHK(enqueue_mm_parts(RowsSplit{xs, kh, M, nullptr, 0, __builtin_ldexpf(1.0f, -L.in_shift)}, L.qkv_f, false,
                                  pw.part, &p, s));
        else
            PCHK(gemm_parts(GemmA{pw.x, H, pw.inv, L.input_norm, M}, L.qkv, pw, &p, s));
        PCHK(by_parts<QkvPost>(p.n, m, L, pw, p, M, start, l, s));
        uint8_t *as = sp ? (uint8_t *)pw.attn : nullptr;
        if (prefill_attn_mx()) {
            if (L.q_shift || L.k_shift || L.v_shift)
                hipLaunchKernelGGL(k_prefill_attn_mx<true>, dim3((M + 7) / 8, 8), dim3(256), 0, s, pw.q, A, M, start,
                                   m.kv, l, pw.attn, A, as, pw.rsc, M, L.q_shift, L.k_shift, L.v_shift);
            else
                hipLaunchKernelGGL(k_prefill_attn_mx<false>, dim3((M + 7) / 8, 8), dim3(256), 0, s, pw.q, A, M, start,
                                   m.kv, l, pw.attn, A, as, pw.rsc, M, 0, 0, 0);
            PCHK(hipGetLastError());
        } else {
            // f32 rows in pw.part (at least M rows of the q|k|v's sums, which
            // have been read), split from there
            float *out = sp ? pw.part : pw.attn;
            hipLaunchKernelGGL(k_prefill_attn<PREFILL_ATTN_QB>, dim3((M + PREFILL_ATTN_QB - 1) / PREFILL_ATTN_QB, 8),
                               dim3(256), 0, s, pw.q, A, M, start, m.kv, l, out, A);
            PCHK(hipGetLastError());
            if (sp) PCHK(enqueue_split_rows(out, A, M, A, as, A / 64, pw.rsc, M, s));
        }
        // o-proj, residual, post-attention norm
        if (sp)
            PCHK(enqueue_mm_parts(RowsSplit{as, A / 64, M, pw.rsc, M, 1.0f}, L.o_f, false, pw.part, &p, s));
        else
            PCHK(gemm_parts(GemmA{pw.attn, A, nullptr, nullptr, M}, L.o, pw, &p, s));
        PCHK(resid(sp, L.post_norm, L.post_shift));
        // gate|up with SwiGLU, down, residual, next layer's input norm
        PCHK(enqueue_gemm_gateup(m, pw, l, M, s));
        if (sp)
            PCHK(enqueue_mm_parts(RowsSplit{(const uint8_t *)pw.h, ki, M, pw.rsc, M, 1.0f}, L.down_f, true, pw.part, &p, s));
        else
            PCHK(gemm_parts(GemmA{pw.h, m.inter, nullptr, nullptr, M}, L.down, pw, &p, s));
        if (l + 1 < m.n_layers)
            PCHK(resid(split_layer(m, l + 1), m.layers[l + 1].input_norm, m.layers[l + 1].in_shift));
        else
            PCHK(resid(false, nullptr, 0));
    }
    hipLaunchKernelGGL(k_final_rms, dim3(1), dim3(256), 0, s, pw.x + (size_t)(M - 1) * H, m.final_norm, H,
                       hidden_out);
    return hipGetLastError();
}

}  // namespace qtts
