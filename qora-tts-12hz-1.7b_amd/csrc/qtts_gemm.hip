// qtts_gemm.hip — the f32-accurate Q4 GEMM on the f16 matrix cores
// (gemm_q4, gemv.rs:349-412), shared by the talker prefill
// (qtts_prefill.hip), the text projection and qtts_gemm_q4.
//
// The contraction: every operand is split into f16 hi + lo (22 of an f32's
// 24 bits; a dequantised weight, a 4-bit integer times an f16 scale, exactly)
// and v_mfma_f32_16x16x32_f16 accumulates lo hi + hi lo + hi hi in f32.
//
// What bounds it: three matrix instructions per useful one, so 3 x 2MNK
// operations at the f16 rate; a kernel that converts both operands while it
// stages them through LDS keeps those pipes busy a fifth of the time.  Here
// neither operand is converted on the way into LDS:
//  - the rows arrive already split (RowsSplit), written once by the kernel
//    that produces them and read by every column tile;
//  - the weight is kept a second time in fragment order (Q4Frag): a lane's
//    nibbles of one 16x16x32 operand are one dword, so a wave dequantises
//    its own columns in registers, 2.4 VALU operations a weight, with no LDS
//    and no barrier between.
//
// Sums: one f32 accumulation per K segment (256 of the contraction, 64 where
// the rows' staging factors change every 64), folded into the running sum
// with the segment's factor.  Short chains keep the rounding below one long
// f32 chain's.  The association is a property of the weight alone (segments
// in order within a slice, slices in order), whatever the rows and however
// the work is cut over workgroups, so a row has the same bits in any batch.
#include "qtts_device.h"
#include "qtts_kernels.h"
#include "qtts_devutil.h"
#include "qtts_mfma.h"

#include <algorithm>
#include <cstdlib>

namespace qtts {

constexpr int MM_MAX_MB = 5;   // row blocks of 16 per tile, at most

// ---------------------------------------------------------------------------
// Fragment order.  Record (group, 64-row chunk): 1024 B of nibbles, lane l's
// four dwords = (block 0, rows 0-31), (block 0, rows 32-63), (block 1, ...),
// then 64 f16 scales (dual: 64 per block).  Block b of a group is its columns
// 16b..16b+15; a dual weight (gate|up) pairs gate columns 16v..+15 (block 0)
// with up columns 16v..+15 (block 1) in virtual group v.  Lane l of a block
// holds column l % 16 at rows 8(l/16)..+7: the nibble of row 2p in bits 4p,
// of row 2p + 1 in bits 16 + 4p, so (w >> 4p) & 0x000F000F is the pair as
// the low bits of two halves.  The scales carry 2^bshift (exact).  Rows past
// k hold scale 0.
// ---------------------------------------------------------------------------

__device__ __forceinline__ void frag_source(const Q4Tiled &w, TileShape ts, int k, int g, const uint8_t *&word,
                                            const uint16_t *&scale)
{
    const int P = ts.T / ts.GB;
    const int s = k / w.KC, rr = k - s * w.KC, r = rr / P, pt = rr - r * P;
    const int ct = g / ts.GB, gt = g - ct * ts.GB;
    const bool wave_groups = (ts.T / 64) % ts.GB == 0;
    const int t = wave_groups ? ((pt >> 6) * ts.GB + gt) * 64 + (pt & 63) : pt * ts.GB + gt;
    const uint8_t *tile = w.data + (size_t)(s * w.CT + ct) * w.tile_bytes;
    word = tile + ((size_t)r * ts.T + t) * 16;
    scale = (const uint16_t *)(tile + (size_t)ts.R * ts.T * 16) + t * ts.R + r;
}

// One wave per record.  Column c of a group: byte c/2, low nibble even c.
__global__ void __launch_bounds__(256)
k_frag_build(Q4Tiled w, Q4Frag f, uint8_t *out)
{
    const int lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
    const int64_t rec = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (rec >= (int64_t)f.ng * f.kc) return;
    const int v = (int)(rec / f.kc), c = (int)(rec - (int64_t)v * f.kc);
    const TileShape ts = tile_shape(w.cfg);
    uint8_t *o = out + rec * f.rec;
    uint32_t nib[4];
    for (int b = 0; b < 2; b++) {
        // dual: groups alternate gate, up; block b of virtual group v is
        // half v % 2 of group 2 (v / 2) + b
        const int g = f.dual ? 2 * (v >> 1) + b : v;
        const int col = f.dual ? 16 * (v & 1) + r16 : 16 * b + r16;
        for (int h = 0; h < 2; h++) {
            uint32_t d = 0;
            for (int e = 0; e < 8; e++) {
                const int k = 64 * c + 32 * h + 8 * q + e;
                uint32_t n = 8;
                if (k < w.k) {
                    const uint8_t *word;
                    const uint16_t *sc;
                    frag_source(w, ts, k, g, word, sc);
                    n = (word[col >> 1] >> (4 * (col & 1))) & 15u;
                }
                d |= n << (4 * (e >> 1) + 16 * (e & 1));
            }
            nib[2 * b + h] = d;
        }
    }
    *(uint4 *)(o + 16 * lane) = uint4{nib[0], nib[1], nib[2], nib[3]};
    const float p2 = __builtin_ldexpf(1.0f, f.bshift);
    for (int b = 0; b < (f.dual ? 2 : 1); b++) {
        const int g = f.dual ? 2 * (v >> 1) + b : v, k = 64 * c + lane;
        _Float16 s = (_Float16)0.0f;
        if (k < w.k) {
            const uint8_t *word;
            const uint16_t *sc;
            frag_source(w, ts, k, g, word, sc);
            s = (_Float16)(h2f(*sc) * p2);
        }
        *(_Float16 *)(o + 1024 + 128 * b + 2 * lane) = s;
    }
}

// ---------------------------------------------------------------------------
// Split rows: row m is kc records of 256 B, one per 64 columns: 32 hi halves,
// 32 lo halves, then the same for the next 32 columns.
// ---------------------------------------------------------------------------

// Rows of f32 into split rows, each 256 columns (a K segment) staged times the
// power of two from their largest |x|: small values keep their bits beside an
// outlier elsewhere in the row.  The factors that undo it go to rsc[s * ldr +
// m].  One workgroup per row.
__global__ void __launch_bounds__(256)
k_split_rows(const float *X, int ld, int K, uint8_t *out, int kc, float *rsc, int ldr)
{
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, m = blockIdx.x;
    const float *x = X + (size_t)m * ld;
    uint8_t *o = out + (size_t)m * kc * 256;
    // four columns a lane, so a wave covers 256 (a caller's rows need not be
    // 16-byte aligned)
    typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
    for (int k0 = 256 * wv; k0 < 64 * kc; k0 += 1024) {
        const int k = k0 + 4 * lane;
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        if (k < K) v = *(const f32x4u *)(x + k);
        const float mx = wave_max_dpp(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        const int sh = range_shift(mx);
        const float p2 = __builtin_ldexpf(1.0f, sh);
        if (k < 64 * kc) {
            uint32_t h0, l0, h1, l1;
            split_f16_pair<true>(v.x * p2, v.y * p2, h0, l0);
            split_f16_pair<true>(v.z * p2, v.w * p2, h1, l1);
            uint8_t *p = o + (k >> 5) * 128 + (k & 31) * 2;
            *(uint2 *)p = uint2{h0, h1};
            *(uint2 *)(p + 64) = uint2{l0, l1};
        }
        if (lane == 0) rsc[(size_t)(k0 >> 8) * ldr + m] = __builtin_ldexpf(1.0f, -sh);
    }
}

// ---------------------------------------------------------------------------
// The GEMM.  Workgroup: 16 MB rows x 128 columns (four groups, one per wave:
// a wave tile of 16 MB x 32), one run of K chunks of 64.  The weight is the
// matrix instruction's A operand and the rows its B operand, so a lane ends
// with four consecutive columns of one row (16-byte stores, one factor).
//
// Rows through double-buffered LDS in fragment order: 256 B per (16 rows,
// part), part = (half of the chunk, hi / lo, q), a row's 16 bytes at slot
// row ^ part: writes (16 lanes of one row, 16 parts) and reads (16 rows of
// one part) both spread over all banks.  Two register sets hold the next two
// chunks' rows and weights.
//
// Measured (a talker layer of a 400-row prompt, against a kernel that
// converted both operands while staging them): gate|up 103 -> 57 us (1.06
// PFLOP/s of f16 products, 87% of what a large matrix product reaches),
// q|k|v 37 -> 26, o 22 -> 21, down 49 -> 47.  The last three make 640 tiles:
// 2.5 rounds over the 256 CUs that run as 3.  More waves a SIMD (row blocks
// of 4: 59 -> 70 us) and an interleave of the instruction groups asked of
// the scheduler (it spills) were slower.
// ---------------------------------------------------------------------------

enum { MM_STORE = 0, MM_PART = 1, MM_PART_DUAL = 2, MM_SWIGLU = 3 };

struct MmOut {
    float *Y;                // STORE: [M][ldy]; PART: [run][M][ldy]
    int ldy;
    int vec;                 // STORE: 16-byte stores fit
    uint8_t *rows;           // SWIGLU: split rows of the next GEMM
    int okc;
    float *rsc;              // SWIGLU: [64-column slot][M]
};

// two weights of a packed nibble pair word: hi and lo halves of (nib - 8) s
__device__ __forceinline__ void dequant_pair(uint32_t w, h16x2 s, h16x2 &hi, h16x2 &lo)
{
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(w), "v"(0x000F000Fu), "s"(0x64006400u));
    const h16x2 n8 = __builtin_bit_cast(h16x2, r) + h16x2{(_Float16)-1032.0f, (_Float16)-1032.0f};
    hi = n8 * s;
    lo = __builtin_elementwise_fma(n8, s, -hi);
}

__device__ __forceinline__ void dequant8(uint32_t w, half8 s, half8 &hi, half8 &lo)
{
    h16x2 h[4], l[4];
#pragma unroll
    for (int p = 0; p < 4; p++) dequant_pair(w >> (4 * p), h16x2{s[2 * p], s[2 * p + 1]}, h[p], l[p]);
    hi = half8{h[0].x, h[0].y, h[1].x, h[1].y, h[2].x, h[2].y, h[3].x, h[3].y};
    lo = half8{l[0].x, l[0].y, l[1].x, l[1].y, l[2].x, l[2].y, l[3].x, l[3].y};
}

template <int MB, int FP, int EPI>
__global__ void __launch_bounds__(256, 2)
k_q4_gemm(RowsSplit a, Q4Frag w, MmOut o, int tm, int nrun, int run_chunks)
{
    constexpr bool DUAL = EPI == MM_SWIGLU || EPI == MM_PART_DUAL, PART = EPI == MM_PART || EPI == MM_PART_DUAL;
    constexpr int BUF = MB * 4096;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * BUF];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, r16 = lane & 15, q = lane >> 4;
    // workgroups are dealt round-robin to the 8 XCDs: each gets a contiguous
    // run of tiles, row tiles fastest, so those that share a weight tile
    // share that XCD's L2
    const int nwg = gridDim.x, id = blockIdx.x, xcd = id & 7, qq = nwg >> 3, rem = nwg & 7;
    const int logical = xcd * qq + min(xcd, rem) + (id >> 3);
    const int mt = logical % tm, rest = logical / tm, run = rest % nrun, nt = rest / nrun;
    const int m0 = mt * 16 * MB;
    const int c0 = run * run_chunks, n = min(run_chunks, w.kc - c0);
    const int grp = __builtin_amdgcn_readfirstlane(4 * nt + wv);

    // rows: thread t moves part t % 16 of row t / 16 of each 16-row block
    const uint32_t rstride = (uint32_t)a.kc * 256;
    const uint8_t *ap = a.p + (size_t)c0 * 256;
    uint32_t ao[MB];                 // the launcher bounds the rows' bytes by 2^31
#pragma unroll
    for (int i = 0; i < MB; i++) ao[i] = (uint32_t)min(m0 + 16 * i + (t >> 4), a.M - 1) * rstride + (t & 15) * 16;
    const int aw = (t & 15) * 256 + (((t >> 4) ^ (t & 15)) * 16);
    const uint8_t *wp = w.data + ((size_t)min(grp, w.ng - 1) * w.kc + c0) * w.rec;

    // register sets of rows and of weights: a tall tile's chunk covers the
    // loads by itself; short tiles run one segment, all of it in flight at once
    constexpr int AS = MB <= 2 ? 4 : FP == 1 && MB >= 5 ? 1 : 2, WS = MB <= 2 ? 4 : 2;
    u32x4 ra[AS][MB];
    u32x4 rn[WS];
    half8 rs[WS][DUAL ? 4 : 2];       // [set][half of the chunk (+ 2 block)]
    const auto fetch_a = [&](int s, int c) {
#pragma unroll
        for (int i = 0; i < MB; i++) ra[s][i] = *(const u32x4 *)(ap + (size_t)c * 256 + ao[i]);
    };
    const auto fetch_w = [&](int s, int c) {
        const uint8_t *p = wp + (size_t)c * w.rec;
        rn[s] = *(const u32x4 *)(p + 16 * lane);
        rs[s][0] = *(const half8 *)(p + 1024 + 16 * q);
        rs[s][1] = *(const half8 *)(p + 1088 + 16 * q);
        if constexpr (DUAL) {
            rs[s][2] = *(const half8 *)(p + 1152 + 16 * q);
            rs[s][3] = *(const half8 *)(p + 1216 + 16 * q);
        }
    };
    const auto stage = [&](int s, int buf) {
#pragma unroll
        for (int i = 0; i < MB; i++) *(u32x4 *)(lds + buf * BUF + i * 4096 + aw) = ra[s][i];
    };
    const float ubs = __builtin_ldexpf(1.0f, -w.bshift);
    f32x4 cur[MB][2], tot[MB][2], seg[FP == 1 ? MB : 1][2];   // seg, FP 1: the segment's 64-column sums
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) tot[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // [half][block]; half 0 is dequantised a chunk ahead (tall tiles: its
    // arithmetic then fills the last products' issue slots, not the wait for
    // the rows after the barrier: 128 / 400 / 1024 rows x 2048 x 12288 40.4 ->
    // 34.9, 59.1 -> 56.7, 151 -> 144 us)
    constexpr bool AHEAD = MB > 2;
    half8 wh[2][2], wl[2][2];
    const auto dequant = [&](int s, int h) {
#pragma unroll
        for (int j = 0; j < 2; j++) dequant8(rn[s][2 * j + h], rs[s][DUAL ? 2 * j + h : h], wh[h][j], wl[h][j]);
    };
    const auto mma = [&](int h, const half8 (&xh)[MB], const half8 (&xl)[MB], bool first) {
        const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                cur[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[h][j], xh[i], first ? z : cur[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                cur[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[h][j], xl[i], cur[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                cur[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[h][j], xh[i], cur[i][j], 0, 0, 0);
    };
    const auto read_x = [&](int buf, int h, half8 (&xh)[MB], half8 (&xl)[MB]) {
        const int ph = 8 * h + q, pl = ph + 4;
#pragma unroll
        for (int i = 0; i < MB; i++) {
            xh[i] = *(const half8 *)(lds + buf * BUF + i * 4096 + ph * 256 + ((r16 ^ ph) * 16));
            xl[i] = *(const half8 *)(lds + buf * BUF + i * 4096 + pl * 256 + ((r16 ^ pl) * 16));
        }
    };
    // chunk in buf with weights of set s; sn: the next chunk's set
    const auto compute = [&](int s, int sn, int buf, bool first) {
        half8 xh[2][MB], xl[2][MB];
        read_x(buf, 0, xh[0], xl[0]);
        if (!AHEAD) dequant(s, 0);
        dequant(s, 1);
        mma(0, xh[0], xl[0], first);
        read_x(buf, 1, xh[1], xl[1]);
        mma(1, xh[1], xl[1], false);
        if (AHEAD) dequant(sn, 0);
    };
    // sums times the power of two that undoes the staging (exact), into the
    // running ones
    const auto fold = [&](const float (&f)[MB]) {
#pragma unroll
        for (int i = 0; i < MB; i++) {
            const float u = f[i] * ubs;
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) tot[i][j][e] = fmaf(cur[i][j][e], u, tot[i][j][e]);
        }
    };
    const auto fold_seg = [&](const float (&f)[MB], bool first) {
#pragma unroll
        for (int i = 0; i < (FP == 1 ? MB : 0); i++) {
            const float u = f[i] * ubs;
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) seg[i][j][e] = first ? cur[i][j][e] * u : fmaf(cur[i][j][e], u, seg[i][j][e]);
        }
    };

#pragma unroll
    for (int u = 0; u < WS; u++) {
        if (u < AS) fetch_a(u, min(u, n - 1));
        fetch_w(u, min(u, n - 1));
    }
    stage(0, 0);
    if (AHEAD) dequant(0, 0);
    __syncthreads();
    for (int c = 0; c < n; c += 4) {
        float f4[MB];
        if constexpr (FP == 4) {
#pragma unroll
            for (int i = 0; i < MB; i++)
                f4[i] = a.rsc ? a.rsc[(size_t)((c0 + c) >> 2) * a.rseg + min(m0 + 16 * i + r16, a.M - 1)] : a.ufac;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (c + u < n) {
                const int s = u % WS, buf = u & 1;
                if (MB > 2 || c + u + AS < n) fetch_a(u % AS, min(c + u + AS, n - 1));
                float f1[MB];            // the chunk's factors, in flight behind its matrix work
                if constexpr (FP == 1) {
#pragma unroll
                    for (int i = 0; i < MB; i++)
                        f1[i] = a.rsc[(size_t)(c0 + c + u) * a.rseg + min(m0 + 16 * i + r16, a.M - 1)];
                }
                compute(s, (u + 1) % WS, buf, FP == 1 || u == 0);
                if constexpr (FP == 1) fold_seg(f1, u == 0);
                if (MB > 2 || c + u + WS < n) fetch_w(s, min(c + u + WS, n - 1));
                stage((u + 1) % AS, buf ^ 1);
                __syncthreads();
            }
        }
        if constexpr (FP == 4) {
            fold(f4);
        } else {
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) tot[i][j] += seg[i][j];
        }
    }

    if constexpr (EPI == MM_SWIGLU) {
        // silu(gate) up of this lane's row: outputs 64 nt + 16 wave + 4q..+3;
        // staged for the next GEMM by the row's largest |value| over the
        // tile's 64 outputs
        float(*wmx)[16 * MB] = (float(*)[16 * MB])lds;   // the loop ended with a barrier
        f32x4 v[MB];
#pragma unroll
        for (int i = 0; i < MB; i++) {
            float mx = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[i][e] = silu_f(tot[i][0][e]) * tot[i][1][e];
                mx = fmaxf(mx, fabsf(v[i][e]));
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            if (q == 0) wmx[wv][16 * i + r16] = mx;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MB; i++) {
            const int m = m0 + 16 * i + r16, s = 16 * i + r16;
            const int sh = range_shift(fmaxf(fmaxf(wmx[0][s], wmx[1][s]), fmaxf(wmx[2][s], wmx[3][s])));
            const float p2 = __builtin_ldexpf(1.0f, sh);
            uint32_t h0, l0, h1, l1;
            split_f16_pair<true>(v[i].x * p2, v[i].y * p2, h0, l0);
            split_f16_pair<true>(v[i].z * p2, v[i].w * p2, h1, l1);
            if (m < a.M) {
                uint8_t *p = o.rows + ((size_t)m * o.okc + nt) * 256 + (wv >> 1) * 128 + (wv & 1) * 32 + 8 * q;
                *(uint2 *)p = uint2{h0, h1};
                *(uint2 *)(p + 64) = uint2{l0, l1};
                if (wv == 0 && q == 0) o.rsc[(size_t)nt * a.M + m] = __builtin_ldexpf(1.0f, -sh);
            }
        }
        return;
    }
    if (grp >= w.ng) return;
    float *Y = o.Y + (PART ? (size_t)run * a.M * o.ldy : 0);
#pragma unroll
    for (int i = 0; i < MB; i++) {
        const int m = m0 + 16 * i + r16;
        if (m >= a.M) continue;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            float *y = Y + (size_t)m * o.ldy + 32 * grp + 16 * j + 4 * q;
            if (PART || o.vec) {
                *(f32x4 *)y = tot[i][j];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) y[e] = tot[i][j][e];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Consumers of partial sums (MmParts, sum_parts in qtts_mfma.h)
// ---------------------------------------------------------------------------

// Y[m][col] = (silu)(sum of parts (+ bias)); one thread per 4 columns
template <int NP>
__global__ void __launch_bounds__(256)
k_fold_store(MmParts p, int M, int ncols, const float *bias, int silu, float *Y, int ldy)
{
    const int m = blockIdx.y, c = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (c >= ncols) return;
    f32x4 v = sum_parts4<NP>(p, (size_t)m * p.ld + c);
    float *y = Y + (size_t)m * ldy + c;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float x = v[e];
        if (bias) x += bias[c + e];
        if (silu) x = silu_f(x);
        y[e] = x;
    }
}

// silu(gate) up of a dual weight's parts into split rows, one wave per (row,
// 64 outputs): output j of virtual group j / 16 has its gate at column
// 32 (j / 16) + j % 16 and its up 16 further.
template <int NP>
__global__ void __launch_bounds__(256)
k_fold_swiglu(MmParts p, int M, int slots, uint8_t *rows, int okc, float *rsc)
{
    const int lane = threadIdx.x & 63, nt = blockIdx.x * 4 + (threadIdx.x >> 6), m = blockIdx.y;
    if (nt >= slots) return;
    const int j = 64 * nt + lane;
    const size_t at = (size_t)m * p.ld + 32 * (j >> 4) + (j & 15);
    const float g = sum_parts<NP>(p, at), u = sum_parts<NP>(p, at + 16);
    const float v = silu_f(g) * u;
    const int sh = range_shift(wave_max_dpp(fabsf(v)));
    const float x = v * __builtin_ldexpf(1.0f, sh);
    uint32_t h, l;
    split_f16_pair<true>(x, 0.0f, h, l);
    uint16_t *r = (uint16_t *)(rows + ((size_t)m * okc + nt) * 256 + (lane >> 5) * 128 + (lane & 31) * 2);
    r[0] = (uint16_t)h;
    r[32] = (uint16_t)l;
    if (lane == 0) rsc[(size_t)nt * M + m] = __builtin_ldexpf(1.0f, -sh);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

#define GCHK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) return e_; } while (0)

bool frag_supported(const Q4Tiled &w)
{
    return w.k % 32 == 0 && w.k >= 64 && w.bshift >= 0 && w.n >= 32 && (!w.interleave || (w.n / 32) % 4 == 0);
}

// Shape of w's fragment order and the bytes it takes.
size_t frag_shape(const Q4Tiled &w, Q4Frag *f)
{
    *f = Q4Frag{nullptr, w.k, (w.k + 63) / 64, w.n / 32, w.interleave, w.interleave ? 1280 : 1152, w.bshift};
    return (size_t)f->ng * f->kc * f->rec;
}

hipError_t enqueue_frag_build(const Q4Tiled &w, const Q4Frag &f, uint8_t *out, hipStream_t s)
{
    const int64_t recs = (int64_t)f.ng * f.kc;
    hipLaunchKernelGGL(k_frag_build, dim3((unsigned)((recs + 3) / 4)), dim3(256), 0, s, w, f, out);
    return hipGetLastError();
}

// k-slices of a weight whose consumer adds partial sums: a divisor of its
// segments, at most 144 column tiles x slices per row tile (128 for the
// talker's q|k|v, o and down).  A property of the weight alone (a row's bits
// do not depend on the batch), so one count serves every row count: 128 is
// half the CUs per row tile, which fills them from two row tiles on; 96 would
// lie better at 400 rows (480 tiles, not 640) and worse at 1100 (6 rounds of
// 4 segments against 7 of 3).
int mm_slices(const Q4Frag &w)
{
    const int tn = (w.ng + 3) / 4, nseg = (w.kc + 3) / 4;
    int best = 1;
    for (int S = 1; S <= 8; S++)
        if (nseg % S == 0 && S * tn <= 144) best = S;
    return best;
}

static int mm_segments(const Q4Frag &w) { return (w.kc + 3) / 4; }

// Row blocks per tile: the row tiles x columns x runs fill the 256 CUs in
// whole rounds; a tile's time is its matrix work (MB) plus what does not
// depend on the rows (the weight's dequantisation, ~1.5 row blocks, fitted to
// gate|up of 128, 400 and 1024 rows: 34.9, 56.7 and 144 us).  Six row blocks
// spill with half a chunk's weights dequantised ahead.
static int mm_mb(int M, int per_tile, int max_mb)
{
    int best = 1;
    double cost = 1e30;
    for (int mb = 1; mb <= max_mb; mb++) {
        const int tm = (M + 16 * mb - 1) / (16 * mb);
        const double c = (double)((tm * per_tile + 255) / 256) * (mb + 1.5);
        if (c < cost - 1e-9) {
            cost = c;
            best = mb;
        }
        if (tm == 1) break;
    }
    return best;
}

template <int FP, int EPI>
static hipError_t launch_mm(const RowsSplit &a, const Q4Frag &w, const MmOut &o, int run_chunks, hipStream_t s)
{
    if (a.M < 1 || a.kc != w.kc || run_chunks < 1 || run_chunks % 4 || !w.data) return hipErrorInvalidValue;
    if ((size_t)a.M * a.kc * 256 > ((size_t)1 << 31)) return hipErrorInvalidValue;
    if ((EPI == MM_SWIGLU || EPI == MM_PART_DUAL) != (w.dual != 0)) return hipErrorInvalidValue;
    if (EPI == MM_SWIGLU && (w.ng % 4 || run_chunks < w.kc)) return hipErrorInvalidValue;
    if (FP == 1 && !a.rsc) return hipErrorInvalidValue;
    const int tn = (w.ng + 3) / 4, nrun = (w.kc + run_chunks - 1) / run_chunks;
    const int mb = mm_mb(a.M, tn * nrun, MM_MAX_MB), tm = (a.M + 16 * mb - 1) / (16 * mb);
    const dim3 grid((unsigned)(tm * tn * nrun));
    switch (mb) {
#define MM_CASE(B) \
    case B: hipLaunchKernelGGL((k_q4_gemm<B, FP, EPI>), grid, dim3(256), 0, s, a, w, o, tm, nrun, run_chunks); break;
        MM_CASE(1) MM_CASE(2) MM_CASE(3) MM_CASE(4)
#undef MM_CASE
    default: hipLaunchKernelGGL((k_q4_gemm<MM_MAX_MB, FP, EPI>), grid, dim3(256), 0, s, a, w, o, tm, nrun, run_chunks); break;
    }
    return hipGetLastError();
}

hipError_t enqueue_split_rows(const float *X, int ld, int M, int K, uint8_t *out, int kc, float *rsc, int ldr,
                              hipStream_t s)
{
    hipLaunchKernelGGL(k_split_rows, dim3(M), dim3(256), 0, s, X, ld, K, out, kc, rsc, ldr);
    return hipGetLastError();
}

// Rows up to which a prompt's GEMMs run one workgroup per K segment (each
// writes its own partial sums) instead of one per slice: few row tiles leave
// the chip idle behind long K loops, and the partial sums are still small:
// 28 layers of 10 rows 1.56 -> 1.44 ms, of 3 rows 1.51 -> 1.38.
constexpr int MM_SEG_ROWS = 64;

static int mm_run_chunks(const Q4Frag &w, int M)
{
    // (down's 24 segments: 24 partial sums are more to add than they save
    // from 17 rows on)
    return M <= (mm_segments(w) > 8 ? 16 : MM_SEG_ROWS) ? 4 : 4 * (mm_segments(w) / mm_slices(w));
}

size_t mm_part_floats(const Q4Frag &w, int M)
{
    const int rc = mm_run_chunks(w, M);
    return (size_t)((w.kc + rc - 1) / rc) * M * w.ng * 32;
}

// A projection into partial sums.  The rows' factors change every 64 columns
// (fp1), every 256 (rsc with rseg) or not at all.
hipError_t enqueue_mm_parts(const RowsSplit &a, const Q4Frag &w, bool fp1, float *part, MmParts *p, hipStream_t s)
{
    const int rc = mm_run_chunks(w, a.M), nseg = mm_segments(w);
    p->p = part;
    p->ld = w.ng * 32;
    p->stride = (size_t)a.M * p->ld;
    p->n = (w.kc + rc - 1) / rc;
    p->per = rc == 4 && mm_slices(w) < nseg ? nseg / mm_slices(w) : 1;
    const MmOut o{part, p->ld, 1, nullptr, 0, nullptr};
    return fp1 ? launch_mm<1, MM_PART>(a, w, o, rc, s) : launch_mm<4, MM_PART>(a, w, o, rc, s);
}

template <int NP>
struct FoldSwiglu {
    static hipError_t go(const MmParts &p, int M, int slots, uint8_t *rows, int okc, float *rsc, hipStream_t s)
    {
        hipLaunchKernelGGL(k_fold_swiglu<NP>, dim3((slots + 3) / 4, M), dim3(256), 0, s, p, M, slots, rows, okc, rsc);
        return hipGetLastError();
    }
};

template <int NP>
struct FoldStore {
    static hipError_t go(const MmParts &p, int M, int ncols, const float *bias, int silu, float *Y, int ldy, hipStream_t s)
    {
        hipLaunchKernelGGL(k_fold_store<NP>, dim3((ncols + 1023) / 1024, M), dim3(256), 0, s, p, M, ncols, bias, silu, Y, ldy);
        return hipGetLastError();
    }
};

// silu(gate) up into split rows [M][okc records], factors rsc[64-column slot][M]
hipError_t enqueue_mm_swiglu(const RowsSplit &a, const Q4Frag &w, float *part, uint8_t *rows, int okc, float *rsc,
                             hipStream_t s)
{
    const int slots = w.ng / 4;
    if (a.M > MM_SEG_ROWS) return launch_mm<4, MM_SWIGLU>(a, w, MmOut{nullptr, 0, 0, rows, okc, rsc}, 4 * mm_segments(w), s);
    MmParts p{part, w.ng * 32, (size_t)a.M * w.ng * 32, mm_segments(w), mm_segments(w)};
    GCHK((launch_mm<4, MM_PART_DUAL>(a, w, MmOut{part, p.ld, 1, nullptr, 0, nullptr}, 4, s)));
    return by_parts<FoldSwiglu>(p.n, p, a.M, slots, rows, okc, rsc, s);
}

size_t mm_swiglu_part_floats(const Q4Frag &w, int M)
{
    return M <= MM_SEG_ROWS ? (size_t)mm_segments(w) * M * w.ng * 32 : 0;
}

// Whether plain rows run one workgroup per (tile, K segment) and add partial
// sums, against one long K loop a tile: a segment saved is 2.2 us while the
// tiles alone do not fill the CUs, the second launch costs 5, a second round
// of workgroups 6 more, and the partial sums go out and back at about 4.2 TB/s.
// Loop / segments, us, calls one behind the other: 6144 x 2048 16 rows 48 / 14,
// 400 rows 72 / 67, 500 rows 72 / 82; 2048 x 4096 64 rows 19 / 16, 100 rows 20 /
// 22; 1024 x 2048 16 rows 11.5 / 8.9, 130 rows 12.0 / 12.8; 512 x 2048 3 rows
// 7.7 / 8.8 (never).
static bool rows_by_segment(int64_t rows, size_t ncols, int nseg)
{
    const bool rounds = (rows + 79) / 80 * ((int64_t)(ncols + 127) / 128) * nseg > 256;
    return 8.0 * rows * ncols * nseg < 4.2e6 * (2.2 * (nseg - 1) - (rounds ? 11 : 5));
}

// Plain rows: Y[M][ldy] columns 0..ng*32-1 = (silu)(X W (+ bias)), the rows
// split into `ws` first.  ws_floats bounds what one batch of rows may use
// (split rows, factors, partial sums); more rows run in batches.  The sums of
// a weight are cut into the same segments at any batch size; whether they
// are added in registers or from partial sums does not change a bit.  Bias and
// SiLU are applied where partial sums are added.
hipError_t enqueue_mm_rows(const Q4Frag &w, const float *X, int ld, int rows, const float *bias, bool silu, float *Y,
                           int ldy, float *ws, size_t ws_floats, hipStream_t s)
{
    const int nseg = mm_segments(w);
    const size_t per_row = (size_t)w.kc * 64 + nseg, ncols = (size_t)w.ng * 32;
    const size_t cap_parts = ws_floats / (per_row + (size_t)nseg * ncols);
    const bool parts = bias || silu || ((size_t)rows <= cap_parts && rows_by_segment(rows, ncols, nseg));
    size_t cap = parts ? cap_parts : ws_floats / per_row;
    if (cap < 1) return hipErrorInvalidValue;
    if ((size_t)rows > cap) {
        // equal batches of whole row blocks
        const size_t nb = (rows + cap - 1) / cap, per = ((rows + nb - 1) / nb + 15) & ~(size_t)15;
        cap = per <= cap ? per : cap >= 16 ? cap & ~(size_t)15 : cap;
    }
    for (int r0 = 0; r0 < rows; r0 += (int)cap) {
        const int M = (int)std::min<size_t>(cap, rows - r0);
        // split rows first (16-byte aligned), then the parts, then the factors
        uint8_t *sp = (uint8_t *)ws;
        float *part = ws + (size_t)M * w.kc * 64;
        float *rsc = part + (parts ? (size_t)nseg * M * ncols : 0);
        GCHK(enqueue_split_rows(X + (size_t)r0 * ld, ld, M, w.k, sp, w.kc, rsc, M, s));
        const RowsSplit a{sp, w.kc, M, rsc, M, 1.0f};
        float *y = Y + (size_t)r0 * ldy;
        if (parts) {
            MmParts p{part, (int)ncols, (size_t)M * ncols, nseg, nseg};
            GCHK((launch_mm<4, MM_PART>(a, w, MmOut{part, p.ld, 1, nullptr, 0, nullptr}, 4, s)));
            GCHK(by_parts<FoldStore>(p.n, p, M, (int)ncols, bias, silu ? 1 : 0, y, ldy, s));
        } else {
            const int vec = ldy % 4 == 0 && ((uintptr_t)y & 15) == 0;
            GCHK((launch_mm<4, MM_STORE>(a, w, MmOut{y, ldy, vec, nullptr, 0, nullptr}, 4 * nseg, s)));
        }
    }
    return hipSuccess;
}

// Workspace of one batch of M rows with partial sums (bias / SiLU), and what
// plain rows take at once, up to a bound.
size_t mm_rows_ws_floats(const Q4Frag &w, int M)
{
    return (size_t)M * (w.kc * 64 + mm_segments(w) * (1 + (size_t)w.ng * 32));
}

size_t mm_plain_ws_floats(const Q4Frag &w, int64_t M, size_t most)
{
    const size_t nseg = mm_segments(w), ncols = (size_t)w.ng * 32;
    const size_t loop = (size_t)M * (w.kc * 64 + nseg), seg = loop + (size_t)M * nseg * ncols;
    return std::min(most, seg <= most && rows_by_segment(M, ncols, (int)nseg) ? seg : loop);
}

}  // namespace qtts
