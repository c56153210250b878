// qtts_dconv.hip — the speech decoder's Vocos stages (decoder.rs:495-560,
// conv.rs:114-349) position-major on the matrix cores.
//
// Between the stages a signal of C channels is kept as split rows, one row
// per position: C / 32 records of 128 B, 32 f16 hi then 32 f16 lo (hi + lo
// carries 22 of an f32's 24 bits), written once by the kernel that produces
// it.  A causal convolution is then a GEMM whose rows are positions and whose
// taps are row offsets: the tile's rows (and the dilated taps' reach) go into
// LDS once per 32 channels and serve every tap, with no conversion and no
// gather on the way.  Weights are split and permuted into fragment order at
// upload and go from L2 straight into registers.
//
// The channels of a record are ordered by the matrix instruction's layout:
// slot 8q + u holds channel 4q + u (u < 4) or 16 + 4q + u - 4, so that the
// eight results a lane has of two 16-channel blocks (channels 4q..+3 of each)
// are one 16-byte store, and are, as they stand, the operand of a 1x1
// convolution over them.
//
// Bound: three f16 matrix instructions per useful one.  A wave's tile of 64
// positions x 96 channels reads 8 KB of rows (LDS) and 12 KB of weights (L1)
// for 72 matrix instructions of 16 cycles.  Channel-first f32 signals,
// converted and gathered tap by tap while staging, kept those pipes busy
// 17-25% of the time.  Measured (160 frames): a k 7 convolution of 192
// channels 267 -> 170 us, the 96-channel residual unit 301 -> 242 us, the
// decode 5.5 -> 4.0 ms with the transformer below.
#include "qtts_device.h"
#include "qtts_kernels.h"
#include "qtts_devutil.h"
#include "qtts_mfma.h"
#include "qtts_snake.h"

#include <algorithm>
#include <cstdlib>

namespace qtts {

// ---------------------------------------------------------------------------
// Weights: f32 [rows][kt * ic] (k = tap * ic + channel) -> per 16 CB output
// channels, 32 input channels and tap, CB blocks of hi then lo fragments
// (1 KB each).  Every row is scaled by the power of two that takes its
// largest |w| into [2^14, 2^15), so both halves are normal f16; un[row]
// undoes it.
// ---------------------------------------------------------------------------

__device__ __forceinline__ int slot_channel(int q, int u) { return u < 4 ? 4 * q + u : 12 + 4 * q + u; }

__global__ void __launch_bounds__(256)
k_dconv_row_scale(const float *w, int rows, int kd, float *un)
{
    const int lane = threadIdx.x & 63, r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    float mx = 0.0f;
    for (int k = lane; k < kd; k += 64) mx = fmaxf(mx, fabsf(w[(size_t)r * kd + k]));
    mx = wave_max_dpp(mx);
    if (lane == 0) un[r] = __builtin_ldexpf(1.0f, -range_shift(mx));
}

// One wave per (16-row block, record); grid covers rows/16 * ic/32 * kt.
__global__ void __launch_bounds__(256)
k_dconv_pack(const float *w, const float *un, int rows, int ic, int kt, int cb, uint8_t *out)
{
    const int lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4, nc = ic / 32;
    const int64_t id = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (id >= (int64_t)(rows / 16) * nc * kt) return;
    const int tap = (int)(id % kt), c = (int)(id / kt % nc), blk = (int)(id / kt / nc);
    const int tile = blk / cb, b = blk - tile * cb, row = 16 * blk + r16;
    const float p2 = 1.0f / un[row];                 // a power of two: exact
    float v[8];
    for (int u = 0; u < 8; u++) v[u] = w[(size_t)row * kt * ic + (size_t)tap * ic + 32 * c + slot_channel(q, u)] * p2;
    uint32_t h[4], l[4];
    for (int i = 0; i < 4; i++) split_f16_pair<true>(v[2 * i], v[2 * i + 1], h[i], l[i]);
    uint8_t *o = out + ((((size_t)tile * nc + c) * kt + tap) * cb + b) * 2048 + 16 * lane;
    *(uint4 *)o = uint4{h[0], h[1], h[2], h[3]};
    *(uint4 *)(o + 1024) = uint4{l[0], l[1], l[2], l[3]};
}

// e^alpha and e^-beta of a SnakeBeta's channels
__global__ void k_snake_par(const float *alpha, const float *beta, int n, float *out)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    out[i] = expf(alpha[i]);
    out[n + i] = expf(-beta[i]);
}

// ---------------------------------------------------------------------------
// The convolution.  Workgroup: 64 PB positions x 16 CB channels, four waves
// of 16 PB positions each; a slice of the input records.  LDS row r of a
// record at 128 r, its 16-byte part p at slot p ^ (r / 2) % 8: sixteen
// consecutive rows of one part (a fragment read, at any tap's offset) take
// sixteen different 16-byte columns of the banks, and so do two whole rows (a
// write).  While a record's taps run, the next record's rows come in, a few
// 16-byte pieces a thread per tap, and each weight block's registers are
// refilled for the next tap as soon as its products are issued.
// ---------------------------------------------------------------------------

enum { DC_SNAKE = 0, DC_X_SNAKE = 1, DC_RAW = 2 };   // RAW: the sums of the slices, for a consumer below

struct DcIn {
    const uint8_t *x;        // split rows
    int nc, L, dil;          // records a row, rows, dilation
};

struct DcOut {
    uint8_t *ys;             // split rows of the stage's snake, or
    float *yf;               // its f32 rows (the last stage)
    float *x;                // DC_X_SNAKE: f32 rows of the signal itself
    const float *res;        // DC_X_SNAKE: residual added to it, or null
    const float *bias, *un;  // [M]; un: [phase][M]
    const float *snake;      // [2][M] e^alpha, e^-beta
    int M, os;               // channels; output row of (position n, phase ph): n os + ph
    float *rm;               // range check: a word a wave (range_note)
};

struct DcGeo {
    int tm, tn, nph, ks, cps;   // channel and position tiles, phases, slices of cps records
    float *part;                // ks > 1: raw sums [slice][output row][M]
};

// conv2 of a residual unit behind its conv1 (FUSE)
struct DcFuse {
    const uint8_t *w;
    DcOut o;
};

// The split holds a value as f16 hi + lo: f32-accurate below the f16 maximum
// and, through lo, to 2^-25 absolute.  So every wave that stores split rows
// notes its largest |value| (a plain store: atomics on words of several waves
// lengthened each launch by 2 us), and workgroups beside the output
// convolution's test them (a launch of their own took 10 us, 1% of a short
// chunk), over all channels of 64 positions (16 before a stride): a group that
// reaches the maximum, or lies wholly below the normal f16 but is not zero, is
// out, and the host repeats the decode on the f32 matrix path.  Quiet channels
// beside loud ones of the same positions lose nothing that shows in the sums
// over them.
__device__ __forceinline__ void range_test(const int32_t *flag, const RangeList &l, int32_t *out, int block)
{
    const RangeSignal g = l.s[block / l.blocks];
    // 2^b lanes a group of `per` words
    const int lane = threadIdx.x & 63, wv = block % l.blocks * 4 + (threadIdx.x >> 6), nw = l.blocks * 4;
    const int b = g.per >= 64 ? 6 : 32 - __clz(g.per - 1), lg = lane >> b, ll = lane & ((1 << b) - 1);
    const uint32_t groups = (g.words + g.per - 1) / g.per;
    bool bad = *flag != 0;
    for (uint32_t g0 = (uint32_t)wv << (6 - b); g0 < groups; g0 += (uint32_t)nw << (6 - b)) {
        const uint32_t w0 = (g0 + lg) * g.per;
        float m = 0.0f;
        for (uint32_t i = ll; i < g.per && w0 + i < g.words; i += 1u << b) m = fmaxf(m, g.p[w0 + i]);
        for (int x = (1 << b) >> 1; x; x >>= 1) m = fmaxf(m, __shfl_xor(m, x));
        bad |= !(m < 65504.0f) || (m > 0.0f && m < 0x1p-14f);
    }
    if (bad) *out = 1;
}

__global__ void __launch_bounds__(256)
k_range_result(const int32_t *flag, RangeList l, int32_t *out)
{
    range_test(flag, l, out, blockIdx.x);
}

__device__ __forceinline__ float dc_snake(float v, float ea, float eb) { return v + eb * snake_sin2(ea * v); }

// eight outputs of one position (two blocks' channels 4q..+3, record rec)
__device__ __forceinline__ void dc_store8(const DcOut &o, size_t row, int rec, int q, const f32x4 &a, const f32x4 &b)
{
    if (o.yf) {
        float *y = o.yf + row * o.M + 32 * rec + 4 * q;
        *(f32x4 *)y = a;
        *(f32x4 *)(y + 16) = b;
        return;
    }
    uint32_t h[4], l[4];
    split_f16_pair<true>(a.x, a.y, h[0], l[0]);
    split_f16_pair<true>(a.z, a.w, h[1], l[1]);
    split_f16_pair<true>(b.x, b.y, h[2], l[2]);
    split_f16_pair<true>(b.z, b.w, h[3], l[3]);
    uint8_t *y = o.ys + row * ((size_t)o.M * 4) + rec * 128 + 16 * q;
    *(uint4 *)y = uint4{h[0], h[1], h[2], h[3]};
    *(uint4 *)(y + 64) = uint4{l[0], l[1], l[2], l[3]};
}

__device__ __forceinline__ float max4(float m, const f32x4 &v)
{
    return fmaxf(fmaxf(fmaxf(m, fabsf(v.x)), fmaxf(fabsf(v.y), fabsf(v.z))), fabsf(v.w));
}

template <int EPI>
__device__ __forceinline__ f32x4 dc_epi(const DcOut &o, f32x4 acc, const f32x4 &un, const f32x4 &bias, const f32x4 &ea,
                                        const f32x4 &eb, const f32x4 &ext, float *x)
{
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float v = acc[e] * un[e] + bias[e];
        if (EPI == DC_X_SNAKE) {
            if (o.res) v += ext[e];
            acc[e] = v;
        }
        y[e] = dc_snake(v, ea[e], eb[e]);
    }
    if (EPI == DC_X_SNAKE) *(f32x4 *)x = acc;
    return y;
}

template <int CB, int PB, int KT, int EPI, bool FUSE, bool SK>
__global__ void __launch_bounds__(256, SK && KT > 2 ? 1 : 2)
k_dconv(DcIn in, const uint8_t *wts, DcOut o, DcGeo g, DcFuse fz)
{
    // SK: the waves share the positions (16 PB) and take every fourth record
    constexpr int TP = (SK ? 16 : 64) * PB, RMAX = TP + (KT == 7 ? 54 : KT - 1), NT = SK ? 64 : 256;
    constexpr int NP = (RMAX * 8 + NT - 1) / NT, PPT = (NP + KT - 1) / KT;   // 16-byte pieces a thread per record, per tap
    constexpr int PE = SK ? PB / 4 : PB;                                     // position blocks a wave ends with
    static_assert(!SK || PB == 4, "the waves end with a position block each");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_all[];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, r16 = lane & 15, q = lane >> 4, ts = SK ? lane : t;
    // each XCD takes a contiguous run of tiles, positions fastest: the tiles
    // that share weights share an L2
    const int nwg = gridDim.x, id = blockIdx.x, xcd = id & 7, qq = nwg >> 3, rem = nwg & 7;
    int lg = xcd * qq + min(xcd, rem) + (id >> 3);
    const int nt = lg % g.tn;
    lg /= g.tn;
    const int slice = lg % g.ks;
    lg /= g.ks;
    const int ct = lg % g.tm, ph = lg / g.tm;
    const int n0 = nt * TP, pad = (KT - 1) * in.dil, R = TP + pad;
    const int s0 = slice * g.cps, s1 = min(s0 + g.cps, in.nc);
    // this wave's records: c0, c0 + CS, .. below s1 (SK: perhaps none)
    constexpr int CS = SK ? 4 : 1;
    const int c0 = SK ? s0 + __builtin_amdgcn_readfirstlane(wv) : s0, nrec = c0 < s1 ? (s1 - c0 + CS - 1) / CS : 0;
    const int lbuf = R * 128;                        // bytes of one staged record
    uint8_t *const lds = lds_all + (SK ? wv * 2 * lbuf : 0);
    const int rowb = in.nc * 128;
    const uint8_t *xb = in.x + (size_t)n0 * rowb;    // the tile's first position

    const auto piece = [&](int i, int c) -> u32x4 {
        const int idx = ts + NT * i, gr = n0 - pad + (idx >> 3), cl = min(max(gr, 0), in.L - 1);
        const u32x4 v = *(const u32x4 *)(xb + (ptrdiff_t)(cl - n0) * rowb + c * 128 + (idx & 7) * 16);
        return gr == cl ? v : u32x4{0, 0, 0, 0};
    };
    const auto put = [&](int i, int buf, const u32x4 &v) {
        const int idx = ts + NT * i, r = idx >> 3;
        if (r < R) *(u32x4 *)&lds[buf * lbuf + r * 128 + (((idx & 7) ^ ((r >> 1) & 7)) * 16)] = v;
    };
    const uint8_t *wb = wts + (((size_t)(ph * g.tm + ct) * in.nc + c0) * KT) * (CB * 2048) + 16 * lane;
    // SK: one wave a SIMD (the staged rows fill the LDS) and nothing else to
    // cover the L2's latency, so its weights come two steps ahead, in the
    // registers that leaves: decode of 5 frames 1.12 -> 1.06 ms, of 21 frames
    // 1.48 -> 1.40 ms, of 40 frames 2.04 -> 1.89 ms.  With one or two taps a
    // wave has too few steps: the second set costs 1 frame 0.02 ms.
    constexpr int WS = SK && KT > 2 ? 2 : 1;
    half8 wr[WS][CB][2];
    // block b of the wave's step st (record st / KT, tap st % KT) into set u
    const int nst = nrec * KT;
    const auto load_w = [&](int u, int b, int st) {
        st = min(st, nst - 1);
        const int i = st / KT, tap = st - i * KT;
        const uint8_t *p = wb + (size_t)(i * CS * KT + tap) * (CB * 2048) + b * 2048;
        wr[u][b][0] = *(const half8 *)p;
        wr[u][b][1] = *(const half8 *)(p + 1024);
    };
    f32x4 acc[PB][CB];
#pragma unroll
    for (int p = 0; p < PB; p++)
#pragma unroll
        for (int b = 0; b < CB; b++) acc[p][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    if (!SK || nrec) {
        u32x4 v[NP];
#pragma unroll
        for (int i = 0; i < NP; i++) v[i] = piece(i, c0);
#pragma unroll
        for (int u = 0; u < WS; u++)
#pragma unroll
            for (int b = 0; b < CB; b++) load_w(u, b, u);
#pragma unroll
        for (int i = 0; i < NP; i++) put(i, 0, v[i]);
    }
    if constexpr (SK) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
    for (int c = 0; c < nrec; c++) {
        const int buf = c & 1, cn = c0 + min(c + 1, nrec - 1) * CS;
#pragma unroll
        for (int tap = 0; tap < KT; tap++) {
            u32x4 v[PPT];
#pragma unroll
            for (int i = 0; i < PPT; i++)
                if (tap * PPT + i < NP) v[i] = piece(tap * PPT + i, cn);
            half8 xh[PB], xl[PB];
#pragma unroll
            for (int p = 0; p < PB; p++) {
                const int r = 16 * ((SK ? 0 : PB * wv) + p) + r16 + tap * in.dil, z = (r >> 1) & 7;
                xh[p] = *(const half8 *)&lds[buf * lbuf + r * 128 + ((q ^ z) * 16)];
                xl[p] = *(const half8 *)&lds[buf * lbuf + r * 128 + (((q + 4) ^ z) * 16)];
            }
            const int u = tap % WS;
#pragma unroll
            for (int b = 0; b < CB; b++) {
#pragma unroll
                for (int p = 0; p < PB; p++)
                    acc[p][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wr[u][b][1], xh[p], acc[p][b], 0, 0, 0);
#pragma unroll
                for (int p = 0; p < PB; p++)
                    acc[p][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wr[u][b][0], xl[p], acc[p][b], 0, 0, 0);
#pragma unroll
                for (int p = 0; p < PB; p++)
                    acc[p][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wr[u][b][0], xh[p], acc[p][b], 0, 0, 0);
                load_w(u, b, c * KT + tap + WS);
            }
#pragma unroll
            for (int i = 0; i < PPT; i++)
                if (tap * PPT + i < NP) put(tap * PPT + i, buf ^ 1, v[i]);
        }
        if constexpr (WS == 2 && KT % 2) {
            // an odd record ends on the other set
#pragma unroll
            for (int b = 0; b < CB; b++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const half8 t = wr[0][b][j];
                    wr[0][b][j] = wr[WS - 1][b][j];
                    wr[WS - 1][b][j] = t;
                }
        }
        if constexpr (SK) {
            // one wave's lanes hand each other rows through LDS
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
            __syncthreads();
        }
    }
    if constexpr (SK) {
        // the waves' sums added in wave order, a position block a wave
        f32x4 *rs = (f32x4 *)lds_all;
        __syncthreads();
#pragma unroll
        for (int p = 0; p < PB; p++)
#pragma unroll
            for (int b = 0; b < CB; b++) rs[((wv * PB + p) * CB + b) * 64 + lane] = acc[p][b];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < CB; b++) {
            f32x4 a = rs[(wv * CB + b) * 64 + lane];
#pragma unroll
            for (int w = 1; w < 4; w++) a += rs[((w * PB + wv) * CB + b) * 64 + lane];
            acc[0][b] = a;
        }
        __syncthreads();
    }

    const int nw = n0 + 16 * PE * wv + r16;          // position of p = 0
    if (EPI == DC_RAW || g.ks > 1) {
        float *pp = g.part + (size_t)slice * in.L * g.nph * o.M;
#pragma unroll
        for (int p = 0; p < PE; p++) {
            const int n = nw + 16 * p;
            if (n >= in.L) continue;
            float *row = pp + ((size_t)n * o.os + ph) * o.M + ct * 16 * CB + 4 * q;
#pragma unroll
            for (int b = 0; b < CB; b++) *(f32x4 *)(row + 16 * b) = acc[p][b];
        }
        return;
    }
    const int n16 = n0 / 16 + PE * wv;               // for the range check's words
    if constexpr (EPI == DC_RAW) {
    } else if constexpr (!FUSE) {
        float mx[PE];
#pragma unroll
        for (int p = 0; p < PE; p++) mx[p] = 0.0f;
#pragma unroll
        for (int b = 0; b < CB; b += 2) {
            const int ch = ct * 16 * CB + 16 * b + 4 * q;
            f32x4 un[2], bi[2], ea[2], eb[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                un[j] = ld4(o.un + ph * o.M + ch + 16 * j);
                bi[j] = ld4(o.bias + ch + 16 * j);
                ea[j] = ld4(o.snake + ch + 16 * j);
                eb[j] = ld4(o.snake + o.M + ch + 16 * j);
            }
            f32x4 ext[PE][2];
            if (EPI == DC_X_SNAKE && o.res) {
#pragma unroll
                for (int p = 0; p < PE; p++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        ext[p][j] = ld4(o.res + ((size_t)min(nw + 16 * p, in.L - 1) * o.os + ph) * o.M + ch + 16 * j);
            }
#pragma unroll
            for (int p = 0; p < PE; p++) {
                const int n = nw + 16 * p;
                if (n >= in.L) continue;
                const size_t row = (size_t)n * o.os + ph;
                f32x4 y[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    y[j] = dc_epi<EPI>(o, acc[p][b + j], un[j], bi[j], ea[j], eb[j], ext[p][j],
                                       EPI == DC_X_SNAKE ? o.x + row * o.M + ch + 16 * j : nullptr);
                    mx[p] = max4(mx[p], y[j]);
                }
                dc_store8(o, row, (ct * CB + b) / 2, q, y[0], y[1]);
            }
        }
        if (o.ys && o.os > 1) {
#pragma unroll
            for (int p = 0; p < PE; p++) range_note(o.rm + ((size_t)(n16 + p) * g.tm + ct) * g.nph + ph, mx[p], lane);
        } else if (o.ys) {
#pragma unroll
            for (int p = 1; p < PE; p++) mx[0] = fmaxf(mx[0], mx[p]);
            range_note(o.rm + (size_t)(n16 / PE) * g.tm + ct, mx[0], lane);
        }
    } else {
        // conv1's snake stays in registers as conv2's operand (the 16 CB
        // channels are all of conv2's input); the same values, products and
        // order as through a split row
        half8 th[PE][CB / 2], tl[PE][CB / 2];
        float mx = 0.0f;
        // the residual, in flight behind conv1's snakes
        const DcOut &o2 = fz.o;
        f32x4 ext[PE][CB];
#pragma unroll
        for (int p = 0; p < PE; p++)
#pragma unroll
            for (int b = 0; b < CB; b++) ext[p][b] = ld4(o2.res + (size_t)min(nw + 16 * p, in.L - 1) * o2.M + 16 * b + 4 * q);
#pragma unroll
        for (int b = 0; b < CB; b += 2) {
            const int ch = 16 * b + 4 * q;
            f32x4 un[2], bi[2], ea[2], eb[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                un[j] = ld4(o.un + ch + 16 * j);
                bi[j] = ld4(o.bias + ch + 16 * j);
                ea[j] = ld4(o.snake + ch + 16 * j);
                eb[j] = ld4(o.snake + o.M + ch + 16 * j);
            }
#pragma unroll
            for (int p = 0; p < PE; p++) {
                f32x4 y[2];
#pragma unroll
                for (int j = 0; j < 2; j++)
                    y[j] = dc_epi<DC_SNAKE>(o, acc[p][b + j], un[j], bi[j], ea[j], eb[j], f32x4{}, nullptr);
                if (nw + 16 * p < in.L) mx = max4(max4(mx, y[0]), y[1]);
                uint32_t h[4], l[4];
                split_f16_pair<true>(y[0].x, y[0].y, h[0], l[0]);
                split_f16_pair<true>(y[0].z, y[0].w, h[1], l[1]);
                split_f16_pair<true>(y[1].x, y[1].y, h[2], l[2]);
                split_f16_pair<true>(y[1].z, y[1].w, h[3], l[3]);
                th[p][b / 2] = __builtin_bit_cast(half8, uint4{h[0], h[1], h[2], h[3]});
                tl[p][b / 2] = __builtin_bit_cast(half8, uint4{l[0], l[1], l[2], l[3]});
            }
        }
        range_note(o.rm + n16 / PE, mx, lane);
        float mx2 = 0.0f;
#pragma unroll
        for (int b = 0; b < CB; b += 2) {
            f32x4 a2[PE][2];
#pragma unroll
            for (int p = 0; p < PE; p++) a2[p][0] = a2[p][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            const int ch = 16 * b + 4 * q;
#pragma unroll
            for (int c = 0; c < CB / 2; c++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint8_t *w2 = fz.w + ((size_t)c * CB + b + j) * 2048 + 16 * lane;
                    const half8 wh = *(const half8 *)w2, wl = *(const half8 *)(w2 + 1024);
#pragma unroll
                    for (int p = 0; p < PE; p++)
                        a2[p][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wl, th[p][c], a2[p][j], 0, 0, 0);
#pragma unroll
                    for (int p = 0; p < PE; p++)
                        a2[p][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh, tl[p][c], a2[p][j], 0, 0, 0);
#pragma unroll
                    for (int p = 0; p < PE; p++)
                        a2[p][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh, th[p][c], a2[p][j], 0, 0, 0);
                }
            f32x4 un[2], bi[2], ea[2], eb[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                un[j] = ld4(o2.un + ch + 16 * j);
                bi[j] = ld4(o2.bias + ch + 16 * j);
                ea[j] = ld4(o2.snake + ch + 16 * j);
                eb[j] = ld4(o2.snake + o2.M + ch + 16 * j);
            }
#pragma unroll
            for (int p = 0; p < PE; p++) {
                const int n = nw + 16 * p;
                if (n >= in.L) continue;
                f32x4 y[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    y[j] = dc_epi<DC_X_SNAKE>(o2, a2[p][j], un[j], bi[j], ea[j], eb[j], ext[p][b + j],
                                              o2.x + (size_t)n * o2.M + ch + 16 * j);
                    mx2 = max4(mx2, y[j]);
                }
                dc_store8(o2, n, b / 2, q, y[0], y[1]);
            }
        }
        if (o2.ys) range_note(o2.rm + n16 / PE, mx2, lane);
    }
}

// Split slices added in slice order, then the epilogue; a thread per output
// row and eight channels (as dc_store8 stores them).
template <int EPI>
__global__ void __launch_bounds__(256)
k_dconv_reduce(const float *part, int ks, int64_t rows, int nph, DcOut o)
{
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x, n8 = o.M / 8;
    float mx = 0.0f;
    if (id < rows * n8) {
        const int64_t row = id / n8;
        const int j8 = (int)(id - row * n8), rec = j8 >> 2, q = j8 & 3, ch = 32 * rec + 4 * q, ph = (int)(row % nph);
        f32x4 a[2];
        for (int j = 0; j < 2; j++) a[j] = ld4(part + row * o.M + ch + 16 * j);
        for (int s = 1; s < ks; s++)
            for (int j = 0; j < 2; j++) a[j] += ld4(part + ((size_t)s * rows + row) * o.M + ch + 16 * j);
        f32x4 y[2];
        for (int j = 0; j < 2; j++) {
            const int c = ch + 16 * j;
            const f32x4 ext = EPI == DC_X_SNAKE && o.res ? ld4(o.res + row * o.M + c) : f32x4{};
            y[j] = dc_epi<EPI>(o, a[j], ld4(o.un + ph * o.M + c), ld4(o.bias + c), ld4(o.snake + c), ld4(o.snake + o.M + c),
                               ext, EPI == DC_X_SNAKE ? o.x + row * o.M + c : nullptr);
            mx = max4(mx, y[j]);
        }
        dc_store8(o, row, rec, q, y[0], y[1]);
    }
    if (o.ys) range_note(o.rm + (id >> 6), mx, threadIdx.x & 63);
}

// ---------------------------------------------------------------------------
// The transformer between VQ and upsampling (decoder.rs:198-340) on the same
// rows: its matrices are 1x1 convolutions whose slices' sums the kernels below
// add, each with what follows in the reference.  A few positions and 512 to
// 3072 channels: the launches are bound by the latency of a record's loads,
// so a launch takes many slices of one record a wave, and the kernels that
// add the slices issue all their loads before the first addition.  The 8
// layers of 512 channels, whole decode, channel-first before and this: 1
// frame 1.20 -> 1.01 ms, 21 frames 1.67 -> 1.48 ms, 160 frames 4.24 -> 4.10.
// ---------------------------------------------------------------------------

struct LinSum {
    const float *part;       // [ks][rows][M]
    const float *un, *bias;  // [M]; bias may be null
    int ks, rows, M;
};

// four consecutive channels of a row (KS > 0: that many slices, every load
// issued before the first addition)
template <int KS>
__device__ __forceinline__ f32x4 lin_sum(const LinSum &p, int row, int ch)
{
    const float *a = p.part + (size_t)row * p.M + ch;
    const size_t st = (size_t)p.rows * p.M;
    f32x4 v;
    if constexpr (KS > 0) {
        f32x4 x[KS];
#pragma unroll
        for (int s = 0; s < KS; s++) x[s] = ld4(a + s * st);
        v = x[0];
#pragma unroll
        for (int s = 1; s < KS; s++) v += x[s];
    } else {
        v = ld4(a);
        for (int s = 1; s < p.ks; s++) v += ld4(a + s * st);
    }
    v *= ld4(p.un + ch);
    return p.bias ? v + ld4(p.bias + ch) : v;
}

// slot store of eight channels (record rec, lane group q) of a split row
__device__ __forceinline__ void split_store8(uint8_t *ys, int row, int C, int rec, int q, const f32x4 &a, const f32x4 &b)
{
    DcOut o{};
    o.ys = ys;
    o.M = C;
    dc_store8(o, row, rec, q, a, b);
}

// plain f32 rows
template <int KS>
__global__ void __launch_bounds__(256)
k_lin_rows(LinSum p, float *y)
{
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x, n4 = p.M / 4;
    if (id >= p.rows * n4) return;
    const int row = (int)(id / n4), ch = 4 * (int)(id - row * n4);
    *(f32x4 *)(y + (size_t)row * p.M + ch) = lin_sum<KS>(p, row, ch);
}

// channel-first [M][rows]: 64 rows x 32 channels through LDS
template <int KS>
__global__ void __launch_bounds__(256)
k_lin_cf(LinSum p, float *y)
{
    __shared__ float tile[64][33];
    const int t = threadIdx.x, r0 = blockIdx.x * 64, c0 = blockIdx.y * 32;
    for (int i = t; i < 64 * 8; i += 256) {
        const int r = i >> 3, c = 4 * (i & 7);
        if (r0 + r < p.rows) {
            const f32x4 v = lin_sum<KS>(p, r0 + r, c0 + c);
            for (int e = 0; e < 4; e++) tile[r][c + e] = v[e];
        }
    }
    __syncthreads();
    for (int i = t; i < 64 * 32; i += 256) {
        const int r = i & 63, c = i >> 6;
        if (r0 + r < p.rows) y[(size_t)(c0 + c) * p.rows + r0 + r] = tile[r][c];
    }
}

// silu(gate) up of interleaved rows (gate 2j, up 2j + 1) into split rows
template <int KS>
__global__ void __launch_bounds__(256)
k_lin_swiglu(LinSum p, uint8_t *ys, float *rm)
{
    const int C = p.M / 2, n8 = C / 8;
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    float mx = 0.0f;
    if (id < (int64_t)p.rows * n8) {
        const int row = (int)(id / n8), j8 = (int)(id - (int64_t)row * n8), rec = j8 >> 2, q = j8 & 3;
        f32x4 y[2];
        for (int j = 0; j < 2; j++) {
            const int c = 2 * (32 * rec + 4 * q + 16 * j);
            const f32x4 a = lin_sum<KS>(p, row, c), b = lin_sum<KS>(p, row, c + 4);
            y[j] = f32x4{silu_f(a.x) * a.y, silu_f(a.z) * a.w, silu_f(b.x) * b.y, silu_f(b.z) * b.w};
            mx = max4(mx, y[j]);
        }
        split_store8(ys, row, C, rec, q, y[0], y[1]);
    }
    range_note(rm + (id >> 6), mx, threadIdx.x & 63);
}

// x (+)= scale * sum, then RMSNorm (eps 1e-5) into split rows; one wave a
// row of at most 512 NV channels, in registers.  scale null: x = sum.
template <int NV, int KS>
__global__ void __launch_bounds__(256)
k_lin_resid_rms(LinSum p, const float *scale, float *x, const float *gamma, uint8_t *ys, float *rm)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, row = blockIdx.x * 4 + wv, H = p.M;
    float mx = 0.0f;
    if (row < p.rows) {
        f32x4 v[NV][2];
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int j8 = lane + 64 * i, ch = 32 * (j8 >> 2) + 4 * (j8 & 3) + 16 * j;
                v[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if (8 * j8 >= H) continue;
                f32x4 a = lin_sum<KS>(p, row, ch);
                float *xr = x + (size_t)row * H + ch;
                if (scale) a = ld4(xr) + ld4(scale + ch) * a;
                *(f32x4 *)xr = a;
                v[i][j] = a;
                ss = fmaf(a.x, a.x, fmaf(a.y, a.y, fmaf(a.z, a.z, fmaf(a.w, a.w, ss))));
            }
        const float inv = 1.0f / sqrtf(wave_sum_dpp(ss) / (float)H + 1e-5f);
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int j8 = lane + 64 * i, rec = j8 >> 2, q = j8 & 3;
            if (8 * j8 >= H) continue;
            const f32x4 a = v[i][0] * inv * ld4(gamma + 32 * rec + 4 * q);
            const f32x4 b = v[i][1] * inv * ld4(gamma + 32 * rec + 4 * q + 16);
            mx = max4(max4(mx, a), b);
            split_store8(ys, row, H, rec, q, a, b);
        }
    }
    range_note(rm + row, mx, lane);
}

// Channel-first f32 [C][L] -> split rows: 64 positions x 32 channels through
// LDS; lane = position.
__global__ void __launch_bounds__(256)
k_cf_split(const float *x, int C, int L, uint8_t *ys, float *rm)
{
    __shared__ float tile[32][65];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, p0 = blockIdx.x * 64, rec = blockIdx.y;
    for (int i = wv; i < 32; i += 4) tile[i][lane] = p0 + lane < L ? x[(size_t)(32 * rec + i) * L + p0 + lane] : 0.0f;
    __syncthreads();
    // thread: position t / 4, lane group q = t % 4
    const int p = t >> 2, q = t & 3;
    float v[8], mx = 0.0f;
    for (int u = 0; u < 8; u++) {
        v[u] = tile[slot_channel(q, u)][p];
        mx = fmaxf(mx, fabsf(v[u]));
    }
    if (p0 + p < L) {
        uint32_t h[4], l[4];
        for (int i = 0; i < 4; i++) split_f16_pair<true>(v[2 * i], v[2 * i + 1], h[i], l[i]);
        uint8_t *y = ys + (size_t)(p0 + p) * ((size_t)C * 4) + rec * 128 + 16 * q;
        *(uint4 *)y = uint4{h[0], h[1], h[2], h[3]};
        *(uint4 *)(y + 64) = uint4{l[0], l[1], l[2], l[3]};
    }
    range_note(rm + ((size_t)blockIdx.x * gridDim.y + rec) * 4 + wv, mx, lane);
}

// One-channel output convolution over f32 rows [L][C], clamp to [-1, 1], the
// first `cut` samples dropped.  Workgroup: 64 positions; thread (position,
// quarter of the channels), four quarters added in order.  Bound: reading the
// rows (118 MB at 160 frames, 41 us; 81 us a channel-first plane at a time).
// Workgroups from nout on: the decode's range check.
template <int K>
__global__ void __launch_bounds__(256)
k_out_rows(const float *x, int C, int L, const float *w, float bias, int dil, int64_t cut, float *out, int nout,
           const int32_t *flag, RangeList l, int32_t *out_of_range)
{
    if ((int)blockIdx.x >= nout) {
        range_test(flag, l, out_of_range, blockIdx.x - nout);
        return;
    }
    extern __shared__ float sm[];
    const int t = threadIdx.x, n0 = blockIdx.x * 64, pad = (K - 1) * dil, R = 64 + pad, ld = C + 4;
    float *ws = sm, *xs = sm + ((K * C + 3) & ~3);   // ws [tap][C], xs [R][ld]
    for (int i = t; i < K * C; i += 256) ws[(i % K) * C + i / K] = w[i];
    const int c4 = C / 4;
    for (int i = t; i < R * c4; i += 256) {
        const int r = i / c4, c = 4 * (i - r * c4), n = n0 - pad + r;
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        if (n >= 0 && n < L) v = ld4(x + (size_t)n * C + c);
        *(f32x4 *)(xs + r * ld + c) = v;
    }
    __syncthreads();
    const int p = t >> 2, qr = t & 3;
    float a = 0.0f;
#pragma unroll
    for (int j = 0; j < K; j++) {
        const float *xr = xs + (p + j * dil) * ld, *wr = ws + j * C;
        for (int c = 4 * qr; c < C; c += 16) {
            const f32x4 xv = *(const f32x4 *)(xr + c), wv = *(const f32x4 *)(wr + c);
            a = fmaf(xv.x, wv.x, a);
            a = fmaf(xv.y, wv.y, a);
            a = fmaf(xv.z, wv.z, a);
            a = fmaf(xv.w, wv.w, a);
        }
    }
    a += dpp_mov<0xB1>(a);
    a += dpp_mov<0x4E>(a);
    const int n = n0 + p;
    if (qr == 0 && n < L && n >= cut) out[n - cut] = fminf(fmaxf(a + bias, -1.0f), 1.0f);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

#define VCHK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) return e_; } while (0)

constexpr int DC_CB = DC_VOCOS_CB, DC_LIN_CB = DC_TF_CB;

bool dconv_fits(int oc, int ic, int kt, int dil)
{
    return oc % (16 * DC_CB) == 0 && ic % 32 == 0 && (kt == 7 ? dil >= 1 && dil <= 9 : kt == 1 || (kt == 2 && dil == 1));
}

size_t dconv_weight_bytes(int rows, int ic, int kt) { return (size_t)rows * ic * kt * 4; }

hipError_t enqueue_dconv_pack(const float *w, int rows, int ic, int kt, int cb, uint8_t *out, float *un, hipStream_t s)
{
    hipLaunchKernelGGL(k_dconv_row_scale, dim3((rows + 3) / 4), dim3(256), 0, s, w, rows, ic * kt, un);
    const int64_t n = (int64_t)(rows / 16) * (ic / 32) * kt;
    hipLaunchKernelGGL(k_dconv_pack, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, w, un, rows, ic, kt, cb, out);
    return hipGetLastError();
}

hipError_t enqueue_snake_par(const float *alpha, const float *beta, int n, float *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_snake_par, dim3((n + 255) / 256), dim3(256), 0, s, alpha, beta, n, out);
    return hipGetLastError();
}

// Words of the range check for T frames at most: of a stage's signal the
// partial sums' kernel has the most waves (one per 64 rows and 8 channels).
static size_t range_words(int64_t L, int M, int os) { return (size_t)(L / 16 + 16) * (M / (16 * DC_CB)) * 3 * os + 16; }

size_t dec_range_words(const DecoderDev &d, int64_t T)
{
    size_t n = 0;
    if (d.tf_rows) {
        const size_t rms = T + 4, cf = (T / 64 + 1) * (d.latent / 8), att = (T / 16 + 1) * 4 * d.n_heads;
        n += rms + cf + d.n_tf * (2 * rms + att + (size_t)T * d.inter / 512 + 4);
    }
    if (d.vocos_rows) {
        int64_t L = T;
        for (int u = 0; u < d.n_up; u++) L *= d.up[u].conv_t.stride;
        n += (size_t)(L / 64 + 1) * (d.voc_init.ic / 8) + range_words(L, d.voc_init.oc, 1);
        for (int b = 0; b < d.n_voc; b++) {
            const DecVocos &B = d.voc[b];
            n += range_words(L, B.up.oc, B.up.stride);
            L *= B.up.stride;
            n += 2 * B.n_res * range_words(L, B.up.oc, 1);
        }
    }
    return n;
}

// `words` words for the next launch, `per` of them a group.
static float *range_take(RangeLog &log, size_t words, int per)
{
    if (words > (size_t)(log.end - log.next)) {
        log.full = true;
        return log.next;
    }
    float *p = log.next;
    log.next += words;
    log.sig.push_back(RangeSignal{p, (uint32_t)words, (uint32_t)per});
    return p;
}

// Signals from..+63 of the log, with one or several workgroups each.
static int range_list(const RangeLog &log, size_t from, RangeList *l)
{
    const int k = (int)std::min<size_t>(log.sig.size() - from, RANGE_SIGNALS);
    uint32_t most = 0;
    for (int i = 0; i < k; i++) {
        l->s[i] = log.sig[from + i];
        most = std::max(most, l->s[i].words);
    }
    if (!k) l->s[0] = RangeSignal{nullptr, 0, 1};
    l->blocks = most < 4096 ? 1 : 8;
    return std::max(k, 1) * l->blocks;
}

// *out (host memory, 0 before) becomes 1 if `flag` is set or a signal from
// `from` on left the split's range.
hipError_t enqueue_range_result(const RangeLog &log, size_t from, const int32_t *flag, int32_t *out, hipStream_t s)
{
    do {
        RangeList l{};
        const int n = range_list(log, from, &l);
        hipLaunchKernelGGL(k_range_result, dim3(n), dim3(256), 0, s, flag, l, out);
        VCHK(hipGetLastError());
        from += RANGE_SIGNALS;
    } while (from < log.sig.size());
    return hipSuccess;
}

// Tile form and slices of the contraction: the launch's rounds over the CUs
// times a workgroup's matrix cycles, plus the partial sums' traffic.  Forms:
// 256 positions; 128 (each wave's weights then outrun the L1 by a third); 64
// positions with the records dealt to the four waves (SK), where the four
// hold different weights: few positions take it (a k 7 convolution of 672
// positions and 192 channels 45 us, on 64-position tiles whose waves share
// the weights 118).  A fused residual unit (one slice) does not run on 256
// positions: its four position blocks a wave spill (160 frames: 325 us a unit,
// with two blocks 242).
constexpr double DC_WAIT = 2500;   // cycles, fitted at 1 to 400 frames (0 and 5000 are up to 2% slower at 160)
enum { DC_P256 = 0, DC_P128 = 1, DC_SK64 = 2 };

static void dc_plan(int L, int tm, int nph, int nc, int kt, int M, size_t part_cap, bool fuse, int *form, int *ks_out)
{
    double best = 1e300;
    for (int f = DC_P256; f <= DC_SK64; f++) {
        const int tp = 256 >> f, tn = (L + tp - 1) / tp;
        for (int ks = 1; ks <= std::min(nc, 16); ks++) {
            const int cps = (nc + ks - 1) / ks;
            if ((nc + cps - 1) / cps != ks) continue;     // no empty slice
            if (fuse && ks == 1 && f == DC_P256) continue;
            const double plane = (double)L * nph * M;
            if (ks > 1 && plane * ks > (double)part_cap) break;
            const int64_t wgs = (int64_t)tn * tm * nph * ks;
            const double rounds = (double)((wgs + 255) / 256);
            const double rec = f == DC_SK64 ? (cps + 3) / 4 * 1152.0 : f == DC_P128 ? cps * 576 * 1.4 : cps * 1152.0;
            // with one tap a record's loads outlast its matrix work: the
            // wait shows unless the waves' records overlap
            const double wait = kt > 2 ? 0 : (f == DC_SK64 ? (cps + 3) / 4 : cps) * DC_WAIT / kt;
            double c = rounds * (rec * kt * (rounds < 2 || f == DC_SK64 ? 1.25 : 1.0) + (f == DC_SK64 ? 4500 : 2500) + wait);
            if (ks > 1) c += plane * (ks + 1) * 4 / 4e12 * 2.4e9 + 10000;
            if (c < best) {
                best = c;
                *form = f;
                *ks_out = ks;
            }
        }
    }
}

template <int PB, int KT, int EPI, bool FUSE, bool SK>
static void dc_launch(const DcIn &in, const uint8_t *w, const DcOut &o, const DcGeo &g, const DcFuse &fz, hipStream_t s)
{
    const int rows = (SK ? 16 : 64) * PB + (KT - 1) * in.dil;
    int lds = (SK ? 4 : 1) * 2 * rows * 128;
    if (SK) lds = std::max(lds, 4 * PB * DC_CB * 1024);
    hipLaunchKernelGGL((k_dconv<DC_CB, PB, KT, EPI, FUSE, SK>), dim3((unsigned)(g.tm * g.tn * g.nph * g.ks)), dim3(256), lds,
                       s, in, w, o, g, fz);
}

template <int KT, int EPI, bool FUSE>
static void dc_launch_form(int form, const DcIn &in, const uint8_t *w, const DcOut &o, const DcGeo &g, const DcFuse &fz,
                           hipStream_t s)
{
    if (form == DC_SK64) {
        dc_launch<4, KT, EPI, FUSE, true>(in, w, o, g, fz, s);
        return;
    }
    if constexpr (!FUSE) {
        if (form == DC_P256) {
            dc_launch<4, KT, EPI, FUSE, false>(in, w, o, g, fz, s);
            return;
        }
    }
    dc_launch<2, KT, EPI, FUSE, false>(in, w, o, g, fz, s);
}

template <int KT, int EPI>
static hipError_t dconv(const DcIn &in, const uint8_t *w, DcOut o, int nph, const DecoderWs &ws, RangeLog &log,
                        hipStream_t s, DcFuse *fz = nullptr, bool *fused = nullptr)
{
    int form = 0, ks = 1;
    DcGeo g{};
    g.tm = o.M / (16 * DC_CB);
    g.nph = nph;
    // one channel tile holds all of a fused conv2's input
    const bool fuse = KT == 7 && fz && g.tm == 1;
    dc_plan(in.L, g.tm, nph, in.nc, KT, o.M, ws.part_cap, fuse, &form, &ks);
    g.tn = (in.L + (256 >> form) - 1) / (256 >> form);
    g.cps = (in.nc + ks - 1) / ks;
    g.ks = ks;
    g.part = ws.part;
    if constexpr (KT == 7) {
        if (fuse && ks == 1) {
            *fused = true;
            const int per = form == DC_SK64 ? 4 : 2;
            o.rm = range_take(log, 4 * (size_t)g.tn, per);
            if (fz->o.ys) fz->o.rm = range_take(log, 4 * (size_t)g.tn, per);
            if (log.full) return hipErrorInvalidValue;
            dc_launch_form<KT, EPI, true>(form, in, w, o, g, *fz, s);
            return hipGetLastError();
        }
    }
    // a word a wave; with a stride one per 16 positions
    const int64_t rows = (int64_t)in.L * nph, n = rows * (o.M / 8);
    if (o.ys && ks > 1) o.rm = range_take(log, (size_t)(n + 255) / 256 * 4, o.M / 8);
    else if (o.ys && o.os > 1) o.rm = range_take(log, (size_t)g.tn * (16 >> form) * g.tm * nph, g.tm * nph);
    else if (o.ys) o.rm = range_take(log, 4 * (size_t)g.tn * g.tm, g.tm << form);
    if (log.full) return hipErrorInvalidValue;
    dc_launch_form<KT, EPI, false>(form, in, w, o, g, DcFuse{}, s);
    VCHK(hipGetLastError());
    if (ks > 1) {
        hipLaunchKernelGGL(k_dconv_reduce<EPI>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ws.part, ks, rows, nph, o);
    }
    return hipGetLastError();
}

// A linear layer over split rows into slice sums: 64-channel tiles, slices of
// one to a few records a wave, as many as give about two workgroups a CU.
static hipError_t linear(const uint8_t *x, int nc, int rows, const DecLin &w, int M, const float *bias, const DecoderWs &ws,
                         LinSum *out, hipStream_t s)
{
    DcGeo g{};
    g.tm = M / (16 * DC_LIN_CB);
    g.tn = (rows + 63) / 64;
    g.nph = 1;
    int ks = std::max(1, std::min({nc / 4, 16, 512 / std::max(1, g.tm * g.tn)}));
    while (ks > 1 && (size_t)ks * rows * M > ws.part_cap) ks--;
    g.cps = (nc + ks - 1) / ks;
    g.ks = (nc + g.cps - 1) / g.cps;
    g.part = ws.part;
    if ((size_t)g.ks * rows * M > ws.part_cap) return hipErrorInvalidValue;
    DcOut o{};
    o.M = M;
    o.os = 1;
    const int lds = std::max(4 * 2 * 64 * 128, 4 * 4 * DC_LIN_CB * 1024);
    hipLaunchKernelGGL((k_dconv<DC_LIN_CB, 4, 1, DC_RAW, false, true>), dim3((unsigned)(g.tm * g.tn * g.ks)), dim3(256), lds,
                       s, DcIn{x, nc, rows, 1}, w.w, o, g, DcFuse{});
    *out = LinSum{ws.part, w.un, bias, g.ks, rows, M};
    return hipGetLastError();
}

// the instance of a consumer of slice sums for p.ks slices
#define LIN_BY_KS(KERNEL, GRID, ...)                                                             \
    do {                                                                                         \
        switch (p.ks) {                                                                          \
        case 1: hipLaunchKernelGGL((KERNEL(1)), GRID, dim3(256), 0, s, __VA_ARGS__); break;      \
        case 2: hipLaunchKernelGGL((KERNEL(2)), GRID, dim3(256), 0, s, __VA_ARGS__); break;      \
        case 4: hipLaunchKernelGGL((KERNEL(4)), GRID, dim3(256), 0, s, __VA_ARGS__); break;      \
        case 8: hipLaunchKernelGGL((KERNEL(8)), GRID, dim3(256), 0, s, __VA_ARGS__); break;      \
        default: hipLaunchKernelGGL((KERNEL(0)), GRID, dim3(256), 0, s, __VA_ARGS__); break;     \
        }                                                                                        \
        VCHK(hipGetLastError());                                                                 \
    } while (0)
#define K_ROWS(KS) k_lin_rows<KS>
#define K_CF(KS) k_lin_cf<KS>
#define K_SWIGLU(KS) k_lin_swiglu<KS>
#define K_RMS1(KS) k_lin_resid_rms<1, KS>
#define K_RMS4(KS) k_lin_resid_rms<4, KS>

static hipError_t resid_rms(const LinSum &p, const float *scale, float *x, const float *gamma, uint8_t *ys, RangeLog &log,
                            hipStream_t s)
{
    const dim3 grid((p.rows + 3) / 4);
    float *rm = range_take(log, 4 * (size_t)grid.x, 64);
    if (log.full) return hipErrorInvalidValue;
    if (p.M <= 512) LIN_BY_KS(K_RMS1, grid, p, scale, x, gamma, ys, rm);
    else LIN_BY_KS(K_RMS4, grid, p, scale, x, gamma, ys, rm);
    return hipSuccess;
}

// The transformer over T positions: in [latent][T] channel-first f32 to out
// likewise.  bufs: four buffers of the workspace other than those two.
hipError_t enqueue_dec_tf(const DecoderDev &d, const DecoderWs &ws, const float *in, float *out, float *const bufs[4], int T,
                          RangeLog &log, hipStream_t s)
{
    const int H = d.hidden, A = d.n_heads * d.head_dim, I = d.inter, LAT = d.latent;
    uint8_t *xs = (uint8_t *)bufs[0], *hs = (uint8_t *)bufs[1];
    float *x = bufs[2], *qkv = bufs[3];
    LinSum p{};
    float *rm = range_take(log, (size_t)((T + 63) / 64) * (LAT / 8), LAT / 8);
    if (log.full) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_cf_split, dim3((T + 63) / 64, LAT / 32), dim3(256), 0, s, in, LAT, T, hs, rm);
    VCHK(hipGetLastError());
    VCHK(linear(hs, LAT / 32, T, d.tf_in, H, d.tf_in_b, ws, &p, s));
    VCHK(resid_rms(p, nullptr, x, d.tf[0].in_norm, xs, log, s));
    for (int l = 0; l < d.n_tf; l++) {
        const DecLayer &L = d.tf[l];
        VCHK(linear(xs, H / 32, T, L.pqkv, 3 * A, nullptr, ws, &p, s));
        LIN_BY_KS(K_ROWS, dim3((unsigned)(((int64_t)T * 3 * A / 4 + 255) / 256)), p, qkv);
        // its blocks of 16 positions: four waves a head
        rm = range_take(log, (size_t)((T + 15) / 16) * d.n_heads * 4, 16 * d.n_heads);
        if (log.full) return hipErrorInvalidValue;
        VCHK(enqueue_dec_attn_rows(d, qkv, T, hs, rm, s));
        VCHK(linear(hs, A / 32, T, L.po, H, nullptr, ws, &p, s));
        VCHK(resid_rms(p, L.attn_scale, x, L.post_norm, xs, log, s));
        VCHK(linear(xs, H / 32, T, L.pgu, 2 * I, nullptr, ws, &p, s));
        const dim3 sg((unsigned)(((int64_t)T * I / 8 + 255) / 256));
        rm = range_take(log, 4 * (size_t)sg.x, I / 8);
        if (log.full) return hipErrorInvalidValue;
        LIN_BY_KS(K_SWIGLU, sg, p, hs, rm);
        VCHK(linear(hs, I / 32, T, L.pdown, H, nullptr, ws, &p, s));
        VCHK(resid_rms(p, L.mlp_scale, x, l + 1 < d.n_tf ? d.tf[l + 1].in_norm : d.tf_norm, xs, log, s));
    }
    VCHK(linear(xs, H / 32, T, d.tf_out, LAT, d.tf_out_b, ws, &p, s));
    LIN_BY_KS(K_CF, dim3((T + 63) / 64, LAT / 32), p, out);
    return hipSuccess;
}

// Whether enqueue_dec_tf runs a decoder's shapes (its slice sums within
// part_floats are checked per call).  It was the faster one at every length
// timed (1 to 400 frames: 11% to 1% of the decode), so no length limits it;
// the shapes are what its tiles need: whole 64-channel tiles, whole records,
// heads of the tiled attention's 64, and a row of at most 2048 in a wave's
// registers.
bool dec_tf_fits(const DecoderDev &d)
{
    const int A = d.n_heads * d.head_dim;
    return !d.weights_f32 && d.n_tf > 0 && d.hidden <= 2048 && d.hidden % 64 == 0 && A % 64 == 0 && d.inter % 32 == 0 &&
           d.latent % 64 == 0 && d.head_dim == 64 && dec_attn_tiled(d);
}

// The most positions whose slice sums fit part_floats.
int dec_tf_rows(const DecoderDev &d, size_t part_floats)
{
    const int widest = std::max({3 * d.n_heads * d.head_dim, 2 * d.inter, d.latent, d.hidden});
    return (int)std::min<size_t>(part_floats / widest, 1 << 20);
}

// The Vocos stages and the output conv from the upsamplers' signal sig
// [voc_init.ic][L] (channel-first f32).  bufs: four buffers of the workspace
// other than sig's.
hipError_t enqueue_vocos(const DecoderDev &d, const DecoderWs &ws, const float *sig, float *const bufs[4], int L, int64_t cut,
                         float *audio, bool fuse, RangeLog &log, int32_t *out_of_range, hipStream_t s)
{
    uint8_t *sn = (uint8_t *)bufs[0], *t1 = (uint8_t *)bufs[1];
    float *x = bufs[2], *last = bufs[3];
    const int ic = d.voc_init.ic;
    float *rm = range_take(log, (size_t)((L + 63) / 64) * (ic / 8), ic / 8);
    if (log.full) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_cf_split, dim3((L + 63) / 64, ic / 32), dim3(256), 0, s, sig, ic, L, t1, rm);
    VCHK(hipGetLastError());
    // the snake that follows residual r of block b: the next residual's, the
    // next block's, or the last one, whose f32 rows the output conv reads
    const auto next = [&](int b, int r, DcOut *o) {
        const bool in_block = b >= 0 && r + 1 < d.voc[b].n_res;
        const bool end = !in_block && b + 1 >= d.n_voc;
        o->snake = in_block ? d.voc[b].res[r + 1].a1_par : (end ? d.final_par : d.voc[b + 1].pre_par);
        o->yf = end ? last : nullptr;
        o->ys = end ? nullptr : o->ys;
    };
    DcOut o{};
    o.ys = sn;
    o.M = d.voc_init.oc;
    o.os = 1;
    o.bias = d.voc_init.b;
    o.un = d.voc_init.un;
    next(-1, 0, &o);
    VCHK((dconv<7, DC_SNAKE>(DcIn{t1, ic / 32, L, d.voc_init.dil}, d.voc_init.pw, o, 1, ws, log, s)));
    for (int b = 0; b < d.n_voc; b++) {
        const DecVocos &B = d.voc[b];
        DcOut u{};
        u.ys = t1;
        u.x = x;
        u.M = B.up.oc;
        u.os = B.up.stride;
        u.bias = B.up.b;
        u.un = B.up.un;
        next(b, -1, &u);
        const DcIn ui{sn, B.up.ic / 32, L, 1};
        if (B.up.taps == 2) VCHK((dconv<2, DC_X_SNAKE>(ui, B.up.pw, u, B.up.stride, ws, log, s)));
        else VCHK((dconv<1, DC_X_SNAKE>(ui, B.up.pw, u, B.up.stride, ws, log, s)));
        L *= B.up.stride;
        std::swap(sn, t1);
        for (int r = 0; r < B.n_res; r++) {
            const DecVocosRes &R = B.res[r];
            DcOut c1{};
            c1.ys = t1;
            c1.M = B.up.oc;
            c1.os = 1;
            c1.bias = R.c1.b;
            c1.un = R.c1.un;
            c1.snake = R.a2_par;
            DcOut c2 = c1;
            c2.ys = sn;
            c2.x = x;
            c2.res = x;
            c2.bias = R.c2.b;
            c2.un = R.c2.un;
            next(b, r, &c2);
            DcFuse fz{R.c2.pw, c2};
            if (fz.o.ys) fz.o.ys = t1;    // neighbouring tiles still read sn
            bool fused = false;
            const DcIn ci{sn, B.up.oc / 32, L, R.c1.dil};
            VCHK((dconv<7, DC_SNAKE>(ci, R.c1.pw, c1, 1, ws, log, s, fuse ? &fz : nullptr, &fused)));
            if (fused) {
                std::swap(sn, t1);
                continue;
            }
            VCHK((dconv<1, DC_X_SNAKE>(DcIn{t1, B.up.oc / 32, L, 1}, R.c2.pw, c2, 1, ws, log, s)));
        }
    }
    const int ch = d.n_voc ? d.voc[d.n_voc - 1].up.oc : d.voc_init.oc;
    const size_t lds = (size_t)(((d.out_k * ch + 3) & ~3) + (64 + (d.out_k - 1) * d.out_dil) * (ch + 4)) * sizeof(float);
    RangeList l{};
    const int nout = (L + 63) / 64, nr = out_of_range ? range_list(log, 0, &l) : 0;
    hipLaunchKernelGGL(k_out_rows<7>, dim3(nout + nr), dim3(256), lds, s, last, ch, L, d.out_w, d.out_b, d.out_dil, cut, audio,
                       nout, ws.range_flag, l, out_of_range);
    VCHK(hipGetLastError());
    if (!out_of_range || log.sig.size() <= RANGE_SIGNALS) return hipSuccess;
    return enqueue_range_result(log, RANGE_SIGNALS, ws.range_flag, out_of_range, s);
}

// Whether enqueue_vocos runs a decoder's shapes.
bool vocos_fits(const DecoderDev &d)
{
    if (d.weights_f32 || !dconv_fits(d.voc_init.oc, d.voc_init.ic, d.voc_init.k, d.voc_init.dil) || d.voc_init.k != 7)
        return false;
    int ch = d.voc_init.oc;
    for (int b = 0; b < d.n_voc; b++) {
        const DecVocos &B = d.voc[b];
        if (!dconv_fits(B.up.oc, B.up.ic, B.up.taps, 1)) return false;
        ch = B.up.oc;
        for (int r = 0; r < B.n_res; r++) {
            const DecVocosRes &R = B.res[r];
            if (R.c1.k != 7 || !dconv_fits(ch, ch, 7, R.c1.dil) || R.c2.k != 1) return false;
        }
    }
    // the output conv's tile in 64 KB of LDS
    return d.out_k == 7 && (size_t)(7 * ch + (64 + 6 * d.out_dil) * (ch + 4)) * sizeof(float) <= 65536;
}

}  // namespace qtts
