// Batched prefill for gfx950: LlamaModel::forward (llama.rs:683-700) with its
// attention (llama.rs:162-266), run over n_seq sequences of seq tokens at once
// so every projection is one GEMM on the matrix cores.  The K/V rows of the
// processed positions are appended to each sequence's KV cache, so decode can
// continue from them.
//
// GEMM numerics.  The reference accumulates f64(a) * f64(q * scale) into f32
// in k order (cpu.rs:1128-1160).  Two forms of the activations here:
//  - int8 per-tensor weights (every projection of an int8 model): each row of
//    activations as 24-bit fixed point, x = X 2^-E with E per row and
//    |x - X 2^-E| <= 2^-23 max|row|, X in three balanced int8 digits; the int8
//    matrix cores sum d q exactly in i32, and the epilogue forms the exact
//    integer dot product and rounds X.q 2^-E scale to f32 once
//    (k_norm_digits, k_gemm_digits);
//  - block-32 weights and bf16 weights: each f32 activation as two bf16
//    values hi = bf16(x), lo = bf16(x - hi) (|x - hi - lo| <= 2^-17 |x|), two
//    bf16 MFMAs per product accumulated in f32 (one for bf16 weights: the
//    reference's bf16 cast), scaled per output or per 32-wide k block.
// The differences from the reference are the activation rounding and the
// summation order, far inside the 1e-3 logit bar.
//
// Data layout.  GEMM inputs are [Mp][ld] planes (three int8 digit planes, or
// the bf16 hi and lo planes): Mp = rows rounded up to the M tile, ld = k
// rounded up to the k step (64); the columns past k are zero.  RMSNorm writes
// its planes directly; the attention and SwiGLU outputs, whose rows no single
// workgroup holds whole, go through f32 rows and a per-row pass into digit
// planes (bf16 planes directly for the other weight types).  Weights are the
// GEMV stream layout (one row of kp bytes per output, byte = q + 128), read
// as they are by the int8 matrix cores, converted to bf16 for the bf16 ones.
#include <cmath>

#include "internal.h"
#include "kdev.h"

namespace scry {
namespace {

using namespace dev;

typedef unsigned short u16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define PF_LAUNCH_CHECK() SCRY_HIP(hipGetLastError()); return SCRY_OK

// hi = bf16(x), lo = bf16(x - hi) with the hardware round-to-nearest-even
// conversion: the bits of bf16_rn for every finite x (NaN stays NaN)
__device__ __forceinline__ void split_bf16(float x, u16 &hi, u16 &lo) {
    const __bf16 h = (__bf16)x;
    hi = __builtin_bit_cast(u16, h);
    lo = __builtin_bit_cast(u16, (__bf16)(x - (float)h));
}

// ------------------------------------------------------------------ RMSNorm
// cpu.rs:574-599 on the rows r*rstep + roff of x: rstd = 1/sqrt(mean(x^2)+eps)
// in f64, out = f32(x * rstd * w).  Writes the bf16 planes of row r (columns
// [k, ld) zeroed) and/or an f32 copy.
__global__ __launch_bounds__(256) void k_norm_split(const float *__restrict__ x, int ldx, int rstep, int roff,
                                                    const float *__restrict__ w, int k, float eps, u16 *hi,
                                                    u16 *lo, int ldp, int kpad, float *outf, int ldf) {
    __shared__ double red[4];
    const int r = blockIdx.x;
    const float *src = x + ((size_t)r * rstep + roff) * ldx;
    double ss = 0.0;
    for (int j = threadIdx.x; j < k; j += 256) ss += (double)src[j] * (double)src[j];
    const double rstd = 1.0 / sqrt(block_sum_d(ss, red) / (double)k + (double)eps);
    for (int j = threadIdx.x; j < kpad; j += 256) {
        const float v = j < k ? (float)((double)src[j] * rstd * (double)w[j]) : 0.f;
        if (hi) {
            u16 a, b;
            split_bf16(v, a, b);
            hi[(size_t)r * ldp + j] = a;
            lo[(size_t)r * ldp + j] = b;
        }
        if (outf && j < k) outf[(size_t)r * ldf + j] = v;
    }
}

// The same with 8 consecutive columns per thread and chunk, the row held in
// registers between the two passes, and 16-byte plane stores (k % 8 == 0,
// rows of x and w 16-byte aligned, planes only, NC = kpad / 2048 rounded up).
template <int NC>
__global__ __launch_bounds__(256) void k_norm_split8(const float *__restrict__ x, int ldx, int rstep, int roff,
                                                     const float *__restrict__ w, int k, float eps, u16 *hi,
                                                     u16 *lo, int ldp, int kpad) {
    __shared__ double red[4];
    const int r = blockIdx.x, t = threadIdx.x;
    const float *src = x + ((size_t)r * rstep + roff) * ldx;
    float4 v[NC][2];
    double ss = 0.0;
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int j = (c * 256 + t) * 8;
        v[c][0] = v[c][1] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (j < k) {
            v[c][0] = *(const float4 *)(src + j);
            v[c][1] = *(const float4 *)(src + j + 4);
        }
        const float e[8] = {v[c][0].x, v[c][0].y, v[c][0].z, v[c][0].w, v[c][1].x, v[c][1].y, v[c][1].z, v[c][1].w};
#pragma unroll
        for (int i = 0; i < 8; i++) ss += (double)e[i] * (double)e[i];
    }
    const double rstd = 1.0 / sqrt(block_sum_d(ss, red) / (double)k + (double)eps);
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int j = (c * 256 + t) * 8;
        if (j >= kpad) break;
        float4 w0 = make_float4(0.f, 0.f, 0.f, 0.f), w1 = w0;
        if (j < k) {
            w0 = *(const float4 *)(w + j);
            w1 = *(const float4 *)(w + j + 4);
        }
        const float e[8] = {v[c][0].x, v[c][0].y, v[c][0].z, v[c][0].w, v[c][1].x, v[c][1].y, v[c][1].z, v[c][1].w};
        const float g[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
        unsigned ph[4], pl[4];
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
            u16 a0, b0, a1, b1;
            split_bf16(j + i < k ? (float)((double)e[i] * rstd * (double)g[i]) : 0.f, a0, b0);
            split_bf16(j + i + 1 < k ? (float)((double)e[i + 1] * rstd * (double)g[i + 1]) : 0.f, a1, b1);
            ph[i / 2] = (unsigned)a0 | ((unsigned)a1 << 16);
            pl[i / 2] = (unsigned)b0 | ((unsigned)b1 << 16);
        }
        *(u32x4 *)(hi + (size_t)r * ldp + j) = u32x4{ph[0], ph[1], ph[2], ph[3]};
        *(u32x4 *)(lo + (size_t)r * ldp + j) = u32x4{pl[0], pl[1], pl[2], pl[3]};
    }
}

// RMSNorm into digit planes (the input of the int8 GEMM, k_gemm_digits):
// the same normalised row y as k_norm_split, then per row an exponent E with
// max|y| 2^E <= 2^23 - 2^16 - 1, X = rint(y 2^E) (exact scaling in f64, one
// rounding: |y - X 2^-E| <= 2^-E-1 <= 2^-23 max|y|), and X = d0 + 2^8 d1 +
// 2^16 d2 in balanced digits (d0, d1 in [-128, 127]; the bound keeps d2 in
// [-127, 127]).  A row holding a NaN or an infinity gets E = DG_NONFINITE
// and the GEMM writes NaN for it, as the split planes do (lo = bf16(inf - inf)).
// Thread t holds columns 8 (c 256 + t) .. +7 of chunk c; VEC: 16-byte loads
// (k % 8 == 0, rows 16-byte aligned).  NORM false: the rows as they are (y = x;
// w and eps unused), for GEMM inputs that no single kernel holds whole rows of.
constexpr int DG_NONFINITE = 0x7fffffff;
constexpr double DG_XMAX = 8323071.0;  // 2^23 - 2^16 - 1

template <int NC, bool VEC, bool NORM>
__global__ __launch_bounds__(256) void k_norm_digits(const float *__restrict__ x, int ldx, const float *__restrict__ w,
                                                     int k, float eps, signed char *dg, size_t dstride, int *de,
                                                     int ldp, int kpad) {
    __shared__ double red[4];
    __shared__ float s_max[4];
    __shared__ int s_bad[4];
    const int r = blockIdx.x, t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const float *src = x + (size_t)r * ldx;
    float y[NC][8];
    double ss = 0.0;
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int j = (c * 256 + t) * 8;
        if (VEC) {
            float4 v0 = make_float4(0.f, 0.f, 0.f, 0.f), v1 = v0;
            if (j < k) {
                v0 = *(const float4 *)(src + j);
                v1 = *(const float4 *)(src + j + 4);
            }
            y[c][0] = v0.x, y[c][1] = v0.y, y[c][2] = v0.z, y[c][3] = v0.w;
            y[c][4] = v1.x, y[c][5] = v1.y, y[c][6] = v1.z, y[c][7] = v1.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) y[c][i] = j + i < k ? src[j + i] : 0.f;
        }
        if (NORM) {
#pragma unroll
            for (int i = 0; i < 8; i++) ss += (double)y[c][i] * (double)y[c][i];
        }
    }
    const double rstd = NORM ? 1.0 / sqrt(block_sum_d(ss, red) / (double)k + (double)eps) : 1.0;
    float amax = 0.f;
    int bad = 0;
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int j = (c * 256 + t) * 8;
        float g[8];
        if (NORM && VEC) {
            float4 w0 = make_float4(0.f, 0.f, 0.f, 0.f), w1 = w0;
            if (j < k) {
                w0 = *(const float4 *)(w + j);
                w1 = *(const float4 *)(w + j + 4);
            }
            g[0] = w0.x, g[1] = w0.y, g[2] = w0.z, g[3] = w0.w, g[4] = w1.x, g[5] = w1.y, g[6] = w1.z, g[7] = w1.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) g[i] = NORM && j + i < k ? w[j + i] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float v = j + i >= k ? 0.f : NORM ? (float)((double)y[c][i] * rstd * (double)g[i]) : y[c][i];  // cpu.rs:574-599
            y[c][i] = v;
            amax = fmaxf(amax, fabsf(v));
            bad |= !isfinite(v);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        amax = fmaxf(amax, __shfl_xor(amax, off));
        bad |= __shfl_xor(bad, off);
    }
    if (lane == 0) s_max[wv] = amax, s_bad[wv] = bad;
    __syncthreads();
    amax = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
    bad = s_bad[0] | s_bad[1] | s_bad[2] | s_bad[3];
    int E = 0;
    if (bad) {
        E = DG_NONFINITE;
    } else if (amax > 0.f) {
        int ex;
        frexpf(amax, &ex);  // amax = m 2^ex, m in [0.5, 1)
        E = 23 - ex;
        if (ldexp((double)amax, E) > DG_XMAX) E--;
    }
    const int Es = bad ? 0 : E;
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int j = (c * 256 + t) * 8;
        if (j >= kpad) break;
        unsigned b[3][2] = {{0u, 0u}, {0u, 0u}, {0u, 0u}};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            // y 2^E is exact in f32 (a power-of-two scaling to at most 2^23), rint then exact
            const int X = bad ? 0 : (int)rintf(ldexpf(y[c][i], Es));
            // balanced digits: d0 = sext8(X), d1 = sext8(X1), d2 = X2 with X1 = (X - d0) / 2^8, X2 = (X1 - d1) / 2^8
            const int X1 = (X - (int)(signed char)X) >> 8;
            const int X2 = (X1 - (int)(signed char)X1) >> 8;
            const int sh = 8 * (i & 3);
            b[0][i >> 2] |= (unsigned)(X & 255) << sh;
            b[1][i >> 2] |= (unsigned)(X1 & 255) << sh;
            b[2][i >> 2] |= (unsigned)(X2 & 255) << sh;
        }
#pragma unroll
        for (int pl = 0; pl < 3; pl++)
            *(uint2 *)(dg + pl * dstride + (size_t)r * ldp + j) = make_uint2(b[pl][0], b[pl][1]);
    }
    if (t == 0) de[r] = E;
}

// f32 rows -> bf16 planes (columns [k, kpad) zeroed)
__global__ void k_split(const float *__restrict__ x, int ldx, int rows, int k, int kpad, u16 *hi, u16 *lo, int ldp) {
    const size_t total = (size_t)rows * kpad;
    for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (size_t)gridDim.x * blockDim.x) {
        const int r = (int)(g / kpad), j = (int)(g % kpad);
        u16 a = 0, b = 0;
        if (j < k) split_bf16(x[(size_t)r * ldx + j], a, b);
        hi[(size_t)r * ldp + j] = a;
        lo[(size_t)r * ldp + j] = b;
    }
}

// ------------------------------------------------------------------ GEMM
// C[m][n] = sum_k (hi + lo)[m][k] * q[n][k], q the int8 weight of output n.
// Workgroup tile BM x BN, k step BK; 4 waves in 2 x 2, each 64 x 128 as 4 x 8
// tiles of v_mfma_f32_16x16x32_bf16.  Operand lane layouts of that
// instruction (16 x 32 A, 32 x 16 B, 16 x 16 D): lane l holds
// A[l % 16][8 (l / 16) + e] and B[8 (l / 16) + e][l % 16] for e = 0..7, and
// D[4 (l / 16) + r][l % 16] for r = 0..3.
// One LDS stage (the next k step is held in registers while the current one
// is consumed) keeps a workgroup at ~75 KB, so two fit on a CU: two waves per
// SIMD hide each other's LDS and barrier latency (measured: 45-48% of the
// bf16 issue rate, against 29-35% for a double-buffered stage at one wave
// per SIMD).
constexpr int BM = 128, BN = 256, BK = 64;
constexpr int LDT = BK + 8;  // LDS row stride in bf16 (144 B): 16-byte row reads hit distinct banks
constexpr int G_THREADS = 256;
constexpr size_t A_TILE = (size_t)BM * LDT, B_TILE = (size_t)BN * LDT;  // u16 elements
constexpr int AC = BM * BK / 8 / G_THREADS;   // 16-byte A chunks per thread and plane
// dynamic LDS: A hi, A lo, B + [BK/32][BN] block-32 scales
constexpr size_t GEMM_LDS = (2 * A_TILE + B_TILE) * sizeof(u16) + (BK / 32) * BN * sizeof(float);
static_assert(GEMM_LDS >= 2 * BM * (BN / 2 + 8) * sizeof(u16), "SwiGLU staging tile");

enum { GE_STORE = PF_STORE, GE_RESID = PF_RESID, GE_SWIGLU = PF_SWIGLU };

struct GemmP {
    const u16 *ahi, *alo;
    int lda;
    const uint8_t *w;
    int kp, N;
    const float *s32;  // block-32 scales [N][nb] (packed-row order) or null
    int nb;
    int M, nk;         // rows, k steps (k rounded up to 32, / 32)
    int n_mb, n_nb;    // tiles along M and N
    float scale, scale2;
    const float *bias;  // GE_STORE: + bias[n] (f32, after scaling)
    float *c;
    int ldc;
    u16 *ohi, *olo;
    int ldo, opad;     // SwiGLU planes: row stride, columns written (with zero pad)
    const signed char *ad;  // digit planes [3][.][lda] (k_gemm_digits), plane stride dstride bytes
    const int *ae;          // row exponents
    size_t dstride;
    float *of;              // SwiGLU output as f32 rows [M][ldo] instead of the planes (k_gemm_digits)
    int splits, kchunk;     // the smaller tiles: k splits of kchunk steps each
    double *part;           // splits > 1: sums [split][M][N]
    float *partf;           // the same for k_gemm_ring
};

// Workgroup -> tile: workgroup b runs on XCD b % 8.  Tiles are numbered by
// super-tiles of 4 M tiles x 8 N tiles (fewer at the last rows and columns) and
// an XCD works through whole runs of 32 of them, so the workgroups it runs
// together share A rows and weight rows in its L2.  Only real tiles are
// numbered: with 32 numbers for every super-tile, 2 row tiles x 112 column
// tiles took two rounds of the chip instead of one (130 x 4096 x 28672 150 ->
// 83 us, 640 x 4096 x 28672 300 -> 231).
__device__ __forceinline__ bool gemm_tile(const GemmP &p, int &mb, int &nb) {
    const int b = blockIdx.x, xcd = b & 7, loc = b >> 3;
    const int t = ((loc >> 5) * 8 + xcd) * 32 + (loc & 31);
    if (t >= p.n_mb * p.n_nb) return false;
    const int nb0 = t / (8 * p.n_mb) * 8, nw = min(8, p.n_nb - nb0);  // panel of column tiles
    const int in = t - nb0 * p.n_mb, mb0 = in / (4 * nw) * 4, mh = min(4, p.n_mb - mb0);
    const int r = in - mb0 * nw;
    mb = mb0 + r % mh;
    nb = nb0 + r / mh;
    return true;
}
int gemm_tile_grid(const GemmP &p) { return (p.n_mb * p.n_nb + 255) / 256 * 256; }

// 16 weight bytes (q + 128) -> 16 bf16 of q, as 8 words.  Flipping bit 7
// gives q's two's-complement byte; |q| <= 128 is exact in bf16
// (v_cvt_f32_i32 on the sign-extended byte, then v_cvt_pk_bf16_f32).
__device__ __forceinline__ void bytes_to_bf16(u32x4 v, u32x4 &o0, u32x4 &o1) {
    bf16x8 r0, r1;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        r0[j] = (__bf16)(float)(int)(signed char)((v.x ^ 0x80808080u) >> (8 * j));
        r0[4 + j] = (__bf16)(float)(int)(signed char)((v.y ^ 0x80808080u) >> (8 * j));
        r1[j] = (__bf16)(float)(int)(signed char)((v.z ^ 0x80808080u) >> (8 * j));
        r1[4 + j] = (__bf16)(float)(int)(signed char)((v.w ^ 0x80808080u) >> (8 * j));
    }
    o0 = __builtin_bit_cast(u32x4, r0);
    o1 = __builtin_bit_cast(u32x4, r1);
}

// GEMM epilogue for a wave's TM x TN tiles of 16 x 16, D[4 (l / 16) + r][l % 16]
// of each tile at rows mw + 16 tm, columns nw + 16 tn; s_a / s_b scale the
// gate / up halves (s_a alone otherwise).
// lane value of the lane l ^ 2 / l ^ 1 (quad permutes, no LDS traffic)
__device__ __forceinline__ float quad_xor2(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, false));
}
__device__ __forceinline__ int quad_xor1(int v) { return __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, false); }

// GEMM epilogue for a wave's TM x TN tiles of 16 x 16, D[4 (l / 16) + r][l % 16]
// of each tile at rows mw + 16 tm, columns nw + 16 tn; s_a / s_b scale the
// gate / up halves (s_a alone otherwise).
template <int EPI, int TM, int TN>
__device__ __forceinline__ void gemm_store(const GemmP &p, const f32x4 (&acc)[TM][TN], int mw, int nw, int lane,
                                           float s_a, float s_b) {
    const int fr = lane & 15;
#pragma unroll
    for (int tn = 0; tn < TN; tn++) {
        const int n = nw + tn * 16 + fr;
#pragma unroll
        for (int tm = 0; tm < TM; tm++) {
            if (EPI == GE_SWIGLU) {
                // fused gate/up rows of a group of 4: gate[2t], gate[2t+1],
                // up[2t], up[2t+1] in lanes 4q .. 4q+3.  Rows are taken in pairs
                // (r0, r1) so that every lane evaluates one SiLU: the gate lanes
                // form output row r0 (their gate, the up lane's r0 value), the up
                // lanes output row r1 (the gate lane's r1 value, their up); lanes
                // 4q and 4q+2 then store columns 2t, 2t+1 of their row as one
                // 32-bit word per plane
                const bool gate = (n & 2) == 0;
                const float sc = gate ? s_a : s_b;
#pragma unroll
                for (int rp = 0; rp < 2; rp++) {
                    const float v0 = acc[tm][tn][2 * rp] * sc, v1 = acc[tm][tn][2 * rp + 1] * sc;
                    const float recv = quad_xor2(gate ? v1 : v0);
                    const float gv = gate ? v0 : recv, uv = gate ? recv : v1;
                    u16 a, b;
                    split_bf16(silu_f(gv) * uv, a, b);  // cpu.rs:666-678
                    const unsigned hw = (unsigned)a | ((unsigned)quad_xor1((int)a) << 16);
                    const unsigned lw = (unsigned)b | ((unsigned)quad_xor1((int)b) << 16);
                    const int m = mw + tm * 16 + ((lane >> 4) << 2) + 2 * rp + (gate ? 0 : 1);
                    if ((n & 1) == 0 && m < p.M && n < p.N) {  // N is a multiple of 4
                        const size_t at = (size_t)m * p.ldo + ((n >> 2) << 1);
                        *(unsigned *)(p.ohi + at) = hw;
                        *(unsigned *)(p.olo + at) = lw;
                    }
                }
            }
        }
        if (EPI != GE_SWIGLU) {
            // this column's residual values (or bias) are all requested before the
            // first store: the compiler cannot tell the stores from later loads of
            // c apart, and would otherwise wait out one round trip per element
            const bool nok = n < p.N;
            const float bn = EPI == GE_STORE && p.bias && nok ? p.bias[n] : 0.f;  // cpu.rs:553-570
            float res[TM][4];
#pragma unroll
            for (int tm = 0; tm < TM; tm++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = mw + tm * 16 + ((lane >> 4) << 2) + r;
                    res[tm][r] = EPI == GE_RESID && nok && m < p.M ? p.c[(size_t)m * p.ldc + n] : 0.f;
                }
#pragma unroll
            for (int tm = 0; tm < TM; tm++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = mw + tm * 16 + ((lane >> 4) << 2) + r;
                    if (nok && m < p.M) {
                        const float v = acc[tm][tn][r] * s_a;
                        // cpu.rs:104-113 add
                        p.c[(size_t)m * p.ldc + n] = EPI == GE_RESID ? res[tm][r] + v : (EPI == GE_STORE && p.bias ? v + bn : v);
                    }
                }
        }
    }
}

// SwiGLU epilogue through LDS.  The MFMA layout leaves each lane one column
// of 4 rows, so direct plane stores are 4-byte pieces of 8 rows per
// instruction; instead each wave puts its outputs (one SiLU per lane and row
// pair, as in gemm_store) into an LDS tile [BM][BN / 2] per plane, and the
// workgroup then writes whole 256-byte plane rows with 16-byte stores.  The
// caller's LDS is free (no loads in flight, every wave past its last read);
// so (>= 2 BM (BN / 2 + 8) u16) holds the tile.  Rows past M are not written
// (they stay zero); columns past N / 2 neither.
// SiLU in f32 for outputs that become digit planes (each row to 2^-23 of
// its largest value) or split-bf16 planes (hi + lo hold x to 2^-17): the f32
// evaluation is within a few 2^-24 of the reference's f64 one
// (cpu.rs:1119-1122), so the planes agree with the f64 path's to their own
// bound, at a quarter of the cost.  Where the next GEMM reads
// one bf16 plane (the bf16 model: the reference's bf16 cast of the f32
// value), the f64 evaluation is kept, since one ulp of f32 can move a bf16
// rounding.
__device__ __forceinline__ float silu_split(float g) { return g / (1.f + expf(-g)); }

template <int TM, int TN, int NT, bool EXACT, int BM_ = BM, int BN_ = BN>
__device__ __forceinline__ void swiglu_store(const GemmP &p, const f32x4 (&acc)[TM][TN], u16 *so, int ml, int nl, int m0,
                                             int n0, int lane) {
    constexpr int OW = BN_ / 2, LDO = OW + 8;  // output columns per tile; LDS row stride (u16)
    constexpr int LDF = OW + 4;               // the same in f32 (p.of: f32 rows instead of planes)
    u16 *sh = so, *sl = so + BM_ * LDO;
    float *sf = reinterpret_cast<float *>(so);
    const int fr = lane & 15;
#pragma unroll
    for (int tn = 0; tn < TN; tn++) {
        const int n = nl + tn * 16 + fr;  // tile column (n0 is a multiple of 4)
        const bool gate = (n & 2) == 0;
        const float sc = gate ? p.scale : p.scale2;
#pragma unroll
        for (int tm = 0; tm < TM; tm++) {
#pragma unroll
            for (int rp = 0; rp < 2; rp++) {
                const float v0 = acc[tm][tn][2 * rp] * sc, v1 = acc[tm][tn][2 * rp + 1] * sc;
                const float recv = quad_xor2(gate ? v1 : v0);
                const float gv = gate ? v0 : recv, uv = gate ? recv : v1;
                const float o = (EXACT ? silu_f(gv) : silu_split(gv)) * uv;  // cpu.rs:666-678
                const int r = ml + tm * 16 + ((lane >> 4) << 2) + 2 * rp + (gate ? 0 : 1);
                if (p.of) {
                    const float po = __int_as_float(quad_xor1(__float_as_int(o)));
                    if ((n & 1) == 0) *(float2 *)(sf + r * LDF + ((n >> 2) << 1)) = make_float2(o, po);
                } else {
                    u16 a, b;
                    split_bf16(o, a, b);
                    const unsigned hw = (unsigned)a | ((unsigned)quad_xor1((int)a) << 16);
                    const unsigned lw = (unsigned)b | ((unsigned)quad_xor1((int)b) << 16);
                    if ((n & 1) == 0) {
                        const int at = r * LDO + ((n >> 2) << 1);
                        *(unsigned *)(sh + at) = hw;
                        *(unsigned *)(sl + at) = lw;
                    }
                }
            }
        }
    }
    __syncthreads();
    const int oc0 = n0 >> 1, ocn = p.N >> 1;
    if (p.of) {  // f32 rows: 4 columns per 16-byte store
        constexpr int CPF = OW / 4;
        for (int idx = threadIdx.x; idx < BM_ * CPF; idx += NT) {
            const int r = idx / CPF, c = idx - r * CPF;
            const int m = m0 + r, col = oc0 + c * 4;
            if (m >= p.M || col >= ocn) continue;
            const float *src = sf + r * LDF + c * 4;
            float *dst = p.of + (size_t)m * p.ldo + col;
            if (col + 4 <= ocn) {
                *(float4 *)dst = *(const float4 *)src;
            } else {
                for (int e = 0; e < ocn - col; e++) dst[e] = src[e];
            }
        }
        return;
    }
    constexpr int CPR = OW / 8;  // 16-byte chunks per row
    for (int idx = threadIdx.x; idx < 2 * BM_ * CPR; idx += NT) {
        const int pl = idx / (BM_ * CPR), rem = idx - pl * (BM_ * CPR), r = rem / CPR, c = rem - r * CPR;
        const int m = m0 + r, col = oc0 + c * 8;
        if (m >= p.M || col >= ocn) continue;
        const u16 *src = (pl ? sl : sh) + r * LDO + c * 8;
        u16 *dst = (pl ? p.olo : p.ohi) + (size_t)m * p.ldo + col;
        if (col + 8 <= ocn) {
            *(u32x4 *)dst = *(const u32x4 *)src;
        } else {
            for (int e = 0; e < ocn - col; e++) dst[e] = src[e];
        }
    }
}

// zero the plane columns past the SwiGLU output (k padding of the next GEMM),
// rows [m0, m0 + BM_); one wave of the last column tile
template <int BM_>
__device__ __forceinline__ void swiglu_pad(const GemmP &p, int m0, int lane) {
    const int c0 = p.N >> 1;
    for (int idx = lane; idx < BM_ * (p.opad - c0); idx += 64) {
        const int m = m0 + idx / (p.opad - c0), col = c0 + idx % (p.opad - c0);
        p.ohi[(size_t)m * p.ldo + col] = 0;
        p.olo[(size_t)m * p.ldo + col] = 0;
    }
}

// (block-32: the per-block scaling needs a second accumulator tile, so one
// workgroup per CU keeps it in registers)
// WBF: bf16 weight rows [N][kp] (2 bytes each, copied to LDS as they are) and
// a single bf16 activation plane (bf16 mode: both operands rounded to bf16,
// products exact, f32 accumulation); p.alo is not read.
template <int EPI, bool B32, bool WBF = false>
__global__ __launch_bounds__(G_THREADS, B32 ? 1 : 2) void k_gemm(GemmP p) {
    static_assert(!(WBF && B32), "bf16 weights carry no block scales");
    extern __shared__ float4 gsm[];
    u16 *sa = reinterpret_cast<u16 *>(gsm);
    u16 *sb = sa + 2 * A_TILE;
    float *s_sc = reinterpret_cast<float *>(sb + B_TILE);  // [BK/32][BN]
    int mb, nbk;
    if (!gemm_tile(p, mb, nbk)) return;
    const int m0 = mb * BM, n0 = nbk * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;

    // global -> LDS assignment: A chunk c = tid + 256 i (row c / (BK/8), 8 bf16
    // at 8 (c % (BK/8))); B chunk c = tid + 256 i (row c / (BK/16), 16 bytes at
    // 16 (c % (BK/16)))
    constexpr int CPR = BK / 8, BPR = WBF ? BK / 8 : BK / 16;  // 16-byte chunks per row
    constexpr int BCW = BN * BPR / G_THREADS;                    // weight chunks per thread
    constexpr int NPL = WBF ? 1 : 2;                             // activation planes
    constexpr unsigned WB = WBF ? 2 : 1;                         // bytes per weight
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(p.w, (size_t)p.N * p.kp * WB);
    const u16 *ga[2][AC];
    unsigned boff[BCW];
#pragma unroll
    for (int i = 0; i < AC; i++) {
        const int c = tid + 256 * i;
        ga[0][i] = p.ahi + (size_t)(m0 + c / CPR) * p.lda + (c % CPR) * 8;
        ga[1][i] = WBF ? ga[0][i] : p.alo + (size_t)(m0 + c / CPR) * p.lda + (c % CPR) * 8;
    }
#pragma unroll
    for (int i = 0; i < BCW; i++) {
        const int c = tid + 256 * i;
        const int n = n0 + c / BPR;
        boff[i] = n < p.N ? (unsigned)((size_t)n * p.kp * WB + (c % BPR) * 16) : 0x80000000u;
    }
    const bool s_ld = B32 && n0 + tid < p.N;
    const __amdgpu_buffer_rsrc_t sr = make_rsrc(p.s32, B32 ? (size_t)p.N * p.nb * sizeof(float) : 0);

    u32x4 ra[2][AC], rb[BCW];
    float rs[BK / 32];
    auto gload = [&](int kt) {
        const int k0 = kt * BK;
#pragma unroll
        for (int pl = 0; pl < NPL; pl++)
#pragma unroll
            for (int i = 0; i < AC; i++) ra[pl][i] = *(const u32x4 *)(ga[pl][i] + k0);
#pragma unroll
        for (int i = 0; i < BCW; i++) rb[i] = bload16(wr, boff[i] + (unsigned)k0 * WB);
        if (B32) {
#pragma unroll
            for (int j = 0; j < BK / 32; j++)  // blocks past the scales read as 0 (their A is 0)
                rs[j] = s_ld ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                             sr, (int)(((n0 + tid) * p.nb + kt * (BK / 32) + j) * 4), 0, 0))
                             : 0.f;
        }
    };
    auto lstore = [&]() {
#pragma unroll
        for (int pl = 0; pl < NPL; pl++)
#pragma unroll
            for (int i = 0; i < AC; i++) {
                const int c = tid + 256 * i;
                *(u32x4 *)(sa + pl * A_TILE + (c / CPR) * LDT + (c % CPR) * 8) = ra[pl][i];
            }
#pragma unroll
        for (int i = 0; i < BCW; i++) {
            const int c = tid + 256 * i;
            if constexpr (WBF) {
                *(u32x4 *)(sb + (c / BPR) * LDT + (c % BPR) * 8) = rb[i];
            } else {
                u32x4 o0, o1;
                bytes_to_bf16(rb[i], o0, o1);
                u16 *d = sb + (c / BPR) * LDT + (c % BPR) * 16;
                *(u32x4 *)d = o0;
                *(u32x4 *)(d + 8) = o1;
            }
        }
        if (B32) {
#pragma unroll
            for (int j = 0; j < BK / 32; j++) s_sc[j * BN + tid] = rs[j];
        }
    };

    f32x4 acc[4][8];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    gload(0);
    lstore();
    __syncthreads();
    const int fr = lane & 15, fk = (lane >> 4) << 3;
    for (int kt = 0; kt < p.nk; kt++) {
        if (kt + 1 < p.nk) gload(kt + 1);  // in flight while this step is consumed
#pragma unroll
        for (int ks = 0; ks < BK / 32; ks++) {
            bf16x8 ah[4], al[4];
#pragma unroll
            for (int tm = 0; tm < 4; tm++) {
                const int r = wm * 64 + tm * 16 + fr;
                ah[tm] = *(const bf16x8 *)(sa + r * LDT + ks * 32 + fk);
                if (!WBF) al[tm] = *(const bf16x8 *)(sa + A_TILE + r * LDT + ks * 32 + fk);
            }
#pragma unroll
            for (int tn = 0; tn < 8; tn++) {
                const int cn = wn * 128 + tn * 16 + fr;
                const bf16x8 bv = *(const bf16x8 *)(sb + cn * LDT + ks * 32 + fk);
                if (B32) {
                    const float sc = s_sc[ks * BN + cn];
#pragma unroll
                    for (int tm = 0; tm < 4; tm++) {
                        f32x4 t = f32x4{0.f, 0.f, 0.f, 0.f};
                        t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[tm], bv, t, 0, 0, 0);
                        t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[tm], bv, t, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[tm][tn][r] = fmaf(sc, t[r], acc[tm][tn][r]);
                    }
                } else {
#pragma unroll
                    for (int tm = 0; tm < 4; tm++) {
                        acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[tm], bv, acc[tm][tn], 0, 0, 0);
                        if (!WBF)
                            acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[tm], bv, acc[tm][tn], 0, 0, 0);
                    }
                }
            }
        }
        if (kt + 1 < p.nk) {
            __syncthreads();  // every wave is done with this step's LDS
            lstore();
        }
        __syncthreads();
    }

    // ---- epilogue: D[4 (l / 16) + r][l % 16] of each tile
    if (EPI == GE_SWIGLU && !B32) {  // (the last k step ended with a barrier: LDS is free)
        swiglu_store<4, 8, G_THREADS, WBF>(p, acc, sa, wm * 64, wn * 128, m0, n0, lane);
        if (wave == 0 && nbk == p.n_nb - 1) swiglu_pad<BM>(p, m0, lane);
    } else {
        gemm_store<EPI, 4, 8>(p, acc, m0 + wm * 64, n0 + wn * 128, lane, B32 ? 1.f : p.scale, B32 ? 1.f : p.scale2);
        if (EPI == GE_SWIGLU && wave == 0 && nbk == p.n_nb - 1) swiglu_pad<BM>(p, m0, lane);
    }
}

// ------------------------------------------------------------------ GEMM, direct-to-LDS ring
// The int8 per-tensor GEMM (every projection of an int8 model).  Same tile
// (128 x 256), numerics and epilogues as k_gemm; the staging differs:
//  - activations and weights go from memory straight into LDS (buffer loads
//    with the LDS destination: M0 = the 1 KB block, lane i writes its 16 bytes
//    at 16 i), through a ring of 3 k steps, so two steps are in flight while
//    one is consumed and no register holds staged data;
//  - the weights stay int8 in LDS (half the bytes of bf16) and each wave
//    converts the 16 bytes it reads (two MFMA k halves) after the read;
//  - one barrier per k step: a step's slot is refilled only after every wave
//    has passed the barrier that follows its last read.
// 8 waves (2 along M x 4 along N) of 64 x 64 outputs; 144 KB of LDS, one
// workgroup per CU.  Measured on the config-5 shapes against k_gemm (same box,
// same run): qkv 811 -> 728 us, gate/up 3129 -> 3045 us, down 1754 -> 1594 us,
// and a higher clock under the power limit.
//
// LDS step layout: hi plane [128 rows][128 B], lo plane likewise, weights
// [256 columns][64 B].  16-byte chunks are XOR-swizzled so the MFMA operand
// reads (16 rows of one chunk per 16 lanes) hit distinct banks: activation
// chunk c of row r sits at c ^ (r & 7), weight chunk c of column n at
// c ^ ((n >> 1) & 3).  MFMA k order within a step: lane group g of the
// 16x16x32 MFMA holds k = 16 g + 8 h + e for k half h, e < 8, which makes
// the weight operand of both halves one 16-byte read per lane.
// WBF: bf16 weight rows (128 B per column and step, read as they are) and one
// activation plane (the bf16 model); else int8 weights and hi, lo planes.
// The bf16 model's short prompts and the op-level bf16 matmul also take
// smaller tiles and k splits (pick_tile, pick_cut): with 128 x 256, 37 rows x 4096
// columns are 16 workgroups.  Without splits a tile changes no bit (the k
// order is the same); a split's f32 sums are added in split order.
// B32: int8 weights with block-32 scales: the two scales a step has per column
// ride in the stage, and a half step's products (one block) are scaled into
// the sums.
template <bool WBF, bool B32, int BM_, int BN_, int WGM_, int WGN_, int S_>
struct RTile {
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, S = S_;
    static constexpr int TM = BM / WGM / 16, TN = BN / WGN / 16, NW = WGM * WGN, T = 64 * NW;
    static constexpr int NPL = WBF ? 1 : 2, WB = WBF ? 2 : 1;  // activation planes; bytes per weight
    static constexpr int A_PL = BM * BK * 2, B_ST = BN * BK * WB, SC = NPL * A_PL + B_ST;
    static constexpr int STAGE = SC + (B32 ? 2 * BN * 4 : 0);  // scales [2][BN]
    static constexpr int JA = A_PL / 1024 / NW, JB = B_ST / 1024 / NW;  // 1 KB loads per wave and step
    static constexpr int L = NPL * JA + JB + (B32 ? 1 : 0);
    static_assert(!B32 || (!WBF && 2 * (BN / 64) <= NW), "one 64-column scale load per wave");
    static constexpr size_t LDS = (size_t)S * STAGE;
    static constexpr bool BIG = BM_ == 128 && BN_ == 256;  // the super-tile map, no k splits
    static_assert(WGM * TM * 16 == BM && WGN * TN * 16 == BN && BK == 64, "ring tile");
    static_assert((A_PL / 1024) % NW == 0 && (B_ST / 1024) % NW == 0, "ring units");
    static_assert(L * (S - 2) < 64, "vmcnt range");
    static_assert(LDS >= 2 * BM * (BN / 2 + 8) * sizeof(u16), "SwiGLU staging tile");
};
template <bool WBF, bool B32>
using RBig = RTile<WBF, B32, BM, BN, 2, 4, 3>;

// buffer descriptor words (base, stride 0, num_records, raw-buffer flags),
// wave-uniform
__device__ __forceinline__ u32x4 ring_desc(const void *base, size_t bytes) {
    const uint64_t b = (uint64_t)(uintptr_t)base;
    const unsigned n = bytes > 0x7fffffffu ? 0x7fffffffu : (unsigned)bytes;
    u32x4 d = u32x4{(unsigned)b, (unsigned)(b >> 32) & 0xffffu, n, 0x00020000u};
#pragma unroll
    for (int i = 0; i < 4; i++) d[i] = __builtin_amdgcn_readfirstlane(d[i]);
    return d;
}

// 64 lanes x 16 bytes of buffer d at voff + soff -> LDS [lds, lds + 1024).
// The compiler does not see this load: callers wait with ring_wait before
// reading the LDS it fills (a vmcnt wait it cannot misplace), and M0 is
// restored.  Every lane's address stays inside the buffer's records or reads
// zero; no load is out of bounds for every lane (those can complete out of
// order and break partial vmcnt waits).
__device__ __forceinline__ void ring_load(u32x4 d, unsigned lds, unsigned voff, unsigned soff) {
    unsigned saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %2, %3, %4 offen lds\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "s"(lds), "v"(voff), "s"(d), "s"(soff)
        : "memory");
}
// 64 lanes x 4 bytes of buffer d -> LDS [lds, lds + 256), as ring_load
__device__ __forceinline__ void ring_load4(u32x4 d, unsigned lds, unsigned voff, unsigned soff) {
    unsigned saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "buffer_load_dword %2, %3, %4 offen lds\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "s"(lds), "v"(voff), "s"(d), "s"(soff)
        : "memory");
}
template <int N>
__device__ __forceinline__ void ring_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// workgroup barrier without a memory fence (a fence would also wait for the
// ring's loads); LDS reads and writes of this wave complete first
__device__ __forceinline__ void ring_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Workgroup -> (tile, k split) of the smaller tiles: XCD b % 8 walks a
// contiguous run, row tiles fastest, so the row tiles of one weight panel
// share an L2 (the super-tile map would leave XCDs without work here).
__device__ __forceinline__ bool small_tile(const GemmP &p, int &mb, int &nb, int &sp) {
    const unsigned total = (unsigned)p.n_mb * p.n_nb * p.splits, per = (total + 7) / 8;
    const unsigned w = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || w >= total) return false;
    mb = (int)(w % p.n_mb);
    nb = (int)(w / p.n_mb % p.n_nb);
    sp = (int)(w / ((unsigned)p.n_mb * p.n_nb));
    return true;
}

template <int EPI, bool WBF, bool B32, class C>
__global__ __launch_bounds__(C::T, C::BIG ? 1 : 2) void k_gemm_ring(GemmP p) {
    constexpr int A_PL = C::A_PL, STAGE = C::STAGE, JA = C::JA, L = C::L, NPL = C::NPL, WB = C::WB, S = C::S;
    constexpr int TM = C::TM, TN = C::TN, NW = C::NW, T = C::T, WGN = C::WGN;
    extern __shared__ float4 rsm[];
    unsigned char *sm = reinterpret_cast<unsigned char *>(rsm);
    int mb, nbk, sp = 0;
    if (C::BIG ? !gemm_tile(p, mb, nbk) : !small_tile(p, mb, nbk, sp)) return;
    const int m0 = mb * C::BM, n0 = nbk * C::BN;
    // this split's k steps
    const int kt0 = C::BIG ? 0 : sp * p.kchunk, kt1 = C::BIG ? p.nk : min(p.nk, kt0 + p.kchunk);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const size_t a_bytes = (size_t)p.n_mb * C::BM * p.lda * 2;
    const u32x4 dh = ring_desc(p.ahi, a_bytes), dl = ring_desc(WBF ? p.ahi : p.alo, a_bytes);
    const u32x4 dw = ring_desc(p.w, (size_t)p.N * p.kp * WB);
    const u32x4 dsc = ring_desc(B32 ? (const void *)p.s32 : p.w, B32 ? (size_t)p.N * p.nb * 4 : 4);
    const unsigned sm0 = (unsigned)(uintptr_t)sm;  // LDS address (low half of the flat address)
    // B32: this wave's scale load fills block sc_h of 64 columns (waves past
    // the last load the same again)
    constexpr int SG = C::BN >= 64 ? C::BN / 64 : 1;
    const int sc_u = wave % (2 * SG), sc_h = sc_u / SG;
    const unsigned sc_lds = (unsigned)(C::SC + (sc_h * C::BN + (sc_u % SG) * 64) * 4);
    const unsigned sc_voff = B32 ? (unsigned)(min(n0 + (sc_u % SG) * 64 + lane, p.N - 1) * p.nb * 4) : 0u;
    // load j of this wave fills 1 KB block u = j NW + wave: j < JA the hi plane
    // (8 rows of 128 B), j < 2 JA the lo plane, else the weights (int8: 16
    // columns of 64 B; bf16: 8 columns of 128 B)
    constexpr int LT = L - (B32 ? 1 : 0);  // loads of the tile
    unsigned voff[LT], loff[LT];
#pragma unroll
    for (int j = 0; j < LT; j++) {
        if (j < NPL * JA) {
            const int pl = j / JA, ua = (j % JA) * NW + wave;
            const int r = 8 * ua + (lane >> 3), c = (lane & 7) ^ (r & 7);
            voff[j] = (unsigned)((m0 + r) * p.lda * 2 + c * 16);
            loff[j] = (unsigned)(pl * A_PL + ua * 1024);
        } else if (WBF) {
            const int ub = (j - NPL * JA) * NW + wave;
            const int n = 8 * ub + (lane >> 3), c = (lane & 7) ^ (n & 7);
            const int row = min(n0 + n, p.N - 1);  // columns past N re-read row N - 1 (never stored)
            voff[j] = (unsigned)(row * p.kp * 2 + c * 16);
            loff[j] = (unsigned)(NPL * A_PL + ub * 1024);
        } else {
            const int ub = (j - NPL * JA) * NW + wave;
            const int n = 16 * ub + (lane >> 2), c = (lane & 3) ^ ((n >> 1) & 3);
            const int row = min(n0 + n, p.N - 1);  // columns past N re-read row N - 1 (never stored)
            voff[j] = (unsigned)(row * p.kp + c * 16);
            loff[j] = (unsigned)(NPL * A_PL + ub * 1024);
        }
    }
    // step kt into ring slot; steps past the last re-read the last (in bounds, never used)
    auto issue = [&](int kt, int slot) {
        const int ks = min(kt, kt1 - 1);
        const unsigned base = sm0 + (unsigned)(slot * STAGE);
        if (B32) ring_load4(dsc, base + sc_lds, sc_voff, (unsigned)(min(2 * ks + sc_h, p.nb - 1) * 4));
#pragma unroll
        for (int j = 0; j < LT; j++) {
            if (j < JA) ring_load(dh, base + loff[j], voff[j], (unsigned)(ks * BK * 2));
            else if (j < NPL * JA) ring_load(dl, base + loff[j], voff[j], (unsigned)(ks * BK * 2));
            else ring_load(dw, base + loff[j], voff[j], (unsigned)(ks * BK * WB));
        }
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    ring_wait<0>();
#pragma unroll
    for (int s = 0; s < S - 1; s++) issue(kt0 + s, s);
    const int fr = lane & 15, g = lane >> 4;
    int cur = 0;  // ring slot of step kt
    for (int kt = kt0; kt < kt1; kt++) {
        ring_wait<L * (S - 2)>();  // this wave's loads of step kt have landed
        ring_barrier();            // every wave's have; slot kt - 1 is free
        issue(kt + S - 1, cur == 0 ? S - 1 : cur - 1);
        const unsigned char *st = sm + cur * STAGE;
        cur = cur == S - 1 ? 0 : cur + 1;
        bf16x8 b0[TN], b1[TN];
#pragma unroll
        for (int tn = 0; tn < TN; tn++) {
            const int n = wn * TN * 16 + tn * 16 + fr;
            if constexpr (WBF) {  // bf16 rows: chunk 2 g + h of the column's 128 bytes
                b0[tn] = *(const bf16x8 *)(st + A_PL + n * 128 + (((2 * g) ^ (fr & 7)) << 4));
                b1[tn] = *(const bf16x8 *)(st + A_PL + n * 128 + (((2 * g + 1) ^ (fr & 7)) << 4));
            } else if constexpr (B32) {  // a half step is one block: 8 weights at k 32 h + 8 g
                const int sw = (fr >> 1) & 3, lo8 = 8 * (g & 1);
                const uint2 v0 = *(const uint2 *)(st + 2 * A_PL + n * 64 + (((g >> 1) ^ sw) << 4) + lo8);
                const uint2 v1 = *(const uint2 *)(st + 2 * A_PL + n * 64 + (((2 + (g >> 1)) ^ sw) << 4) + lo8);
                u32x4 o0, o1;
                bytes_to_bf16(u32x4{v0.x, v0.y, v1.x, v1.y}, o0, o1);
                b0[tn] = __builtin_bit_cast(bf16x8, o0);
                b1[tn] = __builtin_bit_cast(bf16x8, o1);
            } else {
                const u32x4 v = *(const u32x4 *)(st + 2 * A_PL + n * 64 + ((g ^ ((fr >> 1) & 3)) << 4));
                u32x4 o0, o1;
                bytes_to_bf16(v, o0, o1);
                b0[tn] = __builtin_bit_cast(bf16x8, o0);
                b1[tn] = __builtin_bit_cast(bf16x8, o1);
            }
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            bf16x8 ah[TM], al[TM];
#pragma unroll
            for (int tm = 0; tm < TM; tm++) {
                const int ch = B32 ? 4 * h + g : 2 * g + h;  // 16-byte chunk of the row's 128
                const int off = (wm * TM * 16 + tm * 16 + fr) * 128 + ((ch ^ (fr & 7)) << 4);
                ah[tm] = *(const bf16x8 *)(st + off);
                if (!WBF) al[tm] = *(const bf16x8 *)(st + A_PL + off);
            }
            if constexpr (B32) {
#pragma unroll
                for (int tn = 0; tn < TN; tn++) {
                    const float sc = *(const float *)(st + C::SC + (h * C::BN + wn * TN * 16 + tn * 16 + fr) * 4);
                    f32x4 t[TM];
#pragma unroll
                    for (int tm = 0; tm < TM; tm++)
                        t[tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[tm], h ? b1[tn] : b0[tn], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (int tm = 0; tm < TM; tm++)
                        t[tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[tm], h ? b1[tn] : b0[tn], t[tm], 0, 0, 0);
#pragma unroll
                    for (int tm = 0; tm < TM; tm++)
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[tm][tn][r] = fmaf(sc, t[tm][r], acc[tm][tn][r]);
                }
                continue;
            }
#pragma unroll
            for (int tn = 0; tn < TN; tn++)
#pragma unroll
                for (int tm = 0; tm < TM; tm++)
                    acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[tm], h ? b1[tn] : b0[tn], acc[tm][tn], 0, 0, 0);
            if (!WBF) {
#pragma unroll
                for (int tn = 0; tn < TN; tn++)
#pragma unroll
                    for (int tm = 0; tm < TM; tm++)
                        acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[tm], h ? b1[tn] : b0[tn], acc[tm][tn], 0, 0, 0);
            }
        }
    }
    ring_wait<0>();  // the re-read tail steps land before the workgroup's LDS is reused or released
    if (!C::BIG && p.splits > 1) {
        float *part = p.partf + (size_t)sp * p.M * p.N;
#pragma unroll
        for (int tn = 0; tn < TN; tn++) {
            const int n = n0 + wn * TN * 16 + tn * 16 + fr;
#pragma unroll
            for (int tm = 0; tm < TM; tm++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = m0 + wm * TM * 16 + tm * 16 + (g << 2) + r;
                    if (m < p.M && n < p.N) part[(size_t)m * p.N + n] = acc[tm][tn][r];
                }
        }
        return;
    }
    if (EPI == GE_SWIGLU) {
        __syncthreads();  // every wave's tail loads have landed
        swiglu_store<TM, TN, T, WBF || B32, C::BM, C::BN>(p, acc, reinterpret_cast<u16 *>(sm), wm * TM * 16, wn * TN * 16, m0,
                                                   n0, lane);
        if (wave == 0 && nbk == p.n_nb - 1) swiglu_pad<C::BM>(p, m0, lane);
    } else {
        gemm_store<EPI, TM, TN>(p, acc, m0 + wm * TM * 16, n0 + wn * TN * 16, lane, p.scale, p.scale2);
    }
}

// The k splits' f32 sums of k_gemm_ring, added in split order, then
// gemm_store's epilogue.
template <int EPI>
__global__ __launch_bounds__(256) void k_ring_finish(GemmP p) {
    const size_t mn = (size_t)p.M * p.N;
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < mn; t += (size_t)gridDim.x * 256) {
        const int m = (int)(t / p.N), n = (int)(t % p.N);
        float v = p.partf[t];
        for (int sp = 1; sp < p.splits; sp++) v += p.partf[(size_t)sp * mn + t];
        v *= p.scale;
        float *c = p.c + (size_t)m * p.ldc + n;
        *c = EPI == GE_RESID ? *c + v : p.bias ? v + p.bias[n] : v;
    }
}

// ------------------------------------------------------------------ GEMM on the int8 matrix cores
// Activations as digit planes (k_norm_digits): x = (d0 + 2^8 d1 + 2^16 d2)
// 2^-E per row, weights q (byte XOR 0x80).  Three v_mfma_i32_16x16x64_i8
// per 64-wide k step and tile (one per digit plane) accumulate exact integer
// sums in i32 (|d q| <= 2^14, k <= 131008); the epilogue forms
// S = A2 2^16 + A1 2^8 + A0 exactly in f64 and writes f32(S 2^-E scale)
// (one rounding) through the same store / SwiGLU epilogues.  Against the
// split-bf16 kernel: 3 int8 MFMAs at twice the bf16 rate instead of 4 bf16
// ones per 64 k, no weight conversion, 192 activation bytes per row and step
// instead of 256 (measured on the config-5 shapes in a stand-alone harness:
// qkv 715-820 -> 512 us, gate/up 3118-3189 -> 2288 us).
// Staging as k_gemm_ring: a 3-step direct-to-LDS ring; a step holds the three
// digit planes [128 rows][64 B] and the weights [256 columns][64 B], 16-byte
// chunk c of row r at c ^ ((r >> 1) & 3).  Lane group g of a 16x16x64 MFMA
// reads chunk g of its row / column for both operands, so every k pairs with
// itself.  8 waves of 64 x 64 outputs, 120 KB of LDS, one workgroup per CU.
// Small row counts (short prompts, the op-level matmul) leave most CUs idle
// with that tile (512 rows x 4096 columns: 64 workgroups), so launch_gemm also
// picks smaller tiles and splits k: a split writes its exact sums S (integers
// below 2^53) as f64, and k_digits_finish adds them (exactly, in any order)
// and applies the same scale, rounding and epilogue: the same bits whatever
// the tile and the split.
template <int BM_, int BN_, int WGM_, int WGN_, int S_>
struct DTile {
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, S = S_;
    static constexpr int TM = BM / WGM / 16, TN = BN / WGN / 16, NW = WGM * WGN, T = 64 * NW;
    static constexpr int A_PL = BM * BK, B_ST = BN * BK, STAGE = 3 * A_PL + B_ST;
    // 1 KB loads per wave (16 rows of 64 B); weight loads past the last unit repeat it
    static constexpr int JP = 3 * A_PL / 1024 / NW, BU = B_ST / 1024, JB = (BU + NW - 1) / NW, L = JP + JB;
    static constexpr size_t LDS = (size_t)S * STAGE;
    static constexpr bool BIG = BM_ == 128 && BN_ == 256;  // k_gemm_ring's tile and map
    static_assert(BK == 64 && WGM * TM * 16 == BM && WGN * TN * 16 == BN, "digit ring tile");
    static_assert(3 * A_PL / 1024 % NW == 0, "digit ring units");
    static_assert(L * (S - 2) < 64, "vmcnt range");
    static_assert(LDS >= BM * (BN / 2 + 4) * sizeof(float), "SwiGLU staging tile");
};
using DBig = DTile<BM, BN, 2, 4, 3>;
static_assert(DBig::LDS >= 2 * BM * (BN / 2 + 8) * sizeof(u16), "SwiGLU plane staging tile");

// S 2^-E scale in f64, one rounding to f32
__device__ __forceinline__ float digit_value(double S, int E, double sc) {
    return E == DG_NONFINITE ? __builtin_nanf("") : (float)(S * ldexp(1.0, -E) * sc);
}

template <int EPI, class TL>
__global__ __launch_bounds__(TL::T, TL::BIG ? 1 : 2) void k_gemm_digits(GemmP p) {
    constexpr int TM = TL::TM, TN = TL::TN, NW = TL::NW, T = TL::T, S = TL::S, A_PL = TL::A_PL, STAGE = TL::STAGE;
    constexpr int JP = TL::JP, L = TL::L, AU = A_PL / 1024;
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    extern __shared__ float4 dsm[];
    unsigned char *sm = reinterpret_cast<unsigned char *>(dsm);
    int mb, nbk, sp = 0;
    if (TL::BIG ? !gemm_tile(p, mb, nbk) : !small_tile(p, mb, nbk, sp)) return;
    const int m0 = mb * TL::BM, n0 = nbk * TL::BN;
    // this split's k steps
    const int kt0 = TL::BIG ? 0 : sp * p.kchunk, kt1 = TL::BIG ? p.nk : min(p.nk, kt0 + p.kchunk);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wm = wave / TL::WGN, wn = wave % TL::WGN;
    const u32x4 da = ring_desc(p.ad, 3 * p.dstride), dw = ring_desc(p.w, (size_t)p.N * p.kp);
    const unsigned sm0 = (unsigned)(uintptr_t)sm;  // LDS address (low half of the flat address)
    // load j of this wave fills 1 KB block u = j NW + wave: digit plane u / AU
    // (16 rows of 64 B) for j < JP, then the weights (16 columns of 64 B)
    unsigned voff[L], loff[L];
#pragma unroll
    for (int j = 0; j < L; j++) {
        if (j < JP) {
            const int u = j * NW + wave, pl = u / AU, ua = u % AU;
            const int r = 16 * ua + (lane >> 2), c = (lane & 3) ^ ((r >> 1) & 3);
            voff[j] = (unsigned)(pl * p.dstride + (size_t)(m0 + r) * p.lda + c * 16);
            loff[j] = (unsigned)(pl * A_PL + ua * 1024);
        } else {
            const int ub = min((j - JP) * NW + wave, TL::BU - 1);
            const int n = 16 * ub + (lane >> 2), c = (lane & 3) ^ ((n >> 1) & 3);
            const int row = min(n0 + n, p.N - 1);  // columns past N re-read row N - 1 (never stored)
            voff[j] = (unsigned)(row * p.kp + c * 16);
            loff[j] = (unsigned)(3 * A_PL + ub * 1024);
        }
    }
    // step kt into ring slot; steps past the last re-read the last (in bounds, never used)
    auto issue = [&](int kt, int slot) {
        const unsigned ko = (unsigned)(min(kt, kt1 - 1) * BK);
        const unsigned base = sm0 + (unsigned)(slot * STAGE);
#pragma unroll
        for (int j = 0; j < L; j++) ring_load(j < JP ? da : dw, base + loff[j], voff[j], ko);
    };

    i32x4 acc[3][TM][TN];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[d][i][j] = i32x4{0, 0, 0, 0};
    ring_wait<0>();
#pragma unroll
    for (int s = 0; s < S - 1; s++) issue(kt0 + s, s);
    const int fr = lane & 15, g = lane >> 4;
    int cur = 0;  // ring slot of step kt
    for (int kt = kt0; kt < kt1; kt++) {
        ring_wait<L * (S - 2)>();  // this wave's loads of step kt have landed
        ring_barrier();            // every wave's have; slot kt - 1 is free
        issue(kt + S - 1, cur == 0 ? S - 1 : cur - 1);
        const unsigned char *st = sm + cur * STAGE;
        cur = cur == S - 1 ? 0 : cur + 1;
        i32x4 bq[TN];
#pragma unroll
        for (int tn = 0; tn < TN; tn++) {
            const int n = wn * TN * 16 + tn * 16 + fr;
            const u32x4 v = *(const u32x4 *)(st + 3 * A_PL + n * 64 + ((g ^ ((fr >> 1) & 3)) << 4)) ^ 0x80808080u;
            bq[tn] = __builtin_bit_cast(i32x4, v);
        }
#pragma unroll
        for (int d = 0; d < 3; d++) {
            i32x4 a[TM];
#pragma unroll
            for (int tm = 0; tm < TM; tm++) {
                const int r = wm * TM * 16 + tm * 16 + fr;
                a[tm] = *(const i32x4 *)(st + d * A_PL + r * 64 + ((g ^ ((fr >> 1) & 3)) << 4));
            }
#pragma unroll
            for (int tn = 0; tn < TN; tn++)
#pragma unroll
                for (int tm = 0; tm < TM; tm++)
                    acc[d][tm][tn] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[tm], bq[tn], acc[d][tm][tn], 0, 0, 0);
        }
    }
    ring_wait<0>();  // the re-read tail steps land before the workgroup's LDS is reused or released
    auto sum_of = [&](int tm, int tn, int r) {
        return (double)acc[2][tm][tn][r] * 65536.0 + (double)acc[1][tm][tn][r] * 256.0 + (double)acc[0][tm][tn][r];
    };
    if (!TL::BIG && p.splits > 1) {
        double *part = p.part + (size_t)sp * p.M * p.N;
#pragma unroll
        for (int tn = 0; tn < TN; tn++) {
            const int n = n0 + wn * TN * 16 + tn * 16 + fr;
#pragma unroll
            for (int tm = 0; tm < TM; tm++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = m0 + wm * TM * 16 + tm * 16 + (g << 2) + r;
                    if (m < p.M && n < p.N) part[(size_t)m * p.N + n] = sum_of(tm, tn, r);
                }
        }
        return;
    }
    // the scale and the rounding here; the store epilogues then run at unit scale
    int er[TM][4];
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = m0 + wm * TM * 16 + tm * 16 + (g << 2) + r;
            er[tm][r] = m < p.M ? p.ae[m] : 0;
        }
    f32x4 v[TM][TN];
#pragma unroll
    for (int tn = 0; tn < TN; tn++) {
        const int n = n0 + wn * TN * 16 + tn * 16 + fr;
        const double sc = EPI == GE_SWIGLU && (n & 2) ? (double)p.scale2 : (double)p.scale;  // gate / up rows
#pragma unroll
        for (int tm = 0; tm < TM; tm++)
#pragma unroll
            for (int r = 0; r < 4; r++) v[tm][tn][r] = digit_value(sum_of(tm, tn, r), er[tm][r], sc);
    }
    GemmP q = p;
    q.scale = q.scale2 = 1.f;
    if (EPI == GE_SWIGLU) {
        __syncthreads();  // every wave's tail loads have landed
        swiglu_store<TM, TN, T, false, TL::BM, TL::BN>(q, v, reinterpret_cast<u16 *>(sm), wm * TM * 16, wn * TN * 16, m0,
                                                       n0, lane);
        if (TL::BIG && !p.of && wave == 0 && nbk == p.n_nb - 1) swiglu_pad<BM>(p, m0, lane);
    } else {
        gemm_store<EPI, TM, TN>(q, v, m0 + wm * TM * 16, n0 + wn * TN * 16, lane, 1.f, 1.f);
    }
}

// The k splits' sums, added in split order; then gemm_store's (swiglu_store's,
// f32 rows) value and epilogue.  One thread per row and 4 columns (one SwiGLU
// group: gate, gate, up, up).  Bound by reading the partials once.
template <int EPI>
__global__ __launch_bounds__(256) void k_digits_finish(GemmP p) {
    const int nq = (p.N + 3) >> 2;
    const size_t mn = (size_t)p.M * p.N, total = (size_t)p.M * nq;
    const bool vec = p.N % 2 == 0;  // 16-byte pairs of doubles
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < total; t += (size_t)gridDim.x * 256) {
        const int m = (int)(t / nq), n = (int)(t % nq) * 4, w = min(4, p.N - n);
        const double *src = p.part + (size_t)m * p.N + n;
        double S[4] = {0.0, 0.0, 0.0, 0.0};
        for (int sp = 0; sp < p.splits; sp++) {
            const double *q = src + (size_t)sp * mn;
            if (vec) {
                const double2 a = *(const double2 *)q, b = w > 2 ? *(const double2 *)(q + 2) : make_double2(0.0, 0.0);
                S[0] += a.x, S[1] += a.y, S[2] += b.x, S[3] += b.y;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) S[e] += e < w ? q[e] : 0.0;
            }
        }
        const int E = p.ae[m];
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
            v[e] = digit_value(S[e], E, EPI == GE_SWIGLU && e >= 2 ? (double)p.scale2 : (double)p.scale);
        if (EPI == GE_SWIGLU) {
            *(float2 *)(p.of + (size_t)m * p.ldo + (n >> 1)) =
                make_float2(silu_split(v[0]) * v[2], silu_split(v[1]) * v[3]);
        } else {
            float *c = p.c + (size_t)m * p.ldc + n;
            for (int e = 0; e < w; e++)
                c[e] = EPI == GE_RESID ? c[e] + v[e] : EPI == GE_STORE && p.bias ? v[e] + p.bias[n + e] : v[e];
        }
    }
}

// ------------------------------------------------------------------ RoPE + KV append
// Row m = s * seq + i is position p0[s] + i of sequence s.  q pairs are rotated
// in place (llama.rs:208-216 without a pre-scale: forward scales the scores),
// k pairs are rotated into the cache row, v is copied into the cache row
// (kv_cache.rs:99-118).  cpu.rs:655-658 in f32, no contraction.
__global__ void k_rope_kv(float *qkv, int ldq, int M, int seq, int qd, int kvd, int hd, PrefillSeqs t, int l,
                          PrefillKVP kp) {
    const int hh = hd >> 1, nkv = kvd / hd;
    const int per_row = (qd >> 1) + (kvd >> 1) + kvd;
    const size_t total = (size_t)M * per_row;
    for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (size_t)gridDim.x * blockDim.x) {
        const int m = (int)(g / per_row), e = (int)(g % per_row);
        const int s = m / seq, i = m - s * seq;
        const int pos = t.p0[s] + i;
        float *row = qkv + (size_t)m * ldq;
        float *kc = t.k[s] + (size_t)l * t.ls[s] + (size_t)pos * kvd;
        float *vc = t.v[s] + (size_t)l * t.ls[s] + (size_t)pos * kvd;
        if (e < (qd >> 1) + (kvd >> 1)) {
            const bool isq = e < (qd >> 1);
            const int j = isq ? 2 * e : 2 * (e - (qd >> 1));  // element index within q or k
            const float2 cs = t.rope[s][(size_t)pos * hh + ((j % hd) >> 1)];
            float *x = isq ? row + j : row + qd + j;
            const float x0 = x[0], x1 = x[1];
            const float r0 = __fsub_rn(__fmul_rn(x0, cs.x), __fmul_rn(x1, cs.y));
            const float r1 = __fadd_rn(__fmul_rn(x0, cs.y), __fmul_rn(x1, cs.x));
            if (isq) {
                x[0] = r0;
                x[1] = r1;
            } else {
                kc[j] = r0;
                kc[j + 1] = r1;
                if (kp.kh) {  // the attention's planes of this K row
                    const size_t at = ((size_t)(s * nkv + j / hd) * kp.rows + pos) * hd + j % hd;
                    u16 h0, l0, h1, l1;
                    split_bf16(r0, h0, l0);
                    split_bf16(r1, h1, l1);
                    *(unsigned *)(kp.kh + at) = (unsigned)h0 | ((unsigned)h1 << 16);
                    *(unsigned *)(kp.kl + at) = (unsigned)l0 | ((unsigned)l1 << 16);
                }
            }
        } else {
            const int j = e - (qd >> 1) - (kvd >> 1);
            const float v = row[qd + kvd + j];
            vc[j] = v;
            if (kp.kh) {
                const size_t at = ((size_t)(s * nkv + j / hd) * kp.rows + pos) * hd + j % hd;
                split_bf16(v, kp.vh[at], kp.vl[at]);
            }
        }
    }
}

// The same with 8 consecutive elements (four rotation pairs, or eight v
// values) per thread: float4 loads and stores, 16-byte plane stores
// (qd, kvd, hd multiples of 8; ldq, the caches and the tables 16-byte aligned).
__global__ void k_rope_kv8(float *qkv, int ldq, int M, int seq, int qd, int kvd, int hd, PrefillSeqs t, int l,
                           PrefillKVP kp) {
    const int hh = hd >> 1, nkv = kvd / hd;
    const int per_row = (qd + 2 * kvd) >> 3;
    const size_t total = (size_t)M * per_row;
    for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (size_t)gridDim.x * blockDim.x) {
        const int m = (int)(g / per_row), e8 = (int)(g % per_row) * 8;
        const int s = m / seq, i = m - s * seq;
        const int pos = t.p0[s] + i;
        float *row = qkv + (size_t)m * ldq;
        float *kc = t.k[s] + (size_t)l * t.ls[s] + (size_t)pos * kvd;
        float *vc = t.v[s] + (size_t)l * t.ls[s] + (size_t)pos * kvd;
        float o[8];
        int j;  // element index within q, k or v
        int part;  // 0 q, 1 k, 2 v
        if (e8 < qd) {
            part = 0;
            j = e8;
        } else if (e8 < qd + kvd) {
            part = 1;
            j = e8 - qd;
        } else {
            part = 2;
            j = e8 - qd - kvd;
        }
        const float4 a0 = *(const float4 *)(row + e8), a1 = *(const float4 *)(row + e8 + 4);
        const float x[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
        if (part < 2) {
            const float4 *cs4 = (const float4 *)(t.rope[s] + (size_t)pos * hh + ((j % hd) >> 1));
            const float4 c0 = cs4[0], c1 = cs4[1];
            const float cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};  // (cos, sin) x 4
#pragma unroll
            for (int p = 0; p < 4; p++) {  // cpu.rs:655-658 in f32, no contraction
                const float x0 = x[2 * p], x1 = x[2 * p + 1], c = cs[2 * p], sn = cs[2 * p + 1];
                o[2 * p] = __fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, sn));
                o[2 * p + 1] = __fadd_rn(__fmul_rn(x0, sn), __fmul_rn(x1, c));
            }
        } else {
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = x[q];
        }
        float *dst = part == 0 ? row + j : part == 1 ? kc + j : vc + j;
        *(float4 *)dst = make_float4(o[0], o[1], o[2], o[3]);
        *(float4 *)(dst + 4) = make_float4(o[4], o[5], o[6], o[7]);
        if (part > 0 && kp.kh) {  // the attention's planes of this K / V row
            const size_t at = ((size_t)(s * nkv + j / hd) * kp.rows + pos) * hd + j % hd;
            unsigned ph[4], pl[4];
#pragma unroll
            for (int q = 0; q < 8; q += 2) {
                u16 h0, l0, h1, l1;
                split_bf16(o[q], h0, l0);
                split_bf16(o[q + 1], h1, l1);
                ph[q / 2] = (unsigned)h0 | ((unsigned)h1 << 16);
                pl[q / 2] = (unsigned)l0 | ((unsigned)l1 << 16);
            }
            u16 *bh = part == 1 ? kp.kh : kp.vh, *bl = part == 1 ? kp.kl : kp.vl;
            *(u32x4 *)(bh + at) = u32x4{ph[0], ph[1], ph[2], ph[3]};
            *(u32x4 *)(bl + at) = u32x4{pl[0], pl[1], pl[2], pl[3]};
        }
    }
}

// The planes of the K / V rows [0, p0) that earlier calls left in the caches.
__global__ void k_kv_planes(PrefillSeqs t, int l, int n_seq, int kvd, int hd, PrefillKVP kp) {
    const int nkv = kvd / hd;
    for (int s = 0; s < n_seq; s++) {
        const size_t total = (size_t)t.p0[s] * kvd;
        const float *kc = t.k[s] + (size_t)l * t.ls[s], *vc = t.v[s] + (size_t)l * t.ls[s];
        for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (size_t)gridDim.x * blockDim.x) {
            const int row = (int)(g / kvd), c = (int)(g % kvd);
            const size_t at = ((size_t)(s * nkv + c / hd) * kp.rows + row) * hd + c % hd;
            split_bf16(kc[g], kp.kh[at], kp.kl[at]);
            split_bf16(vc[g], kp.vh[at], kp.vl[at]);
        }
    }
}

// ------------------------------------------------------------------ attention
// Causal attention of the processed rows over their cache (llama.rs:218-250:
// scores = q.k, x scale, mask keys after the query position, softmax, P.V),
// online over 32-key tiles.  Workgroup: 128 query rows of one (head, sequence);
// two threads per row, each holding half of head_dim (HT >= hd / 2 values).
// The output row goes straight into the bf16 planes of the o_proj input.
constexpr int AQ = 128, AK = 32;

template <int HT>
__global__ __launch_bounds__(256) void k_attn_prefill(PrefillAttn a, PrefillSeqs t, int l) {
    extern __shared__ float4 asm4[];
    float *sk = reinterpret_cast<float *>(asm4);  // [AK][hd]
    float *sv = sk + AK * a.hd;
    const int tid = threadIdx.x, row = tid >> 1, half = tid & 1;
    const int qb = blockIdx.x, h = blockIdx.y, s = blockIdx.z;
    const int i = qb * AQ + row;
    const bool valid = i < a.seq;
    const int p0 = t.p0[s], pos = p0 + i;
    const int ht = a.hd >> 1, kvh = h / (a.nh / a.nkv);
    const size_t m = (size_t)s * a.seq + i;
    float q[HT], o[HT];
#pragma unroll
    for (int d = 0; d < HT; d++) {
        q[d] = (valid && d < ht) ? a.qkv[m * a.ldq + h * a.hd + half * ht + d] : 0.f;
        o[d] = 0.f;
    }
    float mx = -INFINITY, lsum = 0.f;
    const int kend = p0 + min(a.seq, (qb + 1) * AQ);  // keys [0, kend) cover this block
    const float *kc = t.k[s] + (size_t)l * t.ls[s] + (size_t)kvh * a.hd;
    const float *vc = t.v[s] + (size_t)l * t.ls[s] + (size_t)kvh * a.hd;
    for (int k0 = 0; k0 < kend; k0 += AK) {
        __syncthreads();
        for (int idx = tid; idx < AK * a.hd; idx += 256) {
            const int j = idx / a.hd, d = idx - j * a.hd;
            const bool in = k0 + j < kend;
            sk[idx] = in ? kc[(size_t)(k0 + j) * a.kvd + d] : 0.f;
            sv[idx] = in ? vc[(size_t)(k0 + j) * a.kvd + d] : 0.f;
        }
        __syncthreads();
        float sc[AK];
        float bm = -INFINITY;
#pragma unroll
        for (int j = 0; j < AK; j++) {
            const float *kr = sk + j * a.hd + half * ht;
            float dt = 0.f;
#pragma unroll
            for (int d = 0; d < HT; d++)
                if (d < ht) dt = fmaf(q[d], kr[d], dt);
            dt += __shfl_xor(dt, 1);
            const float v = k0 + j <= pos ? dt * a.scale : -INFINITY;
            sc[j] = v;
            bm = fmaxf(bm, v);
        }
        const float mn = fmaxf(mx, bm);
        if (mn == -INFINITY) continue;  // every key so far masked (rows past seq)
        const float alpha = expf(mx - mn);
        lsum *= alpha;
#pragma unroll
        for (int d = 0; d < HT; d++) o[d] *= alpha;
#pragma unroll
        for (int j = 0; j < AK; j++) {
            const float pj = expf(sc[j] - mn);
            lsum += pj;
            const float *vr = sv + j * a.hd + half * ht;
#pragma unroll
            for (int d = 0; d < HT; d++)
                if (d < ht) o[d] = fmaf(pj, vr[d], o[d]);
        }
        mx = mn;
    }
    if (!valid) return;
    const float inv = 1.f / lsum;
    u16 *ph = a.ohi + m * a.ldo + h * a.hd + half * ht;
    u16 *pl = a.olo + m * a.ldo + h * a.hd + half * ht;
#pragma unroll
    for (int d = 0; d < HT; d++)
        if (d < ht) {
            u16 x0, x1;
            split_bf16(o[d] * inv, x0, x1);
            ph[d] = x0;
            pl[d] = x1;
        }
    if (h == a.nh - 1 && half == 1)  // zero the k padding of the o_proj input
        for (int c = a.nh * a.hd; c < a.opad; c++) {
            a.ohi[m * a.ldo + c] = 0;
            a.olo[m * a.ldo + c] = 0;
        }
}

// The same attention on the fp32 matrix cores (v_mfma_f32_16x16x4_f32: lane
// l holds A[l % 16][l / 16], B[l / 16][l % 16] and D[4 (l / 16) + r][l % 16]).
// Workgroup: MQ query rows of one (head, sequence), one wave per 16 rows; K/V
// tiles of MK keys in LDS.  Per wave and 16-key sub-tile:
//   S^T = K Q^T in HD/4 MFMAs; chunk c, position j holds head dim (HD/4) j + c,
//     so a lane's K and Q values are contiguous.  Lane l receives the scores
//     of query row l % 16 against keys 4 (l / 16) + r, r = 0..3;
//   online softmax per query row, reduced over the 4 lanes l % 16 + 16 g;
//   O^T += V^T P^T in HD/16 x 4 MFMAs; chunk r takes keys 4 j + r, so P^T is
//     the lane's own scores, and lane l accumulates query row l % 16 at head
//     dims 16 t + 4 (l / 16) + r.
// fp32 products and accumulation: the arithmetic of the VALU kernel above,
// in another summation order.
constexpr int MQW = 8, MQ = 16 * MQW, MK = 64;  // waves (16 query rows each) per workgroup; keys per tile

template <int HD>
__global__ __launch_bounds__(64 * MQW) void k_attn_mfma(PrefillAttn a, PrefillSeqs t, int l) {
    constexpr int NC = HD / 4, NT = HD / 16, LD = HD + 4;
    extern __shared__ float4 am4[];
    float *sk = reinterpret_cast<float *>(am4);  // [MK][LD]
    float *sv = sk + MK * LD;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int qb = (int)gridDim.x - 1 - (int)blockIdx.x;  // longest blocks first
    const int h = blockIdx.y, s = blockIdx.z;
    const int lr = lane & 15, lg = lane >> 4;
    const int i = qb * MQ + w * 16 + lr;
    const bool valid = i < a.seq;
    const int p0 = t.p0[s], pos = p0 + i;
    const int kvh = h / (a.nh / a.nkv);
    const size_t m = (size_t)s * a.seq + i;
    float q[NC];
    {
        const float *qr = a.qkv + m * a.ldq + h * HD + NC * lg;
#pragma unroll
        for (int c = 0; c < NC; c++) q[c] = valid ? qr[c] : 0.f;
    }
    f32x4 o[NT];
#pragma unroll
    for (int dt = 0; dt < NT; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float mrow = -INFINITY, lrow = 0.f;
    const int kend = p0 + min(a.seq, (qb + 1) * MQ);                 // keys of the workgroup
    const int wlast = p0 + min(a.seq, qb * MQ + w * 16 + 16) - 1;    // last key of this wave's rows
    const float *kc = t.k[s] + (size_t)l * t.ls[s] + (size_t)kvh * HD;
    const float *vc = t.v[s] + (size_t)l * t.ls[s] + (size_t)kvh * HD;
    for (int k0 = 0; k0 < kend; k0 += MK) {
        __syncthreads();
        for (int idx = tid; idx < MK * (HD / 4); idx += 64 * MQW) {
            const int j = idx / (HD / 4), c4 = idx - j * (HD / 4);
            float4 kv = make_float4(0.f, 0.f, 0.f, 0.f), vv = kv;
            if (k0 + j < kend) {
                kv = *(const float4 *)(kc + (size_t)(k0 + j) * a.kvd + 4 * c4);
                vv = *(const float4 *)(vc + (size_t)(k0 + j) * a.kvd + 4 * c4);
            }
            *(float4 *)(sk + j * LD + 4 * c4) = kv;
            *(float4 *)(sv + j * LD + 4 * c4) = vv;
        }
        __syncthreads();
        for (int sb = 0; sb < MK; sb += 16) {
            const int kb = k0 + sb;
            if (kb > wlast) break;  // wave-uniform: masked for every row of the wave
            f32x4 st = f32x4{0.f, 0.f, 0.f, 0.f};
            const float *kr = sk + (sb + lr) * LD + NC * lg;
#pragma unroll
            for (int c = 0; c < NC; c++) st = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[c], q[c], st, 0, 0, 0);
            float p[4];
            float tmax = -INFINITY;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                p[r] = kb + 4 * lg + r <= pos ? st[r] * a.scale : -INFINITY;  // llama.rs:225-234
                tmax = fmaxf(tmax, p[r]);
            }
            tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
            const float mn = fmaxf(mrow, tmax);  // finite: key 0 is visible to every row
            const float alpha = expf(mrow - mn);
            float ps = 0.f;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                p[r] = expf(p[r] - mn);
                ps += p[r];
            }
            ps += __shfl_xor(ps, 16);
            ps += __shfl_xor(ps, 32);
            lrow = lrow * alpha + ps;
            mrow = mn;
#pragma unroll
            for (int dt = 0; dt < NT; dt++) o[dt] *= alpha;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float *vr = sv + (sb + 4 * lg + r) * LD + lr;
#pragma unroll
                for (int dt = 0; dt < NT; dt++)
                    o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[dt * 16], p[r], o[dt], 0, 0, 0);
            }
        }
    }
    if (!valid) return;
    const float inv = 1.f / lrow;
    u16 *ph = a.ohi + m * a.ldo + h * HD, *pl = a.olo + m * a.ldo + h * HD;
#pragma unroll
    for (int dt = 0; dt < NT; dt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int d = dt * 16 + 4 * lg + r;
            u16 x0, x1;
            split_bf16(o[dt][r] * inv, x0, x1);
            ph[d] = x0;
            pl[d] = x1;
        }
    if (h == a.nh - 1 && lg == 0)  // zero the k padding of the o_proj input
        for (int c = a.nh * HD; c < a.opad; c++) {
            a.ohi[m * a.ldo + c] = 0;
            a.olo[m * a.ldo + c] = 0;
        }
}

// The same attention on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16),
// every f32 operand x carried as hi = bf16(x), lo = bf16(x - hi) and each
// product as hi*hi + hi*lo + lo*hi (the lo*lo term is below 2^-16 of it):
// error ~2^-16 relative per product, where the fp32 matrix cores give 2^-24
// at one sixteenth of the rate.  K and V come as planes written once per row
// (k_rope_kv, k_kv_planes); q is split in registers.
// Workgroup: 16 query rows per wave, 8 waves, one (head, sequence); K / V
// tiles of 64 keys in LDS, K key-major [key][hd], V transposed [hd][key].
// Per wave and 32 keys:
//   S^T = K Q^T for two 16-key halves (A = K [16 keys][32 hd], B = Q^T):
//     lane l gets query l % 16 against keys 4 (l / 16) + r of each half;
//   online softmax per query over the 32 keys (4 lanes l % 16 + 16 g);
//   O^T += V^T P^T with the 32 keys as the MFMA's k: slot 8 g + e is key
//     4 g + e (e < 4) of the first half and 16 + 4 g + (e - 4) of the
//     second, which is exactly the P values lane (l % 16, g) holds.  The V
//     tile stores each 32-key chunk in that slot order, so a lane's 8 keys
//     are one 16-byte read (two 8-byte reads 32 bytes apart made 2-way bank
//     conflicts at the padded row stride).
constexpr int BQW = 8, BQ = 16 * BQW, BKT = 64;  // waves; query rows; keys per tile

// bf16 hi / lo words of two values with the hardware round-to-nearest-even
// conversion (the same bits as split_bf16 for finite inputs; NaN stays NaN)
__device__ __forceinline__ unsigned pack_hl(float a, float b, bool lo_plane) {
    const __bf16 ha = (__bf16)a, hb = (__bf16)b;
    if (!lo_plane) return (unsigned)__builtin_bit_cast(u16, ha) | ((unsigned)__builtin_bit_cast(u16, hb) << 16);
    const __bf16 la = (__bf16)(a - (float)ha), lb = (__bf16)(b - (float)hb);
    return (unsigned)__builtin_bit_cast(u16, la) | ((unsigned)__builtin_bit_cast(u16, lb) << 16);
}

template <int HD>
__global__ __launch_bounds__(64 * BQW) void k_attn_bf3(PrefillAttn a, PrefillSeqs t, PrefillKVP kv) {
    constexpr int NKB = HD / 32, NDT = HD / 16, KLD = HD + 8, VLD = BKT + 8;
    extern __shared__ float4 ab4[];
    u16 *sKh = reinterpret_cast<u16 *>(ab4);
    u16 *sKl = sKh + BKT * KLD, *sVh = sKl + BKT * KLD, *sVl = sVh + HD * VLD;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // 1-D grid, the longest query blocks of every (head, sequence) first; within
    // a block row, index g -> (sequence, KV head) g % (n_seq nkv), query head of
    // the group g / (n_seq nkv): the heads sharing K / V rows land on one XCD
    // (workgroup b runs on XCD b % 8)
    const int nhs = a.nh * a.nseq, nkvs = a.nkv * a.nseq;
    const int qb = a.nqb - 1 - (int)blockIdx.x / nhs, g = (int)blockIdx.x % nhs;
    const int kvg = g % nkvs, rep = g / nkvs;
    const int s = kvg / a.nkv, kvh = kvg % a.nkv, h = kvh * (a.nh / a.nkv) + rep;
    const int lr = lane & 15, lg = lane >> 4;
    const int i = qb * BQ + w * 16 + lr;
    const bool valid = i < a.seq;
    const int p0 = t.p0[s], pos = p0 + i;
    const size_t m = (size_t)s * a.seq + i;
    // Q^T fragments: lane (query lr, group lg) holds head dims 32 kb + 8 lg + e
    bf16x8 qh[NKB], ql[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++) {
        float4 v0 = make_float4(0.f, 0.f, 0.f, 0.f), v1 = v0;
        if (valid) {
            const float *qr = a.qkv + m * a.ldq + h * HD + 32 * kb + 8 * lg;
            v0 = *(const float4 *)qr;
            v1 = *(const float4 *)(qr + 4);
        }
        u32x4 hv, lv;
        hv.x = pack_hl(v0.x, v0.y, false), lv.x = pack_hl(v0.x, v0.y, true);
        hv.y = pack_hl(v0.z, v0.w, false), lv.y = pack_hl(v0.z, v0.w, true);
        hv.z = pack_hl(v1.x, v1.y, false), lv.z = pack_hl(v1.x, v1.y, true);
        hv.w = pack_hl(v1.z, v1.w, false), lv.w = pack_hl(v1.z, v1.w, true);
        qh[kb] = __builtin_bit_cast(bf16x8, hv);
        ql[kb] = __builtin_bit_cast(bf16x8, lv);
    }
    f32x4 o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float mrow = -INFINITY, lrow = 0.f;
    const int kend = p0 + min(a.seq, (qb + 1) * BQ);               // keys of the workgroup
    const int wlast = p0 + min(a.seq, qb * BQ + w * 16 + 16) - 1;  // last key of this wave's rows
    const size_t pb = ((size_t)s * a.nkv + kvh) * kv.rows * HD;     // plane rows of (s, kvh)
    for (int k0 = 0; k0 < kend; k0 += BKT) {
        __syncthreads();
        // K planes: key j, 8 head dims per chunk
        for (int idx = tid; idx < 2 * BKT * (HD / 8); idx += 64 * BQW) {
            const int pl = idx / (BKT * (HD / 8)), r = idx - pl * (BKT * (HD / 8));
            const int j = r / (HD / 8), c = r - j * (HD / 8);
            u32x4 v = u32x4{0u, 0u, 0u, 0u};
            if (k0 + j < kend) v = *(const u32x4 *)((pl ? kv.kl : kv.kh) + pb + (size_t)(k0 + j) * HD + 8 * c);
            *(u32x4 *)((pl ? sKl : sKh) + j * KLD + 8 * c) = v;
        }
        // V planes transposed: keys 2 jp, 2 jp + 1 of 8 head dims -> 8 words [hd][key pair]
        for (int idx = tid; idx < 2 * (BKT / 2) * (HD / 8); idx += 64 * BQW) {
            const int pl = idx / ((BKT / 2) * (HD / 8)), r = idx - pl * ((BKT / 2) * (HD / 8));
            const int c = r / (BKT / 2), jp = r - c * (BKT / 2), j = 2 * jp;
            const u16 *src = (pl ? kv.vl : kv.vh) + pb;
            u32x4 v0 = u32x4{0u, 0u, 0u, 0u}, v1 = v0;
            if (k0 + j < kend) v0 = *(const u32x4 *)(src + (size_t)(k0 + j) * HD + 8 * c);
            if (k0 + j + 1 < kend) v1 = *(const u32x4 *)(src + (size_t)(k0 + j + 1) * HD + 8 * c);
            const int jj = j & 31;  // key 16 h + 4 g + e of its chunk -> slot 8 g + 4 h + e
            u16 *dst = (pl ? sVl : sVh) + (8 * c) * VLD + (j - jj) + 8 * ((jj >> 2) & 3) + 4 * (jj >> 4) + (jj & 3);
            const unsigned a0[4] = {v0.x, v0.y, v0.z, v0.w}, a1[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                *(unsigned *)(dst + (2 * e) * VLD) = (a0[e] & 0xffffu) | (a1[e] << 16);
                *(unsigned *)(dst + (2 * e + 1) * VLD) = (a0[e] >> 16) | (a1[e] & 0xffff0000u);
            }
        }
        __syncthreads();
        for (int c32 = 0; c32 < BKT; c32 += 32) {
            const int kb0 = k0 + c32;
            if (kb0 > wlast) break;  // wave-uniform: masked for every row of the wave
            float p[8];
#pragma unroll
            for (int hf = 0; hf < 2; hf++) {
                f32x4 st = f32x4{0.f, 0.f, 0.f, 0.f};
                const int kr = (c32 + 16 * hf + lr) * KLD + 8 * lg;
#pragma unroll
                for (int kb = 0; kb < NKB; kb++) {
                    const bf16x8 kh = *(const bf16x8 *)(sKh + kr + 32 * kb);
                    const bf16x8 kl = *(const bf16x8 *)(sKl + kr + 32 * kb);
                    st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, qh[kb], st, 0, 0, 0);
                    st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, ql[kb], st, 0, 0, 0);
                    st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kl, qh[kb], st, 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 4; r++)
                    p[4 * hf + r] = kb0 + 16 * hf + 4 * lg + r <= pos ? st[r] * a.scale : -INFINITY;  // llama.rs:225-234
            }
            float tmax = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; e++) tmax = fmaxf(tmax, p[e]);
            tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
            const float mn = fmaxf(mrow, tmax);  // finite: key 0 is visible to every row
            // e^x as 2^(x log2 e) on the hardware exp: within ~1e-6 relative where
            // it matters, below the 2^-17 of the P planes it feeds; the row sum
            // is formed from the same values, so O / l stays consistent
            const float alpha = __builtin_amdgcn_exp2f((mrow - mn) * 1.44269504f);
            float ps = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                p[e] = __builtin_amdgcn_exp2f((p[e] - mn) * 1.44269504f);
                ps += p[e];
            }
            ps += __shfl_xor(ps, 16);
            ps += __shfl_xor(ps, 32);
            lrow = lrow * alpha + ps;
            mrow = mn;
            u32x4 phv, plv;
            phv.x = pack_hl(p[0], p[1], false), plv.x = pack_hl(p[0], p[1], true);
            phv.y = pack_hl(p[2], p[3], false), plv.y = pack_hl(p[2], p[3], true);
            phv.z = pack_hl(p[4], p[5], false), plv.z = pack_hl(p[4], p[5], true);
            phv.w = pack_hl(p[6], p[7], false), plv.w = pack_hl(p[6], p[7], true);
            const bf16x8 ph = __builtin_bit_cast(bf16x8, phv), pl = __builtin_bit_cast(bf16x8, plv);
#pragma unroll
            for (int dt = 0; dt < NDT; dt++) {
                o[dt] *= alpha;
                const int vr = (16 * dt + lr) * VLD + c32 + 8 * lg;
                const bf16x8 bvh = *(const bf16x8 *)(sVh + vr), bvl = *(const bf16x8 *)(sVl + vr);
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bvh, ph, o[dt], 0, 0, 0);
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bvh, pl, o[dt], 0, 0, 0);
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bvl, ph, o[dt], 0, 0, 0);
            }
        }
    }
    if (!valid) return;
    const float inv = 1.f / lrow;
    if (a.of) {  // f32 rows (quantized for the o_proj GEMM afterwards)
        float *orow = a.of + m * a.ldo + h * HD;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
            *(float4 *)(orow + dt * 16 + 4 * lg) =
                make_float4(o[dt][0] * inv, o[dt][1] * inv, o[dt][2] * inv, o[dt][3] * inv);
        return;
    }
    u16 *oh = a.ohi + m * a.ldo + h * HD, *ol = a.olo + m * a.ldo + h * HD;
#pragma unroll
    for (int dt = 0; dt < NDT; dt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int d = dt * 16 + 4 * lg + r;
            u16 x0, x1;
            split_bf16(o[dt][r] * inv, x0, x1);
            oh[d] = x0;
            ol[d] = x1;
        }
    if (h == a.nh - 1 && lg == 0)  // zero the k padding of the o_proj input
        for (int c = a.nh * HD; c < a.opad; c++) {
            a.ohi[m * a.ldo + c] = 0;
            a.olo[m * a.ldo + c] = 0;
        }
}

template <int HD>
int attn_bf3_t(const PrefillAttn &a, int n_seq, const PrefillSeqs &t, const PrefillKVP &kv, hipStream_t s) {
    constexpr size_t lds = (2 * (size_t)BKT * (HD + 8) + 2 * (size_t)HD * (BKT + 8)) * sizeof(u16);
    static bool attr = false;
    if (!attr) {
        SCRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_attn_bf3<HD>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        attr = true;
    }
    PrefillAttn ag = a;
    ag.nqb = (a.seq + BQ - 1) / BQ;
    ag.nseq = n_seq;
    hipLaunchKernelGGL(k_attn_bf3<HD>, dim3(ag.nqb * a.nh * n_seq), dim3(64 * BQW), lds, s, ag, t, kv);
    PF_LAUNCH_CHECK();
}

template <int HD>
int attn_mfma_t(const PrefillAttn &a, int n_seq, const PrefillSeqs &t, int l, hipStream_t s) {
    constexpr size_t lds = 2 * (size_t)MK * (HD + 4) * sizeof(float);
    static bool attr = false;
    if (!attr) {
        SCRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_attn_mfma<HD>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        attr = true;
    }
    const dim3 grid((a.seq + MQ - 1) / MQ, a.nh, n_seq);
    hipLaunchKernelGGL(k_attn_mfma<HD>, grid, dim3(64 * MQW), lds, s, a, t, l);
    PF_LAUNCH_CHECK();
}

template <int EPI, bool B32, bool WBF = false>
int gemm_t(const GemmP &p, hipStream_t s) {
    static bool attr = false;
    if (!attr) {
        SCRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_gemm<EPI, B32, WBF>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)GEMM_LDS));
        attr = true;
    }
    hipLaunchKernelGGL((k_gemm<EPI, B32, WBF>), dim3(gemm_tile_grid(p)), dim3(G_THREADS), GEMM_LDS, s, p);
    PF_LAUNCH_CHECK();
}

template <int EPI, class TL>
int digits_launch(const GemmP &p, int grid, hipStream_t s) {
    static bool attr = false;
    if (!attr) {
        SCRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_gemm_digits<EPI, TL>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)TL::LDS));
        attr = true;
    }
    hipLaunchKernelGGL((k_gemm_digits<EPI, TL>), dim3(grid), dim3(TL::T), TL::LDS, s, p);
    PF_LAUNCH_CHECK();
}

// p's k splits, none empty, and the workspace of their partial sums (el bytes each)
int set_splits(GemmP &p, int splits, size_t el, void **ws) {
    p.kchunk = (p.nk + splits - 1) / splits;
    p.splits = (p.nk + p.kchunk - 1) / p.kchunk;
    SCRY_TRY(split_workspace(el * p.M * p.N, &p.splits, ws));
    if (p.splits == 1) p.kchunk = p.nk;
    return SCRY_OK;
}

template <int EPI, class TL>
int digits_small(GemmP p, int splits, hipStream_t s) {
    p.n_mb = (p.M + TL::BM - 1) / TL::BM;
    p.n_nb = (p.N + TL::BN - 1) / TL::BN;
    void *ws = nullptr;
    SCRY_TRY(set_splits(p, splits, sizeof(double), &ws));
    p.part = (double *)ws;
    SCRY_TRY((digits_launch<EPI, TL>(p, (p.n_mb * p.n_nb * p.splits + 7) / 8 * 8, s)));
    if (p.splits > 1) {
        const size_t g = ((size_t)p.M * ((p.N + 3) / 4) + 255) / 256;
        hipLaunchKernelGGL(k_digits_finish<EPI>, dim3((unsigned)std::min<size_t>(g, 65536)), dim3(256), 0, s, p);
        PF_LAUNCH_CHECK();
    }
    return SCRY_OK;
}

// Tile and k splits for M rows.  The time of a choice: k steps of a split times
// the workgroups each CU runs one after another or together (workgroups / 256)
// times the measured time of one workgroup's step (us, from 17-1024 rows at
// k 768-11008, n 768-28672: alone on a CU / sharing it), plus the partial
// sums' round trip.  From about 224 tiles of 128 x 256 on the large tile stays
// the fastest.  Measured, that tile -> this choice (rows x k x n):
//   digits  512 x 11008 x 4096 193 -> 91 us, 512 x 4096 x 4096 81 -> 43, 130 x
//           4096 x 14336 80 -> 57, 64 x 11008 x 4096 180 -> 29, 200 x 768 x
//           2304 26 -> 11; kept: 512 x 4096 x 14336 89 (next best 113).  128 x
//           192 where the others leave the last round part empty: 130 x 4096 x
//           22016 82 -> 74, 1024 x 4096 x 6144 87 -> 81; not 1024 x 4096 x
//           14336 (167, it 220)
//   bf16    512 x 11008 x 4096 180 -> 65, 37 x 4096 x 12288 63 -> 22, 37 x
//           11008 x 4096 152 -> 22, 130 x 4096 x 28672 134 -> 81, 256 x 768 x
//           2304 22 -> 8; kept: 512 x 4096 x 28672 157 (next best 188)
//   block-32, against the register-staged kernel: 37 x 4096 x 14336 251 -> 38,
//           130 x 11008 x 4096 661 -> 75, 512 x 11008 x 4096 673 -> 144, 1024 x
//           4096 x 14336 523 -> 315 (large tile)
struct TileCost {
    int bm, bn;
    double alone, shared;
};
constexpr TileCost kDigitTiles[6] = {{128, 256, 1.25, 1.25}, {128, 128, 0.80, 0.80}, {64, 128, 0.52, 0.50}, {64, 64, 0.38, 0.345}, {32, 128, 0.376, 0.34}, {128, 192, 1.12, 1.14}};
constexpr TileCost kRingTiles[5] = {{128, 256, 1.15, 1.20}, {128, 128, 0.65, 0.70}, {64, 128, 0.42, 0.36}, {64, 64, 0.33, 0.23}, {32, 128, 0.34, 0.26}};
constexpr TileCost kB32Tiles[5] = {{128, 256, 2.2, 2.4}, {128, 128, 1.42, 1.38}, {64, 128, 0.92, 0.74}, {64, 64, 0.62, 0.49}, {32, 128, 0.60, 0.52}};
struct TilePick {
    int tile, splits;
    double t;
};
TilePick pick_tile(const TileCost *tl, int n_tiles, int M, int N, int nk, int part_bytes, int max_splits) {
    TilePick best{0, 1, 1e30};
    for (int i = 0; i < n_tiles; i++) {
        const double tiles = (double)((M + tl[i].bm - 1) / tl[i].bm) * ((N + tl[i].bn - 1) / tl[i].bn);
        for (int sp = 1; sp <= (i ? max_splits : 1); sp *= 2) {
            const double bytes = (double)sp * M * N * part_bytes;
            if (sp > 1 && (nk < 4 * sp || bytes > 268435456.0)) break;  // at most 256 MB of partial sums
            const double n = std::ceil(tiles * sp / 256.0);
            double t = (nk + sp - 1) / sp * n * (n > 1 ? tl[i].shared : tl[i].alone);
            if (sp > 1) t += 4.0 + 2.0 * bytes / 5.0e6;
            if (t < best.t) best = {i, sp, t};
        }
    }
    return best;
}

// A last round of the chip that is mostly empty costs a whole one.  Where it is
// 4 % cheaper (below that the model cannot tell: 1500 x 11008 x 4096 was 5 %
// slower at 1 %), the columns of the full rounds go to one launch and the rest
// to a second one with its own tile, 6 us allowed for launch and drain.
// Measured, one launch of the best tile -> two:
//   digits    384 x 4096 x 22016 147 -> 103 us, 511 x 4096 x 22016 149 -> 139,
//             600 x 4096 x 14336 146 -> 123, 1500 x 4096 x 22016 377 -> 339
//   block-32  384 x 4096 x 22016 238 -> 177, 600 x 4096 x 14336 244 -> 198,
//             2046 x 4096 x 14336 605 -> 546
struct CutPick {
    TilePick first, rest;
    int cols;  // columns of the first launch; 0 = one launch (first)
};
CutPick pick_cut(const TileCost *tl, int n_tiles, int M, int N, int nk, int part_bytes, int max_splits) {
    CutPick best{pick_tile(tl, n_tiles, M, N, nk, part_bytes, max_splits), {}, 0};
    double bt = 0.96 * best.first.t;
    for (int i = 0; i < n_tiles; i++) {
        const int n_mb = (M + tl[i].bm - 1) / tl[i].bm, n_nb = (N + tl[i].bn - 1) / tl[i].bn;
        const int rounds = (int)((int64_t)n_mb * n_nb / 256);
        const int64_t cols = (int64_t)rounds * 256 / n_mb * tl[i].bn;
        if (cols < 1 || cols >= N) continue;
        const TilePick r = pick_tile(tl, n_tiles, M, N - (int)cols, nk, part_bytes, max_splits);
        const double t = nk * rounds * (rounds > 1 ? tl[i].shared : tl[i].alone) + 6.0 + r.t;
        if (t < bt) bt = t, best = {{i, 1, 0.0}, r, (int)cols};
    }
    return best;
}

// columns [c0, c0 + n) of p as a problem of their own (c0 a multiple of 64;
// el: bytes of a weight)
GemmP gemm_cols(GemmP p, int c0, int n, int el) {
    const bool end = c0 + n == p.N;
    p.w += (size_t)c0 * p.kp * el;
    if (p.s32) p.s32 += (size_t)c0 * p.nb;
    if (p.bias) p.bias += c0;
    if (p.c) p.c += c0;
    if (p.of) p.of += c0 / 2;  // the SwiGLU outputs: one column per two
    if (p.ohi) p.ohi += c0 / 2;
    if (p.olo) p.olo += c0 / 2;
    p.opad = end ? p.opad - c0 / 2 : n / 2;  // the zero pad comes with the last columns
    p.N = n;
    p.n_nb = (n + BN - 1) / BN;
    return p;
}

template <int EPI>
int gemm_digits_tile(const GemmP &p, const TilePick &d, hipStream_t s) {
    switch (d.tile) {
        case 1: return digits_small<EPI, DTile<128, 128, 2, 4, 3>>(p, d.splits, s);
        case 2: return digits_small<EPI, DTile<64, 128, 2, 2, 3>>(p, d.splits, s);
        case 3: return digits_small<EPI, DTile<64, 64, 2, 2, 4>>(p, d.splits, s);
        case 4: return digits_small<EPI, DTile<32, 128, 1, 2, 4>>(p, d.splits, s);
        case 5: return digits_small<EPI, DTile<128, 192, 2, 4, 3>>(p, d.splits, s);
    }
    return digits_launch<EPI, DBig>(p, gemm_tile_grid(p), s);
}

template <int EPI>
int gemm_digits_t(const GemmP &p, hipStream_t s) {
    // the smaller tiles write SwiGLU as f32 rows only
    const CutPick d = pick_cut(kDigitTiles, EPI != GE_SWIGLU || p.of ? 6 : 1, p.M, p.N, p.nk, sizeof(double), 16);
    if (!d.cols) return gemm_digits_tile<EPI>(p, d.first, s);
    SCRY_TRY(gemm_digits_tile<EPI>(gemm_cols(p, 0, d.cols, 1), d.first, s));
    return gemm_digits_tile<EPI>(gemm_cols(p, d.cols, p.N - d.cols, 1), d.rest, s);
}

template <int EPI, bool WBF, bool B32, class C>
int ring_launch(const GemmP &p, int grid, hipStream_t s) {
    static bool attr = false;
    if (!attr) {
        SCRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_gemm_ring<EPI, WBF, B32, C>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS));
        attr = true;
    }
    hipLaunchKernelGGL((k_gemm_ring<EPI, WBF, B32, C>), dim3(grid), dim3(C::T), C::LDS, s, p);
    PF_LAUNCH_CHECK();
}

template <int EPI, bool WBF, bool B32, class C>
int ring_small(GemmP p, int splits, hipStream_t s) {
    p.n_mb = (p.M + C::BM - 1) / C::BM;
    p.n_nb = (p.N + C::BN - 1) / C::BN;
    void *ws = nullptr;
    SCRY_TRY(set_splits(p, splits, sizeof(float), &ws));
    p.partf = (float *)ws;
    SCRY_TRY((ring_launch<EPI, WBF, B32, C>(p, (p.n_mb * p.n_nb * p.splits + 7) / 8 * 8, s)));
    if (p.splits > 1) {
        const size_t g = ((size_t)p.M * p.N + 255) / 256;
        hipLaunchKernelGGL(k_ring_finish<EPI>, dim3((unsigned)std::min<size_t>(g, 65536)), dim3(256), 0, s, p);
        PF_LAUNCH_CHECK();
    }
    return SCRY_OK;
}

template <int EPI, bool WBF, bool B32>
int gemm_ring_tile(const GemmP &p, const TilePick &d, hipStream_t s) {
    if constexpr (WBF || B32) {
        switch (d.tile) {
            case 1: return ring_small<EPI, WBF, B32, RTile<WBF, B32, 128, 128, 2, 4, 3>>(p, d.splits, s);
            case 2: return ring_small<EPI, WBF, B32, RTile<WBF, B32, 64, 128, 2, 2, 3>>(p, d.splits, s);
            case 3: return ring_small<EPI, WBF, B32, RTile<WBF, B32, 64, 64, 2, 2, B32 ? 3 : 4>>(p, d.splits, s);
            case 4: return ring_small<EPI, WBF, B32, RTile<WBF, B32, 32, 128, 1, 4, 4>>(p, d.splits, s);
        }
    }
    return ring_launch<EPI, WBF, B32, RBig<WBF, B32>>(p, gemm_tile_grid(p), s);
}

// WBF or B32: the tile by pick_cut; int8 per-tensor weights through bf16
// planes (k beyond the digit kernel's): the large tile
template <int EPI, bool WBF, bool B32 = false>
int gemm_ring_t(const GemmP &p, hipStream_t s) {
    if (!WBF && !B32) return gemm_ring_tile<EPI, WBF, B32>(p, {0, 1, 0.0}, s);
    // SwiGLU planes come from the whole sums: no k splits
    const CutPick d = pick_cut(B32 ? kB32Tiles : kRingTiles, 5, p.M, p.N, p.nk, sizeof(float), EPI == GE_SWIGLU ? 1 : 8);
    if (!d.cols) return gemm_ring_tile<EPI, WBF, B32>(p, d.first, s);
    SCRY_TRY((gemm_ring_tile<EPI, WBF, B32>(gemm_cols(p, 0, d.cols, WBF ? 2 : 1), d.first, s)));
    return gemm_ring_tile<EPI, WBF, B32>(gemm_cols(p, d.cols, p.N - d.cols, WBF ? 2 : 1), d.rest, s);
}

}  // namespace

int prefill_rows_pad(int M) { return (M + BM - 1) / BM * BM; }
int prefill_k_pad(int k) { return (k + BK - 1) / BK * BK; }

int launch_norm_split(const float *x, int ldx, int rows, int rstep, int roff, const float *w, int k, float eps,
                      u16 *hi, u16 *lo, int ldp, float *outf, int ldf, hipStream_t s) {
    if (rows <= 0) return SCRY_OK;
    const int kpad = hi ? prefill_k_pad(k) : k;
    if (hi && kpad > ldp) return set_error(SCRY_ERR_INVALID, "norm_split: k %d exceeds plane stride %d", k, ldp);
    const bool al16 = ((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0) && ((uintptr_t)hi % 16 == 0) &&
                      ((uintptr_t)lo % 16 == 0) && ldx % 4 == 0 && ldp % 8 == 0 && (rstep * ldx) % 4 == 0 &&
                      (roff * ldx) % 4 == 0;
    const int nc = (kpad + 2047) / 2048;
    if (hi && !outf && k % 8 == 0 && al16 && nc <= 8) {
        switch (nc) {
            case 1: hipLaunchKernelGGL(k_norm_split8<1>, dim3(rows), dim3(256), 0, s, x, ldx, rstep, roff, w, k, eps, hi, lo, ldp, kpad); break;
            case 2: hipLaunchKernelGGL(k_norm_split8<2>, dim3(rows), dim3(256), 0, s, x, ldx, rstep, roff, w, k, eps, hi, lo, ldp, kpad); break;
            case 3:
            case 4: hipLaunchKernelGGL(k_norm_split8<4>, dim3(rows), dim3(256), 0, s, x, ldx, rstep, roff, w, k, eps, hi, lo, ldp, kpad); break;
            default: hipLaunchKernelGGL(k_norm_split8<8>, dim3(rows), dim3(256), 0, s, x, ldx, rstep, roff, w, k, eps, hi, lo, ldp, kpad); break;
        }
        PF_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_norm_split, dim3(rows), dim3(256), 0, s, x, ldx, rstep, roff, w, k, eps, hi, lo, ldp,
                       kpad, outf, ldf);
    PF_LAUNCH_CHECK();
}

bool gemm_takes_digits(const Packed &w) {
    // int8 per-tensor weights; k bound: |sum of d q| <= 2^14 kpad stays in i32
    return !w.bf16 && !w.s32 && prefill_k_pad(w.k) <= 131008;
}

int launch_norm_digits(const float *x, int ldx, int rows, const float *w, int k, float eps, signed char *dg,
                       size_t dstride, int *e, int ldp, hipStream_t s) {
    if (rows <= 0) return SCRY_OK;
    const int kpad = prefill_k_pad(k);
    if (kpad > ldp || ldp % 16 || dstride % 16 || dstride < (size_t)rows * ldp || (uintptr_t)dg % 16)
        return set_error(SCRY_ERR_INVALID, "norm_digits: k %d, plane stride %d / %zu", k, ldp, dstride);
    const int nc = (kpad + 2047) / 2048;
    if (nc > 8) return set_error(SCRY_ERR_UNSUPPORTED, "norm_digits: k %d > 16384", k);
    const bool norm = w != nullptr;
    const bool vec = k % 8 == 0 && (uintptr_t)x % 16 == 0 && ldx % 4 == 0 && (uintptr_t)w % 16 == 0;
#define ND_LAUNCH(NC, V, N) \
    hipLaunchKernelGGL((k_norm_digits<NC, V, N>), dim3(rows), dim3(256), 0, s, x, ldx, w, k, eps, dg, dstride, e, ldp, kpad)
#define ND_NC(NC)                         \
    if (vec && norm) ND_LAUNCH(NC, true, true);   \
    else if (norm) ND_LAUNCH(NC, false, true);    \
    else if (vec) ND_LAUNCH(NC, true, false);     \
    else ND_LAUNCH(NC, false, false)
    switch (nc) {
        case 1: ND_NC(1); break;
        case 2: ND_NC(2); break;
        case 3:
        case 4: ND_NC(4); break;
        default: ND_NC(8); break;
    }
#undef ND_NC
#undef ND_LAUNCH
    PF_LAUNCH_CHECK();
}

int launch_split(const float *x, int ldx, int rows, int k, u16 *hi, u16 *lo, int ldp, hipStream_t s) {
    const int kpad = prefill_k_pad(k);
    if (kpad > ldp) return set_error(SCRY_ERR_INVALID, "split: k %d exceeds plane stride %d", k, ldp);
    const size_t total = (size_t)rows * kpad;
    if (total == 0) return SCRY_OK;
    const unsigned grid = (unsigned)std::min<size_t>((total + 255) / 256, 65536);
    hipLaunchKernelGGL(k_split, dim3(grid), dim3(256), 0, s, x, ldx, rows, k, kpad, hi, lo, ldp);
    PF_LAUNCH_CHECK();
}

int launch_gemm(int epi, const PrefillGemm &g, hipStream_t s) {
    const Packed &w = *g.w;
    const int kp_el = w.bf16 ? w.kp / 2 : w.kp;  // row stride in weights
    if (w.kp % 16 || w.k > kp_el) return set_error(SCRY_ERR_INVALID, "gemm: bad packed layout");
    if (w.bf16 && w.s32) return set_error(SCRY_ERR_INVALID, "gemm: bf16 weights carry no block scales");
    if (w.bytes() >= 0x7fffffffull)  // buffer offsets are 32-bit
        return set_error(SCRY_ERR_UNSUPPORTED, "gemm: %zu weight bytes (limit 2 GiB per tensor)", w.bytes());
    const int kpad = prefill_k_pad(w.k);
    if (kpad > g.lda || g.lda % 8) return set_error(SCRY_ERR_INVALID, "gemm: plane stride %d < k %d", g.lda, w.k);
    if (epi == GE_SWIGLU && (w.fused != 1 || w.rows % 4 || (w.rows >> 1) > g.ldo || g.opad > g.ldo || g.ldo % 8 ||
                             ((uintptr_t)g.ohi | (uintptr_t)g.olo) % 16))
        return set_error(SCRY_ERR_INVALID, "gemm: swiglu needs the fused gate/up layout");
    if (w.s32 && w.nb * 32 < w.k) return set_error(SCRY_ERR_INVALID, "gemm: block-32 scales too short");
    if (g.of && (!g.ad || epi != GE_SWIGLU || (uintptr_t)g.of % 16 || g.ldo % 4))
        return set_error(SCRY_ERR_INVALID, "gemm: f32 SwiGLU rows need digit planes and 16-byte rows");
    if (g.ad) {  // digit planes: the int8 matrix cores
        if (!gemm_takes_digits(w) || !g.ae || g.lda % 16 || (uintptr_t)g.ad % 16 ||
            g.dstride < (size_t)prefill_rows_pad(g.M) * g.lda || 3 * g.dstride >= 0x7fffffffull)
            return set_error(SCRY_ERR_INVALID, "gemm: digit planes need int8 per-tensor weights and a %d-row stride",
                             prefill_rows_pad(g.M));
    }
    GemmP p{};
    p.ahi = g.ahi;
    p.alo = g.alo;
    p.ad = g.ad;
    p.ae = g.ae;
    p.dstride = g.dstride;
    p.of = g.of;
    p.lda = g.lda;
    p.w = w.d;
    p.kp = kp_el;
    p.N = w.rows;
    p.s32 = w.s32;
    p.nb = w.nb;
    p.M = g.M;
    p.nk = kpad / BK;
    p.n_mb = (g.M + BM - 1) / BM;
    p.n_nb = (w.rows + BN - 1) / BN;
    p.scale = w.scale;
    p.scale2 = w.scale2;
    p.bias = g.bias;
    p.c = g.c;
    p.ldc = g.ldc;
    p.ohi = g.ohi;
    p.olo = g.olo;
    p.ldo = g.ldo;
    p.opad = g.opad;
    const bool b32 = w.s32 != nullptr;
    // the ring kernels address the planes through a buffer descriptor (32-bit
    // offsets); larger planes take the register-staged kernel
    const bool ring_ok = (size_t)p.n_mb * BM * p.lda * 2 < 0x7fffffffull;
    if (w.bf16) {  // the bf16 model: weight rows as they are, the hi plane = the reference's bf16 cast
        p.alo = nullptr;
        switch (epi) {
            case GE_STORE: return ring_ok ? gemm_ring_t<GE_STORE, true>(p, s) : gemm_t<GE_STORE, false, true>(p, s);
            case GE_RESID: return ring_ok ? gemm_ring_t<GE_RESID, true>(p, s) : gemm_t<GE_RESID, false, true>(p, s);
            case GE_SWIGLU: return ring_ok ? gemm_ring_t<GE_SWIGLU, true>(p, s) : gemm_t<GE_SWIGLU, false, true>(p, s);
        }
        return set_error(SCRY_ERR_INVALID, "gemm: unknown epilogue %d", epi);
    }
    if (p.ad) {
        switch (epi) {
            case GE_STORE: return gemm_digits_t<GE_STORE>(p, s);
            case GE_RESID: return gemm_digits_t<GE_RESID>(p, s);
            case GE_SWIGLU: return gemm_digits_t<GE_SWIGLU>(p, s);
        }
        return set_error(SCRY_ERR_INVALID, "gemm: unknown epilogue %d", epi);
    }
    if (b32) {
        p.scale = p.scale2 = 1.f;  // the block scales are in the sums
        const bool r = ring_ok && (size_t)p.N * p.nb * 4 < 0x7fffffffull;
        switch (epi) {
            case GE_STORE: return r ? gemm_ring_t<GE_STORE, false, true>(p, s) : gemm_t<GE_STORE, true>(p, s);
            case GE_RESID: return r ? gemm_ring_t<GE_RESID, false, true>(p, s) : gemm_t<GE_RESID, true>(p, s);
            case GE_SWIGLU: return r ? gemm_ring_t<GE_SWIGLU, false, true>(p, s) : gemm_t<GE_SWIGLU, true>(p, s);
        }
        return set_error(SCRY_ERR_INVALID, "gemm: unknown epilogue %d", epi);
    }
    if (!ring_ok) {
        switch (epi) {
            case GE_STORE: return gemm_t<GE_STORE, false>(p, s);
            case GE_RESID: return gemm_t<GE_RESID, false>(p, s);
            case GE_SWIGLU: return gemm_t<GE_SWIGLU, false>(p, s);
        }
        return set_error(SCRY_ERR_INVALID, "gemm: unknown epilogue %d", epi);
    }
    switch (epi) {
        case GE_STORE: return gemm_ring_t<GE_STORE, false>(p, s);
        case GE_RESID: return gemm_ring_t<GE_RESID, false>(p, s);
        case GE_SWIGLU: return gemm_ring_t<GE_SWIGLU, false>(p, s);
    }
    return set_error(SCRY_ERR_INVALID, "gemm: unknown epilogue %d", epi);
}

int launch_gemm_bf16(const unsigned short *w, int kp, int N, int k, const unsigned short *ahi, int lda, int M,
                     float *c, int ldc, const float *bias, hipStream_t s) {
    const int kpad = prefill_k_pad(k);
    if (kp < kpad || kp % BK) return set_error(SCRY_ERR_INVALID, "gemm_bf16: weight rows of %d < k %d", kp, k);
    if (kpad > lda || lda % 8) return set_error(SCRY_ERR_INVALID, "gemm_bf16: plane stride %d < k %d", lda, k);
    if ((size_t)N * kp * 2 >= 0x7fffffffull)
        return set_error(SCRY_ERR_UNSUPPORTED, "gemm_bf16: weight bytes above 2 GiB");
    GemmP p{};
    p.ahi = ahi;
    p.alo = nullptr;
    p.lda = lda;
    p.w = reinterpret_cast<const uint8_t *>(w);
    p.kp = kp;
    p.N = N;
    p.M = M;
    p.nk = kpad / BK;
    p.n_mb = (M + BM - 1) / BM;
    p.n_nb = (N + BN - 1) / BN;
    p.scale = 1.f;
    p.scale2 = 1.f;
    p.bias = bias;
    p.c = c;
    p.ldc = ldc;
    if ((size_t)p.n_mb * BM * p.lda * 2 < 0x7fffffffull) return gemm_ring_t<GE_STORE, true>(p, s);
    return gemm_t<GE_STORE, false, true>(p, s);
}

int launch_rope_kv(float *qkv, int ldq, int M, int seq, int qd, int kvd, int hd, const PrefillSeqs &t, int l,
                   const PrefillKVP &kp, int n_seq, hipStream_t s) {
    if (hd % 2 || qd % hd || kvd % hd) return set_error(SCRY_ERR_INVALID, "rope_kv: bad head dims");
    if (kp.kh) {
        int rmax = 0, any_old = 0;
        for (int i = 0; i < n_seq; i++) {
            rmax = std::max(rmax, t.p0[i] + seq);
            any_old |= t.p0[i] > 0;
        }
        if (rmax > kp.rows) return set_error(SCRY_ERR_INVALID, "rope_kv: %d plane rows < %d", kp.rows, rmax);
        if (any_old) {
            hipLaunchKernelGGL(k_kv_planes, dim3(1024), dim3(256), 0, s, t, l, n_seq, kvd, hd, kp);
            SCRY_HIP(hipGetLastError());
        }
    }
    bool v8 = hd % 8 == 0 && qd % 8 == 0 && kvd % 8 == 0 && ldq % 4 == 0 && (uintptr_t)qkv % 16 == 0 &&
              (!kp.kh || (uintptr_t)kp.kh % 16 == 0);
    for (int i = 0; i < n_seq && v8; i++)
        v8 = (uintptr_t)t.k[i] % 16 == 0 && (uintptr_t)t.v[i] % 16 == 0 && (uintptr_t)t.rope[i] % 16 == 0 &&
             t.ls[i] % 4 == 0;
    if (v8) {
        const size_t total8 = (size_t)M * ((qd + 2 * kvd) >> 3);
        if (total8 == 0) return SCRY_OK;
        const unsigned grid = (unsigned)std::min<size_t>((total8 + 255) / 256, 65536);
        hipLaunchKernelGGL(k_rope_kv8, dim3(grid), dim3(256), 0, s, qkv, ldq, M, seq, qd, kvd, hd, t, l, kp);
        PF_LAUNCH_CHECK();
    }
    const size_t total = (size_t)M * ((qd >> 1) + (kvd >> 1) + kvd);
    if (total == 0) return SCRY_OK;
    const unsigned grid = (unsigned)std::min<size_t>((total + 255) / 256, 65536);
    hipLaunchKernelGGL(k_rope_kv, dim3(grid), dim3(256), 0, s, qkv, ldq, M, seq, qd, kvd, hd, t, l, kp);
    PF_LAUNCH_CHECK();
}

bool attn_prefill_planes(int hd) { return hd == 64 || hd == 128; }

int launch_attn_prefill(const PrefillAttn &a, int n_seq, const PrefillSeqs &t, int l, const PrefillKVP &kv,
                        hipStream_t s) {
    if (a.hd % 2 || a.hd > 128 || a.nkv <= 0 || a.nh % a.nkv)
        return set_error(SCRY_ERR_UNSUPPORTED, "attn_prefill: head_dim %d / heads %d,%d", a.hd, a.nh, a.nkv);
    if (a.of && (!kv.kh || !attn_prefill_planes(a.hd) || (uintptr_t)a.of % 16 || a.ldo % 4))
        return set_error(SCRY_ERR_INVALID, "attn_prefill: f32 output rows need the bf16 matrix-core kernel");
    if (kv.kh && attn_prefill_planes(a.hd)) {  // bf16 matrix cores on the K / V planes
        if (a.hd == 128) return attn_bf3_t<128>(a, n_seq, t, kv, s);
        return attn_bf3_t<64>(a, n_seq, t, kv, s);
    }
    switch (a.hd) {  // matrix-core kernel for the common head sizes
        case 32: return attn_mfma_t<32>(a, n_seq, t, l, s);
        case 48: return attn_mfma_t<48>(a, n_seq, t, l, s);
        case 64: return attn_mfma_t<64>(a, n_seq, t, l, s);
        case 128: return attn_mfma_t<128>(a, n_seq, t, l, s);
        default: break;
    }
    const dim3 grid((a.seq + AQ - 1) / AQ, a.nh, n_seq);
    const size_t lds = 2 * (size_t)AK * a.hd * sizeof(float);
    const int ht = a.hd / 2;
    if (ht <= 8)
        hipLaunchKernelGGL(k_attn_prefill<8>, grid, dim3(256), lds, s, a, t, l);
    else if (ht <= 16)
        hipLaunchKernelGGL(k_attn_prefill<16>, grid, dim3(256), lds, s, a, t, l);
    else if (ht <= 32)
        hipLaunchKernelGGL(k_attn_prefill<32>, grid, dim3(256), lds, s, a, t, l);
    else
        hipLaunchKernelGGL(k_attn_prefill<64>, grid, dim3(256), lds, s, a, t, l);
    PF_LAUNCH_CHECK();
}

}  // namespace scry
