// Op-level glue kernels behind the MathBackend entry points (cpu.rs citations
// per kernel).  The decode step does not use these: its RMSNorm, RoPE, KV
// append, SwiGLU, residual add, embedding and argmax are fused into the GEMV
// and attention kernels.  These serve the per-op API (a Rust HipBackend's
// trait methods) and the parity tests.
#include <algorithm>

#include "internal.h"
#include "kdev.h"

namespace scry {
namespace {

inline unsigned grid1(size_t n, unsigned cap = 65536) {
    size_t g = (n + 255) / 256;
    return (unsigned)(g < 1 ? 1 : (g > cap ? cap : g));
}

#define GRID_STRIDE(i, n) \
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (size_t)gridDim.x * blockDim.x)

// cpu.rs:574-599: one workgroup per row, f64 sum of squares.  The row is read
// once, 16 bytes per load (NV loads per thread, all in flight), and kept in
// registers; few rows take 1024 threads, since one row's latency is then the
// whole kernel (in a layer: 1 x 4096 11.7 -> 3.8 us, 512 x 4096 16.3 -> 8.3 us
// against a loop of 4-byte loads read twice).
template <int NT, int NV>
__global__ __launch_bounds__(NT) void k_rmsnorm4(const float4 *__restrict__ x, const float4 *__restrict__ w, int d4,
                                                 float eps, float4 *__restrict__ out) {
    __shared__ double red[NT / 64];
    const float4 *r = x + (size_t)blockIdx.x * d4;
    float4 v[NV], g[NV];
#pragma unroll
    for (int c = 0; c < NV; c++) {
        const int j = c * NT + threadIdx.x;
        v[c] = j < d4 ? r[j] : make_float4(0.f, 0.f, 0.f, 0.f);
        g[c] = j < d4 ? w[j] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    double ss = 0.0;
#pragma unroll
    for (int c = 0; c < NV; c++)
        ss += (double)v[c].x * v[c].x + (double)v[c].y * v[c].y + ((double)v[c].z * v[c].z + (double)v[c].w * v[c].w);
    ss = dev::wave_sum_d_dpp(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int i = 0; i < NT / 64; i++) tot += red[i];
    const double rstd = 1.0 / sqrt(tot / (double)(4 * d4) + (double)eps);
#pragma unroll
    for (int c = 0; c < NV; c++) {
        const int j = c * NT + threadIdx.x;
        if (j < d4)
            out[(size_t)blockIdx.x * d4 + j] =
                make_float4((float)((double)v[c].x * rstd * (double)g[c].x), (float)((double)v[c].y * rstd * (double)g[c].y),
                            (float)((double)v[c].z * rstd * (double)g[c].z), (float)((double)v[c].w * rstd * (double)g[c].w));
    }
}
// any d
__global__ __launch_bounds__(256) void k_rmsnorm(const float *__restrict__ x,
                                                 const float *__restrict__ w, int d, float eps,
                                                 float *__restrict__ out) {
    const float *r = x + (size_t)blockIdx.x * d;
    double ss = 0.0;
    for (int j = threadIdx.x; j < d; j += 256) ss += (double)r[j] * (double)r[j];
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    __shared__ double red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const double tot = red[0] + red[1] + red[2] + red[3];
    const double rstd = 1.0 / sqrt(tot / (double)d + (double)eps);
    for (int j = threadIdx.x; j < d; j += 256)
        out[(size_t)blockIdx.x * d + j] = (float)((double)r[j] * rstd * (double)w[j]);
}

// cpu.rs:635-664 (+ mod.rs:219-230 scale): one thread per position, pair and
// group of ROPE_H heads, which share the f64 cos / sin (the time of a thread
// per rotated pair: 512 x 32 heads x 128 9.1 -> 6.0 us).
constexpr int ROPE_H = 8;
__global__ void k_rope(const float *__restrict__ x, int seq, int n_heads, int hd, int start_pos,
                       const float *__restrict__ freqs, int scaled, float scale,
                       float *__restrict__ out) {
    const int np = hd / 2, ng = (n_heads + ROPE_H - 1) / ROPE_H;
    const size_t total = (size_t)seq * ng * np;
    GRID_STRIDE(t, total) {
        const int i = (int)(t % np);
        const size_t sg = t / np;
        const int s = (int)(sg / ng), h0 = (int)(sg % ng) * ROPE_H;
        const float2 *p = reinterpret_cast<const float2 *>(x + ((size_t)s * n_heads + h0) * hd) + i;
        float2 *o = reinterpret_cast<float2 *>(out + ((size_t)s * n_heads + h0) * hd) + i;
        float2 v[ROPE_H];
#pragma unroll
        for (int h = 0; h < ROPE_H; h++) v[h] = p[(size_t)min(h, n_heads - 1 - h0) * np];
        const double ang = (double)(start_pos + s) * (double)freqs[i];
        const float c = (float)cos(ang), sn = (float)sin(ang);
#pragma unroll
        for (int h = 0; h < ROPE_H; h++) {
            // the cosine products are fused, as written: of products left to the
            // compiler it fused either, depending on the code around them, and
            // the last bit with it
            float r0 = fmaf(v[h].x, c, -__fmul_rn(v[h].y, sn));
            float r1 = fmaf(v[h].y, c, __fmul_rn(v[h].x, sn));
            if (scaled) {
                r0 = __fmul_rn(r0, scale);
                r1 = __fmul_rn(r1, scale);
            }
            if (h0 + h < n_heads) o[(size_t)h * np] = make_float2(r0, r1);
        }
    }
}

// A cache's RoPE table (cpu.rs:648-652).  Bound by the f64 cos / sin; on the
// host this table was 1 ms per 1000 positions and cache (4 caches of 1031
// positions: 4.1 of a 14 ms batch), here a few us.
__global__ void k_rope_table(const float *__restrict__ freqs, int n_pos, int half, float2 *__restrict__ cs) {
    const size_t total = (size_t)n_pos * half;
    GRID_STRIDE(t, total) {
        const double ang = (double)(t / half) * (double)freqs[t % half];
        cs[t] = make_float2((float)cos(ang), (float)sin(ang));
    }
}

// Elementwise kernels over 16-byte quads (storage blocks are 256-byte
// aligned), the last n % 4 values by the first threads: bound by HBM.
template <class F>
__device__ __forceinline__ void quads(size_t n, F f) {
    const size_t n4 = n >> 2;
    GRID_STRIDE(i, n4) f(i << 2, 4);
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) f((n4 << 2) + threadIdx.x, 1);
}
__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ void st4(float *p, float4 v) { *reinterpret_cast<float4 *>(p) = v; }

__global__ void k_scale(const float *__restrict__ x, size_t n, float s, float *__restrict__ out) {
    quads(n, [&](size_t i, int w) {
        if (w == 1) {
            out[i] = __fmul_rn(x[i], s);
            return;
        }
        const float4 a = ld4(x + i);
        st4(out + i, make_float4(__fmul_rn(a.x, s), __fmul_rn(a.y, s), __fmul_rn(a.z, s), __fmul_rn(a.w, s)));
    });
}

// x * scale rounded to f32: a product that may be contracted (as __fmul_rn's
// may) is fused into the subtraction of the maximum
__device__ __forceinline__ float scaled_value(float x, float scale) {
#pragma clang fp contract(off)
    return x * scale;
}

// softmax (cpu.rs:336-366) and scaled_softmax (cpu.rs:300-334): v = x or x *
// scale (f32), f32 max (NaN ignored), e = expf(v - max) kept as f32, f64 sum,
// out = f32(f64(e) * (1 / sum)) (within an f64 ulp of e / sum: the f64 divide
// per element was most of the time).
// W threads per row (a wave, or a workgroup of 256), NV values each in
// registers: the row is read and written once.  30000 x 1500: 186 -> 64 us
// (360 MB: 5.6 TB/s), 16384 x 512: 29 -> 14 us, against rows read three times.
template <int W, int NV, bool SCALED>
__global__ __launch_bounds__(256) void k_softmax_reg(const float *__restrict__ x, int rows, int cols, float scale,
                                                     float *__restrict__ out) {
    constexpr int RPB = 256 / W;  // rows per workgroup
    const int tid = threadIdx.x, t = tid % W;
    const size_t row = (size_t)blockIdx.x * RPB + tid / W;
    if (W == 64 && row >= (size_t)rows) return;  // (no barriers in a wave's row)
    const float *r = x + row * cols;
    float *o = out + row * cols;
    float v[NV];
    float mx = -INFINITY;
#pragma unroll
    for (int c = 0; c < NV; c++) {
        const int j = c * W + t;
        v[c] = j < cols ? r[j] : -INFINITY;
    }
#pragma unroll
    for (int c = 0; c < NV; c++) {
        if (SCALED && c * W + t < cols) v[c] = scaled_value(v[c], scale);
        mx = fmaxf(mx, v[c]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    __shared__ float redf[4];
    __shared__ double redd[4];
    if (W == 256) {
        if ((tid & 63) == 0) redf[tid >> 6] = mx;
        __syncthreads();
        mx = fmaxf(fmaxf(redf[0], redf[1]), fmaxf(redf[2], redf[3]));
    }
    double sum = 0.0;
#pragma unroll
    for (int c = 0; c < NV; c++) {
        v[c] = expf(__fsub_rn(v[c], mx));
        if (c * W + t < cols) sum += (double)v[c];
    }
    sum = dev::wave_sum_d_dpp(sum);
    if (W == 256) {
        if ((tid & 63) == 0) redd[tid >> 6] = sum;
        __syncthreads();
        sum = (redd[0] + redd[1]) + (redd[2] + redd[3]);
    }
    const double inv = 1.0 / sum;
#pragma unroll
    for (int c = 0; c < NV; c++) {
        const int j = c * W + t;
        if (j < cols) o[j] = (float)((double)v[c] * inv);
    }
}

// rows too long for registers: one workgroup per row, read three times
template <bool SCALED>
__global__ __launch_bounds__(256) void k_softmax(const float *__restrict__ x, int cols, float scale,
                                                 float *__restrict__ out) {
    const float *r = x + (size_t)blockIdx.x * cols;
    float *o = out + (size_t)blockIdx.x * cols;
    __shared__ float redf[4];
    __shared__ double redd[4];
    float mx = -INFINITY;
    for (int j = threadIdx.x; j < cols; j += 256) mx = fmaxf(mx, SCALED ? scaled_value(r[j], scale) : r[j]);
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((threadIdx.x & 63) == 0) redf[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(redf[0], redf[1]), fmaxf(redf[2], redf[3]));
    double sum = 0.0;
    for (int j = threadIdx.x; j < cols; j += 256) {
        const float e = expf(__fsub_rn(SCALED ? scaled_value(r[j], scale) : r[j], mx));
        o[j] = e;
        sum += (double)e;
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if ((threadIdx.x & 63) == 0) redd[threadIdx.x >> 6] = sum;
    __syncthreads();
    const double inv = 1.0 / ((redd[0] + redd[1]) + (redd[2] + redd[3]));
    for (int j = threadIdx.x; j < cols; j += 256) o[j] = (float)((double)o[j] * inv);
}

// cpu.rs:666-678, 1119-1122
__global__ void k_swiglu(const float *__restrict__ g, const float *__restrict__ u, size_t n,
                         float *__restrict__ out) {
    quads(n, [&](size_t i, int w) {
        if (w == 1) {
            out[i] = __fmul_rn(dev::silu_f(g[i]), u[i]);
            return;
        }
        const float4 a = ld4(g + i), b = ld4(u + i);
        st4(out + i, make_float4(__fmul_rn(dev::silu_f(a.x), b.x), __fmul_rn(dev::silu_f(a.y), b.y),
                                 __fmul_rn(dev::silu_f(a.z), b.z), __fmul_rn(dev::silu_f(a.w), b.w)));
    });
}

__global__ void k_add(const float *__restrict__ a, const float *__restrict__ b, size_t n,
                      float *__restrict__ out) {
    quads(n, [&](size_t i, int w) {
        if (w == 1) {
            out[i] = __fadd_rn(a[i], b[i]);
            return;
        }
        const float4 p = ld4(a + i), q = ld4(b + i);
        st4(out + i, make_float4(__fadd_rn(p.x, q.x), __fadd_rn(p.y, q.y), __fadd_rn(p.z, q.z), __fadd_rn(p.w, q.w)));
    });
}

// mod.rs:76-83: the bias row added to every row of c [rows, n], in place
__global__ void k_add_bias_rows(float *__restrict__ c, const float *__restrict__ bias,
                                size_t total, int n) {
    GRID_STRIDE(i, total) c[i] = __fadd_rn(c[i], bias[i % n]);
}

// cpu.rs:485-498 (ids validated on the host)
__global__ void k_embedding(const float *__restrict__ w, const int64_t *__restrict__ ids,
                            int n_ids, int dim, float *__restrict__ out) {
    const size_t total = (size_t)n_ids * dim;
    GRID_STRIDE(t, total) {
        const size_t i = t / dim, d = t % dim;
        out[t] = w[(size_t)ids[i] * dim + d];
    }
}

// cpu.rs:707-730: [max_seq, n_kv*hd] -> [n_q, L, hd].  Workgroups of KV head
// blockIdx.y read each row of theirs once, W values (16 bytes where hd % 4 ==
// 0) per thread, and write it for its n_q / n_kv query heads (32 heads x 1001
// x 128: 17.7 -> 8 us).
template <int W>
struct Vals {
    float v[W];
};
template <>
struct __align__(16) Vals<4> {
    float v[4];
};
template <int W>
__global__ void k_gather_repeat_kv(const float *__restrict__ cache, int L, int n_kv, int n_rep, int hd,
                                   float *__restrict__ out) {
    const int hw = hd / W;
    const size_t n = (size_t)L * hw;
    for (int kv = blockIdx.y; kv < n_kv; kv += gridDim.y) {
        GRID_STRIDE(t, n) {
            const size_t s = t / hw;
            const int d = (int)(t % hw) * W;
            const Vals<W> x = *reinterpret_cast<const Vals<W> *>(cache + (s * n_kv + kv) * hd + d);
            float *o = out + ((size_t)kv * n_rep * L + s) * hd + d;
            for (int r = 0; r < n_rep; r++, o += (size_t)L * hd) *reinterpret_cast<Vals<W> *>(o) = x;
        }
    }
}

// cpu.rs:680-705, the same reading of whole [seq, d_head] heads
template <int W>
__global__ void k_repeat_kv(const float *__restrict__ x, int n_kv, int n_rep, size_t hs, float *__restrict__ out) {
    const size_t n = hs / W;
    for (size_t kv = blockIdx.y; kv < (size_t)n_kv; kv += gridDim.y) {
        GRID_STRIDE(t, n) {
            const Vals<W> v = *reinterpret_cast<const Vals<W> *>(x + kv * hs + t * W);
            float *o = out + kv * n_rep * hs + t * W;
            for (int r = 0; r < n_rep; r++, o += hs) *reinterpret_cast<Vals<W> *>(o) = v;
        }
    }
}

// Logits of the int8 LM head for rows whose normalised input holds an
// infinity or a NaN.  The prefill GEMMs mark such a row and give NaN for all
// of it, while the reference's sum of f64(a) (q s) over k (cpu.rs:1128-1160)
// is +-inf per column unless a NaN term or both infinities occur; only the
// terms of the non-finite inputs decide it.  One workgroup per row:
// RMSNorm's f64 scale (cpu.rs:574-599) and the normalised values
// f32(f64(x) rstd f64(g)); a row with none non-finite is left as it is;
// otherwise each 256-position chunk's non-finite values (at most 256) are
// gathered in LDS and every column's class is folded into its logit (the
// classes combine in any order).
__global__ __launch_bounds__(256) void k_logits_nonfinite(const float *__restrict__ x, int ldx,
                                                          const float *__restrict__ g, float eps, int k,
                                                          const uint8_t *__restrict__ W, int kp,
                                                          const float *__restrict__ s32, int nb, float scale,
                                                          int n, float *__restrict__ y, int ldy) {
    __shared__ double red[4];
    __shared__ int s_cnt;
    __shared__ int s_idx[256];
    __shared__ float s_val[256];
    const int row = blockIdx.x, tid = threadIdx.x;
    const float *xr = x + (size_t)row * ldx;
    float *yr = y + (size_t)row * ldy;
    double ss = 0.0;
    for (int p = tid; p < k; p += 256) ss += (double)xr[p] * (double)xr[p];
    ss = dev::block_sum_d(ss, red);
    const double rstd = 1.0 / sqrt(ss / (double)k + (double)eps);
    bool seen = false;  // uniform: a chunk with non-finite values was folded in
    for (int p0 = 0; p0 < k; p0 += 256) {
        const int p = p0 + tid;
        float t = 0.f;
        if (p < k) t = g ? (float)((double)xr[p] * rstd * (double)g[p]) : xr[p];
        __syncthreads();
        if (tid == 0) s_cnt = 0;
        __syncthreads();
        if (p < k && !isfinite(t)) {
            const int i = atomicAdd(&s_cnt, 1);
            s_idx[i] = p;
            s_val[i] = t;
        }
        __syncthreads();
        const int cnt = s_cnt;
        if (cnt == 0) continue;
        for (int j = tid; j < n; j += 256) {
            int cls = seen ? dev::nonfinite_class(yr[j]) : 0;
            const uint8_t *wr = W + (size_t)j * kp;
            for (int i = 0; i < cnt; i++) {
                const int q = s_idx[i];
                cls |= dev::nonfinite_term(s_val[i], wr[q], s32 ? s32[(size_t)j * nb + (q >> 5)] : scale);
            }
            yr[j] = dev::nonfinite_value(cls);
        }
        seen = true;
    }
}

// Ordered argmax over one vector (generate.rs:167-173): workgroups over
// contiguous ranges, then one over their results.  One workgroup over 50257
// logits took 53 us, the two launches 6.
__global__ __launch_bounds__(dev::TPB) void k_argmax_part(const float *__restrict__ x, int n, int chunk,
                                                          dev::ArgAcc *__restrict__ part) {
    __shared__ dev::ArgAcc sh[dev::TPB];
    const int lo = (int)min((long long)blockIdx.x * chunk, (long long)n);
    const dev::ArgAcc r = dev::block_argmax_range(x, lo, lo + min(chunk, n - lo), sh);
    if (threadIdx.x == 0) part[blockIdx.x] = r;
}
__global__ __launch_bounds__(dev::TPB) void k_argmax_end(const float *__restrict__ x, int n,
                                                         const dev::ArgAcc *__restrict__ part, int np, int64_t *out) {
    __shared__ dev::ArgAcc sh[dev::TPB];
    const dev::ArgAcc a = (int)threadIdx.x < np ? part[threadIdx.x] : dev::ArgAcc{0.f, -1, -1};
    const dev::ArgAcc r = dev::block_argmax(a, sh);
    const int tok = dev::argmax_finish(r, x, n, sh);
    if (threadIdx.x == 0) *out = n <= 0 ? 0 : tok;
}

__global__ void k_fill_f32(float *p, size_t n, float v) { GRID_STRIDE(i, n) p[i] = v; }
__global__ void k_fill_u32(unsigned int *p, size_t n, unsigned int v) { GRID_STRIDE(i, n) p[i] = v; }

}  // namespace

#define LAUNCH_CHECK() SCRY_HIP(hipGetLastError()); return SCRY_OK

int launch_rmsnorm(const float *x, const float *w, int rows, int d, float eps, float *out,
                   hipStream_t s) {
    if (rows <= 0) return SCRY_OK;
    const bool v4 = d % 4 == 0 && ((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 == 0;
    const float4 *x4 = (const float4 *)x, *w4 = (const float4 *)w;
    const int d4 = d / 4;
    if (v4 && rows >= 256 && d4 <= 1024)
        hipLaunchKernelGGL((k_rmsnorm4<256, 4>), dim3(rows), dim3(256), 0, s, x4, w4, d4, eps, (float4 *)out);
    else if (v4 && d4 <= 256)
        hipLaunchKernelGGL((k_rmsnorm4<256, 1>), dim3(rows), dim3(256), 0, s, x4, w4, d4, eps, (float4 *)out);
    else if (v4 && d4 <= 1024)
        hipLaunchKernelGGL((k_rmsnorm4<1024, 1>), dim3(rows), dim3(1024), 0, s, x4, w4, d4, eps, (float4 *)out);
    else if (v4 && d4 <= 4096)
        hipLaunchKernelGGL((k_rmsnorm4<1024, 4>), dim3(rows), dim3(1024), 0, s, x4, w4, d4, eps, (float4 *)out);
    else
        hipLaunchKernelGGL(k_rmsnorm, dim3(rows), dim3(256), 0, s, x, w, d, eps, out);
    LAUNCH_CHECK();
}

int launch_rope(const float *x, int seq, int n_heads, int hd, int start_pos, const float *freqs,
                int scaled, float scale, float *out, hipStream_t s) {
    const size_t total = (size_t)seq * ((n_heads + ROPE_H - 1) / ROPE_H) * (hd / 2);
    if (total == 0) return SCRY_OK;
    hipLaunchKernelGGL(k_rope, dim3(grid1(total)), dim3(256), 0, s, x, seq, n_heads, hd, start_pos,
                       freqs, scaled, scale, out);
    LAUNCH_CHECK();
}

int launch_rope_table(const float *freqs, int n_pos, int half, float2 *cs, hipStream_t s) {
    const size_t total = (size_t)n_pos * half;
    if (total == 0) return SCRY_OK;
    hipLaunchKernelGGL(k_rope_table, dim3(grid1(total)), dim3(256), 0, s, freqs, n_pos, half, cs);
    LAUNCH_CHECK();
}

int launch_scale(const float *x, size_t n, float sc, float *out, hipStream_t s) {
    if (n == 0) return SCRY_OK;
    hipLaunchKernelGGL(k_scale, dim3(grid1((n + 3) / 4)), dim3(256), 0, s, x, n, sc, out);
    LAUNCH_CHECK();
}

namespace {
template <bool SCALED>
int softmax_rows(const float *x, int rows, int cols, float scale, float *out, hipStream_t s) {
    if (rows <= 0 || cols <= 0) return SCRY_OK;
    // a wave per row once there are rows for every CU's waves, else a workgroup
#define SM_LAUNCH(W, NV) \
    hipLaunchKernelGGL((k_softmax_reg<W, NV, SCALED>), dim3((rows + 256 / W - 1) / (256 / W)), dim3(256), 0, s, x, rows, cols, scale, out)
    if (rows >= 1024 && cols <= 2048) {
        if (cols <= 256) SM_LAUNCH(64, 4);
        else if (cols <= 512) SM_LAUNCH(64, 8);
        else if (cols <= 1024) SM_LAUNCH(64, 16);
        else SM_LAUNCH(64, 32);
    } else if (cols <= 8192) {
        if (cols <= 1024) SM_LAUNCH(256, 4);
        else if (cols <= 2048) SM_LAUNCH(256, 8);
        else if (cols <= 4096) SM_LAUNCH(256, 16);
        else SM_LAUNCH(256, 32);
    } else {
        hipLaunchKernelGGL((k_softmax<SCALED>), dim3(rows), dim3(256), 0, s, x, cols, scale, out);
    }
#undef SM_LAUNCH
    LAUNCH_CHECK();
}
}  // namespace

int launch_softmax(const float *x, int rows, int cols, float *out, hipStream_t s) {
    return softmax_rows<false>(x, rows, cols, 1.f, out, s);
}

int launch_scaled_softmax(const float *x, int rows, int cols, float scale, float *out, hipStream_t s) {
    return softmax_rows<true>(x, rows, cols, scale, out, s);
}

int launch_swiglu(const float *g, const float *u, size_t n, float *out, hipStream_t s) {
    if (n == 0) return SCRY_OK;
    hipLaunchKernelGGL(k_swiglu, dim3(grid1((n + 3) / 4)), dim3(256), 0, s, g, u, n, out);
    LAUNCH_CHECK();
}

int launch_add(const float *a, const float *b, size_t n, float *out, hipStream_t s) {
    if (n == 0) return SCRY_OK;
    hipLaunchKernelGGL(k_add, dim3(grid1((n + 3) / 4)), dim3(256), 0, s, a, b, n, out);
    LAUNCH_CHECK();
}

int launch_add_bias_rows(float *c, const float *bias, int rows, int n, hipStream_t s) {
    const size_t total = (size_t)rows * n;
    if (total == 0) return SCRY_OK;
    hipLaunchKernelGGL(k_add_bias_rows, dim3(grid1(total)), dim3(256), 0, s, c, bias, total, n);
    LAUNCH_CHECK();
}

int launch_embedding(const float *w, const int64_t *ids, int n_ids, int dim, float *out,
                     hipStream_t s) {
    const size_t total = (size_t)n_ids * dim;
    if (total == 0) return SCRY_OK;
    hipLaunchKernelGGL(k_embedding, dim3(grid1(total)), dim3(256), 0, s, w, ids, n_ids, dim, out);
    LAUNCH_CHECK();
}

int launch_gather_repeat_kv(const float *cache, int cached_len, int n_kv, int n_q, int hd,
                            float *out, hipStream_t s) {
    const size_t total = (size_t)n_q * cached_len * hd;
    if (total == 0) return SCRY_OK;
    const int n_rep = n_q / n_kv, gy = n_kv < 65535 ? n_kv : 65535;
    if (hd % 4 == 0)
        hipLaunchKernelGGL(k_gather_repeat_kv<4>, dim3(grid1((size_t)cached_len * hd / 4, 4096), gy), dim3(256), 0, s,
                           cache, cached_len, n_kv, n_rep, hd, out);
    else
        hipLaunchKernelGGL(k_gather_repeat_kv<1>, dim3(grid1((size_t)cached_len * hd, 4096), gy), dim3(256), 0, s,
                           cache, cached_len, n_kv, n_rep, hd, out);
    LAUNCH_CHECK();
}

int launch_repeat_kv(const float *x, int n_kv, int n_q, int seq, int d_head, float *out,
                     hipStream_t s) {
    const size_t hs = (size_t)seq * d_head, total = (size_t)n_q * hs;
    if (total == 0) return SCRY_OK;
    const int n_rep = n_q / n_kv, gy = n_kv < 65535 ? n_kv : 65535;
    if (hs % 4 == 0)
        hipLaunchKernelGGL(k_repeat_kv<4>, dim3(grid1(hs / 4, 4096), gy), dim3(256), 0, s, x, n_kv, n_rep, hs, out);
    else
        hipLaunchKernelGGL(k_repeat_kv<1>, dim3(grid1(hs, 4096), gy), dim3(256), 0, s, x, n_kv, n_rep, hs, out);
    LAUNCH_CHECK();
}

int launch_logits_nonfinite(const float *x, int ldx, int rows, const float *norm_w, float eps, const Packed &w,
                            float *y, int ldy, hipStream_t s) {
    if (rows <= 0 || w.bf16) return SCRY_OK;  // bf16 rows: the GEMM's products already give +-inf
    hipLaunchKernelGGL(k_logits_nonfinite, dim3(rows), dim3(256), 0, s, x, ldx, norm_w, eps, w.k, w.d, w.kp, w.s32,
                       w.nb, w.scale, w.rows, y, ldy);
    LAUNCH_CHECK();
}

int launch_argmax(const float *x, int64_t n, int64_t *out, void *part, hipStream_t s) {
    static_assert(sizeof(dev::ArgAcc) * dev::TPB <= kArgmaxScratch, "argmax scratch");
    if (n > 0x7fffffff) return set_error(SCRY_ERR_UNSUPPORTED, "argmax: n too large");
    const int np = (int)std::min<int64_t>(dev::TPB, std::max<int64_t>(1, (n + 1023) / 1024));
    const int chunk = (int)((n + np - 1) / np);
    hipLaunchKernelGGL(k_argmax_part, dim3(np), dim3(dev::TPB), 0, s, x, (int)n, chunk, (dev::ArgAcc *)part);
    hipLaunchKernelGGL(k_argmax_end, dim3(1), dim3(dev::TPB), 0, s, x, (int)n, (const dev::ArgAcc *)part, np, out);
    LAUNCH_CHECK();
}

int launch_fill_f32(float *p, size_t n, float v, hipStream_t s) {
    if (n == 0) return SCRY_OK;
    hipLaunchKernelGGL(k_fill_f32, dim3(grid1(n)), dim3(256), 0, s, p, n, v);
    LAUNCH_CHECK();
}

int launch_fill_u32(unsigned int *p, size_t n, unsigned int v, hipStream_t s) {
    if (n == 0) return SCRY_OK;
    hipLaunchKernelGGL(k_fill_u32, dim3(grid1(n)), dim3(256), 0, s, p, n, v);
    LAUNCH_CHECK();
}

}  // namespace scry
