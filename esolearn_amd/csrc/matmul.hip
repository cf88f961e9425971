// f32 (batched) matmul with f64 accumulation (MathBackend::matmul in f32,
// mod.rs:54-63, and matmul_strided_batched, mod.rs:561-591; the reference's
// m > 1 fallback sums in f64, cpu.rs:875-999).  f32 products are exact in
// f64, so every kernel here differs from the sequential f64 sum only in the
// order of the additions, and rounds to f32 once.
//
//   k_mm_f64      the f64 matrix cores (v_mfma_f64_16x16x4_f64), any transpose
//   k_mv_rows     few rows of A, B stored [n][k]: one lane group per row of B
//   k_mv_cols     few rows of A, B stored [k][n]: lanes over columns
//   k_mm_reduce   adds the k splits' f64 partial sums in split order
#include <algorithm>

#include "internal.h"
#include "kdev.h"

namespace scry {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

struct MMArgs {
    const float *a, *b, *bias;  // bias [n] or null (added in f32 to the rounded sum)
    float *c;
    double *part;  // splits > 1: f64 partial sums [split][batch][m][n]
    int batch, m, k, n, splits;
    unsigned kchunk;
    int tm, tn;  // tiles
};

// ---------------------------------------------------------------- matrix cores
// A workgroup of 4 waves (2 x 2) owns a BM x BN tile of one batch entry and one
// k range.  Both operands are staged in LDS as [row][k] f32 rows of 32 k
// values (36-float stride: the 16 rows x 4 k-quads of a fragment read are 64
// distinct 16-byte slots modulo the 64 banks); lane (g, i) reads row i's k
// quad g of each 16, which feeds four MFMAs: the k order inside a step is
// permuted alike for A and B.  Bound by the f64 matrix rate (64 cycles per
// MFMA, 78.6 TFLOP/s; a library product reaches 73): values are widened on
// the way into the MFMA (one convert each), the next step's values are
// requested before the current step's MFMAs and written to the other LDS
// buffer after them (one barrier per step).
// Measured against one thread per output with a serial f64 loop: 1500 x 1280
// x 5120 (k in the middle) 341-368 us (two cards), 53-58 TFLOP/s, against about
// 10 ms; attention scores 20 x [1500 x 64] x [64 x 1500] 122-134 us against 2.7
// ms, values 111-123 us with k_mm_reduce.
constexpr int MM_T = 256, MM_BK = 32, MM_S = 36;

// KC: the operand is stored k-contiguous ([row][k], ld = k), else [k][row]
// (ld = rows).  Rows past the last are read from the last (never stored);
// k positions past the range read as zero in both operands.
//
// The f64 MFMA leaves hardly any issue slots to other vector instructions
// (counters: with 6 of them per MFMA the matrix cores were 58% busy), so the
// step loop has no branches and no clamps: a step's loads are buffer loads
// from uniform bases that the step moves, per-thread offsets are computed
// once, and the range check zeroes k positions past the range.  [row][k]: the
// offset is replaced by one past every resource.  [k][row]: k position 4 q + u
// goes through a resource of u's own, which starts at k row u and ends with the
// range (scalar instructions only: as fast as one resource and a scalar offset
// of u rows, which the compiler leaves out of what the range check promises).
// LD_QUAD reads 16 bytes along k (k % 4 == 0), LD_WORD single values; LD_WIDE
// is for matrices whose offsets inside a tile do not fit 31 bits, LD_HUGE for
// dimensions whose last tile or step ends past 2^31 - 1 (unsigned indexes, which
// made LD_WIDE 5-12% slower).
enum { LD_WIDE = 0, LD_WORD = 1, LD_QUAD = 2, LD_HUGE = 3 };

// k positions, and rows and columns at a tile's end
template <int LD>
struct Index {
    typedef int T;
};
template <>
struct Index<LD_HUGE> {
    typedef unsigned T;
};

template <int R, bool KC, int LD>
struct Stage {
    typedef typename Index<LD>::T K;
    static constexpr int N = R * MM_BK / 4 / MM_T;  // float4 per thread
    float4 v[N];
    unsigned off[N];   // bytes from the tile's first row (KC) or column at the step's k
    __device__ __forceinline__ static void slot(int j, int &row, int &q) {
        const int t = threadIdx.x;
        if (KC) {
            q = t & 7;
            row = (t >> 3) + 32 * j;
        } else {
            row = t % R;
            q = t / R + (MM_T / R) * j;
        }
    }
    __device__ __forceinline__ void init(int rows, int k, int r0) {
#pragma unroll
        for (int j = 0; j < N; j++) {
            int row, q;
            slot(j, row, q);
            const unsigned r = (unsigned)min(row, rows - 1 - r0);
            off[j] = 4u * (KC ? r * (unsigned)k + 4u * q : 4u * q * (unsigned)rows + r);
        }
    }
    // the values of step [k0, k0 + 32) of a range that ends at kend; none of
    // them is used here, or the wave would wait for the loads before the
    // MFMAs that are to hide them
    __device__ __forceinline__ void load(const float *p, int rows, int k, int r0, K k0, K kend) {
        const int left = (int)(kend - k0);
        if (LD == LD_WIDE || LD == LD_HUGE) {
#pragma unroll
            for (int j = 0; j < N; j++) {
                int row, q;
                slot(j, row, q);
                const K r = min((K)r0 + row, (K)(rows - 1));
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const K c = min(k0 + 4 * q + u, (K)(k - 1));
                    const float y = KC ? p[(size_t)r * k + c] : p[(size_t)c * rows + r];
                    (&v[j].x)[u] = left > 4 * q + u ? y : 0.f;
                }
            }
            return;
        }
        auto rsrc = [&](size_t first, int nb) {
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p) + first, (short)0, nb, 0x00020000);
        };
        if (KC) {
            constexpr unsigned past = 0x80000000u;
            // values left up to the end, capped at the resource limit (scalar 32-bit compares)
            const size_t first = (size_t)r0 * k + k0;
            const long long d = (long long)((size_t)rows * k - first);
            const int hi = (int)(d >> 29);
            const auto rs = rsrc(first, hi < 0 ? 0 : hi > 0 ? 0x7ffffffc : (int)d * 4);
#pragma unroll
            for (int j = 0; j < N; j++) {
                int row, q;
                slot(j, row, q);
                if (LD == LD_QUAD) {
                    v[j] = dev::bload16f(rs, left > 4 * q ? off[j] : past);
                } else {
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        (&v[j].x)[u] = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)(left > 4 * q + u ? off[j] + 4 * u : past), 0, 0));
                }
            }
        } else {
            // k rows of this step inside the range, from row r0 of the first on
            const int here = min(left, MM_BK) * rows - r0;  // below 2^26 (2^21 rows or columns at most)
            const size_t first = (size_t)k0 * rows + r0;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const auto rs = rsrc(first + (size_t)u * rows, 4 * max(here - u * rows, 0));
#pragma unroll
                for (int j = 0; j < N; j++)
                    (&v[j].x)[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off[j], 0, 0));
            }
        }
    }
    __device__ __forceinline__ void store(float *s) const {
#pragma unroll
        for (int j = 0; j < N; j++) {
            int row, q;
            slot(j, row, q);
            *reinterpret_cast<float4 *>(s + row * MM_S + 4 * q) = v[j];
        }
    }
};

// Two waves per SIMD at least: with at most 256 registers the compiler keeps
// the sums in vector registers; otherwise it moved all of them to accumulation
// registers and back in every step (64 moves per 32 MFMAs: 1500 x 1280 x 5120
// 385 us, now 368; attention scores 146 -> 134, values 130 -> 123).
template <int BM, int BN, bool TA, bool TB, int LD>
__global__ __launch_bounds__(MM_T, 2) void k_mm_f64(MMArgs p) {
    __shared__ __align__(16) float sa[2][BM * MM_S];
    __shared__ __align__(16) float sb[2][BN * MM_S];
    constexpr int WM = BM / 2, WN = BN / 2, NM = WM / 16, NN = WN / 16;
    // block -> (batch, split, tile): each XCD (block id mod 8) walks a
    // contiguous run of tiles, rows fastest, so its L2 keeps a B panel
    const unsigned total = (unsigned)p.tm * p.tn * p.splits * p.batch, per = (total + 7) / 8;
    for (unsigned vb = blockIdx.x; vb < 8 * per; vb += gridDim.x) {  // gridDim.x: a multiple of 8
    const unsigned w = (vb & 7) * per + (vb >> 3);
    if (w >= total) continue;
    const int it = (int)(w % p.tm), jt = (int)(w / p.tm % p.tn);
    const int sp = (int)(w / ((unsigned)p.tm * p.tn) % p.splits), bt = (int)(w / ((unsigned)p.tm * p.tn * p.splits));
    const float *A = p.a + (size_t)bt * p.m * p.k, *B = p.b + (size_t)bt * p.k * p.n;
    const int i0 = it * BM, j0 = jt * BN;
    typedef typename Index<LD>::T K;
    const K kb = (K)sp * (K)p.kchunk, ke = min((K)p.k, kb + (K)p.kchunk);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave & 1) * WM, wn = (wave >> 1) * WN;
    const int fo = (lane & 15) * MM_S + 4 * (lane >> 4);
    d4 acc[NM][NN];
#pragma unroll
    for (int x = 0; x < NM; x++)
#pragma unroll
        for (int y = 0; y < NN; y++) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    Stage<BM, !TA, LD> la;
    Stage<BN, TB, LD> lb;
    la.init(p.m, p.k, i0);
    lb.init(p.n, p.k, j0);
    la.load(A, p.m, p.k, i0, kb, ke);
    lb.load(B, p.n, p.k, j0, kb, ke);
    la.store(sa[0]);
    lb.store(sb[0]);
    __syncthreads();
    int cur = 0;
    for (K k0 = kb; k0 < ke; k0 += MM_BK) {
        la.load(A, p.m, p.k, i0, k0 + MM_BK, ke);
        lb.load(B, p.n, p.k, j0, k0 + MM_BK, ke);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float4 fa[NM], fb[NN];
#pragma unroll
            for (int x = 0; x < NM; x++)
                fa[x] = *reinterpret_cast<const float4 *>(&sa[cur][(wm + 16 * x) * MM_S + fo + 16 * h]);
#pragma unroll
            for (int y = 0; y < NN; y++)
                fb[y] = *reinterpret_cast<const float4 *>(&sb[cur][(wn + 16 * y) * MM_S + fo + 16 * h]);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                double da[NM], db[NN];
#pragma unroll
                for (int x = 0; x < NM; x++) da[x] = (double)(&fa[x].x)[r];
#pragma unroll
                for (int y = 0; y < NN; y++) db[y] = (double)(&fb[y].x)[r];
#pragma unroll
                for (int x = 0; x < NM; x++)
#pragma unroll
                    for (int y = 0; y < NN; y++)
                        acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(da[x], db[y], acc[x][y], 0, 0, 0);
            }
        }
        la.store(sa[cur ^ 1]);
        lb.store(sb[cur ^ 1]);
        __syncthreads();
        cur ^= 1;
    }
    // accumulator element r of lane (g, i): row 4 r + g, column i
    const size_t mn = (size_t)p.m * p.n;
    const int ci = lane & 15, cg = lane >> 4;
#pragma unroll
    for (int x = 0; x < NM; x++)
#pragma unroll
        for (int y = 0; y < NN; y++) {
            const K j = (K)j0 + wn + 16 * y + ci;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const K i = (K)i0 + wm + 16 * x + 4 * r + cg;
                if (i >= (K)p.m || j >= (K)p.n) continue;
                const size_t o = (size_t)i * p.n + j;
                if (p.splits > 1) {
                    p.part[((size_t)sp * p.batch + bt) * mn + o] = acc[x][y][r];
                } else {
                    const float v = (float)acc[x][y][r];
                    p.c[(size_t)bt * mn + o] = p.bias ? __fadd_rn(v, p.bias[j]) : v;
                }
            }
        }
    }
}

__global__ __launch_bounds__(256) void k_mm_reduce(const double *__restrict__ part, int splits, size_t total, int n,
                                                   const float *__restrict__ bias, float *__restrict__ c) {
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < total; t += (size_t)gridDim.x * 256) {
        double s = part[t];
        for (int i = 1; i < splits; i++) s += part[(size_t)i * total + t];
        const float v = (float)s;
        c[t] = bias ? __fadd_rn(v, bias[t % n]) : v;
    }
}

// ------------------------------------------------------------ few rows of A
// B stored [n][k]: G lanes (a power of two, 4 k values each) walk one row of
// B, MV_R rows of each lane group in flight; the f64 sums meet by shuffles.
// Bound by reading B once: A's rows stay in L1.
constexpr int MV_R = 4;

template <int MT, int G, bool VEC>
__global__ __launch_bounds__(256) void k_mv_rows(const float *__restrict__ a, const float *__restrict__ b,
                                                 const float *__restrict__ bias, int m, int k, int n, int ta,
                                                 float *__restrict__ c) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = lane / G, l = lane % G;
    const int bt = blockIdx.y;
    const float *A = a + (size_t)bt * m * k, *B = b + (size_t)bt * k * n;
    // row r of this group: j0 + r * (64 / G): a load covers 64 / G adjacent rows
    const int j0 = (blockIdx.x * 4 + wave) * (MV_R * 64 / G) + sub;
    const float *br[MV_R];
#pragma unroll
    for (int r = 0; r < MV_R; r++) br[r] = B + (size_t)min(j0 + r * (64 / G), n - 1) * k;
    double acc[MV_R][MT];
#pragma unroll
    for (int r = 0; r < MV_R; r++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[r][i] = 0.0;
    constexpr int W = VEC ? 4 : 1;
#pragma unroll 2
    for (int p = l * W; p < k; p += G * W) {
        float bv[MV_R][W], av[MT][W];
#pragma unroll
        for (int r = 0; r < MV_R; r++) {
            if (VEC)
                *reinterpret_cast<float4 *>(bv[r]) = *reinterpret_cast<const float4 *>(br[r] + p);
            else
                bv[r][0] = br[r][p];
        }
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const int ii = min(i, m - 1);
            if (VEC && !(ta && m > 1)) {
                *reinterpret_cast<float4 *>(av[i]) = *reinterpret_cast<const float4 *>(A + (size_t)ii * k + p);
            } else {
#pragma unroll
                for (int u = 0; u < W; u++) av[i][u] = ta ? A[(size_t)(p + u) * m + ii] : A[(size_t)ii * k + p + u];
            }
        }
#pragma unroll
        for (int u = 0; u < W; u++)
#pragma unroll
            for (int r = 0; r < MV_R; r++)
#pragma unroll
                for (int i = 0; i < MT; i++) acc[r][i] = fma((double)av[i][u], (double)bv[r][u], acc[r][i]);
    }
#pragma unroll
    for (int r = 0; r < MV_R; r++) {
        const int j = j0 + r * (64 / G);
#pragma unroll
        for (int i = 0; i < MT; i++) {
            double s = acc[r][i];
#pragma unroll
            for (int off = G / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
            if (l == 0 && j < n && i < m) {
                const float v = (float)s;
                c[((size_t)bt * m + i) * n + j] = bias ? __fadd_rn(v, bias[j]) : v;
            }
        }
    }
}

// B stored [k][n]: CG threads side by side own W columns each, 256 / CG k
// groups of a workgroup take every (256 / CG)-th row of its k range; the
// groups meet in LDS in a fixed order.  k splits (blockIdx.y) leave f64
// partials for k_mm_reduce.
template <int MT, int W>
__global__ __launch_bounds__(256) void k_mv_cols(const float *__restrict__ a, const float *__restrict__ b,
                                                 const float *__restrict__ bias, int batch, int m, int k, int n,
                                                 int ta, int cg, int splits, int kchunk, float *__restrict__ c,
                                                 double *__restrict__ part) {
    __shared__ double red[MT * W * 256];
    const int bt = blockIdx.z, sp = blockIdx.y, kg = 256 / cg;
    const int tc = threadIdx.x % cg, tk = threadIdx.x / cg;
    const int j0 = (blockIdx.x * cg + tc) * W;
    const float *A = a + (size_t)bt * m * k;
    const float *B = b + (size_t)bt * k * n + min(j0, n - W);
    const int kb = sp * kchunk, ke = min(k, kb + kchunk);
    double acc[MT][W];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int u = 0; u < W; u++) acc[i][u] = 0.0;
    constexpr int U = 8;  // rows in flight
    for (int p0 = kb + tk; p0 < ke; p0 += U * kg) {
        float bv[U][W], av[U][MT];
#pragma unroll
        for (int q = 0; q < U; q++) {
            const int p = min(p0 + q * kg, ke - 1);
            if (W == 4)
                *reinterpret_cast<float4 *>(bv[q]) = *reinterpret_cast<const float4 *>(B + (size_t)p * n);
            else
                bv[q][0] = B[(size_t)p * n];
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const int ii = min(i, m - 1);
                av[q][i] = ta ? A[(size_t)p * m + ii] : A[(size_t)ii * k + p];
            }
        }
#pragma unroll
        for (int q = 0; q < U; q++) {
            if (p0 + q * kg < ke) {
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int u = 0; u < W; u++) acc[i][u] = fma((double)av[q][i], (double)bv[q][u], acc[i][u]);
            }
        }
    }
    // [value][k group][column thread]: neighbouring threads on neighbouring doubles
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int u = 0; u < W; u++) red[(i * W + u) * 256 + tk * cg + tc] = acc[i][u];
    __syncthreads();
    const int cols = cg * W;
    for (int t = threadIdx.x; t < MT * cols; t += 256) {
        const int i = t / cols, col = t % cols, j = blockIdx.x * cols + col;
        if (i >= m || j >= n) continue;
        const int v0 = (i * W + col % W) * 256 + col / W;
        double s = red[v0];
        for (int g = 1; g < kg; g++) s += red[v0 + g * cg];
        const size_t o = ((size_t)bt * m + i) * n + j;
        if (splits > 1) {
            part[(size_t)sp * batch * m * n + o] = s;
        } else {
            const float v = (float)s;
            c[o] = bias ? __fadd_rn(v, bias[j]) : v;
        }
    }
}

#define LAUNCH_CHECK() SCRY_HIP(hipGetLastError()); return SCRY_OK

constexpr int kHuge = 0x7fffffff - 1024;  // up to here tiles, steps and strides end below 2^31

// parts of p (1 or more) that cover x > 0
unsigned parts(unsigned x, unsigned p) { return (x + p - 1) / p; }

int reduce_parts(const double *part, int splits, size_t total, int n, const float *bias, float *c, hipStream_t s) {
    const size_t g = (total + 255) / 256;
    hipLaunchKernelGGL(k_mm_reduce, dim3((unsigned)(g > 65536 ? 65536 : g)), dim3(256), 0, s, part, splits, total, n,
                       bias, c);
    LAUNCH_CHECK();
}

template <int T, int LD>
void mm_launch(const MMArgs &p, int ta, int tb, hipStream_t s) {
    const unsigned total = (unsigned)p.tm * p.tn * p.splits * p.batch;
    const unsigned g = std::min((total + 7) / 8 * 8, 1u << 22);  // more tiles than that: several per workgroup
    auto kern = ta ? (tb ? k_mm_f64<T, T, true, true, LD> : k_mm_f64<T, T, true, false, LD>)
                   : (tb ? k_mm_f64<T, T, false, true, LD> : k_mm_f64<T, T, false, false, LD>);
    hipLaunchKernelGGL(kern, dim3(g), dim3(MM_T), 0, s, p);
}

template <int MT, int G>
void rows_launch(bool vec, dim3 g, hipStream_t s, const float *a, const float *b, const float *bias, int m, int k,
                 int n, int ta, float *c) {
    if (vec)
        hipLaunchKernelGGL((k_mv_rows<MT, G, true>), g, dim3(256), 0, s, a, b, bias, m, k, n, ta, c);
    else
        hipLaunchKernelGGL((k_mv_rows<MT, G, false>), g, dim3(256), 0, s, a, b, bias, m, k, n, ta, c);
}

template <int MT>
int mv_rows(const float *a, const float *b, const float *bias, int batch, int m, int k, int n, int ta, float *c,
            hipStream_t s) {
    const bool vec = k % 4 == 0;
    const int lanes = vec ? k / 4 : k;  // lanes a row can use
    const int G = lanes > 32 ? 64 : lanes > 16 ? 32 : lanes > 8 ? 16 : 8;
    const int per = 4 * MV_R * 64 / G;  // rows per workgroup
    const dim3 g((n + per - 1) / per, batch);
    switch (G) {
        case 64: rows_launch<MT, 64>(vec, g, s, a, b, bias, m, k, n, ta, c); break;
        case 32: rows_launch<MT, 32>(vec, g, s, a, b, bias, m, k, n, ta, c); break;
        case 16: rows_launch<MT, 16>(vec, g, s, a, b, bias, m, k, n, ta, c); break;
        default: rows_launch<MT, 8>(vec, g, s, a, b, bias, m, k, n, ta, c); break;
    }
    LAUNCH_CHECK();
}

template <int MT>
int mv_cols(const float *a, const float *b, const float *bias, int batch, int m, int k, int n, int ta, float *c,
            hipStream_t s) {
    const int W = n % 4 == 0 ? 4 : 1;
    const int need = (n + W - 1) / W;
    const int cg = need > 32 ? 64 : need > 16 ? 32 : need > 8 ? 16 : 8, kg = 256 / cg;
    const int cb = (need + cg - 1) / cg;
    // about 1024 workgroups (4 per CU), each k group at least 16 rows
    int splits = (1024 + cb * batch - 1) / (cb * batch);
    splits = std::max(1, std::min({splits, k / (16 * kg), 64}));
    splits = (int)parts(k, parts(k, splits));  // none empty
    void *ws = nullptr;
    SCRY_TRY(split_workspace(sizeof(double) * (size_t)batch * m * n, &splits, &ws));
    const int kchunk = (int)parts(k, splits);
    const dim3 g(cb, splits, batch);
    if (W == 4)
        hipLaunchKernelGGL((k_mv_cols<MT, 4>), g, dim3(256), 0, s, a, b, bias, batch, m, k, n, ta, cg, splits, kchunk,
                           c, (double *)ws);
    else
        hipLaunchKernelGGL((k_mv_cols<MT, 1>), g, dim3(256), 0, s, a, b, bias, batch, m, k, n, ta, cg, splits, kchunk,
                           c, (double *)ws);
    SCRY_HIP(hipGetLastError());
    if (splits > 1) return reduce_parts((const double *)ws, splits, (size_t)batch * m * n, n, bias, c, s);
    return SCRY_OK;
}

}  // namespace

int launch_matmul_f32(const float *a, const float *b, int batch, int m, int k, int n, int ta, int tb,
                      const float *bias, float *c, hipStream_t s) {
    if ((size_t)batch * m * n == 0) return SCRY_OK;
    // few rows: reading B is the work and the f64 vector units keep up (the
    // batch and n limits are the grid's, k's that of int strides)
    if (m <= 4 && batch <= 65535 && n <= (1 << 26) && k <= kHuge) {
        if (tb) return m == 1   ? mv_rows<1>(a, b, bias, batch, m, k, n, ta, c, s)
                       : m == 2 ? mv_rows<2>(a, b, bias, batch, m, k, n, ta, c, s)
                                : mv_rows<4>(a, b, bias, batch, m, k, n, ta, c, s);
        return m == 1   ? mv_cols<1>(a, b, bias, batch, m, k, n, ta, c, s)
               : m == 2 ? mv_cols<2>(a, b, bias, batch, m, k, n, ta, c, s)
                        : mv_cols<4>(a, b, bias, batch, m, k, n, ta, c, s);
    }
    MMArgs p{};
    p.a = a;
    p.b = b;
    p.bias = bias;
    p.c = c;
    p.batch = batch;
    p.m = m;
    p.k = k;
    p.n = n;
    auto tiles = [&](int t) { return (size_t)batch * parts(m, t) * parts(n, t); };
    const int dim = std::max({m, n, k});
    const bool huge = dim > kHuge;
    const bool wide = dim > (1 << 21);  // 31-bit offsets: 64 rows of k, or 32 k rows of m or n values
    // 64 x 64 tiles where they fill the CUs or a long k can be split over
    // them, else 32 x 32 (12 x 200 x 200 x 64: 6 against 14 us; 64 x 4096 x
    // 4096, split: 62 against 49 us).  128 x 128 was slower everywhere
    // (1500 x 1280 x 5120: 513 against 368 us, one wave per SIMD).
    const int steps = (int)parts(k, MM_BK);
    const int t = huge ? 32 : tiles(64) >= 256 || (steps >= 64 && m > 32 && n > 32) ? 64 : 32;
    p.tm = (int)parts(m, t);
    p.tn = (int)parts(n, t);
    const size_t nt = tiles(t);
    p.splits = nt >= 512 ? 1 : (int)std::max<size_t>(1, std::min<size_t>({(512 + nt - 1) / nt, (size_t)steps / 8, 16}));
    p.splits = (int)parts(steps, parts(steps, p.splits));  // none empty
    void *ws = nullptr;
    SCRY_TRY(split_workspace(sizeof(double) * (size_t)batch * m * n, &p.splits, &ws));
    p.part = (double *)ws;
    p.kchunk = parts(steps, p.splits) * MM_BK;
    if (huge)
        mm_launch<32, LD_HUGE>(p, ta, tb, s);
    else if (wide)
        t == 32 ? mm_launch<32, LD_WIDE>(p, ta, tb, s) : mm_launch<64, LD_WIDE>(p, ta, tb, s);
    else if (k % 4 == 0)
        t == 32 ? mm_launch<32, LD_QUAD>(p, ta, tb, s) : mm_launch<64, LD_QUAD>(p, ta, tb, s);
    else
        t == 32 ? mm_launch<32, LD_WORD>(p, ta, tb, s) : mm_launch<64, LD_WORD>(p, ta, tb, s);
    SCRY_HIP(hipGetLastError());
    if (p.splits > 1) return reduce_parts(p.part, p.splits, (size_t)batch * m * n, n, bias, c, s);
    return SCRY_OK;
}

}  // namespace scry
