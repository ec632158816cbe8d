// (f) Global extended Kalman filter update of the MLP weights on the device.
//
// Replaces KalmanFilter.update_state_vector
// (potentials/nnp/kalman_filter.py:196-233).  With n_w weights (all elements,
// one state vector) and m observations of one structure (m = 1 for the
// energy, m = 3 N for the force components):
//
//   X = P H                                 n_w x m
//   A = H^T X + r I = L L^T                 m x m     k_gemm_f64, chol_lower
//   [Z; z^T] = [X; xi^T] L^-T               rows carried by the factorisation
//   P = c (P - Z Z^T) + q I,  W = W + Z z   (K = X A^-1, K X^T = Z Z^T, K xi = Z z)
//
// r is the measurement noise (1/eta for the filter of type 0, lambda for
// type 1), c the fading-memory factor (1 or 1/lambda) and q the process
// noise; the schedules of eta, q and lambda are host scalars.  The
// reference forms inv(A) and multiplies; the Cholesky factor gives the same
// K (A is symmetric positive definite: H^T P H is semi-definite and r > 0)
// without forming the inverse.
//
// With more observations than weights (m > n_w: the force update of a large
// structure) the same update is computed through n_w x n_w factors instead
// of m x m ones.  With P = L L^T and G = L^T H, A = G^T G + r I, and by the
// push-through identity K = X A^-1 = L S^-1 G with S = G G^T + r I (n_w x n_w),
// so that P - K X^T = r L S^-1 L^T.  With S = Ls Ls^T and M = L Ls^-T:
//
//   L = chol(P)
//   G = L^T H                               n_w x m
//   S = G G^T + r I = Ls Ls^T,  [M; y^T] = [L; (G xi)^T] Ls^-T   (one factorisation)
//   W = W + M y  (= L S^-1 G xi),  P = c r M M^T + q I
//
// about 2 n_w^2 m + 8/3 n_w^3 flops against 3 n_w^2 m + 2 m^2 n_w + m^3 / 3,
// and factorisations of n_w rows instead of m.  All matrices are column-major FP64:
// P (n_w x n_w, ld n_w) and H (n_w x m, ld ldh) -- H column o is the
// gradient of observation o, i.e. a row-major (m x n_w) Jacobian.
//
// Every product and factorisation is a kernel of this file: the library's
// triangular kernels and its many small products per block took most of the
// update (student network, n_w = 1,698, m = 4,608: 11.0 ms, now 2.2).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"

namespace pt {
namespace {

// M ((n + 1) x n, ld ldm > n) = the lower triangle of A (zeros above) with g^T as its last row
__global__ void k_lower_copy(int n, const double* __restrict__ A, long long lda, const double* __restrict__ g,
                             double* __restrict__ M, long long ldm) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;   // row
    const int j = blockIdx.y;                             // column
    if (i < n) M[(size_t)j * ldm + i] = i >= j ? A[(size_t)j * lda + i] : 0.0;
    else if (i == n) M[(size_t)j * ldm + n] = g[j];
}

// the first of two factorisations' info codes that is not zero
__global__ void k_merge_info(int* __restrict__ info, const int* __restrict__ info2) {
    if (threadIdx.x == 0 && *info == 0) *info = *info2;
}

// dst[i * ldd] = src[i]
__global__ void k_set_row(int n, const double* __restrict__ src, double* __restrict__ dst, long long ldd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[(size_t)i * ldd] = src[i];
}

// One observation: a = h . x + r with x = P h; x -> x / sqrt(a), z = xi / sqrt(a).  One workgroup.
__global__ __launch_bounds__(1024) void k_one_obs(int n, const double* __restrict__ h, double* __restrict__ x,
                                                  const double* __restrict__ xi, double r, double* __restrict__ z,
                                                  int* __restrict__ info) {
    __shared__ double part[16];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 1024) s += h[i] * x[i];
    s = wave_sum(s);
    if (wave_lane() == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    double a = r;
    for (int q = 0; q < 16; ++q) a += part[q];
    const double ir = 1.0 / sqrt(a);
    for (int i = threadIdx.x; i < n; i += 1024) x[i] *= ir;
    if (threadIdx.x == 0) {
        *z = *xi * ir;
        *info = a > 0.0 ? 0 : 1;
    }
}

// ---- FP64 products on the matrix cores -------------------------------------
//
// C (M x N) = alpha A B + beta C [+ diag I], column-major, one workgroup of four
// wavefronts per 64 x 64 tile (a 2 x 2 block of 16 x 16 MFMA tiles per
// wavefront).  K runs in chunks of 16
// through LDS; loads are issued two chunks ahead (a chunk's products take about
// the latency of a load that misses L2).  Bound: the matrix cores.  A CU needs four
// workgroups to keep them fed (one wavefront per SIMD each), so products of fewer
// tiles split K over blockIdx.z: every part goes to its slice of `part`, k_gemm_sum adds them in
// order.  Measured, one part | split: 1,698 x 1,698 x 4,608 (lower half) 503 | 313 + 11 us
// = 41 TFLOP/s of the 64 that a large product reaches, x 1,698 188 | 120 + 13, 1,698 x 576 x 1,698
// 91 (in 32 x 32 tiles) | 75 + 10.  The
// operands' layouts are compile-time: LA = 0: A(r, k) at r + k lda, 1: at
// k + r lda; LB = 0: B(k, c) at c + k ldb, 1: at k + c ldb.  LDS holds [k][row]
// with rows T + 1 doubles apart (both the column-wise stores of a k-contiguous
// operand and the fragment reads then spread over the banks).
// lower: only tiles on or below the diagonal, each also written transposed when
// mirror is set (symmetric results).  tri: A is a lower triangle read
// transposed (LA = 1): k starts at the tile's first row and entries k < r
// count as zero.
constexpr int kKc = 16;
typedef double mf_d4 __attribute__((ext_vector_type(4)));

struct GemmArgs {
    int M, N, K;
    const double* A;
    long long lda;
    const double* B;
    long long ldb;
    double* C;
    long long ldc;
    double alpha, beta, diag;
    int lower, mirror, tri;
    int split;       // parts of K (a slice of part each, M x N)
    double* part;
};

template <int LA, int LB>
__global__ __launch_bounds__(256) void k_gemm_f64(GemmArgs g) {
    constexpr int T = 64, W = T / 32;             // MFMA tiles per wavefront and dimension
    constexpr int LDP = T + 1;
    constexpr int PER = T * kKc / 256;    // elements per thread, chunk and operand
    __shared__ double sA[2][kKc * LDP], sB[2][kKc * LDP];
    // (a triangle's longest rows, the first ones, start first)
    const int r0 = (g.tri ? blockIdx.y : blockIdx.x) * T, c0 = (g.tri ? blockIdx.x : blockIdx.y) * T;
    if (g.lower && r0 + T <= c0) return;
    const int l = wave_lane(), wv = uniform(threadIdx.x >> 6);
    const int row = l & 15, grp = l >> 4;
    const int wr = (wv & 1) * 16 * W, wc = (wv >> 1) * 16 * W;
    // this part's columns: whole chunks, the last part takes the remainder
    const int k_begin = g.tri ? r0 / kKc * kKc : 0, chunks = max(0, (g.K - k_begin) / kKc);
    const int per = (chunks + g.split - 1) / g.split, first = min((int)blockIdx.z * per, chunks);
    const int kb = k_begin + first * kKc, nk = min(per, chunks - first);
    const bool last_part = (int)blockIdx.z == g.split - 1;
    struct Chunk {
        double a[PER], b[PER];
    };
    // the thread's elements of chunk 0 and the way to the next chunk (rows and columns
    // past the end repeat the last one: their products are not stored)
    const double *pa[PER], *pb[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int t = threadIdx.x + 256 * i;
        const size_t ka = kb + (LA ? t % kKc : t / T), ra = min(r0 + (LA ? t / kKc : t % T), g.M - 1);
        const size_t kc = kb + (LB ? t % kKc : t / T), cb = min(c0 + (LB ? t / kKc : t % T), g.N - 1);
        pa[i] = g.A + (LA ? ka + ra * g.lda : ra + ka * g.lda);
        pb[i] = g.B + (LB ? kc + cb * g.ldb : cb + kc * g.ldb);
    }
    // loads a chunk and moves on by `chunks` (the last whole chunk is loaded again past the end)
    auto fetch = [&](Chunk& v, int chunks) {
        const long long da = LA ? kKc * chunks : kKc * chunks * g.lda, db = LB ? kKc * chunks : kKc * chunks * g.ldb;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            v.a[i] = *pa[i];
            v.b[i] = *pb[i];
            pa[i] += da;
            pb[i] += db;
        }
    };
    auto put = [&](const Chunk& v, int s, int k0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int t = threadIdx.x + 256 * i;
            const int ka = LA ? t % kKc : t / T, ra = LA ? t / kKc : t % T;
            sA[s][ka * LDP + ra] = LA && g.tri && k0 + ka < r0 + ra ? 0.0 : v.a[i];
            sB[s][(LB ? t % kKc : t / T) * LDP + (LB ? t / kKc : t % T)] = v.b[i];
        }
    };
    mf_d4 acc[W][W] = {};
    auto products = [&](int s) {
        double a[kKc / 4][W], b[kKc / 4][W];
#pragma unroll
        for (int k = 0; k < kKc / 4; ++k)
#pragma unroll
            for (int i = 0; i < W; ++i) {
                a[k][i] = sA[s][(4 * k + grp) * LDP + wr + 16 * i + row];
                b[k][i] = sB[s][(4 * k + grp) * LDP + wc + 16 * i + row];
            }
#pragma unroll
        for (int k = 0; k < kKc / 4; ++k)
#pragma unroll
            for (int i = 0; i < W; ++i)
#pragma unroll
                for (int j = 0; j < W; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[k][j], a[k][i], acc[i][j], 0, 0, 0);
    };
    // chunk c: products from LDS buffer c & 1; chunk c + 1 goes from registers to
    // the other buffer (last read before the barrier), chunk c + 2 is loaded.  No
    // branch around a load: the wait at its use would cover every later load too.
    if (nk > 0) {
        Chunk u, v;
        fetch(u, nk > 1);
        put(u, 0, kb);
        fetch(u, nk > 2);
        __syncthreads();
        for (int c = 0;; c += 2) {
            fetch(v, c + 3 < nk);
            products(0);
            put(u, 1, kb + (c + 1) * kKc);
            __syncthreads();
            if (c + 1 >= nk) break;
            fetch(u, c + 4 < nk);
            products(1);
            put(v, 0, kb + (c + 2) * kKc);
            __syncthreads();
            if (c + 2 >= nk) break;
        }
    }
    const int kr = kb + nk * kKc;
    if (last_part && kr < g.K) {   // the last columns, fewer than a chunk
        for (int t = threadIdx.x; t < T * kKc; t += 256) {
            const int ka = kr + t / T, ra = r0 + t % T, cb = c0 + t % T;
            const bool in = ka < g.K;
            sA[0][t / T * LDP + t % T] =
                in && ra < g.M && !(LA && g.tri && ka < ra) ? g.A[LA ? ka + ra * (size_t)g.lda : ra + ka * (size_t)g.lda] : 0.0;
            sB[0][t / T * LDP + t % T] = in && cb < g.N ? g.B[LB ? ka + cb * (size_t)g.ldb : cb + ka * (size_t)g.ldb] : 0.0;
        }
        __syncthreads();
        products(0);
    }
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
        for (int j = 0; j < W; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = r0 + wr + 16 * i + row, cc = c0 + wc + 16 * j + grp + 4 * q;
                if (r >= g.M || cc >= g.N || (g.lower && r < cc)) continue;
                if (g.split > 1) {
                    g.part[((size_t)blockIdx.z * g.N + cc) * g.M + r] = acc[i][j][q];
                    continue;
                }
                const double p = g.alpha * acc[i][j][q] + (r == cc ? g.diag : 0.0);
                double* o = g.C + r + (size_t)cc * g.ldc;
                *o = g.beta != 0.0 ? p + g.beta * *o : p;
                if (g.mirror && r > cc) {
                    o = g.C + cc + (size_t)r * g.ldc;
                    *o = g.beta != 0.0 ? p + g.beta * *o : p;
                }
            }
}

// The parts' sums into C, as the single-part kernel stores its products: 32 x 32 entries per
// workgroup, the mirrored ones through LDS so that both go to consecutive addresses (written
// straight from the lower triangle they took 49 us at 1,698 x 1,698, not 17).
__global__ __launch_bounds__(256) void k_gemm_sum(GemmArgs g) {
    __shared__ double tile[32][33];
    const int r0 = blockIdx.x * 32, c0 = blockIdx.y * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    if (g.lower && r0 + 32 <= c0) return;
    const int r = r0 + tx;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int cc = c0 + ty + 8 * q;
        if (r >= g.M || cc >= g.N || (g.lower && r < cc)) continue;
        double s = 0.0;
        for (int z = 0; z < g.split; ++z) s += g.part[((size_t)z * g.N + cc) * g.M + r];
        const double p = g.alpha * s + (r == cc ? g.diag : 0.0);
        double* o = g.C + r + (size_t)cc * g.ldc;
        *o = g.beta != 0.0 ? p + g.beta * *o : p;
        tile[ty + 8 * q][tx] = p;
    }
    if (!g.mirror) return;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int rr = r0 + ty + 8 * q, cc = c0 + tx;   // entry (rr, cc) of the triangle to (cc, rr)
        if (rr >= g.M || cc >= g.N || rr <= cc) continue;
        const double p = tile[tx][ty + 8 * q];
        double* o = g.C + cc + (size_t)rr * g.ldc;
        *o = g.beta != 0.0 ? p + g.beta * *o : p;
    }
}

// Workgroups that fill the chip (four per CU), most parts of a product, chunks of K that a
// part has at least (below that its start and its part's way through memory cost more than it saves)
constexpr int kGemmFill = 1024, kGemmParts = 8, kGemmChunks = 12;

long long gemm_tiles(const GemmArgs& g) {
    const long long r = (g.M + 63) / 64, c = (g.N + 63) / 64;
    return g.lower ? r * (r + 1) / 2 : r * c;
}

int gemm_parts(const GemmArgs& g) {
    if (g.tri) return 1;
    const long long want = (kGemmFill + gemm_tiles(g) - 1) / gemm_tiles(g);
    return (int)std::max(1LL, std::min({want, (long long)kGemmParts, (long long)(g.K / kKc / kGemmChunks)}));
}

// Doubles that the parts of any product of at most n x n results take: gemm_parts < fill /
// tiles + 1, and a result has at most 2 x 64 x 64 entries per tile (lower: half the tiles of
// a full one).  Not less for a smaller product, so a workspace serves all up to its size.
size_t gemm_part_doubles(int n) {
    const long long r = (n + 63) / 64;
    const long long by_tiles = 2LL * 64 * 64 * (kGemmFill + std::min<long long>(kGemmFill, r * r));
    return (size_t)std::min<long long>((long long)kGemmParts * n * n, by_tiles);
}

template <int LA, int LB>
int gemm_f64(GemmArgs g, double* part, hipStream_t st) {
    g.split = gemm_parts(g);
    g.part = part;
    const dim3 rc((g.M + 63) / 64, (g.N + 63) / 64, g.split), cr((g.N + 63) / 64, (g.M + 63) / 64, 1);
    hipLaunchKernelGGL((k_gemm_f64<LA, LB>), g.tri ? cr : rc, dim3(256), 0, st, g);
    if (g.split > 1) hipLaunchKernelGGL(k_gemm_sum, dim3((g.M + 31) / 32, (g.N + 31) / 32), dim3(256), 0, st, g);
    return launch_check("k_gemm_f64");
}

// ---- Cholesky factorisation A = L L^T (lower, in place), right-looking in
// blocks of 64 columns, one launch per block (k_chol_step).  A may carry further
// rows below its n x n part (rows n .. rows - 1): they come out as B L^-T, the
// triangular solve with the factor, at the cost of more tiles in the same launches.
//
// The launch of block k holds two kinds of workgroups, both starting from the
// finished columns of block k - 1:
//  * a strip: 64 rows of block k's own columns.  It applies block k - 1 to them and
//    to the 64 x 64 diagonal block (MFMA),
//    factorises the diagonal block itself (in LDS; a launch and a round trip
//    through memory cost more than the repeated work) and solves its rows.  The last
//    two go in 16-column steps: two wavefronts factorise the 16 x 16 diagonal
//    block, each with the rows of its own below it (the rest of the block, the
//    strip's rows) -- panel16 -- and all subtract the step's products from the
//    columns to the right by MFMA;
//  * a tile: 64 x 64 entries further right, from which block k - 1 is subtracted.
// Nothing that a workgroup writes is read by another of the same launch.  What
// bounds it: the serial chain of the 64 pivots; the tiles run beside it.  Measured per
// block at n = 1,698: 22.4 us, with 1,699 rows carried 25.6 (as two launches, panel
// and trailing update, 15.4 + 8 to 20 and a launch more); 16.5 without a block before it.
constexpr int kNb = 64, kSb = 16, kLd = kNb + 1;

// lane C's value of each 16-lane row, in every lane of the row
template <int C>
__device__ __forceinline__ double row_bcast(double v) {
    const long long u = __builtin_bit_cast(long long, v);
    const long long r = __builtin_amdgcn_update_dpp(0LL, u, 0x150 + C, 0xF, 0xF, true);   // row_newbcast:C
    return __builtin_bit_cast(double, r);
}

template <int B, int N, typename F>
__device__ __forceinline__ void static_range(F&& f) {
    if constexpr (B < N) {
        f(std::integral_constant<int, B>{});
        static_range<B + 1, N>(f);
    }
}

// 1 / sqrt(p): the hardware estimate with two Newton steps (a third of the latency
// of a root and a division), on p scaled by an even power of two into [1/2, 2), so
// that every positive p is in the estimate's range.  Not positive -> NaN.
__device__ __forceinline__ double pivot_rsqrt(double p) {
    const int e = __builtin_amdgcn_frexp_exp(p) & ~1;
    const double m = __builtin_amdgcn_ldexp(p, -e), h = 0.5 * m;
    double y = __builtin_amdgcn_rsq(m);
    y = y * fma(-h, y * y, 1.5);
    y = y * fma(-h, y * y, 1.5);
    y = __builtin_amdgcn_ldexp(y, -(e >> 1));
    return p > 1.7976931348623157e308 ? 0.0 : y;
}

// A 16-column step of one wavefront: a (lane l of each 16-lane row holds row l of
// the 16 x 16 diagonal block, the same in all four) -> its Cholesky factor, x (a
// row of the panel per lane) -> x L^-T; the entries of other rows come by a row
// broadcast, one for both.  The next column and its pivot's chain come before the
// other columns' products, which then fill that chain's gaps.  Returns the 1-based
// column of the first pivot that is not positive, else 0.
__device__ __forceinline__ int panel16(double (&a)[kSb], double (&x)[kSb]) {
    const int l = wave_lane() & (kSb - 1);
    double rd = pivot_rsqrt(row_bcast<0>(a[0]));
    static_range<0, kSb>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        a[j] *= rd;                        // (the pivot's own lane: p / sqrt(p))
        x[j] *= rd;
        if constexpr (j + 1 < kSb) {
            const double f = row_bcast<j + 1>(a[j]);
            a[j + 1] = fma(-a[j], f, a[j + 1]);
            x[j + 1] = fma(-x[j], f, x[j + 1]);
            rd = pivot_rsqrt(row_bcast<j + 1>(a[j + 1]));
            static_range<j + 2, kSb>([&](auto cc) {
                constexpr int c = decltype(cc)::value;
                const double g = row_bcast<c>(a[j]);
                a[c] = fma(-a[j], g, a[c]);
                x[c] = fma(-x[j], g, x[c]);
            });
            __builtin_amdgcn_sched_barrier(0);
        }
    });
    double d = a[0];
#pragma unroll
    for (int c = 1; c < kSb; ++c) d = l == c ? a[c] : d;
    const unsigned long long m = __ballot(!(d > 0.0)) & 0xFFFFull;
    return m ? __ffsll(m) : 0;
}

// acc += s * X(16 rows at x, stride ldx) Y(16 rows at y, stride ldy)^T over 16 columns
__device__ __forceinline__ mf_d4 mul16(const double* x, int ldx, const double* y, int ldy, double s, mf_d4 acc) {
    const int row = wave_lane() & 15, grp = wave_lane() >> 4;
#pragma unroll
    for (int k = 0; k < kSb; k += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(s * x[row * ldx + k + grp], y[row * ldy + k + grp], acc, 0, 0, 0);
    return acc;
}

__device__ __forceinline__ mf_d4 tile_load(const double* x) {
    const int row = wave_lane() & 15, grp = wave_lane() >> 4;
    mf_d4 v;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = x[(grp + 4 * q) * kLd + row];
    return v;
}

__device__ __forceinline__ void tile_store(double* x, const mf_d4& v) {
    const int row = wave_lane() & 15, grp = wave_lane() >> 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) x[(grp + 4 * q) * kLd + row] = v[q];
}

constexpr size_t kStepLds = sizeof(double) * 2 * kNb * kLd;   // a strip's diagonal block and rows; a tile's operands

constexpr int kStepThreads = 512;

// Rows x0 .. x0 + 63 (the last one xmax repeated past the end) of the 64 columns from kp,
// one thread's part: entry i is row t % 64 of column t / 64, t = thread + kStepThreads i
constexpr int kStepPer = kNb * kNb / kStepThreads;

__device__ __forceinline__ void block_fetch(const double* __restrict__ A, long long lda, int kp, int x0, int xmax,
                                            double (&v)[kStepPer]) {
    const double* p = A + min(x0 + (int)(threadIdx.x % kNb), xmax) + (size_t)(kp + threadIdx.x / kNb) * lda;
#pragma unroll
    for (int i = 0; i < kStepPer; ++i) v[i] = p[(size_t)(i * (kStepThreads / kNb)) * lda];
}

// into LDS as [column][row]
__device__ __forceinline__ void block_put(double* s, const double (&v)[kStepPer]) {
#pragma unroll
    for (int i = 0; i < kStepPer; ++i) {
        const int t = threadIdx.x + kStepThreads * i;
        s[t / kNb * kLd + t % kNb] = v[i];
    }
}

// acc[j] += sum over the 64 columns of x(row) y(16 j + row): x, y point at the first row of such a block's tiles
template <int N, int M>
__device__ __forceinline__ void block_products(const double* x, const double* y, mf_d4 (&acc)[M]) {
    const int row = wave_lane() & 15, grp = wave_lane() >> 4;
#pragma unroll 4
    for (int k = 0; k < kNb; k += 4) {
        const double a = x[(k + grp) * kLd + row];
#pragma unroll
        for (int j = 0; j < N; ++j)
            acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[(k + grp) * kLd + 16 * j + row], a, acc[j], 0, 0, 0);
    }
}

__device__ __forceinline__ void chol_strip(int rows, int n, double* __restrict__ A, long long lda, int k0, int strip,
                                           double* __restrict__ Ldiag, int* __restrict__ info, double* sm) {
    double* D = sm;                        // diagonal block, row-major (lower 16 x 16 tiles)
    double* X = sm + kNb * kLd;            // this workgroup's 64 rows of the block's columns
    const int nb = min(kNb, n - k0);
    const int wv = uniform(threadIdx.x >> 6);
    const int R0 = k0 + nb + strip * kNb;
    const int nr = max(0, min(kNb, rows - R0));
    if (strip == 0 && k0 > 0) {
        // the factor of the previous diagonal block goes to its place (until now other
        // workgroups read the unfactorised one); thread t reads what it overwrites below
        for (int t = threadIdx.x; t < kNb * kNb; t += kStepThreads) {
            const int r = t % kNb, c = t / kNb;
            if (c <= r) A[k0 - kNb + r + (size_t)(k0 - kNb + c) * lda] = Ldiag[t];
        }
    }
    {
        // wavefront w < 4: row tile w of the diagonal block, column tiles 0 .. w; w >= 4: row tile w - 4 of the strip
        const bool diag = wv < 4;
        const int t = wv & 3, nu = diag ? t + 1 : 4;
        const int x = (diag ? k0 : R0) + 16 * t, xmax = diag ? k0 + nb - 1 : rows - 1;
        const int l = wave_lane(), row = l & 15, grp = l >> 4;
        double old[4][4], vd[kStepPer], vx[kStepPer];
        if (k0 > 0) {
            block_fetch(A, lda, k0 - kNb, k0, k0 + nb - 1, vd);
            block_fetch(A, lda, k0 - kNb, R0, rows - 1, vx);
        }
        const double* px = A + min(x + row, xmax);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) old[u][q] = px[(size_t)min(k0 + 16 * u + grp + 4 * q, n - 1) * lda];
        mf_d4 acc[4] = {};
        if (k0 > 0) {
            block_put(D, vd);
            block_put(X, vx);
            __syncthreads();
            const double* xo = (diag ? D : X) + 16 * t;
            if (nu == 4) block_products<4>(xo, D, acc);
            else if (nu == 3) block_products<3>(xo, D, acc);
            else if (nu == 2) block_products<2>(xo, D, acc);
            else block_products<1>(xo, D, acc);
            __syncthreads();   // the operands' LDS becomes the block's and the strip's
        }
        // (a block of fewer columns is completed with the unit matrix)
        const int r = 16 * t + row;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (u < nu) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int c = 16 * u + grp + 4 * q;
                    const double v = old[u][q] - acc[u][q];
                    if (diag) D[r * kLd + c] = r < nb && c <= r ? v : (r == c ? 1.0 : 0.0);
                    else X[r * kLd + c] = r < nr && c < nb ? v : 0.0;
                }
            }
        }
    }
    __syncthreads();
    int bad = 0;
    const int l = wave_lane();
#pragma unroll 1
    for (int b = 0; b < kNb / kSb; ++b) {
        double a[kSb], x[kSb];
        const double* dg = D + b * kSb * (kLd + 1) + (l & (kSb - 1)) * kLd;
        const bool mine = wv == 1 || (wv == 0 && l < kNb - kSb * (b + 1));
        double* xr = (wv == 0 ? D + (kSb * (b + 1) + (mine ? l : 0)) * kLd : X + l * kLd) + b * kSb;
        int e = 0;
        if (wv < 2) {
            // (a lane without a row of its own works on some row of the buffers and stores nothing)
#pragma unroll
            for (int c = 0; c < kSb; ++c) { a[c] = dg[c]; x[c] = xr[c]; }
            e = panel16(a, x);
        }
        __syncthreads();   // both wavefronts have read the diagonal block
        if (wv < 2) {
            if (wv == 0 && l < kSb) {
#pragma unroll
                for (int c = 0; c < kSb; ++c) D[b * kSb * (kLd + 1) + l * kLd + c] = c <= l ? a[c] : 0.0;
            }
            if (mine) {
#pragma unroll
                for (int c = 0; c < kSb; ++c) xr[c] = x[c];
            }
            if (e != 0 && bad == 0) bad = b * kSb + e;
        }
        __syncthreads();
        // columns to the right: D_t,u -= D_t,b D_u,b^T for b < u <= t, X_t,u -= X_t,b D_u,b^T
        int q = 0;
        for (int u = b + 1; u < kNb / kSb; ++u) {
            const double* Du = D + u * kSb * kLd + b * kSb;
            for (int t = u; t < kNb / kSb + 4; ++t, ++q)
                if (q % (kStepThreads / kWave) == wv) {
                    double* row = t < kNb / kSb ? D + t * kSb * kLd : X + (t - kNb / kSb) * kSb * kLd;
                    tile_store(row + u * kSb, mul16(row + b * kSb, kLd, Du, kLd, -1.0, tile_load(row + u * kSb)));
                }
        }
        __syncthreads();
    }
    if (strip == 0) {
        for (int t = threadIdx.x; t < kNb * kNb; t += kStepThreads) Ldiag[t] = D[(t % kNb) * kLd + t / kNb];
        if (threadIdx.x == 0) {
            if (k0 == 0) *info = bad;
            else if (bad != 0 && *info == 0) *info = k0 + bad;
        }
    }
    for (int t = threadIdx.x; t < kNb * kNb; t += kStepThreads) {
        const int r = t % kNb, c = t / kNb;
        if (r < nr && c < nb) A[R0 + r + (size_t)(k0 + c) * lda] = X[r * kLd + c];
    }
}

// A(r, c) -= sum_k A(r, k) A(c, k) over the 64 columns of block kp, rows from r0, columns
// from c0 (entries on or below the diagonal)
__device__ __forceinline__ void chol_tile(int rows, int n, double* __restrict__ A, long long lda, int kp, int r0, int c0,
                                          double* sm) {
    double *sR = sm, *sC = sm + kNb * kLd;
    // (rows and columns past the end repeat the last one, their products are not stored)
    double va[kStepPer], vb[kStepPer];
    block_fetch(A, lda, kp, r0, rows - 1, va);
    block_fetch(A, lda, kp, c0, n - 1, vb);
    const int l = wave_lane(), wv = uniform(threadIdx.x >> 6);
    const int row = l & 15, grp = l >> 4;
    const int wr = (wv & 3) * 16, wc = (wv >> 2) * 32;
    // the tile itself, in flight with the block's rows (a lane's rows are consecutive in memory)
    double old[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            old[j][q] = A[min(r0 + wr + row, rows - 1) + (size_t)min(c0 + wc + 16 * j + grp + 4 * q, n - 1) * lda];
    block_put(sR, va);
    block_put(sC, vb);
    __syncthreads();
    mf_d4 acc[2] = {};
    block_products<2>(sR + wr, sC + wc, acc);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = r0 + wr + row, c = c0 + wc + 16 * j + grp + 4 * q;
            if (r < rows && c < n && r >= c) A[r + (size_t)c * lda] = old[j][q] - acc[j][q];
        }
}

// Block k0: workgroups 0 .. strips - 1 are its strips (the longest work, started first),
// the others the tiles to its right, column by column.
__global__ __launch_bounds__(kStepThreads) void k_chol_step(int rows, int n, double* __restrict__ A, long long lda, int k0,
                                                            int strips, double* __restrict__ Ldiag,
                                                            int* __restrict__ info) {
    extern __shared__ __align__(16) double sm[];
    if ((int)blockIdx.x < strips) {
        chol_strip(rows, n, A, lda, k0, blockIdx.x, Ldiag, info, sm);
        return;
    }
    const int k1 = k0 + kNb;               // (a block with tiles to its right has all 64 columns)
    int t = blockIdx.x - strips, j = 0;
    while (t >= strips - j) { t -= strips - j; ++j; }
    chol_tile(rows, n, A, lda, k0 - kNb, k1 + (j + t) * kNb, k1 + j * kNb, sm);
}

// the factor of the last diagonal block to its place
__global__ __launch_bounds__(256) void k_chol_last(int nb, double* __restrict__ A, long long lda,
                                                   const double* __restrict__ Ldiag) {
    for (int t = threadIdx.x; t < kNb * kNb; t += 256) {
        const int r = t % kNb, c = t / kNb;
        if (r < nb && c <= r) A[r + (size_t)c * lda] = Ldiag[t];
    }
}

// A (rows x n, rows >= n, ld lda): the lower triangle of its first n rows -> L,
// the rows below -> B L^-T.  *info = 0 or the 1-based column of the first pivot
// that is not positive (as dpotrf reports it).  Ldiag: kNb * kNb doubles.
int chol_lower(hipStream_t st, int rows, int n, double* A, long long lda, double* Ldiag, int* info) {
    int k0 = 0;
    for (; k0 < n; k0 += kNb) {
        const int k1 = std::min(k0 + kNb, n);
        const int strips = std::max(1, (rows - k1 + kNb - 1) / kNb);
        // the first block has nothing before it to subtract
        const int cols = k0 == 0 ? 0 : (n - k1 + kNb - 1) / kNb;
        const int tiles = cols * strips - cols * (cols - 1) / 2;
        hipLaunchKernelGGL(k_chol_step, dim3(strips + tiles), dim3(kStepThreads), kStepLds, st, rows, n, A, lda, k0,
                           strips, Ldiag, info);
        if (int e = launch_check("k_chol_step")) return e;
    }
    k0 -= kNb;
    hipLaunchKernelGGL(k_chol_last, dim3(1), dim3(256), 0, st, n - k0, A + k0 + (size_t)k0 * lda, lda, (const double*)Ldiag);
    return launch_check("k_chol_last");
}

// y (n) += A (n x m, ld lda) x (stride incx): kGemvCols columns per workgroup and
// 256 rows, partial sums in part[chunk][n], added in order by k_gemv_sum
constexpr int kGemvCols = 64;

__global__ __launch_bounds__(256) void k_gemv(int n, int m, const double* __restrict__ A, long long lda,
                                              const double* __restrict__ x, long long incx,
                                              double* __restrict__ part) {
    const int r = blockIdx.x * 256 + threadIdx.x;
    const int c0 = blockIdx.y * kGemvCols, c1 = min(m, c0 + kGemvCols);
    if (r >= n) return;
    double s = 0.0;
#pragma unroll 8
    for (int c = c0; c < c1; ++c) s += A[r + (size_t)c * lda] * x[(size_t)c * incx];
    part[(size_t)blockIdx.y * n + r] = s;
}

__global__ __launch_bounds__(256) void k_gemv_sum(int n, int chunks, const double* __restrict__ part, double beta,
                                                  double* __restrict__ y, long long incy) {
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    double s = 0.0;
    for (int c = 0; c < chunks; ++c) s += part[(size_t)c * n + r];
    y[(size_t)r * incy] = beta != 0.0 ? y[(size_t)r * incy] + s : s;
}

size_t gemv_ws_doubles(int n, int m) { return (size_t)n * ((m + kGemvCols - 1) / kGemvCols); }

// y = [y +] A x
int gemv(hipStream_t st, int n, int m, const double* A, long long lda, const double* x, long long incx, bool add,
         double* y, long long incy, double* part) {
    const int chunks = (m + kGemvCols - 1) / kGemvCols;
    hipLaunchKernelGGL(k_gemv, dim3((n + 255) / 256, chunks), dim3(256), 0, st, n, m, A, lda, x, incx, part);
    hipLaunchKernelGGL(k_gemv_sum, dim3((n + 255) / 256), dim3(256), 0, st, n, chunks, (const double*)part,
                       add ? 1.0 : 0.0, y, incy);
    return launch_check("gemv");
}

// xi = (ref - pred) * scale, loss += sum xi^2 (one block of 256 per 256 entries)
__global__ void k_residual(int n, const double* __restrict__ pred, const double* __restrict__ ref, double ref_scalar,
                           double scale, double* __restrict__ xi, double* __restrict__ loss) {
    __shared__ double part[4];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (i < n) {
        v = ((ref ? ref[i] : ref_scalar) - pred[i]) * scale;
        xi[i] = v;
    }
    double s = wave_sum(v * v);
    if (wave_lane() == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(loss, part[0] + part[1] + part[2] + part[3]);
}

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// the n_w x n_w form when the observations outnumber the weights
bool factored_form(int n_w, int m) { return m > n_w; }

}  // namespace
}  // namespace pt

using namespace pt;

namespace {
// Workspace: the factorised matrix with the rows it carries, G (n_w x n_w form only),
// partial sums of the products with a vector and of those split over K, a vector, the diagonal block, info.
struct KalmanWs {
    size_t aug, G, part, gpart, vec, diag, info, total;
    long long lda;
    KalmanWs(int n_w, int m) {
        const size_t nw = (size_t)n_w, mm = (size_t)m;
        const bool f = factored_form(n_w, m);
        lda = f ? 2 * (long long)n_w + 1 : (long long)m + n_w + 1;
        size_t o = 0;
        aug = o; o += align256(8 * (size_t)lda * (f ? nw : mm));
        G = o; o += f ? align256(8 * nw * mm) : 0;
        part = o; o += align256(8 * gemv_ws_doubles(n_w, std::max(n_w, m)));
        gpart = o; o += align256(8 * gemm_part_doubles(n_w));
        vec = o; o += align256(8 * nw);
        diag = o; o += align256(8 * (size_t)kNb * kNb);
        info = o; o += align256(sizeof(int));
        total = o;
    }
};
}  // namespace

extern "C" size_t pt_kalman_workspace_bytes(int n_w, int m) {
    if (n_w < 1 || m < 1) return 0;
    return KalmanWs(n_w, m).total;
}

extern "C" int pt_kalman_residual(int n, const double* pred, const double* ref, double ref_scalar, double scale,
                                  double* xi, double* loss, pt_stream_t stream) {
    PT_REQUIRE(n >= 1 && pred && xi && loss, "pt_kalman_residual: bad arguments");
    hipLaunchKernelGGL(k_residual, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, n, pred, ref,
                       ref_scalar, scale, xi, loss);
    return launch_check("pt_kalman_residual");
}

extern "C" int pt_kalman_update(int n_w, int m, double* P, const double* H, long long ldh, const double* xi,
                                double* W, double r, double c, double q, void* ws, size_t ws_bytes, int* info,
                                pt_stream_t stream) {
    PT_REQUIRE(n_w >= 1 && m >= 1, "pt_kalman_update: n_w and m must be positive");
    PT_REQUIRE(P && H && xi && W && ws && info, "pt_kalman_update: null argument");
    PT_REQUIRE(ldh >= n_w, "pt_kalman_update: ldh < n_w");
    PT_REQUIRE(r > 0.0, "pt_kalman_update: the measurement noise must be positive");
    PT_REQUIRE(ws_bytes >= pt_kalman_workspace_bytes(n_w, m), "pt_kalman_update: workspace too small");
    PT_REQUIRE((size_t)n_w * n_w < (1ull << 31) && (factored_form(n_w, m) || (size_t)m * m < (1ull << 31)) &&
                   (size_t)n_w * m < (1ull << 31) && ldh < (1LL << 31),
               "pt_kalman_update: matrices of 2^31 entries and more");
    hipStream_t st = (hipStream_t)stream;
    const KalmanWs L(n_w, m);
    char* base = (char*)ws;
    double* S = (double*)(base + L.aug);
    double* G = (double*)(base + L.G);
    double* part = (double*)(base + L.part);
    double* gpart = (double*)(base + L.gpart);
    double* vec = (double*)(base + L.vec);
    double* diag = (double*)(base + L.diag);
    int* info2 = (int*)(base + L.info);
    const long long ld = L.lda;
    if (factored_form(n_w, m)) {
        // L = chol(P), lower triangle in place
        if (int e = chol_lower(st, n_w, n_w, P, n_w, diag, info)) return e;
        // G = L^T H
        if (int e = gemm_f64<1, 1>({n_w, m, n_w, P, n_w, H, ldh, G, n_w, 1.0, 0.0, 0.0, 0, 0, 1}, gpart, st)) return e;
        // S = G G^T + r I, below it L and (G xi)^T
        if (int e = gemm_f64<0, 0>({n_w, n_w, m, G, n_w, G, n_w, S, ld, 1.0, 0.0, r, 1, 0, 0}, gpart, st)) return e;
        if (int e = gemv(st, n_w, m, G, n_w, xi, 1, false, vec, 1, part)) return e;
        hipLaunchKernelGGL(k_lower_copy, dim3((n_w + 256) / 256, n_w), dim3(256), 0, st, n_w, (const double*)P,
                           (long long)n_w, (const double*)vec, S + n_w, ld);
        if (int e = launch_check("k_lower_copy")) return e;
        // S = Ls Ls^T, M = L Ls^-T, y = Ls^-1 G xi
        if (int e = chol_lower(st, 2 * n_w + 1, n_w, S, ld, diag, info2)) return e;
        hipLaunchKernelGGL(k_merge_info, dim3(1), dim3(64), 0, st, info, (const int*)info2);
        if (int e = launch_check("k_merge_info")) return e;
        // W += M y (= L S^-1 G xi), then P = c r M M^T + q I
        const double* M = S + n_w;
        if (int e = gemv(st, n_w, n_w, M, ld, S + 2 * (size_t)n_w, ld, true, W, 1, part)) return e;
        return gemm_f64<0, 0>({n_w, n_w, n_w, M, ld, M, ld, P, n_w, c * r, 0.0, q, 1, 1, 0}, gpart, st);
    }
    double* X = S + m;                       // n_w rows below the m x m matrix
    double* z = S + m + (size_t)n_w;         // and the row of the residuals
    if (m == 1) {
        if (int e = gemv(st, n_w, n_w, P, n_w, H, 1, false, X, 1, part)) return e;
        hipLaunchKernelGGL(k_one_obs, dim3(1), dim3(1024), 0, st, n_w, H, X, xi, r, z, info);
        if (int e = launch_check("k_one_obs")) return e;
    } else {
        // X = P H, A = H^T X + r I, the residuals as the last row
        if (int e = gemm_f64<0, 1>({n_w, m, n_w, P, n_w, H, ldh, X, ld, 1.0, 0.0, 0.0, 0, 0, 0}, gpart, st)) return e;
        if (int e = gemm_f64<1, 1>({m, m, n_w, H, ldh, X, ld, S, ld, 1.0, 0.0, r, 1, 0, 0}, gpart, st)) return e;
        hipLaunchKernelGGL(k_set_row, dim3((m + 255) / 256), dim3(256), 0, st, m, xi, z, ld);
        if (int e = launch_check("k_set_row")) return e;
        // A = L L^T, Z = X L^-T, z = L^-1 xi
        if (int e = chol_lower(st, m + n_w + 1, m, S, ld, diag, info)) return e;
    }
    // W += Z z, P = c (P - Z Z^T) + q I
    if (int e = gemv(st, n_w, m, X, ld, z, ld, true, W, 1, part)) return e;
    return gemm_f64<0, 0>({n_w, n_w, m, X, ld, X, ld, P, n_w, -c, c, q, 1, 1, 0}, gpart, st);
}
