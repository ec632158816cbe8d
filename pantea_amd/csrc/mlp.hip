// (c) Element-grouped atomic MLPs on gfx950 matrix cores.
//
// Replaces _compute_energy_per_atom (potentials/nnp/energy.py:23-39):
// scaler (descriptors/scaler.py:206-246) -> [Dense -> act] x hidden ->
// Dense(1) -> act_out (models/nn/model.py:24-58, y = x @ W + b), plus the
// reverse-mode gradient dE_i/dG_i that the force adjoint consumes.
//
// Atoms of one element are contiguous (internal order), so each layer is a
// plain GEMM over a 16-atom tile:
//   PT_MLP_F64    v_mfma_f64_16x16x4_f64   (FP64 in, FP64 accumulate)
//   PT_MLP_BF16   v_mfma_f32_16x16x32_bf16 (BF16 in, FP32 accumulate)
//   PT_MLP_BF16X3 the same with split operands x = hi + lo (hi*hi + hi*lo +
//                 lo*hi), giving about 16 mantissa bits per product.
// A workgroup owns a block of rows; layer inputs go through LDS (in the
// matrix instruction's input type), activation derivatives stay in registers,
// weights come from a packed device buffer (both W and W^T layouts, so that
// every MFMA operand fragment is a contiguous run of K elements) built once by
// pt_mlp_pack.
//
// Operand layouts (16x16 output tile, lane l, accumulator element i = 0..3):
//   A[row = l % 16][k = kc + l / 16 (f64) | kc + 8 (l / 16) + 0..7 (bf16)]
//   B[k (same as A)][col = l % 16]
//   C[row][col = l % 16] with row = l / 16 + 4 i   (v_mfma_f64_16x16x4_f64)
//                         or  row = 4 (l / 16) + i (v_mfma_f32_16x16x32_bf16)
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"

typedef double pt_d4 __attribute__((ext_vector_type(4)));
typedef float pt_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 pt_bf8 __attribute__((ext_vector_type(8)));

namespace pt {
namespace {

constexpr int kPad = 32;     // K/N padding of every layer
constexpr int kMaxW = 128;   // widest padded layer
constexpr int kMaxHidden = 3;

inline int padw(int w) { return (w + kPad - 1) / kPad * kPad; }

struct MlpShape {
    int n_hidden;
    int in_p;
    int w[kMaxHidden];    // true widths
    int wp[kMaxHidden];   // padded widths
    int act[kMaxHidden];
    int act_out;
    int kout;             // padded input width of the output layer
    int wmax;
    // packed buffer offsets (bytes)
    size_t W64[kMaxHidden], b64[kMaxHidden], wout64, bout64;
    size_t WTh[kMaxHidden], WTl[kMaxHidden], Wh[kMaxHidden], Wl[kMaxHidden], b32[kMaxHidden];
    size_t wout32, bout32;
    size_t total;
    // offsets into the unpacked FP64 parameter vector (W then b per layer)
    size_t pW[kMaxHidden + 1], pb[kMaxHidden + 1];
    int in_dim;
};

int make_shape(const pt_mlp_desc* d, MlpShape& s) {
    if (!d || d->n_layers < 1 || d->n_layers > kMaxHidden + 1) {
        set_error("mlp: n_layers must be in [1, %d]", kMaxHidden + 1);
        return PT_ERR_UNSUPPORTED;
    }
    if (d->width[d->n_layers - 1] != 1) {
        set_error("mlp: the output layer must have width 1");
        return PT_ERR_ARG;
    }
    s = MlpShape{};
    s.n_hidden = d->n_layers - 1;
    s.in_dim = d->in_dim;
    s.in_p = padw(d->in_dim);
    if (d->in_dim < 1 || s.in_p > kMaxW) {
        set_error("mlp: input width %d unsupported (max %d)", d->in_dim, kMaxW);
        return PT_ERR_UNSUPPORTED;
    }
    s.wmax = s.in_p;
    for (int l = 0; l < s.n_hidden; ++l) {
        s.w[l] = d->width[l];
        s.wp[l] = padw(d->width[l]);
        s.act[l] = d->act[l];
        if (s.w[l] < 1 || s.wp[l] > kMaxW) {
            set_error("mlp: hidden width %d unsupported (max %d)", s.w[l], kMaxW);
            return PT_ERR_UNSUPPORTED;
        }
        s.wmax = std::max(s.wmax, s.wp[l]);
    }
    s.act_out = d->act[d->n_layers - 1];
    s.kout = s.n_hidden > 0 ? s.wp[s.n_hidden - 1] : s.in_p;
    size_t o = 0, p = 0;
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    int fan_in = d->in_dim;
    for (int l = 0; l <= s.n_hidden; ++l) {
        int fo = l < s.n_hidden ? s.w[l] : 1;
        s.pW[l] = p; p += (size_t)fan_in * fo;
        s.pb[l] = p; p += (size_t)fo;
        fan_in = fo;
    }
    int kin = s.in_p;
    for (int l = 0; l < s.n_hidden; ++l) {
        const size_t mn = (size_t)kin * s.wp[l];
        s.W64[l] = o; o = al(o + 8 * mn);
        s.b64[l] = o; o = al(o + 8 * (size_t)s.wp[l]);
        s.WTh[l] = o; o = al(o + 2 * mn);
        s.WTl[l] = o; o = al(o + 2 * mn);
        s.Wh[l] = o; o = al(o + 2 * mn);
        s.Wl[l] = o; o = al(o + 2 * mn);
        s.b32[l] = o; o = al(o + 4 * (size_t)s.wp[l]);
        kin = s.wp[l];
    }
    s.wout64 = o; o = al(o + 8 * (size_t)s.kout);
    s.bout64 = o; o = al(o + 8);
    s.wout32 = o; o = al(o + 4 * (size_t)s.kout);
    s.bout32 = o; o = al(o + 4);
    s.total = o;
    return PT_OK;
}

// ---- activations (models/nn/activation.py:7-60) ---------------------------
template <typename T>
__device__ __forceinline__ void activate(int a, T z, T& y, T& dy) {
    switch (a) {
    case PT_ACT_IDENTITY: y = z; dy = T(1); return;
    case PT_ACT_TANH: { T t = tanh(z); y = t; dy = T(1) - t * t; return; }
    case PT_ACT_LOGISTIC: { T s = T(1) / (T(1) + exp(-z)); y = s; dy = s * (T(1) - s); return; }
    case PT_ACT_SOFTPLUS: {
        // log(1 + e^z) computed stably; derivative = logistic(z)
        T az = z > T(0) ? z : -z;
        y = (z > T(0) ? z : T(0)) + log1p(exp(-az));
        dy = T(1) / (T(1) + exp(-z));
        return;
    }
    case PT_ACT_RELU: y = z > T(0) ? z : T(0); dy = z > T(0) ? T(1) : T(0); return;
    case PT_ACT_GAUSSIAN: { T g = exp(T(-0.5) * z * z); y = g; dy = -z * g; return; }
    case PT_ACT_COS: y = cos(z); dy = -sin(z); return;
    case PT_ACT_EXP: { T e = exp(-z); y = e; dy = -e; return; }
    case PT_ACT_HARMONIC: y = z * z; dy = T(2) * z; return;
    }
    y = z; dy = T(1);
}

// The same for N values of one activation (the kind is uniform: one branch for all of them).
template <typename T, int N>
__device__ __forceinline__ void activate_n(int a, T (&y)[N], T (&dy)[N]) {
    auto each = [&](auto kind) {
#pragma unroll
        for (int i = 0; i < N; ++i) activate<T>(decltype(kind)::value, y[i], y[i], dy[i]);
    };
    switch (a) {
    case PT_ACT_TANH: each(std::integral_constant<int, PT_ACT_TANH>{}); return;
    case PT_ACT_LOGISTIC: each(std::integral_constant<int, PT_ACT_LOGISTIC>{}); return;
    case PT_ACT_SOFTPLUS: each(std::integral_constant<int, PT_ACT_SOFTPLUS>{}); return;
    case PT_ACT_RELU: each(std::integral_constant<int, PT_ACT_RELU>{}); return;
    case PT_ACT_GAUSSIAN: each(std::integral_constant<int, PT_ACT_GAUSSIAN>{}); return;
    case PT_ACT_COS: each(std::integral_constant<int, PT_ACT_COS>{}); return;
    case PT_ACT_EXP: each(std::integral_constant<int, PT_ACT_EXP>{}); return;
    case PT_ACT_HARMONIC: each(std::integral_constant<int, PT_ACT_HARMONIC>{}); return;
    default: each(std::integral_constant<int, PT_ACT_IDENTITY>{}); return;
    }
}

// y, dy/dz and d2y/dz2 (the training kernel differentiates the input gradient)
template <typename T>
__device__ __forceinline__ void activate2(int a, T z, T& y, T& dy, T& ddy) {
    switch (a) {
    case PT_ACT_IDENTITY: y = z; dy = T(1); ddy = T(0); return;
    case PT_ACT_TANH: { T t = tanh(z); y = t; dy = T(1) - t * t; ddy = T(-2) * t * dy; return; }
    case PT_ACT_LOGISTIC: {
        T s = T(1) / (T(1) + exp(-z)); y = s; dy = s * (T(1) - s); ddy = dy * (T(1) - T(2) * s); return;
    }
    case PT_ACT_SOFTPLUS: {
        T az = z > T(0) ? z : -z;
        y = (z > T(0) ? z : T(0)) + log1p(exp(-az));
        T s = T(1) / (T(1) + exp(-z));
        dy = s; ddy = s * (T(1) - s);
        return;
    }
    case PT_ACT_RELU: y = z > T(0) ? z : T(0); dy = z > T(0) ? T(1) : T(0); ddy = T(0); return;
    case PT_ACT_GAUSSIAN: { T g = exp(T(-0.5) * z * z); y = g; dy = -z * g; ddy = (z * z - T(1)) * g; return; }
    case PT_ACT_COS: y = cos(z); dy = -sin(z); ddy = -y; return;
    case PT_ACT_EXP: { T e = exp(-z); y = e; dy = -e; ddy = e; return; }
    case PT_ACT_HARMONIC: y = z * z; dy = T(2) * z; ddy = T(2); return;
    }
    y = z; dy = T(1); ddy = T(0);
}

__device__ __forceinline__ unsigned short bf16_bits(float x) {
    // round to nearest even
    unsigned u = __float_as_uint(x);
    unsigned r = u + 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(r >> 16);
}
__device__ __forceinline__ float bf16_to_f(unsigned short b) { return __uint_as_float(((unsigned)b) << 16); }

__device__ __forceinline__ void split_bf16(float x, unsigned short& hi, unsigned short& lo) {
    hi = bf16_bits(x);
    lo = bf16_bits(x - bf16_to_f(hi));
}

// ---- packing: FP64 params -> padded W/W^T (f64, bf16 hi/lo), biases ------
__global__ void k_pack(MlpShape s, const double* __restrict__ params, char* __restrict__ out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    int kin = s.in_p, fan_in = s.in_dim;
    for (int l = 0; l < s.n_hidden; ++l) {
        const int n = s.wp[l];
        const int mn = kin * n;
        if (t < mn) {
            const int k = t / n, c = t % n;  // W[k][c]
            const double v = (k < fan_in && c < s.w[l]) ? params[s.pW[l] + (size_t)k * s.w[l] + c] : 0.0;
            ((double*)(out + s.W64[l]))[t] = v;
            unsigned short hi, lo;
            split_bf16((float)v, hi, lo);
            ((unsigned short*)(out + s.Wh[l]))[t] = hi;
            ((unsigned short*)(out + s.Wl[l]))[t] = lo;
            ((unsigned short*)(out + s.WTh[l]))[c * kin + k] = hi;
            ((unsigned short*)(out + s.WTl[l]))[c * kin + k] = lo;
        }
        if (t < n) {
            const double b = t < s.w[l] ? params[s.pb[l] + t] : 0.0;
            ((double*)(out + s.b64[l]))[t] = b;
            ((float*)(out + s.b32[l]))[t] = (float)b;
        }
        fan_in = s.w[l];
        kin = n;
    }
    const int L = s.n_hidden;
    if (t < s.kout) {
        const double v = t < fan_in ? params[s.pW[L] + t] : 0.0;
        ((double*)(out + s.wout64))[t] = v;
        ((float*)(out + s.wout32))[t] = (float)v;
    }
    if (t == 0) {
        ((double*)(out + s.bout64))[0] = params[s.pb[L]];
        ((float*)(out + s.bout32))[0] = (float)params[s.pb[L]];
    }
}

// ---- the MLP kernel -----------------------------------------------------------
template <int MODE>
struct MT { typedef float T; };
template <>
struct MT<PT_MLP_F64> { typedef double T; };

// One network of a launch: the atoms of one element.
struct MlpNet {
    MlpShape s;
    int n_atoms;
    int block0;           // first workgroup of this network
    const void* G;
    const double* scale;  // [2][in_dim]: sub, mul
    double scale_add;
    const char* packed;
    double* e_atom;
    void* dEdG;
};

constexpr int kMlpNets = 4;   // networks per launch (the arguments stay well below the 4 KB limit)

struct MlpArgs {
    MlpNet net[kMlpNets];
    int n_net;
    int ldg;
    int g_f64;
    int stride;           // LDS row stride (elements)
};

// C = A(16 x K, LDS row-major, stride) * B, accumulating one 16-column tile.
// Row of accumulator element i in lane group grp = l / 16.
template <int MODE>
__device__ __forceinline__ int crow(int grp, int i) {
    return MODE == PT_MLP_F64 ? grp + 4 * i : 4 * grp + i;
}

template <int MODE>
__device__ __forceinline__ void gemm_tile(const typename MT<MODE>::T* A, int stride, int K,
                                          const char* packed, size_t off_hi, size_t off_lo,
                                          int ldb, bool bt, int n0, typename MT<MODE>::T acc[4]) {
    const int l = wave_lane();
    const int row = l & 15, grp = l >> 4;
    if constexpr (MODE == PT_MLP_F64) {
        pt_d4 c = {acc[0], acc[1], acc[2], acc[3]};
        const double* W = (const double*)(packed + off_hi);
        for (int k0 = 0; k0 < K; k0 += 4) {
            const int k = k0 + grp;
            const double a = A[row * stride + k];
            // bt == false: B[k][n] = W[k][n] (W is K x ldb);  bt == true: B[k][n] = W[n][k]
            const double b = bt ? W[(size_t)(n0 + row) * ldb + k] : W[(size_t)k * ldb + n0 + row];
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
        }
        acc[0] = c[0]; acc[1] = c[1]; acc[2] = c[2]; acc[3] = c[3];
    } else {
        pt_f4 c = {acc[0], acc[1], acc[2], acc[3]};
        const unsigned short* Bh = (const unsigned short*)(packed + off_hi);
        const unsigned short* Bl = (const unsigned short*)(packed + off_lo);
        for (int k0 = 0; k0 < K; k0 += 32) {
            const int kb = k0 + 8 * grp;
            pt_bf8 ah, al, bh, bl;
            const float* ap = A + row * stride + kb;
            // B fragment: 8 consecutive k of column n0 + row, from the k-contiguous layout
            const size_t bo = (size_t)(n0 + row) * ldb + kb;
            const uint4 vh = *reinterpret_cast<const uint4*>(Bh + bo);
            const uint4 vl = *reinterpret_cast<const uint4*>(Bl + bo);
            const unsigned short* ph = reinterpret_cast<const unsigned short*>(&vh);
            const unsigned short* pl = reinterpret_cast<const unsigned short*>(&vl);
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                unsigned short hi, lo;
                split_bf16(ap[q], hi, lo);
                ah[q] = __builtin_bit_cast(__bf16, hi);
                al[q] = __builtin_bit_cast(__bf16, lo);
                bh[q] = __builtin_bit_cast(__bf16, ph[q]);
                bl[q] = __builtin_bit_cast(__bf16, pl[q]);
            }
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, c, 0, 0, 0);
            if (MODE == PT_MLP_BF16X3) {
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, c, 0, 0, 0);
            }
        }
        acc[0] = c[0]; acc[1] = c[1]; acc[2] = c[2]; acc[3] = c[3];
    }
    (void)bt;
}

// ---- inference: energies and input gradients ---------------------------------
//
// One workgroup of four wavefronts takes ROWS = 16 MTW WR atoms through the
// whole network.  The wavefronts form a WR x WC grid: WR blocks of MTW row
// tiles times WC interleaved sets of 16-column tiles (CT tiles each in a
// hidden layer).  A weight fragment is loaded once for the MTW row tiles of
// its wavefront, and the MTW products of one fragment are independent chains.
// Between layers only the next product's input goes through LDS, stored as
// the matrix instruction takes it (FP64, or the BF16 halves, split once where
// they are produced); the activation derivatives stay in the registers of the
// lanes that need them again in the reverse sweep (same C layout).
//
// What bounds it: below ~10k atoms the serial chain of one row tile through
// the layers (13.5 us FP64, 9.0 us BF16x3 for 52-64-64-1; one wavefront doing
// all columns of 16 rows took 66 and 28 us); above, the weight fragments
// re-read from L2 by every workgroup and the MFMA issue (98,304 rows: 137 us
// FP64 = 21 TFLOP/s, 50 us BF16x3; before 245 and 85 us).
template <int MODE>
struct MlpLds;
template <>
struct MlpLds<PT_MLP_F64> {
    double* x;
    int stride;
    static constexpr size_t bytes(int rows, int stride) { return sizeof(double) * (size_t)rows * stride; }
    __device__ __forceinline__ void put(int r, int k, double v) const { x[r * stride + k] = v; }
};
template <int MODE>
struct MlpLds {
    unsigned short* hi;
    unsigned short* lo;
    int stride;
    static constexpr size_t bytes(int rows, int stride) { return 2 * sizeof(unsigned short) * (size_t)rows * stride; }
    __device__ __forceinline__ void put(int r, int k, float v) const {
        unsigned short h, l;
        split_bf16(v, h, l);
        hi[r * stride + k] = h;
        lo[r * stride + k] = l;
    }
};

template <int MODE>
__device__ __forceinline__ MlpLds<MODE> mlp_lds(char* base, int rows, int stride) {
    MlpLds<MODE> b;
    b.stride = stride;
    if constexpr (MODE == PT_MLP_F64) {
        b.x = reinterpret_cast<double*>(base);
    } else {
        b.hi = reinterpret_cast<unsigned short*>(base);
        b.lo = b.hi + (size_t)rows * stride;
    }
    return b;
}

// acc[m] += X(rows r0 + 16 m ..) * B(columns n0 ..) for the MTW row tiles of a
// wavefront, K a multiple of 32.  Every fragment of a K chunk is loaded before
// the chunk's products.
template <int MODE, int MTW>
__device__ __forceinline__ void mlp_gemm(const MlpLds<MODE>& X, int r0, int K, const char* packed, size_t off_hi,
                                         size_t off_lo, int ldb, bool bt, int n0,
                                         typename MT<MODE>::T (&acc)[MTW][4]) {
    const int l = wave_lane();
    const int row = l & 15, grp = l >> 4;
    if constexpr (MODE == PT_MLP_F64) {
        (void)off_lo;
        pt_d4 c[MTW];
#pragma unroll
        for (int m = 0; m < MTW; ++m) c[m] = pt_d4{0.0, 0.0, 0.0, 0.0};
        const double* W = (const double*)(packed + off_hi);
        // bt == false: B[k][n] = W[k][n] (W is K x ldb);  bt == true: B[k][n] = W[n][k]
        const double* Wl = bt ? W + (size_t)(n0 + row) * ldb + grp : W + (size_t)grp * ldb + n0 + row;
        const size_t ks = bt ? 4 : (size_t)4 * ldb;
        const double* A = X.x + (r0 + row) * X.stride + grp;
        for (int k0 = 0; k0 < K; k0 += 32) {
            double b[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) b[u] = Wl[(size_t)(k0 / 4 + u) * ks];
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int m = 0; m < MTW; ++m)
                    c[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[16 * m * X.stride + k0 + 4 * u], b[u], c[m], 0, 0, 0);
        }
#pragma unroll
        for (int m = 0; m < MTW; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[m][i] = c[m][i];
    } else {
        (void)bt;
        pt_f4 c[MTW];
#pragma unroll
        for (int m = 0; m < MTW; ++m) c[m] = pt_f4{0.f, 0.f, 0.f, 0.f};
        // B fragment: 8 consecutive k of column n0 + row, from the k-contiguous layout
        const size_t bo = (size_t)(n0 + row) * ldb + 8 * grp;
        const unsigned short* Bh = (const unsigned short*)(packed + off_hi) + bo;
        const unsigned short* Bl = (const unsigned short*)(packed + off_lo) + bo;
        const int ao = (r0 + row) * X.stride + 8 * grp;
        for (int k0 = 0; k0 < K; k0 += 32) {
            const pt_bf8 bh = __builtin_bit_cast(pt_bf8, *reinterpret_cast<const uint4*>(Bh + k0));
            const pt_bf8 bl = MODE == PT_MLP_BF16X3 ? __builtin_bit_cast(pt_bf8, *reinterpret_cast<const uint4*>(Bl + k0))
                                                    : pt_bf8{};
#pragma unroll
            for (int m = 0; m < MTW; ++m) {
                const int o = ao + 16 * m * X.stride + k0;
                const pt_bf8 ah = __builtin_bit_cast(pt_bf8, *reinterpret_cast<const uint4*>(X.hi + o));
                c[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, c[m], 0, 0, 0);
                if (MODE == PT_MLP_BF16X3) {
                    const pt_bf8 al = __builtin_bit_cast(pt_bf8, *reinterpret_cast<const uint4*>(X.lo + o));
                    c[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, c[m], 0, 0, 0);
                    c[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, c[m], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int m = 0; m < MTW; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[m][i] = c[m][i];
    }
}

// sum over the 16 lanes of a DPP row (the 16 columns of a C tile), in every lane
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_f32<kDppXor1, 0xF>(v);
    v += dpp_f32<kDppXor2, 0xF>(v);
    v += dpp_f32<kDppHalfMirror, 0xF>(v);
    v += dpp_f32<kDppMirror, 0xF>(v);
    return v;
}
__device__ __forceinline__ double row16_sum(double v) {
    v += dpp_f64<kDppXor1, 0xF>(v);
    v += dpp_f64<kDppXor2, 0xF>(v);
    v += dpp_f64<kDppHalfMirror, 0xF>(v);
    v += dpp_f64<kDppMirror, 0xF>(v);
    return v;
}

// f(0), ..., f(N - 1) with compile-time indices (the layer loops index register arrays)
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

template <int CT, int WC, int MTW>
constexpr int mlp_rows() { return 16 * MTW * (4 / WC); }

// HM: most hidden layers; hidden layers have at most 16 CT WC columns (padded).
template <int MODE, int CT, int WC, int MTW, int HM>
__global__ __launch_bounds__(256) void k_mlp(MlpArgs a) {
    typedef typename MT<MODE>::T T;
    constexpr int ROWS = mlp_rows<CT, WC, MTW>();
    extern __shared__ __align__(16) char smem[];
    __shared__ T esum[WC][ROWS];
    int gi = 0;
    while (gi + 1 < a.n_net && (int)blockIdx.x >= a.net[gi + 1].block0) ++gi;
    const MlpNet& net = a.net[gi];
    const MlpShape& s = net.s;
    const int stride = a.stride;
    // the two LDS buffers of layer inputs, swapped after each layer
    MlpLds<MODE> X = mlp_lds<MODE>(smem, ROWS, stride);
    MlpLds<MODE> Y = mlp_lds<MODE>(smem + MlpLds<MODE>::bytes(ROWS, stride), ROWS, stride);
    auto swap_xy = [&]() { const MlpLds<MODE> t = X; X = Y; Y = t; };
    const int l = wave_lane();
    const int wv = uniform(threadIdx.x >> 6);
    const int wc = wv % WC;
    const int r0 = (wv / WC) * 16 * MTW;     // this wavefront's first row
    const int row = l & 15, grp = l >> 4;
    const int a0 = ((int)blockIdx.x - net.block0) * ROWS;
    const char* packed = net.packed;
    const int H = s.n_hidden;
    const T* wout = (MODE == PT_MLP_F64) ? (const T*)(packed + s.wout64) : (const T*)(packed + s.wout32);
    const T bout = (MODE == PT_MLP_F64) ? (T)((const double*)(packed + s.bout64))[0]
                                        : (T)((const float*)(packed + s.bout32))[0];
    auto g_at = [&](int atom, int k) {
        const size_t o = (size_t)atom * a.ldg + k;
        return a.g_f64 ? ((const double*)net.G)[o] : (double)((const float*)net.G)[o];
    };

    // 1. scaled input, zero padded: 32 columns x 8 rows per step (a linear model reads it where it is)
    for (int k0 = 0; H > 0 && k0 < s.in_p; k0 += 32) {
        const int k = k0 + (threadIdx.x & 31);
        const bool ok = k < s.in_dim;
        const double sub = ok ? net.scale[k] : 0.0, mul = ok ? net.scale[s.in_dim + k] : 0.0;
        double g[ROWS / 8];
#pragma unroll
        for (int j = 0; j < ROWS / 8; ++j) {
            const int atom = a0 + (threadIdx.x >> 5) + 8 * j;
            g[j] = ok && atom < net.n_atoms ? g_at(atom, k) : 0.0;
        }
#pragma unroll
        for (int j = 0; j < ROWS / 8; ++j) {
            const int r = (threadIdx.x >> 5) + 8 * j;
            X.put(r, k, ok && a0 + r < net.n_atoms ? (T)((g[j] - sub) * mul + net.scale_add) : T(0));
        }
    }
    __syncthreads();

    // 2. hidden layers; part: this lane's share of the output layer's dot product
    T D[HM][CT][MTW][4];                     // activation derivatives
    T part[MTW][4] = {};
    int kin = s.in_p;
    static_for<HM>([&](auto hc) {
        constexpr int h = decltype(hc)::value;
        if (h < H) {
            const int wp = s.wp[h];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const int n0 = 16 * (wc + WC * ct);
                T z[MTW][4] = {}, dz[MTW][4] = {};
                const int col = n0 + row;
                if (n0 < s.w[h]) {
                    T acc[MTW][4];
                    if (MODE == PT_MLP_F64)
                        mlp_gemm<MODE, MTW>(X, r0, kin, packed, s.W64[h], 0, wp, false, n0, acc);
                    else
                        mlp_gemm<MODE, MTW>(X, r0, kin, packed, s.WTh[h], s.WTl[h], kin, true, n0, acc);
                    const T bias = (MODE == PT_MLP_F64) ? (T)((const double*)(packed + s.b64[h]))[col]
                                                        : (T)((const float*)(packed + s.b32[h]))[col];
                    const bool pad = col >= s.w[h];
#pragma unroll
                    for (int m = 0; m < MTW; ++m) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) z[m][i] = acc[m][i] + bias;
                        activate_n<T, 4>(s.act[h], z[m], dz[m]);
#pragma unroll
                        for (int i = 0; i < 4; ++i) { z[m][i] = pad ? T(0) : z[m][i]; dz[m][i] = pad ? T(0) : dz[m][i]; }
                    }
                }
                const T wk = (h == H - 1 && n0 < wp) ? wout[col] : T(0);
#pragma unroll
                for (int m = 0; m < MTW; ++m)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        D[h][ct][m][i] = dz[m][i];
                        if (h == H - 1) part[m][i] += z[m][i] * wk;
                        else if (n0 < wp) Y.put(r0 + 16 * m + crow<MODE>(grp, i), col, z[m][i]);
                    }
            }
            if (h < H - 1) {
                __syncthreads();
                swap_xy();
                kin = wp;
            }
        }
    });
    if (H == 0) {   // linear model: the scaled input itself
        for (int n0 = 16 * wc; n0 < s.in_p; n0 += 16 * WC) {
            const int k = n0 + row;
            if (k < s.in_dim) {
                const double sub = net.scale[k], mul = net.scale[s.in_dim + k];
#pragma unroll
                for (int m = 0; m < MTW; ++m)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int atom = a0 + r0 + 16 * m + crow<MODE>(grp, i);
                        if (atom < net.n_atoms) part[m][i] += (T)((g_at(atom, k) - sub) * mul + net.scale_add) * wout[k];
                    }
            }
        }
    }

    // 3. output layer (width 1): 16 columns by DPP, the WC column sets through LDS
    T go[MTW][4];                            // output derivatives of this lane's rows
#pragma unroll
    for (int m = 0; m < MTW; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const T v = row16_sum(part[m][i]);
            if (row == 0) esum[wc][r0 + 16 * m + crow<MODE>(grp, i)] = v;
        }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MTW; ++m) {
        T y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + 16 * m + crow<MODE>(grp, i);
            y[i] = esum[0][r];
#pragma unroll
            for (int q = 1; q < WC; ++q) y[i] += esum[q][r];
            y[i] += bout;
        }
        activate_n<T, 4>(s.act_out, y, go[m]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + 16 * m + crow<MODE>(grp, i);
            if (wc == 0 && row == 0 && a0 + r < net.n_atoms) net.e_atom[a0 + r] = (double)y[i];
        }
    }
    if (!net.dEdG) return;

    // 4. reverse sweep: dZ of layer h goes through LDS, the derivatives come from registers
    static_for<HM>([&](auto hc) {
        constexpr int h = HM - 1 - decltype(hc)::value;
        constexpr int hn = h + 1 < HM ? h + 1 : h;
        if (h < H) {
            const int wp = s.wp[h];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const int n0 = 16 * (wc + WC * ct);
                if (n0 < wp) {
                    T acc[MTW][4];
                    if (h == H - 1) {
                        const T wk = wout[n0 + row];
#pragma unroll
                        for (int m = 0; m < MTW; ++m)
#pragma unroll
                            for (int i = 0; i < 4; ++i) acc[m][i] = go[m][i] * wk;
                    } else if (n0 < s.w[h]) {
                        // dZ_h = (dZ_{h+1} . W_{h+1}^T) * D[h]
                        const int wn = s.wp[hn];
                        if (MODE == PT_MLP_F64)
                            mlp_gemm<MODE, MTW>(X, r0, wn, packed, s.W64[hn], 0, wn, true, n0, acc);
                        else
                            mlp_gemm<MODE, MTW>(X, r0, wn, packed, s.Wh[hn], s.Wl[hn], wn, true, n0, acc);
                    } else {
#pragma unroll
                        for (int m = 0; m < MTW; ++m)
#pragma unroll
                            for (int i = 0; i < 4; ++i) acc[m][i] = T(0);
                    }
#pragma unroll
                    for (int m = 0; m < MTW; ++m)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            Y.put(r0 + 16 * m + crow<MODE>(grp, i), n0 + row, D[h][ct][m][i] * acc[m][i]);
                }
            }
            __syncthreads();
            swap_xy();
        }
    });
    // 5. dE/dx' = dZ_0 . W_0^T (or wout for a linear model), then chain the scaler
    for (int n0 = 16 * wc; n0 < s.in_p; n0 += 16 * WC) {
        const int k = n0 + row;
        if (n0 >= s.in_dim) break;
        T acc[MTW][4];
        if (H > 0) {
            if (MODE == PT_MLP_F64)
                mlp_gemm<MODE, MTW>(X, r0, s.wp[0], packed, s.W64[0], 0, s.wp[0], true, n0, acc);
            else
                mlp_gemm<MODE, MTW>(X, r0, s.wp[0], packed, s.Wh[0], s.Wl[0], s.wp[0], true, n0, acc);
        } else {
#pragma unroll
            for (int m = 0; m < MTW; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[m][i] = go[m][i] * wout[k];
        }
        if (k < s.in_dim) {
            const double mk = net.scale[s.in_dim + k];
#pragma unroll
            for (int m = 0; m < MTW; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int atom = a0 + r0 + 16 * m + crow<MODE>(grp, i);
                    if (atom < net.n_atoms) {
                        const double gk = (double)acc[m][i] * mk;
                        const size_t o = (size_t)atom * a.ldg + k;
                        if (a.g_f64) ((double*)net.dEdG)[o] = gk;
                        else ((float*)net.dEdG)[o] = (float)gk;
                    }
                }
        }
    }
}

// ---- training: forward-over-reverse through the MLP -------------------------
//
// Per atom the loss gradient w.r.t. the weights is
//   gy * dy/dtheta + tseed * d(ydot)/dtheta,
// y = MLP(x'), ydot = grad_x' MLP . xdot' (xdot' = T * mul, the descriptor
// tangent in scaled space).  Rows 0..15 of a 32-row tile carry the 16 atoms'
// primal values, rows 16..31 their tangents, so every layer (and its reverse)
// is one GEMM over 32 rows on the matrix cores; the weight gradients are
// GEMMs over those 32 rows (K = atoms x {primal, tangent}).

// C(16 x 16) = A^T B over the 32 rows of two LDS tiles: A[r][i0 + ..], B[r][o0 + ..].
template <int MODE>
__device__ __forceinline__ void wgrad_tile(const typename MT<MODE>::T* A, const typename MT<MODE>::T* B,
                                           int stride, int i0, int o0, typename MT<MODE>::T out[4]) {
    const int l = wave_lane();
    const int row = l & 15, grp = l >> 4;
    if constexpr (MODE == PT_MLP_F64) {
        pt_d4 c = {0.0, 0.0, 0.0, 0.0};
        for (int k0 = 0; k0 < 32; k0 += 4) {
            const int k = k0 + grp;
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(A[k * stride + i0 + row], B[k * stride + o0 + row], c, 0, 0, 0);
        }
        out[0] = c[0]; out[1] = c[1]; out[2] = c[2]; out[3] = c[3];
    } else {
        pt_f4 c = {0.f, 0.f, 0.f, 0.f};
        pt_bf8 ah, al, bh, bl;
        const int kb = 8 * grp;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            unsigned short h1, l1, h2, l2;
            split_bf16(A[(kb + q) * stride + i0 + row], h1, l1);
            split_bf16(B[(kb + q) * stride + o0 + row], h2, l2);
            ah[q] = __builtin_bit_cast(__bf16, h1);
            al[q] = __builtin_bit_cast(__bf16, l1);
            bh[q] = __builtin_bit_cast(__bf16, h2);
            bl[q] = __builtin_bit_cast(__bf16, l2);
        }
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, c, 0, 0, 0);
        if (MODE == PT_MLP_BF16X3) {
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, c, 0, 0, 0);
        }
        out[0] = c[0]; out[1] = c[1]; out[2] = c[2]; out[3] = c[3];
    }
}

// What bounds it: one tile's chain of small products and elementwise passes
// between barriers; the four wavefronts of a workgroup share a tile (column tiles
// and halves of the products, cells of the elementwise passes), where one
// wavefront per tile needed the same LDS and left three of a CU's four SIMDs idle.
// Measured, student networks of two elements: Jacobian of 4,608 rows 240 -> 58 us
// (FP64), gradient sums of 26,000 atoms 226 -> 72 us (BF16x3), 123 -> 24 us for one
// structure (FP64); the elements share the launch.
struct TrainNet {
    MlpShape s;
    int n_atoms;
    int block0, nblocks;  // this network's workgroups
    int nparam;
    const void* G;
    const void* T;        // TRAIN: tangents; JACOBIAN: T[d * t_dir + atom * ldg + k]
    const double* scale;
    double scale_add;
    const char* packed;
    const double* gy;     // TRAIN: per-atom seed of y
    double* out;          // TRAIN: parameter gradient (FP64, layout of the unpacked params); JACOBIAN: J
};

struct TrainArgs {
    TrainNet net[kMlpNets];
    int n_net;
    int ldg;
    int g_f64;
    double tseed;         // seed of ydot (same for every atom); JACOBIAN: the sign
    int stride;
    // JACOBIAN
    int n_dir;
    long long t_dir, ldj;
};

// LDS of a workgroup: layer inputs (H + 1), pre-activations (H) and two reverse
// buffers of 32 rows, 32 per-row scalars, and the gradient sums (TRAIN)
inline size_t train_lds(size_t word, int H, int stride, int nparam) {
    return word * ((size_t)(2 * H + 3) * 32 * stride + 32 + nparam);
}

// cells of 16 rows x `width` columns (a multiple of 32) over the 256 threads
template <typename F>
__device__ __forceinline__ void for_cells(int width, F&& f) {
    for (int k = threadIdx.x & 31; k < width; k += 32) {
        f((int)(threadIdx.x >> 5), k);
        f((int)(threadIdx.x >> 5) + 8, k);
    }
}

// JAC = false: sums of the loss gradient over the atoms.  JAC = true (FP64): one
// row of J per (atom, direction), nothing summed: a dense layer's block of a row
// is the outer product a[r] (x) zbar[r] + adot[r] (x) zdotbar[r] and a bias block
// is zbar[r], written to HBM with consecutive threads on consecutive parameters.
template <int MODE, bool JAC>
__global__ __launch_bounds__(256) void k_mlp_train(TrainArgs a) {
    typedef typename MT<MODE>::T T;
    extern __shared__ __align__(16) char smem[];
    int gi = 0;
    while (gi + 1 < a.n_net && (int)blockIdx.x >= a.net[gi + 1].block0) ++gi;
    const TrainNet& net = a.net[gi];
    const MlpShape& s = net.s;
    const int H = s.n_hidden;
    const int l = wave_lane(), tid = threadIdx.x;
    const int wv = uniform(tid >> 6);
    const int stride = a.stride;
    const size_t tile = (size_t)32 * stride;
    T* base = reinterpret_cast<T*>(smem);
    auto Abuf = [&](int h) { return base + h * tile; };
    auto Zbuf = [&](int h) { return base + (H + 1 + h) * tile; };
    T* P = base + (2 * H + 1) * tile;     // reverse buffers, swapped after each layer
    T* Q = P + tile;
    T* outv = Q + tile;                   // [0,16): zbar_L, [16,32): zdotbar_L
    T* gacc = outv + 32;
    const char* packed = net.packed;
    if (!JAC)
        for (int k = tid; k < net.nparam; k += 256) gacc[k] = T(0);
    const int row = l & 15, grp = l >> 4;
    const T* wout = (MODE == PT_MLP_F64) ? (const T*)(packed + s.wout64) : (const T*)(packed + s.wout32);
    const T bout = (MODE == PT_MLP_F64) ? (T)((const double*)(packed + s.bout64))[0]
                                        : (T)((const float*)(packed + s.bout32))[0];
    const int L = H;
    const int fan_L = H > 0 ? s.w[H - 1] : s.in_dim;
    const int ndir = JAC ? a.n_dir : 1;
    const int items = (net.n_atoms + 15) / 16 * ndir;
    for (int it = blockIdx.x - net.block0; it < items; it += net.nblocks) {
        const int a0 = it / ndir * 16, d = it % ndir;
        const int nrows = min(16, net.n_atoms - a0);
        // row r of this item in J
        auto Jrow = [&](int r) { return net.out + (size_t)((long long)(a0 + r) * ndir + d) * a.ldj; };
        // scaled input (rows 0..15) and its tangent (rows 16..31)
        for_cells(s.in_p, [&](int r, int k) {
            T v = T(0), t = T(0);
            if (r < nrows && k < s.in_dim) {
                const size_t o = (size_t)(a0 + r) * a.ldg + k, ot = o + (JAC ? (size_t)d * a.t_dir : 0);
                const double g = a.g_f64 ? ((const double*)net.G)[o] : (double)((const float*)net.G)[o];
                const double gt = a.g_f64 ? ((const double*)net.T)[ot] : (double)((const float*)net.T)[ot];
                v = (T)((g - net.scale[k]) * net.scale[s.in_dim + k] + net.scale_add);
                t = (T)(gt * net.scale[s.in_dim + k]);
            }
            Abuf(0)[r * stride + k] = v;
            Abuf(0)[(16 + r) * stride + k] = t;
        });
        __syncthreads();
        // forward: the products of (column tile, half) units in turn, then the activations
        int kin = s.in_p;
        for (int h = 0; h < H; ++h) {
            const int wp = s.wp[h];
            for (int u = wv; u < wp / 8; u += 4) {
                const int n0 = (u >> 1) * 16, half = (u & 1) * 16;
                const int col = n0 + row;
                T z[4] = {T(0), T(0), T(0), T(0)};
                if (n0 < s.w[h]) {
                    if (MODE == PT_MLP_F64)
                        gemm_tile<MODE>(Abuf(h) + half * stride, stride, kin, packed, s.W64[h], 0, wp, false, n0, z);
                    else
                        gemm_tile<MODE>(Abuf(h) + half * stride, stride, kin, packed, s.WTh[h], s.WTl[h], kin, true, n0, z);
                }
                const T bias = half ? T(0) : (MODE == PT_MLP_F64) ? (T)((const double*)(packed + s.b64[h]))[col]
                                                                  : (T)((const float*)(packed + s.b32[h]))[col];
                const bool pad = col >= s.w[h];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    Zbuf(h)[(half + crow<MODE>(grp, i)) * stride + col] = pad ? T(0) : z[i] + bias;
            }
            __syncthreads();
            for_cells(wp, [&](int r, int k) {
                T y, dy;
                activate<T>(s.act[h], Zbuf(h)[r * stride + k], y, dy);
                const bool pad = k >= s.w[h];
                Abuf(h + 1)[r * stride + k] = pad ? T(0) : y;
                Abuf(h + 1)[(16 + r) * stride + k] = pad ? T(0) : dy * Zbuf(h)[(16 + r) * stride + k];
            });
            __syncthreads();
            kin = wp;
        }
        // output layer and its reverse seeds: 4 lanes per atom, one wavefront
        if (wv == 0) {
            const int r = l >> 2, part = l & 3;
            T z = T(0), zd = T(0);
            for (int k = part; k < kin; k += 4) {
                z += Abuf(H)[r * stride + k] * wout[k];
                zd += Abuf(H)[(16 + r) * stride + k] * wout[k];
            }
            z += __shfl_xor(z, 1, kWave); z += __shfl_xor(z, 2, kWave);
            zd += __shfl_xor(zd, 1, kWave); zd += __shfl_xor(zd, 2, kWave);
            z += bout;
            T y, dy, ddy;
            activate2<T>(s.act_out, z, y, dy, ddy);
            const bool ok = r < nrows;
            const T gy = !JAC && ok ? (T)net.gy[a0 + r] : T(0);
            const T gt = ok ? (T)a.tseed : T(0);
            if (part == 0) {
                outv[r] = gy * dy + gt * ddy * zd;  // zbar_L
                outv[16 + r] = gt * dy;                  // zdotbar_L
            }
        }
        __syncthreads();
        // gradients of the output layer; abar, adotbar of the last hidden output -> P
        if constexpr (JAC) {
            for (int k = tid; k < fan_L; k += 256)
                for (int r = 0; r < nrows; ++r)
                    Jrow(r)[s.pW[L] + k] = Abuf(H)[r * stride + k] * outv[r] + Abuf(H)[(16 + r) * stride + k] * outv[16 + r];
            if (tid < nrows) Jrow(tid)[s.pb[L]] = outv[tid];
        } else {
            for (int k = tid; k < fan_L; k += 256) {
                T gw = T(0);
                for (int r = 0; r < 16; ++r)
                    gw += Abuf(H)[r * stride + k] * outv[r] + Abuf(H)[(16 + r) * stride + k] * outv[16 + r];
                gacc[s.pW[L] + k] += gw;
            }
            if (tid == 255) {
                T gb = T(0);
                for (int r = 0; r < 16; ++r) gb += outv[r];
                gacc[s.pb[L]] += gb;
            }
        }
        for (int h = H - 1; h >= 0; --h) {
            const int wp = s.wp[h];
            const int kin_h = h > 0 ? s.wp[h - 1] : s.in_p;
            // zbar = abar f'(z) + adotbar f''(z) zdot ; zdotbar = adotbar f'(z)   (in place)
            for_cells(wp, [&](int r, int k) {
                const T z = Zbuf(h)[r * stride + k], zd = Zbuf(h)[(16 + r) * stride + k];
                T y, dy, ddy;
                activate2<T>(s.act[h], z, y, dy, ddy);
                const T ab = h == H - 1 ? outv[r] * wout[k] : P[r * stride + k];
                const T adb = h == H - 1 ? outv[16 + r] * wout[k] : P[(16 + r) * stride + k];
                const bool pad = k >= s.w[h];
                P[r * stride + k] = pad ? T(0) : ab * dy + adb * ddy * zd;
                P[(16 + r) * stride + k] = pad ? T(0) : adb * dy;
            });
            __syncthreads();
            const int fan_in = h > 0 ? s.w[h - 1] : s.in_dim;
            const int wo = s.w[h];
            const T* A = Abuf(h);
            if constexpr (JAC) {
                // rows of J: W_h[in][out], q = in * wo + out (in and out advance without a division)
                const int nW = fan_in * wo, dq = 256 / wo, rq = 256 - dq * wo;
                int in = tid / wo, out = tid - in * wo;
                for (int q = tid; q < nW; q += 256) {
                    for (int r = 0; r < nrows; ++r)
                        Jrow(r)[s.pW[h] + q] = A[r * stride + in] * P[r * stride + out] +
                                               A[(16 + r) * stride + in] * P[(16 + r) * stride + out];
                    in += dq; out += rq;
                    if (out >= wo) { out -= wo; ++in; }
                }
                for (int k = tid; k < wo; k += 256)
                    for (int r = 0; r < nrows; ++r) Jrow(r)[s.pb[h] + k] = P[r * stride + k];
            } else {
                // dW_h += A_h^T [zbar; zdotbar]  (K = 32 rows), tiles in turn over the wavefronts
                const int to = (wo + 15) / 16, ti = (fan_in + 15) / 16;
                for (int u = wv; u < ti * to; u += 4) {
                    const int i0 = u / to * 16, o0 = u % to * 16;
                    T c[4];
                    wgrad_tile<MODE>(A, P, stride, i0, o0, c);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int in = i0 + crow<MODE>(grp, i), out = o0 + row;
                        if (in < fan_in && out < wo) gacc[s.pW[h] + (size_t)in * wo + out] += c[i];
                    }
                }
                for (int k = tid; k < wo; k += 256) {
                    T gb = T(0);
                    for (int r = 0; r < 16; ++r) gb += P[r * stride + k];
                    gacc[s.pb[h] + k] += gb;
                }
            }
            if (h > 0) {
                // [abar; adotbar] of layer h's input = [zbar; zdotbar] W_h^T  -> Q
                for (int u = wv; u < kin_h / 8; u += 4) {
                    const int n0 = (u >> 1) * 16, half = (u & 1) * 16;
                    T c[4] = {T(0), T(0), T(0), T(0)};
                    if (n0 < s.w[h - 1]) {
                        if (MODE == PT_MLP_F64)
                            gemm_tile<MODE>(P + half * stride, stride, wp, packed, s.W64[h], 0, wp, true, n0, c);
                        else
                            gemm_tile<MODE>(P + half * stride, stride, wp, packed, s.Wh[h], s.Wl[h], wp, true, n0, c);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) Q[(half + crow<MODE>(grp, i)) * stride + n0 + row] = c[i];
                }
                T* t = P; P = Q; Q = t;
            }
            __syncthreads();
        }
        __syncthreads();
    }
    if constexpr (!JAC) {
        __syncthreads();
        for (int k = tid; k < net.nparam; k += 256) {
            const double v = (double)gacc[k];
            if (v != 0.0) atomicAdd(&net.out[k], v);
        }
    }
}

constexpr int kTrainBlocks = 4096;   // of the sums: each ends with an atomic per parameter

// Workgroups of a launch's networks: an item each, shared out by items beyond
// kTrainBlocks.  Networks whose widest, deepest and largest need more LDS together
// than a workgroup has are launched one by one.
template <int MODE, bool JAC>
int launch_train(TrainArgs& a, hipStream_t st) {
    typedef typename MT<MODE>::T T;
    int wmax = 0, hid = 0, np = 0;
    long long total = 0;
    for (int g = 0; g < a.n_net; ++g) {
        wmax = std::max(wmax, a.net[g].s.wmax);
        hid = std::max(hid, a.net[g].s.n_hidden);
        np = std::max(np, a.net[g].nparam);
        total += (long long)((a.net[g].n_atoms + 15) / 16) * (JAC ? a.n_dir : 1);
    }
    a.stride = wmax + (sizeof(T) == 8 ? 1 : 4);
    const size_t bytes = train_lds(sizeof(T), hid, a.stride, JAC ? 0 : np);
    if (bytes > lds_limit() && a.n_net > 1) {
        TrainArgs one = a;
        one.n_net = 1;
        for (int g = 0; g < a.n_net; ++g) {
            one.net[0] = a.net[g];
            if (int rc = launch_train<MODE, JAC>(one, st)) return rc;
        }
        return PT_OK;
    }
    if (bytes > lds_limit()) {
        set_error("mlp training: %zu bytes of LDS per workgroup exceed the device limit", bytes);
        return PT_ERR_UNSUPPORTED;
    }
    const long long most = JAC ? 1 << 20 : kTrainBlocks;
    int blocks = 0;
    for (int g = 0; g < a.n_net; ++g) {
        const long long items = (long long)((a.net[g].n_atoms + 15) / 16) * (JAC ? a.n_dir : 1);
        a.net[g].block0 = blocks;
        a.net[g].nblocks = (int)std::max<long long>(1, std::min(items, items * most / std::max(total, 1LL) + 1));
        blocks += a.net[g].nblocks;
    }
    hipLaunchKernelGGL((k_mlp_train<MODE, JAC>), dim3(blocks), dim3(256), bytes, st, a);
    return launch_check("k_mlp_train");
}

// ---- loss seeds and Adam --------------------------------------------------------

__global__ void k_train_seeds(int n, const double* __restrict__ f, const double* __restrict__ fref,
                              const double* __restrict__ energy, double eref, double we, double wf,
                              double* __restrict__ delta, double* __restrict__ gy, double* __restrict__ loss) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const double de = energy[0] - eref;
    double s = 0.0;
    if (i < n) {
        for (int d = 0; d < 3; ++d) {
            const double r = f[3 * i + d] - fref[3 * i + d];
            delta[3 * i + d] = wf * 2.0 * r / (3.0 * n);
            s += r * r;
        }
        gy[i] = we * 2.0 * de / ((double)n * n);
    }
    s = wave_sum(s);  // all lanes of the (full) block take part
    if (wave_lane() == 0 && s != 0.0) atomicAdd(&loss[1], wf * s / (3.0 * n));
    if (i == 0) atomicAdd(&loss[0], we * de * de / ((double)n * n));
}

// Adam (Kingma & Ba 2015) with optional decoupled weight decay (AdamW).
__global__ void k_adam(int n, double* __restrict__ p, const double* __restrict__ g, double* __restrict__ m,
                       double* __restrict__ v, double lr, double b1, double b2, double eps, double wd,
                       double c1, double c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double gi = g[i];
    const double mi = b1 * m[i] + (1.0 - b1) * gi;
    const double vi = b2 * v[i] + (1.0 - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const double mh = mi / c1, vh = vi / c2;
    p[i] = p[i] - lr * (mh / (sqrt(vh) + eps) + wd * p[i]);
}

template <int MODE, int CT, int WC, int MTW, int HM>
int launch_mlp_cfg(MlpArgs& a, hipStream_t st) {
    typedef typename MT<MODE>::T T;
    constexpr int ROWS = mlp_rows<CT, WC, MTW>();
    int wmax = 0, blocks = 0;
    for (int g = 0; g < a.n_net; ++g) {
        wmax = std::max(wmax, a.net[g].s.wmax);
        a.net[g].block0 = blocks;
        blocks += (a.net[g].n_atoms + ROWS - 1) / ROWS;
    }
    // FP64 rows an odd number of 8-byte words apart; BF16 rows 16 bytes (a fragment) past a multiple of 64
    a.stride = wmax + (sizeof(T) == 8 ? 1 : 8);
    const size_t bytes = 2 * MlpLds<MODE>::bytes(ROWS, a.stride);
    if (bytes + sizeof(T) * WC * ROWS > lds_limit()) {
        set_error("mlp: layer widths need %zu bytes of LDS per workgroup", bytes);
        return PT_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL((k_mlp<MODE, CT, WC, MTW, HM>), dim3(blocks), dim3(256), bytes, st, a);
    return launch_check("k_mlp");
}

// Shape of the workgroup by the launch's rows.  Below the lines: 16 rows per
// workgroup, a column tile per wavefront, for the most wavefronts in flight.
// Above: 32 rows per workgroup, so that a weight fragment serves two row tiles;
// narrow FP64 networks (hidden layers of at most two column tiles, which leave
// wavefronts idle) split 64 rows over the four wavefronts instead.
// Measured, us per launch (16 rows | the other shape):
//   52-64-64-1 FP64      12,288 rows 26.9 | 31.5   32,768 rows 58.8 | 53.9   98,304 rows 153 | 137
//   52-64-64-1 BF16x3    12,288 rows 12.2 | 14.6   32,768 rows 23.0 | 19.2   98,304 rows 58.8 | 50.0
//   34-16-16-1 FP64      12,288 rows 12.8 | 17.8   32,768 rows 29.4 | 24.5   98,304 rows 78.3 | 65.0
//   34-16-16-1 BF16x3    32,768 rows 11.4 | 15.7   65,536 rows 21.0 | 19.6   98,304 rows 29.6 | 33.8 (16 rows stay)
//   linear, 120 inputs FP64, 30,000 rows 17.0 | 38.3   98,304 rows 47.1 | 109 (one wavefront for all columns: 16 rows stay)
// (64 rows per workgroup for the wide networks, 54.7 us at 98,304 rows in
// BF16x3, never won.)  One wavefront per 16 rows took 66 / 28 / 32 / 17 us for
// any size up to 12,288 rows and 245 / 85 / 117 / 42 us at 98,304.
constexpr long long kMlpWideRows = 20480, kMlpNarrowRows = 24576;

template <int MODE>
int launch_mlp(MlpArgs& a, hipStream_t st) {
    int wp = 0, hid = 0;
    long long n = 0;
    for (int g = 0; g < a.n_net; ++g) {
        const MlpShape& s = a.net[g].s;
        for (int h = 0; h < s.n_hidden; ++h) wp = std::max(wp, s.wp[h]);
        hid = std::max(hid, s.n_hidden);
        n += a.net[g].n_atoms;
    }
    if (wp > 64) return launch_mlp_cfg<MODE, 2, 4, 1, 3>(a, st);
    if (MODE == PT_MLP_F64 && hid > 0 && wp <= 32 && n >= kMlpNarrowRows) return launch_mlp_cfg<PT_MLP_F64, 2, 1, 1, 3>(a, st);
    if (hid <= 2 && wp > 32 && n >= kMlpWideRows) return launch_mlp_cfg<MODE, 1, 4, 2, 2>(a, st);
    return launch_mlp_cfg<MODE, 1, 4, 1, 3>(a, st);
}

}  // namespace
}  // namespace pt

using namespace pt;

extern "C" size_t pt_mlp_packed_bytes(const pt_mlp_desc* desc) {
    MlpShape s;
    if (make_shape(desc, s) != PT_OK) return 0;
    return s.total;
}

extern "C" int pt_mlp_pack(const pt_mlp_desc* desc, const double* params, void* packed,
                           pt_stream_t stream) {
    PT_REQUIRE(desc && params && packed, "pt_mlp_pack: null argument");
    MlpShape s;
    if (int rc = make_shape(desc, s)) return rc;
    int work = s.kout;
    int kin = s.in_p;
    for (int l = 0; l < s.n_hidden; ++l) { work = std::max(work, kin * s.wp[l]); kin = s.wp[l]; }
    hipLaunchKernelGGL(k_pack, dim3((work + 255) / 256), dim3(256), 0, (hipStream_t)stream, s, params,
                       (char*)packed);
    return launch_check("pt_mlp_pack");
}

extern "C" int pt_mlp_energy_grad_multi(int mode, int n_jobs, const pt_mlp_job* jobs, int ldg, int g_precision,
                                        pt_stream_t stream) {
    PT_REQUIRE(n_jobs >= 0 && (jobs || n_jobs == 0), "pt_mlp_energy_grad: bad job list");
    PT_REQUIRE(g_precision == PT_F64 || g_precision == PT_F32, "pt_mlp_energy_grad: bad precision");
    PT_REQUIRE(mode == PT_MLP_F64 || mode == PT_MLP_BF16 || mode == PT_MLP_BF16X3, "pt_mlp_energy_grad: unknown mode %d",
               mode);
    hipStream_t st = (hipStream_t)stream;
    MlpArgs a{};
    a.ldg = ldg;
    a.g_f64 = g_precision == PT_F64;
    for (int j = 0; j < n_jobs; ++j) {
        const pt_mlp_job& q = jobs[j];
        PT_REQUIRE(q.n_atoms >= 0, "pt_mlp_energy_grad: n_atoms < 0");
        if (q.n_atoms > 0) {
            PT_REQUIRE(q.G && q.scale && q.desc && q.packed && q.e_atom, "pt_mlp_energy_grad: null argument");
            MlpNet& t = a.net[a.n_net];
            if (int rc = make_shape(q.desc, t.s)) return rc;
            PT_REQUIRE(ldg >= q.desc->in_dim, "pt_mlp_energy_grad: ldg < in_dim");
            t.n_atoms = q.n_atoms;
            t.G = q.G;
            t.scale = q.scale;
            t.scale_add = q.desc->scale_add;
            t.packed = (const char*)q.packed;
            t.e_atom = q.e_atom;
            t.dEdG = q.dEdG;
            ++a.n_net;
        }
        if (a.n_net == kMlpNets || (j == n_jobs - 1 && a.n_net > 0)) {
            const int rc = mode == PT_MLP_F64    ? launch_mlp<PT_MLP_F64>(a, st)
                           : mode == PT_MLP_BF16 ? launch_mlp<PT_MLP_BF16>(a, st)
                                                 : launch_mlp<PT_MLP_BF16X3>(a, st);
            if (rc) return rc;
            a.n_net = 0;
        }
    }
    return PT_OK;
}

extern "C" int pt_mlp_energy_grad(int mode, int n_atoms, const void* G, int ldg, int g_precision,
                                  const double* scale, const pt_mlp_desc* desc, const void* packed,
                                  double* e_atom, void* dEdG, pt_stream_t stream) {
    PT_REQUIRE(n_atoms >= 0, "pt_mlp_energy_grad: n_atoms < 0");
    if (n_atoms == 0) return PT_OK;
    const pt_mlp_job job{n_atoms, G, scale, desc, packed, e_atom, dEdG};
    return pt_mlp_energy_grad_multi(mode, 1, &job, ldg, g_precision, stream);
}

extern "C" size_t pt_mlp_param_count(const pt_mlp_desc* desc) {
    MlpShape s;
    if (make_shape(desc, s) != PT_OK) return 0;
    return s.pb[s.n_hidden] + 1;
}

// a job of pt_mlp_train_grad_multi / pt_mlp_jacobian_multi as a network of the launch
static int train_net(const pt_mlp_train_job& q, int ldg, const char* what, pt::TrainNet& t) {
    PT_REQUIRE(q.n_atoms >= 0, "%s: n_atoms < 0", what);
    if (q.n_atoms == 0) return PT_OK;
    PT_REQUIRE(q.G && q.T && q.scale && q.desc && q.packed && q.out, "%s: null argument", what);
    if (int rc = make_shape(q.desc, t.s)) return rc;
    PT_REQUIRE(ldg >= q.desc->in_dim, "%s: ldg < in_dim", what);
    t.n_atoms = q.n_atoms;
    t.G = q.G;
    t.T = q.T;
    t.scale = q.scale;
    t.scale_add = q.desc->scale_add;
    t.packed = (const char*)q.packed;
    t.gy = q.gy;
    t.out = q.out;
    t.nparam = (int)(t.s.pb[t.s.n_hidden] + 1);
    return PT_OK;
}

extern "C" int pt_mlp_train_grad_multi(int mode, int n_jobs, const pt_mlp_train_job* jobs, int ldg, int g_precision,
                                       double tseed, pt_stream_t stream) {
    PT_REQUIRE(n_jobs >= 0 && (jobs || n_jobs == 0), "pt_mlp_train_grad: bad job list");
    PT_REQUIRE(g_precision == PT_F64 || g_precision == PT_F32, "pt_mlp_train_grad: bad precision");
    PT_REQUIRE(mode == PT_MLP_F64 || mode == PT_MLP_BF16 || mode == PT_MLP_BF16X3, "pt_mlp_train_grad: unknown mode %d",
               mode);
    hipStream_t st = (hipStream_t)stream;
    TrainArgs a{};
    a.ldg = ldg;
    a.g_f64 = g_precision == PT_F64;
    a.tseed = tseed;
    for (int j = 0; j < n_jobs; ++j) {
        PT_REQUIRE(jobs[j].gy || jobs[j].n_atoms == 0, "pt_mlp_train_grad: null argument");
        if (int rc = train_net(jobs[j], ldg, "pt_mlp_train_grad", a.net[a.n_net])) return rc;
        if (jobs[j].n_atoms > 0) ++a.n_net;
        if (a.n_net == kMlpNets || (j == n_jobs - 1 && a.n_net > 0)) {
            const int rc = mode == PT_MLP_F64    ? launch_train<PT_MLP_F64, false>(a, st)
                           : mode == PT_MLP_BF16 ? launch_train<PT_MLP_BF16, false>(a, st)
                                                 : launch_train<PT_MLP_BF16X3, false>(a, st);
            if (rc) return rc;
            a.n_net = 0;
        }
    }
    return PT_OK;
}

extern "C" int pt_mlp_train_grad(int mode, int n_atoms, const void* G, const void* T, int ldg,
                                 int g_precision, const double* scale, const pt_mlp_desc* desc,
                                 const void* packed, const double* gy, double tseed, double* grad,
                                 pt_stream_t stream) {
    PT_REQUIRE(n_atoms >= 0, "pt_mlp_train_grad: n_atoms < 0");
    if (n_atoms == 0) return PT_OK;
    const pt_mlp_train_job job{n_atoms, G, T, scale, desc, packed, gy, grad};
    return pt_mlp_train_grad_multi(mode, 1, &job, ldg, g_precision, tseed, stream);
}

extern "C" int pt_mlp_jacobian_multi(int n_dir, int n_jobs, const pt_mlp_train_job* jobs, long long t_dir, int ldg,
                                     double sign, long long ldj, pt_stream_t stream) {
    PT_REQUIRE(n_dir >= 1, "pt_mlp_jacobian: n_atoms < 0 or n_dir < 1");
    PT_REQUIRE(n_jobs >= 0 && (jobs || n_jobs == 0), "pt_mlp_jacobian: bad job list");
    TrainArgs a{};
    a.ldg = ldg;
    a.g_f64 = 1;
    a.tseed = sign;
    a.n_dir = n_dir;
    a.t_dir = t_dir;
    a.ldj = ldj;
    for (int j = 0; j < n_jobs; ++j) {
        TrainNet& t = a.net[a.n_net];
        if (int rc = train_net(jobs[j], ldg, "pt_mlp_jacobian", t)) return rc;
        if (jobs[j].n_atoms > 0) {
            PT_REQUIRE(t_dir >= (long long)(t.n_atoms - 1) * ldg + jobs[j].desc->in_dim || n_dir == 1,
                       "pt_mlp_jacobian: tangent directions overlap");
            PT_REQUIRE(ldj >= t.nparam, "pt_mlp_jacobian: ldj below the parameter count");
            PT_REQUIRE((long long)t.n_atoms * n_dir < (1LL << 31), "pt_mlp_jacobian: too many rows");
            ++a.n_net;
        }
        if (a.n_net == kMlpNets || (j == n_jobs - 1 && a.n_net > 0)) {
            if (int rc = launch_train<PT_MLP_F64, true>(a, (hipStream_t)stream)) return rc;
            a.n_net = 0;
        }
    }
    return PT_OK;
}

extern "C" int pt_mlp_jacobian(int n_atoms, int n_dir, const double* G, const double* T, long long t_dir, int ldg,
                               const double* scale, const pt_mlp_desc* desc, const void* packed, double sign,
                               double* J, long long ldj, pt_stream_t stream) {
    PT_REQUIRE(n_atoms >= 0 && n_dir >= 1, "pt_mlp_jacobian: n_atoms < 0 or n_dir < 1");
    if (n_atoms == 0) return PT_OK;
    const pt_mlp_train_job job{n_atoms, G, T, scale, desc, packed, nullptr, J};
    return pt_mlp_jacobian_multi(n_dir, 1, &job, t_dir, ldg, sign, ldj, stream);
}

extern "C" int pt_train_seeds(int n, const double* force, const double* force_ref, const double* energy,
                              double energy_ref, double w_energy, double w_force, double* delta, double* gy,
                              double* loss, pt_stream_t stream) {
    PT_REQUIRE(n > 0 && force && force_ref && energy && delta && gy && loss, "pt_train_seeds: bad arguments");
    hipLaunchKernelGGL(k_train_seeds, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, n, force,
                       force_ref, energy, energy_ref, w_energy, w_force, delta, gy, loss);
    return launch_check("pt_train_seeds");
}

extern "C" int pt_adam_step(int n, double* params, const double* grad, double* m, double* v, double lr,
                            double beta1, double beta2, double eps, double weight_decay, int step,
                            pt_stream_t stream) {
    PT_REQUIRE(n >= 0 && params && grad && m && v && step >= 1, "pt_adam_step: bad arguments");
    if (n == 0) return PT_OK;
    const double c1 = 1.0 - pow(beta1, step), c2 = 1.0 - pow(beta2, step);
    hipLaunchKernelGGL(k_adam, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, n, params, grad, m, v,
                       lr, beta1, beta2, eps, weight_decay, c1, c2);
    return launch_check("pt_adam_step");
}
