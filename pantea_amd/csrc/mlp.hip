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

    // 1. scaled input, zero padded: 32 columns x 8 rows per step
    for (int k0 = 0; k0 < s.in_p; k0 += 32) {
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

struct TrainArgs {
    MlpShape s;
    int n_atoms;
    const void* G;
    const void* T;
    int ldg;
    int g_f64;
    const double* scale;
    double scale_add;
    const char* packed;
    const double* gy;     // per-atom seed of y
    double tseed;         // seed of ydot (same for every atom)
    double* grad;         // parameter gradient, FP64, layout of the unpacked params
    int stride;
    int nparam;
};

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int MODE>
__global__ __launch_bounds__(256) void k_mlp_train(TrainArgs a) {
    typedef typename MT<MODE>::T T;
    extern __shared__ __align__(16) char smem[];
    const MlpShape& s = a.s;
    const int H = s.n_hidden;
    const int l = wave_lane();
    const int wv = threadIdx.x >> 6;
    const int wpb = blockDim.x >> 6;
    const int stride = a.stride;
    const size_t tile = (size_t)32 * stride;
    const size_t per_wave = (size_t)(2 * H + 3) * tile + 64 + a.nparam;
    T* base = reinterpret_cast<T*>(smem) + (size_t)wv * per_wave;
    T* Abuf[kMaxHidden + 1];
    T* Zbuf[kMaxHidden];
    for (int h = 0; h <= H; ++h) Abuf[h] = base + h * tile;
    for (int h = 0; h < H; ++h) Zbuf[h] = base + (H + 1 + h) * tile;
    T* P[2] = {base + (2 * H + 1) * tile, base + (2 * H + 2) * tile};
    T* outv = base + (2 * H + 3) * tile;  // [0,16): z_L, [16,32): zdot_L, [32,48): zbar_L, [48,64): zdotbar_L
    T* gacc = outv + 64;
    for (int k = l; k < a.nparam; k += kWave) gacc[k] = T(0);
    const int row = l & 15, grp = l >> 4;
    const T* wout = (MODE == PT_MLP_F64) ? (const T*)(a.packed + s.wout64) : (const T*)(a.packed + s.wout32);
    const T bout = (MODE == PT_MLP_F64) ? (T)((const double*)(a.packed + s.bout64))[0]
                                        : (T)((const float*)(a.packed + s.bout32))[0];
    const int ntiles = (a.n_atoms + 15) / 16;
    for (int tl = blockIdx.x * wpb + wv; tl < ntiles; tl += gridDim.x * wpb) {
        const int a0 = tl * 16;
        // scaled input and its tangent
        for (int e = l; e < 16 * s.in_p; e += kWave) {
            const int r = e / s.in_p, k = e % s.in_p;
            const int atom = a0 + r;
            T v = T(0), t = T(0);
            if (atom < a.n_atoms && k < s.in_dim) {
                const size_t o = (size_t)atom * a.ldg + k;
                const double g = a.g_f64 ? ((const double*)a.G)[o] : (double)((const float*)a.G)[o];
                const double gt = a.g_f64 ? ((const double*)a.T)[o] : (double)((const float*)a.T)[o];
                v = (T)((g - a.scale[k]) * a.scale[s.in_dim + k] + a.scale_add);
                t = (T)(gt * a.scale[s.in_dim + k]);
            }
            Abuf[0][r * stride + k] = v;
            Abuf[0][(16 + r) * stride + k] = t;
        }
        wave_fence();
        // forward: primal rows 0..15, tangent rows 16..31
        int kin = s.in_p;
        for (int h = 0; h < H; ++h) {
            const int wp = s.wp[h];
            for (int n0 = 0; n0 < wp; n0 += 16) {
                T az[4] = {T(0), T(0), T(0), T(0)}, at[4] = {T(0), T(0), T(0), T(0)};
                if (MODE == PT_MLP_F64) {
                    gemm_tile<MODE>(Abuf[h], stride, kin, a.packed, s.W64[h], 0, wp, false, n0, az);
                    gemm_tile<MODE>(Abuf[h] + 16 * stride, stride, kin, a.packed, s.W64[h], 0, wp, false, n0, at);
                } else {
                    gemm_tile<MODE>(Abuf[h], stride, kin, a.packed, s.WTh[h], s.WTl[h], kin, true, n0, az);
                    gemm_tile<MODE>(Abuf[h] + 16 * stride, stride, kin, a.packed, s.WTh[h], s.WTl[h], kin, true, n0, at);
                }
                const int col = n0 + row;
                const T bias = (MODE == PT_MLP_F64) ? (T)((const double*)(a.packed + s.b64[h]))[col]
                                                    : (T)((const float*)(a.packed + s.b32[h]))[col];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = crow<MODE>(grp, i);
                    const T z = az[i] + bias, zd = at[i];
                    T y, dy;
                    activate<T>(s.act[h], z, y, dy);
                    const bool pad = col >= s.w[h];
                    Zbuf[h][r * stride + col] = pad ? T(0) : z;
                    Zbuf[h][(16 + r) * stride + col] = pad ? T(0) : zd;
                    Abuf[h + 1][r * stride + col] = pad ? T(0) : y;
                    Abuf[h + 1][(16 + r) * stride + col] = pad ? T(0) : dy * zd;
                }
            }
            wave_fence();
            kin = wp;
        }
        // output layer and its reverse seeds: 4 lanes per atom
        {
            const int r = l >> 2, part = l & 3;
            T z = T(0), zd = T(0);
            for (int k = part; k < kin; k += 4) {
                z += Abuf[H][r * stride + k] * wout[k];
                zd += Abuf[H][(16 + r) * stride + k] * wout[k];
            }
            z += __shfl_xor(z, 1, kWave); z += __shfl_xor(z, 2, kWave);
            zd += __shfl_xor(zd, 1, kWave); zd += __shfl_xor(zd, 2, kWave);
            z += bout;
            T y, dy, ddy;
            activate2<T>(s.act_out, z, y, dy, ddy);
            const int atom = a0 + r;
            const bool ok = atom < a.n_atoms;
            const T gy = ok ? (T)a.gy[atom] : T(0);
            const T gt = ok ? (T)a.tseed : T(0);
            if (part == 0) {
                outv[r] = z;
                outv[16 + r] = zd;
                outv[32 + r] = gy * dy + gt * ddy * zd;  // zbar_L
                outv[48 + r] = gt * dy;                  // zdotbar_L
            }
        }
        wave_fence();
        // gradients of the output layer
        const int L = H;
        for (int k = l; k < kin; k += kWave) {
            T gw = T(0);
            for (int r = 0; r < 16; ++r)
                gw += Abuf[H][r * stride + k] * outv[32 + r] + Abuf[H][(16 + r) * stride + k] * outv[48 + r];
            const int fan_in = H > 0 ? s.w[H - 1] : s.in_dim;
            if (k < fan_in) gacc[s.pW[L] + k] += gw;
        }
        if (l == 0) {
            T gb = T(0);
            for (int r = 0; r < 16; ++r) gb += outv[32 + r];
            gacc[s.pb[L]] += gb;
        }
        // abar, adotbar of the last hidden output -> P[0]
        for (int e = l; e < 16 * kin; e += kWave) {
            const int r = e / kin, k = e % kin;
            P[0][r * stride + k] = outv[32 + r] * wout[k];
            P[0][(16 + r) * stride + k] = outv[48 + r] * wout[k];
        }
        wave_fence();
        int cur = 0;
        for (int h = H - 1; h >= 0; --h) {
            const int wp = s.wp[h];
            const int kin_h = h > 0 ? s.wp[h - 1] : s.in_p;
            // zbar = abar f'(z) + adotbar f''(z) zdot ; zdotbar = adotbar f'(z)   (in place)
            for (int e = l; e < 16 * wp; e += kWave) {
                const int r = e / wp, k = e % wp;
                const T z = Zbuf[h][r * stride + k], zd = Zbuf[h][(16 + r) * stride + k];
                T y, dy, ddy;
                activate2<T>(s.act[h], z, y, dy, ddy);
                const T ab = P[cur][r * stride + k], adb = P[cur][(16 + r) * stride + k];
                const bool pad = k >= s.w[h];
                P[cur][r * stride + k] = pad ? T(0) : ab * dy + adb * ddy * zd;
                P[cur][(16 + r) * stride + k] = pad ? T(0) : adb * dy;
            }
            wave_fence();
            // dW_h += A_h^T [zbar; zdotbar]  (K = 32 rows)
            const int fan_in = h > 0 ? s.w[h - 1] : s.in_dim;
            for (int i0 = 0; i0 < kin_h; i0 += 16) {
                for (int o0 = 0; o0 < wp; o0 += 16) {
                    T c[4];
                    wgrad_tile<MODE>(Abuf[h], P[cur], stride, i0, o0, c);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int in = i0 + crow<MODE>(grp, i), out = o0 + row;
                        if (in < fan_in && out < s.w[h]) gacc[s.pW[h] + (size_t)in * s.w[h] + out] += c[i];
                    }
                }
            }
            for (int k = l; k < s.w[h]; k += kWave) {
                T gb = T(0);
                for (int r = 0; r < 16; ++r) gb += P[cur][r * stride + k];
                gacc[s.pb[h] + k] += gb;
            }
            if (h > 0) {
                // [abar; adotbar] of layer h's input = [zbar; zdotbar] W_h^T  -> P[cur ^ 1]
                for (int n0 = 0; n0 < kin_h; n0 += 16) {
                    T c0[4] = {T(0), T(0), T(0), T(0)}, c1[4] = {T(0), T(0), T(0), T(0)};
                    if (MODE == PT_MLP_F64) {
                        gemm_tile<MODE>(P[cur], stride, wp, a.packed, s.W64[h], 0, wp, true, n0, c0);
                        gemm_tile<MODE>(P[cur] + 16 * stride, stride, wp, a.packed, s.W64[h], 0, wp, true, n0, c1);
                    } else {
                        gemm_tile<MODE>(P[cur], stride, wp, a.packed, s.Wh[h], s.Wl[h], wp, true, n0, c0);
                        gemm_tile<MODE>(P[cur] + 16 * stride, stride, wp, a.packed, s.Wh[h], s.Wl[h], wp, true, n0, c1);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = crow<MODE>(grp, i);
                        P[cur ^ 1][r * stride + n0 + row] = c0[i];
                        P[cur ^ 1][(16 + r) * stride + n0 + row] = c1[i];
                    }
                }
                cur ^= 1;
            }
            wave_fence();
        }
    }
    wave_fence();
    for (int k = l; k < a.nparam; k += kWave) {
        const double v = (double)gacc[k];
        if (v != 0.0) atomicAdd(&a.grad[k], v);
    }
}

template <int MODE>
int launch_train(TrainArgs a, hipStream_t st) {
    typedef typename MT<MODE>::T T;
    const int H = a.s.n_hidden;
    a.stride = a.s.wmax + (sizeof(T) == 8 ? 1 : 4);
    const size_t per_wave = sizeof(T) * ((size_t)(2 * H + 3) * 32 * a.stride + 64 + a.nparam);
    const size_t budget = lds_limit();
    if (per_wave > budget) {
        set_error("mlp training: %zu bytes of LDS per wavefront exceed the device limit", per_wave);
        return PT_ERR_UNSUPPORTED;
    }
    const int wpb = (int)std::min<size_t>(4, budget / per_wave);
    const int ntiles = (a.n_atoms + 15) / 16;
    const int blocks = std::max(1, std::min((ntiles + wpb - 1) / wpb, 1024));
    hipLaunchKernelGGL(k_mlp_train<MODE>, dim3(blocks), dim3(64 * wpb), wpb * per_wave, st, a);
    return launch_check("k_mlp_train");
}

// ---- per-row Jacobian of the input-gradient projection (FP64) -----------------
//
// Row (atom r, direction d) of J is  sign * d(ydot_d)/dtheta,  with
// ydot_d = grad_x' MLP . (T_d * mul) the MLP output's derivative along the
// scaled tangent of direction d.  The forward-over-reverse sweep is the one of
// k_mlp_train (primal rows 0..15 once per tile, tangent rows 16..31 once per
// direction), but nothing is summed over atoms: a dense layer's block of a
// row is the outer product  a[r] (x) zbar[r] + adot[r] (x) zdotbar[r]  and a
// bias block is zbar[r], written straight to HBM with consecutive lanes on
// consecutive parameters of one row.
struct JacArgs {
    MlpShape s;
    int n_atoms;
    const double* G;
    const double* T;      // T[d * t_dir + atom * ldg + k]
    long long t_dir;
    int n_dir;
    int ldg;
    const double* scale;
    double scale_add;
    const char* packed;
    double sign;
    double* J;            // row (atom * n_dir + d), unpacked parameter layout
    long long ldj;
    int stride;
};

__global__ __launch_bounds__(256) void k_mlp_jacobian(JacArgs a) {
    typedef double T;
    constexpr int MODE = PT_MLP_F64;
    extern __shared__ __align__(16) char smem[];
    const MlpShape& s = a.s;
    const int H = s.n_hidden;
    const int l = wave_lane();
    const int wv = threadIdx.x >> 6;
    const int wpb = blockDim.x >> 6;
    const int stride = a.stride;
    const size_t tile = (size_t)32 * stride;
    const size_t per_wave = (size_t)(2 * H + 3) * tile + 64;
    T* base = reinterpret_cast<T*>(smem) + (size_t)wv * per_wave;
    T* Abuf[kMaxHidden + 1];
    T* Zbuf[kMaxHidden];
    for (int h = 0; h <= H; ++h) Abuf[h] = base + h * tile;
    for (int h = 0; h < H; ++h) Zbuf[h] = base + (H + 1 + h) * tile;
    T* P[2] = {base + (2 * H + 1) * tile, base + (2 * H + 2) * tile};
    T* outv = base + (2 * H + 3) * tile;  // [0,16): z_L, [32,48): zbar_L, [48,64): zdotbar_L
    const int row = l & 15, grp = l >> 4;
    const T* wout = (const T*)(a.packed + s.wout64);
    const T bout = ((const double*)(a.packed + s.bout64))[0];
    const int L = H;
    const int fan_L = H > 0 ? s.w[H - 1] : s.in_dim;
    const int ntiles = (a.n_atoms + 15) / 16;
    // one work item = (16-atom tile, direction): the primal sweep is redone per direction
    for (int it = blockIdx.x * wpb + wv; it < ntiles * a.n_dir; it += gridDim.x * wpb) {
        const int a0 = (it / a.n_dir) * 16;
        const int d = it % a.n_dir;
        const int nrows = min(16, a.n_atoms - a0);
        for (int e = l; e < 16 * s.in_p; e += kWave) {
            const int r = e / s.in_p, k = e % s.in_p;
            T v = T(0);
            if (r < nrows && k < s.in_dim)
                v = (a.G[(size_t)(a0 + r) * a.ldg + k] - a.scale[k]) * a.scale[s.in_dim + k] + a.scale_add;
            Abuf[0][r * stride + k] = v;
        }
        wave_fence();
        // primal forward, rows 0..15 (kept for every direction)
        int kin = s.in_p;
        for (int h = 0; h < H; ++h) {
            const int wp = s.wp[h];
            for (int n0 = 0; n0 < wp; n0 += 16) {
                T az[4] = {T(0), T(0), T(0), T(0)};
                gemm_tile<MODE>(Abuf[h], stride, kin, a.packed, s.W64[h], 0, wp, false, n0, az);
                const int col = n0 + row;
                const T bias = ((const double*)(a.packed + s.b64[h]))[col];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = crow<MODE>(grp, i);
                    T y, dy;
                    const T z = az[i] + bias;
                    activate<T>(s.act[h], z, y, dy);
                    const bool pad = col >= s.w[h];
                    Zbuf[h][r * stride + col] = pad ? T(0) : z;
                    Abuf[h + 1][r * stride + col] = pad ? T(0) : y;
                }
            }
            wave_fence();
            kin = wp;
        }
        {
            const int r = l >> 2, part = l & 3;
            T z = T(0);
            for (int k = part; k < kin; k += 4) z += Abuf[H][r * stride + k] * wout[k];
            z += __shfl_xor(z, 1, kWave);
            z += __shfl_xor(z, 2, kWave);
            if (part == 0) outv[r] = z + bout;
        }
        wave_fence();
        {
            // tangent input, rows 16..31
            for (int e = l; e < 16 * s.in_p; e += kWave) {
                const int r = e / s.in_p, k = e % s.in_p;
                T t = T(0);
                if (r < nrows && k < s.in_dim)
                    t = a.T[(size_t)d * a.t_dir + (size_t)(a0 + r) * a.ldg + k] * a.scale[s.in_dim + k];
                Abuf[0][(16 + r) * stride + k] = t;
            }
            wave_fence();
            kin = s.in_p;
            for (int h = 0; h < H; ++h) {
                const int wp = s.wp[h];
                for (int n0 = 0; n0 < wp; n0 += 16) {
                    T at[4] = {T(0), T(0), T(0), T(0)};
                    gemm_tile<MODE>(Abuf[h] + 16 * stride, stride, kin, a.packed, s.W64[h], 0, wp, false, n0, at);
                    const int col = n0 + row;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = crow<MODE>(grp, i);
                        T y, dy;
                        activate<T>(s.act[h], Zbuf[h][r * stride + col], y, dy);
                        const bool pad = col >= s.w[h];
                        Zbuf[h][(16 + r) * stride + col] = pad ? T(0) : at[i];
                        Abuf[h + 1][(16 + r) * stride + col] = pad ? T(0) : dy * at[i];
                    }
                }
                wave_fence();
                kin = wp;
            }
            // output layer: seeds of the projection's reverse sweep
            {
                const int r = l >> 2, part = l & 3;
                T zd = T(0);
                for (int k = part; k < kin; k += 4) zd += Abuf[H][(16 + r) * stride + k] * wout[k];
                zd += __shfl_xor(zd, 1, kWave);
                zd += __shfl_xor(zd, 2, kWave);
                T y, dy, ddy;
                activate2<T>(s.act_out, outv[r], y, dy, ddy);
                const T gt = r < nrows ? (T)a.sign : T(0);
                if (part == 0) {
                    outv[32 + r] = gt * ddy * zd;  // zbar_L
                    outv[48 + r] = gt * dy;        // zdotbar_L
                }
            }
            wave_fence();
            // rows of J: output layer
            for (int e = l; e < 16 * fan_L; e += kWave) {
                const int r = e / fan_L, k = e % fan_L;
                if (r < nrows)
                    a.J[(size_t)((a0 + r) * a.n_dir + d) * a.ldj + s.pW[L] + k] =
                        Abuf[H][r * stride + k] * outv[32 + r] + Abuf[H][(16 + r) * stride + k] * outv[48 + r];
            }
            if (l < nrows) a.J[(size_t)((a0 + l) * a.n_dir + d) * a.ldj + s.pb[L]] = outv[32 + l];
            for (int e = l; e < 16 * kin; e += kWave) {
                const int r = e / kin, k = e % kin;
                P[0][r * stride + k] = outv[32 + r] * wout[k];
                P[0][(16 + r) * stride + k] = outv[48 + r] * wout[k];
            }
            wave_fence();
            int cur = 0;
            for (int h = H - 1; h >= 0; --h) {
                const int wp = s.wp[h];
                const int kin_h = h > 0 ? s.wp[h - 1] : s.in_p;
                for (int e = l; e < 16 * wp; e += kWave) {
                    const int r = e / wp, k = e % wp;
                    const T z = Zbuf[h][r * stride + k], zd = Zbuf[h][(16 + r) * stride + k];
                    T y, dy, ddy;
                    activate2<T>(s.act[h], z, y, dy, ddy);
                    const T ab = P[cur][r * stride + k], adb = P[cur][(16 + r) * stride + k];
                    const bool pad = k >= s.w[h];
                    P[cur][r * stride + k] = pad ? T(0) : ab * dy + adb * ddy * zd;
                    P[cur][(16 + r) * stride + k] = pad ? T(0) : adb * dy;
                }
                wave_fence();
                // rows of J: W_h[in][out] and b_h[out]
                const int fan_in = h > 0 ? s.w[h - 1] : s.in_dim;
                const int wo = s.w[h];
                const int nW = fan_in * wo;
                for (int e = l; e < 16 * nW; e += kWave) {
                    const int r = e / nW, q = e % nW;
                    const int in = q / wo, out = q % wo;
                    if (r < nrows)
                        a.J[(size_t)((a0 + r) * a.n_dir + d) * a.ldj + s.pW[h] + q] =
                            Abuf[h][r * stride + in] * P[cur][r * stride + out] +
                            Abuf[h][(16 + r) * stride + in] * P[cur][(16 + r) * stride + out];
                }
                for (int e = l; e < 16 * wo; e += kWave) {
                    const int r = e / wo, out = e % wo;
                    if (r < nrows) a.J[(size_t)((a0 + r) * a.n_dir + d) * a.ldj + s.pb[h] + out] = P[cur][r * stride + out];
                }
                if (h > 0) {
                    for (int n0 = 0; n0 < kin_h; n0 += 16) {
                        T c0[4] = {T(0), T(0), T(0), T(0)}, c1[4] = {T(0), T(0), T(0), T(0)};
                        gemm_tile<MODE>(P[cur], stride, wp, a.packed, s.W64[h], 0, wp, true, n0, c0);
                        gemm_tile<MODE>(P[cur] + 16 * stride, stride, wp, a.packed, s.W64[h], 0, wp, true, n0, c1);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int r = crow<MODE>(grp, i);
                            P[cur ^ 1][r * stride + n0 + row] = c0[i];
                            P[cur ^ 1][(16 + r) * stride + n0 + row] = c1[i];
                        }
                    }
                    cur ^= 1;
                }
                wave_fence();
            }
        }
    }
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
    if (MODE == PT_MLP_F64 && wp <= 32 && n >= kMlpNarrowRows) return launch_mlp_cfg<PT_MLP_F64, 2, 1, 1, 3>(a, st);
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

extern "C" int pt_mlp_train_grad(int mode, int n_atoms, const void* G, const void* T, int ldg,
                                 int g_precision, const double* scale, const pt_mlp_desc* desc,
                                 const void* packed, const double* gy, double tseed, double* grad,
                                 pt_stream_t stream) {
    PT_REQUIRE(n_atoms >= 0, "pt_mlp_train_grad: n_atoms < 0");
    if (n_atoms == 0) return PT_OK;
    PT_REQUIRE(G && T && scale && desc && packed && gy && grad, "pt_mlp_train_grad: null argument");
    PT_REQUIRE(g_precision == PT_F64 || g_precision == PT_F32, "pt_mlp_train_grad: bad precision");
    TrainArgs a{};
    if (int rc = make_shape(desc, a.s)) return rc;
    PT_REQUIRE(ldg >= desc->in_dim, "pt_mlp_train_grad: ldg < in_dim");
    a.n_atoms = n_atoms;
    a.G = G;
    a.T = T;
    a.ldg = ldg;
    a.g_f64 = g_precision == PT_F64;
    a.scale = scale;
    a.scale_add = desc->scale_add;
    a.packed = (const char*)packed;
    a.gy = gy;
    a.tseed = tseed;
    a.grad = grad;
    a.nparam = (int)(a.s.pb[a.s.n_hidden] + 1);
    hipStream_t st = (hipStream_t)stream;
    switch (mode) {
    case PT_MLP_F64: return launch_train<PT_MLP_F64>(a, st);
    case PT_MLP_BF16: return launch_train<PT_MLP_BF16>(a, st);
    case PT_MLP_BF16X3: return launch_train<PT_MLP_BF16X3>(a, st);
    }
    set_error("pt_mlp_train_grad: unknown mode %d", mode);
    return PT_ERR_ARG;
}

extern "C" int pt_mlp_jacobian(int n_atoms, int n_dir, const double* G, const double* T, long long t_dir, int ldg,
                               const double* scale, const pt_mlp_desc* desc, const void* packed, double sign,
                               double* J, long long ldj, pt_stream_t stream) {
    PT_REQUIRE(n_atoms >= 0 && n_dir >= 1, "pt_mlp_jacobian: n_atoms < 0 or n_dir < 1");
    if (n_atoms == 0) return PT_OK;
    PT_REQUIRE(G && T && scale && desc && packed && J, "pt_mlp_jacobian: null argument");
    JacArgs a{};
    if (int rc = make_shape(desc, a.s)) return rc;
    PT_REQUIRE(ldg >= desc->in_dim, "pt_mlp_jacobian: ldg < in_dim");
    PT_REQUIRE(t_dir >= (long long)(n_atoms - 1) * ldg + desc->in_dim || n_dir == 1,
               "pt_mlp_jacobian: tangent directions overlap");
    const long long np = (long long)(a.s.pb[a.s.n_hidden] + 1);
    PT_REQUIRE(ldj >= np, "pt_mlp_jacobian: ldj below the parameter count");
    PT_REQUIRE((long long)n_atoms * n_dir < (1LL << 31), "pt_mlp_jacobian: too many rows");
    a.n_atoms = n_atoms;
    a.n_dir = n_dir;
    a.G = G;
    a.T = T;
    a.t_dir = t_dir;
    a.ldg = ldg;
    a.scale = scale;
    a.scale_add = desc->scale_add;
    a.packed = (const char*)packed;
    a.sign = sign;
    a.J = J;
    a.ldj = ldj;
    a.stride = a.s.wmax + 1;
    const size_t per_wave = sizeof(double) * ((size_t)(2 * a.s.n_hidden + 3) * 32 * a.stride + 64);
    const size_t budget = lds_limit();
    if (per_wave > budget) {
        set_error("pt_mlp_jacobian: %zu bytes of LDS per wavefront exceed the device limit", per_wave);
        return PT_ERR_UNSUPPORTED;
    }
    const int wpb = (int)std::min<size_t>(4, budget / per_wave);
    const long long items = (long long)((n_atoms + 15) / 16) * n_dir;
    const int blocks = (int)std::max<long long>(1, std::min<long long>((items + wpb - 1) / wpb, 8192));
    hipLaunchKernelGGL(k_mlp_jacobian, dim3(blocks), dim3(64 * wpb), wpb * per_wave, (hipStream_t)stream, a);
    return launch_check("k_mlp_jacobian");
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
