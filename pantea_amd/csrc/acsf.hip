// (b) ACSF descriptors, their adjoint and their tangent on gfx950.
//
// One wavefront (64 lanes) per centre, or a team of 4 or 8 when a
// launch has too few centres to fill the chip.  The centre's neighbour row is staged
// in LDS (relative vectors R_ij = r_i - r_j under the minimum image with r_ij
// or 1/r_ij, and per mode the cutoff values), compacted to r_ij <= rc_max and
// r_ij > 0 (atoms/neighbor.py:102-107).  Rows arrive sorted by type, so each
// neighbour element is a contiguous LDS segment.
//
// Radial groups (descriptors/acsf/radial.py:38-61, acsf.py:231-246):
//   G2_s = sum_j exp(-eta_s (r_ij - rs_s)^2) fc(r_ij), lanes over neighbours.
// Angular groups (angular.py:50-107, acsf.py:249-330): every unordered pair
// {j, k} of the group's segments is visited once (for equal neighbour
// elements this equals the reference's ordered sum halved).  With
//   S = r_ij^2 + r_ik^2 + r_jk^2,  F = fc(r_ij) fc(r_ik) fc(r_jk)
// (G9: S and F without the r_jk terms), each function of the group is a cell
// (eta e, angular term a) of an outer product:
//   term(e, a) = exp(-eta_e S) F * pre_a (1 + lam_a cos)^zeta_a .
// r_jk = |MIC(R_ij - R_ik)| as in the reference (the MIC is skipped when the
// box exceeds 4 rc, where it cannot act), and pairs with r_jk = 0 are
// excluded (acsf.py:325).  Pairs are first screened (r_jk < rc for G3) and
// the live ones compacted into a per-wave LDS queue, so the heavy per-pair
// work runs on full wavefronts.
//
// The adjoint (MODE_ADJ) reverses the same loops with w = dE/dG.  Per pair
// only two eta sums are needed, SP = sum_e P_e and SEP = sum_e eta_e P_e with
// P_e = exp(-eta_e S) sum_a w_ea ang_a, from which dT/dr_ij, dT/dr_ik,
// dT/dr_jk follow; dT/dcos uses sum_e exp(-eta_e S) sum_a w_ea dang_a.  These
// become gradients g_ij, g_ik w.r.t. R_ij and R_ik; -g goes into the LDS slot
// of each neighbour (LDS atomics) and g into the centre.  The neighbour slots
// become the per-edge buffer dE_i/dr_j; the centre part is -F_self
// (potentials/nnp/force.py:16-43).  The tangent (MODE_TAN) pushes a
// displacement field delta forward: T_is = sum_m dG_is/dr_m . delta_m.
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <type_traits>

#include "common.h"

namespace pt {
namespace {

enum { MODE_FWD = 0, MODE_ADJ = 1, MODE_TAN = 2 };

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ---- precision-specific math -------------------------------------------------
// ex2k(x): exponential of x scaled by kexp (FP32: v_exp_f32 = 2^x with the
// log2(e) factor folded into the caller's constants; FP64: libm exp).
template <typename R> struct M;
// FP64 elementary functions for the pair loops (the kernels' accuracy goal is
// ~1e-15 relative, far inside the 1e-10 parity bound):
//  * exp: Tang's table-driven method (ACM TOMS 15(2), 1989): x = (32 m + j)
//    ln2/32 + r with |r| <= ln2/64 (two-constant Cody-Waite reduction),
//    e^x = 2^m * 2^(j/32) * e^r, e^r by its degree-6 Taylor polynomial
//    (remainder < 4e-18); the 32 values 2^(j/32) live in LDS;
//  * 1/x and 1/sqrt(x): the hardware estimates refined by two Newton steps.
__constant__ double kExp2Tab[32] = {
    0x1.0000000000000p+0, 0x1.059b0d3158574p+0, 0x1.0b5586cf9890fp+0, 0x1.11301d0125b51p+0,
    0x1.172b83c7d517bp+0, 0x1.1d4873168b9aap+0, 0x1.2387a6e756238p+0, 0x1.29e9df51fdee1p+0,
    0x1.306fe0a31b715p+0, 0x1.371a7373aa9cbp+0, 0x1.3dea64c123422p+0, 0x1.44e086061892dp+0,
    0x1.4bfdad5362a27p+0, 0x1.5342b569d4f82p+0, 0x1.5ab07dd485429p+0, 0x1.6247eb03a5585p+0,
    0x1.6a09e667f3bcdp+0, 0x1.71f75e8ec5f74p+0, 0x1.7a11473eb0187p+0, 0x1.82589994cce13p+0,
    0x1.8ace5422aa0dbp+0, 0x1.93737b0cdc5e5p+0, 0x1.9c49182a3f090p+0, 0x1.a5503b23e255dp+0,
    0x1.ae89f995ad3adp+0, 0x1.b7f76f2fb5e47p+0, 0x1.c199bdd85529cp+0, 0x1.cb720dcef9069p+0,
    0x1.d5818dcfba487p+0, 0x1.dfc97337b9b5fp+0, 0x1.ea4afa2a490dap+0, 0x1.f50765b6e4540p+0,
};
__shared__ double g_exp2_tab[32];

// every thread of the block calls this before any early exit
__device__ __forceinline__ void exp2_tab_load() {
    if (threadIdx.x < 32) g_exp2_tab[threadIdx.x] = kExp2Tab[threadIdx.x];
    __syncthreads();
}

__device__ __forceinline__ double exp_tab(double x) {
    x = fmax(x, -708.0);
    const double nf = __builtin_rint(x * 0x1.71547652b82fep+5);          // 32 / ln2
    double r = fma(nf, -0x1.62e42fee00000p-6, x);                       // ln2/32, high part
    r = fma(nf, -0x1.a39ef35793c76p-38, r);                             // ln2/32, low part
    const int n = (int)nf;
    double p = fma(r, 1.0 / 720.0, 1.0 / 120.0);
    p = fma(p, r, 1.0 / 24.0);
    p = fma(p, r, 1.0 / 6.0);
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return __builtin_amdgcn_ldexp(g_exp2_tab[n & 31] * p, n >> 5);
}

__device__ __forceinline__ double rcp_nr(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y = fma(y, fma(-x, y, 1.0), y);
    y = fma(y, fma(-x, y, 1.0), y);
    return y;
}

__device__ __forceinline__ double rsq_nr(double x) {
    double y = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * x;
    y = y * fma(-h, y * y, 1.5);
    y = y * fma(-h, y * y, 1.5);
    return y;
}

template <> struct M<double> {
    static constexpr double kexp = 1.0;
    static __device__ __forceinline__ double ex2k(double x) { return exp_tab(x); }
    static __device__ __forceinline__ double ex(double x) { return exp_tab(x); }
    static __device__ __forceinline__ double th(double x) {
        // tanh(u) = (1 - e^{-2u}) / (1 + e^{-2u}); used for u in [-1, 1]
        const double e = exp_tab(-2.0 * x);
        return (1.0 - e) * rcp_nr(1.0 + e);
    }
    static __device__ __forceinline__ double co(double x) { return cos(x); }
    static __device__ __forceinline__ double si(double x) { return sin(x); }
    static __device__ __forceinline__ double sq(double x) { return sqrt(x); }
    static __device__ __forceinline__ double pw(double b, double z) { return pow(b, z); }
    static __device__ __forceinline__ double rcp(double x) { return rcp_nr(x); }
    // r and 1/r from r^2 > 0
    static __device__ __forceinline__ void root(double r2, double& r, double& ir) {
        ir = rsq_nr(r2);
        r = r2 * ir;
    }
};
template <> struct M<float> {
    static constexpr float kexp = 1.4426950408889634f;  // log2(e)
    static __device__ __forceinline__ float ex2k(float x) { return __builtin_amdgcn_exp2f(x); }
    static __device__ __forceinline__ float ex(float x) { return __builtin_amdgcn_exp2f(x * kexp); }
    static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
    static __device__ __forceinline__ float th(float x) {
        // tanh(u) = (1 - e^{-2u}) / (1 + e^{-2u}); used for u in [-1, 1]
        const float e = __builtin_amdgcn_exp2f(x * (-2.0f * kexp));
        return (1.0f - e) * rcp(1.0f + e);
    }
    static __device__ __forceinline__ float co(float x) { return __cosf(x); }
    static __device__ __forceinline__ float si(float x) { return __sinf(x); }
    static __device__ __forceinline__ float sq(float x) { return __builtin_amdgcn_sqrtf(x); }
    static __device__ __forceinline__ float pw(float b, float z) { return powf(b, z); }
    static __device__ __forceinline__ void root(float r2, float& r, float& ir) {
        ir = __builtin_amdgcn_rsqf(r2);
        r = r2 * ir;
    }
};

// Cutoff value and derivative (descriptors/acsf/cutoff.py:66-110).
template <typename R>
__device__ __forceinline__ void cutoff(int type, R rc, R inv_rc, R tanh_pre, R r, R& f, R& df) {
    if (!(r < rc)) { f = R(0); df = R(0); return; }
    switch (type) {
    case PT_CUT_HARD: f = R(1); df = R(0); return;
    case PT_CUT_TANHU:
    case PT_CUT_TANH: {
        const R t = M<R>::th(R(1) - r * inv_rc);
        const R pre = (type == PT_CUT_TANH) ? tanh_pre : R(1);
        const R t2 = t * t;
        f = pre * t2 * t;
        df = -pre * R(3) * t2 * (R(1) - t2) * inv_rc;
        return;
    }
    case PT_CUT_COS: {
        const R x = R(M_PI) * r * inv_rc;
        f = R(0.5) * (M<R>::co(x) + R(1));
        df = R(-0.5) * M<R>::si(x) * R(M_PI) * inv_rc;
        return;
    }
    case PT_CUT_EXP: {
        const R x = r * inv_rc, q = R(1) - x * x;
        const R iq = M<R>::rcp(q);
        f = M<R>::ex(R(1) - iq);
        df = f * (R(-2) * x * iq * iq) * inv_rc;
        return;
    }
    case PT_CUT_POLY1:
        f = (R(2) * r - R(3)) * r * r + R(1);
        df = R(6) * r * r - R(6) * r;
        return;
    case PT_CUT_POLY2:
        f = ((R(15) - R(6) * r) * r - R(10)) * r * r * r + R(1);
        df = ((R(-30) * r + R(60)) * r - R(30)) * r * r;
        return;
    }
    f = R(0); df = R(0);
}

// Cutoff specialised per group: CUTK_TANH (tanh / tanhu, cpre = prefactor),
// CUTK_COS, or the generic switch.  Branch-free for the first two.
enum { CUTK_TANH = 0, CUTK_COS = 1, CUTK_GEN = 2 };

template <typename R, int CUT>
__device__ __forceinline__ void cutoff_k(int type, R rc, R irc, R cpre, R tanh_pre, R r, R& f, R& df) {
    if (CUT == CUTK_TANH) {
        const R t = M<R>::th(R(1) - r * irc);
        const R t2 = t * t;
        const bool in = r < rc;
        f = in ? cpre * t2 * t : R(0);
        df = in ? R(-3) * cpre * t2 * (R(1) - t2) * irc : R(0);
    } else if (CUT == CUTK_COS) {
        const R x = R(M_PI) * r * irc;
        const bool in = r < rc;
        f = in ? R(0.5) * (M<R>::co(x) + R(1)) : R(0);
        df = in ? R(-0.5 * M_PI) * irc * M<R>::si(x) : R(0);
    } else {
        cutoff<R>(type, rc, irc, tanh_pre, r, f, df);
    }
}

// pre (1 + lam c)^zeta and its derivative w.r.t. c (angular.py:60-65).
template <typename R>
__device__ __forceinline__ void angular_term(R c, R lam, R zeta, int izeta, R pre, R& v, R& dv) {
    const R b = R(1) + lam * c;
    if (izeta >= 0) {
        // pm1 = b^(izeta - 1) by square-and-multiply over the bits of izeta - 1 (<= 15)
        const int z1 = izeta > 0 ? izeta - 1 : 0;
        R pm1 = R(1), q = b;
        if (z1 & 1) pm1 *= q;
        q *= q;
        if (z1 & 2) pm1 *= q;
        q *= q;
        if (z1 & 4) pm1 *= q;
        q *= q;
        if (z1 & 8) pm1 *= q;
        v = pre * (izeta > 0 ? pm1 * b : R(1));
        dv = (izeta == 0) ? R(0) : pre * R(izeta) * lam * pm1;
    } else {
        v = pre * M<R>::pw(b, zeta);
        dv = pre * zeta * lam * M<R>::pw(b, zeta - R(1));
    }
}

// Angular-term evaluation specialised per group: ANGK_Z1 (every zeta = 1),
// ANGK_Z1N2 (every zeta = 1, at most two terms), ANGK_P4 (every zeta in
// {1, 2, 4}), ANGK_Z14 (exactly the four terms zeta in {1, 4} x lambda in
// {+1, -1}, evaluated in that canonical order from the shared powers of
// 1 +- cos; the group's columns are mapped to it) or the generic
// square-and-multiply / pow.  The specialised forms leave the factor
// pre = 2^(1 - zeta) out of the pair loop: it scales the group's sums
// (forward) or dE/dG (adjoint) once per centre.
enum { ANGK_Z1 = 0, ANGK_P4 = 1, ANGK_GEN = 2, ANGK_Z1N2 = 3, ANGK_Z14 = 4 };

template <int ANG>
__host__ __device__ constexpr int ang_terms() { return ANG == ANGK_Z1N2 ? 2 : PT_AG_ANG; }

template <typename R> struct alignas(4 * sizeof(R)) V4 { R x, y, z, w; };
template <typename R> struct alignas(2 * sizeof(R)) V2 { R x, y; };

// Live-pair queue of one wavefront: (a | b << 16) indices of pairs that
// pass the r_jk screen; a batch of 64 is taken as soon as it is full, so it
// never holds more than 63 + 64 entries.
template <int MODE>
__host__ __device__ constexpr int queue_len() { return 128; }

template <typename R>
struct Stage {
    V4<R>* P;      // (x, y, z, 1/r) of R_ij = r_i - r_j
    V4<R>* Q;      // TAN: (r, r^2, fc, dfc/dr) -- cutoff of the current group
    V2<R>* Q2;     // FWD: (r, fc)
    V2<R>* QF;     // ADJ: (fc, dfc / r) of the current group
    R* D;          // [3][cap] TAN: delta_i - delta_j
    double* DA;    // [cap][3] ADJ: per-edge accumulators (FP64: fast LDS atomics; x, y, z
                   // adjacent so the three adds of an edge share one address)
    unsigned long long* keep;   // ADJ and teams: the staging ballots, one per 64 row entries
    unsigned* queue;
    R* W;          // ADJ, FP64: the group's dE/dG weights (read by broadcast)
};

// The adjoint keeps a compact record (x, y, z, 1/r) + per group (fc, dfc / r)
// and no per-neighbour row slot (r^2 is recomputed per pair from x, y, z,
// edge positions come back from the staging ballots): the LDS per wave then
// allows three waves per SIMD in FP64 and four and a half in FP32.

template <typename R, int MODE, int WPC>
__host__ __device__ constexpr size_t stage_bytes_per_nbr() {
    return MODE == MODE_ADJ ? sizeof(double) * 3 * WPC + sizeof(R) * 6
                            : sizeof(R) * (MODE == MODE_FWD ? 6 : 11);
}

// cap is a multiple of 4 and >= the row length; the per-wave area is a
// multiple of 32 bytes
// (WPC wavefronts share the stage: each has a queue and, in the adjoint,
// weights and accumulators of its own -- added in a fixed order at the end, so that the
// result does not depend on the wavefronts' timing -- and the staging ballots
// are kept in every mode)
template <typename R, int MODE, int WPC>
__host__ __device__ constexpr size_t stage_bytes(int cap) {
    return ((size_t)cap * stage_bytes_per_nbr<R, MODE, WPC>() + WPC * queue_len<MODE>() * sizeof(unsigned) +
            (MODE == MODE_ADJ ? WPC * PT_AG_ETA * PT_AG_ANG * sizeof(R) : 0) +
            (MODE == MODE_ADJ || WPC > 1 ? (size_t)((cap + kWave - 1) / kWave) * sizeof(unsigned long long) : 0) +
            31) / 32 * 32;
}

template <typename R, int MODE, int WPC>
__device__ __forceinline__ Stage<R> carve(char* base, int cap, int sub) {
    Stage<R> s;
    char* p = base;
    s.DA = nullptr;
    if (MODE == MODE_ADJ) { s.DA = reinterpret_cast<double*>(p) + 3 * cap * sub; p += 3 * cap * WPC * sizeof(double); }
    s.P = reinterpret_cast<V4<R>*>(p); p += cap * sizeof(V4<R>);
    s.Q = nullptr; s.Q2 = nullptr; s.QF = nullptr;
    if ((MODE == MODE_ADJ)) {
        s.QF = reinterpret_cast<V2<R>*>(p); p += cap * sizeof(V2<R>);
    } else if (MODE == MODE_FWD) {
        s.Q2 = reinterpret_cast<V2<R>*>(p); p += cap * sizeof(V2<R>);
    } else {
        s.Q = reinterpret_cast<V4<R>*>(p); p += cap * sizeof(V4<R>);
    }
    if (MODE == MODE_TAN) { s.D = reinterpret_cast<R*>(p); p += 3 * cap * sizeof(R); } else { s.D = nullptr; }
    s.queue = reinterpret_cast<unsigned*>(p) + sub * queue_len<MODE>();
    p += WPC * queue_len<MODE>() * sizeof(unsigned);
    s.W = nullptr;
    s.keep = nullptr;
    if (MODE == MODE_ADJ) {
        s.W = reinterpret_cast<R*>(p) + sub * PT_AG_ETA * PT_AG_ANG;
        p += WPC * PT_AG_ETA * PT_AG_ANG * sizeof(R);
    }
    if (MODE == MODE_ADJ || WPC > 1) s.keep = reinterpret_cast<unsigned long long*>(p);
    return s;
}

__device__ __forceinline__ void lds_add(double* p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <typename R>
__device__ __forceinline__ R mic_r(R d, R L, R half) {
    d = (d > half) ? d - L : d;
    d = (d < -half) ? d + L : d;
    return d;
}

template <typename R>
__device__ __forceinline__ void mic3(const BoxArg& b, R& x, R& y, R& z) {
    x = mic_r(x, (R)b.L[0], (R)b.half[0]);
    y = mic_r(y, (R)b.L[1], (R)b.half[1]);
    z = mic_r(z, (R)b.L[2], (R)b.half[2]);
}

// Staged neighbours with type < t for t = 0 .. kSegTypes (rows are type-sorted,
// so each element is one contiguous segment).  Types are 1-based.
constexpr int kSegTypes = 9;

// the counts live in lanes 0 .. kSegTypes of one VGPR (no private array)
__device__ __forceinline__ int seg_below(int segv, int t) {
    return __builtin_amdgcn_readlane(segv, t < 0 ? 0 : (t > kSegTypes ? kSegTypes : t));
}

// One run of a launch: centres that share a descriptor table.
struct KRun {
    const pt_sf_table* table;
    const int* centers;
    void* out;            // FWD: G, TAN: T (n x ld)
    const void* w;        // ADJ: dE/dG (n x ld)
    double* f_self;       // ADJ (n x 3)
    const double* delta;  // TAN (atoms x 3, internal order); nullptr: the unit vector of dir
    int n, begin;
    int item0;            // first work item of the run
    int dir;
};

constexpr int kMaxRuns = 8;

struct KArgs {
    const double* pos4;
    BoxArg box;
    const double* boxes;  // when set: the box lengths of several structures, box_id of each atom
    const int* box_id;
    const long long* row_off;
    const int* nbr;
    int ld;
    void* edge_grad;      // ADJ (n_pairs x 3)
    const int* rev;       // ADJ: when set, edge e's gradient goes to slot rev[e] (the reverse edge)
    int center_only;
    int cap;
    int n_items, n_runs;
    KRun run[kMaxRuns];
};

// A group of the table in registers: lane k holds the group's k-th 32-bit word
// and its k-th double.  One load each (the fields follow by v_readlane),
// where reading the fields one by one was a chain of ~35 dependent loads per
// angular group -- most of a wavefront's latency for a short row.
struct GroupWords {
    int w;
    double d;
};

template <typename G>
__device__ __forceinline__ GroupWords group_words(const G* g) {
    static_assert(sizeof(G) % 8 == 0 && sizeof(G) <= 4 * kWave, "a group fits one word per lane");
    const int lane = wave_lane();
    GroupWords r;
    r.w = lane < (int)(sizeof(G) / 4) ? reinterpret_cast<const int*>(g)[lane] : 0;
    r.d = lane < (int)(sizeof(G) / 8) ? reinterpret_cast<const double*>(g)[lane] : 0.0;
    return r;
}

__device__ __forceinline__ int lane_word(int v, int k) { return __builtin_amdgcn_readlane(v, k); }
__device__ __forceinline__ float lane_value(float v, int k) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
}
__device__ __forceinline__ double lane_value(double v, int k) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u & 0xffffffffu), k);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), k);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// word / double index of a field
#define PT_WORD(type, field) ((int)(offsetof(type, field) / 4))
#define PT_DBL(type, field) ((int)(offsetof(type, field) / 8))

// all wavefronts of a centre
template <int WPC>
__device__ __forceinline__ void centre_sync() {
    if constexpr (WPC == 1) wave_sync();
    else __syncthreads();
}

__device__ __forceinline__ double uniform_f64(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)uniform((int)(unsigned)(u & 0xffffffffu)), hi = (unsigned)uniform((int)(unsigned)(u >> 32));
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Uniform description of one angular group inside the kernel.
template <typename R>
struct AngGroup {
    int bj, nj, bk, nk;
    bool same, g3, mic;
    int n_eta, n_ang, cut;
    R rc, irc, cpre, tanh_pre;
    const BoxArg* box;
    R keta[PT_AG_ETA];     // -eta * kexp: exp(-eta S) = ex2k(keta S)
    R lam[PT_AG_ANG], zeta[PT_AG_ANG], pre[PT_AG_ANG], zl[PT_AG_ANG];   // zl = zeta * lambda
    int izeta[PT_AG_ANG];
};

template <typename R, int ANG, bool DER>
__device__ __forceinline__ void ang_eval(const AngGroup<R>& X, R cs, R (&v)[PT_AG_ANG], R (&dv)[PT_AG_ANG]) {
    // terms q >= n_ang carry pre = lam = zl = 0 and izeta = 1; in the
    // specialised forms v = (1 + lam c)^zeta and dv = zeta lam (1 + lam c)^(zeta - 1)
    // without pre, in the generic one both include pre
    constexpr int NA = ang_terms<ANG>();
    if constexpr (ANG == ANGK_Z14) {
        // (1 + c), (1 - c), (1 + c)^4, (1 - c)^4 and their derivatives in c
        const R bp = R(1) + cs, bm = R(1) - cs;
        const R bp2 = bp * bp, bm2 = bm * bm;
        v[0] = bp; v[1] = bm; v[2] = bp2 * bp2; v[3] = bm2 * bm2;
        dv[0] = DER ? R(1) : R(0);
        dv[1] = DER ? R(-1) : R(0);
        dv[2] = DER ? R(4) * bp * bp2 : R(0);
        dv[3] = DER ? R(-4) * bm * bm2 : R(0);
        return;
    }
#pragma unroll
    for (int q = 0; q < NA; ++q) {
        if (ANG == ANGK_Z1 || ANG == ANGK_Z1N2) {
            v[q] = R(1) + X.lam[q] * cs;
            dv[q] = DER ? X.zl[q] : R(0);
        } else if (ANG == ANGK_P4) {
            const R b = R(1) + X.lam[q] * cs;
            const R b2 = b * b;
            const int z = X.izeta[q];
            v[q] = z == 1 ? b : (z == 2 ? b2 : b2 * b2);
            dv[q] = DER ? X.zl[q] * (z == 1 ? R(1) : (z == 2 ? b : b * b2)) : R(0);
        } else {
            angular_term<R>(cs, X.lam[q], X.zeta[q], X.izeta[q], X.pre[q], v[q], dv[q]);
        }
    }
}

// All unordered pairs {j, k} of one angular group: screening on r_jk, a
// per-wave queue of live pairs, and the pair body in full-wave batches.
// The WPC wavefronts of a centre take the screening steps in turn (turn: this one's
// first).  have_cut: the stage holds the cutoff values already.  Returns the number of steps.
template <typename R, int MODE, int CUT, int ANG, int WPC>
__device__ __forceinline__ int angular_group(const Stage<R>& S, const AngGroup<R>& X,
                                             const R (&Win)[PT_AG_ETA][PT_AG_ANG],
                                             R (&acc)[PT_AG_ETA][PT_AG_ANG], int cap, int sub, int turn, bool have_cut) {
    const int lane = wave_lane();
    constexpr int NA = ang_terms<ANG>();
    constexpr bool kPreOut = ANG != ANGK_GEN;   // pre applied outside the pair loop
    // FP64 adjoint: the weights live in LDS (broadcast reads), which frees
    // 32 VGPRs in the pair loop.  So they do in FP32 where the angular terms take a
    // power each: their values fill the scalar registers, and 16 weights more were
    // spilled and read back lane by lane (12 Bohr, 12,288 centres 1,320 -> 1,260 us).
    constexpr bool kPowers = ANG == ANGK_GEN && CUT != CUTK_GEN && WPC == 1;
    constexpr bool kWLds = MODE == MODE_ADJ && (sizeof(R) == 8 || kPowers);
    R W[PT_AG_ETA][PT_AG_ANG];
#pragma unroll
    for (int e = 0; e < PT_AG_ETA; ++e)
#pragma unroll
        for (int q = 0; q < PT_AG_ANG; ++q) W[e][q] = kPreOut ? Win[e][q] * X.pre[q] : Win[e][q];
    // Adjoint of the zeta {1, 4} x lambda +-1 class: the weighted angular sum
    // of one eta, U(c) = w0 (1 + c) + w1 (1 - c) + w2 (1 + c)^4 + w3 (1 - c)^4,
    // is a quartic in c.  With sp = w2 + w3, sm = w2 - w3, W[e] becomes
    // (u0, u1, sp, sm4) = (w0 + w1 + sp, w0 - w1 + 4 sm, sp, 4 sm) and
    //   U = u0 + u1 c + sp c^2 (6 + c^2) + sm4 c^3,
    //   U' = u1 + sp (12 c + 4 c^3) + 3 sm4 c^2,
    // so the pair body needs no angular terms, and the powers of c are
    // shared by the eta values.
    constexpr bool kQuartic = MODE == MODE_ADJ && ANG == ANGK_Z14;
    if (kQuartic) {
#pragma unroll
        for (int e = 0; e < PT_AG_ETA; ++e) {
            const R w0 = W[e][0], w1 = W[e][1], sp = W[e][2] + W[e][3], sm = W[e][2] - W[e][3];
            W[e][0] = (w0 + w1) + sp;
            W[e][1] = (w0 - w1) + R(4) * sm;
            W[e][2] = sp;
            W[e][3] = R(4) * sm;
        }
    }
    if (kWLds) {
        if (lane == 0) {
#pragma unroll
            for (int e = 0; e < PT_AG_ETA; ++e)
#pragma unroll
                for (int q = 0; q < PT_AG_ANG; ++q) S.W[e * PT_AG_ANG + q] = W[e][q];
        }
    }
    // cutoff values of the group's neighbours
    if (have_cut) {
        wave_sync();
    } else {
        for (int pass = 0; pass < (X.same ? 1 : 2); ++pass) {
            const int sb = pass == 0 ? X.bj : X.bk, sn = pass == 0 ? X.nj : X.nk;
            for (int s = sb + lane + sub * kWave; s < sb + sn; s += WPC * kWave) {
                R f, df;
                if constexpr ((MODE == MODE_ADJ)) {
                    const R ir = S.P[s].w;
                    cutoff_k<R, CUT>(X.cut, X.rc, X.irc, X.cpre, X.tanh_pre, M<R>::rcp(ir), f, df);
                    V2<R> fv;
                    fv.x = f; fv.y = df * ir;   // dfc / r
                    S.QF[s] = fv;
                } else if constexpr (MODE == MODE_FWD) {
                    cutoff_k<R, CUT>(X.cut, X.rc, X.irc, X.cpre, X.tanh_pre, S.Q2[s].x, f, df);
                    S.Q2[s].y = f;
                } else {
                    cutoff_k<R, CUT>(X.cut, X.rc, X.irc, X.cpre, X.tanh_pre, S.Q[s].x, f, df);
                    S.Q[s].z = f;
                    S.Q[s].w = df;
                }
            }
        }
        centre_sync<WPC>();
    }

    // one live pair (ia, ib)
    auto body = [&](const int ia, const int ib) {
        const V4<R> pa = S.P[ia], pb = S.P[ib];
        V4<R> qa, qb;   // (r, r^2, fc, dfc); ADJ: (unused, r^2, fc, dfc / r)
        R ira, irb;     // 1 / r
        if constexpr ((MODE == MODE_ADJ)) {
            const V2<R> ua = S.QF[ia], ub = S.QF[ib];
            ira = pa.w;
            irb = pb.w;
            qa.y = pa.x * pa.x + pa.y * pa.y + pa.z * pa.z;
            qb.y = pb.x * pb.x + pb.y * pb.y + pb.z * pb.z;
            qa.x = R(0); qa.z = ua.x; qa.w = ua.y;
            qb.x = R(0); qb.z = ub.x; qb.w = ub.y;
        } else if constexpr (MODE == MODE_FWD) {
            const V2<R> ua = S.Q2[ia], ub = S.Q2[ib];
            qa.x = ua.x; qa.y = ua.x * ua.x; qa.z = ua.y; qa.w = R(0);
            qb.x = ub.x; qb.y = ub.x * ub.x; qb.z = ub.y; qb.w = R(0);
        } else {
            qa = S.Q[ia];
            qb = S.Q[ib];
        }
        if constexpr ((MODE != MODE_ADJ)) {
            ira = pa.w;
            irb = pb.w;
        }
        R jx = pa.x - pb.x, jy = pa.y - pb.y, jz = pa.z - pb.z;
        if (X.mic) mic3(*X.box, jx, jy, jz);
        const R rjk2 = jx * jx + jy * jy + jz * jz;   // > 0 (screened)
        R rjk, irjk;
        M<R>::root(rjk2, rjk, irjk);
        R fjk = R(1), dfjk = R(0);
        if (X.g3) cutoff_k<R, CUT>(X.cut, X.rc, X.irc, X.cpre, X.tanh_pre, rjk, fjk, dfjk);
        const R Ssum = X.g3 ? qa.y + qb.y + rjk2 : qa.y + qb.y;
        const R F = qa.z * qb.z * fjk;
        const R iab = ira * irb;
        const R cs = (pa.x * pb.x + pa.y * pb.y + pa.z * pb.z) * iab;
        R ang[PT_AG_ANG], dang[PT_AG_ANG];
        if constexpr (!kQuartic) ang_eval<R, ANG, MODE != MODE_FWD>(X, cs, ang, dang);
        if (MODE == MODE_FWD) {
#pragma unroll
            for (int e = 0; e < PT_AG_ETA; ++e) {
                if (e < X.n_eta) {
                    const R rad = M<R>::ex2k(X.keta[e] * Ssum) * F;
#pragma unroll
                    for (int q = 0; q < NA; ++q) acc[e][q] += rad * ang[q];
                }
            }
            return;
        }
        // derivative building blocks
        const R ra = qa.x, rb = qb.x;
        const R ira2 = ira * ira, irb2 = irb * irb;
        if (!X.g3) irjk = R(0);
        // d F / d r_ij etc. (without the exp factor)
        const R Fa = qa.w * qb.z * fjk, Fb = qa.z * qb.w * fjk, Fj = qa.z * qb.z * dfjk;
        if (MODE == MODE_ADJ) {
            R SP = R(0), SKP = R(0), SV = R(0);
            R c3 = R(0), t4 = R(0), dt4 = R(0), c2x3 = R(0);
            if constexpr (kQuartic) {
                const R c2 = cs * cs;
                c3 = c2 * cs;
                t4 = c2 * (R(6) + c2);
                dt4 = R(12) * cs + R(4) * c3;
                c2x3 = R(3) * c2;
            }
#pragma unroll
            for (int e = 0; e < PT_AG_ETA; ++e) {
                if (e < X.n_eta) {
                    const R ex = M<R>::ex2k(X.keta[e] * Ssum);
                    R U = R(0), V = R(0);
                    if constexpr (kQuartic) {
                        const R u0 = kWLds ? S.W[e * PT_AG_ANG + 0] : W[e][0];
                        const R u1 = kWLds ? S.W[e * PT_AG_ANG + 1] : W[e][1];
                        const R sp = kWLds ? S.W[e * PT_AG_ANG + 2] : W[e][2];
                        const R sm4 = kWLds ? S.W[e * PT_AG_ANG + 3] : W[e][3];
                        U = u0 + u1 * cs + sp * t4 + sm4 * c3;
                        V = u1 + sp * dt4 + sm4 * c2x3;
                    } else {
#pragma unroll
                        for (int q = 0; q < NA; ++q) {
                            const R wq = kWLds ? S.W[e * PT_AG_ANG + q] : W[e][q];
                            U += wq * ang[q];
                            V += wq * dang[q];
                        }
                    }
                    const R P = ex * U;
                    SP += P;
                    SKP += X.keta[e] * P;
                    SV += ex * V;
                }
            }
            // dT/dr = d/dr [exp(-eta S) F]: F' sum_e P_e - 2 r F sum_e eta_e P_e,
            // sum_e eta_e P_e = -SKP / kexp.  With Fa, Fb built from dfc / r,
            // d T / d r_ij / r_ij = Fa SP + F2 SKP (and the same for r_ik).
            const R F2S = F * R(2.0 / M<R>::kexp) * SKP;
            const R d_rjk = X.g3 ? (Fj * SP + rjk * F2S) : R(0);
            const R d_c = F * SV;
            // d cos / d R_ij = R_ik/(r_ij r_ik) - cos R_ij / r_ij^2 (and a <-> b), folded:
            // g_a = (d_rij / r_ij - d_c cos / r_ij^2) R_ij + (d_c / (r_ij r_ik)) R_ik + s_j R_jk
            const R sj = d_rjk * irjk;
            const R dcc = d_c * cs;
            const R al = Fa * SP + F2S - dcc * ira2;
            const R bl = Fb * SP + F2S - dcc * irb2;
            const R be = d_c * iab;
            const R gax = al * pa.x + be * pb.x + sj * jx;
            const R gay = al * pa.y + be * pb.y + sj * jy;
            const R gaz = al * pa.z + be * pb.z + sj * jz;
            const R gbx = bl * pb.x + be * pa.x - sj * jx;
            const R gby = bl * pb.y + be * pa.y - sj * jy;
            const R gbz = bl * pb.z + be * pa.z - sj * jz;
            lds_add(&S.DA[3 * ia], -(double)gax); lds_add(&S.DA[3 * ia + 1], -(double)gay);
            lds_add(&S.DA[3 * ia + 2], -(double)gaz);
            lds_add(&S.DA[3 * ib], -(double)gbx); lds_add(&S.DA[3 * ib + 1], -(double)gby);
            lds_add(&S.DA[3 * ib + 2], -(double)gbz);
        } else {  // MODE_TAN
            const R cax = pb.x * iab - cs * pa.x * ira2, cay = pb.y * iab - cs * pa.y * ira2,
                    caz = pb.z * iab - cs * pa.z * ira2;  // d cos / d R_ij
            const R cbx = pa.x * iab - cs * pb.x * irb2, cby = pa.y * iab - cs * pb.y * irb2,
                    cbz = pa.z * iab - cs * pb.z * irb2;  // d cos / d R_ik
            const R ax = S.D[ia], ay = S.D[cap + ia], az = S.D[2 * cap + ia];
            const R bx = S.D[ib], by = S.D[cap + ib], bz = S.D[2 * cap + ib];
            const R tij = (pa.x * ax + pa.y * ay + pa.z * az) * ira;
            const R tik = (pb.x * bx + pb.y * by + pb.z * bz) * irb;
            const R tjk = X.g3 ? (jx * (ax - bx) + jy * (ay - by) + jz * (az - bz)) * irjk : R(0);
            const R cdot = cax * ax + cay * ay + caz * az + cbx * bx + cby * by + cbz * bz;
            // d/dt [exp(-eta S) F] = exp(-eta S) (X0 - 2 eta X1)
            const R X0 = Fa * tij + Fb * tik + Fj * tjk;
            const R X1 = F * (ra * tij + rb * tik + rjk * tjk);
#pragma unroll
            for (int e = 0; e < PT_AG_ETA; ++e) {
                if (e < X.n_eta) {
                    const R ex = M<R>::ex2k(X.keta[e] * Ssum);
                    const R rdot = ex * (X0 + R(2.0 / M<R>::kexp) * X.keta[e] * X1);
                    const R radc = ex * F * cdot;
#pragma unroll
                    for (int q = 0; q < NA; ++q) acc[e][q] += rdot * ang[q] + radc * dang[q];
                }
            }
        }
    };

    // Pair enumeration, ordered so that the 64 lanes of one step touch
    // distinct neighbour slots (few LDS atomic conflicts in the adjoint):
    //  - cross segments: lanes run over the shorter segment q, the other
    //    index is the diagonal k = (q + d) mod n_long, d = 0 .. n_long-1;
    //  - one segment: k = (q + 1 + d) mod n for d < n/2 -- each unordered
    //    pair once (see below for the last diagonal of an even n).
    // Pair p = d * nrow + q; each lane advances p by 64 WPC per step.
    const bool jrow = X.nj <= X.nk;
    const int nrow = X.same ? X.nj : (jrow ? X.nj : X.nk);
    const int ncol = X.same ? X.nj : (jrow ? X.nk : X.nj);
    const int brow = X.same ? X.bj : (jrow ? X.bj : X.bk);
    const int bcol = X.same ? X.bj : (jrow ? X.bk : X.bj);
    // one segment: h = n/2 diagonals d (k = q + 1 + d mod n); for even n the
    // last diagonal pairs q with q + n/2 and holds each pair twice, so only
    // q < n/2 is taken there
    const int h = X.same ? X.nj / 2 : ncol;
    const int npairs = nrow * h;
    if (npairs <= 0) return 0;   // (the same for every wavefront of the centre)
    const int half_d = (X.same && X.nj % 2 == 0) ? h - 1 : -1;   // the doubled diagonal
    const int half_q = X.nj / 2;
    constexpr int kStep = kWave * WPC;
    const int d64 = uniform(kStep / nrow), r64 = uniform(kStep - d64 * nrow);
    const int p0 = WPC == 1 ? lane : lane + turn * kWave;
    int d = p0 / nrow, q = p0 - (p0 / nrow) * nrow;
    // screen r_jk^2 < rc^2 (loosened by 1e-4 relative); the exact r_jk < rc
    // test is the cutoff's own (it is 0 beyond rc)
    const R rc2 = X.g3 ? X.rc * X.rc * R(1.0001) : R(INFINITY);
    const int sk = X.same ? 1 : 0;
    int qn = 0, base = WPC == 1 ? 0 : turn * kWave;
    // one batch of up to 64 queued pairs through the body; the rest moves up
    auto drain = [&]() {
        wave_sync();
        const int take = qn < kWave ? qn : kWave;
        const unsigned e = lane < take ? S.queue[lane] : 0u;
        const int rem = qn - take;
        const unsigned mv0 = lane < rem ? S.queue[kWave + lane] : 0u;
        const unsigned mv1 = lane + kWave < rem ? S.queue[2 * kWave + lane] : 0u;
        wave_sync();
        if (lane < rem) S.queue[lane] = mv0;
        if (lane + kWave < rem) S.queue[kWave + lane] = mv1;
        qn = rem;
        if (lane < take) body((int)(e & 0xffffu), (int)(e >> 16));
    };
    // kDiag diagonals per lane and step: lane (D, q) screens d = kDiag D + u,
    // u = 0 .. kDiag - 1, which share the row slot and the index arithmetic;
    // the queue is drained whenever it holds a full batch, so it never holds
    // more than 63 + 64 entries.  (Measured on gfx950: 4 beats 2 and 8 in
    // FP32, and 2 in the FP64 adjoint by 2.5 %.)
    constexpr int kDiag = 4;
    const int hh = (h + kDiag - 1) / kDiag;
    const int npairs2 = nrow * hh;
    while (true) {
        if (base < npairs2) {
            const int ia = brow + q;
            const int d0 = kDiag * d;
            // the lane's diagonals d0 + u exist for u < nu; the doubled diagonal
            // of an even segment (the last one, half_d = h - 1) only for q < n/2
            int nu = min(max(h - d0, 0), kDiag);
            if (q >= half_q && half_d >= d0 && half_d < d0 + kDiag) nu = half_d - d0;
            if (base + lane >= npairs2) nu = 0;
            // column k = (q + sk + d0 + u) mod ncol: q + sk + d0 + u < 2 ncol for
            // every existing diagonal, so k0 + u wraps at most once; a lane with
            // no diagonal reads from the segment start (loads stay in the stage)
            int k0 = q + sk + d0;
            k0 = k0 >= ncol ? k0 - ncol : k0;
            k0 = nu > 0 ? k0 : 0;
            const V4<R>* pseg = S.P + bcol;
            const unsigned eb = (unsigned)ia | ((unsigned)bcol << 16);
#pragma unroll
            for (int u = 0; u < kDiag; ++u) {
                // (k0 + u) mod ncol as an unsigned minimum: k0 + u - ncol is
                // negative (huge) unless the column wraps; at most 2 past the
                // segment start for a lane beyond nu
                const unsigned kk = min((unsigned)(k0 + u), (unsigned)(k0 + u - ncol));
                const V4<R> pa = S.P[ia], pb = pseg[kk];
                R jx = pa.x - pb.x, jy = pa.y - pb.y, jz = pa.z - pb.z;
                if (X.mic) mic3(*X.box, jx, jy, jz);
                const R r2 = jx * jx + jy * jy + jz * jz;
                const bool live = (u < nu) & (r2 > R(0)) & (r2 < rc2);
                // (a ballot per compare: no lane mask rebuilt from the bool)
                const unsigned long long b = __builtin_amdgcn_ballot_w64(u < nu) &
                                             __builtin_amdgcn_ballot_w64(r2 > R(0)) &
                                             __builtin_amdgcn_ballot_w64(r2 < rc2);
                if (live) S.queue[qn + lanes_below(b)] = eb + (kk << 16);
                qn += __popcll(b);
                if (qn >= kWave) drain();
            }
            base += kStep;
            q += r64;
            d += d64;
            if (q >= nrow) { q -= nrow; ++d; }
        }
        const bool last = base >= npairs2;
        while (qn >= kWave || (last && qn > 0)) drain();
        if (last && qn == 0) break;
    }
    if (kPreOut && MODE != MODE_ADJ) {
#pragma unroll
        for (int e = 0; e < PT_AG_ETA; ++e)
#pragma unroll
            for (int q = 0; q < PT_AG_ANG; ++q) acc[e][q] *= X.pre[q];
    }
    wave_sync();
    return (npairs2 + kWave - 1) / kWave;
}

// 1 when the group's terms are exactly zeta {1, 4} x lambda {+1, -1} (any
// order); qmap[k] then gives the term of canonical slot k = 2 [zeta = 4] +
// [lambda = -1].
__device__ __forceinline__ int z14_order(const GroupWords& G, int n_ang, int (&qmap)[PT_AG_ANG]) {
    int seen = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) qmap[q] = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int iz = lane_word(G.w, PT_WORD(pt_angular_group, izeta) + q);
        const double lam = lane_value(G.d, PT_DBL(pt_angular_group, lam) + q);
        const bool ok = (iz == 1 || iz == 4) && (lam == 1.0 || lam == -1.0);
        const int k = ok ? (iz == 4 ? 2 : 0) + (lam < 0.0 ? 1 : 0) : 4;
        seen |= 1 << k;
#pragma unroll
        for (int t = 0; t < 4; ++t) qmap[t] = uniform(t == k ? q : qmap[t]);
    }
    return n_ang == 4 && uniform(seen) == 15 ? 1 : 0;
}

// Shared between the wavefronts of a centre (beyond the stage).
template <typename R, int WPC>
struct Team {
    static constexpr int kPending = 4;                   // groups whose parts wait for the other wavefronts'
    static_assert(WPC >= kPending, "a wavefront per pending group adds its parts");
    R part[WPC][kPending][PT_AG_ETA * PT_AG_ANG];        // groups' sums of each wavefront
    int seg[WPC][16];                               // segment counts of each wavefront's row chunks
};
template <typename R>
struct Team<R, 1> {
    static constexpr int kPending = 1;
};

// Sums of a group's first N cells over the wavefront.  One wavefront per centre: into their
// columns.  A team: into its part of pending group `slot`, whose lane's column
// (or -1) and cell wavefront `slot` keeps.
// gw: the group's words (GroupWords).
template <int N, typename R, int WPC>
__device__ __forceinline__ void store_cells(const R (&acc)[PT_AG_ETA][PT_AG_ANG], const int (&qmap)[PT_AG_ANG], int gw,
                                            int n_eta, int n_ang, Team<R, WPC>& T, int sub, int slot, int& pending_col, int& pending_cell,
                                            R* row) {
    R flat[N];
#pragma unroll
    for (int k = 0; k < N; ++k) flat[k] = acc[k / PT_AG_ANG][k % PT_AG_ANG];
    const R v = wave_sums<N>(flat);
    const int cell = sum_of_lane<N>(), q = cell & (PT_AG_ANG - 1);
    // (the map packed: indexed by lane the array would live in scratch)
    const unsigned packed = (unsigned)(qmap[0] | qmap[1] << 8 | qmap[2] << 16 | qmap[3] << 24);
    const int tq = (int)((packed >> (8 * q)) & 3u);
    const int k = __shfl(gw, PT_WORD(pt_angular_group, col) + max(cell - q, 0) + tq, kWave);
    const bool own = cell >= 0 && cell / PT_AG_ANG < n_eta && q < n_ang && k >= 0;
    if constexpr (WPC > 1) {
        if (own) T.part[sub][slot][cell] = v;
        if (sub == slot) { pending_col = own ? k : -1; pending_cell = cell; }
    } else if (own) {
        row[k] = v;
    }
}

template <typename R, int MODE, int KIND, int WPC>
__device__ __forceinline__ void acsf_centre(const KArgs& a, char* smem, Team<R, WPC>& T) {
    if (sizeof(R) == 8) exp2_tab_load();
    const int lane = wave_lane();
    const int wv = uniform(threadIdx.x >> 6);
    const int wpb = blockDim.x >> 6;
    const int sub = WPC == 1 ? 0 : wv;                                    // wavefront of this centre
    const int item = uniform(WPC == 1 ? xcd_block() * wpb + wv : xcd_block());
    if (item >= a.n_items) return;
    int ri = 0;
    while (ri + 1 < a.n_runs && item >= a.run[ri + 1].item0) ++ri;
    const KRun& rn = a.run[ri];
    const int c = item - rn.item0;
    const int cap = a.cap;
    Stage<R> S = carve<R, MODE, WPC>(WPC == 1 ? smem + (size_t)wv * stage_bytes<R, MODE, WPC>(cap) : smem, cap, sub);
    const pt_sf_table* __restrict__ tab = rn.table;
    const int i = uniform(rn.centers ? rn.centers[c] : rn.begin + c);
    const double4 pi = reinterpret_cast<const double4*>(a.pos4)[i];
    const long long off = a.row_off[i];
    const int len = (int)(a.row_off[i + 1] - off);
    if (len > cap) {
        // the row does not fit the staging slice sized by the caller's max_row:
        // stage nothing and report the centre as NaN (outputs, f_self, the row's edges)
        const R nan = __builtin_nan("");
        const int t0 = lane + sub * kWave;
        if (MODE != MODE_ADJ) {
            R* out = (R*)rn.out;
            for (int q = t0; q < a.ld; q += WPC * kWave) out[(size_t)c * a.ld + q] = nan;
        } else {
            if (a.edge_grad) {
                R* eg = (R*)a.edge_grad;
                for (int t = t0; t < len; t += WPC * kWave) {
                    const long long e = a.rev ? (long long)a.rev[off + t] : off + t;
                    if (e >= 0) { eg[3 * e] = nan; eg[3 * e + 1] = nan; eg[3 * e + 2] = nan; }
                }
            }
            if (rn.f_self && t0 < 3) rn.f_self[3 * c + t0] = (double)nan;
        }
        return;
    }
    BoxArg box = a.box;
    if (a.boxes) {
        const double* bl = a.boxes + 3 * (size_t)a.box_id[i];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            box.L[d] = uniform_f64(bl[d]);
            box.half[d] = 0.5 * box.L[d];
        }
        box.periodic = uniform((box.L[0] > 0.0) ? 1 : 0);
    }
    const double rcmax = tab->rc_max;
    const R tanh_pre = (R)tab->tanh_pre;
    // |R_ij - R_ik| <= 2 rc_max: the image shift can only act when L/2 < 2 rc_max
    const double lim = 4.0 * rcmax * (1.0 + 1e-9);
    const bool mic_jk = box.periodic && (!(box.L[0] > lim) || !(box.L[1] > lim) || !(box.L[2] > lim));

    double dix = 0, diy = 0, diz = 0;
    if (MODE == MODE_TAN) {
        if (rn.delta) {
            dix = rn.delta[3 * i]; diy = rn.delta[3 * i + 1]; diz = rn.delta[3 * i + 2];
        } else {
            dix = rn.dir == 0; diy = rn.dir == 1; diz = rn.dir == 2;
        }
    }

    // segment counts are needed up to one past the largest type the table uses
    static_assert(PT_MAX_GROUPS <= kWave, "a lane per group");
    const int n_rg = uniform(tab->n_rg), n_ag = uniform(tab->n_ag);
    int tg = lane < n_rg ? tab->rg[lane].elem : 0;
    if (lane < n_ag) tg = max(tg, max(tab->ag[lane].ej, tab->ag[lane].ek));
    // Tables whose angular groups share one tanh cutoff (and whose radial groups do too:
    // cut_r): its values are computed as the row is staged, once per neighbour, where
    // every group computed them for its own segments (two elements: five times)
    bool cut_a = false, cut_r = false;
    R rc0 = R(0), irc0 = R(0), cpre0 = R(1);
    int cut0 = 0;
    if constexpr (KIND != PT_ACSF_GENERIC) {
        const int ca = lane < n_ag ? tab->ag[lane].cut : -1, cr = lane < n_rg ? tab->rg[lane].cut : -1;
        const double ra = lane < n_ag ? tab->ag[lane].rc : 0.0, rr = lane < n_rg ? tab->rg[lane].rc : 0.0;
        cut0 = lane_word(ca, 0);
        const double r0 = lane_value(ra, 0);
        cut_a = (cut0 == PT_CUT_TANH || cut0 == PT_CUT_TANHU) && __ballot(lane < n_ag && (ca != cut0 || ra != r0)) == 0ull;
        cut_r = cut_a && __ballot(lane < n_rg && (cr != cut0 || rr != r0)) == 0ull;
        rc0 = (R)r0;
        irc0 = (R)(1.0 / r0);
        cpre0 = cut0 == PT_CUT_TANH ? tanh_pre : R(1);
    }
    // a team's next angular group, loaded while the one before is worked on
    GroupWords Gn{0, 0.0};
    if (WPC > 1 && n_ag > 0) Gn = group_words(&tab->ag[0]);
    // and the adjoint's weights by column
    R wrow = R(0);
    if (MODE == MODE_ADJ && WPC > 1 && lane < a.ld) wrow = ((const R*)rn.w)[(size_t)c * a.ld + lane];
    int tmax = 0;
    while (tmax < kSegTypes && __ballot(tg > tmax) != 0ull) ++tmax;
    const int nseg = min(tmax + 1, kSegTypes);

    // ---- stage the row ----------------------------------------------------
    // one entry of a 64-entry chunk per lane
    struct Entry {
        double dx, dy, dz, r, tj;
        int j;
        bool in, keep;
    };
    auto load = [&](int t0) {
        Entry e{0, 0, 0, 0, 0, 0, t0 + lane < len, false};
        if (e.in) {
            e.j = a.nbr[off + t0 + lane];
            const double4 pj = reinterpret_cast<const double4*>(a.pos4)[e.j];
            e.dx = pi.x - pj.x; e.dy = pi.y - pj.y; e.dz = pi.z - pj.z;
            e.r = exact_dist(e.dx, e.dy, e.dz, box);
            e.tj = pj.w;
            e.keep = (e.r <= rcmax) && (e.r > 0.0);
        }
        return e;
    };
    int seg = 0;   // lane q: staged neighbours with type < q
    // kept entries go to the slots m, m + 1, ...
    auto store = [&](const Entry& e, int t0, unsigned long long bal, int m) {
        if (e.keep) {
            const int s = m + lanes_below(bal);
            V4<R> pv, qv;
            pv.x = (R)e.dx; pv.y = (R)e.dy; pv.z = (R)e.dz;
            pv.w = (R)(1.0 / e.r);
            qv.x = (R)e.r; qv.y = (R)e.r * (R)e.r; qv.z = R(0); qv.w = R(0);
            S.P[s] = pv;
            R f = R(0), df = R(0);
            if (cut_a) cutoff_k<R, CUTK_TANH>(cut0, rc0, irc0, cpre0, tanh_pre, qv.x, f, df);
            if constexpr ((MODE == MODE_ADJ)) {
                if (cut_a) {   // (else written per group)
                    V2<R> fv;
                    fv.x = f; fv.y = df * pv.w;
                    S.QF[s] = fv;
                }
            } else if constexpr (MODE == MODE_FWD) {
                V2<R> uv;
                uv.x = qv.x; uv.y = f;
                S.Q2[s] = uv;
            } else {
                qv.z = f; qv.w = df;
                S.Q[s] = qv;
            }
            if (MODE == MODE_ADJ && WPC == 1) { S.DA[3 * s] = 0.0; S.DA[3 * s + 1] = 0.0; S.DA[3 * s + 2] = 0.0; }
            if (MODE == MODE_TAN) {
                double ex = dix, ey = diy, ez = diz;
                if (!a.center_only) {
                    ex -= rn.delta[3 * e.j]; ey -= rn.delta[3 * e.j + 1]; ez -= rn.delta[3 * e.j + 2];
                }
                S.D[s] = (R)ex; S.D[cap + s] = (R)ey; S.D[2 * cap + s] = (R)ez;
            }
        } else if (MODE == MODE_ADJ && e.in && a.edge_grad) {
            // (a reverse index of -1 would mean an asymmetric list: no slot to write)
            const long long k = a.rev ? (long long)a.rev[off + t0 + lane] : off + t0 + lane;
            if (k >= 0) {
                R* eg = (R*)a.edge_grad + 3 * k;
                eg[0] = R(0); eg[1] = R(0); eg[2] = R(0);
            }
        }
        const int tk = (int)e.tj;
        for (int q = 1; q <= nseg; ++q) {
            const int cq = __popcll(__ballot(e.keep && tk < q));
            seg += lane == q ? cq : 0;
        }
    };
    int m = 0;
    if constexpr (WPC == 1) {
        for (int t0 = 0; t0 < len; t0 += kWave) {
            const Entry e = load(t0);
            const unsigned long long bal = __ballot(e.keep);
            if (MODE == MODE_ADJ && lane == 0) S.keep[t0 / kWave] = bal;
            store(e, t0, bal, m);
            m += __popcll(bal);
        }
        m = uniform(m);
        wave_sync();
    } else {
        // chunks in turn; the ballots of all chunks first (a chunk's slots start after
        // those of the chunks before it), the first chunk of a wavefront stays in registers
        const Entry e0 = load(sub * kWave);
        for (int t0 = sub * kWave; t0 < len; t0 += WPC * kWave) {
            const unsigned long long bal = __ballot(t0 == sub * kWave ? e0.keep : load(t0).keep);
            if (lane == 0) S.keep[t0 / kWave] = bal;
        }
        __syncthreads();
        for (int t0 = 0; t0 < len; t0 += kWave) {
            const unsigned long long bal = S.keep[t0 / kWave];
            if (t0 / kWave % WPC == sub) store(t0 == sub * kWave ? e0 : load(t0), t0, bal, m);
            m += __popcll(bal);
        }
        m = uniform(m);
        if (MODE == MODE_ADJ)
            for (int s = lane; s < 3 * m; s += kWave) S.DA[s] = 0.0;
        if (lane < 16) T.seg[sub][lane] = seg;
        __syncthreads();
        seg = 0;
        if (lane < 16) {
#pragma unroll
            for (int k = 0; k < WPC; ++k) seg += T.seg[k][lane];
        }
    }

    R* out = (R*)rn.out;
    const R* w = (const R*)rn.w;

    // ---- radial groups -----------------------------------------------------
    // (a team takes halves of groups in turn: no sums across wavefronts)
    constexpr int kHalves = WPC > 1 ? 2 : 1, kFun = PT_RG_MAX / kHalves;
    for (int g2 = sub; g2 < n_rg * kHalves; g2 += WPC) {
        const int g = g2 / kHalves, f0 = g2 % kHalves * kFun;
        constexpr int kCol = PT_WORD(pt_radial_group, col), kEta = PT_DBL(pt_radial_group, eta),
                      kRs = PT_DBL(pt_radial_group, rs), kRc = PT_DBL(pt_radial_group, rc);
        const GroupWords G = group_words(&tab->rg[g]);
        const int el = lane_word(G.w, PT_WORD(pt_radial_group, elem));
        const int cut = lane_word(G.w, PT_WORD(pt_radial_group, cut));
        const int nfun = lane_word(G.w, PT_WORD(pt_radial_group, n)) - f0;   // from f0 on
        if (nfun <= 0) continue;
        const int b = seg_below(seg, el), e = seg_below(seg, el + 1);
        const R gr = (R)G.d;
        const R rc = lane_value(gr, kRc), irc = lane_value((R)(1.0 / G.d), kRc);
        const bool mine = lane >= kCol + f0 && lane < kCol + f0 + nfun;   // lane kCol + q: function q's column
        R wl = R(0);
        if (MODE == MODE_ADJ && mine) wl = w[(size_t)c * a.ld + G.w];   // its dE/dG
        R wgt[kFun], acc[kFun], keta[kFun], eta[kFun], rs[kFun];
#pragma unroll
        for (int q = 0; q < kFun; ++q) {
            acc[q] = R(0);
            eta[q] = (q < nfun) ? lane_value(gr, kEta + f0 + q) : R(0);
            keta[q] = -eta[q] * M<R>::kexp;
            rs[q] = (q < nfun) ? lane_value(gr, kRs + f0 + q) : R(0);
            wgt[q] = MODE == MODE_ADJ ? lane_value(wl, kCol + f0 + q) : R(0);
        }
        for (int s = b + lane; s < e; s += kWave) {
            R r;
            if constexpr ((MODE == MODE_ADJ)) r = M<R>::rcp(S.P[s].w);
            else if constexpr (MODE == MODE_FWD) r = S.Q2[s].x;
            else r = S.Q[s].x;
            R f, df = R(0);
            if (cut_r) {
                if constexpr (MODE == MODE_ADJ) { f = S.QF[s].x; df = S.QF[s].y * r; }
                else if constexpr (MODE == MODE_FWD) f = S.Q2[s].y;
                else { f = S.Q[s].z; df = S.Q[s].w; }
            } else {
                cutoff<R>(cut, rc, irc, tanh_pre, r, f, df);
            }
            R rdot = R(0);
            V4<R> pv;
            if (MODE != MODE_FWD) pv = S.P[s];
            if (MODE == MODE_TAN)
                rdot = (pv.x * S.D[s] + pv.y * S.D[cap + s] + pv.z * S.D[2 * cap + s]) * pv.w;
            R dsum = R(0);
#pragma unroll
            for (int q = 0; q < kFun; ++q) {
                if (q < nfun) {
                    const R d = r - rs[q];
                    const R ex = M<R>::ex2k(keta[q] * d * d);
                    if (MODE == MODE_FWD) acc[q] += ex * f;
                    if (MODE == MODE_ADJ) dsum += wgt[q] * ex * (df - R(2) * eta[q] * d * f);
                    if (MODE == MODE_TAN) acc[q] += ex * (df - R(2) * eta[q] * d * f) * rdot;
                }
            }
            if (MODE == MODE_ADJ) {
                const R sc = dsum * pv.w;
                const R gx = sc * pv.x, gy = sc * pv.y, gz = sc * pv.z;
                S.DA[3 * s] -= (double)gx; S.DA[3 * s + 1] -= (double)gy; S.DA[3 * s + 2] -= (double)gz;
            }
        }
        if (MODE != MODE_ADJ) {
            const R v = wave_sums<kFun>(acc);
            const int f = sum_of_lane<kFun>();
            const int col = __shfl(G.w, kCol + f0 + max(f, 0), kWave);
            if (f >= 0 && f < nfun) out[(size_t)c * a.ld + col] = v;
        }
        wave_sync();
    }

    // ---- angular groups ----------------------------------------------------
    bool bad = false;   // a group outside this kernel's table class
    int turn = sub;              // a team's wavefronts take the steps of all groups in turn
    int pending_col = -1, pending_cell = 0;   // this wavefront's pending group: the lane's column and cell
    for (int g = 0; g < n_ag; ++g) {
        typedef pt_angular_group AG;
        constexpr int kCol = PT_WORD(AG, col), kCells = PT_AG_ETA * PT_AG_ANG;
        const GroupWords G = WPC > 1 ? Gn : group_words(&tab->ag[g]);
        if (WPC > 1 && g + 1 < n_ag) Gn = group_words(&tab->ag[g + 1]);
        const R gr = (R)G.d;
        AngGroup<R> X;
        const int ej = lane_word(G.w, PT_WORD(AG, ej)), ek = lane_word(G.w, PT_WORD(AG, ek));
        X.bj = seg_below(seg, ej);
        X.nj = seg_below(seg, ej + 1) - X.bj;
        X.bk = seg_below(seg, ek);
        X.nk = seg_below(seg, ek + 1) - X.bk;
        X.same = ej == ek;
        X.g3 = lane_word(G.w, PT_WORD(AG, kind)) == 3;
        X.mic = mic_jk;
        X.n_eta = lane_word(G.w, PT_WORD(AG, n_eta));
        X.n_ang = lane_word(G.w, PT_WORD(AG, n_ang));
        X.cut = lane_word(G.w, PT_WORD(AG, cut));
        X.rc = lane_value(gr, PT_DBL(AG, rc));
        X.irc = lane_value((R)(1.0 / G.d), PT_DBL(AG, rc));
        X.cpre = X.cut == PT_CUT_TANH ? tanh_pre : R(1);
        X.tanh_pre = tanh_pre;
        X.box = &box;
        // qmap[k]: the table term evaluated in slot k (the identity, or the
        // canonical order of a ZETA {1, 4} x LAMBDA {+1, -1} group)
        int qmap[PT_AG_ANG];
        const int z14 = (KIND == PT_ACSF_TANH_Z14) ? z14_order(G, X.n_ang, qmap) : 0;
        if (!z14) {
#pragma unroll
            for (int q = 0; q < PT_AG_ANG; ++q) qmap[q] = q;
        }
        // lane kCol + cell holds the cell's column and its weight (adjoint)
        const int cell = lane - kCol;
        const bool mine = cell >= 0 && cell < kCells && cell / PT_AG_ANG < X.n_eta && cell % PT_AG_ANG < X.n_ang && G.w >= 0;
        R wl = R(0);
        if (MODE == MODE_ADJ) {
            if (WPC > 1 && a.ld <= kWave) {
                const R v = __shfl(wrow, mine ? G.w : 0, kWave);
                wl = mine ? v : R(0);
            } else if (mine) {
                wl = w[(size_t)c * a.ld + G.w];
            }
        }
        R W[PT_AG_ETA][PT_AG_ANG], acc[PT_AG_ETA][PT_AG_ANG];
        const R keta_l = (R)(-G.d * M<R>::kexp);
#pragma unroll
        for (int e = 0; e < PT_AG_ETA; ++e) {
            X.keta[e] = (e < X.n_eta) ? lane_value(keta_l, PT_DBL(AG, eta) + e) : R(0);
#pragma unroll
            for (int q = 0; q < PT_AG_ANG; ++q) {
                acc[e][q] = R(0);
                W[e][q] = MODE == MODE_ADJ ? lane_value(wl, kCol + e * PT_AG_ANG + qmap[q]) : R(0);
            }
        }
        const R zl_l = (R)(G.d * __shfl(G.d, lane + PT_DBL(AG, lam) - PT_DBL(AG, zeta)));   // zeta lambda, in zeta's lanes
        bool z1 = true, p4 = true;
#pragma unroll
        for (int q = 0; q < PT_AG_ANG; ++q) {
            const bool on = q < X.n_ang;
            const int tq = qmap[q];
            X.lam[q] = on ? lane_value(gr, PT_DBL(AG, lam) + tq) : R(0);
            X.zeta[q] = on ? lane_value(gr, PT_DBL(AG, zeta) + tq) : R(1);
            X.pre[q] = on ? lane_value(gr, PT_DBL(AG, pre) + tq) : R(0);
            X.izeta[q] = on ? lane_word(G.w, PT_WORD(AG, izeta) + tq) : 1;
            X.zl[q] = on ? lane_value(zl_l, PT_DBL(AG, zeta) + tq) : R(0);
            z1 = z1 && X.izeta[q] == 1;
            p4 = p4 && (X.izeta[q] == 1 || X.izeta[q] == 2 || X.izeta[q] == 4);
        }
        const int ck = (X.cut == PT_CUT_TANH || X.cut == PT_CUT_TANHU) ? CUTK_TANH
                       : (X.cut == PT_CUT_COS ? CUTK_COS : CUTK_GEN);
        const int ak = z14 ? ANGK_Z14
                           : (z1 ? (X.n_ang <= 2 ? ANGK_Z1N2 : ANGK_Z1) : (p4 ? ANGK_P4 : ANGK_GEN));
        if (!cut_a) centre_sync<WPC>();   // the previous group's cutoff values are no longer read
        int steps = 0;
        if constexpr (KIND == PT_ACSF_TANH_Z14) {
            if (ck == CUTK_TANH && ak == ANGK_Z14)
                steps = angular_group<R, MODE, CUTK_TANH, ANGK_Z14, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else
                bad = true;
        } else if constexpr (KIND == PT_ACSF_TANH_P4) {
            if (ck == CUTK_TANH && ak != ANGK_GEN)
                steps = angular_group<R, MODE, CUTK_TANH, ANGK_P4, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else
                bad = true;
        } else if constexpr (KIND == PT_ACSF_TANH_Z1N2) {
            if (ck == CUTK_TANH && ak == ANGK_Z1N2)
                steps = angular_group<R, MODE, CUTK_TANH, ANGK_Z1N2, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else
                bad = true;
        } else if (MODE == MODE_TAN || (sizeof(R) == 8 && ck != CUTK_TANH)) {
            steps = angular_group<R, MODE, CUTK_GEN, ANGK_GEN, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
        } else if (sizeof(R) == 8) {
            if (ak == ANGK_GEN) steps = angular_group<R, MODE, CUTK_TANH, ANGK_GEN, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else steps = angular_group<R, MODE, CUTK_TANH, ANGK_P4, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
        } else if (ck == CUTK_TANH) {
            if (ak == ANGK_Z1N2) steps = angular_group<R, MODE, CUTK_TANH, ANGK_Z1N2, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else if (ak == ANGK_Z1) steps = angular_group<R, MODE, CUTK_TANH, ANGK_Z1, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else if (ak == ANGK_P4) steps = angular_group<R, MODE, CUTK_TANH, ANGK_P4, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else steps = angular_group<R, MODE, CUTK_TANH, ANGK_GEN, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
        } else if (ck == CUTK_COS) {
            if (ak == ANGK_Z1N2) steps = angular_group<R, MODE, CUTK_COS, ANGK_Z1N2, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else if (ak == ANGK_Z1) steps = angular_group<R, MODE, CUTK_COS, ANGK_Z1, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else if (ak == ANGK_P4) steps = angular_group<R, MODE, CUTK_COS, ANGK_P4, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
            else steps = angular_group<R, MODE, CUTK_COS, ANGK_GEN, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
        } else {
            steps = angular_group<R, MODE, CUTK_GEN, ANGK_GEN, WPC>(S, X, W, acc, cap, sub, turn, cut_a);
        }

        if (MODE != MODE_ADJ) {
            // three eta values and fewer leave the last row of cells out
            R* row = out + (size_t)c * a.ld;
            constexpr int kPending = Team<R, WPC>::kPending;
            const int slot = g % kPending;
            if (X.n_eta < PT_AG_ETA)
                store_cells<kCells - PT_AG_ANG>(acc, qmap, G.w, X.n_eta, X.n_ang, T, sub, slot, pending_col, pending_cell, row);
            else
                store_cells<kCells>(acc, qmap, G.w, X.n_eta, X.n_ang, T, sub, slot, pending_col, pending_cell, row);
            if constexpr (WPC > 1) {
                if (slot == kPending - 1 || g + 1 == n_ag) {
                    // each pending group's parts, in order, by one wavefront
                    __syncthreads();
                    if (sub <= slot && pending_col >= 0) {
                        R v = T.part[0][sub][pending_cell];
#pragma unroll
                        for (int k = 1; k < WPC; ++k) v += T.part[k][sub][pending_cell];
                        row[pending_col] = v;
                    }
                    if (g + 1 < n_ag) __syncthreads();
                }
            }
        }
        if constexpr (WPC == 1) wave_sync();
        else turn = (turn + WPC - steps % WPC) % WPC;
    }
    centre_sync<WPC>();

    const R nan = __builtin_nan("");
    if (MODE != MODE_ADJ && bad && sub == 0) {
        for (int q = lane; q < a.ld; q += kWave) out[(size_t)c * a.ld + q] = nan;
    }
    if (MODE == MODE_ADJ) {
        if constexpr (WPC > 1) {
            // the wavefronts' accumulators, in order, into those of the first
            double* D0 = S.DA - 3 * cap * sub;
            for (int s = threadIdx.x; s < 3 * m; s += WPC * kWave) {
                double v = D0[s];
#pragma unroll
                for (int k = 1; k < WPC; ++k) v += D0[3 * cap * k + s];
                D0[s] = v;
            }
            S.DA = D0;
            __syncthreads();
        }
        if (a.edge_grad) {
            R* eg = (R*)a.edge_grad;
            // the staging ballots give each kept row entry its staged slot
            int ms = 0;
            for (int t0 = 0; t0 < len; t0 += kWave) {
                const unsigned long long bal = S.keep[t0 / kWave];
                if ((WPC == 1 || t0 / kWave % WPC == sub) && ((bal >> lane) & 1ull)) {
                    const int s = ms + lanes_below(bal);
                    const long long e = a.rev ? (long long)a.rev[off + t0 + lane] : off + t0 + lane;
                    if (e >= 0) {
                        eg[3 * e + 0] = bad ? nan : (R)S.DA[3 * s];
                        eg[3 * e + 1] = bad ? nan : (R)S.DA[3 * s + 1];
                        eg[3 * e + 2] = bad ? nan : (R)S.DA[3 * s + 2];
                    }
                }
                ms += __popcll(bal);
            }
        }
        if (rn.f_self && sub == 0) {
            // G_i depends on r_i only through R_ij = r_i - r_j, so dE_i/dr_i = -sum_j dE_i/dr_j
            // and F_self = -dE_i/dr_i = sum_j dE_i/dr_j, the per-edge accumulators
            double fx = 0.0, fy = 0.0, fz = 0.0;
            for (int s = lane; s < m; s += kWave) {
                fx += S.DA[3 * s];
                fy += S.DA[3 * s + 1];
                fz += S.DA[3 * s + 2];
            }
            const double sx = wave_sum(fx), sy = wave_sum(fy), sz = wave_sum(fz);
            if (lane == 0) {
                rn.f_self[3 * c + 0] = bad ? (double)nan : sx;
                rn.f_self[3 * c + 1] = bad ? (double)nan : sy;
                rn.f_self[3 * c + 2] = bad ? (double)nan : sz;
            }
        }
    }
}

// Entry kernels over the same body: the others ask the compiler for four
// (<= 128 VGPRs) or eight (<= 64 VGPRs) resident waves per SIMD; the FP64
// forwards of the specialised table classes and the FP32 forwards of the
// zeta {1, 4} and zeta = 1 classes fit those without spills.
template <typename R, int MODE, int KIND>
__global__ __launch_bounds__(256) void k_acsf(KArgs a) {
    extern __shared__ __align__(32) char smem[];
    Team<R, 1> T;
    acsf_centre<R, MODE, KIND, 1>(a, smem, T);
}

template <typename R, int MODE, int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_acsf_w4(KArgs a) {
    extern __shared__ __align__(32) char smem[];
    Team<R, 1> T;
    acsf_centre<R, MODE, KIND, 1>(a, smem, T);
}

template <typename R, int MODE, int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_acsf_w8(KArgs a) {
    extern __shared__ __align__(32) char smem[];
    Team<R, 1> T;
    acsf_centre<R, MODE, KIND, 1>(a, smem, T);
}

// A team of WPC wavefronts per centre.
// (the FP64 tangent of the table classes is held to three waves per SIMD: with two, 768
// items took 73 us, not 59)
template <typename R, int MODE, int KIND, int WPC>
__global__ __launch_bounds__(64 * WPC, sizeof(R) == 8 && MODE == MODE_TAN && KIND != PT_ACSF_GENERIC ? 3 : 1)
void k_acsf_team(KArgs a) {
    extern __shared__ __align__(32) char smem[];
    __shared__ Team<R, WPC> T;
    acsf_centre<R, MODE, KIND, WPC>(a, smem, T);
}

// Launches of at most this many centres run a team per centre: of 8 wavefronts while all
// teams are resident at two to a CU (one, for the FP64 tangent's registers), of 4 until a
// wavefront per centre fills the chip as well.  Rows of fewer than kTeamRow entries leave
// a team little to share; teams of 8 gain them nothing.  A centre's wavefronts meet only where the
// row is staged and where sums are added: radial groups go by halves, the pair steps of
// all angular groups in turn, and a group's table words are loaded while the one before
// runs.  (With barriers around every group FP64 took 31 and 37 us at 96 centres, FP32 27 and 33 at 384.)
// Measured, us per launch (HIP events over 40 launches in a row), wavefronts per centre
// 1 | 4 | 8 (52 functions at 12 Bohr, ~110 neighbours; 34 at 8 Bohr, ~32):
//   12 Bohr FP64 forward  96 centres 60.0 | 24.9 | 19.8   512 66.0 | 30.5 | 29.7   640 66.1 | 34.5 | 38.4   1,792 78.7 | 66.5
//   12 Bohr FP64 adjoint  96 centres 73.3 | 31.7 | 25.0   512 81.4 | 40.7 | 38.1   640 81.7 | 46.6 | 50.8   1,792 102 | 92.1
//   12 Bohr FP64 tangent  96 centres 70.8 | 30.1 | 23.6   256 75.2 | 31.1 | 25.4   512 78.3 | 39.2 | 46.4   1,792 98.1 | 93.8   2,048 102 | 106
//   12 Bohr FP32 forward  96 centres 43.1 | 18.8 | 14.8   512 47.4 | 21.3 | 19.7   640 47.4 | 22.8 | 23.6   1,792 50.7 | 40.6
//   12 Bohr FP32 adjoint  96 centres 53.4 | 23.5 | 18.6   512 58.8 | 27.5 | 25.1   640 59.1 | 29.7 | 35.3   1,792 66.5 | 55.7
//   12 Bohr FP32 tangent  96 centres 54.2 | 22.7 | 17.5   512 60.3 | 26.1 | 23.8   640 59.7 | 28.3 | 32.9   1,792 64.2 | 54.6
//   8 Bohr FP32 forward   96 centres 13.0 | 10.1 | 9.3    768 13.8 | 12.4          1,280 15.5 | 15.6
//   8 Bohr FP64 adjoint   96 centres 21.2 | 15.0 | 14.1   768 22.5 | 19.5          1,280 26.3 | 29.7
// (teams of 2 win 5 to 15 % between 1,536 and 2,048 centres: not worth a third set of kernels.)
// The general table class has no teams of 8, and its FP64 kernels' registers leave two teams of 4
// to a CU, not four: long rows gain up to 1,280 centres, short ones while all teams are
// resident.  Cosine cutoff, 1 | 4:
//   12 Bohr FP64 forward  512 centres 104 | 49.7   640 104 | 73.4   1,280 122 | 116   1,536 124 | 130
//   12 Bohr FP64 adjoint  512 centres 146 | 72.1   640 146 | 107    1,280 176 | 170   1,536 180 | 191
//   12 Bohr FP32 adjoint  512 centres 65.3 | 32.9                   1,792 74.0 | 67.9
//   8 Bohr FP64 forward   512 centres 28.2 | 25.5  640 27.8 | 40.7
//   8 Bohr FP64 adjoint   512 centres 39.0 | 34.8  640 38.6 | 56.3
//   8 Bohr FP32 adjoint   768 centres 18.6 | 18.2
constexpr int kTeam8 = 512, kTeam8Tan64 = 256, kTeamLong = 1792, kTeamShort = 768, kTeamRow = 80;
constexpr int kTeamLongGeneral64 = 1280, kTeamShortGeneral64 = 512;

template <typename R, int MODE, int KIND>
int launch(KArgs a, hipStream_t stream) {
    if (a.n_items <= 0) return PT_OK;
    a.cap = (std::max(a.cap, 1) + 3) / 4 * 4;
    if (a.cap > 65535) {
        set_error("acsf: neighbour rows longer than 65535 entries are not supported");
        return PT_ERR_UNSUPPORTED;
    }
    const size_t per_wave = stage_bytes<R, MODE, 1>(a.cap);
    const size_t lds_budget = lds_limit();
    if (per_wave > lds_budget) {
        set_error("acsf: neighbour row of %d entries exceeds the LDS budget", a.cap);
        return PT_ERR_UNSUPPORTED;
    }
    // (a row that only fits the LDS without a team's extra arrays keeps one wavefront)
    auto team = [&](auto wpc, int most) {
        constexpr int W = decltype(wpc)::value;
        const size_t bytes = stage_bytes<R, MODE, W>(a.cap);
        if (a.n_items > most || bytes + sizeof(Team<R, W>) + 512 > lds_budget) return false;
        hipLaunchKernelGGL((k_acsf_team<R, MODE, KIND, W>), dim3(a.n_items), dim3(64 * W), bytes, stream, a);
        return true;
    };
    auto some_team = [&]() {
        constexpr std::integral_constant<int, 4> w4{};
        constexpr bool general64 = KIND == PT_ACSF_GENERIC && sizeof(R) == 8;
        if (a.cap < kTeamRow) return team(w4, general64 ? kTeamShortGeneral64 : kTeamShort);
        if constexpr (KIND != PT_ACSF_GENERIC)
            if (team(std::integral_constant<int, 8>{}, sizeof(R) == 8 && MODE == MODE_TAN ? kTeam8Tan64 : kTeam8)) return true;
        return team(w4, general64 ? kTeamLongGeneral64 : kTeamLong);
    };
    if (some_team())
        return launch_check("k_acsf_team");
    // waves per workgroup: the most resident waves per CU under the LDS limit,
    // ties to the smaller workgroup (a workgroup's LDS is held until its
    // slowest wave ends; one-wave groups ran the FP32 adjoint 2.5 % faster
    // than two-wave groups at the same 18 resident waves)
    const size_t cu = std::max(lds_per_cu(), lds_budget);
    int wpb = 1;
    size_t best = 0;
    for (int w = 1; w <= 4; w *= 2) {
        if ((size_t)w * per_wave > lds_budget) break;
        const size_t waves = (size_t)w * (cu / ((size_t)w * per_wave));
        if (waves > best) { best = waves; wpb = w; }
    }
    const int blocks = (a.n_items + wpb - 1) / wpb;
    if constexpr (sizeof(R) == 8 && MODE == MODE_FWD && KIND != PT_ACSF_GENERIC)
        hipLaunchKernelGGL((k_acsf_w4<R, MODE, KIND>), dim3(blocks), dim3(64 * wpb), wpb * per_wave, stream, a);
    else if constexpr (sizeof(R) == 4 && MODE == MODE_FWD && (KIND == PT_ACSF_TANH_Z14 || KIND == PT_ACSF_TANH_Z1N2))
        hipLaunchKernelGGL((k_acsf_w8<R, MODE, KIND>), dim3(blocks), dim3(64 * wpb), wpb * per_wave, stream, a);
    else
        hipLaunchKernelGGL((k_acsf<R, MODE, KIND>), dim3(blocks), dim3(64 * wpb), wpb * per_wave, stream, a);
    return launch_check("k_acsf");
}

template <typename R, int MODE>
int run_kind(int kind, const KArgs& a, hipStream_t st) {
    switch (kind) {
    case PT_ACSF_GENERIC: return launch<R, MODE, PT_ACSF_GENERIC>(a, st);
    case PT_ACSF_TANH_P4: return launch<R, MODE, PT_ACSF_TANH_P4>(a, st);
    case PT_ACSF_TANH_Z1N2: return launch<R, MODE, PT_ACSF_TANH_Z1N2>(a, st);
    case PT_ACSF_TANH_Z14: return launch<R, MODE, PT_ACSF_TANH_Z14>(a, st);
    }
    set_error("acsf: unknown kernel kind %d", kind);
    return PT_ERR_ARG;
}

// The runs of one table kind go into one launch (kMaxRuns at a time), in order.
template <int MODE>
int run_all(int precision, KArgs& a, int n_runs, const pt_acsf_run* runs, hipStream_t st) {
    PT_REQUIRE(precision == PT_F64 || precision == PT_F32, "acsf: unknown precision %d", precision);
    for (int r = 0; r < n_runs; ++r) {
        PT_REQUIRE(runs[r].n_centers >= 0, "acsf: bad sizes");
        PT_REQUIRE(runs[r].table, "acsf: null argument");
    }
    for (int r = 0; r < n_runs;) {
        const int kind = runs[r].kind;
        long long items = 0;
        a.n_runs = 0;
        for (; r < n_runs && runs[r].kind == kind && a.n_runs < kMaxRuns; ++r) {
            const pt_acsf_run& q = runs[r];
            if (q.n_centers == 0) continue;
            KRun& k = a.run[a.n_runs++];
            k.table = q.table;
            k.centers = q.centers;
            k.out = q.out;
            k.w = q.w;
            k.f_self = q.f_self;
            k.delta = q.delta;
            k.dir = q.dir;
            k.n = q.n_centers;
            k.begin = q.center_begin;
            k.item0 = (int)items;
            items += q.n_centers;
        }
        PT_REQUIRE(items < (1LL << 31), "acsf: too many centres in one launch");
        a.n_items = (int)items;
        const int rc = precision == PT_F64 ? run_kind<double, MODE>(kind, a, st) : run_kind<float, MODE>(kind, a, st);
        if (rc) return rc;
    }
    return PT_OK;
}

KArgs common_args(const double* pos4, const double* box, const long long* row_off, const int* nbr, int max_row) {
    KArgs a{};
    a.pos4 = pos4;
    a.box.periodic = box != nullptr;
    for (int d = 0; d < 3; ++d) {
        a.box.L[d] = box ? box[d] : 0.0;
        a.box.half[d] = box ? 0.5 * box[d] : 0.0;
    }
    a.row_off = row_off;
    a.nbr = nbr;
    a.cap = max_row;
    return a;
}

// a run of the single-table entry points (their precision argument carries the table kind)
pt_acsf_run single_run(int precision_kind, const pt_sf_table* table, int n_centers, int center_begin,
                       const int* centers) {
    pt_acsf_run r{};
    r.table = table;
    r.kind = precision_kind >> PT_ACSF_KIND_SHIFT;
    r.n_centers = n_centers;
    r.center_begin = center_begin;
    r.centers = centers;
    return r;
}

int base_precision(int precision_kind) { return precision_kind & ((1 << PT_ACSF_KIND_SHIFT) - 1); }

}  // namespace
}  // namespace pt

using namespace pt;

extern "C" int pt_acsf_forward_multi(int precision, const double* pos4, const double* box, const long long* row_off,
                                     const int* nbr, int max_row, int n_runs, const pt_acsf_run* runs, int ldg,
                                     pt_stream_t stream) {
    PT_REQUIRE(pos4 && row_off && n_runs >= 0 && (runs || n_runs == 0), "pt_acsf_forward: null argument");
    PT_REQUIRE(ldg >= 0, "pt_acsf_forward: bad sizes");
    for (int r = 0; r < n_runs; ++r)
        PT_REQUIRE(runs[r].out || runs[r].n_centers == 0, "pt_acsf_forward: null argument");
    KArgs a = common_args(pos4, box, row_off, nbr, max_row);
    a.ld = ldg;
    return run_all<MODE_FWD>(precision, a, n_runs, runs, (hipStream_t)stream);
}

extern "C" int pt_acsf_forward(int precision, const double* pos4, const double* box,
                               const long long* row_off, const int* nbr, int max_row,
                               int n_centers, int center_begin, const int* centers,
                               const pt_sf_table* table, void* G, int ldg, pt_stream_t stream) {
    pt_acsf_run r = single_run(precision, table, n_centers, center_begin, centers);
    r.out = G;
    return pt_acsf_forward_multi(base_precision(precision), pos4, box, row_off, nbr, max_row, 1, &r, ldg, stream);
}

extern "C" int pt_acsf_adjoint_multi(int precision, const double* pos4, const double* box, const double* boxes,
                                     const int* box_id, const long long* row_off, const int* nbr, const int* rev,
                                     int max_row, int n_runs, const pt_acsf_run* runs, int ldw, void* edge_grad,
                                     pt_stream_t stream) {
    PT_REQUIRE(pos4 && row_off && n_runs >= 0 && (runs || n_runs == 0), "pt_acsf_adjoint: null argument");
    PT_REQUIRE(!boxes || (box_id && !box), "pt_acsf_adjoint: box table without box indices");
    for (int r = 0; r < n_runs; ++r)
        PT_REQUIRE(runs[r].w || runs[r].n_centers == 0, "pt_acsf_adjoint: null argument");
    KArgs a = common_args(pos4, box, row_off, nbr, max_row);
    a.boxes = boxes;
    a.box_id = box_id;
    a.ld = ldw;
    a.edge_grad = edge_grad;
    a.rev = rev;
    return run_all<MODE_ADJ>(precision, a, n_runs, runs, (hipStream_t)stream);
}

extern "C" int pt_acsf_adjoint(int precision, const double* pos4, const double* box,
                               const long long* row_off, const int* nbr, int max_row,
                               int n_centers, int center_begin, const int* centers,
                               const pt_sf_table* table, const void* w, int ldw, double* f_self,
                               void* edge_grad, pt_stream_t stream) {
    pt_acsf_run r = single_run(precision, table, std::max(n_centers, 0), center_begin, centers);
    r.w = w;
    r.f_self = f_self;
    return pt_acsf_adjoint_multi(base_precision(precision), pos4, box, nullptr, nullptr, row_off, nbr, nullptr,
                                 max_row, 1, &r, ldw, edge_grad, stream);
}

extern "C" int pt_acsf_adjoint_transposed(int precision, const double* pos4, const double* box,
                                          const long long* row_off, const int* nbr, const int* rev, int max_row,
                                          int n_centers, int center_begin, const int* centers,
                                          const pt_sf_table* table, const void* w, int ldw, double* f_self,
                                          void* edge_grad_t, pt_stream_t stream) {
    PT_REQUIRE(rev, "pt_acsf_adjoint_transposed: null argument");
    pt_acsf_run r = single_run(precision, table, std::max(n_centers, 0), center_begin, centers);
    r.w = w;
    r.f_self = f_self;
    return pt_acsf_adjoint_multi(base_precision(precision), pos4, box, nullptr, nullptr, row_off, nbr, rev, max_row,
                                 1, &r, ldw, edge_grad_t, stream);
}

extern "C" int pt_acsf_tangent_multi(int precision, const double* pos4, const double* box, const double* boxes,
                                     const int* box_id, const long long* row_off, const int* nbr, int max_row,
                                     int n_runs, const pt_acsf_run* runs, int center_only, int ldt,
                                     pt_stream_t stream) {
    PT_REQUIRE(pos4 && row_off && n_runs >= 0 && (runs || n_runs == 0), "pt_acsf_tangent: null argument");
    PT_REQUIRE(!boxes || (box_id && !box), "pt_acsf_tangent: box table without box indices");
    for (int r = 0; r < n_runs; ++r) {
        PT_REQUIRE(runs[r].out || runs[r].n_centers == 0, "pt_acsf_tangent: null argument");
        PT_REQUIRE(runs[r].delta || (center_only && runs[r].dir >= 0 && runs[r].dir <= 2),
                   "pt_acsf_tangent: a run without a displacement field needs a direction and center_only");
    }
    KArgs a = common_args(pos4, box, row_off, nbr, max_row);
    a.boxes = boxes;
    a.box_id = box_id;
    a.ld = ldt;
    a.center_only = center_only;
    return run_all<MODE_TAN>(precision, a, n_runs, runs, (hipStream_t)stream);
}

extern "C" int pt_acsf_tangent(int precision, const double* pos4, const double* box,
                               const long long* row_off, const int* nbr, int max_row,
                               int n_centers, int center_begin, const int* centers,
                               const pt_sf_table* table, const double* delta, int center_only,
                               void* T, int ldt, pt_stream_t stream) {
    PT_REQUIRE(delta, "pt_acsf_tangent: null argument");
    pt_acsf_run r = single_run(precision, table, std::max(n_centers, 0), center_begin, centers);
    r.out = T;
    r.delta = delta;
    return pt_acsf_tangent_multi(base_precision(precision), pos4, box, nullptr, nullptr, row_off, nbr, max_row, 1,
                                 &r, center_only, ldt, stream);
}

extern "C" int pt_sf_table_kind(const pt_sf_table* t) {
    if (!t) return PT_ACSF_GENERIC;
    if (t->n_ag <= 0) return PT_ACSF_GENERIC;
    bool p4 = true, z1n2 = true, z14 = true;
    for (int g = 0; g < t->n_ag && g < PT_MAX_GROUPS; ++g) {
        const pt_angular_group& G = t->ag[g];
        const bool tanh = G.cut == PT_CUT_TANH || G.cut == PT_CUT_TANHU;
        bool allz1 = true, allp4 = true;
        int seen = 0;
        for (int q = 0; q < G.n_ang; ++q) {
            allz1 = allz1 && G.izeta[q] == 1;
            allp4 = allp4 && (G.izeta[q] == 1 || G.izeta[q] == 2 || G.izeta[q] == 4);
            // the kernel's test (z14_order): zeta 1 or 4, lambda exactly +1 or -1, each pair once
            if ((G.izeta[q] == 1 || G.izeta[q] == 4) && (G.lam[q] == 1.0 || G.lam[q] == -1.0))
                seen |= 1 << ((G.izeta[q] == 4 ? 2 : 0) + (G.lam[q] < 0.0 ? 1 : 0));
            else
                seen |= 1 << 4;
        }
        p4 = p4 && tanh && allp4;
        z1n2 = z1n2 && tanh && allz1 && G.n_ang <= 2;
        z14 = z14 && tanh && G.n_ang == 4 && seen == 15;
    }
    return z1n2 ? PT_ACSF_TANH_Z1N2 : (z14 ? PT_ACSF_TANH_Z14 : (p4 ? PT_ACSF_TANH_P4 : PT_ACSF_GENERIC));
}
