// (c'') A training batch as one list: the neighbour lists, descriptors and
// labels of several structures are copied into one set of arrays, so that every
// step of the loss gradient (MLP, adjoint, force gather, seeds, tangent, weight
// gradient) is one launch over all structures instead of one per structure.
//
// Layout of the batch: segment q = e * n_struct + k holds the atoms of element e
// of structure k, in the structure's internal order.  Atoms of one element are
// contiguous (plain GEMM rows for the MLP); a row keeps its order (type-sorted,
// as the descriptor kernels need it), so an edge keeps its position in its row
// and the reverse index follows from the reverse edge's row.  Why: a structure of a few hundred atoms leaves most of the chip
// idle and every launch costs its fixed latency; 32 structures of 96 to 1,536
// atoms took 393 launches and 7.5 ms per gradient.
#include <cmath>

#include "common.h"

namespace pt {
namespace {

// Words of a structure's record in the plan (pt_train_batch_* in the header).
enum { R_POS4, R_ROWOFF, R_NBR, R_REV, R_G, R_FREF, R_EREF, R_BOX, R_N = R_BOX + 3, R_WORDS };

constexpr int kMaxElem = 8;

struct Plan {
    const long long* rec;     // [n_struct][R_WORDS]
    const long long* begin;   // [n_struct][n_elem] first atom of element e's block (structure order)
    const long long* edge0;   // [n_struct][n_elem] row_off at that atom
    const long long* atom;    // [n_elem * n_struct + 1] first batch atom of a segment
    const long long* edge;    // [n_elem * n_struct + 1] first batch edge of a segment
    int ns, ne;
};

__host__ __device__ inline Plan make_plan(const long long* p, int ns, int ne) {
    Plan q;
    q.ns = ns;
    q.ne = ne;
    q.rec = p;
    q.begin = q.rec + (size_t)ns * R_WORDS;
    q.edge0 = q.begin + (size_t)ns * ne;
    q.atom = q.edge0 + (size_t)ns * ne;
    q.edge = q.atom + (size_t)ns * ne + 1;
    return q;
}

__device__ __forceinline__ double as_f64(long long v) { return __builtin_bit_cast(double, v); }

// One wavefront per batch atom: position, descriptors, label, list row.
template <typename R>
__global__ __launch_bounds__(256) void k_batch_assemble(Plan p, int n_atoms, int ld, double* __restrict__ pos4,
                                                        long long* __restrict__ row_off, int* __restrict__ nbr,
                                                        int* __restrict__ rev, R* __restrict__ G,
                                                        double* __restrict__ f_ref, int* __restrict__ box_id,
                                                        double* __restrict__ boxes) {
    const int lane = wave_lane();
    const int i = uniform(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (i >= n_atoms) return;
    int lo = 0, hi = p.ne * p.ns;   // the segment of atom i: the largest q with atom[q] <= i
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (p.atom[mid] <= i) lo = mid; else hi = mid;
    }
    const int q = lo, e = q / p.ns, k = q - e * p.ns;
    const long long* rec = p.rec + (size_t)k * R_WORDS;
    const int li = (int)p.begin[(size_t)k * p.ne + e] + (i - (int)p.atom[q]);
    const long long* ro = (const long long*)rec[R_ROWOFF];
    const long long b = ro[li], len = ro[li + 1] - b;
    const long long ob = p.edge[q] + (b - p.edge0[(size_t)k * p.ne + e]);
    if (lane < 4) pos4[4 * (size_t)i + lane] = ((const double*)rec[R_POS4])[4 * (size_t)li + lane];
    if (lane < 3) f_ref[3 * (size_t)i + lane] = ((const double*)rec[R_FREF])[3 * (size_t)li + lane];
    if (lane == 0) {
        row_off[i] = ob;
        if (i == n_atoms - 1) row_off[n_atoms] = ob + len;
        box_id[i] = k;
    }
    if (li == 0 && lane < 3) boxes[3 * (size_t)k + lane] = as_f64(rec[R_BOX + lane]);
    const R* g = (const R*)rec[R_G] + (size_t)li * ld;
    for (int c = lane; c < ld; c += kWave) G[(size_t)i * ld + c] = g[c];
    // element blocks of the structure: local atom -> batch atom, local edge -> batch edge
    int blk[kMaxElem];
    long long da[kMaxElem], de[kMaxElem];
#pragma unroll
    for (int t = 0; t < kMaxElem; ++t) {
        if (t < p.ne) {
            const int s = t * p.ns + k;
            blk[t] = (int)p.begin[(size_t)k * p.ne + t];
            da[t] = p.atom[s] - blk[t];
            de[t] = p.edge[s] - p.edge0[(size_t)k * p.ne + t];
        } else {
            blk[t] = 0; da[t] = 0; de[t] = 0;
        }
    }
    const int* nb = (const int*)rec[R_NBR];
    const int* rv = (const int*)rec[R_REV];
    for (long long t = lane; t < len; t += kWave) {
        const int j = nb[b + t];
        // the block of j: the one with the largest first atom <= j
        int best = -1;
        long long a = 0, d = 0;
#pragma unroll
        for (int s = 0; s < kMaxElem; ++s) {
            if (s < p.ne && blk[s] <= j && blk[s] > best) { best = blk[s]; a = da[s]; d = de[s]; }
        }
        nbr[ob + t] = (int)(j + a);
        rev[ob + t] = (int)(rv[b + t] + d);
    }
}

// One wavefront per batch atom: F = f_self - row sum of the transposed edge
// gradients, delta = dL/dF, |F - F*|^2.
template <typename E>
__global__ __launch_bounds__(256) void k_batch_forces(Plan p, int n_atoms, const long long* __restrict__ row_off,
                                                      const double* __restrict__ f_self, const E* __restrict__ gT,
                                                      const int* __restrict__ box_id,
                                                      const double* __restrict__ f_ref, double wf,
                                                      double* __restrict__ delta, double* __restrict__ sq) {
    const int lane = wave_lane();
    const int i = uniform(xcd_block() * 4 + (threadIdx.x >> 6));
    if (i >= n_atoms) return;
    const long long b = row_off[i], e = row_off[i + 1];
    double f[3] = {0, 0, 0};
    for (long long k = b + lane; k < e; k += kWave)
        for (int d = 0; d < 3; ++d) f[d] += (double)gT[3 * k + d];
    for (int d = 0; d < 3; ++d) f[d] = wave_sum(f[d]);
    if (lane == 0) {
        const double n = (double)p.rec[(size_t)box_id[i] * R_WORDS + R_N];
        double s = 0.0;
        for (int d = 0; d < 3; ++d) {
            const double r = f_self[3 * (size_t)i + d] - f[d] - f_ref[3 * (size_t)i + d];
            delta[3 * (size_t)i + d] = wf * 2.0 * r / (3.0 * n);
            s += r * r;
        }
        sq[i] = s;
    }
}

__device__ __forceinline__ double block_sum256(double v, double* part) {
    v = wave_sum(v);
    __syncthreads();
    if (wave_lane() == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    return part[0] + part[1] + part[2] + part[3];
}

// One workgroup per structure: E, the energy seed of its atoms, both loss terms.
__global__ __launch_bounds__(256) void k_batch_seeds(Plan p, const double* __restrict__ e_atom,
                                                     const double* __restrict__ sq, double we, double wf,
                                                     double* __restrict__ gy, double* __restrict__ loss) {
    __shared__ double part[4];
    const int k = blockIdx.x;
    double es = 0.0, ss = 0.0;
    for (int t = 0; t < p.ne; ++t) {
        const int a = (int)p.atom[t * p.ns + k], z = (int)p.atom[t * p.ns + k + 1];
        for (int i = a + threadIdx.x; i < z; i += 256) { es += e_atom[i]; ss += sq[i]; }
    }
    const double E = block_sum256(es, part), S = block_sum256(ss, part);
    const long long* rec = p.rec + (size_t)k * R_WORDS;
    const double n = (double)rec[R_N], de = E - as_f64(rec[R_EREF]);
    const double g = we * 2.0 * de / (n * n);
    for (int t = 0; t < p.ne; ++t) {
        const int a = (int)p.atom[t * p.ns + k], z = (int)p.atom[t * p.ns + k + 1];
        for (int i = a + threadIdx.x; i < z; i += 256) gy[i] = g;
    }
    if (threadIdx.x == 0) {
        atomicAdd(&loss[0], we * de * de / (n * n));
        atomicAdd(&loss[1], wf * S / (3.0 * n));
    }
}

int check_batch(const char* what, int ns, int ne, const long long* plan, int n_atoms) {
    PT_REQUIRE(ns >= 1 && ne >= 1 && ne <= kMaxElem && plan && n_atoms >= 1, "%s: bad batch", what);
    return PT_OK;
}

}  // namespace
}  // namespace pt

using namespace pt;

extern "C" int pt_train_batch_words(int n_struct, int n_elem) {
    return n_struct * (R_WORDS + 2 * n_elem) + 2 * (n_struct * n_elem + 1);
}

extern "C" int pt_train_batch_assemble(int n_struct, int n_elem, const long long* plan, int n_atoms, int ld,
                                       int g_precision, double* pos4, long long* row_off, int* nbr, int* rev, void* G,
                                       double* f_ref, int* box_id, double* boxes, pt_stream_t stream) {
    if (int rc = check_batch("pt_train_batch_assemble", n_struct, n_elem, plan, n_atoms)) return rc;
    PT_REQUIRE(pos4 && row_off && nbr && rev && G && f_ref && box_id && boxes && ld >= 0,
               "pt_train_batch_assemble: null argument");
    PT_REQUIRE(g_precision == PT_F64 || g_precision == PT_F32, "pt_train_batch_assemble: bad precision");
    const Plan p = make_plan(plan, n_struct, n_elem);
    const dim3 grid((n_atoms + 3) / 4);
    if (g_precision == PT_F64)
        hipLaunchKernelGGL(k_batch_assemble<double>, grid, dim3(256), 0, (hipStream_t)stream, p, n_atoms, ld, pos4,
                           row_off, nbr, rev, (double*)G, f_ref, box_id, boxes);
    else
        hipLaunchKernelGGL(k_batch_assemble<float>, grid, dim3(256), 0, (hipStream_t)stream, p, n_atoms, ld, pos4,
                           row_off, nbr, rev, (float*)G, f_ref, box_id, boxes);
    return launch_check("k_batch_assemble");
}

extern "C" int pt_train_batch_seeds(int n_struct, int n_elem, const long long* plan, int n_atoms,
                                    const long long* row_off, const double* f_self, const void* edge_grad_t,
                                    int edge_precision, const int* box_id, const double* f_ref, const double* e_atom,
                                    double w_energy, double w_force, double* delta, double* gy, double* sq,
                                    double* loss, pt_stream_t stream) {
    if (int rc = check_batch("pt_train_batch_seeds", n_struct, n_elem, plan, n_atoms)) return rc;
    PT_REQUIRE(row_off && f_self && edge_grad_t && box_id && f_ref && e_atom && delta && gy && sq && loss,
               "pt_train_batch_seeds: null argument");
    PT_REQUIRE(edge_precision == PT_F64 || edge_precision == PT_F32, "pt_train_batch_seeds: bad precision");
    const Plan p = make_plan(plan, n_struct, n_elem);
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((n_atoms + 3) / 4);
    if (edge_precision == PT_F64)
        hipLaunchKernelGGL(k_batch_forces<double>, grid, dim3(256), 0, st, p, n_atoms, row_off, f_self,
                           (const double*)edge_grad_t, box_id, f_ref, w_force, delta, sq);
    else
        hipLaunchKernelGGL(k_batch_forces<float>, grid, dim3(256), 0, st, p, n_atoms, row_off, f_self,
                           (const float*)edge_grad_t, box_id, f_ref, w_force, delta, sq);
    if (int rc = launch_check("k_batch_forces")) return rc;
    hipLaunchKernelGGL(k_batch_seeds, dim3(n_struct), dim3(256), 0, st, p, e_atom, (const double*)sq, w_energy, w_force,
                       gy, loss);
    return launch_check("k_batch_seeds");
}
