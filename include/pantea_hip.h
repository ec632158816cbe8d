/*
 * pantea_hip.h -- C ABI of libpantea_hip.so, the gfx950 (MI355X) kernels of
 * the Behler-Parrinello NNP hot path.
 *
 * Conventions
 *  - Every pointer argument marked (device) is a device pointer (for example
 *    torch.Tensor.data_ptr() of a CUDA/HIP tensor); (host) pointers are read
 *    before the call returns.
 *  - Work is enqueued asynchronously on `stream` (a hipStream_t; pass
 *    torch.cuda.current_stream().cuda_stream).  Only pt_nbr_build
 *    synchronises `stream` (once, to read the pair count back, through a
 *    pageable copy: it allocates nothing); pt_nbr_build_async does not.
 *  - Return value: PT_OK (0) or a negative PT_ERR_*; pt_last_error() gives a
 *    thread-local message.  Buffers are owned by the caller; scratch comes in
 *    through `ws`/`ws_bytes`, sized by the *_workspace_bytes() queries.
 *  - Atom order: the neighbour build returns `perm` (internal -> input
 *    index) and all other entry points work on that internal order, in which
 *    atoms are grouped by type (ascending) and, inside a type, by cell.
 *
 * The reference (pantea 0.11.0) is pure Python on JAX; it has no FFI.  Each
 * entry point names the reference function it replaces (path:line in the
 * reference tree).
 */
#ifndef PANTEA_HIP_H
#define PANTEA_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef void *pt_stream_t; /* hipStream_t */

enum {
    PT_OK = 0,
    PT_ERR_ARG = -1,
    PT_ERR_CAPACITY = -2,
    PT_ERR_HIP = -3,
    PT_ERR_UNSUPPORTED = -4
};

/* Arithmetic of the descriptor kernels. */
enum { PT_F64 = 0, PT_F32 = 1 };

/* Descriptor kernel variants.  The precision argument of pt_acsf_forward /
 * pt_acsf_adjoint / pt_acsf_tangent may carry (kind << PT_ACSF_KIND_SHIFT), kind from
 * pt_sf_table_kind() of the table's host copy: the launch then uses a kernel
 * compiled for that table class only (fewer registers, higher occupancy).
 * Results are those of PT_ACSF_GENERIC; a kernel that meets a group outside
 * its class writes NaN for that centre instead of a wrong number. */
#define PT_ACSF_KIND_SHIFT 8
enum { PT_ACSF_GENERIC = 0,     /* any table */
       PT_ACSF_TANH_P4 = 1,     /* every angular group: tanh/tanhu cutoff, zeta in {1, 2, 4} */
       PT_ACSF_TANH_Z1N2 = 2,   /* every angular group: tanh/tanhu cutoff, zeta = 1, <= 2 terms */
       PT_ACSF_TANH_Z14 = 3 };  /* every angular group: tanh/tanhu cutoff, exactly the four terms
                                   zeta {1, 4} x lambda {+1, -1} */

/* Arithmetic of the MLP kernels (matrix cores). */
enum {
    PT_MLP_F64 = 0,    /* v_mfma_f64_16x16x4_f64 */
    PT_MLP_BF16 = 1,   /* v_mfma_f32_16x16x32_bf16, one product */
    PT_MLP_BF16X3 = 2  /* split bf16 (hi*hi + hi*lo + lo*hi), FP32 accumulate */
};

/* Cutoff function codes (n2p2 numbering, potentials/nnp/settings.py:43-51). */
enum { PT_CUT_HARD = 0, PT_CUT_COS = 1, PT_CUT_TANHU = 2, PT_CUT_TANH = 3,
       PT_CUT_EXP = 4, PT_CUT_POLY1 = 5, PT_CUT_POLY2 = 6 };

/* MLP activation codes (models/nn/activation.py:48-60). */
enum { PT_ACT_IDENTITY = 0, PT_ACT_TANH = 1, PT_ACT_LOGISTIC = 2, PT_ACT_SOFTPLUS = 3,
       PT_ACT_RELU = 4, PT_ACT_GAUSSIAN = 5, PT_ACT_COS = 6, PT_ACT_EXP = 7,
       PT_ACT_HARMONIC = 8 };

/* Scaler kinds (descriptors/scaler.py:206-246). */
enum { PT_SCALE_CENTER = 0, PT_SCALE_SCALE = 1, PT_SCALE_SCALE_CENTER = 2,
       PT_SCALE_SCALE_CENTER_SIGMA = 3 };

const char *pt_last_error(void);
int pt_version(void);

/* ------------------------------------------------------------------------
 * Symmetry-function table of one ACSF descriptor (descriptors/acsf/acsf.py:
 * 43-45), compiled on the host into groups that share their neighbour loop.
 *  - radial group: functions of one neighbour type and one cutoff;
 *    G1 is G2 with eta = 0, r_shift = 0 (radial.py:38-61).
 *  - angular group: functions of one unordered neighbour-type pair, one
 *    cutoff and one kind (G3/G9); each function is a cell (eta e, angular
 *    term a) of an n_eta x n_ang grid; col[e*4+a] = output column or -1.
 * The table lives in device memory (one upload per descriptor).
 * ---------------------------------------------------------------------- */
#define PT_RG_MAX 8
#define PT_AG_ETA 4
#define PT_AG_ANG 4
#define PT_MAX_GROUPS 24

typedef struct {
    int elem;   /* neighbour atom type, 1-based */
    int cut;    /* PT_CUT_* */
    int n;      /* functions in the group (<= PT_RG_MAX) */
    int pad_;
    double rc;
    double eta[PT_RG_MAX];
    double rs[PT_RG_MAX];
    int col[PT_RG_MAX];
} pt_radial_group;

typedef struct {
    int ej, ek;   /* neighbour atom types, 1-based, ej <= ek */
    int cut;      /* PT_CUT_* */
    int kind;     /* 3 = G3, 9 = G9 (angular.py:50-107) */
    int n_eta, n_ang;
    double rc;
    double half;  /* 0.5 when ej == ek (acsf.py:285-290), else 1 */
    double eta[PT_AG_ETA];
    double zeta[PT_AG_ANG];
    double lam[PT_AG_ANG];
    double pre[PT_AG_ANG];    /* 2^(1 - zeta) */
    int izeta[PT_AG_ANG];     /* zeta as a small integer (0..16) or -1 */
    int col[PT_AG_ETA * PT_AG_ANG];
} pt_angular_group;

typedef struct {
    int n_sf;
    int n_rg, n_ag;
    int pad_;
    double rc_max;
    double tanh_pre; /* ((e + 1/e) / (e - 1/e))^3, cutoff.py:82 */
    pt_radial_group rg[PT_MAX_GROUPS];
    pt_angular_group ag[PT_MAX_GROUPS];
} pt_sf_table;

/* ------------------------------------------------------------------------
 * (a) Neighbour list.  Replaces the dense cutoff masks of
 * atoms/neighbor.py:47-64,102-107 (mask (r <= rc) & (r > 0) over the
 * minimum-image distances of atoms/distance.py:63-78).
 * Atoms are sorted stably by (type, cell), then a CSR list is built whose rows
 * hold internal neighbour indices in ascending order.
 *  pos      (device) n rows of pos_stride (>= 3) FP64, x y z first, input
 *           order (pos_stride 4 lets a previous pos4 be the input);
 *           types (device) n, 1-based
 *  box      (host) 3 box lengths, or NULL for a non-periodic structure
 *  perm     (device, out) n: internal -> input index
 *  pos4     (device, out) n x 4 FP64: x, y, z, type (internal order)
 *  row_off  (device, out) n + 1
 *  nbr      (device, out) cap; rev (device, out, optional) cap: index of the
 *           reverse edge j->i for every edge i->j
 *  n_pairs, max_row (host, out)
 * Returns PT_ERR_CAPACITY (with *n_pairs set) when cap is too small.
 * ---------------------------------------------------------------------- */
size_t pt_nbr_workspace_bytes(int n, int n_types);
int pt_nbr_build(int n, const double *pos, int pos_stride, const int *types, int n_types,
                 const double *box, double rc,
                 int *perm, double *pos4, long long *row_off, int *nbr, int *rev,
                 long long cap, long long *n_pairs, int *max_row,
                 void *ws, size_t ws_bytes, pt_stream_t stream);

/* The same build for an MD step that never waits on the host (periodic
 * boxes only); no counterpart in the reference, which has no neighbour list.
 * Differences from pt_nbr_build:
 *  - gate (device, optional): when *gate == 0 every kernel of the build
 *    returns at once and perm, pos4, row_off, nbr and rev keep their
 *    contents (pt_skin_check sets the gate from the skin criterion);
 *  - nothing is read back: totals (device, 4 x int64, cleared by the caller)
 *    get [0] the pair count of the last build, [1] the longest row and [2]
 *    the largest pair count since they were cleared, [3] += 1 per build.
 *    [2] > cap means a build overflowed the arrays (the list is then
 *    incomplete); the caller checks [1] against the max_row it passes to the
 *    descriptor kernels (a longer row turns that centre's outputs into NaN);
 *  - rows longer than 256 entries take a second pass, decided on the device;
 *    it is enqueued only when row_limit (the longest row the caller's kernels
 *    read, i.e. the max_row it passes them) exceeds 256: a list with a row
 *    over row_limit is unusable either way, and totals[1] reports it.
 * No synchronisation and no host read: every launch is enqueued whatever the
 * data, so the sequence can be replayed or captured.
 * A list that does not fit (more pairs than cap, or a row over 256 entries
 * without the second pass) is not written, while row_off holds the offsets it
 * would have: read the totals before the rows.  pt_nbr_build_async_or_empty
 * is for callers whose kernels walk the list before the totals are known (the
 * MD step): the rows of such a list are all empty (row_off holds zeros). */
int pt_nbr_build_async(int n, const double *pos, int pos_stride, const int *types, int n_types,
                       const double *box, double rc, int *perm, double *pos4, long long *row_off,
                       int *nbr, int *rev, long long cap, const int *gate, long long *totals,
                       int row_limit, void *ws, size_t ws_bytes, pt_stream_t stream);
int pt_nbr_build_async_or_empty(int n, const double *pos, int pos_stride, const int *types, int n_types,
                                const double *box, double rc, int *perm, double *pos4, long long *row_off,
                                int *nbr, int *rev, long long cap, const int *gate, long long *totals,
                                int row_limit, void *ws, size_t ws_bytes, pt_stream_t stream);

/* Mark the closed neighbourhoods of n_sel atoms: flags[s] = 1 and
 * flags[j] = 1 for every j in the row of s (flags: device, n entries, not
 * cleared here).  Used to evaluate a potential on the centres whose
 * descriptors a few atoms' full forces depend on (the sampled judge of the
 * surrogate MD driver); no counterpart in the reference. */
int pt_nbr_mark_rows(int n_sel, const int *sel, const long long *row_off, const int *nbr,
                     unsigned char *flags, pt_stream_t stream);

/* Table class of a host-side table (host code, no device access). */
int pt_sf_table_kind(const pt_sf_table *host_table);

/* ------------------------------------------------------------------------
 * (b) ACSF forward: descriptor rows of the centres
 *     centers[c] (or center_begin + c when centers == NULL), internal order.
 * Replaces _calculate_acsf_descriptor (descriptors/acsf/acsf.py:163-213).
 *  G (device, out): n_centers x ldg, FP64 (PT_F64) or FP32 (PT_F32).
 *  max_row: the longest neighbour row (from pt_nbr_build); it sizes each
 *           centre's LDS staging, and a centre whose row is longer is
 *           written as NaN (for the adjoint: f_self and the row's edges).
 * ---------------------------------------------------------------------- */
int pt_acsf_forward(int precision, const double *pos4, const double *box,
                    const long long *row_off, const int *nbr, int max_row,
                    int n_centers, int center_begin, const int *centers,
                    const pt_sf_table *table, void *G, int ldg, pt_stream_t stream);

/* ------------------------------------------------------------------------
 * (b') ACSF adjoint.  With w = dE/dG (n_centers x ldw, same precision),
 * writes per centre i
 *   f_self[i]         = -sum_s w_is dG_is/dr_i     (potentials/nnp/force.py:
 *                       16-43: the reference's gradient w.r.t. the central
 *                       positions, neighbours frozen)
 *   edge_grad[e(i,j)] =  sum_s w_is dG_is/dr_j     (all j in row i)
 * f_self is FP64 (device, n_centers x 3, optional).  edge_grad is FP64 for
 * PT_F64 and FP32 for PT_F32 (device, n_pairs x 3, optional); entries of
 * row i beyond the descriptor cutoff are written as zero.
 * ---------------------------------------------------------------------- */
int pt_acsf_adjoint(int precision, const double *pos4, const double *box,
                    const long long *row_off, const int *nbr, int max_row,
                    int n_centers, int center_begin, const int *centers,
                    const pt_sf_table *table, const void *w, int ldw,
                    double *f_self, void *edge_grad, pt_stream_t stream);

/* The adjoint with a transposed edge buffer: edge e(i,j)'s gradient
 * sum_s w_is dG_is/dr_j goes to the slot of the reverse edge, rev[e]
 * (device, from pt_nbr_build), so that edge_grad_t[e(j,i)] = dE_i/dr_j and
 * row j of the buffer holds everything atom j receives.  Every slot whose
 * reverse edge belongs to a launched centre is written (zero beyond the
 * cutoff); f_self as in pt_acsf_adjoint.  Same forces as pt_acsf_adjoint +
 * pt_force_gather, read contiguously by pt_force_gather_transposed; no
 * counterpart in the reference (force.py:16-43 is autodiff). */
int pt_acsf_adjoint_transposed(int precision, const double *pos4, const double *box,
                               const long long *row_off, const int *nbr, const int *rev, int max_row,
                               int n_centers, int center_begin, const int *centers,
                               const pt_sf_table *table, const void *w, int ldw,
                               double *f_self, void *edge_grad_t, pt_stream_t stream);

/* Full forces F = -grad E by a scatter-free gather over the edge buffer:
 *   F[i] = sum_{e in row i} (edge_grad[e] - edge_grad[rev[e]]).
 * (FP64 accumulation; edge_precision PT_F64 or PT_F32.)  Replaces the
 * autodiff of potentials/nnp/force.py:16-43 for the -grad E force mode. */
int pt_force_gather(int n, const long long *row_off, const int *rev,
                    const void *edge_grad, int edge_precision, double *f_full,
                    pt_stream_t stream);
/* F[i] = f_self[i] - sum_{e in row i} edge_grad_t[e] over the transposed
 * buffer of pt_acsf_adjoint_transposed (f_self: device, n x 3 FP64, the
 * adjoint's own output): one contiguous read per row. */
int pt_force_gather_transposed(int n, const long long *row_off, const double *f_self,
                               const void *edge_grad_t, int edge_precision, double *f_full,
                               pt_stream_t stream);

/* ------------------------------------------------------------------------
 * Descriptor tangent: T[c, s] = sum_m dG_{i,s}/dr_m . delta[m] for centre
 * i = centers[c].  With center_only != 0 only the centre's own delta
 * contributes (delta of neighbours taken as 0); with delta = unit vector
 * this is one column of the self-Jacobian of descriptors/acsf/acsf.py:
 * 88-120,215-228 (ACSF.grad).  delta: (device) n x 3 FP64, internal order.
 * ---------------------------------------------------------------------- */
int pt_acsf_tangent(int precision, const double *pos4, const double *box,
                    const long long *row_off, const int *nbr, int max_row,
                    int n_centers, int center_begin, const int *centers,
                    const pt_sf_table *table, const double *delta, int center_only,
                    void *T, int ldt, pt_stream_t stream);

/* ------------------------------------------------------------------------
 * Several tables (or tangent directions) in one launch.  A run is a set of
 * centres that share a table: n_centers centres center_begin, ... or
 * centers[] (device), kind = pt_sf_table_kind of the table, its rows of out
 * (G or T), w and f_self (as in the single-table calls; unused members may be
 * NULL).  delta == NULL in a center_only tangent means the unit vector of
 * direction dir (0, 1, 2).  boxes (device, 3 lengths per structure; 0: not
 * periodic) with box_id (device, a structure index per atom) replaces box for
 * lists that hold several structures.  rev == NULL: edge_grad in the edges'
 * own slots (pt_acsf_adjoint), else transposed (pt_acsf_adjoint_transposed).
 * ---------------------------------------------------------------------- */
typedef struct {
    const pt_sf_table *table;
    int kind;
    int n_centers;
    int center_begin;
    int dir;
    const int *centers;
    void *out;
    const void *w;
    double *f_self;
    const double *delta;
} pt_acsf_run;
int pt_acsf_forward_multi(int precision, const double *pos4, const double *box, const long long *row_off,
                          const int *nbr, int max_row, int n_runs, const pt_acsf_run *runs, int ldg,
                          pt_stream_t stream);
int pt_acsf_adjoint_multi(int precision, const double *pos4, const double *box, const double *boxes,
                          const int *box_id, const long long *row_off, const int *nbr, const int *rev, int max_row,
                          int n_runs, const pt_acsf_run *runs, int ldw, void *edge_grad, pt_stream_t stream);
int pt_acsf_tangent_multi(int precision, const double *pos4, const double *box, const double *boxes,
                          const int *box_id, const long long *row_off, const int *nbr, int max_row, int n_runs,
                          const pt_acsf_run *runs, int center_only, int ldt, pt_stream_t stream);

/* ------------------------------------------------------------------------
 * (c) Atomic MLP of one element on matrix cores: scaler + dense layers +
 * output, and the input gradient.  Replaces _compute_energy_per_atom
 * (potentials/nnp/energy.py:23-39) = scaler (descriptors/scaler.py:206-246)
 * + NeuralNetworkModel (models/nn/model.py:24-58), and its reverse-mode
 * gradient w.r.t. the descriptor.
 *  G      (device) n_atoms x ldg, FP64 or FP32 (g_precision)
 *  scale  (device) 2 x in_dim FP64: x' = (x - scale[0,k]) * scale[1,k] + add
 *         (every scaler kind of scaler.py:206-246 is such an affine map)
 *  packed (device) from pt_mlp_pack
 *  e_atom (device, out) n_atoms FP64 (model output, per atom)
 *  dEdG   (device, out, optional) n_atoms x ldg in g_precision
 * ---------------------------------------------------------------------- */
typedef struct {
    int n_layers;      /* hidden layers + the output layer (<= 4) */
    int in_dim;        /* descriptor width (<= 128) */
    int width[4];      /* outputs per layer; the last is 1; hidden <= 128 */
    int act[4];        /* PT_ACT_* per layer */
    double scale_add;  /* scaler offset: smin for the min-max kinds, else 0 */
} pt_mlp_desc;

/* Packed weights: FP64 W/b plus bf16 hi/lo copies in both W and W^T
 * layouts, padded to multiples of 32.  params (device, FP64) holds per layer
 * W (fan_in x fan_out, row-major, the flax kernel layout of model.py:28-38)
 * then b (fan_out). */
size_t pt_mlp_packed_bytes(const pt_mlp_desc *desc);
int pt_mlp_pack(const pt_mlp_desc *desc, const double *params, void *packed,
                pt_stream_t stream);

int pt_mlp_energy_grad(int mode, int n_atoms, const void *G, int ldg, int g_precision,
                       const double *scale, const pt_mlp_desc *desc, const void *packed,
                       double *e_atom, void *dEdG, pt_stream_t stream);

/* Several elements' networks in one launch: every job is one call of
 * pt_mlp_energy_grad (its n_atoms, G, scale, desc, packed, e_atom, dEdG) at
 * the common mode, ldg and g_precision. */
typedef struct {
    int n_atoms;
    const void *G;
    const double *scale;
    const pt_mlp_desc *desc;
    const void *packed;
    double *e_atom;
    void *dEdG;
} pt_mlp_job;
int pt_mlp_energy_grad_multi(int mode, int n_jobs, const pt_mlp_job *jobs, int ldg, int g_precision,
                             pt_stream_t stream);

/* ------------------------------------------------------------------------
 * (c') Training of an atomic MLP (the student surrogate).  No counterpart in
 * the reference runs (its trainer, potentials/nnp/gradient_descent.py:
 * 157-233, is broken); the loss is the energy MSE per atom plus a weighted
 * force MSE, w_E ((E - E*)/N)^2 + w_F / (3N) sum |F - F*|^2 per structure.
 * pt_mlp_train_grad accumulates into grad (FP64, layout of the unpacked
 * params) the gradient  sum_i gy[i] dy_i/dtheta + tseed d(ydot_i)/dtheta,
 * y = MLP(scaled G), ydot = grad_G y . T (T: descriptor tangent).  With
 * gy = dL/dE and T = J delta, delta = dL/dF, tseed = -1, this is dL/dtheta.
 * ---------------------------------------------------------------------- */
size_t pt_mlp_param_count(const pt_mlp_desc *desc);
int pt_mlp_train_grad(int mode, int n_atoms, const void *G, const void *T, int ldg,
                      int g_precision, const double *scale, const pt_mlp_desc *desc,
                      const void *packed, const double *gy, double tseed, double *grad,
                      pt_stream_t stream);
/* Several elements' networks in one launch, for the weight gradient and for
 * the per-row Jacobian below: every job is one call of pt_mlp_train_grad (out:
 * grad) or pt_mlp_jacobian (out: J; gy unused). */
typedef struct {
    int n_atoms;
    const void *G;
    const void *T;
    const double *scale;
    const pt_mlp_desc *desc;
    const void *packed;
    const double *gy;
    double *out;
} pt_mlp_train_job;
int pt_mlp_train_grad_multi(int mode, int n_jobs, const pt_mlp_train_job *jobs, int ldg, int g_precision,
                            double tseed, pt_stream_t stream);
int pt_mlp_jacobian_multi(int n_dir, int n_jobs, const pt_mlp_train_job *jobs, long long t_dir, int ldg, double sign,
                          long long ldj, pt_stream_t stream);
/* delta = w_F 2 (F - F*) / (3N), gy = w_E 2 (E - E*) / N^2 (per atom), and
 * loss[0] += w_E ((E - E*)/N)^2, loss[1] += w_F / (3N) sum |F - F*|^2.
 * energy: device scalar. */
int pt_train_seeds(int n, const double *force, const double *force_ref, const double *energy,
                   double energy_ref, double w_energy, double w_force, double *delta, double *gy,
                   double *loss, pt_stream_t stream);
/* A batch of labelled structures as one list, so that every step of the loss
 * gradient is one launch.  Segment q = e * n_struct + k of the batch holds the
 * atoms of element e of structure k.  plan (device, pt_train_batch_words 64-bit
 * words): per structure the device addresses of pos4, row_off, nbr, rev, the
 * descriptors G (n x ld) and the labels F* (n x 3), then E* (FP64 bits), the
 * three box lengths (FP64 bits; 0: not periodic) and the atom count; per
 * (structure, element) the element block's first atom (past the last atom if
 * the structure has none) and row_off there; the first batch atom and the first
 * batch edge of every segment, each closed by the total.  Every atom belongs to
 * an element block.
 * pt_train_batch_assemble copies the lists into pos4 .. boxes (n_atoms + 1
 * row offsets, n_struct x 3 box lengths, a structure index per atom: the box
 * table of pt_acsf_*_multi).  pt_train_batch_seeds: from f_self and the
 * transposed edge gradients of the batch and e_atom, per structure delta, gy
 * and the loss sums of pt_train_seeds (sq: n_atoms doubles of workspace). */
int pt_train_batch_words(int n_struct, int n_elem);
int pt_train_batch_assemble(int n_struct, int n_elem, const long long *plan, int n_atoms, int ld, int g_precision,
                            double *pos4, long long *row_off, int *nbr, int *rev, void *G, double *f_ref,
                            int *box_id, double *boxes, pt_stream_t stream);
int pt_train_batch_seeds(int n_struct, int n_elem, const long long *plan, int n_atoms, const long long *row_off,
                         const double *f_self, const void *edge_grad_t, int edge_precision, const int *box_id,
                         const double *f_ref, const double *e_atom, double w_energy, double w_force, double *delta,
                         double *gy, double *sq, double *loss, pt_stream_t stream);
/* Adam (decoupled weight decay when weight_decay > 0), step counts from 1;
 * optax.adamw semantics (gradient_descent.py:70-76). */
int pt_adam_step(int n, double *params, const double *grad, double *m, double *v, double lr,
                 double beta1, double beta2, double eps, double weight_decay, int step,
                 pt_stream_t stream);

/* ------------------------------------------------------------------------
 * (f) Global extended Kalman filter trainer
 * (potentials/nnp/kalman_filter.py:42-335).
 *
 * pt_mlp_jacobian: per-row Jacobian of the reference's self-term forces
 * (the jacrev of _compute_forces_error, kalman_filter.py:305-335).  Row
 * (atom a, direction d) of J (row-major, leading dimension ldj, columns in
 * the layout of the unpacked params) is
 *     sign * d/dtheta [ grad_x' y(x'_a) . (T_d[a] * mul) ],
 * with T_d the centre-only descriptor tangent along axis d (pt_acsf_tangent
 * with center_only and delta = e_d): sign = -1 gives dF_self[a, d]/dtheta.
 * G: (device) n_atoms x ldg FP64; T: n_dir blocks of n_atoms x ldg FP64,
 * t_dir doubles apart; J: (device, out) n_atoms * n_dir rows; only the
 * columns of this element's parameters are written.  FP64 only.
 * ---------------------------------------------------------------------- */
int pt_mlp_jacobian(int n_atoms, int n_dir, const double *G, const double *T, long long t_dir, int ldg,
                    const double *scale, const pt_mlp_desc *desc, const void *packed, double sign,
                    double *J, long long ldj, pt_stream_t stream);
/* xi[i] = (ref[i] - pred[i]) * scale (ref == NULL: ref_scalar for every i) and
 * loss[0] += sum_i xi[i]^2: the energy and force errors of
 * kalman_filter.py:276-303 and the loss of :243, :268. */
int pt_kalman_residual(int n, const double *pred, const double *ref, double ref_scalar, double scale,
                       double *xi, double *loss, pt_stream_t stream);
/* One update of KalmanFilter.update_state_vector (kalman_filter.py:196-233)
 * with the schedules applied by the caller:
 *   X = P H, A = H^T X + r I, K = X A^-1, P <- c (P - K X^T) + q I, W <- W + K xi
 * r = 1/eta (type 0) or lambda (type 1), c = 1 (type 0) or 1/lambda (type 1).
 * P: (device, in/out) n_w x n_w FP64; H: (device) m columns of n_w (leading
 * dimension ldh), column o = gradient of observation o; xi: m; W: n_w.
 * A is factorised by Cholesky (blocked) instead of being
 * inverted; with m > n_w the same update is computed from the n_w x n_w
 * factors of P and of S = G G^T + r I, G = L^T H (push-through identity:
 * P - K X^T = r L S^-1 L^T).  info (device int) receives the first nonzero
 * dpotrf status (0 = success).
 * ws: pt_kalman_workspace_bytes(n_w, m) bytes of device memory. */
size_t pt_kalman_workspace_bytes(int n_w, int m);
int pt_kalman_update(int n_w, int m, double *P, const double *H, long long ldh, const double *xi,
                     double *W, double r, double c, double q, void *ws, size_t ws_bytes, int *info,
                     pt_stream_t stream);

/* ------------------------------------------------------------------------
 * Scaler statistics and extrapolation counter on the device
 * (descriptors/scaler.py:84-142, 249-295).  params (device) holds 4 x n_cols
 * FP64: mean | sigma | minval | maxval (the ScalerParams fields).  G: n_rows
 * descriptor rows, leading dimension ldg, FP64 or FP32 (g_precision).
 * ---------------------------------------------------------------------- */
size_t pt_scaler_workspace_bytes(int n_rows, int n_cols);
/* nsamples == 0: params = the statistics of G (_fit, scaler.py:249-259:
 * mean, population std, min, max).  nsamples > 0: params (the statistics of
 * nsamples earlier rows) are merged with those of G as _partial_fit does
 * (scaler.py:262-283).  Deterministic (fixed reduction order). */
int pt_scaler_partial_fit(int n_rows, int n_cols, const void *G, int ldg, int g_precision,
                          double nsamples, double *params, void *ws, size_t ws_bytes, pt_stream_t stream);
/* Extrapolation count (_calculate_number_of_warnings, scaler.py:286-295,
 * which reports whether any value lies outside [minval, maxval]): a value
 * outside [minval - margin w, maxval + margin w], w = maxval - minval, or
 * NaN, is out of range (margin 0: the reference's test).  Accumulates into
 * counters (device, 3 x uint64, cleared by the caller):
 *   [0] += rows with an out-of-range value, [1] += out-of-range values,
 *   [2] = max([2], bit pattern of the largest excess in units of w).
 * No synchronisation: the counters can be read whenever the caller syncs. */
int pt_scaler_extrapolation(int n_rows, int n_cols, const void *G, int ldg, int g_precision,
                            const double *params, double margin, unsigned long long *counters,
                            pt_stream_t stream);

/* ------------------------------------------------------------------------
 * (d) Reductions and the velocity-Verlet step (FP64).
 * ---------------------------------------------------------------------- */
size_t pt_reduce_workspace_bytes(int n);
/* out[0] = sum x[i] in a fixed order (deterministic).  Replaces the sums of
 * potentials/nnp/energy.py:54-63. */
int pt_reduce_sum_f64(int n, const double *x, double *out, void *ws, size_t ws_bytes,
                      pt_stream_t stream);
/* The same sum without a workspace and without any allocation: for callers
 * that cannot allocate device memory (code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc).  It has no counterpart in
 * the reference.  The partial sums live in a 512 KiB device array of the
 * library, one copy per GPU, held until the process ends; n is limited to
 * 2^26 = 67,108,864 elements (PT_ERR_ARG beyond, nothing launched).  The
 * stream must belong to the current device.  Calls that overlap on one GPU
 * (several streams or threads) share that array and race.  Results are
 * bitwise those of pt_reduce_sum_f64 (same kernels, same order). */
int pt_reduce_sum_f64_noalloc(int n, const double *x, double *out, pt_stream_t stream);

/* x <- wrap(x + v dt + 1/2 a dt^2), a = F (inv_mass == NULL, the reference
 * integrator of simulation/molecular_dynamics.py:16-20,65-72) or F/m.
 * pos4 is updated in place (type column untouched); wrap = jnp.remainder
 * (atoms/box.py:123-126) when box != NULL (host, 3 lengths). */
int pt_verlet_positions(int n, double *pos4, const double *vel, const double *force,
                        const double *inv_mass, double dt, const double *box,
                        pt_stream_t stream);
/* pos (n x 3, device) <- jnp.remainder(pos, box) (atoms/box.py:123-126,
 * applied by atoms/structure.py:80-81 when a structure is created). */
int pt_wrap_positions(int n, double *pos, const double *box, pt_stream_t stream);
/* v <- v + 1/2 (a_old + a_new) dt (molecular_dynamics.py:23-30,73-76). */
int pt_verlet_velocities(int n, double *vel, const double *f_old, const double *f_new,
                         const double *inv_mass, double dt, pt_stream_t stream);
/* out[0] = 1/2 sum m v^2 (simulation/system.py:20-22), deterministic. */
int pt_kinetic_energy(int n, const double *vel, const double *mass, double *out,
                      void *ws, size_t ws_bytes, pt_stream_t stream);
/* Berendsen rescale v *= 1/sqrt(1 + dt/tau (T/T0 - 1)), T from ke[0]
 * (simulation/thermostat.py:12-22, system.py:25-29). */
int pt_berendsen_rescale(int n, double *vel, const double *ke, double dt, double tau,
                         double t0, double kb, pt_stream_t stream);

/* out[0], out[1] = the largest and the second largest |MIC(pos4_i - ref_i)|
 * over the atoms (device scalars; out holds 514 doubles, out[2..513] are
 * scratch).  A skin list stays exact while out[0] + out[1] <= skin: no pair
 * has moved by more than the sum of its two displacements.  Drives the
 * rebuild of skin neighbour lists (no counterpart in the reference, which
 * has no neighbour list). */
int pt_max_displacement(int n, const double *pos4, const double *ref, const double *box,
                        double *out, pt_stream_t stream);

/* *flag (device int) = 1 when a skin list built at ref must be rebuilt at
 * pos4: the two largest |MIC(pos4_i - ref_i)| sum to more than skin (or skin
 * <= 0, or a displacement is NaN), else 0.  scratch (device): 514 doubles,
 * as the out array of pt_max_displacement.  No host read. */
int pt_skin_check(int n, const double *pos4, const double *ref, const double *box, double skin,
                  double *scratch, int *flag, pt_stream_t stream);
/* The work of an MD step around its rebuild and forces in three calls, with
 * the results of the separate calls above bit for bit:
 * pt_md_positions: pt_verlet_positions, the new pos4 also to pos_out (n x 4);
 * ref != NULL (n x 4): *flag as pt_skin_check(pos4, ref, box, skin, scratch).
 * pt_md_velocities: unless gate (device, optional) holds 0, the new state of
 * atom i follows from the old one of atom perm[i] (the order of a gated
 * rebuild; f_old is in the old order, f_new in the new one), else from that
 * of atom i: velocities as pt_verlet_velocities (with_mass: a = F / m), the
 * rest moved.  in and out share no array.  ref_pos (optional): takes pos4
 * under the same gate.  ke_part (optional): ceil(n / 1024) partial sums of
 * the kinetic energy, as pt_reduce_workspace_bytes(n) holds.
 * pt_md_berendsen: pt_berendsen_rescale from those partial sums. */
typedef struct {
    double *vel;       /* (device) n x 3 */
    double *mass, *inv_mass;
    int *orig, *types;
} pt_md_state;
int pt_md_positions(int n, double *pos4, const double *vel, const double *force, const double *inv_mass,
                    double dt, const double *box, double *pos_out, const double *ref, double skin,
                    double *scratch, int *flag, pt_stream_t stream);
int pt_md_velocities(int n, const int *gate, const int *perm, const pt_md_state *in, const pt_md_state *out,
                     const double *f_old, const double *f_new, int with_mass, double dt, const double *pos4,
                     double *ref_pos, double *ke_part, pt_stream_t stream);
int pt_md_berendsen(int n, double *vel, const double *ke_part, double dt, double tau, double t0, double kb,
                    pt_stream_t stream);
/* The state of atom i from input-order arrays: atom perm[i]'s velocity, mass,
 * 1 / mass, perm[i] itself and type. */
int pt_md_start(int n, const int *perm, const double *vel, const double *mass, const int *types,
                const pt_md_state *out, pt_stream_t stream);
/* inv[perm[i]] = i: the internal index of each input atom. */
int pt_invert_perm(int n, const int *perm, int *inv, pt_stream_t stream);
/* Up to PT_COPY_MAX copies (device, a multiple of 4 bytes each, ranges that do
 * not overlap) in one launch. */
#define PT_COPY_MAX 8
typedef struct {
    const void *src;
    void *dst;
    long long bytes;
} pt_copy_array;
int pt_copy_arrays(int n, const pt_copy_array *arrays, pt_stream_t stream);
/* dst[idx[i]] (n x 3) = the first three of row i of src (rows src_stride apart). */
int pt_scatter_rows3_f64(int n, const int *idx, const double *src, int src_stride, double *dst,
                         pt_stream_t stream);
/* dst <- src (n_words words of word_bytes = 4 or 8), unless gate (device,
 * optional) holds 0. */
int pt_copy_gated(long long n_words, int word_bytes, const void *src, void *dst, const int *gate,
                  pt_stream_t stream);
/* In place, unless gate (device, optional) holds 0: row i of buf (width
 * words of word_bytes = 4 or 8) <- old row perm[i], through tmp (same size).
 * Moves the MD state into the order of a gated rebuild. */
int pt_permute_rows_gated(int n, int width, int word_bytes, const int *perm, void *buf, void *tmp,
                          const int *gate, pt_stream_t stream);
/* The same for up to PT_PERMUTE_MAX arrays in two launches (gather of every
 * array into tmp, then copy back): tmp holds n * sum(width * word_bytes)
 * bytes (pt_permute_state_tmp_bytes). */
#define PT_PERMUTE_MAX 8
typedef struct {
    void *buf;       /* (device) n rows of width words */
    int width;
    int word_bytes;  /* 4 or 8 */
} pt_permute_array;
size_t pt_permute_state_tmp_bytes(int n, int n_arrays, const pt_permute_array *arrays);
int pt_permute_state_gated(int n, const int *perm, int n_arrays, const pt_permute_array *arrays, void *tmp,
                           size_t tmp_bytes, const int *gate, pt_stream_t stream);

/* Row gathers/scatters between input order and internal order. */
int pt_gather_rows_f64(int n, int width, const int *idx, const double *src, double *dst,
                       pt_stream_t stream); /* dst[i] = src[idx[i]] */
int pt_scatter_rows_f64(int n, int width, const int *idx, const double *src, double *dst,
                        pt_stream_t stream); /* dst[idx[i]] = src[i] */
int pt_gather_rows_i32(int n, int width, const int *idx, const int *src, int *dst,
                       pt_stream_t stream);

#ifdef __cplusplus
}
#endif

#endif /* PANTEA_HIP_H */
