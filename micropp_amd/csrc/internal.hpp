// internal.hpp -- device-side data layout of micropp_amd and the launchers
// shared by the .hip translation units.
//
// ELL on the device (SELL-64): rows are grouped into slices of 64 (one
// wavefront); inside a slice the 81 slots are slot-major, so slot s of the 64
// rows of slice q sits at [(q * 81 + s) * 64 + lane].  One wavefront streams
// a slice with 81 fully coalesced 512-byte loads of values and 256-byte loads
// of columns.  Row and slot numbering are the reference's (row = node*3 + fi,
// slot = nb*3 + fj, nb = (dz+1)*9 + (dy+1)*3 + (dx+1)); rows are padded to a
// multiple of 256 with zero values and column 0.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <string>
#include <utility>
#include <vector>

#include "material_base.h"
#include "mppd.h"

namespace mpp {

constexpr int kSlots = 81;
constexpr int kBlock = 256;     // threads per block of the row-space kernels
constexpr int kRowPad = 256;    // row padding (a block of rows)
constexpr int kMaxSpheres = 64; // MIC3D_RANDOM_SPHERES list length
constexpr int kNumMicroTypes = 14;     // MIC_HOMOGENEOUS .. MIC3D_RANDOM_SPHERES
constexpr int kMicRandomSpheres = 13;  // MIC3D_RANDOM_SPHERES

// Geometry passed by value to kernels.
struct Grid {
  int nx, ny, nz;
  int nex, ney, nez;
  int nn, nrow, nrow_pad, nelem;
  double dx, dy, dz, wg, vol_tot, evol;
};

// Jacobi-PCG scalars of one system (device resident).
struct CgState {
  double rz, pn0, pn, beta, min_err, rel_err;
  int its, max_its, done;
  int fresh;  // the scalars hold the sums of the last iteration queued (kernels.hpp)
};

// Status of an averaging / norm reduction.
struct RedState {
  double v[8];
  int flag;
};

size_t round_up(size_t v, size_t m);
void set_error(const std::string &msg);
int fail(int code, const std::string &msg);
int hip_fail(hipError_t e, const char *what);

#define MPP_HIP(call)                                  \
  do {                                                 \
    hipError_t _e = (call);                            \
    if (_e != hipSuccess) return mpp::hip_fail(_e, #call); \
  } while (0)

// Device allocation of n elements, zero-filled unless asked otherwise.
template <typename T>
inline int dalloc(T **p, size_t n, bool zero = true) {
  *p = nullptr;
  if (n == 0) n = 1;
  hipError_t e = hipMalloc((void **)p, n * sizeof(T));
  if (e != hipSuccess) return hip_fail(e, "hipMalloc");
  if (zero) {
    e = hipMemset(*p, 0, n * sizeof(T));
    // hipMemset runs on the null stream, which the solvers' non-blocking
    // streams do not order against: finish it before the buffer is used
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) return hip_fail(e, "hipMemset");
  }
  return MPPD_OK;
}

// The device buffers of an object as one allocation with 256-byte aligned
// parts: hipMalloc and hipFree cost 20 to 700 us each, a set of one or two
// dozen buffers several milliseconds.  add() every part, then alloc().
class Arena {
 public:
  template <typename T>
  void add(T **p, size_t n) {
    parts_.push_back({reinterpret_cast<void **>(p), size_});
    size_ += (std::max<size_t>(n, 1) * sizeof(T) + 255) & ~(size_t)255;
  }
  size_t size() const { return size_; }
  // *base owns the parts
  int alloc(void **base) {
    *base = nullptr;
    const hipError_t e = hipMalloc(base, size_);
    if (e != hipSuccess) return hip_fail(e, "hipMalloc");
    for (auto &p : parts_) *p.first = static_cast<char *>(*base) + p.second;
    return MPPD_OK;
  }

 private:
  size_t size_ = 0;
  std::vector<std::pair<void **, size_t>> parts_;
};

// Device allocation of n elements, zero-filled on stream st: the fill is
// ordered before st's later work, and the caller synchronizes st before the
// buffer is used from another stream or by a blocking copy.
template <typename T>
inline int dalloc(T **p, size_t n, hipStream_t st) {
  *p = nullptr;
  if (n == 0) n = 1;
  hipError_t e = hipMalloc((void **)p, n * sizeof(T));
  if (e != hipSuccess) return hip_fail(e, "hipMalloc");
  e = hipMemsetAsync(*p, 0, n * sizeof(T), st);
  return e == hipSuccess ? MPPD_OK : hip_fail(e, "hipMemsetAsync");
}

inline void dfree(void *p) {
  if (p) (void)hipFree(p);
}

// Test hook: with MPPD_FAIL_ALLOC=1 in the environment, the buffers an entry
// point makes on its first call (mppd_newton_mixed, mppd_msolver_adjoint) are
// freed again after they are allocated and the call fails with
// MPPD_ERR_NOMEM, as an out-of-memory failure would; a test then checks that
// the next call allocates afresh and gives the normal result.
inline bool alloc_fault_injected() {
  const char *v = std::getenv("MPPD_FAIL_ALLOC");
  return v && std::atoi(v) != 0;
}

// Two-level preconditioner of the multi-RHS inner CG (mixed.hip k_c_*): the
// Jacobi weights plus a Galerkin coarse space of trilinear hats on a coarse
// grid aligned with the fine one (h fine elements per coarse element and
// side).  Only interior coarse nodes carry unknowns (the boundary is
// Dirichlet); coarse DOF q * 3 + d of interior coarse node q = ((cz - 1) my +
// (cy - 1)) mx + (cx - 1).
struct CGrid {
  int hx, hy, hz;  // fine elements per coarse element
  int lx, ly, lz;  // = h where all are h wide; else some are l wide
  int tx, ty, tz;  // width of the last, where neither (= h otherwise)
  int mx, my, mz;  // interior coarse nodes per side
  int nq, nc;      // interior coarse nodes, coarse DOFs (3 nq)
  int even;        // sides (bit 0 x, 1 y, 2 z) whose coarse nodes have even fine indices
};

// fine index of coarse node q (0 .. d) along a side of ne elements
__host__ __device__ inline int coarse_node(int q, int ne, int d, int even) {
  if (!even) return q * ne / d;
  return q < d ? 2 * (q * ((ne + 1) / 2) / d) : ne;
}
// device buffers of the coarse level of one K-field system
struct CoarseDev {
  CGrid cg;
  const float *ainv;  // nc x nc: the inverse of the Galerkin coarse matrix (symmetric)
  float *t1;          // x-restricted residual: 3 K nz ny mx floats
  float *rc;          // restricted residual, nc x K
  float *ecp;         // split partials of the coarse solve, kCoarseSplit x nc x K
  float *ec;          // coarse correction, nc x K
  float *z;           // the preconditioned residual z, in R's layout
  double *prz;        // partials of (r, z) at the inner CG's start: 3 K x (vector blocks)
  void *arena;        // the one device allocation holding all of the above
};
constexpr int kCoarseSplit = 16;    // column splits of the coarse solve (one partial each)
constexpr int kCoarseMaxLine = 256;  // nodes per side a coarse level allows
constexpr int kCoarseMaxDofs = 2200;  // coarse DOFs of a multi-RHS solver (3 x 9^3 = 2187: 10^3 coarse elements)
constexpr double kHighContrast = 30.0;  // of the moduli: beyond it, coarse grids of the multilevel form made for it
constexpr int kCoarseMaxPos = 4096;   // positions of a fine element that the set-up's table holds at once (57 MB)
// Trilinear hats along one side at one fine index: the interior coarse nodes
// below and above it, as offsets into the coarse vectors, and their weights
// (0 for a node on the boundary, with a valid offset).
struct HatEntry {
  float w0, w1;
  int q0, q1;
};

// Multilevel (V-cycle) preconditioner of the multi-RHS inner CG on a stencil
// dictionary (vcycle.hip): Jacobi smoothing on the fine grid and on the grid of
// twice its spacing (its Galerkin operator stored as FP32 node blocks), and the
// dense inverse of a coarse Galerkin matrix.  Small RVEs have no second level
// (mid.nq = 0): their coarse grid is that fine itself.
struct VCycleDev {
  CGrid mid, cg;  // second level (h = 2), coarse grid
  // along x, y, z: the coarse hats at the nodes of the level above, and the
  // first node there beyond coarse node q (0 .. d - 1), and at or beyond it (1 .. d)
  const HatEntry *hat[3];
  const int *past[3], *upto[3];
  Grid g1;           // the second level as a grid: m + 2 nodes a side, the boundary among them
  const float *ainv;          // nc x nc
  float *rc, *ec;             // restricted residual and coarse correction (nc x K)
  float *A1, *kinv1;          // second level: node blocks (63 float4 a node, A1[quad * NP1 + node]) and Jacobi weights
  float *R1, *E0, *T1, *E;    // second level: residual, Jacobi part, smoothed residual, correction
  float *z;                   // fine work vector, in R's layout
  double *prz;                // partials of (r, z) at the inner CG's start: K x stencil_blocks
  float w0, w1;               // damping of the two Jacobi smoothers
  void *arena;
};
// MPPD_COARSE=0 in the environment turns the coarse levels off
bool coarse_enabled();
// the largest coarse grid aligned with g with at most max_dofs coarse DOFs
// (false: none)
bool coarse_grid(const Grid &g, int max_dofs, CGrid *out);
// the grid of twice the spacing (an odd side's last element 1 wide; false: a side of fewer than 4 elements)
bool coarse_grid_by_two(const Grid &g, CGrid *out);
// the coarse grid of the multilevel preconditioner of an RVE with this contrast: about 4 or 5 fine elements per coarse
// element and side; false: none
bool coarse_grid_cycle(const Grid &g, double contrast, CGrid *out);
// a coarse grid of elements of at least `least` fine ones a side, as narrow as max_dofs coarse DOFs allow: coarse node
// q of a side of ne elements and d = m + 1 coarse ones at fine index floor(q ne / d) (widths h and, where d does not
// divide the side, l = h + 1); false: none
bool coarse_grid_wide(const Grid &g, int least, int max_dofs, CGrid *out);
// the longest cell side over the shortest, and a coarse grid of elements of one length on every side (a side's own
// elements where those are longer), as short as max_dofs coarse DOFs allow; false: none
double cell_aspect(const Grid &g);
bool coarse_grid_long(const Grid &g, int max_dofs, CGrid *out);
// the coarse grid beside Jacobi: elements at least 2 wide, or of one length where the cells are long; false: none
bool coarse_grid_additive(const Grid &g, int max_dofs, CGrid *out);
// C (device, coarse_table_len(cg, nz) doubles) = the Galerkin contributions P_e^T Ke P_e per phase and position,
// for nz of the coarse_table_planes(cg) planes of positions from z0 on
// (positions of a side: those in an element h wide, in one l wide, in the last one)
int coarse_table_planes(const CGrid &cg);
size_t coarse_table_len(const CGrid &cg, int nz);
hipError_t launch_cs_table(const CGrid &cg, int z0, int nz, const double *ke, double *C, hipStream_t st);
// ainv (nc x nc floats, device) = the FP32 inverse of the Galerkin coarse
// matrix of the RVE (phase map et_d, per-phase element stiffness ke_d) on cg;
// *ok = false when that matrix is not positive definite
int coarse_inverse(const Grid &g, const CGrid &cg, const int *et_d, const double *ke_d, float *ainv, hipStream_t st,
                   bool *ok);
// coarse.hip: the coarse level of a K-field system on the RVE grid g (per-phase
// element stiffness ke_d, phase map et_d); *out = nullptr when the grid has
// none (or MPPD_COARSE=0 in the environment)
int coarse_setup(const Grid &g, const int *et_d, const double *ke_d, int K, hipStream_t st, CoarseDev **out);
void coarse_free(CoarseDev *c);

// Mixed-precision Newton (mppd_newton_mixed, batches with mixed_precision):
// the linear solve of the last Newton iteration nr_max_its permits stops at
// cg_rel_tol times this factor.  When the Newton ends there unconverged (the
// reference's exit at the iteration cap), that correction is the last term of
// the returned state and no later iteration corrects its error, so that
// solve is taken closer to the exact Newton step.
constexpr double kMixedLastStepTighten = 1e-2;

// Mixed-precision defect correction: each FP32 inner solve stops at
// max(inner_tol, kInnerAim * target / ||D^-1 r||), target being the outer
// test's on the true FP64 residual.  The outer test alone decides
// convergence, so this factor only trades inner iterations against the risk
// of one more outer pass.  A second pass reduces its residual by about 1e-3,
// where the FP32 recursive residual stays within a fraction of a percent of
// the true one; on the 50^3 random-sphere RVE with 12 fields the final
// ||D^-1 r|| came to 0.70 of the target at most (0.30 with a factor of 0.3),
// with 73 instead of 76-77 inner iterations and still two outer passes.
constexpr double kInnerAim = 0.7;

// material_base with the derived constants of the reference's constructors
// (mppd_api.hip); MPPD_ERR_ARG for an unknown law.
int make_material(const material_base &in, material_base &m);

// ---------------- launchers (geometry.hip) ----------------
hipError_t launch_bmat(const Grid &g, double *bmat, hipStream_t st);
hipError_t launch_random_spheres(const double *geo, double *spheres, hipStream_t st);
hipError_t launch_phase_map(const Grid &g, int type, const double *geo, const double *spheres, int nsph, int *et,
                            int *bad, hipStream_t st);
// elements of phase 0 and of phases >= 1 (counts[2], zero on entry)
hipError_t launch_phase_counts(const Grid &g, const int *et, unsigned long long *counts, hipStream_t st);
hipError_t launch_ell_cols(const Grid &g, int *cols, hipStream_t st);
hipError_t launch_sell_to_rows(const Grid &g, const int *cols, const double *vals, int *cols_rm, double *vals_rm,
                               hipStream_t st);
hipError_t launch_rows_to_sell(const Grid &g, const double *vals_rm, double *vals, hipStream_t st);

// ---------------- launchers (assembly.hip) ----------------
hipError_t launch_material_eval(const material_base &m, int n, const double *eps, const double *hist, double *sig,
                                double *ctan, double *hist_new, int *nl, hipStream_t st);
hipError_t launch_set_displ_bc(const Grid &g, const double *eps6, double *u, hipStream_t st);
// Element stiffness: per phase (phase_mode: one 24x24 block per material,
// u/vars ignored) or per element.
hipError_t launch_elem_ke(const Grid &g, const double *bmat, const material_base *mats_d, const int *et, const double *u,
                          const double *vars, int phase_mode, double *ke, hipStream_t st);
hipError_t launch_gather_vals(const Grid &g, const int *et, const double *ke, int phase_mode, double *vals,
                              hipStream_t st);
hipError_t launch_elem_be(const Grid &g, const double *bmat, const material_base *mats, const int *et, const double *u,
                          const double *vars, double *be, hipStream_t st);
hipError_t launch_gather_rhs(const Grid &g, const double *be, double *b, double *partials, RedState *red,
                             hipStream_t st);
hipError_t launch_ave_stress(const Grid &g, const double *bmat, const material_base *mats, const int *et,
                             const double *u, const double *vars, double *partials, RedState *red, hipStream_t st);
hipError_t launch_vars_new(const Grid &g, const double *bmat, const material_base *mats, const int *et, const double *u,
                           const double *vars_old, double *vars_new, RedState *red, hipStream_t st);
// calc_fields: strain / stress nelem x 6 each
hipError_t launch_elem_fields(const Grid &g, const double *bmat, const material_base *mats, const int *et,
                              const double *u, const double *vars, double *strain, double *stress, hipStream_t st);

// ---------------- launchers (solver.hip) ----------------
// CG state is a pair: iteration k reads state[k & 1] and writes
// state[(k + 1) & 1] (parity = k); so are the search directions p[0], p[1].
// part needs 3 * (nrow_pad / 256) doubles.  Before state[q & 1] is read after
// q iterations, launch_cg_tail(.., q, ..) takes in the last one's sums.
hipError_t launch_spmv(const Grid &g, const int *cols, const double *vals, const double *x, double *y, hipStream_t st);
// The FP64 matrix of an all-elastic RVE as a stencil table: code[node] (of
// nrow_pad / 3 + 1) and 81 values of each of a code's three rows
struct Stencil64 {
  uint16_t *code = nullptr;
  double *tab = nullptr;
};
constexpr int kStencilCodes = 6561 + 2;  // 3^8 phase patterns, a boundary node, a padding node
// Nodes from which an all-elastic RVE's FP64 CG reads the table: its 12.8 MB
// (of which a solve touches the RVE's own patterns) against 1944 bytes a node
// of stored values.  Below, both come from L2: 16^3 nodes 10.3 us an iteration
// either way, 21^3 10.0 / 10.7, 26^3 11.0 / 12.7, 51^3 28.3 / 58.0.
constexpr int kDictNodes = 8000;
inline size_t stencil64_codes(const Grid &g) { return (size_t)g.nrow_pad / 3 + 1; }
inline size_t stencil64_table() { return (size_t)kStencilCodes * 3 * kSlots; }
hipError_t launch_stencil64(const Grid &g, const int *et, const double *ke, const Stencil64 &s, hipStream_t st);
// The working set of one Jacobi-PCG: vectors of nrow_pad doubles, the partial
// table and the state pair.
struct CgVecs {
  double *x, *r, *p[2], *Ap, *kinv, *part;
  CgState *state;
};
hipError_t launch_cg_init(const Grid &g, const double *vals, const double *b, const CgVecs &w, double min_err,
                          double rel_err, int max_its, hipStream_t st);
// step1 of an iteration; cols == nullptr: the matrix was assembled here and
// the stencil columns are computed; dict: it is dict's, whose table is read.  dir = false leaves out the kernel that
// forms p where step1 does not (timing of the SpMV alone, after one call with it)
hipError_t launch_cg_step1(const Grid &g, const int *cols, const double *vals, const Stencil64 *dict, const CgVecs &w,
                           int parity, hipStream_t st, bool dir = true);
hipError_t launch_cg_iter(const Grid &g, const int *cols, const double *vals, const Stencil64 *dict, const CgVecs &w,
                          int parity, hipStream_t st);
hipError_t launch_cg_tail(const Grid &g, const CgVecs &w, int queued, hipStream_t st);
hipError_t launch_axpy(int n, double a, const double *x, double *y, hipStream_t st);
hipError_t launch_copy(int n, const double *x, double *y, hipStream_t st);

// ---------------- launchers (vcycle.hip) ----------------
// The FP32 operator of an all-elastic RVE as a stencil dictionary: a 16-bit
// code per node (the phases of its eight elements), the table of stencils, the
// nodes whose elements differ in phase (nif of them, ascending) and the
// symmetric stencils of the others.
struct StencilOp {
  const uint16_t *code = nullptr;
  const int *list = nullptr;
  const float *tab = nullptr, *hom = nullptr;
  int nif = 0;
};
size_t stencil_bytes(const Grid &g);  // device bytes of an operator
// partials per field of a stencil kernel (at most ..._max, whatever the phases)
int stencil_blocks(const Grid &g, const StencilOp &op);
int stencil_blocks_max(const Grid &g);
// fills buf (stencil_bytes) and *op; ke: the FP64 element stiffness per phase (3 x 576); synchronizes st
hipError_t launch_d_setup(const Grid &g, const int *et, const double *ke, void *buf, StencilOp *op, hipStream_t st);
// AP = A P and the (p, Ap) partials part1[field * stencil_blocks + block]
hipError_t launch_d_spmv(const Grid &g, int K, const StencilOp &op, const float *P, float *AP, double *part1,
                         const void *state, hipStream_t st);
// the multilevel preconditioner of a K-field system (*out = nullptr: no
// coarse grid, or MPPD_COARSE=0); P and AP are its scratch during the set-up
// (contrast: of the RVE's materials, at least 1)
int vcycle_setup(const Grid &g, int K, double contrast, const int *et_d, const double *ke_d, const StencilOp &op, const float *kinv,
                 float *P, float *AP, hipStream_t st, VCycleDev **out);
void vcycle_free(VCycleDev *v);
// OUT = M R with Z = D^-1 R given (Z may be v.z), T a work vector, and the (r, OUT) partials
// pr[field * stencil_blocks + block]; OUT may be Z or T, not v.z
hipError_t launch_vcycle(const Grid &g, int K, const VCycleDev &v, const StencilOp &op, const float *kinv,
                         const float *R, const float *Z, float *T, float *OUT, double *pr, const void *cur,
                         hipStream_t st);
// after launch_m_resid: the inner CG's start direction P = M R and the state's (r, z)
hipError_t launch_v_start(const Grid &g, int K, const VCycleDev &v, const StencilOp &op, const float *kinv,
                          const float *R, float *P, float *AP, void *state, hipStream_t st);

// ---------------- launchers (mixed.hip): K right-hand sides, K in {4,8,12,16} ----------------
size_t mixed_matrix_floats(const Grid &g);
size_t mixed_vector_len(const Grid &g, int K);
size_t mixed_partials(const Grid &g, int K);
size_t mixed_state_bytes();
// the FP32 Jacobi weights of an all-elastic RVE (zero off the interior)
hipError_t launch_m_kinv(const Grid &g, const int *et, const double *ke, float *kinv, hipStream_t st);
hipError_t launch_m_setbc(const Grid &g, int K, const double *eps, double *U, hipStream_t st);
// F: adjoint sources (FP64, the layout of U) or null
hipError_t launch_m_resid(const Grid &g, int K, const int *et, const double *ke, const double *U, const double *F,
                          const float *kinv, float *R, float *X, float *P, double *part, int first, double rel,
                          double abs_tol, double tau_min, int max_inner, void *state, hipStream_t st,
                          const int *active = nullptr);
// U's K fields = the n <= K displacement vectors u[k] (reference numbering, node * 3 + d; a null one, or null u: zero),
// zero beyond; and back to those not null (the last of those that are the same)
hipError_t launch_m_load_u(const Grid &g, int K, int n, const double *const *u, double *U, hipStream_t st);
hipError_t launch_m_store_u(const Grid &g, int K, int n, const double *U, double *const *u, hipStream_t st);
// adjoint: G (3 x 24 x 6 doubles) and the sources F of fields 0 .. nadj-1
hipError_t launch_m_adj_src(const Grid &g, int K, int nadj, const double *bmat, const material_base *mats_d,
                            const int *et, double *G, double *F, hipStream_t st);
// adjoint derivatives from U (fields 0..5 = adjoint fields, s0 .. s0+ns-1 =
// forward fields): ctan[36] = d sigma_v / d eps_i (v * 6 + i), dmat[ns * 36] =
// d sigma_v / d (E, nu) of phase p ((s * 6 + v) * 6 + p * 2 + {0, 1})
size_t mixed_adj_partials(const Grid &g, int ns);
// (ke: the per-phase FP64 element stiffness, 3 x 576)
hipError_t launch_m_adj(const Grid &g, int K, const double *bmat, const material_base *mats_d, const int *et,
                        const double *ke, const double *U, int s0, int ns, double *part, double *ctan, double *dmat,
                        hipStream_t st);
// one inner CG iteration; R X P AP in the 4-field-group layout
// Two-level preconditioner: coarse (may be null: Jacobi alone).  start:
// after launch_m_resid, the inner CG's start direction P = z = D^-1 R +
// P_c A_c^-1 P_c^T R and the state's (r, z); launch_m_iter with coarse applies
// it in every iteration.
hipError_t launch_c_start(const Grid &g, int K, const CoarseDev &c, const float *kinv, const float *R, float *P,
                          void *state, hipStream_t st);
// one iteration of the inner CG (operator: the stored FP32 matrix A, K = 4 only,
// or, when A is null, the stencil dictionary op)
hipError_t launch_m_iter(const Grid &g, int K, const float *A, const StencilOp &op, const float *kinv, float *R, float *X, float *P,
                         float *AP, double *part, void *state, int parity, hipStream_t st,
                         const CoarseDev *coarse = nullptr, const VCycleDev *vc = nullptr);
// s0's (r, z) from partials prz[field * row + i]; guard: with the test of a positive definite preconditioner
hipError_t launch_c_rzfix(int K, int row, const double *prz, bool guard, void *state, hipStream_t st);
// blocks per component of the vector kernels (the partial tables' stride)
size_t coarse_vec_blocks(const Grid &g);
hipError_t launch_m_accum(const Grid &g, int K, const float *X, double *U, hipStream_t st);
// mixed-precision solves of an assembled FP64 ELL system (field 0 of K = 4):
// FP32 node-block copy of the interior block + Jacobi weights; FP64 residual
// b - A du with the outer test and inner start state; du += X
hipError_t launch_m_from_ell(const Grid &g, const double *vals, float *A, double *kinv64, float *kinv,
                             hipStream_t st);
hipError_t launch_m_resid_ell(const Grid &g, int K, const int *cols, const double *vals, const double *b,
                              const double *du, const double *kinv64, const float *kinv, float *R, float *X,
                              float *P, double *part, int first, double rel, double abs_tol, double tau_min,
                              int max_inner, void *state, hipStream_t st);
hipError_t launch_m_accum_ell(const Grid &g, int K, const float *X, double *du, hipStream_t st);
hipError_t launch_m_ave(const Grid &g, int K, const double *bmat, const material_base *mats_d, const int *et,
                        const double *U, double *part, double *out, hipStream_t st);
}  // namespace mpp

// One RVE: geometry, materials, B, phase map (the opaque mppd_rve of mppd.h).
struct mppd_rve {
  mpp::Grid g;
  int micro_type = 0;
  double geo[4];
  material_base mats[3];
  material_base *mats_d = nullptr;  // the same three on the device
  double *bmat = nullptr;
  int *et = nullptr;
  double *spheres = nullptr;
  void *arena = nullptr;  // owns the above
  int nsph = 0;
  double vf[2] = {0, 0};
  int all_elastic = 1;
};

namespace mpp {

void mixed_state_view(const void *state_h, int parity, int *its, int *all_done);
bool mixed_state_broken(const void *state_h, int parity);
// field k of the inner state: returns its done flag; *pn its preconditioned
// residual norm, *target the norm at which it stops
int mixed_state_field(const void *state_h, int parity, int k, double *pn, double *target);
void mixed_outer_view(const void *state_h, int K, int *all_conv, double *pn, double *pn0);
// per field: converged flag of the last outer test, ||r||_2 now and at the last `first` test
void mixed_outer_norms(const void *state_h, int K, int *conv, double *rn, double *rn0);

}  // namespace mpp
