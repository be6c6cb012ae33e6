// batch.hip -- many RVEs of uneven size, geometry and material state per
// launch (gfx950).
//
// A batch holds B RVEs, one per macro Gauss point.  Every finite-element
// operation of the Newton / CG path is ONE launch over the whole batch: the
// launch's blocks are the concatenation of each RVE's blocks, and a
// block -> RVE table (one int per block) tells a block which RVE it works on
// and its index inside that RVE.  The per-RVE arithmetic is the single-RVE
// kernels' (kernels.hpp bodies, same block shapes, same fixed reduction
// order), so a batched RVE's results are bit-identical to solving it alone.
// RVEs switched off in the per-RVE activity mask return at once; converged
// CGs stop through their own device-side flag.
//
// Launch shapes (blocks per RVE):
//   row   nrow_pad / 256       rows / nodes / CG vectors / SpMV
//   elem  ceil(nelem / 256)    one thread per element
//   ke    ceil(items / 4)      one wave per element stiffness (phase mode: 3)
//   rve   1                    per-RVE finishing reductions
#include "kernels.hpp"
#include "batch.hpp"

namespace mpp {

#define MPP_BATCH_PROLOGUE(MAP)                 \
  const int rid = MAP[blockIdx.x];              \
  if (!act[rid]) return;                        \
  const BRve &R = rv[rid];

// ---------------- boundary values and vector moves ----------------
__global__ void __launch_bounds__(256) kb_set_bc(const BRve *rv, const int *map, const int *act, const int *blk0,
                                                 const double *eps) {
  MPP_BATCH_PROLOGUE(map)
  const int lb = blockIdx.x - blk0[rid];
  set_bc_node(R.g, lb * 256 + threadIdx.x, eps + (size_t)rid * 6, R.uw);
}

// which: 0 uw <- u_n, 1 u_k <- uw, 2 uw <- u_k, 3 uw <- 0
__global__ void __launch_bounds__(256) kb_move(const BRve *rv, const int *map, const int *act, const int *blk0,
                                               int which) {
  MPP_BATCH_PROLOGUE(map)
  const int row = (blockIdx.x - blk0[rid]) * 256 + threadIdx.x;
  if (row >= R.g.nrow) return;
  switch (which) {
    case 0: R.uw[row] = R.u_n[row]; break;
    case 1: R.u_k[row] = R.uw[row]; break;
    case 2: R.uw[row] = R.u_k[row]; break;
    default: R.uw[row] = 0.0; break;
  }
}

// history moves: what 0: vars_n <- 0 and vars_k <- vars_aux (first
// nonlinearity); what 1: vars_aux <- 0
__global__ void __launch_bounds__(256) kb_vars_move(const BRve *rv, const int *map, const int *act, const int *blk0,
                                                    int what) {
  MPP_BATCH_PROLOGUE(map)
  const size_t n = (size_t)R.g.nelem * 8 * NVAR;
  const size_t t0 = (size_t)(blockIdx.x - blk0[rid]) * 256 + threadIdx.x;
  const size_t stride = (size_t)R.nb_elem * 256;
  for (size_t t = t0; t < n; t += stride) {
    if (what == 0) {
      R.vars_n[t] = 0.0;
      R.vars_k[t] = R.vars_aux[t];
    } else {
      R.vars_aux[t] = 0.0;
    }
  }
}

// ---------------- assembly ----------------
__global__ void __launch_bounds__(256) kb_elem_ke(const BRve *rv, const int *map, const int *act, const int *blk0) {
  MPP_BATCH_PROLOGUE(map)
  elem_ke_body(R.g, blockIdx.x - blk0[rid], R.bmat, R.mats, R.et, R.uw, R.use_vars ? R.vars_n : nullptr,
               R.phase_mode, R.ke);
}

__global__ void __launch_bounds__(256) kb_gather_vals(const BRve *rv, const int *map, const int *act,
                                                      const int *blk0) {
  MPP_BATCH_PROLOGUE(map)
  // four slices per row block
  gather_vals_slice(R.g, (blockIdx.x - blk0[rid]) * 4 + blockIdx.y, R.et, R.ke, R.phase_mode, R.vals);
}

__global__ void __launch_bounds__(256) kb_elem_be(const BRve *rv, const int *map, const int *act, const int *blk0) {
  MPP_BATCH_PROLOGUE(map)
  elem_be_body(R.g, (blockIdx.x - blk0[rid]) * (256 / kGpElems) + blockIdx.y, R.bmat, R.mats, R.et, R.uw, R.use_vars ? R.vars_n : nullptr, R.be);
}

__global__ void __launch_bounds__(256) kb_gather_rhs(const BRve *rv, const int *map, const int *act,
                                                     const int *blk0) {
  MPP_BATCH_PROLOGUE(map)
  gather_rhs_body(R.g, blockIdx.x - blk0[rid], R.be, R.b, R.part);
}

// one block per RVE: ||b||
__global__ void __launch_bounds__(256) kb_norm_finish(const BRve *rv, const int *act, double *out) {
  const int rid = blockIdx.x;
  if (!act[rid]) return;
  const BRve &R = rv[rid];
  double t[1];
  seg_sum<1>(R.part, R.nb_row, t);
  if (threadIdx.x == 0) out[rid] = sqrt(t[0]);
}

// u = uw (which 0) or u_k (which 1); vars as the RVE's use_vars says
__global__ void __launch_bounds__(8 * kAveElems) kb_ave_stress(const BRve *rv, const int *map, const int *act, const int *blk0,
                                                     int which) {
  MPP_BATCH_PROLOGUE(map)
  ave_stress_body(R.g, (blockIdx.x - blk0[rid]) * (256 / kAveElems) + blockIdx.y, R.bmat, R.mats, R.et, which ? R.u_k : R.uw,
                  R.use_vars ? R.vars_n : nullptr, R.part);
}

__global__ void __launch_bounds__(256) kb_ave_finish(const BRve *rv, const int *act, double *out) {
  const int rid = blockIdx.x;
  if (!act[rid]) return;
  const BRve &R = rv[rid];
  double t[6];
  ave_total(R.part, R.nb_elem, t);
  if (threadIdx.x == 0)
    for (int v = 0; v < 6; ++v) out[(size_t)rid * 6 + v] = t[v] / R.g.vol_tot;
}

// calc_vars_new on u_k: vars_old = vars_n if the RVE has history, else none;
// vars_new = vars_k if it has history, else vars_aux.  flags[rid] |= nonlinear.
__global__ void __launch_bounds__(256) kb_vars_new(const BRve *rv, const int *map, const int *act, const int *blk0,
                                                   int *flags) {
  MPP_BATCH_PROLOGUE(map)
  vars_new_body(R.g, (blockIdx.x - blk0[rid]) * (256 / kGpElems) + blockIdx.y, R.bmat, R.mats, R.et, R.u_k, R.use_vars ? R.vars_n : nullptr,
                R.use_vars ? R.vars_k : R.vars_aux, flags + rid);
}

__global__ void kb_zero_ints(int n, int *p) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---------------- CG ----------------
__device__ __forceinline__ const double *cg_matrix(const BRve &R, const int *a0on, int rid) {
  return a0on[rid] && R.a0 ? R.a0 : R.vals;
}

__global__ void __launch_bounds__(256) kb_cg_init(const BRve *rv, const int *map, const int *act, const int *blk0,
                                                  const int *a0on) {
  MPP_BATCH_PROLOGUE(map)
  cg_init_body(R.g, blockIdx.x - blk0[rid], cg_matrix(R, a0on, rid), R.b, R.x, R.r, R.kinv, R.part);
}

// one block per RVE; an inactive RVE's CG starts (and stays) done
__global__ void __launch_bounds__(256) kb_cg_init_state(const BRve *rv, const int *act, double min_err,
                                                        double rel_err, int max_its) {
  const int rid = blockIdx.x;
  const BRve &R = rv[rid];
  if (!act[rid]) {
    if (threadIdx.x == 0) {
      CgState c{};
      c.done = 1;
      R.cg[0] = c;
    }
    return;
  }
  cg_init_state_body(R.part, R.nb_row, min_err, rel_err, max_its, R.cg);
}

// The SpMV of the batch in one of its tuned shapes: CH slots of a row in
// flight per load round; XCD: launch block b takes logical block
// (b & 7) * per + (b >> 3), so each XCD streams a contiguous run of blocks
// (blocks are dispatched round-robin over the 8 XCDs).  The arithmetic is
// the same in every shape.
// DICT: some RVE's matrix is a stencil table (its branch costs the others 40
// registers, hence kernels of their own).  SRC: the stored ones (mat_source).
template <int CH, bool XCD, bool DICT, int SRC, bool AHEAD>
__global__ void __launch_bounds__(256) kb_cg_step1(const BRve *rv, const int2 *at, CgState *cg, const int *a0on,
                                                   int nb, int per, int parity) {
  const int b = XCD ? (int)((blockIdx.x & 7) * per + (blockIdx.x >> 3)) : (int)blockIdx.x;
  if (b >= nb) return;
  const int rid = at[b].x, k = parity & 1;
  const BRve &R = rv[rid];
  __shared__ double seg[kSegDoubles];
  CgState *cur = cg + 2 * rid + k, *nxt = cg + 2 * rid + (k ^ 1);
  if (DICT && R.dict.tab)
    cg_step1_body64<CH, kMatTable, AHEAD>(R.g, at[b].y, R.nb_row, R.dict.tab, R.dict.code, R.kinv, R.r, R.p[k], R.p[k ^ 1], R.Ap,
                           R.part, cur, nxt, seg);
  else  // vals and a0 are assembled here: the stencil columns follow from the grid
    cg_step1_body64<CH, SRC, AHEAD>(R.g, at[b].y, R.nb_row, cg_matrix(R, a0on, rid), nullptr, R.kinv, R.r, R.p[k], R.p[k ^ 1],
                        R.Ap, R.part, cur, nxt, seg);
}

__global__ void __launch_bounds__(256) kb_cg_step2(const BRve *rv, const int2 *at, const CgState *cg, int parity) {
  const int rid = at[blockIdx.x].x, n = (parity & 1) ^ 1;
  const BRve &R = rv[rid];
  cg_step2_body64(at[blockIdx.x].y, R.nb_row, R.x, R.r, R.p[n], R.Ap, R.kinv, R.part, cg + 2 * rid + n);
}

// one block per RVE
__global__ void __launch_bounds__(256) kb_cg_tail(const BRve *rv) {
  const BRve &R = rv[blockIdx.x];
  cg_tail_body(R.part + R.nb_row, R.nb_row, R.cg);
}

// uw += x
__global__ void __launch_bounds__(256) kb_axpy(const BRve *rv, const int *map, const int *act, const int *blk0) {
#pragma clang fp contract(off)
  MPP_BATCH_PROLOGUE(map)
  const int row = (blockIdx.x - blk0[rid]) * 256 + threadIdx.x;
  if (row < R.g.nrow) R.uw[row] += 1.0 * R.x[row];
}

// ---------------- device-side Newton control ----------------
__device__ __forceinline__ void nt_test(BNewton &s, const BNewtonTest &t) {
  // the reference tests at the top of an iteration: at the cap it stops
  // unconverged, even when the last residual passes (src/solve.cpp:43-78)
  if (s.its >= t.max_its) {
    s.run = 0;
  } else if (s.norm < t.max_tol || s.norm < s.norm0 * t.rel_tol) {
    s.conv = 1;
    s.run = 0;
  }
}

__global__ void kb_nt_start(int n, const int *on, const double *norms, BNewtonTest t, BNewton *nst) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  BNewton s = nst[r];
  s.its = s.sits = s.conv = s.applied = 0;
  s.run = on[r] != 0;
  if (s.run) {
    s.norm0 = s.norm = norms[r];
    nt_test(s, t);
  }
  nst[r] = s;
}

__global__ void kb_nt_prepare(int n, const BRve *rv, BNewton *nst, int has_a0, int its_with_A0, int *act, int *ke,
                              int *gather, int *a0on, int *pend) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  BNewton s = nst[r];
  const int run = s.run;
  const int a0sel = run && has_a0 && s.its < its_with_A0;
  const int phase = rv[r].phase_mode;
  act[r] = run;
  if (has_a0) a0on[r] = a0sel;
  ke[r] = run && !a0sel && !phase;
  gather[r] = run && !a0sel && (!phase || !s.vals_ready);
  if (run && !a0sel && phase) s.vals_ready = 1;
  s.applied = 0;
  pend[r] = 0;
  nst[r] = s;
}

// rows: uw += x of the RVEs whose CG stopped and whose correction is not in uw
__global__ void __launch_bounds__(256) kb_nt_axpy(const BRve *rv, const int *map, const int *blk0,
                                                  const BNewton *nst) {
#pragma clang fp contract(off)
  const int rid = map[blockIdx.x];
  const BNewton &s = nst[rid];
  const BRve &R = rv[rid];
  if (!s.run || s.applied || !R.cg[0].done) return;
  const int row = (blockIdx.x - blk0[rid]) * 256 + threadIdx.x;
  if (row < R.g.nrow) R.uw[row] += 1.0 * R.x[row];
}

__global__ void kb_nt_mark(int n, const BRve *rv, BNewton *nst, int *pend) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  BNewton s = nst[r];
  const CgState c = rv[r].cg[0];
  const int now = s.run && !s.applied && c.done;
  if (now) {
    s.applied = 1;
    s.sits += c.its;
    nst[r] = s;
  }
  pend[r] = now;
}

__global__ void kb_nt_after(int n, const int *pend, const double *norms, BNewtonTest t, BNewton *nst) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n || !pend[r]) return;
  BNewton s = nst[r];
  s.its += 1;
  s.norm = norms[r];
  nt_test(s, t);
  nst[r] = s;
}

// ---------------- mixed precision ----------------
__global__ void __launch_bounds__(256) kb_m_prep(const BRve *rv, const int *map, const int *act, const int *blk0,
                                                 const int *a0on) {
  MPP_BATCH_PROLOGUE(map)
  const int row = (blockIdx.x - blk0[rid]) * 256 + threadIdx.x;  // < nrow_pad
  const double *A = cg_matrix(R, a0on, rid);
  const size_t base = (size_t)(row >> 6) * kSlots * 64 + (row & 63);
  for (int s = 0; s < kSlots; ++s) R.vals32[base + (size_t)s * 64] = (float)A[base + (size_t)s * 64];
  double k = 0.0;
  if (row < R.g.nrow) k = 1 / A[base + (size_t)(13 * 3 + row % 3) * 64];
  R.kinv[row] = k;
  R.kinv32[row] = (float)k;
  R.x[row] = 0.0;
}

// partials per row block: (D^-1 r)^2, r32.z32, z32.z32
__global__ void __launch_bounds__(256) kb_m_resid(const BRve *rv, const int *map, const int *act, const int *blk0,
                                                  const int *a0on) {
#pragma clang fp contract(off)
  __shared__ double lds[4 * 3];
  MPP_BATCH_PROLOGUE(map)
  const int lb = blockIdx.x - blk0[rid];
  const int row = lb * 256 + threadIdx.x;
  const double rr = R.b[row] - row_dot_grid(R.g, cg_matrix(R, a0on, rid), (const double *)R.x, row);
  const double zr = R.kinv[row] * rr;
  const float r32 = (float)rr;
  const float z32 = R.kinv32[row] * r32;
  R.r[row] = rr;
  R.r32[0][row] = r32;
  R.x32[row] = 0.0f;
  double v[3] = {zr * zr, (double)r32 * z32, (double)z32 * z32};
  block_sum<3, 256>(v, lds);
  if (threadIdx.x == 0)
    for (int q = 0; q < 3; ++q) R.part[(size_t)lb * 3 + q] = v[q];
}

// the coarse solve's blocks of one RVE (none without a coarse level)
__device__ __forceinline__ int coarse_blocks(const BRve &R) { return (R.cgrid.nc + kGemvRows - 1) / kGemvRows; }

// one block per RVE: the outer test and the inner CG's start state (an
// inactive or converged RVE's inner CG starts done)
__global__ void __launch_bounds__(256) kb_m_outer(const BRve *rv, const int *act, int first, double rel,
                                                  double abs_tol, double tau_min, int max_inner, const int *tight,
                                                  double tight_factor, BOuter *out) {
  const int rid = blockIdx.x;
  if (tight && tight[rid]) rel *= tight_factor;
  const BRve &R = rv[rid];
  if (!act[rid]) {
    if (threadIdx.x == 0) {
      CgState c{};
      c.done = 1;
      R.cg[0] = c;
    }
    return;
  }
  double t[3], cz[1];
  seg_sum<3>(R.part, R.nb_row, t);
  seg_sum<1>(R.cpart, coarse_blocks(R), cz);
  if (threadIdx.x == 0) {
    BOuter &o = out[rid];
    const double pn = sqrt(t[0]);
    const double target = first ? fmax(abs_tol, rel * pn) : o.target;
    const int conv = pn < target || pn == 0.0;
    if (first) {
      o.pn0 = pn;
      o.target = target;
    }
    o.pn = pn;
    o.conv = conv;
    CgState c{};
    c.fresh = 1;
    c.rz = t[1] + cz[0];
    c.pn0 = sqrt(t[2]);
    c.pn = c.pn0;
    c.min_err = 0.0;
    // aim a little below what the outer test needs, but not below what FP32 resolves
    c.rel_err = pn > 0.0 ? fmax(tau_min, kInnerAim * target / pn) : 1.0;
    c.max_its = max_inner;
    c.its = 0;
    c.done = conv || cg_done(c);
    R.cg[0] = c;
  }
}

// ---------------------------------------------------------------------------
// The inner FP32 CG, four kernels per iteration:
//   dir    the scalars that the previous iteration's sums give (beta, the
//          stopping test), z = D^-1 r + P_c e and p = z + beta p
//   spmv   Ap = A p, partials of p.Ap (shapes as kb_cg_step1)
//   upd    alpha, x, r, partials of r.D^-1 r and of the stopping test's
//          ||D^-1 r||^2 on the row blocks; r_c = P_c^T r on the coarse ones
//   gemv   e = A_c^-1 r_c and partials of r_c.e
// with e the coarse correction of the two-level preconditioner: trilinear
// hats of the RVE's coarse grid (R.cgrid) and the inverse of the Galerkin
// coarse matrix of its initial (elastic) tangent.  (r, z) is r.D^-1 r +
// r_c.e, so z needs no kernel (nor vector) of its own.  The coarse blocks of
// upd form r - alpha Ap from the old r, beside the row blocks that store it:
// r lives in two vectors, read from r[k & 1] and written to r[(k + 1) & 1].
// States as in the FP64 CG (kernels.hpp).  FP32 residual rows: row = node * 3
// + d; sums over the rows, r_c among them, are FP64 in fixed orders.
// What bounds it: the SpMV streams 324 bytes per row (6.3 TB/s with eight
// RVEs of 25..31 nodes a side live); the other kernels, and the SpMV once most
// RVEs have stopped, wait for their launch, the state and the partial sums
// (4 to 6 us each), hence as few of them as the data allow.
// Eight J2 RVEs of 25..31 nodes a side, all live, us: SpMV 28.6, dir 4.4, upd
// 11.3, gemv 4.8 (eight kernels before, of 4 to 7 beside the SpMV); two live:
// 10, 3.4, 5.3, 3.5.  With a coarse level on every side (not only those with a
// suitable divisor) the slowest of them takes 392 iterations a load step
// instead of 1233, and the step 28 ms instead of 75.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void m_scalars(CgRegs &c, const BRve &R) {
#pragma clang fp contract(off)
  if (c.done || c.fresh) return;
  double t[2], cz[1];
  seg_sum<2>(R.part + R.nb_row, R.nb_row, t);
  seg_sum<1>(R.cpart, coarse_blocks(R), cz);
  const double rz = t[1] + cz[0];
  c.beta = rz / c.rz;
  c.pn = sqrt(t[0]);
  c.rz = rz;
  c.its += 1;
  c.done = cg_done(c);
}

// one thread per node: the weights of the 8 coarse nodes around it (zero
// outside) serve its three rows
__global__ void __launch_bounds__(256) kb_m_dir(const BRve *rv, const int2 *at, CgState *cg, int parity) {
  const int rid = at[blockIdx.x].x, lb = at[blockIdx.x].y, k = parity & 1;
  const BRve &R = rv[rid];
  CgRegs c = cg_load(cg + 2 * rid + k);
  const Grid &g = R.g;
  const CGrid &cgd = R.cgrid;
  const int node = lb * 256 + threadIdx.x;
  const bool in = node < g.nn;
  float z[3] = {}, p[3] = {};
  if (in && !c.done) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      z[d] = R.kinv32[node * 3 + d] * R.r32[k][node * 3 + d];
      p[d] = R.p32[node * 3 + d];
    }
    if (cgd.nc) {
      const int i = node % g.nx, j = (node / g.nx) % g.ny, l = node / (g.nx * g.ny);
      const HatEntry hx = R.hat[0][i], hy = R.hat[1][j], hz = R.hat[2][l];
      float acc[3] = {};
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const float w = (t & 1 ? hx.w1 : hx.w0) * ((t & 2 ? hy.w1 : hy.w0) * (t & 4 ? hz.w1 : hz.w0));
        const float *e = R.cec + ((t & 1 ? hx.q1 : hx.q0) + (t & 2 ? hy.q1 : hy.q0) + (t & 4 ? hz.q1 : hz.q0));
#pragma unroll
        for (int d = 0; d < 3; ++d) acc[d] += w * e[d];
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) z[d] += acc[d];
    }
  }
  m_scalars(c, R);
  if (lb == 0 && threadIdx.x == 0) cg_store(c, c.done, cg + 2 * rid + (k ^ 1));
  if (c.done || !in) return;
#pragma unroll
  for (int d = 0; d < 3; ++d) R.p32[node * 3 + d] = c.its == 0 ? z[d] : (float)(z[d] + c.beta * p[d]);
}

template <int CH, bool XCD, int SRC>
__global__ void __launch_bounds__(256) kb_m_spmv(const BRve *rv, const int2 *at, const CgState *cg, int nb, int per,
                                                 int parity) {
  const int b = XCD ? (int)((blockIdx.x & 7) * per + (blockIdx.x >> 3)) : (int)blockIdx.x;
  if (b >= nb) return;
  const int rid = at[b].x;
  const BRve &R = rv[rid];
  cg_spmv_body32<CH, SRC>(R.g, at[b].y, R.vals32, R.p32, R.Ap32, R.part, cg + 2 * rid + ((parity & 1) ^ 1));
}

// START: r_c of the residual kb_m_resid has stored (RVEs in act); the row
// blocks have nothing to do
template <bool START>
__global__ void __launch_bounds__(256) kb_m_upd(const BRve *rv, const int2 *at, const int *act, const CgState *cg,
                                                int parity) {
#pragma clang fp contract(off)
  __shared__ double lds[4 * 2];
  const int rid = at[blockIdx.x].x, lb = at[blockIdx.x].y, k = START ? 0 : parity & 1;
  const BRve &R = rv[rid];
  const CgState *cur = cg + 2 * rid + (k ^ 1);
  if (START ? !act[rid] || lb < R.nb_row : cur->done != 0) return;
  double alpha = 0.0;
  const float *r = R.r32[k], *Ap = R.Ap32;
  if (lb < R.nb_row) {
    const int row = lb * 256 + threadIdx.x;
    const float xo = R.x32[row], ro = r[row], po = R.p32[row], ao = Ap[row], ko = R.kinv32[row];
    double pap[1];
    seg_sum<1>(R.part, R.nb_row, pap);
    alpha = cur->rz / pap[0];
    R.x32[row] = xo + alpha * po;
    const float rv2 = ro - alpha * ao;
    R.r32[k ^ 1][row] = rv2;
    const float zv = ko * rv2;
    double v[2] = {(double)zv * zv, (double)rv2 * zv};
    block_sum<2, 256>(v, lds);
    if (threadIdx.x == 0) {
      R.part[R.nb_row + (size_t)lb * 2 + 0] = v[0];
      R.part[R.nb_row + (size_t)lb * 2 + 1] = v[1];
    }
    return;
  }
  const CGrid &cgd = R.cgrid;
  const int q = lb - R.nb_row;
  if (q >= cgd.nq) return;
  if (!START) {
    double pap[1];
    seg_sum<1>(R.part, R.nb_row, pap);
    alpha = cur->rz / pap[0];
  }
  // the nodes under the hat of coarse node (cx, cy, cz), between its neighbours
  const int dx = cgd.mx + 1, dy = cgd.my + 1, dz = cgd.mz + 1;
  const int cx = q % cgd.mx, cy = (q / cgd.mx) % cgd.my, cz = q / (cgd.mx * cgd.my);  // interior index, 0-based
  const int i0 = cx * R.g.nex / dx + 1, j0 = cy * R.g.ney / dy + 1, l0 = cz * R.g.nez / dz + 1;
  const int wx = (cx + 2) * R.g.nex / dx - i0, wy = (cy + 2) * R.g.ney / dy - j0;
  const int n = wx * wy * ((cz + 2) * R.g.nez / dz - l0);
  const int ox = 3 * cx, oy = 3 * cgd.mx * cy, oz = 3 * cgd.mx * cgd.my * cz;
  const auto weight = [](const HatEntry &h, int o) { return (h.q0 == o ? h.w0 : 0.0f) + (h.q1 == o ? h.w1 : 0.0f); };
  double acc[3] = {};
#pragma unroll 2
  for (int s = threadIdx.x; s < n; s += 256) {
    const int i = i0 + s % wx, j = j0 + (s / wx) % wy, l = l0 + s / (wx * wy);
    const float w = weight(R.hat[0][i], ox) * (weight(R.hat[1][j], oy) * weight(R.hat[2][l], oz));
    const int e = ((l * R.g.ny + j) * R.g.nx + i) * 3;
#pragma unroll
    for (int d = 0; d < 3; ++d) acc[d] += (double)w * (START ? r[e + d] : (float)(r[e + d] - alpha * Ap[e + d]));
  }
  __shared__ double ldc[4 * 3];
  block_sum<3, 256>(acc, ldc);
  if (threadIdx.x < 3) {
    R.crc[q * 3 + threadIdx.x] = acc[threadIdx.x];
    R.crc32[q * 3 + threadIdx.x] = (float)acc[threadIdx.x];
  }
}

// e = A_c^-1 r_c: a wave per two coarse rows (the inverse's rows read along
// their length); act: at the start, else the RVEs whose CG goes on
__global__ void __launch_bounds__(256) kb_c_gemv(const BRve *rv, const int2 *at, const int *act, const CgState *cg,
                                                 int parity) {
  __shared__ double lds[4];
  const int rid = at[blockIdx.x].x, lb = at[blockIdx.x].y, nc = rv[rid].cgrid.nc;
  const BRve &R = rv[rid];
  if (lb * kGemvRows >= nc || (act ? !act[rid] : cg[2 * rid + ((parity & 1) ^ 1)].done != 0)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, row = lb * kGemvRows + 2 * w;
  const float *rc = R.crc32;
  const float *a0 = R.cainv + (size_t)min(row, nc - 1) * nc, *a1 = R.cainv + (size_t)min(row + 1, nc - 1) * nc;
  const double r0 = R.crc[min(row, nc - 1)], r1 = R.crc[min(row + 1, nc - 1)];
  float s0 = 0.0f, s1 = 0.0f;
#pragma unroll 8
  for (int c = lane; c < nc; c += 64) {
    const float v = rc[c];
    s0 = fmaf(a0[c], v, s0);
    s1 = fmaf(a1[c], v, s1);
  }
  s0 = wave_sum_dpp(s0);
  s1 = wave_sum_dpp(s1);
  if (lane == 0) {
    double z = 0.0;
    if (row < nc) R.cec[row] = s0, z += r0 * s0;
    if (row + 1 < nc) R.cec[row + 1] = s1, z += r1 * s1;
    lds[w] = z;
  }
  lds_barrier();
  if (threadIdx.x == 0) R.cpart[lb] = ((lds[0] + lds[1]) + lds[2]) + lds[3];
}

// one block per RVE
__global__ void __launch_bounds__(256) kb_m_tail(const BRve *rv, CgState *cg) {
  CgState *state = cg + 2 * blockIdx.x;
  CgRegs c = cg_load(state);
  if (c.done || c.fresh) return;
  m_scalars(c, rv[blockIdx.x]);
  if (threadIdx.x == 0) cg_store(c, 1, state);
}

__global__ void __launch_bounds__(256) kb_m_accum(const BRve *rv, const int *map, const int *act, const int *blk0) {
  MPP_BATCH_PROLOGUE(map)
  const int row = (blockIdx.x - blk0[rid]) * 256 + threadIdx.x;
  R.x[row] += (double)R.x32[row];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_b_set_bc(const BLaunch &L, const double *eps, hipStream_t st) {
  hipLaunchKernelGGL(kb_set_bc, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.map, L.act, L.row.blk0, eps);
  return hipGetLastError();
}
hipError_t launch_b_move(const BLaunch &L, int which, hipStream_t st) {
  hipLaunchKernelGGL(kb_move, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.map, L.act, L.row.blk0, which);
  return hipGetLastError();
}
hipError_t launch_b_vars_move(const BLaunch &L, int what, hipStream_t st) {
  hipLaunchKernelGGL(kb_vars_move, dim3(L.elem.nb), dim3(256), 0, st, L.rv, L.elem.map, L.act, L.elem.blk0, what);
  return hipGetLastError();
}
hipError_t launch_b_mat(const BLaunch &L, const int *act_ke, const int *act_gather, hipStream_t st) {
  hipLaunchKernelGGL(kb_elem_ke, dim3(L.ke.nb), dim3(64 * kKeWaves), 0, st, L.rv, L.ke.map, act_ke, L.ke.blk0);
  hipLaunchKernelGGL(kb_gather_vals, dim3(L.row.nb, 4), dim3(256), 0, st, L.rv, L.row.map, act_gather, L.row.blk0);
  return hipGetLastError();
}
hipError_t launch_b_rhs(const BLaunch &L, double *norms, hipStream_t st) {
  hipLaunchKernelGGL(kb_elem_be, dim3(L.elem.nb, 256 / kGpElems), dim3(8 * kGpElems), 0, st, L.rv, L.elem.map, L.act, L.elem.blk0);
  hipLaunchKernelGGL(kb_gather_rhs, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.map, L.act, L.row.blk0);
  hipLaunchKernelGGL(kb_norm_finish, dim3(L.nrve), dim3(256), 0, st, L.rv, L.act, norms);
  return hipGetLastError();
}
hipError_t launch_b_ave(const BLaunch &L, int which, double *sig, hipStream_t st) {
  hipLaunchKernelGGL(kb_ave_stress, dim3(L.elem.nb, 256 / kAveElems), dim3(8 * kAveElems), 0, st, L.rv, L.elem.map, L.act, L.elem.blk0, which);
  hipLaunchKernelGGL(kb_ave_finish, dim3(L.nrve), dim3(256), 0, st, L.rv, L.act, sig);
  return hipGetLastError();
}
hipError_t launch_b_vars_new(const BLaunch &L, int *flags, hipStream_t st) {
  hipLaunchKernelGGL(kb_zero_ints, dim3((L.nrve + 255) / 256), dim3(256), 0, st, L.nrve, flags);
  hipLaunchKernelGGL(kb_vars_new, dim3(L.elem.nb, 256 / kGpElems), dim3(8 * kGpElems), 0, st, L.rv, L.elem.map, L.act, L.elem.blk0, flags);
  return hipGetLastError();
}
hipError_t launch_b_cg_init(const BLaunch &L, double min_err, double rel_err, int max_its, hipStream_t st) {
  hipLaunchKernelGGL(kb_cg_init, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.map, L.act, L.row.blk0, L.a0on);
  hipLaunchKernelGGL(kb_cg_init_state, dim3(L.nrve), dim3(256), 0, st, L.rv, L.act, min_err, rel_err, max_its);
  return hipGetLastError();
}
template <int CH, bool XCD>
static void launch_step1(const BLaunch &L, int parity, hipStream_t st) {
  const int nb = L.row.nb, per = (nb + 7) / 8;
  const bool stream = mat_source((double)nb * 256 * kSlots * sizeof(double)) == kMatStream;
  const bool ahead = cg_ahead(nb, L.nx_max);
  const auto k = stream ? (L.dict ? kb_cg_step1<CH, XCD, true, kMatStream, false>
                                  : kb_cg_step1<CH, XCD, false, kMatStream, false>)
                 : L.dict ? (ahead ? kb_cg_step1<CH, XCD, true, kMatCached, true>
                                   : kb_cg_step1<CH, XCD, true, kMatCached, false>)
                          : (ahead ? kb_cg_step1<CH, XCD, false, kMatCached, true>
                                   : kb_cg_step1<CH, XCD, false, kMatCached, false>);
  hipLaunchKernelGGL(k, dim3(XCD ? 8 * per : nb), dim3(256), 0, st, L.rv, L.row.at, L.cg, L.a0on, nb, per, parity);
}

hipError_t launch_b_spmv(const BLaunch &L, int shape, int parity, hipStream_t st) {
  switch (shape) {
    case 0: launch_step1<9, false>(L, parity, st); break;
    case 1: launch_step1<27, false>(L, parity, st); break;
    case 2: launch_step1<81, false>(L, parity, st); break;
    case 3: launch_step1<9, true>(L, parity, st); break;
    case 4: launch_step1<27, true>(L, parity, st); break;
    case 5: launch_step1<81, true>(L, parity, st); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_b_cg_iter(const BLaunch &L, int parity, hipStream_t st) {
  hipError_t e = launch_b_spmv(L, L.spmv_shape, parity, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kb_cg_step2, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.at, L.cg, parity);
  return hipGetLastError();
}
hipError_t launch_b_cg_tail(const BLaunch &L, hipStream_t st) {
  hipLaunchKernelGGL(kb_cg_tail, dim3(L.nrve), dim3(256), 0, st, L.rv);
  return hipGetLastError();
}
hipError_t launch_b_axpy(const BLaunch &L, hipStream_t st) {
  hipLaunchKernelGGL(kb_axpy, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.map, L.act, L.row.blk0);
  return hipGetLastError();
}

static unsigned per_rve_blocks(int n) { return (unsigned)((n + 255) / 256); }

hipError_t launch_b_nt_start(const BLaunch &L, const int *on, const double *norms, BNewtonTest t, BNewton *nst,
                             hipStream_t st) {
  hipLaunchKernelGGL(kb_nt_start, dim3(per_rve_blocks(L.nrve)), dim3(256), 0, st, L.nrve, on, norms, t, nst);
  return hipGetLastError();
}
hipError_t launch_b_nt_prepare(const BLaunch &L, BNewton *nst, int has_a0, int its_with_A0, int *act, int *ke,
                               int *gather, int *a0on, int *pend, hipStream_t st) {
  hipLaunchKernelGGL(kb_nt_prepare, dim3(per_rve_blocks(L.nrve)), dim3(256), 0, st, L.nrve, L.rv, nst, has_a0,
                     its_with_A0, act, ke, gather, a0on, pend);
  return hipGetLastError();
}
hipError_t launch_b_nt_finish(const BLaunch &L, BNewtonTest t, BNewton *nst, int *pend, double *norms,
                              hipStream_t st) {
  hipLaunchKernelGGL(kb_nt_axpy, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.map, L.row.blk0, nst);
  hipLaunchKernelGGL(kb_nt_mark, dim3(per_rve_blocks(L.nrve)), dim3(256), 0, st, L.nrve, L.rv, nst, pend);
  BLaunch P = L;
  P.act = pend;
  hipError_t e = launch_b_rhs(P, norms, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kb_nt_after, dim3(per_rve_blocks(L.nrve)), dim3(256), 0, st, L.nrve, pend, norms, t, nst);
  return hipGetLastError();
}

hipError_t launch_bm_prep(const BLaunch &L, hipStream_t st) {
  hipLaunchKernelGGL(kb_m_prep, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.map, L.act, L.row.blk0, L.a0on);
  return hipGetLastError();
}
hipError_t launch_bm_resid(const BLaunch &L, int first, double rel, double abs_tol, double tau_min, int max_inner,
                           const int *tight, double tight_factor, BOuter *out, hipStream_t st) {
  hipLaunchKernelGGL(kb_m_resid, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.map, L.act, L.row.blk0, L.a0on);
  if (L.coarse) {
    hipLaunchKernelGGL(kb_m_upd<true>, dim3(L.upd.nb), dim3(256), 0, st, L.rv, L.upd.at, L.act, L.cg, 0);
    hipLaunchKernelGGL(kb_c_gemv, dim3(L.gemv.nb), dim3(256), 0, st, L.rv, L.gemv.at, L.act, L.cg, 0);
  }
  hipLaunchKernelGGL(kb_m_outer, dim3(L.nrve), dim3(256), 0, st, L.rv, L.act, first, rel, abs_tol, tau_min,
                     max_inner, tight, tight_factor, out);
  return hipGetLastError();
}
template <int CH, bool XCD>
static void launch_m_spmv(const BLaunch &L, int parity, hipStream_t st) {
  const int nb = L.row.nb, per = (nb + 7) / 8;
  const bool stream = mat_source((double)nb * 256 * kSlots * sizeof(float)) == kMatStream;
  const auto k = stream ? kb_m_spmv<CH, XCD, kMatStream> : kb_m_spmv<CH, XCD, kMatCached>;
  hipLaunchKernelGGL(k, dim3(XCD ? 8 * per : nb), dim3(256), 0, st, L.rv, L.row.at, L.cg, nb, per, parity);
}
hipError_t launch_bm_spmv(const BLaunch &L, int shape, int parity, hipStream_t st) {
  switch (shape) {
    case 0: launch_m_spmv<9, false>(L, parity, st); break;
    case 1: launch_m_spmv<27, false>(L, parity, st); break;
    case 2: launch_m_spmv<81, false>(L, parity, st); break;
    case 3: launch_m_spmv<9, true>(L, parity, st); break;
    case 4: launch_m_spmv<27, true>(L, parity, st); break;
    case 5: launch_m_spmv<81, true>(L, parity, st); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
hipError_t launch_bm_iter(const BLaunch &L, int parity, hipStream_t st) {
  hipLaunchKernelGGL(kb_m_dir, dim3(L.node.nb), dim3(256), 0, st, L.rv, L.node.at, L.cg, parity);
  const hipError_t e = launch_bm_spmv(L, L.spmv_shape32, parity, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kb_m_upd<false>, dim3(L.upd.nb), dim3(256), 0, st, L.rv, L.upd.at, L.act, L.cg, parity);
  if (L.coarse)
    hipLaunchKernelGGL(kb_c_gemv, dim3(L.gemv.nb), dim3(256), 0, st, L.rv, L.gemv.at, (const int *)nullptr, L.cg,
                       parity);
  return hipGetLastError();
}
hipError_t launch_bm_tail(const BLaunch &L, hipStream_t st) {
  hipLaunchKernelGGL(kb_m_tail, dim3(L.nrve), dim3(256), 0, st, L.rv, L.cg);
  return hipGetLastError();
}
hipError_t launch_bm_accum(const BLaunch &L, hipStream_t st) {
  hipLaunchKernelGGL(kb_m_accum, dim3(L.row.nb), dim3(256), 0, st, L.rv, L.row.map, L.act, L.row.blk0);
  return hipGetLastError();
}

}  // namespace mpp
