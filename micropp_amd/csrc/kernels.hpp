// kernels.hpp -- device bodies of the FP64 hot path, shared by the
// single-RVE kernels (assembly.hip, solver.hip) and the batched kernels
// (batch.hip).
//
// A body works on one block's share of one RVE: `lb` is the block's index
// inside that RVE and `nb` the RVE's block count, so a single-RVE kernel
// passes blockIdx.x / gridDim.x and a batched kernel passes its block's
// position inside its RVE.  Both therefore do the same arithmetic in the same
// order, and a batched RVE's results are bit-identical to a single solve.
//
// Reductions are fence-free: every block writes its partial, and a later
// kernel re-sums the partials of an RVE in a fixed order (seg_sum).
#pragma once

#include "internal.hpp"
#include "physics.hpp"
#include "reduce.hpp"

namespace mpp {

constexpr int kKeWaves = 4;  // element-stiffness items (waves) per block

__device__ __forceinline__ void elem_coords(const Grid &g, int e, int &ex, int &ey, int &ez) {
  ex = e % g.nex;
  ey = (e / g.nex) % g.ney;
  ez = e / (g.nex * g.ney);
}

// Global node id of local node a of element (ex, ey, ez) (src/common.cpp:28-41)
__device__ __forceinline__ int elem_node(const Grid &g, int ex, int ey, int ez, int a) {
  return ((ez + kHexPos[a][2]) * g.ny + (ey + kHexPos[a][1])) * g.nx + ex + kHexPos[a][0];
}

__device__ __forceinline__ bool on_boundary(const Grid &g, int i, int j, int k) {
  return i == 0 || j == 0 || k == 0 || i == g.nx - 1 || j == g.ny - 1 || k == g.nz - 1;
}

// get_strain (src/common.cpp:56-72) from the gathered element displacements
__device__ __forceinline__ void strain_at(const double *b /* [6][24] */, const double *ue, double *eps) {
#pragma clang fp contract(off)
  for (int v = 0; v < 6; ++v) {
    double s = 0;
    for (int i = 0; i < 24; ++i) s += b[v * 24 + i] * ue[i];
    eps[v] = s;
  }
}

__device__ __forceinline__ void gather_ue(const Grid &g, int ex, int ey, int ez, const double *u, double *ue) {
  for (int a = 0; a < 8; ++a) {
    const size_t base = (size_t)elem_node(g, ex, ey, ez, a) * 3;
    ue[a * 3 + 0] = u[base + 0];
    ue[a * 3 + 1] = u[base + 1];
    ue[a * 3 + 2] = u[base + 2];
  }
}

__device__ __forceinline__ void stage_bmat(const double *bmat_g, double *bm) {
  for (int i = threadIdx.x; i < 8 * 144; i += blockDim.x) bm[i] = bmat_g[i];
}

// Fixed-order sum of NV interleaved partials [nparts][NV] by one block of 256
// threads; every thread gets the totals.
template <int NV>
__device__ __forceinline__ void seg_sum(const double *part, int nparts, double (&out)[NV]) {
  __shared__ double lds[4 * NV];
  double acc[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) acc[k] = 0.0;
  for (int b = threadIdx.x; b < nparts; b += 256)
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] += part[(size_t)b * NV + k];
  block_sum<NV, 256>(acc, lds);
#pragma unroll
  for (int k = 0; k < NV; ++k) out[k] = acc[k];
}

// ---------------------------------------------------------------------------
// set_displ_bc (src/micro3D.cpp:26-78).  The reference visits the faces
// z=0, z=lz, y=0, y=ly, x=0, x=lx and later faces overwrite shared edges, so
// a node takes the coordinates of the last face containing it.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void set_bc_node(const Grid &g, int node, const double *e, double *u) {
#pragma clang fp contract(off)
  if (node >= g.nn) return;
  const int i = node % g.nx, j = (node / g.nx) % g.ny, k = node / (g.nx * g.ny);
  if (!on_boundary(g, i, j, k)) return;
  const double L = 1.0;
  double x[3];
  if (i == g.nx - 1) {
    x[0] = L, x[1] = j * g.dy, x[2] = k * g.dz;
  } else if (i == 0) {
    x[0] = 0, x[1] = j * g.dy, x[2] = k * g.dz;
  } else if (j == g.ny - 1) {
    x[0] = i * g.dx, x[1] = L, x[2] = k * g.dz;
  } else if (j == 0) {
    x[0] = i * g.dx, x[1] = 0, x[2] = k * g.dz;
  } else if (k == g.nz - 1) {
    x[0] = i * g.dx, x[1] = j * g.dy, x[2] = L;
  } else {
    x[0] = i * g.dx, x[1] = j * g.dy, x[2] = 0;
  }
  const double et[3][3] = {{e[0], 0.5 * e[3], 0.5 * e[4]}, {0.5 * e[3], e[1], 0.5 * e[5]}, {0.5 * e[4], 0.5 * e[5], e[2]}};
  for (int d = 0; d < 3; ++d) {
    double s = 0.0;
    for (int c = 0; c < 3; ++c) s += et[d][c] * x[c];
    u[(size_t)node * 3 + d] = s;
  }
}

// ---------------------------------------------------------------------------
// Element stiffness, get_elem_mat (src/assembly.cpp:140-178): Ke = sum_gp B^T
// (C B wg), one wavefront per element (or per material in phase mode); block
// lb holds items lb*4 .. lb*4+3.  B of a node holds its three shape gradients
// (gx, gy, gz) and zeros, so every sum over strain components has three
// products instead of six; they are added in the reference's order (gp, then
// component), without contraction, and the zero products left out change no
// sum (it starts at +0).  The waves share nothing but the gradients, so after
// those there are no block barriers.
//
// What bounds it: FP64 mul and add (about 600 per lane of an element) beside
// the 4.6 KB written per element.  A lane owns one (gp, node) of C B and one
// (node, node) 3x3 tile of Ke; sig, C and C B take turns in 9.2 KB of LDS a
// wave (four blocks a CU).  40^3 J2 elements: 168 us (460 with the zero products,
// 15 KB a wave and block barriers), 1.8 TB/s of writes.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void wave_lds_sync() {  // LDS written by other lanes of this wave
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// one strain component at a Gauss point with gradients gr[node * 3 + d]
// (strain_at, the products with B's zeros left out)
__device__ __forceinline__ double strain_row(const double *gr, const double *ue, int v) {
#pragma clang fp contract(off)
  const int d0 = v < 3 ? v : v == 5 ? 1 : 0, d1 = v == 3 ? 1 : 2;
  double s = 0;
#pragma unroll
  for (int a = 0; a < 8; ++a) {
    if (v < 3) {
      s += gr[a * 3 + v] * ue[a * 3 + v];
    } else {
      s += gr[a * 3 + d1] * ue[a * 3 + d0];
      s += gr[a * 3 + d0] * ue[a * 3 + d1];
    }
  }
  return s;
}

constexpr int kKeWork = 8 * 8 * 18;  // doubles of a wave's turn-taking LDS: C B
__device__ __forceinline__ void elem_ke_body(const Grid &g, int lb, const double *bmat_g, const material_base *mats,
                                             const int *et, const double *u, const double *vars, int phase_mode,
                                             double *ke) {
#pragma clang fp contract(off)
  __shared__ double grad[8 * 24];  // gx, gy, gz of (gp, node)
  __shared__ double ue_s[kKeWaves][24];
  __shared__ double work[kKeWaves][kKeWork];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  if (tid < 8 * 24) grad[tid] = bmat_g[(tid / 24) * 144 + (tid % 3) * 24 + tid % 24];
  const int item = lb * kKeWaves + w;
  const int nitems = phase_mode ? 3 : g.nelem;
  const bool active = item < nitems;
  int ex = 0, ey = 0, ez = 0, ph = 0;
  if (active) {
    if (phase_mode) {
      ph = item;
    } else {
      elem_coords(g, item, ex, ey, ez);
      ph = et[item];
    }
  }
  if (lane < 24) {
    double v = 0.0;
    if (active && !phase_mode && u) v = u[(size_t)elem_node(g, ex, ey, ez, lane / 3) * 3 + lane % 3];
    ue_s[w][lane] = v;
  }
  __syncthreads();
  if (!active) return;
  // mat_ctan per GP.  Elastic: the closed form, one lane per GP.  Otherwise
  // the forward-difference tangent's 7 stress evaluations per GP (base and
  // 6 perturbed strains) run on 56 lanes at once, then each tangent entry is
  // (s1 - s0) / D_EPS_CTAN as in mat_ctan: the same values bit for bit.
  double *C_s = work[w], *eps_s = C_s + 8 * 36, *sig_s = eps_s + 8 * 6;  // sig: 8 x 7 x 6
  if (mats[ph].type != MATERIAL_ELASTIC) {
    if (lane < 48) eps_s[lane] = strain_row(&grad[(lane / 6) * 24], ue_s[w], lane % 6);
    wave_lds_sync();
    if (lane < 56) {
      const int gp = lane / 7, c = lane % 7;  // c = 0: base strain; c > 0: component c - 1 perturbed
      double e1[6];
      for (int i = 0; i < 6; ++i) e1[i] = eps_s[gp * 6 + i] + (i == c - 1 ? D_EPS_CTAN : 0.0);
      const double *h = (vars && !phase_mode) ? vars + ((size_t)item * 8 + gp) * NVAR : nullptr;
      mat_stress(mats[ph], e1, h, &sig_s[lane * 6]);
    }
    wave_lds_sync();
    for (int q = lane; q < 8 * 36; q += 64) {
      const int gp = q / 36, r = (q / 6) % 6, c = q % 6;
      const double *sg = &sig_s[gp * 7 * 6];
      C_s[q] = (sg[(c + 1) * 6 + r] - sg[r]) / D_EPS_CTAN;
    }
  } else if (lane < 8) {
    mat_ctan(mats[ph], nullptr, nullptr, &C_s[lane * 36]);
  }
  wave_lds_sync();
  const int hi = lane >> 3, lo = lane & 7;
  {  // C B wg of Gauss point hi and node lo: 6 rows x 3 columns
    const double gx = grad[hi * 24 + lo * 3], gy = grad[hi * 24 + lo * 3 + 1], gz = grad[hi * 24 + lo * 3 + 2];
    double C[36];
#pragma unroll
    for (int q = 0; q < 36; ++q) C[q] = C_s[hi * 36 + q];
    wave_lds_sync();  // C B takes C's place
    double *cb = &work[w][lane * 18];
#pragma unroll
    for (int m = 0; m < 6; ++m) {
      const double *c = &C[m * 6];
      cb[m * 3 + 0] = (c[0] * gx + c[3] * gy + c[4] * gz) * g.wg;
      cb[m * 3 + 1] = (c[1] * gy + c[3] * gx + c[5] * gz) * g.wg;
      cb[m * 3 + 2] = (c[2] * gz + c[4] * gx + c[5] * gy) * g.wg;
    }
  }
  wave_lds_sync();
  // lane (hi, lo) = node pair: rows 3 hi .. 3 hi + 2, columns 3 lo .. 3 lo + 2
  double acc[3][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
#pragma unroll 2
  for (int gp = 0; gp < 8; ++gp) {
    const double *gr = &grad[gp * 24 + hi * 3], *cb = &work[w][(gp * 8 + lo) * 18];
    const double gx = gr[0], gy = gr[1], gz = gr[2];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      acc[0][c] += gx * cb[0 + c];
      acc[0][c] += gy * cb[9 + c];
      acc[0][c] += gz * cb[12 + c];
      acc[1][c] += gy * cb[3 + c];
      acc[1][c] += gx * cb[9 + c];
      acc[1][c] += gz * cb[15 + c];
      acc[2][c] += gz * cb[6 + c];
      acc[2][c] += gx * cb[12 + c];
      acc[2][c] += gy * cb[15 + c];
    }
  }
  wave_lds_sync();  // Ke takes C B's place on its way out, for whole lines
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int c = 0; c < 3; ++c) work[w][(3 * hi + a) * 24 + 3 * lo + c] = acc[a][c];
  wave_lds_sync();
  double *out = ke + (size_t)item * 576;
#pragma unroll
  for (int q = 0; q < 9; ++q) out[q * 64 + lane] = work[w][q * 64 + lane];
}

// ---------------------------------------------------------------------------
// Row-owner gather of the element blocks into SELL vals: assembly_mat's
// element loop + ell_add_3D (src/assembly.cpp:105-121,
// src/ell-common.cpp:166-198) and ell_set_bc_3D (:238-297).  For row
// (node N, fi) and slot (neighbour M, fj) the contributing elements are those
// holding both N and M, visited in reference order ex, ey, ez.
//
// A block of 256 threads makes one slice (64 rows) in LDS.  A wave takes 8
// rows at a time: its 8 x 8 lanes load, for each of the 8 elements around the
// row's node, the row's 3 entries towards local node p: 192 bytes in a line
// per row and element, all 24 loads of a lane in flight, every entry of ke
// read once.  Then it adds them element by element (LDS operations of a wave
// keep their order), and the slice is stored by whole lines.  Bound: memory,
// the element matrices in and the values out.  40^3 elements: 85 us
// (a thread per row: 188), 5.0 TB/s.
// ---------------------------------------------------------------------------
constexpr int kGatherPitch = 66;  // doubles per slot of the slice in LDS
__device__ __forceinline__ void gather_vals_slice(const Grid &g, int slice, const int *et, const double *ke,
                                                  int phase_mode, double *vals) {
#pragma clang fp contract(off)
  __shared__ double acc[kSlots * kGatherPitch];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, p = lane & 7;
  for (int t = threadIdx.x; t < kSlots * kGatherPitch; t += 256) acc[t] = 0.0;
  __syncthreads();
  const int px = kHexPos[p][0], py = kHexPos[p][1], pz = kHexPos[p][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = (h * 4 + w) * 8 + (lane >> 3), row = slice * 64 + r;  // (rows of one wave only)
    if (row >= g.nrow) continue;
    const int node = row / 3, fi = row % 3;
    const int i = node % g.nx, j = (node / g.nx) % g.ny, k = node / (g.nx * g.ny);
    if (on_boundary(g, i, j, k)) {
      if (p == 0) acc[(13 * 3 + fi) * kGatherPitch + r] = 1.0;
      continue;
    }
    double v[8][3];
#pragma unroll
    for (int q = 0; q < 8; ++q) {  // reference order (a, b, c) = (x, y, z)
      const int a = q >> 2, b = (q >> 1) & 1, c = q & 1;
      const int e = ((k - 1 + c) * g.ney + j - 1 + b) * g.nex + i - 1 + a;  // interior node: always inside
      const int la = local_node(1 - a, 1 - b, 1 - c);
      const double *s = ke + (size_t)(phase_mode ? et[e] : e) * 576 + (la * 3 + fi) * 24 + p * 3;
#pragma unroll
      for (int d = 0; d < 3; ++d) v[q][d] = s[d];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      // neighbour of the node at local node p of element q
      const int n = ((pz + (q & 1)) * 3 + py + ((q >> 1) & 1)) * 3 + px + (q >> 2);
      double *o = &acc[n * 3 * kGatherPitch + r];
#pragma unroll
      for (int d = 0; d < 3; ++d) o[d * kGatherPitch] += v[q][d];
      wave_lds_sync();
    }
  }
  __syncthreads();
  double *out = vals + (size_t)slice * kSlots * 64;
  for (int t = threadIdx.x; t < kSlots * 64; t += 256) out[t] = acc[(t >> 6) * kGatherPitch + (t & 63)];
}

// A third (neighbours of plane Z) of one row of an all-elastic RVE's matrix (ke:
// its phases' element stiffness, in the caches) by one thread, the same sums.
// Bound: the stores alone.  A call, us, with slices made in LDS / a thread per
// row / per third: 11^3 nodes 18 / 23 / 17, 31^3 32 / 36 / 29, 41^3 52 / 47 / 46,
// 51^3 85 / 70 / 69, 71^3 217 / 215 / 189.
template <int Z>
__device__ __forceinline__ void gather_vals_row(const Grid &g, int row, const int *et, const double *ke,
                                                double *vals) {
#pragma clang fp contract(off)
  if (row >= g.nrow_pad) return;
  double *out = vals + (size_t)(row >> 6) * kSlots * 64 + (row & 63);
  const int node = row / 3, fi = row % 3;
  const int i = node % g.nx, j = (node / g.nx) % g.ny, k = node / (g.nx * g.ny);
  if (row >= g.nrow || on_boundary(g, i, j, k)) {
    for (int s = 27 * Z; s < 27 * Z + 27; ++s) out[s * 64] = row < g.nrow && s == 13 * 3 + fi ? 1.0 : 0.0;
    return;
  }
  const double *s[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {  // reference order (a, b, c) = (x, y, z)
    const int a = q >> 2, b = (q >> 1) & 1, c = q & 1;
    const int e = ((k - 1 + c) * g.ney + j - 1 + b) * g.nex + i - 1 + a;
    s[q] = ke + (size_t)et[e] * 576 + (local_node(1 - a, 1 - b, 1 - c) * 3 + fi) * 24;
  }
#pragma unroll
  for (int n = 9 * Z; n < 9 * Z + 9; ++n) {
    double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int px = n % 3 - (q >> 2), py = (n / 3) % 3 - ((q >> 1) & 1), pz = n / 9 - (q & 1);
      if (px < 0 || px > 1 || py < 0 || py > 1 || pz < 0 || pz > 1) continue;
#pragma unroll
      for (int d = 0; d < 3; ++d) acc[d] += s[q][local_node(px, py, pz) * 3 + d];
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) out[(n * 3 + d) * 64] = acc[d];
  }
}

// ---------------------------------------------------------------------------
// The Gauss-point kernels: a thread per Gauss point (8 lanes an element), so
// that an RVE of a few hundred elements is not a handful of waves that each
// evaluate eight laws in a row.  gp_stage puts the gradients and the
// displacements of the block's NE elements (from e0 on) into LDS, gp_strain is
// get_strain at the thread's point (strain_row, in the reference's order).
// ---------------------------------------------------------------------------
template <int NE>
__device__ __forceinline__ void gp_stage(const Grid &g, int e0, const double *bmat_g, const double *u,
                                         double *grad /* [8 * 24] */, double *ue /* [NE * 24] */) {
  for (int t = threadIdx.x; t < 8 * 24; t += 8 * NE) grad[t] = bmat_g[(t / 24) * 144 + (t % 3) * 24 + t % 24];
  for (int t = threadIdx.x; t < NE * 24; t += 8 * NE) {
    const int e = e0 + t / 24, i = t % 24;
    if (e >= g.nelem) break;
    int ex, ey, ez;
    elem_coords(g, e, ex, ey, ez);
    ue[t] = u[(size_t)elem_node(g, ex, ey, ez, i / 3) * 3 + i % 3];
  }
  __syncthreads();
}

__device__ __forceinline__ void gp_strain(const double *grad, const double *ue, double *eps) {
#pragma unroll
  for (int v = 0; v < 6; ++v) eps[v] = strain_row(&grad[(threadIdx.x & 7) * 24], &ue[(threadIdx.x >> 3) * 24], v);
}

constexpr int kGpElems = 32;    // elements per block of 256 threads
constexpr int kAveElems = 64;   // elements per block of 512 (ave_stress_body)

// ---------------------------------------------------------------------------
// Element internal forces, get_elem_rhs (src/assembly.cpp:123-138).  The
// stresses of the block's points go through LDS; then three of the 24 entries
// of an element per thread, summed over (gp, component) in the reference's
// order, B's zeros left out (elem_ke_body).  40^3 J2 elements 25
// us, 125 elements 6 (a thread per element: 37.5 and 24).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void elem_be_body(const Grid &g, int lb, const double *bmat_g, const material_base *mats,
                                             const int *et, const double *u, const double *vars, double *be) {
#pragma clang fp contract(off)
  __shared__ double grad[8 * 24], ue[kGpElems * 24], sig_s[kGpElems * 48];
  const int e0 = lb * kGpElems;
  gp_stage<kGpElems>(g, e0, bmat_g, u, grad, ue);
  const int e = e0 + (threadIdx.x >> 3);
  if (e < g.nelem) {
    double eps[6];
    gp_strain(grad, ue, eps);
    mat_stress(mats[et[e]], eps, vars ? vars + ((size_t)e0 * 8 + threadIdx.x) * NVAR : nullptr,
               &sig_s[threadIdx.x * 6]);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int t = k * 256 + threadIdx.x, i = t % 24, a = i / 3, d = i % 3;
    if (e0 + t / 24 >= g.nelem) break;
    // the three components with row i of B not zero, ascending, and its entries there
    const int v0 = d, v1 = d == 2 ? 4 : 3, v2 = d == 0 ? 4 : 5;
    const int g0 = d, g1 = d == 1 ? 0 : d == 0 ? 1 : 0, g2 = d == 0 ? 2 : d == 1 ? 2 : 1;
    double acc = 0;
#pragma unroll
    for (int gp = 0; gp < 8; ++gp) {
      const double *b = &grad[gp * 24 + a * 3], *sig = &sig_s[(t / 24) * 48 + gp * 6];
      acc += b[g0] * sig[v0] * g.wg;
      acc += b[g1] * sig[v1] * g.wg;
      acc += b[g2] * sig[v2] * g.wg;
    }
    be[(size_t)e0 * 24 + t] = acc;
  }
}

// ---------------------------------------------------------------------------
// Row-owner gather of the element forces: assembly_rhs (src/assembly.cpp:
// 27-103): element order ez, ey, ex; Dirichlet DOFs zeroed; negated.  The
// block's partial of ||b||^2 goes to part[lb].
// ---------------------------------------------------------------------------
__device__ __forceinline__ void gather_rhs_body(const Grid &g, int lb, const double *be, double *bvec, double *part) {
#pragma clang fp contract(off)
  __shared__ double lds[4];
  const int row = lb * 256 + threadIdx.x;
  double sq = 0.0;
  if (row < g.nrow) {
    const int node = row / 3, d = row % 3;
    const int i = node % g.nx, j = (node / g.nx) % g.ny, k = node / (g.nx * g.ny);
    double acc = 0.0;
    if (!on_boundary(g, i, j, k)) {
      for (int c = 0; c < 2; ++c)
        for (int b = 0; b < 2; ++b)
          for (int a = 0; a < 2; ++a) {
            const int e = ((k - 1 + c) * g.ney + (j - 1 + b)) * g.nex + (i - 1 + a);
            acc += be[(size_t)e * 24 + local_node(1 - a, 1 - b, 1 - c) * 3 + d];
          }
    }
    const double v = -acc;
    bvec[row] = v;
    sq = v * v;
  }
  double val[1] = {sq};
  block_sum<1, 256>(val, lds);
  if (threadIdx.x == 0) part[lb] = val[0];
}

// ---------------------------------------------------------------------------
// calc_ave_stress (src/average.cpp:57-82): per-element sums over the Gauss
// points, and the sum of a block's 64 elements (one wave of them) to
// part[lb * 6 ..]; ave_total adds those.  40^3 J2 elements
// 15.5 us, 125 elements 5 (a thread per element: 21 and 13).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void ave_stress_body(const Grid &g, int lb, const double *bmat_g, const material_base *mats,
                                                const int *et, const double *u, const double *vars, double *part) {
#pragma clang fp contract(off)
  __shared__ double grad[8 * 24], ue[kAveElems * 24], sig_s[kAveElems * 48];
  const int e0 = lb * kAveElems;
  gp_stage<kAveElems>(g, e0, bmat_g, u, grad, ue);
  const int e = e0 + (threadIdx.x >> 3);
  if (e < g.nelem) {
    double eps[6];
    gp_strain(grad, ue, eps);
    mat_stress(mats[et[e]], eps, vars ? vars + ((size_t)e0 * 8 + threadIdx.x) * NVAR : nullptr,
               &sig_s[threadIdx.x * 6]);
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  double s6[6] = {0, 0, 0, 0, 0, 0};
  if (e0 + (int)threadIdx.x < g.nelem)
    for (int gp = 0; gp < 8; ++gp)
#pragma unroll
      for (int v = 0; v < 6; ++v) s6[v] += sig_s[threadIdx.x * 48 + gp * 6 + v] * g.wg;
#pragma unroll
  for (int v = 0; v < 6; ++v) {
    const double s = wave_sum(s6[v]);
    if (threadIdx.x == 0) part[(size_t)lb * 6 + v] = s;
  }
}

// the 6 totals of nb blocks of 256 elements, four partials each, by one block
// of 256 threads (every thread gets them)
__device__ __forceinline__ void ave_total(const double *part, int nb, double (&t)[6]) {
#pragma clang fp contract(off)
  __shared__ double lds[4 * 6];
#pragma unroll
  for (int v = 0; v < 6; ++v) t[v] = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256)
#pragma unroll
    for (int v = 0; v < 6; ++v) {
      double s = 0;
#pragma unroll
      for (int w = 0; w < 4; ++w) s += part[((size_t)b * 4 + w) * 6 + v];
      t[v] += s;
    }
  block_sum<6, 256>(t, lds);
}

// ---------------------------------------------------------------------------
// calc_fields (src/average.cpp:84-112): per element, the Gauss-point strain
// and stress summed with weight wg, times ivol = 1 / (8 wg)
// (src/micropp.cpp:59); element-major [e * 6 + v].
// ---------------------------------------------------------------------------
__device__ __forceinline__ void elem_fields_body(const Grid &g, int lb, const double *bmat_g,
                                                 const material_base *mats, const int *et, const double *u,
                                                 const double *vars, double *strain, double *stress) {
#pragma clang fp contract(off)
  __shared__ double bm[8 * 144];
  stage_bmat(bmat_g, bm);
  __syncthreads();
  const int e = lb * 256 + threadIdx.x;
  if (e >= g.nelem) return;
  int ex, ey, ez;
  elem_coords(g, e, ex, ey, ez);
  double ue[24];
  gather_ue(g, ex, ey, ez, u, ue);
  const material_base &m = mats[et[e]];
  double ea[6] = {0, 0, 0, 0, 0, 0}, sa[6] = {0, 0, 0, 0, 0, 0};
  for (int gp = 0; gp < 8; ++gp) {
    double eps[6], sig[6];
    strain_at(&bm[gp * 144], ue, eps);
    mat_stress(m, eps, vars ? vars + ((size_t)e * 8 + gp) * NVAR : nullptr, sig);
    for (int v = 0; v < 6; ++v) {
      ea[v] += eps[v] * g.wg;
      sa[v] += sig[v] * g.wg;
    }
  }
  const double ivol = 1.0 / (g.wg * 8);
  for (int v = 0; v < 6; ++v) {
    strain[(size_t)e * 6 + v] = ea[v] * ivol;
    stress[(size_t)e * 6 + v] = sa[v] * ivol;
  }
}

// ---------------------------------------------------------------------------
// calc_vars_new (src/update.cpp:32-56): evolute per Gauss point; any
// nonlinear point sets *flag.  A call on 40^3 J2 elements takes 28 us, with
// history 40 (a thread per element: 46 and 60), on 10^3 20 and 21 (33 and 45).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void vars_new_body(const Grid &g, int lb, const double *bmat_g, const material_base *mats,
                                              const int *et, const double *u, const double *vars_old,
                                              double *vars_new, int *flag) {
#pragma clang fp contract(off)
  __shared__ double grad[8 * 24], ue[kGpElems * 24];
  const int e0 = lb * kGpElems;
  gp_stage<kGpElems>(g, e0, bmat_g, u, grad, ue);
  const int e = e0 + (threadIdx.x >> 3);
  if (e >= g.nelem) return;
  double eps[6];
  gp_strain(grad, ue, eps);
  const size_t off = ((size_t)e0 * 8 + threadIdx.x) * NVAR;
  const int nl = mat_evolute(mats[et[e]], eps, vars_old ? vars_old + off : nullptr, vars_new + off);
  // Every wave with a nonlinear point stores the same 1, read after the kernel.
  // (An atomic operation each, all on one address: 10 ns a wave; 50^3 J2
  // elements, all yielding, 161 us a call instead of 38.)
  if (__ballot(nl != 0) && (threadIdx.x & 63) == 0)
    __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ---------------------------------------------------------------------------
// ell_mvp (src/ell.cpp:35-44) row: the 81 slots in chunks of CH (9, 27 or
// 81 slots in flight): the chunk's columns and values first (non-temporal,
// streamed once), then its x gathers, then the products added in slot order
// without contraction, so y is bit-identical to the reference SpMV whatever
// the chunk width.
// ---------------------------------------------------------------------------
constexpr int kChunk = 27;

template <int CH = kChunk>
__device__ __forceinline__ double row_dot(const int *cols, const double *vals, const double *x, int row) {
#pragma clang fp contract(off)
  static_assert(kSlots % CH == 0, "chunks tile the row");
  const size_t base = (size_t)(row >> 6) * kSlots * 64 + (row & 63);
  const int *c = cols + base;
  const double *v = vals + base;
  double acc = 0;
#pragma unroll
  for (int ch = 0; ch < kSlots / CH; ++ch) {
    int ci[CH];
    double vi[CH], xv[CH];
#pragma unroll
    for (int k = 0; k < CH; ++k) ci[k] = __builtin_nontemporal_load(&c[(ch * CH + k) * 64]);
#pragma unroll
    for (int k = 0; k < CH; ++k) vi[k] = __builtin_nontemporal_load(&v[(ch * CH + k) * 64]);
#pragma unroll
    for (int k = 0; k < CH; ++k) xv[k] = x[ci[k]];
#pragma unroll
    for (int k = 0; k < CH; ++k) acc += vi[k] * xv[k];
  }
  return acc;
}

// row_dot on the structured grid: the column of slot nb*3 + fj of row 3n + fi
// is 3 m + fj for the stencil neighbour m = n + offset(nb) (ell_init,
// src/ell-common.cpp:102-130), computed instead of loaded, which leaves 8 of
// the 12 bytes per slot.  m is clamped into the grid.  For a matrix assembled
// here only the rows of boundary nodes (Dirichlet rows, zero off the
// diagonal) and padding rows (zero) have stencil slots outside the grid,
// where the reference's column 0 + fj and the clamped column both give a zero
// product for a finite x, and a sum that starts at +0 is unchanged by adding
// either signed zero.  So the result equals row_dot's bit for bit.  (A matrix
// uploaded from the host may hold values in those slots: use row_dot.)
// T = float: the FP32 inner CG of the mixed-precision batch (FP32 sums).
template <int CH = kChunk, typename T>
__device__ __forceinline__ T row_dot_grid(const Grid &g, const T *vals, const T *x, int row) {
#pragma clang fp contract(off)
  static_assert(kSlots % CH == 0 && CH % 3 == 0, "chunks tile the row in whole neighbours");
  const size_t base = (size_t)(row >> 6) * kSlots * 64 + (row & 63);
  const T *v = vals + base;
  const int n = row / 3, nxny = g.nx * g.ny, hi = g.nn - 1;
  T acc = 0;
#pragma unroll
  for (int ch = 0; ch < kSlots / CH; ++ch) {
    T vi[CH], xv[CH];
#pragma unroll
    for (int k = 0; k < CH; ++k) vi[k] = __builtin_nontemporal_load(&v[(ch * CH + k) * 64]);
#pragma unroll
    for (int k = 0; k < CH; k += 3) {
      const int nb = (ch * CH + k) / 3;
      const int off = (nb / 9 - 1) * nxny + ((nb / 3) % 3 - 1) * g.nx + (nb % 3 - 1);
      const int m3 = 3 * min(max(n + off, 0), hi);
#pragma unroll
      for (int fj = 0; fj < 3; ++fj) xv[k + fj] = x[m3 + fj];
    }
#pragma unroll
    for (int k = 0; k < CH; ++k) acc += vi[k] * xv[k];
  }
  return acc;
}

// The gathers of row_dot_grid for a block of 256 consecutive rows, staged in
// LDS.  The rows belong to 86 nodes from n_lo = row0 / 3 on (wherever the
// block starts), whose stencil neighbours lie on runs of consecutive nodes:
// one of 88 nodes per (dz, dy), or, while those of one dz overlap (a line of
// at most 88 nodes), one run per dz.  The block writes f(entry) of every node
// on the runs (clamped node indices, as row_dot_grid clamps each neighbour)
// once, coalesced, and every row reads its 81 values there instead of
// gathering them from L1/L2: the same values in the same slot order, so the
// result is bit-identical to row_dot_grid.  ly and lz are the LDS distances,
// in nodes, of a line and of a plane.  Every thread of the block must call it.
constexpr int kSegNodes = 88, kSegDoubles = 9 * kSegNodes * 3;
struct SegPitch {
  int ly, lz;
};
template <typename T, typename F>
__device__ __forceinline__ SegPitch stage_runs(const Grid &g, int row0, T *seg /* [9 * kSegNodes * 3] */, F f) {
  const bool joined = g.nx <= kSegNodes;
  const int len = joined ? kSegNodes + 2 * g.nx : kSegNodes;
  const SegPitch pt{joined ? g.nx : kSegNodes, joined ? len : 3 * kSegNodes};
  const int n_lo = row0 / 3, nxny = g.nx * g.ny, hi = g.nn - 1, runs = joined ? 1 : 3;
  for (int dz = -1; dz <= 1; ++dz)
    for (int y = 0; y < runs; ++y) {
      const int n0 = n_lo - 1 + dz * nxny + (y - 1) * g.nx;
      T *out = seg + ((dz + 1) * pt.lz + y * kSegNodes) * 3;
#pragma unroll 2
      for (int e3 = threadIdx.x; e3 < 3 * len; e3 += 256)
        out[e3] = f(3 * min(max(n0 + e3 / 3, 0), hi) + e3 % 3);
    }
  lds_barrier();
  return pt;
}

// One row's products with the staged runs (own: its node there), in slot
// order: the first chunk's values are loaded by the caller, each later chunk's
// before the products of the one in front.
// Where the values come from: a stored matrix (slot k at v[k * 64]) read past
// the caches or through them, or a row of a stencil table (v[k]).
enum MatSource { kMatStream, kMatCached, kMatTable };
template <int SRC, typename T>
__device__ __forceinline__ T load_value(const T *v, int k) {
  if constexpr (SRC == kMatStream)
    return __builtin_nontemporal_load(&v[k * 64]);
  else
    return v[SRC == kMatTable ? k : k * 64];
}
// The stored matrix of a CG is read once an iteration.  While most of it (of
// every RVE of a launch) fits the 256 MB last-level cache, plain loads find it
// there, or in L2; beyond, non-temporal ones keep it from evicting the vectors.
// us per SpMV, plain / non-temporal: 21 MB 6.4 / 8.5, 101 MB 18.4 / 18.8, 171 MB
// (FP32) 28.7 / 30.0, 270 MB (FP32) 42.1 / 43.0, 381 MB 72.8 / 65.0.
inline int mat_source(double bytes) { return bytes > 320e6 ? kMatStream : kMatCached; }
template <int CH, int SRC, typename T>
__device__ __forceinline__ T dot_runs(const T *v, T (&vi)[2][CH], const T *own, SegPitch pt) {
#pragma clang fp contract(off)
  static_assert(kSlots % CH == 0 && CH % 3 == 0, "chunks tile the row in whole neighbours");
  T acc = 0;
#pragma unroll
  for (int ch = 0; ch < kSlots / CH; ++ch) {
    if (ch + 1 < kSlots / CH)
#pragma unroll
      for (int k = 0; k < CH; ++k) vi[(ch + 1) & 1][k] = load_value<SRC>(v, (ch + 1) * CH + k);
#pragma unroll
    for (int k = 0; k < CH; k += 3) {
      const int n = (ch * CH + k) / 3;
      const T *sv = own + ((n / 9 - 1) * pt.lz + ((n / 3) % 3 - 1) * pt.ly + n % 3 - 1) * 3;
#pragma unroll
      for (int fj = 0; fj < 3; ++fj) acc += vi[ch & 1][k + fj] * sv[fj];
    }
  }
  return acc;
}

// ---------------------------------------------------------------------------
// ell_solve_cgpd (src/ell.cpp:66-122), the reference recurrence in two
// kernels per iteration (FP64):
//   step1  the scalars that the previous iteration's sums give (beta, the
//          stopping test), p = z + beta p with z = k r, Ap = A p and the
//          per-block partials of p.Ap
//   step2  alpha = r.z / sum(partials); x += alpha p; r -= alpha Ap; z = k r;
//          per-block partials of z.z and r.z
// The new p has to be read by every row's neighbours, so each block of step1
// forms it, from k, r and the old p, for all nodes on its 9 stencil runs while
// it stages them in LDS (about 9 times each value, the same products each
// time), and stores its own rows' share: p lives in two vectors, read from
// p[i & 1] and written to p[(i + 1) & 1] in iteration i.  z is not stored.
// Every block re-sums all partials of its RVE in the same fixed order, so
// every block holds identical scalars.  Iteration i reads state[i & 1] and
// block 0 of its step1 writes state[(i + 1) & 1], which step2 reads.  The
// sums of the last step2 queued are taken in by cg_tail (before the host
// reads the state), which marks the state fresh: the next step1 then only
// applies its beta.  Once the stopping test holds, later iterations return at
// once and step1 only carries the final state forward.
// Partials: part1 = part[0 .. nb), part2 = part[nb .. 3 nb).
// ---------------------------------------------------------------------------
template <typename C>
__device__ __forceinline__ int cg_done(const C &c) {
  const bool conv = (c.pn < c.min_err) || (c.pn < c.pn0 * c.rel_err);
  return (c.its >= c.max_its || conv) ? 1 : 0;
}

// k = 1/diag; x = 0; r = b - A*0 = b; partials of r.z, z.z with z = k r (the
// first step1 takes p = z)
__device__ __forceinline__ void cg_init_body(const Grid &g, int lb, const double *vals, const double *b, double *x,
                                             double *r, double *kinv, double *part) {
#pragma clang fp contract(off)
  __shared__ double lds[4 * 2];
  const int row = lb * 256 + threadIdx.x;
  double k = 0.0, rv = 0.0;
  if (row < g.nrow) {
    const size_t d = ((size_t)(row >> 6) * kSlots + 13 * 3 + row % 3) * 64 + (row & 63);
    k = 1 / vals[d];
    rv = b[row] - 0.0;
  }
  const double zv = k * rv;
  kinv[row] = k;
  x[row] = 0.0;
  r[row] = rv;
  double v[2] = {rv * zv, zv * zv};
  block_sum<2, 256>(v, lds);
  if (threadIdx.x == 0) {
    part[(size_t)lb * 2 + 0] = v[0];
    part[(size_t)lb * 2 + 1] = v[1];
  }
}

// one block: the initial scalars into state[0]
__device__ __forceinline__ void cg_init_state_body(const double *part, int nparts, double min_err, double rel_err,
                                                   int max_its, CgState *state) {
  double t[2];
  seg_sum<2>(part, nparts, t);
  if (threadIdx.x == 0) {
    CgState c{};
    c.min_err = min_err;
    c.rel_err = rel_err;
    c.max_its = max_its;
    c.rz = t[0];
    c.pn0 = sqrt(t[1]);
    c.pn = c.pn0;
    c.its = 0;
    c.fresh = 1;
    c.done = cg_done(c);
    state[0] = c;
  }
}

// a CgState in registers: only the fields that the CG reads.  (A copy of the
// whole struct goes through LDS, whose addresses take the block size from the
// dispatch packet: a read of host memory by every wave, 11 us at 1555 blocks.)
struct CgRegs {
  double rz, pn0, pn, beta, min_err, rel_err;
  int its, max_its, done, fresh;
};

__device__ __forceinline__ CgRegs cg_load(const CgState *s) {
  return CgRegs{s->rz, s->pn0, s->pn, s->beta, s->min_err, s->rel_err, s->its, s->max_its, s->done, s->fresh};
}

__device__ __forceinline__ void cg_store(const CgRegs &c, int fresh, CgState *s) {
  s->rz = c.rz;
  s->pn0 = c.pn0;
  s->pn = c.pn;
  s->beta = c.beta;
  s->min_err = c.min_err;
  s->rel_err = c.rel_err;
  s->its = c.its;
  s->max_its = c.max_its;
  s->done = c.done;
  s->fresh = fresh;
}

// the scalars of the iteration that c's last step2 belongs to, from the sums
// of its partials (no-op on a fresh state)
__device__ __forceinline__ void cg_scalars(CgRegs &c, const double *part2, int nb) {
#pragma clang fp contract(off)
  if (c.fresh) return;
  double t[2];
  seg_sum<2>(part2, nb, t);
  c.beta = t[1] / c.rz;
  c.pn = sqrt(t[0]);
  c.rz = t[1];
  c.its += 1;
  c.done = cg_done(c);
}

// the state entering an iteration: true if the CG goes on.  part2 holds the
// previous iteration's sums; block 0 writes the state that step2 and the next
// step1 read.
__device__ __forceinline__ bool cg_enter(CgRegs &c, int lb, int nb, const double *part2, CgState *nxt) {
  if (!c.done) cg_scalars(c, part2, nb);
  if (lb == 0 && threadIdx.x == 0) cg_store(c, c.done, nxt);  // a stopped state has no sums to come
  return !c.done;
}

// p of the iteration at one row: p = z + beta p, and p = z in the first
__device__ __forceinline__ double cg_dir(const CgRegs &c, double k, double r, double p) {
#pragma clang fp contract(off)
  const double z = k * r;
  return c.its == 0 ? z : z + c.beta * p;
}

// AHEAD of cg_step1_body64: lines of at most 41 nodes (two entries of a run per
// thread, and one run per plane), and so few row blocks that the 36 registers
// more do not keep any of them waiting.  Iteration, us, ahead / not: 6^3 nodes
// 8.7 / 9.5, 11^3 9.0 / 10.4, 21^3 9.5 / 10.4, 31^3 12.7 / 13.2, eight J2 RVEs of
// 11^3 9.3 / 10.1.
inline bool cg_ahead(int row_blocks, int nx) { return row_blocks <= 768 && 3 * (kSegNodes + 2 * nx) <= 512; }

// step1 of a matrix assembled here (computed stencil columns).  What bounds
// it: at 50^3 nodes the 648 bytes of values per row; on RVEs of a few
// thousand rows the chain of waits (state, sums, stage, values).  The first
// chunk of the row's values does not depend on any of the others, so it is
// loaded before them, and each later chunk before the previous one's products;
// the barriers in between wait for LDS alone.
// code != nullptr: the matrix of an all-elastic RVE as a stencil table (tab, in
// place of vals: 81 values of each of the three rows per code, k_s_table), the
// same values in the same order (kDictNodes).  51^3 nodes: 22.6 us against 47.2
// with the stored matrix, what is left being LDS and L1 reads; 31^3 8.6 / 12.5.
template <int CH, int SRC, bool AHEAD>
__device__ __forceinline__ void cg_step1_body64(const Grid &g, int lb, int nb, const double *vals,
                                                const uint16_t *code, const double *kinv, const double *r,
                                                const double *p, double *pn, double *Ap, double *part1,
                                                const CgState *cur, CgState *nxt, double *seg /* LDS, kSegDoubles */) {
#pragma clang fp contract(off)
  __shared__ double lds[4];
  CgRegs c = cg_load(cur);
  const int row0 = lb * 256, row = row0 + threadIdx.x;
  const double *v = SRC == kMatTable ? vals + ((size_t)code[row / 3] * 3 + row % 3) * kSlots
                                     : vals + (size_t)(row >> 6) * kSlots * 64 + (row & 63);
  double vi[2][CH];
  if (!c.done)
#pragma unroll
    for (int k = 0; k < CH; ++k) vi[0][k] = load_value<SRC>(v, k);
  // AHEAD: the (at most two) entries of each plane's run that the thread
  // stages, loaded before the sums that beta waits for
  const int len = kSegNodes + 2 * g.nx, n_lo = row0 / 3, hi = g.nn - 1;
  double pre[AHEAD ? 18 : 1];
  if constexpr (AHEAD) {
    if (!c.done)
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const int e3 = min((int)threadIdx.x + (k & 1) * 256, 3 * len - 1);
        const int q = 3 * min(max(n_lo - 1 - g.nx + (k / 2 - 1) * g.nx * g.ny + e3 / 3, 0), hi) + e3 % 3;
        pre[k * 3] = kinv[q];
        pre[k * 3 + 1] = r[q];
        pre[k * 3 + 2] = p[q];
      }
  }
  if (!cg_enter(c, lb, nb, part1 + nb, nxt)) return;
  SegPitch pt{g.nx, len};
  if constexpr (AHEAD) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const int e3 = threadIdx.x + (k & 1) * 256;
      if (e3 < 3 * len) seg[(k / 2) * 3 * len + e3] = cg_dir(c, pre[k * 3], pre[k * 3 + 1], pre[k * 3 + 2]);
    }
    lds_barrier();
  } else {
    pt = stage_runs(g, row0, seg, [&](int q) { return cg_dir(c, kinv[q], r[q], p[q]); });
  }
  const double *own = seg + (row / 3 - row0 / 3 + 1 + pt.ly + pt.lz) * 3;
  // rows past the last node lie on its run's clamped end; p is zero there
  const double pv = row < g.nrow ? own[row % 3] : 0.0;
  const double acc = dot_runs<CH, SRC>(v, vi, own, pt);
  pn[row] = pv;
  Ap[row] = acc;
  double t[1] = {pv * acc};
  block_sum<1, 256>(t, lds);
  if (threadIdx.x == 0) part1[lb] = t[0];
}

// p = z + beta p and the state of the iteration alone, ahead of the SpMV of an
// uploaded matrix: its columns are read, so its gathers are not staged
__device__ __forceinline__ void cg_dir_body(int lb, int nb, const double *kinv, const double *r, const double *p,
                                            double *pn, const double *part2, const CgState *cur, CgState *nxt) {
  CgRegs c = cg_load(cur);
  if (!cg_enter(c, lb, nb, part2, nxt)) return;
  const int row = lb * 256 + threadIdx.x;
  pn[row] = cg_dir(c, kinv[row], r[row], p[row]);
}

__device__ __forceinline__ void cg_spmv_cols_body(int lb, const int *cols, const double *vals, const double *p,
                                                  double *Ap, double *part1, const CgState *cur) {
#pragma clang fp contract(off)
  __shared__ double lds[4];
  if (cur->done) return;
  const int row = lb * 256 + threadIdx.x;
  const double y = row_dot(cols, vals, p, row);
  Ap[row] = y;
  double t[1] = {p[row] * y};
  block_sum<1, 256>(t, lds);
  if (threadIdx.x == 0) part1[lb] = t[0];
}

// step2; its vectors are loaded before the sums that alpha waits for
__device__ __forceinline__ void cg_step2_body64(int lb, int nb, double *x, double *r, const double *p,
                                                const double *Ap, const double *kinv, double *part,
                                                const CgState *cur) {
#pragma clang fp contract(off)
  __shared__ double lds[4 * 2];
  if (cur->done) return;
  const int row = lb * 256 + threadIdx.x;
  const double xo = x[row], ro = r[row], po = p[row], ao = Ap[row], ko = kinv[row];
  double pap[1];
  seg_sum<1>(part, nb, pap);
  const double alpha = cur->rz / pap[0];
  x[row] = xo + alpha * po;
  const double rv = ro - alpha * ao;
  r[row] = rv;
  const double zv = ko * rv;
  double v[2] = {zv * zv, rv * zv};
  block_sum<2, 256>(v, lds);
  if (threadIdx.x == 0) {
    part[nb + (size_t)lb * 2 + 0] = v[0];
    part[nb + (size_t)lb * 2 + 1] = v[1];
  }
}

// one block: the sums of the last step2 queued into the state, in place
__device__ __forceinline__ void cg_tail_body(const double *part2, int nb, CgState *state) {
  CgRegs c = cg_load(state);
  if (c.done || c.fresh) return;
  cg_scalars(c, part2, nb);
  if (threadIdx.x == 0) cg_store(c, 1, state);
}

// Ap = A p and the partials of p.Ap of the FP32 inner CG (mixed-precision
// batch), p in memory; products of p and Ap are formed in FP64
template <int CH, int SRC>
__device__ __forceinline__ void cg_spmv_body32(const Grid &g, int lb, const float *vals, const float *p, float *Ap,
                                               double *part1, const CgState *cur) {
#pragma clang fp contract(off)
  __shared__ float seg[9 * kSegNodes * 3];
  __shared__ double lds[4];
  const int row0 = lb * 256, row = row0 + threadIdx.x;
  const float *v = vals + (size_t)(row >> 6) * kSlots * 64 + (row & 63);
  if (cur->done) return;
  float vi[2][CH];
#pragma unroll
  for (int k = 0; k < CH; ++k) vi[0][k] = load_value<SRC>(v, k);
  const SegPitch pt = stage_runs(g, row0, seg, [&](int q) { return p[q]; });
  const float *own = seg + (row / 3 - row0 / 3 + 1 + pt.ly + pt.lz) * 3;
  const float pv = row < g.nrow ? own[row % 3] : 0.0f;
  const float y = dot_runs<CH, SRC>(v, vi, own, pt);
  Ap[row] = y;
  double t[1] = {(double)pv * (double)y};
  block_sum<1, 256>(t, lds);
  if (threadIdx.x == 0) part1[lb] = t[0];
}

// ---------------------------------------------------------------------------
// Coarse-grid hats of the two-level preconditioners (mixed.hip k_c_*,
// batch.hip kb_c_*): trilinear hats of the interior nodes of a coarse grid
// with h fine elements per coarse element and side.
// ---------------------------------------------------------------------------

// hat of interior coarse node q (1 .. m) at fine index i along one side
__device__ __forceinline__ float hat(int i, int q, int h) {
  const int dd = abs(i - q * h);
  return dd < h ? 1.0f - (float)dd / (float)h : 0.0f;
}

// weights and interior coarse indices (0-based) of the two coarse nodes at
// and above fine index i along one side; a node outside 1 .. m gets weight 0
// and index 0 (a valid address)
__device__ __forceinline__ void hat_pair(int i, int h, int m, float (&w)[2], int (&q)[2]) {
  const int q0 = i / h;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int c = q0 + a;
    const bool in = c >= 1 && c <= m;
    w[a] = in ? hat(i, c, h) : 0.0f;
    q[a] = in ? c - 1 : 0;
  }
}

}  // namespace mpp
