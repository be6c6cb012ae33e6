// solver.hip -- FP64 ELL SpMV and Jacobi-preconditioned CG (gfx950).
//
// ell_mvp (src/ell.cpp:35-44): one thread per row of a SELL-64 slice.  The
// 81 slots are consumed in three chunks of 27: the chunk's columns and values
// are loaded first (non-temporal, they are streamed once), then the 27 x
// gathers, then the 27 products are added in slot order without contraction,
// so y is bit-identical to the reference SpMV while every wavefront keeps 27
// value/column loads in flight.  Bound: HBM bandwidth, 12 bytes per slot plus
// 16 bytes per row.
//
// ell_solve_cgpd (src/ell.cpp:66-122): the reference recurrence, one
// iteration = two kernels (kernels.hpp: step1 forms p and Ap, step2 x and r),
// or three for an uploaded matrix, where k_cg_dir forms p ahead of the SpMV.  No kernel uses
// atomics or fences: each block writes its partial, and every block of the
// next kernel re-sums all partials in the same fixed order, so every block
// holds identical scalars.  The parity is a kernel argument, so a run of
// iterations can be queued or captured in a graph ahead of time.
// Time per iteration (us) in two kernels, and as three (SpMV, x and r, p) with
// shuffled block sums: 6^3 nodes 8.7 / 14.1, 11^3 9.0 / 15.6, 21^3 9.9 /
// 16.2, 31^3 17.2 / 23.0, 41^3 33.0 / 37.8, 51^3 58.0 / 60.4.  Small RVEs wait
// for launches and block sums (kernels of about 5 and 3 us), 51^3 for 259 MB of
// values a pass (5.5 TB/s); with the stencil table of an all-elastic RVE 51^3
// takes 28.3, 31^3 12.7.
#include "kernels.hpp"

namespace mpp {

__global__ void __launch_bounds__(256) k_spmv(Grid g, const int *cols, const double *vals, const double *x, double *y) {
  const int row = blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= g.nrow_pad) return;
  const double acc = row_dot(cols, vals, x, row);
  if (row < g.nrow) y[row] = acc;
}

__global__ void __launch_bounds__(256) k_cg_init(Grid g, const double *vals, const double *b, double *x, double *r,
                                                 double *kinv, double *part) {
  cg_init_body(g, blockIdx.x, vals, b, x, r, kinv, part);
}

__global__ void __launch_bounds__(256) k_cg_init_state(const double *part, int nparts, double min_err,
                                                       double rel_err, int max_its, CgState *state) {
  cg_init_state_body(part, nparts, min_err, rel_err, max_its, state);
}

// Blocks are dispatched round-robin over the 8 XCDs: the 8 * per launched
// blocks give XCD x the row blocks [x * per, (x + 1) * per), so each XCD's
// L2 holds a contiguous slab of the gathered vector (2-5% faster SpMV).
template <int SRC, bool AHEAD>
__global__ void __launch_bounds__(256) k_cg_step1(Grid g, int nb, int per, const double *vals, const uint16_t *code,
                                                  const double *kinv, const double *r, const double *p, double *pn,
                                                  double *Ap, double *part, const CgState *cur, CgState *nxt) {
  const int lb = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (lb >= nb) return;
  __shared__ double seg[kSegDoubles];
  cg_step1_body64<kChunk, SRC, AHEAD>(g, lb, nb, vals, code, kinv, r, p, pn, Ap, part, cur, nxt, seg);
}

// step1 on the stencil table with a thread per node: the three rows share the
// staged values, and a wave whose interior nodes have one code (most of them,
// away from phase interfaces) takes the 243 values as scalars.  Blocks of 256
// nodes, three row blocks each, whose partials are those of k_cg_step1: the
// same rows in the same tree.
constexpr int kNodeBlock = 256;
// Row blocks from which it runs: fewer than two node blocks a CU leave its nine
// lines of scalar loads, one after the other, in the open.  Iteration, us, by
// node / by row: 31^3 nodes (350 row blocks) 15.7 / 13.4, 41^3 (808) 23.1 /
// 21.3, 46^3 (1141) 24.9 / 28.1, 51^3 (1555) 28.3 / 33.7.  Lines of more than
// 256 nodes would need more LDS than a launch has by default.
constexpr int kNodeRowBlocks = 1100, kNodeMaxLine = 256;
__global__ void __launch_bounds__(kNodeBlock) k_cg_step1_node(Grid g, int nb, int nblocks, int per,
                                                              const double *__restrict__ tab,
                                                              const uint16_t *__restrict__ code, const double *kinv,
                                                              const double *r, const double *p, double *pn, double *Ap,
                                                              double *part1, const CgState *cur, CgState *nxt) {
#pragma clang fp contract(off)
  extern __shared__ double seg[];  // three runs of nodes, one per dz; then the products
  const int lb = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (lb >= nblocks) return;
  CgRegs c = cg_load(cur);
  const int n0 = lb * kNodeBlock, n = n0 + threadIdx.x;
  const int own_code = code[min(n, g.nrow_pad / 3)];
  if (!cg_enter(c, lb, nb, part1 + nb, nxt)) return;
  const int len = kNodeBlock + 2 + 2 * g.nx, nxny = g.nx * g.ny, hi = g.nn - 1;
  for (int dz = -1; dz <= 1; ++dz)
#pragma unroll 2
    for (int e3 = threadIdx.x; e3 < 3 * len; e3 += kNodeBlock) {
      const int q = 3 * min(max(n0 - 1 - g.nx + dz * nxny + e3 / 3, 0), hi) + e3 % 3;
      seg[(dz + 1) * 3 * len + e3] = cg_dir(c, kinv[q], r[q], p[q]);
    }
  lds_barrier();
  const double *own = seg + (threadIdx.x + 1 + g.nx + len) * 3;
  const bool row = own_code < kStencilCodes - 2, node = n < g.nn;
  double acc[3] = {0.0, 0.0, 0.0};
  const unsigned long long rows = __ballot(row);
  const int first = rows ? __ffsll(rows) - 1 : 0;
  const int wave_code = __builtin_amdgcn_readlane(own_code, first);
  // line m of the stencil's nine: 3 neighbours x 3 values for each of the rows
  const auto line = [&](const auto *t, int m) {
    const double *x = own + ((m / 3 - 1) * len + (m % 3 - 1) * g.nx - 1) * 3;
#pragma unroll
    for (int k = 0; k < 9; ++k)
#pragma unroll
      for (int fi = 0; fi < 3; ++fi) acc[fi] += t[fi * kSlots + m * 9 + k] * x[k];
  };
  if (__ballot(row && own_code != wave_code) == 0) {
    // the constant address space makes these scalar loads
    typedef const __attribute__((address_space(4))) double *Scalars;
    const Scalars t = (Scalars)(uintptr_t)(tab + (size_t)wave_code * 3 * kSlots);
#pragma unroll 1
    for (int m = 0; m < 9; ++m) line(t, m);
  } else {
    const double *t = tab + (size_t)own_code * 3 * kSlots;
#pragma unroll 1
    for (int m = 0; m < 9; ++m) line(t, m);
  }
  double pv[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    pv[d] = node ? own[d] : 0.0;
    if (!row) acc[d] = node ? 0.0 + pv[d] : 0.0;  // a Dirichlet row's only value is its 1.0
  }
  lds_barrier();
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int q = 3 * n + d;
    if (q < g.nrow_pad) {
      pn[q] = pv[d];
      Ap[q] = acc[d];
    }
    seg[threadIdx.x * 3 + d] = pv[d] * acc[d];
  }
  lds_barrier();
  __shared__ double lds[4 * 3];
  double t[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) t[k] = seg[k * 256 + threadIdx.x];
  block_sum<3, 256>(t, lds);
  if (threadIdx.x < 3 && lb * 3 + (int)threadIdx.x < nb) part1[lb * 3 + threadIdx.x] = t[threadIdx.x];
}

// code[n]: sum over the elements q = (a*2+b)*2+c around interior node n of
// phase * 3^q; the last two for a boundary node and a padding node
__global__ void __launch_bounds__(256) k_s_code(Grid g, int n, const int *et, uint16_t *code) {
  const int node = blockIdx.x * 256 + threadIdx.x;
  if (node >= n) return;
  const int i = node % g.nx, j = (node / g.nx) % g.ny, k = node / (g.nx * g.ny);
  int c = kStencilCodes - 1;
  if (node < g.nn) {
    c = kStencilCodes - 2;
    if (!on_boundary(g, i, j, k)) {
      c = 0;
      for (int q = 7; q >= 0; --q)
        c = 3 * c + et[((k - 1 + (q & 1)) * g.ney + j - 1 + ((q >> 1) & 1)) * g.nex + i - 1 + (q >> 2)];
    }
  }
  code[node] = (uint16_t)c;
}

// one block per code, a thread per value: the sums of gather_vals_slice
__global__ void __launch_bounds__(256) k_s_table(const double *ke, double *tab) {
#pragma clang fp contract(off)
  const int code = blockIdx.x, t = threadIdx.x;
  if (t >= 3 * kSlots) return;
  const int fi = t / kSlots, slot = t % kSlots, n = slot / 3, fj = slot % 3;
  double acc = 0.0;
  if (code == kStencilCodes - 2) {
    acc = slot == 13 * 3 + fi ? 1.0 : 0.0;
  } else if (code < kStencilCodes - 2) {
    int rest = code;
    for (int q = 0; q < 8; ++q, rest /= 3) {
      const int a = q >> 2, b = (q >> 1) & 1, c = q & 1;
      const int px = n % 3 - a, py = (n / 3) % 3 - b, pz = n / 9 - c;  // neighbour n in element q
      if (px < 0 || px > 1 || py < 0 || py > 1 || pz < 0 || pz > 1) continue;
      acc += ke[(rest % 3) * 576 + (local_node(1 - a, 1 - b, 1 - c) * 3 + fi) * 24 + local_node(px, py, pz) * 3 + fj];
    }
  }
  tab[(size_t)code * 3 * kSlots + t] = acc;
}

__global__ void __launch_bounds__(256) k_cg_dir(const double *kinv, const double *r, const double *p, double *pn,
                                                const double *part2, const CgState *cur, CgState *nxt) {
  cg_dir_body(blockIdx.x, gridDim.x, kinv, r, p, pn, part2, cur, nxt);
}

__global__ void __launch_bounds__(256) k_cg_spmv_cols(int nb, int per, const int *cols, const double *vals,
                                                      const double *p, double *Ap, double *part1,
                                                      const CgState *cur) {
  const int lb = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (lb >= nb) return;
  cg_spmv_cols_body(lb, cols, vals, p, Ap, part1, cur);
}

__global__ void __launch_bounds__(256) k_cg_step2(double *x, double *r, const double *p, const double *Ap,
                                                  const double *kinv, double *part, const CgState *cur) {
  cg_step2_body64(blockIdx.x, gridDim.x, x, r, p, Ap, kinv, part, cur);
}

__global__ void __launch_bounds__(256) k_cg_tail(const double *part2, int nb, CgState *state) {
  cg_tail_body(part2, nb, state);
}

__global__ void k_axpy(int n, double a, const double *x, double *y) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] += a * x[i];
}

__global__ void k_copy(int n, const double *x, double *y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i];
}

static unsigned nblk(size_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

hipError_t launch_spmv(const Grid &g, const int *cols, const double *vals, const double *x, double *y,
                       hipStream_t st) {
  hipLaunchKernelGGL(k_spmv, dim3(nblk(g.nrow_pad, 256)), dim3(256), 0, st, g, cols, vals, x, y);
  return hipGetLastError();
}

hipError_t launch_cg_init(const Grid &g, const double *vals, const double *b, const CgVecs &w, double min_err,
                          double rel_err, int max_its, hipStream_t st) {
  const unsigned nb = nblk(g.nrow_pad, 256);
  hipLaunchKernelGGL(k_cg_init, dim3(nb), dim3(256), 0, st, g, vals, b, w.x, w.r, w.kinv, w.part);
  hipLaunchKernelGGL(k_cg_init_state, dim3(1), dim3(256), 0, st, w.part, (int)nb, min_err, rel_err, max_its, w.state);
  return hipGetLastError();
}

hipError_t launch_stencil64(const Grid &g, const int *et, const double *ke, const Stencil64 &s, hipStream_t st) {
  const int n = g.nrow_pad / 3 + 1;
  hipLaunchKernelGGL(k_s_code, dim3(nblk(n, 256)), dim3(256), 0, st, g, n, et, s.code);
  hipLaunchKernelGGL(k_s_table, dim3(kStencilCodes), dim3(256), 0, st, ke, s.tab);
  return hipGetLastError();
}

hipError_t launch_cg_step1(const Grid &g, const int *cols, const double *vals, const Stencil64 *dict, const CgVecs &w,
                           int parity, hipStream_t st, bool dir) {
  const int nb = (int)nblk(g.nrow_pad, 256), per = (nb + 7) / 8, k = parity & 1;
  CgState *cur = w.state + k, *nxt = w.state + (k ^ 1);
  if (cols) {
    if (dir)
      hipLaunchKernelGGL(k_cg_dir, dim3(nb), dim3(256), 0, st, w.kinv, w.r, w.p[k], w.p[k ^ 1], w.part + nb, cur, nxt);
    hipLaunchKernelGGL(k_cg_spmv_cols, dim3(8 * per), dim3(256), 0, st, nb, per, cols, vals, w.p[k ^ 1], w.Ap, w.part,
                       nxt);
  } else if (dict && nb >= kNodeRowBlocks && g.nx <= kNodeMaxLine) {
    const int nn = (nb + 2) / 3, pern = (nn + 7) / 8;
    const size_t lds = (size_t)3 * 3 * (kNodeBlock + 2 + 2 * g.nx) * sizeof(double);
    hipLaunchKernelGGL(k_cg_step1_node, dim3(8 * pern), dim3(kNodeBlock), lds, st, g, nb, nn, pern, dict->tab,
                       dict->code, w.kinv, w.r, w.p[k], w.p[k ^ 1], w.Ap, w.part, cur, nxt);
  } else {
    const int src = dict ? kMatTable : mat_source((double)g.nrow_pad * kSlots * sizeof(double));
    const bool ahead = cg_ahead(nb, g.nx);
    const auto step1 = src == kMatTable    ? (ahead ? k_cg_step1<kMatTable, true> : k_cg_step1<kMatTable, false>)
                       : src == kMatCached ? (ahead ? k_cg_step1<kMatCached, true> : k_cg_step1<kMatCached, false>)
                                           : k_cg_step1<kMatStream, false>;
    hipLaunchKernelGGL(step1, dim3(8 * per), dim3(256), 0, st, g, nb, per, dict ? dict->tab : vals,
                       dict ? dict->code : nullptr, w.kinv, w.r, w.p[k], w.p[k ^ 1], w.Ap, w.part, cur, nxt);
  }
  return hipGetLastError();
}

hipError_t launch_cg_iter(const Grid &g, const int *cols, const double *vals, const Stencil64 *dict, const CgVecs &w,
                          int parity, hipStream_t st) {
  const hipError_t e = launch_cg_step1(g, cols, vals, dict, w, parity, st);
  if (e != hipSuccess) return e;
  const int n = (parity & 1) ^ 1;
  hipLaunchKernelGGL(k_cg_step2, dim3(nblk(g.nrow_pad, 256)), dim3(256), 0, st, w.x, w.r, w.p[n], w.Ap, w.kinv, w.part,
                     w.state + n);
  return hipGetLastError();
}

hipError_t launch_cg_tail(const Grid &g, const CgVecs &w, int queued, hipStream_t st) {
  const unsigned nb = nblk(g.nrow_pad, 256);
  hipLaunchKernelGGL(k_cg_tail, dim3(1), dim3(256), 0, st, w.part + nb, (int)nb, w.state + (queued & 1));
  return hipGetLastError();
}

hipError_t launch_axpy(int n, double a, const double *x, double *y, hipStream_t st) {
  hipLaunchKernelGGL(k_axpy, dim3(nblk(n, 256)), dim3(256), 0, st, n, a, x, y);
  return hipGetLastError();
}

hipError_t launch_copy(int n, const double *x, double *y, hipStream_t st) {
  hipLaunchKernelGGL(k_copy, dim3(nblk(n, 256)), dim3(256), 0, st, n, x, y);
  return hipGetLastError();
}

}  // namespace mpp
