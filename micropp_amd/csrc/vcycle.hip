// vcycle.hip -- the FP32 operator of an all-elastic RVE as a stencil
// dictionary.
//
// With one element stiffness per phase, the 27 neighbour blocks of an interior
// node depend only on the phases of its eight elements: 3^8 = 6561 possible
// stencils (2^8 with two phases), whatever the grid.  The matrix is therefore
// not stored per node (1008 B a node) but as a table of stencils
// (tab[code * 252 + mslot(nb, fi, fj)], 6.6 MB of which an RVE touches a few
// hundred KB at most) and a 16-bit code per node; kNoRow marks the nodes
// without a row (boundary, padding).  Rows and columns of Dirichlet nodes need
// no zeros: the CG vectors are zero there.  The table entries are the FP64
// sums of the element blocks in the reference element order, rounded once.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "mixed.hpp"

namespace mpp {

constexpr int kStencilFloats = kNodeQuads * 4;  // 252
constexpr int kNumStencils = 6561;              // 3^8
constexpr unsigned kNoRow = 0xffffu;

// code[n] = sum over the elements q = (a*2+b)*2+c around interior node n of
// phase * 3^q
__global__ void __launch_bounds__(256) k_d_code(Grid g, int NP, const int *et, uint16_t *code) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= NP) return;
  unsigned c = kNoRow;
  if (n < g.nn) {
    const int i = n % g.nx, j = (n / g.nx) % g.ny, k = n / (g.nx * g.ny);
    if (!node_on_boundary(g, i, j, k)) {
      c = 0;
      unsigned w = 1;
      for (int q = 0; q < 8; ++q, w *= 3) {
        const int ex = i - 1 + (q >> 2), ey = j - 1 + ((q >> 1) & 1), ez = k - 1 + (q & 1);
        c += w * (unsigned)et[(ez * g.ney + ey) * g.nex + ex];
      }
    }
  }
  code[n] = (uint16_t)c;
}

// one block per stencil, one thread per float of it (row pads are zero)
__global__ void __launch_bounds__(256) k_d_table(const double *ke, float *tab) {
  const int code = blockIdx.x, t = threadIdx.x;
  if (t >= kStencilFloats) return;
  const int row = t / 28, rem = t % 28;
  double acc = 0.0;
  if (rem < 27) {
    const int dz = row / 3 - 1, dy = row % 3 - 1, dx = rem / 9 - 1, fi = (rem % 9) / 3, fj = rem % 3;
    int rest = code;
    for (int q = 0; q < 8; ++q, rest /= 3) {
      const int a = q >> 2, b = (q >> 1) & 1, c = q & 1;
      const int px = 1 - a + dx, py = 1 - b + dy, pz = 1 - c + dz;
      if (px < 0 || px > 1 || py < 0 || py > 1 || pz < 0 || pz > 1) continue;
      acc += ke[(rest % 3) * 576 + (local_node(1 - a, 1 - b, 1 - c) * 3 + fi) * 24 + local_node(px, py, pz) * 3 + fj];
    }
  }
  tab[(size_t)code * kStencilFloats + t] = (float)acc;
}

// A node whose eight elements share one phase ("homogeneous") has code
// kHomStep * phase; the others with a row are interface nodes.
constexpr unsigned kHomStep = (kNumStencils - 1) / 2;  // 1 + 3 + ... + 3^7
__device__ __forceinline__ bool is_hom(unsigned c) { return c == 0 || c == kHomStep || c == 2 * kHomStep; }

// The stencil of a homogeneous node: an isotropic phase on box-shaped cells is
// symmetric under reflection of each axis, so the diagonal entries are even in
// dx, dy and dz and entry (x, y) is odd in dx and dy and even in dz (likewise
// (x, z) and (y, z)): 30 numbers instead of 243.  hom[phase * 32 + ...]: a * 8 +
// |dx| + 2 |dy| + 4 |dz| entry (a, a); 24 + |dz|, 26 + |dy|, 28 + |dx| entries
// (x, y), (x, z), (y, z) at the positive offsets.
constexpr int kHomFloats = 32;
__global__ void __launch_bounds__(128) k_d_hom(const float *tab, float *hom) {
  const int ph = threadIdx.x / kHomFloats, t = threadIdx.x % kHomFloats;
  if (ph >= 3) return;
  int dx = 0, dy = 0, dz = 0, fi = 0, fj = 0;
  if (t < 24) {
    fi = fj = t / 8;
    dx = t & 1, dy = (t >> 1) & 1, dz = (t >> 2) & 1;
  } else if (t < 26) {
    dx = dy = 1, dz = t - 24, fj = 1;
  } else if (t < 28) {
    dx = dz = 1, dy = t - 26, fj = 2;
  } else if (t < 30) {
    dy = dz = 1, dx = t - 28, fi = 1, fj = 2;
  }
  const int nb = (dz + 1) * 9 + (dy + 1) * 3 + dx + 1;
  hom[threadIdx.x] = t < 30 ? tab[(size_t)ph * kHomStep * kStencilFloats + mslot(nb, fi, fj)] : 0.0f;
}

// The interface nodes in ascending order (list) and their number: per block of
// 256 nodes its count (k_d_count), the exclusive sums (k_d_scan: one block;
// cnt[nb] = the total), then the nodes (k_d_list).
__global__ void __launch_bounds__(256) k_d_count(const uint16_t *code, int *cnt) {
  __shared__ int w4[4];
  const unsigned c = code[blockIdx.x * 256 + threadIdx.x];
  const unsigned long long m = __ballot(c != kNoRow && !is_hom(c));
  if ((threadIdx.x & 63) == 0) w4[threadIdx.x >> 6] = __popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) cnt[blockIdx.x] = w4[0] + w4[1] + w4[2] + w4[3];
}
__global__ void __launch_bounds__(256) k_d_scan(int nb, int *cnt) {
  __shared__ int s[256];
  const int per = (nb + 255) / 256, i0 = threadIdx.x * per;
  int t = 0;
  for (int i = i0; i < min(i0 + per, nb); ++i) t += cnt[i];
  s[threadIdx.x] = t;
  __syncthreads();
  int base = 0;
  for (int i = 0; i < (int)threadIdx.x; ++i) base += s[i];
  for (int i = i0; i < min(i0 + per, nb); ++i) {
    const int v = cnt[i];
    cnt[i] = base;
    base += v;
  }
  if (threadIdx.x == 255) cnt[nb] = base;
}
__global__ void __launch_bounds__(256) k_d_list(const uint16_t *code, const int *cnt, int *list) {
  __shared__ int w4[4];
  const int n = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned c = code[n];
  const bool on = c != kNoRow && !is_hom(c);
  const unsigned long long m = __ballot(on);
  if (lane == 0) w4[w] = __popcll(m);
  __syncthreads();
  int at = cnt[blockIdx.x];
  for (int i = 0; i < w; ++i) at += w4[i];
  if (on) list[at + __popcll(m & ((1ull << lane) - 1))] = n;
}

// ---------------------------------------------------------------------------
// y = A p of one field group (4 fields).
//
// hom_apply: at the homogeneous nodes of one phase among 62 consecutive nodes,
// by one wave.  Lane l holds node n = n0 - 1 + l: lanes 1 .. 62 own an output,
// lanes 0 and 63 only contribute to their neighbours.  A lane loads p on the 9
// stencil rows (dy, dz) at dx = 0 alone, one direction at a time, and forms the
// sums and differences over dy and dz that the symmetries leave (31 additions
// a field for the three directions); with 36 multiply-adds these give its own
// node's term C and what the node left and right of it takes: S + D to the left
// (this node is its dx = +1 neighbour), S - D to the right, moved one lane over
// at the end.  79 vector instructions a field instead of 243 FMAs.  The
// coefficients are scalar loads.  A wave holding homogeneous nodes of several
// phases runs once per phase (neighbouring homogeneous nodes share four
// elements, so the side terms always meet a node of the phase they are formed
// for); interface nodes are left to iface_apply.
//
// iface_apply: at one interface node per lane, with the lane's own stencil and
// gathered neighbours.
//
// Addresses are clamped into [0, NP); every neighbour of a node with a row lies
// in the grid, and the results of the other lanes are not used.
//
// Bound: a wave is 27 loads of 1 KB and about 480 vector instructions, so the
// loads (three waves a SIMD, nine in flight each) and the 38 MB of P and A P
// weigh as much as the arithmetic.  50^3, 12 fields: 17.2 us with 8 spheres, 14.0
// us with one phase, against 24.9 and 19.9 us with all 243 coefficients (scalar
// loads where a run had one stencil, per lane elsewhere) and 31.8 us for the
// matrix stored (1008 B a node); 4 fields 9.9 us, 14.5 and 25.1 us.
// ---------------------------------------------------------------------------
constexpr int kApNodes = 62;  // outputs per wave
constexpr int kApWaves = 4;   // waves per block (consecutive runs of nodes, one field group)
constexpr int kIfaceNodes = 64;  // interface nodes per block

typedef const __attribute__((address_space(4))) float *const_f32;

__device__ __forceinline__ void fma4(float4 &y, float a, const float4 &x) {
  y.x += a * x.x;
  y.y += a * x.y;
  y.z += a * x.z;
  y.w += a * x.w;
}
__device__ __forceinline__ float4 add4(const float4 &a, const float4 &b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
__device__ __forceinline__ float4 sub4(const float4 &a, const float4 &b) {
  return make_float4(a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w);
}

// lane i takes lane i - 1's value (0x138) or lane i + 1's (0x130); the end
// lane without a source takes 0
template <int CTRL>
__device__ __forceinline__ float4 lane_shift(const float4 &v) {
  auto f = [](float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
  };
  return make_float4(f(v.x), f(v.y), f(v.z), f(v.w));
}

// byte offsets of node n's neighbours at dx = 0 on the 9 stencil rows
// ((dz + 1) * 3 + dy + 1) in one direction of a vector: 32 bits, so that a load
// is a scalar base and one register of offset
__device__ __forceinline__ void row_offsets(const Grid &g, int NP, int n, unsigned (&o)[9]) {
  const int nxny = g.nx * g.ny;
#pragma unroll
  for (int w = 0; w < 9; ++w) o[w] = 16u * (unsigned)min(max(n + (w / 3 - 1) * nxny + (w % 3 - 1) * g.nx, 0), NP - 1);
}
__device__ __forceinline__ void load_rows(const float4 *pd, const unsigned (&o)[9], float4 (&r)[9]) {
#pragma unroll
  for (int w = 0; w < 9; ++w) {
    // (opaque: the 64-bit addresses would otherwise be formed ahead and held in registers)
    unsigned t = o[w];
    asm volatile("" : "+v"(t));
    r[w] = *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(pd) + t);
  }
}

// q: direction 0's rows, already loaded (left with direction 2's)
template <int KG>
__device__ __forceinline__ void hom_apply(int NP, const unsigned (&o)[9], const float *hom, const float4 *pg,
                                          float4 (&q)[9], float4 (&y)[3]) {
  const const_f32 h = (const_f32)(uintptr_t)hom;
  float4 C[3], S[3], D[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) C[a] = S[a] = D[a] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    // q[(dz + 1) * 3 + dy + 1]: over dy = +-1 at dz = +1 and -1, then over dz
    const float4 sp = add4(q[8], q[6]), dp = sub4(q[8], q[6]), sm = add4(q[2], q[0]), dm = sub4(q[2], q[0]);
    const float4 e00 = q[4], e10 = add4(q[5], q[3]), e01 = add4(q[7], q[1]), e11 = add4(sp, sm);
    const float4 o10 = sub4(q[5], q[3]), o11 = add4(dp, dm);                      // odd in dy
    const float4 z01 = sub4(q[7], q[1]), z11 = sub4(sp, sm), yz = sub4(dp, dm);  // odd in dz; in both
    fma4(C[f], h[f * 8 + 0], e00);  // own entry (f, f)
    fma4(S[f], h[f * 8 + 1], e00);
    fma4(C[f], h[f * 8 + 2], e10);
    fma4(S[f], h[f * 8 + 3], e10);
    fma4(C[f], h[f * 8 + 4], e01);
    fma4(S[f], h[f * 8 + 5], e01);
    fma4(C[f], h[f * 8 + 6], e11);
    fma4(S[f], h[f * 8 + 7], e11);
    if (f < 2) {  // entries (x, y): odd in dx and dy
      fma4(D[1 - f], h[24], o10);
      fma4(D[1 - f], h[25], o11);
    }
    if (f != 1) {  // entries (x, z): odd in dx and dz
      fma4(D[2 - f], h[26], z01);
      fma4(D[2 - f], h[27], z11);
    }
    if (f > 0) {  // entries (y, z): odd in dy and dz
      fma4(C[3 - f], h[28], yz);
      fma4(S[3 - f], h[29], yz);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (f < 2) load_rows(pg + (size_t)(f + 1) * KG * NP, o, q);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int a = 0; a < 3; ++a)
    y[a] = add4(C[a], add4(lane_shift<0x138>(sub4(S[a], D[a])), lane_shift<0x130>(add4(S[a], D[a]))));
}

// the rows of plane dz only
template <int KG>
__device__ __forceinline__ void iface_apply(const Grid &g, int NP, int n, int dz, unsigned c, const float *tab,
                                            const float4 *pg, float4 (&y)[3]) {
  const float4 *tc = reinterpret_cast<const float4 *>(tab) + c * (unsigned)kNodeQuads + (dz + 1) * 21;
#pragma unroll
  for (int d = 0; d < 3; ++d) y[d] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
  for (int w = 0; w < 3; ++w) {
    const int m = n + (dz * g.ny + w - 1) * g.nx;
    float4 q[7], p[9];
#pragma unroll
    for (int u = 0; u < 7; ++u) q[u] = tc[w * 7 + u];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int fj = 0; fj < 3; ++fj) p[j * 3 + fj] = pg[(size_t)fj * KG * NP + m + j - 1];
    __builtin_amdgcn_sched_barrier(0);
    float a[28];
#pragma unroll
    for (int u = 0; u < 7; ++u) {
      a[u * 4] = q[u].x;
      a[u * 4 + 1] = q[u].y;
      a[u * 4 + 2] = q[u].z;
      a[u * 4 + 3] = q[u].w;
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int fj = 0; fj < 3; ++fj)
#pragma unroll
        for (int fi = 0; fi < 3; ++fi) fma4(y[fi], a[j * 9 + fi * 3 + fj], p[j * 3 + fj]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// k_d_apply: the operator with an epilogue (ApplyMode, mixed.hpp) for every
// field: kApplyCg OUT = A P and the partials of (P, A P); kApplyRes OUT = R -
// omega A P; kApplyPost OUT = P + omega kinv (R - A P) and the partials of (R,
// OUT); kApplyPow OUT = kinv A P and the partials of (OUT, D OUT).  Partials
// part[field * nblk + block].  Grid (8 peri + 8 per, K/4), nblk = nbi + nbm
// blocks that do work, field group blockIdx.y: first the nbi blocks of
// kIfaceNodes interface nodes each (they start first: most loads to wait for;
// waves 0 .. 2 take a plane dz each, added in LDS in order), then the nbm blocks
// of kApWaves runs of kApNodes nodes (XCD-aware run order).
template <int K, int MODE>
__global__ void __launch_bounds__(256, 3) k_d_apply(Grid g, int NP, int nbi, int peri, int nbm, int per, int nif,
                                                    const uint16_t *code, const int *list, const float *tab,
                                                    const float *hom, const float4 *P, const float4 *R,
                                                    const float *kinv, float omega, float4 *OUT, double *part,
                                                    const MState *cur) {
  constexpr int KG = K / 4;
  __shared__ double lds[kApWaves][4];
  __shared__ float4 lp[2][3][kIfaceNodes];
  const int grp = blockIdx.y, r0 = grp * 4;
  const bool iface = (int)blockIdx.x < 8 * peri;  // whole block
  const int bx = (int)blockIdx.x - (iface ? 0 : 8 * peri);
  const int lb = (bx & 7) * (iface ? peri : per) + (bx >> 3);
  if (lb >= (iface ? nbi : nbm)) return;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const float4 *pg = P + (size_t)grp * NP;
  float4 y[3];
  int n;
  bool out;
  if (iface) {
    const int i = lb * kIfaceNodes + lane;
    n = list[min(i, nif - 1)];
    const unsigned c = code[n];
    if (MODE != kApplyPow && group_stopped(cur, r0)) return;  // whole block
    out = wv == 0 && i < nif;
    if (wv < 3) iface_apply<KG>(g, NP, n, wv - 1, c, tab, pg, y);
    if (wv == 1 || wv == 2)
#pragma unroll
      for (int d = 0; d < 3; ++d) lp[wv - 1][d][lane] = y[d];
    __syncthreads();
    if (wv == 0)
#pragma unroll
      for (int d = 0; d < 3; ++d) y[d] = add4(add4(y[d], lp[0][d][lane]), lp[1][d][lane]);
  } else {
    n = (lb * kApWaves + wv) * kApNodes - 1 + lane;
    const bool in = n >= 0 && n < NP;
    const unsigned c = in ? (unsigned)code[n] : kNoRow;
    unsigned o[9];
    row_offsets(g, NP, n, o);
    float4 rows[9];
    load_rows(pg, o, rows);
    __builtin_amdgcn_sched_barrier(0);  // (in flight while the codes and the state arrive)
    if (MODE != kApplyPow && group_stopped(cur, r0)) return;  // whole block
#pragma unroll
    for (int d = 0; d < 3; ++d) y[d] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    out = in && lane >= 1 && lane <= kApNodes && (c == kNoRow || is_hom(c));
    bool loaded = true;
#pragma unroll 1
    for (int ph = 0; ph < 3; ++ph) {
      const bool mine = c == kHomStep * ph;
      if (__ballot(mine) == 0) continue;
      if (!loaded) load_rows(pg, o, rows);
      loaded = false;
      float4 v[3];
      hom_apply<KG>(NP, o, hom + ph * kHomFloats, pg, rows, v);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        // (pinned: the compiler would otherwise move the multiply-adds under the
        // selection, with all their inputs held until then)
        asm volatile("" : "+v"(v[d].x), "+v"(v[d].y), "+v"(v[d].z), "+v"(v[d].w));
        y[d].x = mine ? v[d].x : y[d].x;
        y[d].y = mine ? v[d].y : y[d].y;
        y[d].z = mine ? v[d].z : y[d].z;
        y[d].w = mine ? v[d].w : y[d].w;
      }
    }
  }
  double s4[4] = {0, 0, 0, 0};
  if (out) {
#pragma unroll
    for (int d = 0; d < 3; ++d)
      apply_out<MODE>(pg[(size_t)d * KG * NP + n], y[d], R, kinv, omega, OUT, (size_t)(d * KG + grp) * NP + n,
                      (size_t)d * NP + n, s4);
  }
  if constexpr (MODE == kApplyRes) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const double s = wave_sum_dpp(s4[r]);
    if (lane == 0) lds[wv][r] = s;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kApWaves; ++w) s += lds[w][threadIdx.x];
    part[(size_t)(r0 + threadIdx.x) * (nbi + nbm) + (iface ? 0 : nbi) + lb] = s;
  }
}

// ---------------------------------------------------------------------------
// Multilevel preconditioner OUT = M R of the inner CG: a V-cycle with one
// damped Jacobi step before and after each coarse correction,
//   Z0 = w0 D^-1 R,  e = M1 P1^T (R - A Z0),  Z1 = Z0 + P1 e,
//   OUT = Z1 + w0 D^-1 (R - A Z1),
// P1 the trilinear interpolation from the grid of twice the spacing (an odd
// side's last element is 1 wide, so every side of at least 4 elements has one).  M1 is the
// same cycle on that grid (small RVEs, vcycle_setup: P1 the coarse hats and M1
// the dense inverse, nothing in between) with its Galerkin operator A1 = P1^T A P1 and the
// dense inverse of the coarse Galerkin matrix as its correction (P2: the coarse
// hats at the second level's nodes; at high contrasts these include the coarse
// ones, coarse_grid_cycle).  M is symmetric positive definite while w0 and w1 stay
// below 2 / lambda_max(D^-1 A) of their levels (estimated at set-up by a power
// iteration on the operators themselves, since isolated stiff elements raise
// it: 2.7-2.9 for cubes, up to 4.5 in thin cells and beside one stiff element).
//
// 50^3, contrast 10, 12 fields: 22 iterations to 1e-8 against 73 with the
// additive two-level form (Jacobi plus the same coarse inverse; one operator
// application an iteration instead of three), 160 us an iteration against 85:
// sigma and ctan of six strains to 1e-10 in 4.8 ms against 7.5 ms.  Sides
// without a common divisor (29 x 37 x 23 elements) had no coarse level before:
// 33 iterations against 250, 2.3 ms against 5.9 ms.
// ---------------------------------------------------------------------------
// a hat's weight at an index with entry h, the hat's node at offset o
__device__ __forceinline__ float hat_weight(const HatEntry &h, int o) {
  return (h.q0 == o ? h.w0 : 0.0f) + (h.q1 == o ? h.w1 : 0.0f);
}
struct Hats {  // along x, y and z (VCycleDev)
  const HatEntry *x, *y, *z;
  const int *past[3], *upto[3];
};

// R1 = P1^T T and E0 = D1^-1 R1.  One thread per second-level node (boundary
// ones write zero) and component c = d KG + grp.
template <int K>
__global__ void __launch_bounds__(256) k_v_restrict(Grid g, Grid g1, int NP, int NP1, const float4 *T,
                                                    const float *kinv1, float4 *R1, float4 *E0, const MState *cur) {
  constexpr int KG = K / 4;
  const int c = blockIdx.y, d = c / KG, grp = c % KG;
  const int n1 = blockIdx.x * 256 + threadIdx.x;
  if (n1 >= NP1) return;
  const float w = kinv1[(size_t)d * NP1 + n1];
  if (group_stopped(cur, grp * 4)) return;
  const int q = n1 % g1.nx, r = (n1 / g1.nx) % g1.ny, s = n1 / (g1.nx * g1.ny);
  float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (n1 < g1.nn && !node_on_boundary(g1, q, r, s)) {
    const float4 *t = T + (size_t)c * NP + ((size_t)(2 * s) * g.ny + 2 * r) * g.nx + 2 * q;
#pragma unroll
    for (int z = -1; z <= 1; ++z)
#pragma unroll
      for (int y = -1; y <= 1; ++y)
#pragma unroll
        for (int x = -1; x <= 1; ++x)
          fma4(acc, (x ? 0.5f : 1.0f) * (y ? 0.5f : 1.0f) * (z ? 0.5f : 1.0f), t[((ptrdiff_t)z * g.ny + y) * g.nx + x]);
  }
  R1[(size_t)c * NP1 + n1] = acc;
  E0[(size_t)c * NP1 + n1] = make_float4(w * acc.x, w * acc.y, w * acc.z, w * acc.w);
}

// k_v_mid: the second level's operator with an epilogue (ApplyMode).  Block:
// one run of kApNodes nodes (lanes as in hom_apply), a wave per stencil plane
// dz and field group, all 30 loads of a wave in flight together (the grid has
// few blocks: a launch is a few memory latencies long, not bytes); the groups'
// waves read the same coefficients at about the same time, from L1 after the
// first.  The planes are added in LDS in order.  kApplyPow: one group (grid's
// block of 192 threads), partials part[field * gridDim.x + block].
template <int K, int MODE>
__global__ void __launch_bounds__(MODE == kApplyPow ? 192 : 48 * K)
    k_v_mid(Grid g1, int NP1, const float4 *A1, const float4 *P, const float4 *R, const float *kinv, float omega,
            float4 *OUT, double *part, const MState *cur) {
  constexpr int KG = K / 4, NG = MODE == kApplyPow ? 1 : KG;
  __shared__ float4 lds[2][NG][3][64];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int pl = wv / NG, gq = wv % NG;  // plane dz = pl - 1, field group
  const int n = (int)blockIdx.x * kApNodes - 1 + lane, nc = min(max(n, 0), NP1 - 1);
  float4 q[3][7], p[3][3];
#pragma unroll
  for (int w = 0; w < 3; ++w) {
    const int m = min(max(n + ((pl - 1) * g1.ny + w - 1) * g1.nx, 0), NP1 - 1);
#pragma unroll
    for (int u = 0; u < 7; ++u) q[w][u] = A1[(size_t)((pl * 3 + w) * 7 + u) * NP1 + nc];
#pragma unroll
    for (int fj = 0; fj < 3; ++fj) p[w][fj] = P[(size_t)(fj * KG + gq) * NP1 + m];
  }
  __builtin_amdgcn_sched_barrier(0);  // (keeps the compiler from moving the loads down to their use)
  if (MODE != kApplyPow && cur->all_done) return;  // whole block
  float4 y[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) y[d] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
  for (int w = 0; w < 3; ++w) {
    float a[28];
#pragma unroll
    for (int u = 0; u < 7; ++u) {
      a[u * 4] = q[w][u].x;
      a[u * 4 + 1] = q[w][u].y;
      a[u * 4 + 2] = q[w][u].z;
      a[u * 4 + 3] = q[w][u].w;
    }
#pragma unroll
    for (int fj = 0; fj < 3; ++fj) {
      const float4 c = p[w][fj], l = lane_shift<0x138>(c), r = lane_shift<0x130>(c);
#pragma unroll
      for (int fi = 0; fi < 3; ++fi) {
        fma4(y[fi], a[fi * 3 + fj], l);
        fma4(y[fi], a[9 + fi * 3 + fj], c);
        fma4(y[fi], a[18 + fi * 3 + fj], r);
      }
    }
  }
  if (pl > 0)
#pragma unroll
    for (int d = 0; d < 3; ++d) lds[pl - 1][gq][d][lane] = y[d];
  __syncthreads();
  if (pl > 0) return;
  double s4[4] = {0, 0, 0, 0};
  if (lane >= 1 && lane <= kApNodes && n < NP1)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const size_t o = (size_t)(d * KG + gq) * NP1 + n;
      apply_out<MODE>(P[o], add4(add4(y[d], lds[0][gq][d][lane]), lds[1][gq][d][lane]), R, kinv, omega, OUT, o,
                      (size_t)d * NP1 + n, s4);
    }
  if constexpr (MODE == kApplyPow) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double s = wave_sum_dpp(s4[r]);
      if (lane == 0) part[(size_t)r * gridDim.x + blockIdx.x] = s;
    }
  }
}

// rc = P^T T for the coarse hats at the nodes of grid gt (the second level or
// the fine grid itself): a wave per coarse node and component, its lanes over
// the nodes under the node's hat
template <int K>
__global__ void __launch_bounds__(256) k_v_coarse_rhs(Grid gt, CGrid cg, Hats hats, int NPt, const float4 *T,
                                                      float4 *rc4, const MState *cur) {
  constexpr int KG = K / 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int id = blockIdx.x * 4 + wv, c = blockIdx.y, d = c / KG, grp = c % KG;
  if (id >= cg.nq || group_stopped(cur, grp * 4)) return;
  const int cx = id % cg.mx, cy = (id / cg.mx) % cg.my, cz = id / (cg.mx * cg.my);  // interior index, 0-based
  // nodes with a non-zero hat: strictly between the neighbouring coarse nodes
  const int x0 = hats.past[0][cx], y0 = hats.past[1][cy], z0 = hats.past[2][cz];
  const int wx = hats.upto[0][cx + 2] - x0, wy = hats.upto[1][cy + 2] - y0;
  const int n = wx * wy * (hats.upto[2][cz + 2] - z0);
  const int ox = 3 * cx, oy = 3 * cg.mx * cy, oz = 3 * cg.mx * cg.my * cz;
  const float4 *t = T + (size_t)c * NPt;
  float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 2
  for (int s = lane; s < n; s += 64) {
    const int r = s / wx, x = x0 + s % wx, y = y0 + r % wy, z = z0 + r / wy;
    const float w = hat_weight(hats.x[x], ox) * (hat_weight(hats.y[y], oy) * hat_weight(hats.z[z], oz));
    fma4(acc, w, t[((size_t)z * gt.ny + y) * gt.nx + x]);
  }
  acc = make_float4(wave_sum_dpp(acc.x), wave_sum_dpp(acc.y), wave_sum_dpp(acc.z), wave_sum_dpp(acc.w));
  if (lane == 0) rc4[(size_t)(id * 3 + d) * KG + grp] = acc;
}

// ec = A_c^-1 rc, FP32 matrix instructions.  Block: 16 rows, its waves each a
// share of the columns, 16 at a time: lane (r = l % 16, k = l / 16) loads the
// four columns 4 k .. 4 k + 3 of row r (one 16-byte load; four lanes a 64-byte
// line) and of rc the field r of the same four, so the step t of four 16x16x4
// products takes column 4 k + t of both operands.  The waves' tiles are added
// in LDS in order.  What bounds it is two memory latencies, and from about 2000
// DOFs the inverse (19 MB at 2187, out of L2 and MALL); hence AHEAD steps of a
// wave are loaded together, all of them up to 1280 columns.  12 fields, us: 375
// DOFs 4, 2187 DOFs 8.6 (14.4 with one step at a time; a wave per 64 rows and
// split columns, summed by the next kernel: 10 and 10).
constexpr int kGemvWaves = 16;
constexpr int kGemvRowsV = 16;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // rows start at any multiple of 4 bytes
template <int K, int AHEAD>
__global__ void __launch_bounds__(64 * kGemvWaves) k_v_gemv(int nc, const float *__restrict__ ainv,
                                                            const float *__restrict__ rc, float *__restrict__ ec,
                                                            const MState *cur) {
  __shared__ float tile[kGemvWaves][256];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, k = lane >> 4, row0 = blockIdx.x * kGemvRowsV;
  // rows past nc are clamped (not stored); columns past nc read on (into the
  // next row, or the zeros behind the inverse) or, a whole step past it, the
  // row's start, and meet zeros in place of rc
  const float *a = ainv + (size_t)min(row0 + r, nc - 1) * nc + 4 * k;
  if (cur->all_done) return;  // whole grid
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int c0 = 16 * w; c0 < nc; c0 += 16 * kGemvWaves * AHEAD) {
    f32x4u av[AHEAD];
    float b[AHEAD][4];
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) {
      const int c = c0 + 16 * kGemvWaves * s;
      av[s] = *reinterpret_cast<const f32x4u *>(a + (c < nc ? c : 0));
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int col = c + 4 * k + t;
        const bool in = r < K && col < nc;
        b[s][t] = rc[in ? col * K + r : 0];
        b[s][t] = in ? b[s][t] : 0.0f;
      }
    }
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s][t], b[s][t], acc, 0, 0, 0);
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) tile[w][(4 * k + v) * 16 + r] = acc[v];  // row 4 k + v, field r
  __syncthreads();
  const int i = threadIdx.x >> 4, f = threadIdx.x & 15;
  if (threadIdx.x >= 256 || f >= K || row0 + i >= nc) return;
  float s = 0.0f;
#pragma unroll
  for (int q = 0; q < kGemvWaves; ++q) s += tile[q][threadIdx.x];
  ec[(size_t)(row0 + i) * K + f] = s;
}

// OUT = w IN + P ec at the nodes of grid gt (as k_v_coarse_rhs; OUT may be IN);
// boundary nodes keep IN, zero there
template <int K>
__global__ void __launch_bounds__(256) k_v_coarse_add(Grid gt, Hats hats, int NPt, float w, const float4 *ec,
                                                      const float4 *IN, float4 *OUT, const MState *cur) {
  constexpr int KG = K / 4;
  const int c = blockIdx.y, d = c / KG, grp = c % KG;
  const int n = blockIdx.x * 256 + threadIdx.x;  // < NPt
  const float4 e0 = IN[(size_t)c * NPt + n];
  if (group_stopped(cur, grp * 4)) return;
  const int x = n % gt.nx, y = (n / gt.nx) % gt.ny, z = n / (gt.nx * gt.ny);
  float4 acc = make_float4(w * e0.x, w * e0.y, w * e0.z, w * e0.w);
  if (n < gt.nn && !node_on_boundary(gt, x, y, z)) {
    const HatEntry hx = hats.x[x], hy = hats.y[y], hz = hats.z[z];
    float4 e[8];
#pragma unroll
    for (int t = 0; t < 8; ++t)
      e[t] = ec[((t & 1 ? hx.q1 : hx.q0) + (t & 2 ? hy.q1 : hy.q0) + (t & 4 ? hz.q1 : hz.q0) + d) * KG + grp];
#pragma unroll
    for (int t = 0; t < 8; ++t)
      fma4(acc, (t & 1 ? hx.w1 : hx.w0) * ((t & 2 ? hy.w1 : hy.w0) * (t & 4 ? hz.w1 : hz.w0)), e[t]);
  }
  OUT[(size_t)c * NPt + n] = acc;
}

// OUT = w0 Z + P1 E; OUT may be Z.  Along a side a fine node lies on a
// second-level node (even index) or half-way between two: the mean of the
// nodes i / 2 and (i + 1) / 2 either way.
template <int K>
__global__ void __launch_bounds__(256) k_v_prolong(Grid g, Grid g1, int NP, int NP1, float w0, const float4 *E,
                                                   const float4 *Z, float4 *OUT, const MState *cur) {
  constexpr int KG = K / 4;
  const int c = blockIdx.y, grp = c % KG;
  const int n = blockIdx.x * 256 + threadIdx.x;
  const float4 z = Z[(size_t)c * NP + n];  // (n < NP: the grid covers NP)
  if (group_stopped(cur, grp * 4)) return;
  float4 acc = make_float4(w0 * z.x, w0 * z.y, w0 * z.z, w0 * z.w);
  const int i = n % g.nx, j = (n / g.nx) % g.ny, k = n / (g.nx * g.ny);
  if (n < g.nn && !node_on_boundary(g, i, j, k)) {
    const float4 *ec = E + (size_t)c * NP1;
    float4 e[8];
#pragma unroll
    for (int t = 0; t < 8; ++t)
      e[t] = ec[(((k + (t >> 2)) / 2) * g1.ny + (j + ((t >> 1) & 1)) / 2) * g1.nx + (i + (t & 1)) / 2];
#pragma unroll
    for (int t = 0; t < 8; ++t) fma4(acc, 0.125f, e[t]);
  }
  OUT[(size_t)c * NP + n] = acc;
}

// The second level's operator: node blocks (A1[quad * NP1 + node], the quads
// of a node as in k_m_spmv's layout) and Jacobi weights.  The block towards a neighbour sums, over the second-level elements
// holding both nodes, the Galerkin contributions of their fine elements (C,
// k_cs_table on mid), in FP64, rounded once; rows and columns of boundary nodes
// are zero.  Block of 64 nodes x 4: thread (lane, y) takes neighbours y, y + 4, ...
__global__ void __launch_bounds__(256) k_v_asm(Grid g, Grid g1, CGrid mid, int NP1, const int *et, const double *C,
                                               float *A1, float *kinv1) {
  const int lane = threadIdx.x & 63, n = blockIdx.x * 64 + lane;
  const int tx = mid.lx == 2 ? 2 : 3, ty = mid.ly == 2 ? 2 : 3;  // positions per side (k_cs_table)
  float *base = A1 + (size_t)n * 4;
  auto put = [&](int s, float v) { base[(size_t)(s >> 2) * NP1 * 4 + (s & 3)] = v; };
  const int i = n % g1.nx, j = (n / g1.nx) % g1.ny, k = n / (g1.nx * g1.ny);
  const bool row = n < g1.nn && !node_on_boundary(g1, i, j, k);
  for (int nb = threadIdx.x >> 6; nb < 27; nb += 4) {
    const int dz = nb / 9 - 1, dy = (nb / 3) % 3 - 1, dx = nb % 3 - 1;
    double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (row && !node_on_boundary(g1, i + dx, j + dy, k + dz)) {
      for (int q = 0; q < 8; ++q) {
        const int a = q >> 2, b = (q >> 1) & 1, c = q & 1;
        const int px = 1 - a + dx, py = 1 - b + dy, pz = 1 - c + dz;
        if (px < 0 || px > 1 || py < 0 || py > 1 || pz < 0 || pz > 1) continue;
        const int Ex = i - 1 + a, Ey = j - 1 + b, Ez = k - 1 + c;
        const int ro = (local_node(1 - a, 1 - b, 1 - c) * 3) * 24 + local_node(px, py, pz) * 3;
        const bool lx = Ex == mid.mx && mid.lx == 1, ly = Ey == mid.my && mid.ly == 1, lz = Ez == mid.mz && mid.lz == 1;
        for (int z = 0; z < (lz ? 1 : 2); ++z)
          for (int y = 0; y < (ly ? 1 : 2); ++y)
            for (int x = 0; x < (lx ? 1 : 2); ++x) {
              const int e = ((Ez * 2 + z) * g.ney + Ey * 2 + y) * g.nex + Ex * 2 + x;
              const int pos = (((lz ? 2 : 0) + z) * ty + (ly ? 2 : 0) + y) * tx + (lx ? 2 : 0) + x;
              const double *s = C + ((size_t)pos * 3 + et[e]) * 576 + ro;
#pragma unroll
              for (int t = 0; t < 9; ++t) acc[t] += s[(t / 3) * 24 + t % 3];
            }
      }
    }
#pragma unroll
    for (int t = 0; t < 9; ++t) put(mslot(nb, t / 3, t % 3), (float)acc[t]);
    if (nb % 3 == 2) put((nb / 3) * 28 + 27, 0.0f);  // the row's pad
    if (nb == 13)
#pragma unroll
      for (int d = 0; d < 3; ++d) kinv1[(size_t)d * NP1 + n] = row ? (float)(1.0 / acc[d * 4]) : 0.0f;
  }
}

// start of the power iteration: a fixed pattern of +-1 on the nodes with a row
// (kinv != 0), four fields
__global__ void __launch_bounds__(256) k_v_rand(int NP, int stride, const float *kinv, float4 *P) {
  const int n = blockIdx.x * 256 + threadIdx.x, d = blockIdx.y;
  if (n >= NP) return;
  unsigned h = (unsigned)(n * 3 + d) * 2654435761u;
  h ^= h >> 15;
  h *= 2246822519u;
  h ^= h >> 13;
  const bool row = kinv[(size_t)d * NP + n] != 0.0f;
  auto s = [&](int b) { return row ? ((h >> b) & 1u ? 1.0f : -1.0f) : 0.0f; };
  P[(size_t)d * stride + n] = make_float4(s(3), s(9), s(17), s(25));
}

// *out = the largest growth of (v, D v) between two iterates of the power
// iteration, over four fields and the blocks of the kernel that formed it
// (partials p0, then p1, n a field).  A mode on a few nodes, of one stiff element
// say, has outgrown what else its block holds after a dozen steps, while the sum
// over a large grid does not show it yet.  Blocks below kGrowthShare of the mean
// are left out: a node or two whose value passes through zero grow by anything.
constexpr double kGrowthShare = 0.1;
__global__ void __launch_bounds__(kRedThreads) k_v_growth(const double *p0, const double *p1, int n, double *out) {
  __shared__ double least[4], most[kRedThreads];
  const double sum = rows_sum<4>(p0, n, n);
  if (threadIdx.x < 4) least[threadIdx.x] = kGrowthShare * sum / n;
  __syncthreads();
  double m = 0.0;
  for (int f = 0; f < 4; ++f)
    for (int i = threadIdx.x; i < n; i += kRedThreads) {
      const double a = p0[(size_t)f * n + i], g = p1[(size_t)f * n + i] / a;
      if (a > least[f]) m = g < 1e6 ? fmax(m, g) : 1e6;  // (1e6, as for NaN: not usable)
    }
  most[threadIdx.x] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < kRedThreads; ++i) m = fmax(m, most[i]);
    *out = m;
  }
}

// the main and the interface blocks of a stencil kernel
static int main_blocks(const Grid &g) { return (int)nblk(mshape(g).NP, kApNodes * kApWaves); }
int stencil_blocks(const Grid &g, const StencilOp &op) { return main_blocks(g) + (int)nblk(op.nif, kIfaceNodes); }
int stencil_blocks_max(const Grid &g) { return main_blocks(g) + (int)nblk(g.nn, kIfaceNodes); }
// codes | interface list | block counts | stencils | homogeneous stencils, 256-byte aligned parts
static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }
size_t stencil_bytes(const Grid &g) {
  const size_t NP = mshape(g).NP;
  return align256(NP * sizeof(uint16_t)) + align256(NP * sizeof(int)) + align256((NP / 256 + 1) * sizeof(int)) +
         align256((size_t)kNumStencils * kStencilFloats * sizeof(float)) + align256(128 * sizeof(float));
}

hipError_t launch_d_setup(const Grid &g, const int *et, const double *ke, void *buf, StencilOp *op, hipStream_t st) {
  const int NP = mshape(g).NP, nb = NP / 256;
  char *p = static_cast<char *>(buf);
  auto take = [&p](size_t bytes) {
    char *q = p;
    p += align256(bytes);
    return q;
  };
  uint16_t *code = reinterpret_cast<uint16_t *>(take(NP * sizeof(uint16_t)));
  int *list = reinterpret_cast<int *>(take(NP * sizeof(int)));
  int *cnt = reinterpret_cast<int *>(take((nb + 1) * sizeof(int)));
  float *tab = reinterpret_cast<float *>(take((size_t)kNumStencils * kStencilFloats * sizeof(float)));
  float *hom = reinterpret_cast<float *>(take(128 * sizeof(float)));
  hipLaunchKernelGGL(k_d_code, dim3(nb), dim3(256), 0, st, g, NP, et, code);
  hipLaunchKernelGGL(k_d_count, dim3(nb), dim3(256), 0, st, code, cnt);
  hipLaunchKernelGGL(k_d_scan, dim3(1), dim3(256), 0, st, nb, cnt);
  hipLaunchKernelGGL(k_d_list, dim3(nb), dim3(256), 0, st, code, cnt, list);
  hipLaunchKernelGGL(k_d_table, dim3(kNumStencils), dim3(256), 0, st, ke, tab);
  hipLaunchKernelGGL(k_d_hom, dim3(1), dim3(128), 0, st, tab, hom);
  op->code = code;
  op->list = list;
  op->tab = tab;
  op->hom = hom;
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(&op->nif, cnt + nb, sizeof(int), hipMemcpyDeviceToHost, st);
  return e == hipSuccess ? hipStreamSynchronize(st) : e;
}

template <int MODE>
static hipError_t launch_d_apply(const Grid &g, int K, const StencilOp &op, const float *P, const float *R,
                                 const float *kinv, float omega, float *OUT, double *part, const void *state,
                                 hipStream_t st) {
  const int NP = mshape(g).NP, nbm = main_blocks(g), per = (nbm + 7) / 8;
  const int nbi = (int)nblk(op.nif, kIfaceNodes), peri = (nbi + 7) / 8;
  MPP_K_DISPATCH(K, hipLaunchKernelGGL((k_d_apply<KK, MODE>), dim3(8 * (peri + per), MODE == kApplyPow ? 1 : KK / 4),
                                       dim3(64 * kApWaves), 0, st, g, NP, nbi, peri, nbm, per, op.nif, op.code,
                                       op.list, op.tab, op.hom, reinterpret_cast<const float4 *>(P),
                                       reinterpret_cast<const float4 *>(R), kinv, omega,
                                       reinterpret_cast<float4 *>(OUT), part, static_cast<const MState *>(state)));
  return hipGetLastError();
}

hipError_t launch_d_spmv(const Grid &g, int K, const StencilOp &op, const float *P, float *AP, double *part1,
                         const void *state, hipStream_t st) {
  return launch_d_apply<kApplyCg>(g, K, op, P, nullptr, nullptr, 0.0f, AP, part1, state, st);
}

template <int MODE>
static hipError_t launch_mid(const Grid &g1, int K, const VCycleDev &v, const float *P, const float *R, float *OUT,
                             double *part, const void *state, hipStream_t st) {
  const int NP1 = mshape(g1).NP;
  MPP_K_DISPATCH(K, hipLaunchKernelGGL((k_v_mid<KK, MODE>), dim3(nblk(NP1, kApNodes)),
                                       dim3(MODE == kApplyPow ? 192 : 48 * KK), 0, st, g1, NP1, reinterpret_cast<const float4 *>(v.A1),
                                       reinterpret_cast<const float4 *>(P), reinterpret_cast<const float4 *>(R),
                                       v.kinv1, v.w1, reinterpret_cast<float4 *>(OUT), part,
                                       static_cast<const MState *>(state)));
  return hipGetLastError();
}

template <int K>
static void launch_gemv(const VCycleDev &v, const MState *cur, hipStream_t st) {
  const dim3 grid(nblk(v.cg.nc, kGemvRowsV)), block(64 * kGemvWaves);
  const int nc = v.cg.nc, steps = (int)nblk(nc, 16 * kGemvWaves);  // of a wave
  if (steps == 1)
    hipLaunchKernelGGL((k_v_gemv<K, 1>), grid, block, 0, st, nc, v.ainv, v.rc, v.ec, cur);
  else if (steps == 2)
    hipLaunchKernelGGL((k_v_gemv<K, 2>), grid, block, 0, st, nc, v.ainv, v.rc, v.ec, cur);
  else
    hipLaunchKernelGGL((k_v_gemv<K, 5>), grid, block, 0, st, nc, v.ainv, v.rc, v.ec, cur);
}

hipError_t launch_vcycle(const Grid &g, int K, const VCycleDev &v, const StencilOp &op, const float *kinv,
                         const float *R, const float *Z, float *T, float *OUT, double *pr, const void *state,
                         hipStream_t st) {
  const int NP = mshape(g).NP;
  const MState *cur = static_cast<const MState *>(state);
  const dim3 grid0(NP / 256, 3 * K / 4);
  hipError_t e = launch_d_apply<kApplyRes>(g, K, op, Z, R, kinv, v.w0, T, nullptr, state, st);
  if (e != hipSuccess) return e;
  const Hats hats{v.hat[0], v.hat[1], v.hat[2], {v.past[0], v.past[1], v.past[2]}, {v.upto[0], v.upto[1], v.upto[2]}};
  const dim3 nq(nblk(v.cg.nq, 4), 3 * K / 4);
  float4 *rc4 = reinterpret_cast<float4 *>(v.rc), *ec4 = reinterpret_cast<float4 *>(v.ec);
  if (!v.mid.nq) {  // two levels
    MPP_K_DISPATCH(K, {
      hipLaunchKernelGGL(k_v_coarse_rhs<KK>, nq, dim3(256), 0, st, g, v.cg, hats, NP,
                         reinterpret_cast<const float4 *>(T), rc4, cur);
      launch_gemv<KK>(v, cur, st);
      hipLaunchKernelGGL(k_v_coarse_add<KK>, grid0, dim3(256), 0, st, g, hats, NP, v.w0, ec4,
                         reinterpret_cast<const float4 *>(Z), reinterpret_cast<float4 *>(v.z), cur);
    });
    return launch_d_apply<kApplyPost>(g, K, op, v.z, R, kinv, v.w0, OUT, pr, state, st);
  }
  const int NP1 = mshape(v.g1).NP;
  const dim3 grid1(NP1 / 256, 3 * K / 4);
  float4 *E0 = reinterpret_cast<float4 *>(v.E0);
  MPP_K_DISPATCH(K, hipLaunchKernelGGL(k_v_restrict<KK>, grid1, dim3(256), 0, st, g, v.g1, NP, NP1,
                                       reinterpret_cast<const float4 *>(T), v.kinv1, reinterpret_cast<float4 *>(v.R1),
                                       E0, cur));
  if ((e = launch_mid<kApplyRes>(v.g1, K, v, v.E0, v.R1, v.T1, nullptr, state, st)) != hipSuccess) return e;
  MPP_K_DISPATCH(K, {
    hipLaunchKernelGGL(k_v_coarse_rhs<KK>, nq, dim3(256), 0, st, v.g1, v.cg, hats, NP1,
                       reinterpret_cast<const float4 *>(v.T1), rc4, cur);
    launch_gemv<KK>(v, cur, st);
    hipLaunchKernelGGL(k_v_coarse_add<KK>, grid1, dim3(256), 0, st, v.g1, hats, NP1, v.w1, ec4, E0, E0, cur);
  });
  if ((e = launch_mid<kApplyPost>(v.g1, K, v, v.E0, v.R1, v.E, nullptr, state, st)) != hipSuccess) return e;
  MPP_K_DISPATCH(K, hipLaunchKernelGGL(k_v_prolong<KK>, grid0, dim3(256), 0, st, g, v.g1, NP, NP1, v.w0,
                                       reinterpret_cast<const float4 *>(v.E), reinterpret_cast<const float4 *>(Z),
                                       reinterpret_cast<float4 *>(v.z), cur));
  return launch_d_apply<kApplyPost>(g, K, op, v.z, R, kinv, v.w0, OUT, pr, state, st);
}

hipError_t launch_v_start(const Grid &g, int K, const VCycleDev &v, const StencilOp &op, const float *kinv,
                          const float *R, float *P, float *AP, void *state, hipStream_t st) {
  const hipError_t e = launch_vcycle(g, K, v, op, kinv, R, P, AP, P, v.prz, state, st);
  return e == hipSuccess ? launch_c_rzfix(K, stencil_blocks(g, op), v.prz, true, state, st) : e;
}

void vcycle_free(VCycleDev *v) {
  if (!v) return;
  dfree(v->arena);
  delete v;
}

namespace {
// Smoother damping: kDamp / lambda with lambda the power iteration's estimate
// after kPowerIts steps (k_v_growth); the smoothers need damping * lambda_max <
// 2.  The estimate is 0.94 to 1.05 lambda_max (damping * lambda_max 1.57 to 1.75)
// in homogeneous, spherical and random media of contrasts to 1000, with one
// stiff element on 24^3 to 160^3, in thin cells, with Poisson's ratios to 0.49,
// and on the second level.  The ratio of the sums over the whole grid instead
// reads 2.71 where one stiff element makes it 3.52 (80^3, contrast 15), and has
// to be met with a smaller kDamp: 45 RVEs of 11 to 80 elements a side take 1501
// iterations against 1511 with 1.55 over that ratio (1531 at kDamp = 1.6).
constexpr int kPowerIts = 12;
constexpr float kDamp = 1.65f;
// The two-level form: coarse elements of at most 2 fine ones a side while their
// inverse has at most kCoarseMaxDofs DOFs (20 elements a side), of at most 3
// while it has at most 1536 (26).  The second level's five kernels fall away:
// 60 us an iteration of 8 fields become 40 at 10 to 16 elements a side, 54 at
// 20 and 47 to 54 at 22 to 26, with as many iterations (22 to 27; 33 at 24).
// Above, the inverse's set-up (2.1 ms at 2187 DOFs against 1.4) costs more than
// the iterations gain.
// Cells kLongCells times as long along one side as along another have it with
// coarse elements of one length, where that is at most two of the long cells:
// twice the spacing on every side loses what the smoother leaves along the
// long ones.  Three levels and this, inner iterations to 1e-8 and ms (contrast
// 10, spheres, eight fields, nodes): 6 x 60 x 61 141, 7.2 and 44, 2.6; 13 x 60 x
// 60 72, 6.2 and 57, 4.1; 17 x 41 x 41 38, 3.2 and 38, 2.5; 9 x 10 x 41 65, 3.3
// and 28, 1.7; at 2.4 long cells (23 x 91 x 91) 64, 10.2 and 72, 9.8; at 3.3 (31
// x 91 x 91) 52, 10.4 and 72, 11.8.  With the 2200 DOFs that stiff phases are
// worth instead of 1536 the set-up takes 0.6 ms more (9 x 61 x 62, contrast 1e4:
// 12.4 ms become 6.9; 10: 3.4 become 3.2).
constexpr double kLongCells = 2.5;
bool coarse_grid_two_level(const Grid &g, double contrast, CGrid *out) {
  if (cell_aspect(g) >= kLongCells && coarse_grid_long(g, contrast > kHighContrast ? kCoarseMaxDofs : 1536, out) &&
      std::max({out->lx * g.dx, out->ly * g.dy, out->lz * g.dz}) <= 2.001 * std::max({g.dx, g.dy, g.dz}))
    return true;
  for (int width = 2; width <= 3; ++width)
    if (coarse_grid_wide(g, width, width == 2 ? kCoarseMaxDofs : 1536, out) &&
        std::max({out->hx, out->lx, out->hy, out->ly, out->hz, out->lz}) <= width)
      return true;
  return false;
}

// The tables of a side of ne fine and d coarse elements at the nodes of the
// level above the coarse one, node i at fine index min(step i, ne): the hats
// (offsets of stride per interior coarse node), then, each for q = 0 .. d, the
// first node beyond coarse node q and the first one at or beyond it
void side_tables(int ne, int d, int even, int step, int stride, std::vector<HatEntry> &hats, std::vector<int> &ends) {
  const int n = (ne + step - 1) / step + 1;
  ends.assign(2 * (d + 1), n);
  int e = 0;
  for (int i = n - 1; i >= 0; --i)
    for (int q = 0; q <= d; ++q) {
      const int x = std::min(step * i, ne), at = coarse_node(q, ne, d, even);
      if (x > at) ends[q] = i;
      if (x >= at) ends[d + 1 + q] = i;
    }
  for (int i = 0; i < n; ++i) {
    const int x = std::min(step * i, ne);
    while (e + 1 < d && x >= coarse_node(e + 1, ne, d, even)) ++e;
    const int a = coarse_node(e, ne, d, even), b = coarse_node(e + 1, ne, d, even);
    const float f = (float)(x - a) / (float)(b - a);
    hats.push_back({e >= 1 ? 1.0f - f : 0.0f, e + 1 < d ? f : 0.0f, (std::max(e, 1) - 1) * stride,
                    (std::min(e + 1, d - 1) - 1) * stride});
  }
}
}  // namespace

int vcycle_setup(const Grid &g, int K, double contrast, const int *et_d, const double *ke_d, const StencilOp &op, const float *kinv,
                 float *P, float *AP, hipStream_t st, VCycleDev **out) {
  *out = nullptr;
  CGrid cg, mid;
  if (!coarse_enabled()) return MPPD_OK;
  const bool two = coarse_grid_two_level(g, contrast, &cg);
  if (two)
    mid = CGrid{};
  else if (!coarse_grid_cycle(g, contrast, &cg) || !coarse_grid_by_two(g, &mid))
    return MPPD_OK;
  VCycleDev *v = new VCycleDev();
  v->arena = nullptr;
  v->cg = cg;
  v->mid = mid;
  Grid &g1 = v->g1;
  g1 = Grid{};  // (without a second level: 2 nodes a side, unused)
  g1.nx = mid.mx + 2;
  g1.ny = mid.my + 2;
  g1.nz = mid.mz + 2;
  g1.nex = g1.nx - 1;
  g1.ney = g1.ny - 1;
  g1.nez = g1.nz - 1;
  g1.nn = g1.nx * g1.ny * g1.nz;
  g1.nrow = 3 * g1.nn;
  g1.nrow_pad = (int)round_up(g1.nrow, kRowPad);
  g1.nelem = g1.nex * g1.ney * g1.nez;
  const MLaunch s1 = mshape(g1);
  const int nc = cg.nc, nb = stencil_blocks(g, op), nb1 = (int)nblk(s1.NP, kApNodes);
  double *C = nullptr, growth_h[2] = {};
  int rc = MPPD_OK;
  bool ok = false;
  do {
    // one allocation, 256-byte aligned parts, all but the coarse inverse and
    // the second level's operator zero-filled
    size_t off = 0;
    auto carve = [&off](size_t bytes) {
      const size_t o = off;
      off += (bytes + 255) & ~(size_t)255;
      return o;
    };
    const size_t n1 = two ? 0 : (size_t)s1.NP * 3 * K * sizeof(float);
    const size_t o_rc = carve((size_t)nc * K * sizeof(float)), o_ec = carve((size_t)nc * K * sizeof(float));
    // the sides' tables (VCycleDev), one copy
    std::vector<HatEntry> hats[3];
    std::vector<int> ends[3];
    size_t o_hat[3], o_end[3];
    const int ne[3] = {g.nex, g.ney, g.nez}, mq[3] = {cg.mx, cg.my, cg.mz};
    for (int a = 0, stride = 3; a < 3; stride *= mq[a++]) {
      side_tables(ne[a], mq[a] + 1, cg.even & (1 << a), two ? 1 : 2, stride, hats[a], ends[a]);
      o_hat[a] = carve(hats[a].size() * sizeof(HatEntry));
      o_end[a] = carve(ends[a].size() * sizeof(int));
    }
    const size_t o_z = carve(mixed_vector_len(g, K) * sizeof(float));
    const size_t o_prz = carve(std::max((size_t)K * nb, 2 * 4 * (size_t)std::max(nb, nb1)) * sizeof(double));
    const size_t o_grow = carve(2 * sizeof(double));
    const size_t o_R1 = carve(n1), o_E0 = carve(n1), o_T1 = carve(n1), o_E = carve(n1);
    const size_t o_k1 = carve(two ? 0 : (size_t)s1.NP * 3 * sizeof(float));
    const size_t zeroed = off, o_ainv = carve(((size_t)nc * nc + 16) * sizeof(float));  // (k_v_gemv reads 15 past it)
    const size_t o_A1 = carve(two ? 0 : mixed_matrix_floats(g1) * sizeof(float));
    hipError_t e = hipMalloc(&v->arena, off);
    if (e == hipSuccess) e = hipMemsetAsync(v->arena, 0, zeroed, st);
    if (e == hipSuccess)
      e = hipMemsetAsync(static_cast<char *>(v->arena) + o_ainv + (size_t)nc * nc * sizeof(float), 0,
                         16 * sizeof(float), st);
    if (e != hipSuccess) {
      rc = hip_fail(e, "preconditioner buffers");
      break;
    }
    char *base = static_cast<char *>(v->arena);
    auto at = [base](size_t o) { return reinterpret_cast<float *>(base + o); };
    v->rc = at(o_rc);
    v->ec = at(o_ec);
    std::vector<char> tables(o_z - o_hat[0]);
    for (int a = 0; a < 3; ++a) {
      std::memcpy(tables.data() + (o_hat[a] - o_hat[0]), hats[a].data(), hats[a].size() * sizeof(HatEntry));
      std::memcpy(tables.data() + (o_end[a] - o_hat[0]), ends[a].data(), ends[a].size() * sizeof(int));
      v->hat[a] = reinterpret_cast<HatEntry *>(base + o_hat[a]);
      v->past[a] = reinterpret_cast<int *>(base + o_end[a]);
      v->upto[a] = v->past[a] + mq[a] + 2;
    }
    e = hipMemcpyAsync(base + o_hat[0], tables.data(), tables.size(), hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
      rc = hip_fail(e, "preconditioner tables");
      break;
    }
    v->z = at(o_z);
    v->R1 = at(o_R1);
    v->E0 = at(o_E0);
    v->T1 = at(o_T1);
    v->E = at(o_E);
    v->kinv1 = at(o_k1);
    v->A1 = at(o_A1);
    v->prz = reinterpret_cast<double *>(base + o_prz);
    double *growth = reinterpret_cast<double *>(base + o_grow);
    float *ainv = at(o_ainv);
    v->ainv = ainv;
    // lambda_max(D^-1 A) of the fine operator, on four fields: the growth of
    // (v, D v) over the last two iterates
    const int NP = mshape(g).NP;
    double *p0 = v->prz, *p1 = v->prz + 4 * (size_t)nb;
    float *a = P, *b = AP;
    hipLaunchKernelGGL(k_v_rand, dim3(NP / 256, 3), dim3(256), 0, st, NP, NP * (K / 4), kinv,
                       reinterpret_cast<float4 *>(a));
    for (int i = 0; i < kPowerIts && e == hipSuccess; ++i) {
      e = launch_d_apply<kApplyPow>(g, K, op, a, nullptr, kinv, 0.0f, b, i & 1 ? p1 : p0, nullptr, st);
      std::swap(a, b);
    }
    hipLaunchKernelGGL(k_v_growth, dim3(1), dim3(kRedThreads), 0, st, p0, p1, nb, growth);
    if (e == hipSuccess && !two) {
      const int planes = coarse_table_planes(mid);
      if ((rc = dalloc(&C, coarse_table_len(mid, planes), false))) break;
      e = launch_cs_table(mid, 0, planes, ke_d, C, st);
      hipLaunchKernelGGL(k_v_asm, dim3(s1.NP / 64), dim3(256), 0, st, g, g1, mid, s1.NP, et_d, C, v->A1, v->kinv1);
      float *a1 = v->E0, *b1 = v->T1;  // four fields fit: K >= 4
      double *q0 = v->prz, *q1 = v->prz + 4 * (size_t)nb1;
      hipLaunchKernelGGL(k_v_rand, dim3(s1.NP / 256, 3), dim3(256), 0, st, s1.NP, s1.NP, v->kinv1,
                         reinterpret_cast<float4 *>(a1));
      for (int i = 0; i < kPowerIts && e == hipSuccess; ++i) {
        e = launch_mid<kApplyPow>(g1, 4, *v, a1, nullptr, b1, i & 1 ? q1 : q0, nullptr, st);
        std::swap(a1, b1);
      }
      hipLaunchKernelGGL(k_v_growth, dim3(1), dim3(kRedThreads), 0, st, q0, q1, nb1, growth + 1);
    }
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(growth_h, growth, sizeof(growth_h), hipMemcpyDeviceToHost, st);
    if (e != hipSuccess) {
      rc = hip_fail(e, "preconditioner set-up");
      break;
    }
    if ((rc = coarse_inverse(g, cg, et_d, ke_d, ainv, st, &ok))) break;  // synchronizes st
    // test hook: MPPD_VCYCLE_DAMPING in kDamp's place (above 2: a preconditioner
    // that is not positive definite, and the solver's return to Jacobi)
    const char *env = std::getenv("MPPD_VCYCLE_DAMPING");
    const float damp = env ? (float)std::atof(env) : kDamp;
    auto damping = [damp](double growth) {  // NaN or no growth: not usable
      const double lam = std::sqrt(growth);
      return lam > 0.1 && lam < 1e3 ? damp / (float)lam : 0.0f;
    };
    v->w0 = damping(growth_h[0]);
    v->w1 = two ? 1.0f : damping(growth_h[1]);
    ok = ok && v->w0 > 0.0f && v->w1 > 0.0f;
  } while (0);
  (void)hipStreamSynchronize(st);  // C may still be in use after a failed step
  dfree(C);
  if (rc || !ok) {
    vcycle_free(v);
    return rc;
  }
  *out = v;
  return MPPD_OK;
}

}  // namespace mpp
