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

// ---------------------------------------------------------------------------
// y = A p of one field group (4 fields) at 62 consecutive nodes by one wave.
// Lane l holds node n = n0 - 1 + l: lanes 1 .. 62 own an output, lanes 0 and
// 63 only contribute to their neighbours.  Per stencil row (dz, dy) a lane
// loads p at the dx = 0 neighbour alone (3 loads of 16 B) and forms what that
// value gives to its own node (C) and to the nodes left and right of it (it is
// their dx = +1 and dx = -1 neighbour: R, L), with those nodes' coefficients;
// after the nine rows the L and R sums move one lane over, 24 lane moves in
// all instead of 24 per row.
//
// A wave whose nodes with a row share one stencil (most waves: an interface
// node differs) takes the coefficients from scalar loads, so that its vector
// instructions are the FMAs and 27 loads; the others load them per lane from
// the table (mostly equal addresses, L1 hits).
//
// Addresses are clamped into [0, NP); every neighbour of a node with a row lies
// in the grid, and the results of the other lanes are not used.
//
// Bound: vector issue (972 FMAs a wave, 1193 vector instructions in the
// one-stencil form; 6.3 waves a SIMD at 50^3 with 12 fields: 12.5 us).  At 50^3
// with 12 fields and 8 spheres 24.7 us, one phase 19.5 us (about 4 us of either
// is the launch and the first loads), against 31.8 us for the stored matrix
// (1008 B a node); with 4 fields 14.3 against 25.1 us.
// ---------------------------------------------------------------------------
constexpr int kApNodes = 62;  // outputs per wave
constexpr int kApWaves = 4;   // waves per block (consecutive runs of nodes, one field group)

typedef const __attribute__((address_space(4))) float *const_f32;

__device__ __forceinline__ void fma4(float4 &y, float a, const float4 &x) {
  y.x += a * x.x;
  y.y += a * x.y;
  y.z += a * x.z;
  y.w += a * x.w;
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

template <int KG>
__device__ __forceinline__ void stencil_apply(const Grid &g, int NP, int n, unsigned c, const float *tab,
                                              const float4 *pg, float4 (&y)[3]) {
  const int nxny = g.nx * g.ny;
  auto load_p = [&](float4(&p)[3], int w) {
    const int m = min(max(n + (w / 3 - 1) * nxny + (w % 3 - 1) * g.nx, 0), NP - 1);
#pragma unroll
    for (int fj = 0; fj < 3; ++fj) p[fj] = pg[(size_t)fj * KG * NP + m];
  };
  float4 p[2][3];
  load_p(p[0], 0);  // in flight while the codes arrive
  __builtin_amdgcn_sched_barrier(0);
  const unsigned long long rows = __ballot(c != kNoRow);
#pragma unroll
  for (int d = 0; d < 3; ++d) y[d] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (rows == 0) return;  // boundary nodes only
  const unsigned c0 = __builtin_amdgcn_readlane(c, (int)__builtin_ctzll(rows));
  if (__ballot(c != kNoRow && c != c0) == 0) {
    float4 L[3], R[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) L[d] = R[d] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const const_f32 t = (const_f32)(uintptr_t)(tab + (size_t)c0 * kStencilFloats);
    // row w + 1's p is loaded before row w's FMAs, its coefficients after the
    // first third of them (a scalar load in flight would make that third wait
    // for it as well); the scheduling barriers keep the compiler from moving
    // the loads down to their use
    float a[2][27];
    auto load_a = [&](int w) {
#pragma unroll
      for (int u = 0; u < 27; ++u) a[w & 1][u] = t[w * 28 + u];
    };
    load_a(0);
#pragma unroll
    for (int w = 0; w < kRows; ++w) {
      if (w + 1 < kRows) load_p(p[(w + 1) & 1], w + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int fj = 0; fj < 3; ++fj) {
#pragma unroll
        for (int fi = 0; fi < 3; ++fi) {
          fma4(L[fi], a[w & 1][fi * 3 + fj], p[w & 1][fj]);
          fma4(y[fi], a[w & 1][9 + fi * 3 + fj], p[w & 1][fj]);
          fma4(R[fi], a[w & 1][18 + fi * 3 + fj], p[w & 1][fj]);
        }
        if (fj == 0) {
          __builtin_amdgcn_sched_barrier(0);
          if (w + 1 < kRows) load_a(w + 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const float4 l = lane_shift<0x138>(L[d]), r = lane_shift<0x130>(R[d]);
      y[d].x += l.x + r.x;
      y[d].y += l.y + r.y;
      y[d].z += l.z + r.z;
      y[d].w += l.w + r.w;
    }
  } else {
    // 27 steps, one 3x3 block of the lane's own coefficients each, loaded a
    // step ahead; the dx = -1 and +1 values are the adjacent lanes', moved
    // over per row (12 sums instead of 36 leave registers for the coefficients)
    const float4 *tc = reinterpret_cast<const float4 *>(tab) + (c == kNoRow ? c0 : c) * (unsigned)kNodeQuads;
    float4 q[2][3];
    auto load_q = [&](int s) {
      // floats 0 .. 11 of the row hold dx = -1 (0 .. 8), 8 .. 19 dx = 0 (9 .. 17), 16 .. 27 dx = +1 (18 .. 26)
#pragma unroll
      for (int u = 0; u < 3; ++u) q[s & 1][u] = tc[(s / 3) * 7 + (s % 3) * 2 + u];
    };
    load_q(0);
#pragma unroll
    for (int s = 0; s < 3 * kRows; ++s) {
      const int j = s % 3;
      if (s + 1 < 3 * kRows) load_q(s + 1);
      __builtin_amdgcn_sched_barrier(0);
      const float4 *qs = q[s & 1];
      const float a[12] = {qs[0].x, qs[0].y, qs[0].z, qs[0].w, qs[1].x, qs[1].y,
                           qs[1].z, qs[1].w, qs[2].x, qs[2].y, qs[2].z, qs[2].w};
#pragma unroll
      for (int fj = 0; fj < 3; ++fj) {
        const float4 v = j == 0 ? lane_shift<0x138>(p[0][fj]) : j == 1 ? p[0][fj] : lane_shift<0x130>(p[0][fj]);
#pragma unroll
        for (int fi = 0; fi < 3; ++fi) fma4(y[fi], a[j + fi * 3 + fj], v);
      }
      if (j == 2 && s + 1 < 3 * kRows) load_p(p[0], s / 3 + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// k_d_spmv: AP = A P for every field and the partials of (p, Ap),
// part1[field * nblk + block].  Grid (8 per, K/4): block (b, g) takes kApWaves
// runs of kApNodes nodes of field group g (XCD-aware run order).
template <int K>
__global__ void __launch_bounds__(256) k_d_spmv(Grid g, int NP, int nblk, int per, const uint16_t *code,
                                                const float *tab, const float4 *P, float4 *AP, double *part1,
                                                const MState *cur) {
  constexpr int KG = K / 4;
  __shared__ double lds[kApWaves][4];
  const int lb = xcd_block(per), grp = blockIdx.y, r0 = grp * 4;
  if (lb >= nblk) return;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n = (lb * kApWaves + wv) * kApNodes - 1 + lane;
  const bool in = n >= 0 && n < NP, out = in && lane >= 1 && lane <= kApNodes;
  const unsigned c = in ? (unsigned)code[n] : kNoRow;
  if (group_stopped(cur, r0)) return;  // whole block
  const float4 *pg = P + (size_t)grp * NP;
  float4 y[3];
  stencil_apply<KG>(g, NP, n, c, tab, pg, y);
  double pap[4] = {0, 0, 0, 0};
  if (out) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const float4 pc = pg[(size_t)d * KG * NP + n];
      const float4 v = c != kNoRow ? y[d] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      AP[(size_t)(d * KG + grp) * NP + n] = v;
      pap[0] += (double)pc.x * v.x;
      pap[1] += (double)pc.y * v.y;
      pap[2] += (double)pc.z * v.z;
      pap[3] += (double)pc.w * v.w;
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const double s = wave_sum_dpp(pap[r]);
    if (lane == 0) lds[wv][r] = s;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kApWaves; ++w) s += lds[w][threadIdx.x];
    part1[(size_t)(r0 + threadIdx.x) * nblk + lb] = s;
  }
}

// blocks of a stencil kernel over NP nodes
int stencil_blocks(const Grid &g) { return (int)nblk(mshape(g).NP, kApNodes * kApWaves); }
size_t stencil_code_len(const Grid &g) { return mshape(g).NP; }
size_t stencil_table_len() { return (size_t)kNumStencils * kStencilFloats; }

hipError_t launch_d_setup(const Grid &g, const int *et, const double *ke, uint16_t *code, float *tab, hipStream_t st) {
  const int NP = mshape(g).NP;
  hipLaunchKernelGGL(k_d_code, dim3(NP / 256), dim3(256), 0, st, g, NP, et, code);
  hipLaunchKernelGGL(k_d_table, dim3(kNumStencils), dim3(256), 0, st, ke, tab);
  return hipGetLastError();
}

hipError_t launch_d_spmv(const Grid &g, int K, const StencilOp &op, const float *P, float *AP, double *part1,
                         const void *state, hipStream_t st) {
  const int NP = mshape(g).NP, nb = stencil_blocks(g), per = (nb + 7) / 8;
  MPP_K_DISPATCH(K, hipLaunchKernelGGL(k_d_spmv<KK>, dim3(8 * per, KK / 4), dim3(64 * kApWaves), 0, st, g, NP, nb,
                                       per, op.code, op.tab, reinterpret_cast<const float4 *>(P),
                                       reinterpret_cast<float4 *>(AP), part1, static_cast<const MState *>(state)));
  return hipGetLastError();
}

}  // namespace mpp
