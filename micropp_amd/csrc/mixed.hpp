// mixed.hpp -- what the FP32 inner solver's translation units share: the CG
// state of the K fields, fixed-order sums of partial tables, block order and
// lane shifts (mixed.hip: the CG and its stored-matrix SpMV; vcycle.hip: the
// stencil-dictionary SpMV and the multilevel preconditioner).
#pragma once

#include "internal.hpp"
#include "kernels.hpp"
#include "physics.hpp"
#include "reduce.hpp"

namespace mpp {

constexpr int kMaxRhs = 16;
constexpr int kRowQuads = 7, kRows = 9;         // stencil rows (dz, dy) of 27 floats + 1 pad
constexpr int kNodeQuads = kRowQuads * kRows;  // 63 float4 per node
__host__ __device__ constexpr int mslot(int nb, int fi, int fj) { return (nb / 3) * 28 + (nb % 3) * 9 + fi * 3 + fj; }
constexpr int kRedThreads = 256;  // threads of the one-block reducers
constexpr int kVecNodes = 2048;   // nodes per block of the vector kernels
// Blocks of kVecNodes nodes from which the vector kernels of the multi-RHS CG
// keep them; with fewer, blocks of 512 nodes.  Iteration, us, 512 / 2048 nodes:
// 11^3 nodes of 8 fields (6 blocks) 37.0 / 38.5, 26^3 of 16 (108) 64.2 / 67.6,
// 31^3 of 16 (180) 81.4 / 83.9, 41^3 of 8 (204) 86.6 / 85.3, 46^3 of 12 (432)
// 127 / 121.
constexpr size_t kVecWide = 200;

// inner CG scalars per field: rz = (r, z), alpha / beta of the iteration, pn
// the current ||z||, pn0 the start value, tau the relative stop; broken: the
// preconditioner has shown itself not positive definite (spd_broken)
struct MState {
  double rz[kMaxRhs], alpha[kMaxRhs], beta[kMaxRhs], pn[kMaxRhs], pn0[kMaxRhs], tau[kMaxRhs];
  int done[kMaxRhs];
  int its, max_its, all_done, broken;
};

// (r, z) not positive on a field that has not reached its stop: z = M r with a
// preconditioner that is not positive definite (a start value that is not a
// number is not its doing)
__device__ __forceinline__ bool spd_broken(double rz, double pn, double pn0, double tau) {
  return !(rz > 0.0) && !(pn < tau * pn0) && pn0 - pn0 == 0.0;
}

// all fields, or the four fields r0 .. r0 + 3 of a group, have stopped (one
// round of loads: no test waits for another's)
__device__ __forceinline__ bool group_stopped(const MState *s, int r0) {
  const int all = s->all_done;
  const int4 d = *reinterpret_cast<const int4 *>(&s->done[r0]);
  return (all | (d.x & d.y & d.z & d.w)) != 0;
}

// outer (defect-correction) test per field: pn = ||kinv r|| (the reference
// CG's metric), rn = ||r||_2 over the interior DOFs (assembly_rhs's norm:
// its Dirichlet rows are zero), and their values at the last `first` call
struct MOuter {
  double pn[kMaxRhs], pn0[kMaxRhs], target[kMaxRhs], rn[kMaxRhs], rn0[kMaxRhs];
  int conv[kMaxRhs];
  int all_conv, pad[3];
};

typedef float f4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bool node_on_boundary(const Grid &g, int i, int j, int k) {
  return i == 0 || j == 0 || k == 0 || i == g.nx - 1 || j == g.ny - 1 || k == g.nz - 1;
}

// Blocks are dispatched round-robin over the 8 XCDs; launch 8 * per blocks and
// give XCD x the logical blocks [x * per, (x + 1) * per).
__device__ __forceinline__ int xcd_block(int per) {
  const int b = blockIdx.x;
  return (b & 7) * per + (b >> 3);
}

// Row sums of a partial table part[row * stride + j], j < n, rows < NR, by
// one block of kRedThreads: every thread accumulates its entries j = t,
// t + kRedThreads, ... of all rows (independent loads, all in flight), each
// wave adds its lanes with DPP moves, and thread t < NR adds the waves' sums
// of row t.  Fixed order throughout.  Thread t < NR returns the sum of row t
// (others return 0).
// The two halves of rows_sum, for callers that issue other loads in between
// (vector-memory loads complete in issue order, so loads issued after the
// partials' do not delay their sum): rows_load adds this thread's entries of
// each row in index order, rows_finish combines the threads.
template <int NR, int UNROLL = 1>
__device__ __forceinline__ void rows_load(const double *part, size_t stride, int n, double (&s)[NR]) {
#pragma unroll
  for (int q = 0; q < NR; ++q) s[q] = 0.0;
  // UNROLL > 1 keeps several rounds of loads in flight (long rows)
#pragma unroll UNROLL
  for (int j = threadIdx.x; j < n; j += kRedThreads)
#pragma unroll
    for (int q = 0; q < NR; ++q) s[q] += part[(size_t)q * stride + j];
}
template <int NR>
__device__ __forceinline__ double rows_finish(double (&s)[NR]) {
  static_assert(NR <= kRedThreads, "one row per thread at the end");
  constexpr int kW = kRedThreads / 64;
  __shared__ double lds[kW][NR];
  const int t = threadIdx.x, w = t >> 6;
  __syncthreads();  // lds may still be read by a previous call
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    const double v = wave_sum_dpp(s[q]);
    if ((t & 63) == 0) lds[w][q] = v;
  }
  __syncthreads();
  double r = 0.0;
  if (t < NR)
    for (int i = 0; i < kW; ++i) r += lds[i][t];
  return r;
}
template <int NR, int UNROLL = 1>
__device__ __forceinline__ double rows_sum(const double *part, size_t stride, int n) {
  double s[NR];
  rows_load<NR, UNROLL>(part, stride, n, s);
  return rows_finish<NR>(s);
}

// ---------------------------------------------------------------------------
// What an operator kernel does with y = A P at a node (one direction, four
// fields; pc = P there): see k_m_spmv and k_d_apply.
// ---------------------------------------------------------------------------
enum ApplyMode { kApplyCg, kApplyRes, kApplyPost, kApplyPow };
template <int MODE>
__device__ __forceinline__ void apply_out(const float4 &pc, const float4 &y, const float4 *R, const float *kinv,
                                          float omega, float4 *OUT, size_t o, size_t ok, double (&s)[4]) {
  float4 v = y;
  if constexpr (MODE == kApplyRes || MODE == kApplyPost) {
    const float4 r = R[o];
    if constexpr (MODE == kApplyRes) {
      v = make_float4(r.x - omega * y.x, r.y - omega * y.y, r.z - omega * y.z, r.w - omega * y.w);
    } else {
      const float w = omega * kinv[ok];
      v = make_float4(pc.x + w * (r.x - y.x), pc.y + w * (r.y - y.y), pc.z + w * (r.z - y.z), pc.w + w * (r.w - y.w));
      s[0] += (double)r.x * v.x;
      s[1] += (double)r.y * v.y;
      s[2] += (double)r.z * v.z;
      s[3] += (double)r.w * v.w;
    }
  } else if constexpr (MODE == kApplyCg) {
    s[0] += (double)pc.x * y.x;
    s[1] += (double)pc.y * y.y;
    s[2] += (double)pc.z * y.z;
    s[3] += (double)pc.w * y.w;
  } else {  // kApplyPow
    const float w = kinv[ok];
    v = make_float4(w * y.x, w * y.y, w * y.z, w * y.w);
    s[0] += (double)v.x * y.x;
    s[1] += (double)v.y * y.y;
    s[2] += (double)v.z * y.z;
    s[3] += (double)v.w * y.w;
  }
  OUT[o] = v;
}

// ---------------------------------------------------------------------------
// The element blocks (phase table or per element) around interior node n:
// blk[q] the 24x24 block of element q = (a*2+b)*2+c, la[q] the node's local
// index in it.  Entry (fi, fj) of the node block towards neighbour nb is the
// FP64 sum of the element contributions in the reference element order.
// ---------------------------------------------------------------------------
struct NodeBlocks {
  const double *blk[8];
  int la[8];
  __device__ NodeBlocks(const Grid &g, int i, int j, int k, const int *et, const double *ke, int phase_mode) {
    for (int a = 0; a < 2; ++a)
      for (int b = 0; b < 2; ++b)
        for (int c = 0; c < 2; ++c) {
          const int q = (a * 2 + b) * 2 + c;
          const int e = ((k - 1 + c) * g.ney + (j - 1 + b)) * g.nex + (i - 1 + a);
          blk[q] = ke + (size_t)(phase_mode ? et[e] : e) * 576;
          la[q] = local_node(1 - a, 1 - b, 1 - c);
        }
  }
  __device__ double entry(int nb, int fi, int fj) const {
    const int dz = nb / 9 - 1, dy = (nb / 3) % 3 - 1, dx = nb % 3 - 1;
    double acc = 0.0;
    for (int a = 0; a < 2; ++a) {
      const int px = 1 - a + dx;
      if (px < 0 || px > 1) continue;
      for (int b = 0; b < 2; ++b) {
        const int py = 1 - b + dy;
        if (py < 0 || py > 1) continue;
        for (int c = 0; c < 2; ++c) {
          const int pz = 1 - c + dz;
          if (pz < 0 || pz > 1) continue;
          const int q = (a * 2 + b) * 2 + c;
          acc += blk[q][(la[q] * 3 + fi) * 24 + local_node(px, py, pz) * 3 + fj];
        }
      }
    }
    return acc;
  }
};

// DPP wave shifts: lane i takes lane i - 1's value (lane 0 keeps `old`), or
// lane i + 1's (lane 63 keeps `old`)
__device__ __forceinline__ float4 from_left(const float4 &v, const float4 &old) {
  auto f = [](float x, float o) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(o), __float_as_int(x), 0x138, 0xf, 0xf, false));
  };
  return make_float4(f(v.x, old.x), f(v.y, old.y), f(v.z, old.z), f(v.w, old.w));
}
__device__ __forceinline__ float4 from_right(const float4 &v, const float4 &old) {
  auto f = [](float x, float o) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(o), __float_as_int(x), 0x130, 0xf, 0xf, false));
  };
  return make_float4(f(v.x, old.x), f(v.y, old.y), f(v.z, old.z), f(v.w, old.w));
}

inline unsigned nblk(size_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

struct MLaunch {
  int NP;         // nodes rounded up to 256
  int per, nb;    // node blocks of 256 per XCD, blocks launched (8 * per)
  int nsl, pers;  // slices of 64 nodes, slices per XCD (8 * pers launched)
  int nbx;        // blocks of 256 float4 per component
};

inline MLaunch mshape(const Grid &g) {
  MLaunch s;
  s.NP = (int)round_up((size_t)g.nn, 256);
  s.per = (s.NP / 256 + 7) / 8;
  s.nb = s.per * 8;
  s.nsl = s.NP / 64;
  s.pers = (s.nsl + 7) / 8;
  s.nbx = (int)nblk((size_t)s.NP / 4, 256);
  return s;
}

#define MPP_K_DISPATCH(K, CALL)                     \
  switch (K) {                                      \
    case 4: {                                       \
      constexpr int KK = 4;                         \
      CALL;                                         \
    } break;                                        \
    case 8: {                                       \
      constexpr int KK = 8;                         \
      CALL;                                         \
    } break;                                        \
    case 12: {                                      \
      constexpr int KK = 12;                        \
      CALL;                                         \
    } break;                                        \
    case 16: {                                      \
      constexpr int KK = 16;                        \
      CALL;                                         \
    } break;                                        \
    default:                                        \
      return hipErrorInvalidValue;                  \
  }

}  // namespace mpp
