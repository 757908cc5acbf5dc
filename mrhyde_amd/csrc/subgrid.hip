// subgrid.hip — batched multiscale subgrid solves: thousands of independent
// small Q1 thermal problems assembled and solved (Jacobi-PCG to a relative
// residual) in ONE persistent launch.
//
// Replaces the per-macro-group loop of the reference multiscale layer, which
// solves one subgrid system at a time with its own assembly and Krylov solve:
//   MultiscaleManager::evaluateMacroMicroMacroMap   multiscaleManager.cpp:866-1188
//   SubGridDtN::subgridSolver                        subgridDtN.cpp:985-1121
//   SubGridDtN_Solver::nonlinearSolver / assembleJacobianResidual
//                                                    subgridDtN_solver.cpp:903-1043, :681-902
// with the PCG of SolverManager::PCG (solverManager_solvers.hpp:812-905).
//
// Instance: a box [0,Lx]x[0,Ly]x[0,Lz] (the unit cube by default) cut into
// n^3 Q1 hexahedra (n per instance), element conductivity k_e, optional
// element source f_e, Dirichlet data g on every boundary node.  The system is
// J du = -F(u0) with u0 = g on the boundary (reference strong-DBC convention)
// and F(u) = A u - b, b_i = sum over the elements e of node i of f_e |e| / 8,
// solved on the interior nodes; the result is u = u0 + du.
//
// Mapping: one workgroup owns one instance at a time and pulls the next from
// a global counter (largest instances first) until the queue is empty, so
// every workgroup reaches the exit.  The instance lives on chip: the search
// direction p and the element conductivities in LDS, each thread's share of
// x, r and the Jacobi scaling in registers.  A thread owns a run of interior
// nodes of one z column and sweeps its planes upwards: the operator is the
// closed-form Q1 stiffness of the instance's box element (exact for the
// 2x2x2 Gauss rule the reference uses), and a plane's values are read once
// for the nodes below, in and above it.  Per node 9 p values and 4
// conductivities from LDS and about 30 floating-point operations on the unit
// cube; one node at a time from its 27 neighbours and 8 elements took 35 LDS
// reads, 72 operations and two index divisions.  Milliseconds a batch, before
// -> now: 1,024 unit cubes in FP64 0.79 -> 0.49, 256 boxes with sources in
// FP32-refined 0.73 -> 0.39, 4,096 unit cubes 2.73 -> 1.71 and 2.53 -> 1.42.

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "mhx_internal.hpp"

namespace mhx {

// ---- box trilinear stiffness -------------------------------------------------
// On a box element of sides (hx, hy, hz) the Q1 stiffness is
//   K = cx S(x)M(x)M + cy M(x)S(x)M + cz M(x)M(x)S,
//   cx = hy hz / hx, cy = hx hz / hy, cz = hx hy / hz,
// with the 1-D S = [1 -1; -1 1] and M = [1/3 1/6; 1/6 1/3].  An entry depends
// only on which of the two nodes' coordinates differ: kv[dx + 2 dy + 4 dz].
inline void box_stencil(double hx, double hy, double hz, double kv[8]) {
  const double cx = hy * hz / hx, cy = hx * hz / hy, cz = hx * hy / hz;
  const double S[2] = {1.0, -1.0}, M[2] = {1.0 / 3.0, 1.0 / 6.0};
  for (int p = 0; p < 8; ++p) {
    const int dx = p & 1, dy = (p >> 1) & 1, dz = (p >> 2) & 1;
    kv[p] = cx * S[dx] * M[dy] * M[dz] + cy * M[dx] * S[dy] * M[dz] + cz * M[dx] * M[dy] * S[dz];
  }
}

constexpr int kSgMaxN = 16;                                   // elements per axis
constexpr int kSgMaxNodes = (kSgMaxN + 1) * (kSgMaxN + 1) * (kSgMaxN + 1);
constexpr int kSgMaxElems = kSgMaxN * kSgMaxN * kSgMaxN;

struct SgInst {
  int n;       // elements per axis
  int k_off;   // offset of the instance's element coefficients
  int x_off;   // offset of the instance's nodal arrays
  int pad;
  double kv[8];  // element stiffness entries by coordinate-difference pattern
  double vol8;   // element volume / 8: the share of a node in a constant source
};

struct SgArgs {
  const SgInst* inst;
  const int* order;      // queue position -> instance (largest first)
  int n_inst;
  const double* k;
  const double* src;     // element sources (nullptr: none)
  const double* g;
  double* x;
  int* iters;
  double* relres;
  int* refinements;
  unsigned int* queue;
  double tol;
  int max_iters;
  int fp32;              // FP32 inner CG inside FP64 iterative refinement
  double inner_tol;
  int max_refine;
};

__global__ void k_sg_reset(unsigned int* q) { *q = 0u; }

// A thread's nodes: the interior column (ix, iy), z = z0 .. z0 + cnt - 1.
struct SgCol {
  int p, e;  // node (ix, iy, z0) in the nodal arrays; element (ix-1, iy-1, z0-1)
  int cnt;
};

// q = A p at the thread's nodes, p and k in LDS: out(s, q_s, p_s) for s <
// cnt.  BOX (the general instance: a box, possibly with sources): kv holds
// the box element's stiffness entries by coordinate-difference pattern; else
// the instance is the unit cube, whose element couples a node to itself (1/3)
// and to its face and body diagonals (-1/12) and not along edges, scaled by
// h = 1 / n.
//
// Plane j (z = z0 - 1 + j) lies below node j, holds node j - 1 and lies above
// node j - 2; element layer j is between planes j and j + 1.  Straight-line
// over C slots; slots from cnt on give values that the caller drops.
template <class T, int C, bool BOX, class Out>
__device__ __forceinline__ void sg_apply(const T* __restrict__ p, const T* __restrict__ kk, int n, const T (&kv)[8],
                                         const SgCol& c, Out&& out) {
  const int n1 = n + 1, pl = n1 * n1, el = n * n;
  const T* P = p + c.p - pl;
  const T* K = kk + c.e;
  const T h = (T)-1 / (T)(12 * n);
  T kl[4] = {0, 0, 0, 0}, prev = 0, cur = 0, pc_prev = 0;
#pragma unroll
  for (int j = 0; j < C + 2; ++j) {
    // one plane at a time (bounds the live registers)
    __builtin_amdgcn_sched_barrier(0);
    // corner ab of the plane: a = 0, 1: x - 1, x + 1; b: y; edge neighbours x, y
    const T m0 = P[-1 - n1], m1 = P[1 - n1], m2 = P[-1 + n1], m3 = P[1 + n1];
    const T xm = P[-1], xp = P[1], ym = P[-n1], yp = P[n1], pc = P[0];
    const T kh[4] = {K[0], K[1], K[n], K[n + 1]};
    // what an element above or below the plane adds per unit conductivity
    T t[4];
    if constexpr (BOX) {
      const T ax = kv[5] * xm, bx = kv[5] * xp, cz = kv[4] * pc;
      const T ay = fma(kv[6], ym, cz), by = fma(kv[6], yp, cz);
      t[0] = fma(kv[7], m0, ax + ay);
      t[1] = fma(kv[7], m1, bx + ay);
      t[2] = fma(kv[7], m2, ax + by);
      t[3] = fma(kv[7], m3, bx + by);
    } else {
      t[0] = m0 + (xm + ym);
      t[1] = m1 + (xp + ym);
      t[2] = m2 + (xm + yp);
      t[3] = m3 + (xp + yp);
    }
    if (j >= 2) {
      const T q = fma(kl[0], t[0], fma(kl[1], t[1], fma(kl[2], t[2], fma(kl[3], t[3], prev))));
      if constexpr (BOX) out(j - 2, q, pc_prev);
      else out(j - 2, q * h, pc_prev);
    }
    if (j >= 1 && j <= C) {
      const T s0 = kl[0] + kh[0], s1 = kl[1] + kh[1], s2 = kl[2] + kh[2], s3 = kl[3] + kh[3];
      if constexpr (BOX) {
        const T ax = kv[1] * xm, bx = kv[1] * xp, cc = kv[0] * pc;
        const T ay = fma(kv[2], ym, cc), by = fma(kv[2], yp, cc);
        cur = fma(s0, fma(kv[3], m0, ax + ay), cur);
        cur = fma(s1, fma(kv[3], m1, bx + ay), cur);
        cur = fma(s2, fma(kv[3], m2, ax + by), cur);
        cur = fma(s3, fma(kv[3], m3, bx + by), cur);
      } else {
        const T d = fma(s0, m0, fma(s1, m1, fma(s2, m2, fma(s3, m3, cur))));
        // in units of -h / 12: the diagonals, and -4 (h / 3) for the node itself
        cur = fma((T)-4 * ((s0 + s1) + (s2 + s3)), pc, d);
      }
    }
    T nxt = 0;
    if (j < C) nxt = fma(kh[0], t[0], fma(kh[1], t[1], fma(kh[2], t[2], kh[3] * t[3])));
    prev = cur;
    cur = nxt;
    pc_prev = pc;
#pragma unroll
    for (int q = 0; q < 4; ++q) kl[q] = kh[q];
    // past the thread's last plane and layer: stay there (unused slots)
    P += j <= c.cnt ? pl : 0;
    K += j < c.cnt ? el : 0;
  }
}

// sum of the eight conductivities around the thread's nodes (the operator's
// diagonal is kv[0] times it, h / 3 on the unit cube) and, where f is given,
// of the element sources: out(s, sum k, sum f)
template <int C, class Out>
__device__ __forceinline__ void sg_around(const double* __restrict__ kk, const double* __restrict__ f, int n,
                                          const SgCol& c, Out&& out) {
  double klo = 0.0, flo = 0.0;
#pragma unroll
  for (int j = 0; j < C + 1; ++j) {
    const int e = c.e + min(j, max(c.cnt - 1, 0) + 1) * n * n;
    const double khi = (kk[e] + kk[e + 1]) + (kk[e + n] + kk[e + n + 1]);
    const double fhi = f ? (f[e] + f[e + 1]) + (f[e + n] + f[e + n + 1]) : 0.0;
    if (j >= 1) out(j - 1, klo + khi, flo + fhi);
    klo = khi;
    flo = fhi;
  }
}

// Sum of two values over the workgroup, returned to every thread; red holds
// two copies used in turn (buf), so one barrier separates a copy's readers
// from its next writers.
template <int WG, class T>
__device__ __forceinline__ void wg_sum2(T& a, T& b, T* red, int& buf) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_xor(a, off, 64);
    b += __shfl_xor(b, off, 64);
  }
  T* r = red + buf * 2 * (WG / 64);
  buf ^= 1;
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  if (l == 0) {
    r[2 * w] = a;
    r[2 * w + 1] = b;
  }
  __syncthreads();
  a = 0;
  b = 0;
#pragma unroll
  for (int i = 0; i < WG / 64; ++i) {
    a += r[2 * i];
    b += r[2 * i + 1];
  }
}

// Jacobi-PCG on the interior nodes (SolverManager::PCG algorithm):
//   x += CG solution of A x = r_in (r_in given in the thread's slots),
// stopping when ||r|| / ||r_in|| <= tol.  p_lds is 0 on the boundary nodes.
// Returns iterations; rr_out = ||r||^2.
template <int WG, int C, class T, bool BOX>
__device__ __forceinline__ int sg_pcg(int n, const T* kk, const T (&kv)[8], T* p_lds, T* red, T (&x)[C], T (&r)[C],
                                      const T (&dinv)[C], SgCol& c, double tol, int max_iters, T& rr_out) {
  const int pl = (n + 1) * (n + 1);
  int buf = 0;
  T rr = 0, rz = 0;
#pragma unroll
  for (int s = 0; s < C; ++s) {
    rr += r[s] * r[s];
    rz += r[s] * (dinv[s] * r[s]);  // z = D^-1 r (dinv is 0 in unused slots)
  }
  wg_sum2<WG>(rr, rz, red, buf);
  const T rr0 = rr;
  int it = 0;
  if (rr0 > (T)0) {
#pragma unroll
    for (int s = 0; s < C; ++s)
      if (s < c.cnt) p_lds[c.p + s * pl] = dinv[s] * r[s];
    __syncthreads();
    const T tol2 = (T)(tol * tol);
    while (it < max_iters) {
      // (opaque once per iteration: the planes' addresses are formed in the
      // sweep instead of being hoisted and held across iterations)
      __asm__ volatile("" : "+v"(c.p), "+v"(c.e), "+v"(c.cnt));
      T q[C];
#pragma unroll
      for (int s = 0; s < C; ++s) q[s] = 0;
      T pq = 0, dummy = 0;
      sg_apply<T, C, BOX>(p_lds, kk, n, kv, c, [&](int s, T qs, T ps) __attribute__((always_inline)) {
        q[s] = s < c.cnt ? qs : (T)0;
        pq = fma(s < c.cnt ? ps : (T)0, q[s], pq);
      });
      wg_sum2<WG>(pq, dummy, red, buf);
      const T alpha = rz / pq;
      T rr1 = 0, rz1 = 0, pp[C];
#pragma unroll
      for (int s = 0; s < C; ++s) {
        pp[s] = s < c.cnt ? p_lds[c.p + s * pl] : (T)0;
        x[s] += alpha * pp[s];
        r[s] -= alpha * q[s];
        rr1 += r[s] * r[s];
        rz1 += r[s] * (dinv[s] * r[s]);
      }
      wg_sum2<WG>(rr1, rz1, red, buf);
      ++it;
      rr = rr1;
      if (!(rr > tol2 * rr0)) break;  // also leaves on NaN
      const T beta = rz1 / rz;
      rz = rz1;
#pragma unroll
      for (int s = 0; s < C; ++s)
        if (s < c.cnt) p_lds[c.p + s * pl] = dinv[s] * r[s] + beta * pp[s];
      __syncthreads();
    }
  }
  rr_out = rr;
  return it;
}

// One instance by one workgroup; C: slots of a thread, at least its run of nodes.
template <int WG, int C, bool MIXED, bool BOX>
__device__ __forceinline__ void sg_instance(const SgArgs& a, int id, double* p64, double* k64, double* red,
                                            float* red32) {
  float* p32 = reinterpret_cast<float*>(p64);  // FP32 views: p in the lower, k in the upper half of p64's storage
  float* k32 = reinterpret_cast<float*>(p64) + kSgMaxNodes;
  const SgInst in_ = a.inst[id];
  const int n = in_.n, n1 = n + 1, pl = n1 * n1, nn = n1 * pl, ne = n * n * n;
  const double* kg = a.k + in_.k_off;
  const double* fg = a.src ? a.src + in_.k_off : nullptr;
  const double* gg = a.g + in_.x_off;
  double kv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) kv[i] = in_.kv[i];

  // the thread's run of nodes (idle threads: the first column, no node)
  SgCol c{n1 + 1 + pl, 0, 0};
  {
    const int m = n - 1, cols = m * m, per = min(WG / cols, m), run = (m + per - 1) / per;
    const int part = threadIdx.x / cols, col = threadIdx.x - part * cols;
    const int cy = col / m, cx = col - cy * m, z0 = part * run;
    if (part < per && z0 < m) {
      c.cnt = min(run, m - z0);
      c.p = (cx + 1) + n1 * (cy + 1) + pl * (z0 + 1);
      c.e = cx + n * cy + n * n * z0;
    }
  }
  for (int e = threadIdx.x; e < ne; e += WG) k64[e] = kg[e];
  // u0: the Dirichlet lift (data) or 0 on the boundary nodes, 0 inside
  auto lift = [&](bool data) {
    for (int v = threadIdx.x; v < nn; v += WG) {
      const int iz = v / pl, w = v - iz * pl, iy = w / n1, ix = w - iy * n1;
      const bool bnd = ix == 0 || iy == 0 || iz == 0 || ix == n || iy == n || iz == n;
      p64[v] = data && bnd ? gg[v] : 0.0;
    }
  };
  lift(true);
  __syncthreads();
  // b - A u0 = -F(u0) on interior rows (assembled residual with the Dirichlet lift)
  double r[C], x[C], dinv[C], b[BOX ? C : 1];
#pragma unroll
  for (int s = 0; s < C; ++s) x[s] = 0.0;
  sg_around<C>(k64, BOX ? fg : nullptr, n, c, [&](int s, double ks, double fs) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);  // one division at a time
    dinv[s] = s < c.cnt ? 1.0 / (kv[0] * ks) : 0.0;
    if constexpr (BOX) b[s] = in_.vol8 * fs;
  });
  auto residual = [&]() __attribute__((always_inline)) {
    sg_apply<double, C, BOX>(p64, k64, n, kv, c, [&](int s, double q, double) __attribute__((always_inline)) {
      r[s] = s < c.cnt ? (BOX ? b[BOX ? s : 0] : 0.0) - q : 0.0;
    });
  };
  residual();
  int its = 0, refs = 0;
  double rr = 0.0, bb = 0.0, dummy = 0.0;
#pragma unroll
  for (int s = 0; s < C; ++s) bb += r[s] * r[s];
  int buf = 0;
  wg_sum2<WG>(bb, dummy, red, buf);
  if constexpr (!MIXED) {
    lift(false);
    __syncthreads();
    its = sg_pcg<WG, C, double, BOX>(n, k64, kv, p64, red, x, r, dinv, c, a.tol, a.max_iters, rr);
  } else {
    // FP32 inner PCG inside FP64 iterative refinement: the residual, the
    // accumulated correction and the convergence test stay FP64.
    const double target2 = a.tol * a.tol * bb;
    rr = bb;
    while (refs < a.max_refine && rr > target2 && its < a.max_iters) {
      const double scale = std::sqrt(rr);
      __syncthreads();
      for (int e = threadIdx.x; e < ne; e += WG) k32[e] = (float)k64[e];
      for (int v = threadIdx.x; v < nn; v += WG) p32[v] = 0.f;
      float xf[C], rf[C], df[C];
#pragma unroll
      for (int s = 0; s < C; ++s) {
        xf[s] = 0.f;
        rf[s] = (float)(r[s] / scale);
        df[s] = (float)dinv[s];
      }
      __syncthreads();
      float rrf = 0.f, kvf[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) kvf[i] = (float)kv[i];
      its += sg_pcg<WG, C, float, BOX>(n, k32, kvf, p32, red32, xf, rf, df, c, a.inner_tol, a.max_iters - its, rrf);
      ++refs;
      // x += scale * xf ; r = b - A (u0 + x) in FP64
      __syncthreads();
      lift(true);
      __syncthreads();
#pragma unroll
      for (int s = 0; s < C; ++s) {
        x[s] += scale * (double)xf[s];
        if (s < c.cnt) p64[c.p + s * pl] = x[s];
      }
      __syncthreads();
      residual();
      double rr2 = 0.0, d2 = 0.0;
#pragma unroll
      for (int s = 0; s < C; ++s) rr2 += r[s] * r[s];
      wg_sum2<WG>(rr2, d2, red, buf);
      rr = rr2;
    }
  }
  // u = u0 + du, through LDS (a thread's nodes are a plane apart)
  __syncthreads();
#pragma unroll
  for (int s = 0; s < C; ++s)
    if (s < c.cnt) p64[c.p + s * pl] = x[s];
  __syncthreads();
  for (int v = threadIdx.x; v < nn; v += WG) {
    const int iz = v / pl, w = v - iz * pl, iy = w / n1, ix = w - iy * n1;
    const bool bnd = ix == 0 || iy == 0 || iz == 0 || ix == n || iy == n || iz == n;
    a.x[in_.x_off + v] = bnd ? gg[v] : p64[v];
  }
  if (threadIdx.x == 0) {
    a.iters[id] = its;
    a.relres[id] = bb > 0.0 ? std::sqrt(rr / bb) : 0.0;
    if (a.refinements) a.refinements[id] = refs;
  }
}

// A thread's run of nodes: the n - 1 interior nodes of a column over as many
// threads as the workgroup holds per column (16 elements, 225 columns: 8 at
// 512 threads, 4 at 1024).  The sweep is built for the runs that occur, so a
// small instance does not walk a large one's slots.
template <int WG, bool MIXED, bool BOX>
__global__ __launch_bounds__(WG) void k_subgrid(SgArgs a) {
  __shared__ double p64[kSgMaxNodes];
  __shared__ double k64[kSgMaxElems];
  __shared__ double red[2 * 2 * (WG / 64)];
  __shared__ float red32[MIXED ? 2 * 2 * (WG / 64) : 1];
  __shared__ int s_next;

  for (;;) {
    if (threadIdx.x == 0) s_next = (int)atomicAdd(a.queue, 1u);
    __syncthreads();
    // (wave-uniform: the instance's description is then read with scalar
    // loads and its stencil entries stay in scalar registers)
    const int qpos = __builtin_amdgcn_readfirstlane(s_next);
    __syncthreads();
    if (qpos >= a.n_inst) break;
    const int id = a.order[qpos];
    const int m = a.inst[id].n - 1, per = min(WG / (m * m), m), run = (m + per - 1) / per;
    if (run == 1) sg_instance<WG, 1, MIXED, BOX>(a, id, p64, k64, red, red32);
    else if (run == 2) sg_instance<WG, 2, MIXED, BOX>(a, id, p64, k64, red, red32);
    else if (run == 3) sg_instance<WG, 3, MIXED, BOX>(a, id, p64, k64, red, red32);
    else if (WG == 1024 || run == 4) sg_instance<WG, 4, MIXED, BOX>(a, id, p64, k64, red, red32);
    else if (run == 5) sg_instance<WG, WG == 1024 ? 4 : 5, MIXED, BOX>(a, id, p64, k64, red, red32);
    else sg_instance<WG, WG == 1024 ? 4 : 8, MIXED, BOX>(a, id, p64, k64, red, red32);
    __syncthreads();
  }
}

}  // namespace mhx

// =============================================================================
// host side: batch object, autotuner, graph capture, C ABI
// =============================================================================
namespace mhx {

// Copies of large results to ordinary host memory.  The runtime's own path
// moves them through one staging buffer with one copying thread (14.2 MB took
// 0.86 ms, longer than the solve; now 0.52).  Here kWorkers threads each take
// every kWorkers-th chunk through a pinned buffer of their own, so the device
// fills some buffers while others are copied out.  Chunks of a quarter of the
// array, up to 2 MiB: each transfer costs about 15 us of its own (512 KiB
// chunks 0.74 ms, 1 MiB 0.55).  One ring of 8 MiB per device, shared by its
// batches (one copy at a time; a second caller takes the runtime's path).  It
// outlives them until mhx_release_host_buffers: a macro loop that creates and
// destroys a batch per step would allocate and free it in every step (results
// and destruction of 4 and 14 MB: 0.47 and 0.76 ms, kept 0.42 and 0.72, the
// runtime's path 0.39 and 0.99).
struct CopyRing {
  static constexpr int kWorkers = 4;
  static constexpr size_t kChunk = 2u << 20;
  // From 3.5 MiB on: the threads and transfers cost about 0.13 ms whatever the
  // size.  Runtime's path / ring, us: 1 MiB 72/142, 2 MiB 133/161, 3 MiB
  // 224/236, 3.6 MiB 262/259, 4.2 MiB 308/272, 8 MiB 498/336.
  static constexpr size_t kMinBytes = 7u << 19;
  int dev = 0;
  char* buf = nullptr;
  hipEvent_t ev[kWorkers] = {};
  std::mutex busy;
  explicit CopyRing(int d) : dev(d) {
    MHX_HIP(hipHostMalloc((void**)&buf, kWorkers * kChunk, hipHostMallocDefault));
    for (auto& e : ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        release();
        throw Error{MHX_ERR_DEVICE, "result copies: event creation failed"};
      }
  }
  CopyRing(const CopyRing&) = delete;
  CopyRing& operator=(const CopyRing&) = delete;
  ~CopyRing() { release(); }
  void release() {
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    if (buf) (void)hipHostFree(buf);
    buf = nullptr;
  }
  // worker w's chunks w, w + kWorkers, ... of src -> dst
  hipError_t work(int w, hipStream_t stream, char* dst, const char* src, size_t bytes, size_t chunk, bool own_thread) {
    char* mine = buf + (size_t)w * kChunk;
    hipError_t e = own_thread ? hipSetDevice(dev) : hipSuccess;
    for (size_t at = (size_t)w * chunk; at < bytes && e == hipSuccess; at += kWorkers * chunk) {
      const size_t len = std::min(chunk, bytes - at);
      e = hipMemcpyAsync(mine, src + at, len, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipEventRecord(ev[w], stream);
      if (e == hipSuccess) e = hipEventSynchronize(ev[w]);
      if (e == hipSuccess) std::memcpy(dst + at, mine, len);
    }
    return e;
  }
};

// the devices' rings (never destroyed: at process exit the runtime may be gone)
struct CopyRings {
  std::mutex mu;
  std::map<int, std::shared_ptr<CopyRing>> of;
};
static CopyRings& copy_rings() {
  static CopyRings* r = new CopyRings;
  return *r;
}
static std::shared_ptr<CopyRing> copy_ring(int dev) {
  CopyRings& all = copy_rings();
  std::lock_guard<std::mutex> lk(all.mu);
  std::shared_ptr<CopyRing>& r = all.of[dev];
  if (!r) r = std::make_shared<CopyRing>(dev);
  return r;
}

struct Batch {
  int dev = 0;  // the device it was created on
  int n_inst = 0;
  long total_nodes = 0, total_elems = 0;
  std::vector<SgInst> h_inst;
  std::vector<int> h_order;
  DevBuf<SgInst> inst;
  DevBuf<int> order, iters, refs;
  DevBuf<double> k, src, g, x, relres;
  DevBuf<unsigned int> queue;
  hipStream_t stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int graph_wg = 0;
  bool box = false;  // instances with their own side lengths or sources (else unit cubes, no source)
  int wg = 0;
  int grid[2] = {0, 0};  // per WG variant (512, 1024)
  mhx_batch_desc desc{};
  double last_ms = 0.0;
  std::string err;
  ~Batch() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

static SgArgs make_args(Batch& b) {
  SgArgs a{};
  a.inst = b.inst.p;
  a.order = b.order.p;
  a.n_inst = b.n_inst;
  a.k = b.k.p;
  a.src = b.src.p;
  a.g = b.g.p;
  a.x = b.x.p;
  a.iters = b.iters.p;
  a.relres = b.relres.p;
  a.refinements = b.refs.p;
  a.queue = b.queue.p;
  a.tol = b.desc.tol;
  a.max_iters = b.desc.max_iters;
  a.fp32 = b.desc.precision == MHX_BATCH_FP32_REFINED;
  a.inner_tol = b.desc.inner_tol;
  a.max_refine = b.desc.max_refine;
  return a;
}

static void enqueue(Batch& b, int wg) {
  SgArgs a = make_args(b);
  hipLaunchKernelGGL(k_sg_reset, dim3(1), dim3(1), 0, b.stream, b.queue.p);
  auto go = [&](auto BX) {
    constexpr bool X = decltype(BX)::value;
    if (wg == 1024) {
      if (a.fp32) hipLaunchKernelGGL((k_subgrid<1024, true, X>), dim3(b.grid[1]), dim3(1024), 0, b.stream, a);
      else hipLaunchKernelGGL((k_subgrid<1024, false, X>), dim3(b.grid[1]), dim3(1024), 0, b.stream, a);
    } else {
      if (a.fp32) hipLaunchKernelGGL((k_subgrid<512, true, X>), dim3(b.grid[0]), dim3(512), 0, b.stream, a);
      else hipLaunchKernelGGL((k_subgrid<512, false, X>), dim3(b.grid[0]), dim3(512), 0, b.stream, a);
    }
  };
  if (b.box) go(std::true_type{});
  else go(std::false_type{});
  MHX_HIP(hipGetLastError());
}

// Ordinary host memory, which the runtime would copy through a staging buffer:
// pinned and managed memory takes a transfer straight from the device (14.4 MB
// into pinned memory 0.26 ms, through the ring 0.48).
static bool ordinary_memory(const void* p) {
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, p) != hipSuccess) {
    (void)hipGetLastError();  // memory that the runtime does not know
    return true;
  }
  return at.type == hipMemoryTypeUnregistered;
}

// device array -> host array, complete on return
static void copy_to_host(Batch& b, void* dst, const void* src, size_t bytes) {
  int dev = -1;
  MHX_HIP(hipGetDevice(&dev));
  std::shared_ptr<CopyRing> ring;
  if (bytes >= CopyRing::kMinBytes && dev == b.dev && ordinary_memory(dst)) {
    try {
      ring = copy_ring(dev);
    } catch (...) {  // no pinned memory to be had: the runtime's path
      (void)hipGetLastError();
    }
  }
  if (ring) {
    std::unique_lock<std::mutex> lk(ring->busy, std::try_to_lock);
    if (lk.owns_lock()) {
      const size_t chunk = std::min(CopyRing::kChunk, (bytes + CopyRing::kWorkers - 1) / CopyRing::kWorkers);
      hipError_t err[CopyRing::kWorkers] = {};
      std::thread th[CopyRing::kWorkers];
      auto run = [&](int w, bool own_thread) {
        err[w] = ring->work(w, b.stream, (char*)dst, (const char*)src, bytes, chunk, own_thread);
      };
      int started = 1;
      try {
        for (; started < CopyRing::kWorkers; ++started) th[started] = std::thread(run, started, true);
      } catch (const std::exception&) {
        // no thread to be had: the remaining workers' chunks follow here
      }
      run(0, false);
      for (int w = started; w < CopyRing::kWorkers; ++w) run(w, false);
      for (int w = 1; w < started; ++w) th[w].join();
      for (hipError_t e : err) {
        // (no transfer of this call into buffers that the next caller gets)
        if (e != hipSuccess) (void)hipStreamSynchronize(b.stream);
        MHX_HIP(e);
      }
      return;
    }
  }
  MHX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, b.stream));
  MHX_HIP(hipStreamSynchronize(b.stream));
}

// a pair of timing events destroyed on every exit path, including the
// MHX_HIP throws between creation and the end of the timed region
struct EventPair {
  hipEvent_t a = nullptr, b = nullptr;
  EventPair() {
    MHX_HIP(hipEventCreate(&a));
    hipError_t e = hipEventCreate(&b);
    if (e != hipSuccess) {
      (void)hipEventDestroy(a);
      throw Error{MHX_ERR_DEVICE, std::string("hipEventCreate: ") + hipGetErrorString(e)};
    }
  }
  EventPair(const EventPair&) = delete;
  EventPair& operator=(const EventPair&) = delete;
  ~EventPair() {
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
  }
  float elapsed_ms() const {
    float ms = 0.f;
    MHX_HIP(hipEventElapsedTime(&ms, a, b));
    return ms;
  }
};

static double timed_run(Batch& b, int wg) {
  EventPair ev;
  MHX_HIP(hipEventRecord(ev.a, b.stream));
  enqueue(b, wg);
  MHX_HIP(hipEventRecord(ev.b, b.stream));
  MHX_HIP(hipEventSynchronize(ev.b));
  return ev.elapsed_ms();
}

static void setup_grid(Batch& b) {
  int dev = 0, cus = 0;
  MHX_HIP(hipGetDevice(&dev));
  MHX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  int occ512 = 0, occ1024 = 0;
  auto occ = [&](auto MX, auto BX) {
    constexpr bool M = decltype(MX)::value, X = decltype(BX)::value;
    MHX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ512, (const void*)k_subgrid<512, M, X>, 512, 0));
    MHX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ1024, (const void*)k_subgrid<1024, M, X>, 1024, 0));
  };
  const bool mixed = b.desc.precision == MHX_BATCH_FP32_REFINED;
  if (mixed && b.box) occ(std::true_type{}, std::true_type{});
  else if (mixed) occ(std::true_type{}, std::false_type{});
  else if (b.box) occ(std::false_type{}, std::true_type{});
  else occ(std::false_type{}, std::false_type{});
  MHX_REQUIRE(occ512 > 0 && occ1024 > 0, MHX_ERR_DEVICE, "subgrid kernel does not fit on a CU");
  b.grid[0] = std::max(1, std::min(b.n_inst, cus * occ512));
  b.grid[1] = std::max(1, std::min(b.n_inst, cus * occ1024));
}

}  // namespace mhx

using namespace mhx;

struct mhx_batch : public Batch {};

extern "C" {

int mhx_batch_create(const mhx_batch_desc* d, mhx_batch** out) {
  mhx_batch* b = nullptr;
  try {
    MHX_REQUIRE(d && out && d->n_inst > 0 && d->n_axis && d->k && d->g, MHX_ERR_ARG, "bad batch description");
    *out = nullptr;
    b = new mhx_batch();
    MHX_HIP(hipGetDevice(&b->dev));
    b->desc = *d;
    if (b->desc.tol <= 0) b->desc.tol = 1e-10;
    if (b->desc.max_iters <= 0) b->desc.max_iters = 10000;
    if (b->desc.inner_tol <= 0) b->desc.inner_tol = 1e-5;
    if (b->desc.max_refine <= 0) b->desc.max_refine = 20;
    MHX_REQUIRE(b->desc.precision == MHX_BATCH_FP64 || b->desc.precision == MHX_BATCH_FP32_REFINED, MHX_ERR_ARG,
                "unknown batch precision");
    b->n_inst = d->n_inst;
    b->box = d->extent != nullptr || d->src != nullptr;
    b->h_inst.resize(b->n_inst);
    long ko = 0, xo = 0;
    for (int i = 0; i < b->n_inst; ++i) {
      const int n = d->n_axis[i];
      MHX_REQUIRE(n >= 2 && n <= kSgMaxN, MHX_ERR_UNSUPPORTED, "subgrid instances need 2..16 elements per axis");
      double L[3] = {1.0, 1.0, 1.0};
      if (d->extent)
        for (int c = 0; c < 3; ++c) {
          L[c] = d->extent[3 * (long)i + c];
          MHX_REQUIRE(std::isfinite(L[c]) && L[c] > 0.0, MHX_ERR_ARG, "subgrid box extents must be positive");
        }
      SgInst& si = b->h_inst[i];
      si = SgInst{};
      si.n = n, si.k_off = (int)ko, si.x_off = (int)xo;
      const double hx = L[0] / n, hy = L[1] / n, hz = L[2] / n;
      box_stencil(hx, hy, hz, si.kv);
      si.vol8 = hx * hy * hz / 8.0;
      ko += (long)n * n * n;
      xo += (long)(n + 1) * (n + 1) * (n + 1);
    }
    MHX_REQUIRE(xo < (1L << 31), MHX_ERR_UNSUPPORTED, "batch too large");
    b->total_elems = ko;
    b->total_nodes = xo;
    b->h_order.resize(b->n_inst);
    for (int i = 0; i < b->n_inst; ++i) b->h_order[i] = i;
    std::stable_sort(b->h_order.begin(), b->h_order.end(),
                     [&](int p, int q) { return b->h_inst[p].n > b->h_inst[q].n; });
    MHX_HIP(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
    b->inst.alloc(b->n_inst);
    b->order.alloc(b->n_inst);
    b->iters.alloc(b->n_inst);
    b->refs.alloc(b->n_inst);
    b->relres.alloc(b->n_inst);
    b->k.alloc(ko);
    if (d->src) b->src.alloc(ko);
    b->g.alloc(xo);
    b->x.alloc(xo);
    b->queue.alloc(1);
    MHX_HIP(hipMemcpyAsync(b->inst.p, b->h_inst.data(), b->n_inst * sizeof(SgInst), hipMemcpyHostToDevice, b->stream));
    MHX_HIP(hipMemcpyAsync(b->order.p, b->h_order.data(), b->n_inst * sizeof(int), hipMemcpyHostToDevice, b->stream));
    MHX_HIP(hipMemcpyAsync(b->k.p, d->k, ko * sizeof(double), hipMemcpyHostToDevice, b->stream));
    if (d->src) MHX_HIP(hipMemcpyAsync(b->src.p, d->src, ko * sizeof(double), hipMemcpyHostToDevice, b->stream));
    MHX_HIP(hipMemcpyAsync(b->g.p, d->g, xo * sizeof(double), hipMemcpyHostToDevice, b->stream));
    MHX_HIP(hipStreamSynchronize(b->stream));
    setup_grid(*b);
    b->wg = d->wg_size == 512 || d->wg_size == 1024 ? d->wg_size : 0;
    if (!b->wg) {
      // autotuner: time each workgroup shape on this batch (after one warm-up) and keep the fastest
      double best = 1e300;
      for (int wg : {512, 1024}) {
        (void)timed_run(*b, wg);
        const double t = timed_run(*b, wg);
        if (t < best) {
          best = t;
          b->wg = wg;
        }
      }
    }
    *out = b;
    return MHX_OK;
  } catch (const Error& e) {
    delete b;
    return e.code;
  }
}

void mhx_batch_destroy(mhx_batch* b) {
  if (!b) return;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  delete b;
}

int mhx_batch_solve(mhx_batch* b, int32_t flags) {
  (void)flags;
  try {
    if (!b) return MHX_ERR_ARG;
    EventPair ev;
    if (b->desc.use_graph) {
      if (!b->exec || b->graph_wg != b->wg) {
        if (b->exec) (void)hipGraphExecDestroy(b->exec);
        if (b->graph) (void)hipGraphDestroy(b->graph);
        b->exec = nullptr;
        b->graph = nullptr;
        MHX_HIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        enqueue(*b, b->wg);
        MHX_HIP(hipStreamEndCapture(b->stream, &b->graph));
        MHX_HIP(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
        b->graph_wg = b->wg;
      }
      MHX_HIP(hipEventRecord(ev.a, b->stream));
      MHX_HIP(hipGraphLaunch(b->exec, b->stream));
    } else {
      MHX_HIP(hipEventRecord(ev.a, b->stream));
      enqueue(*b, b->wg);
    }
    MHX_HIP(hipEventRecord(ev.b, b->stream));
    MHX_HIP(hipEventSynchronize(ev.b));
    b->last_ms = ev.elapsed_ms();
    return MHX_OK;
  } catch (const Error& e) {
    if (b) b->err = e.msg;
    return e.code;
  }
}

int mhx_batch_results(mhx_batch* b, double* x, int32_t* iters, double* relres, int32_t* refinements) {
  try {
    if (!b) return MHX_ERR_ARG;
    if (x) copy_to_host(*b, x, b->x.p, b->total_nodes * sizeof(double));
    if (iters) MHX_HIP(hipMemcpyAsync(iters, b->iters.p, b->n_inst * sizeof(int), hipMemcpyDeviceToHost, b->stream));
    if (relres) MHX_HIP(hipMemcpyAsync(relres, b->relres.p, b->n_inst * sizeof(double), hipMemcpyDeviceToHost, b->stream));
    if (refinements)
      MHX_HIP(hipMemcpyAsync(refinements, b->refs.p, b->n_inst * sizeof(int), hipMemcpyDeviceToHost, b->stream));
    MHX_HIP(hipStreamSynchronize(b->stream));
    return MHX_OK;
  } catch (const Error& e) {
    b->err = e.msg;
    return e.code;
  }
}

int64_t mhx_release_host_buffers(void) {
  try {
    std::map<int, std::shared_ptr<CopyRing>> drop;  // freed outside the lock
    {
      CopyRings& all = copy_rings();
      std::lock_guard<std::mutex> lk(all.mu);
      drop.swap(all.of);
    }
    return (int64_t)(drop.size() * CopyRing::kWorkers * CopyRing::kChunk);
  } catch (const std::exception&) {
    return MHX_ERR_STATE;
  }
}

int mhx_batch_info(const mhx_batch* b, int64_t* total_nodes, int32_t* wg_size, double* last_ms) {
  if (!b) return MHX_ERR_ARG;
  if (total_nodes) *total_nodes = b->total_nodes;
  if (wg_size) *wg_size = b->wg;
  if (last_ms) *last_ms = b->last_ms;
  return MHX_OK;
}

int mhx_batch_set_wg(mhx_batch* b, int32_t wg) {
  if (!b || (wg != 512 && wg != 1024)) return MHX_ERR_ARG;
  b->wg = wg;
  return MHX_OK;
}

}  // extern "C"
