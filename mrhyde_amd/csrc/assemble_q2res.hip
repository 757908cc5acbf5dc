// assemble_q2res.hip — nonlinear thermal residual (no Jacobian) of Q2 hexahedra
// with 3x3x3 Gauss points on axis-aligned box elements, CDNA4 (gfx950).
//
// Same reference steps and mesh class as assemble_q2box.hip, for calls that
// want the residual alone (line searches and convergence checks of Newton's
// method), with an element source but no sine modes.
//
// What bounds it: latency.  About 1,400 operations an element (1.6 times that
// with the elements evaluated twice) take 20 of the 64 us of a 64^3 mesh; two
// thirds of the wavefronts' cycles wait, at two wavefronts per SIMD, for loads
// and for the 50 registers that spill.  So there are no barriers and a lane
// evaluates one element in registers by sum factorisation; a wavefront covers
// 8 x 8 elements in x and y and walks z.  Node
// rows 2e and 2e + 1 of block e sum the elements e - 1 and e: the z neighbour's
// share comes from the layer before (through LDS, 27 doubles a lane, to keep
// the registers at two wavefronts per SIMD), the y neighbour's by a lane
// permute, the x neighbour's by a DPP move.  The first lane in x and y and the
// first layer of a walk only feed the others (7 x 7 of 64 lanes own rows), and
// every row is written once.
// 64^3: 162 us in the row-owned Jacobian kernel's residual form (four barriers a
// layer, 27 of 32 lanes), here 64 us.
//
// The operations and their order are those of k_q2box, so both give the same
// residual to the bit: forward y, z, x, backward z, y, x, the two elements of a
// row summed apart.  (Products with the centre point's shape values 0 and 1 are
// left out.)

#include <algorithm>
#include <cmath>

#include "lattice.hpp"
#include "lattice_product.hpp"
#include "mhx_internal.hpp"
#include "thermal.hpp"

// every operation rounds as it is written (see the head comment)
#pragma clang fp contract(off)

namespace mhx {

namespace {

constexpr const Tab1& kT = T1<2, 3>::v;

static_assert(kT.B[0][1] == 0.0 && kT.B[1][1] == 1.0 && kT.B[2][1] == 0.0 && kT.D[1][1] == 0.0,
              "the centre point is a node");
static_assert(kT.B[0][0] == kT.B[2][2] && kT.B[1][0] == kT.B[1][2] && kT.B[2][0] == kT.B[0][2] &&
                  kT.D[0][0] == -kT.D[2][2] && kT.D[1][0] == -kT.D[1][2] && kT.D[2][0] == -kT.D[0][2],
              "the outer points mirror each other");

// weight W of axis point Q times that of P times that of T (a copy with internal
// linkage: the table's own entries would be loaded at run time)
struct Weights {
  double w[3][3][3];
};
constexpr Weights weights() {
  Weights r{};
  for (int q = 0; q < 3; ++q)
    for (int p = 0; p < 3; ++p)
      for (int t = 0; t < 3; ++t) r.w[q][p][t] = kT.W[q] * kT.W[p] * kT.W[t];
  return r;
}
constexpr Weights kW = weights();

// B[I][0] and D[I][0] in scalar registers (the compiler would keep every table
// constant in a vector register through the loop, and spill)
struct Outer {
  double b[3], d[3];
};

// s + c x with c = D[I][Q] (DER) or B[I][Q]; FIRST: the term starts the chain
template <bool DER, int I, int Q, bool FIRST = false>
__device__ __forceinline__ double term(const Outer& o, double x, double s = 0.0) {
  constexpr double k = DER ? kT.D[I][Q] : kT.B[I][Q];
  const double c = Q == 1 ? k : DER ? (Q == 0 ? o.d[I] : -o.d[2 - I]) : (Q == 0 ? o.b[I] : o.b[2 - I]);
  if constexpr (k == 0.0) return s;
  else if constexpr (FIRST) return c * x;
  else if constexpr (k == 1.0) return s + x;
  else return fma(c, x, s);
}
// node values to the points
template <bool DER, int Q>
__device__ __forceinline__ double point(const Outer& t, double u0, double u1, double u2) {
  if constexpr (!DER && Q == 1) return u1;
  else return term<DER, 2, Q>(t, u2, term<DER, 1, Q>(t, u1, term<DER, 0, Q, true>(t, u0)));
}
template <bool DER>
__device__ __forceinline__ void fwd(const Outer& t, double u0, double u1, double u2, double (&o)[3]) {
  o[0] = point<DER, 0>(t, u0, u1, u2);
  o[1] = point<DER, 1>(t, u0, u1, u2);
  o[2] = point<DER, 2>(t, u0, u1, u2);
}
// point values f to the nodes by values
__device__ __forceinline__ void bwd(const Outer& t, const double (&f)[3], double (&r)[3]) {
  r[0] = term<false, 0, 2>(t, f[2], term<false, 0, 0, true>(t, f[0]));
  r[1] = term<false, 1, 2>(t, f[2], term<false, 1, 1>(t, f[1], term<false, 1, 0, true>(t, f[0])));
  r[2] = term<false, 2, 2>(t, f[2], term<false, 2, 0, true>(t, f[0]));
}
// g by slopes and f by values, point by point: slopes first (DF) or values
template <bool DF, int I>
__device__ __forceinline__ double node2(const Outer& t, const double (&g)[3], const double (&f)[3]) {
  const double s0 = DF ? term<false, I, 0>(t, f[0], term<true, I, 0, true>(t, g[0]))
                       : term<true, I, 0>(t, g[0], term<false, I, 0, true>(t, f[0]));
  const double s1 = DF ? term<false, I, 1>(t, f[1], term<true, I, 1>(t, g[1], s0))
                       : term<true, I, 1>(t, g[1], term<false, I, 1>(t, f[1], s0));
  return DF ? term<false, I, 2>(t, f[2], term<true, I, 2>(t, g[2], s1)) : term<true, I, 2>(t, g[2], term<false, I, 2>(t, f[2], s1));
}
template <bool DF>
__device__ __forceinline__ void bwd2(const Outer& t, const double (&g)[3], const double (&f)[3], double (&r)[3]) {
  r[0] = node2<DF, 0>(t, g, f);
  r[1] = node2<DF, 1>(t, g, f);
  r[2] = node2<DF, 2>(t, g, f);
}

constexpr int kDppShr1 = 0x111;  // row_shr 1: from the lane before

}  // namespace

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_q2res(AsmArgs args, int tx, int ty) {
  const double* __restrict__ u = args.u;
  const double* __restrict__ vx = args.vx;
  const uint8_t* __restrict__ fixed = args.fixed;
  const double* __restrict__ ck0 = args.coef.k0;
  const double* __restrict__ csrc = args.coef.src;
  double* __restrict__ res = args.res;
  const double a2 = args.coef.diff_u2;
  const bool add = args.first_touch == 0;
  const int n0 = args.m.nel[0], n1 = args.m.nel[1], n2 = args.m.nel[2];
  const int N0 = 2 * n0 + 1, N1 = 2 * n1 + 1, N2 = 2 * n2 + 1;
  const int nvx0 = args.m.nvx[0], nvx1 = args.m.nvx[1];
  const int lane = threadIdx.x, lx = lane & 7, ly = lane >> 3;
  int b = blockIdx.x;
  const int bx = b % tx;
  b /= tx;
  const int by = b % ty, bz = b / ty;
  const int ex = 7 * bx + lx - 1, ey = 7 * by + ly - 1;  // element and block of the lane
  const int z0 = bz * args.gpb, z1 = min(z0 + args.gpb, n2 + 1);
  const bool act = ex >= 0 && ex < n0 && ey >= 0 && ey < n1;
  const int cx = act ? ex : 0, cy = act ? ey : 0;
  const double Jx = 0.5 * (vx[3 * (cx + 1)] - vx[3 * cx]);
  const double Jy = 0.5 * (vx[3 * ((long)nvx0 * (cy + 1)) + 1] - vx[3 * ((long)nvx0 * cy) + 1]);
  const double iJx2 = 1.0 / (Jx * Jx), iJy2 = 1.0 / (Jy * Jy);
  const bool own = lx > 0 && ly > 0 && ex <= n0 && ey <= n1;
  const long node0 = 2 * cx + (long)N0 * (2 * cy);
  const long plane = (long)N0 * N1;
  // the layer before: its share of node plane 2z, [field][q2][q1]
  __shared__ double s_carry[27][64];
#pragma unroll
  for (int k = 0; k < 27; ++k) s_carry[k][lane] = 0.0;
  for (int z = max(z0 - 1, 0); z < z1; ++z) {
    const bool on = act && z < n2;
    Outer tb{{kT.B[0][0], kT.B[1][0], kT.B[2][0]}, {kT.D[0][0], kT.D[1][0], kT.D[2][0]}};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      asm volatile("" : "+s"(tb.b[i]));
      asm volatile("" : "+s"(tb.d[i]));
    }
    int cl = lane;  // (opaque, or the compiler keeps the carry in registers)
    asm volatile("" : "+v"(cl));
    const int cz = z < n2 ? z : 0;
    const double Jz = 0.5 * (vx[3 * ((long)nvx0 * nvx1 * (cz + 1)) + 2] - vx[3 * ((long)nvx0 * nvx1 * cz) + 2]);
    const double iJz2 = 1.0 / (Jz * Jz);
    double un[3][3][3], k0 = 1.0, f = 0.0;  // nodes [z][y][x]; 0 off the mesh
#pragma unroll
    for (int k = 0; k < 27; ++k) (&un[0][0][0])[k] = 0.0;
    if (on) {
      const long el = ex + (long)n0 * (ey + (long)n1 * z);
      const double* up = u + node0 + plane * (2 * z);
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
          for (int i = 0; i < 3; ++i) un[k][j][i] = up[plane * k + N0 * j + i];
      if (ck0) k0 = ck0[el];
      if (csrc) f = csrc[el];
    }
    // y contraction: value and slope at the three q2 of every node line
    double v[3][3][3], s[3][3][3];  // [q2][x][z]
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        double o[3], d[3];
        fwd<false>(tb, un[k][0][i], un[k][1][i], un[k][2][i], o);
        fwd<true>(tb, un[k][0][i], un[k][1][i], un[k][2][i], d);
#pragma unroll
        for (int p = 0; p < 3; ++p) v[p][i][k] = o[p], s[p][i][k] = d[p];
      }
    const double aj = fabs(Jy * Jz) * fabs(Jx), wk = on ? aj * k0 : 0.0, wf = on ? aj * f : 0.0;
    double P[2][3][3][3];  // rows 2z and 2z + 1: [plane][field x, y, value][q1][q2]
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      // z and x contractions and the weighted fluxes at the nine points of q2 = p
      double a[3][3], ay[3][3], az[3][3];  // [x, then q1][q3]
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        fwd<false>(tb, v[p][i][0], v[p][i][1], v[p][i][2], a[i]);
        fwd<true>(tb, v[p][i][0], v[p][i][1], v[p][i][2], az[i]);
        fwd<false>(tb, s[p][i][0], s[p][i][1], s[p][i][2], ay[i]);
      }
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        double U[3], Gx[3], Gy[3], Gz[3];
        fwd<false>(tb, a[0][t], a[1][t], a[2][t], U);
        fwd<true>(tb, a[0][t], a[1][t], a[2][t], Gx);
        fwd<false>(tb, ay[0][t], ay[1][t], ay[2][t], Gy);
        fwd<false>(tb, az[0][t], az[1][t], az[2][t], Gz);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          // k = k0 (1 + a u^2) (ThermalPhysics in thermal.hpp)
          const double kap = kW.w[q][p][t] * wk * fma(a2 * U[q], U[q], 1.0);
          a[q][t] = kap * (Gx[q] * iJx2);
          ay[q][t] = kap * (Gy[q] * iJy2);
          az[q][t] = kap * (Gz[q] * iJz2);
        }
      }
      // back along z: planes 2z, 2z + 1 and, for the next layer, 2z + 2
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        double rx[3], ry[3], rv[3];
        bwd(tb, a[q], rx);
        bwd(tb, ay[q], ry);
        const double fs[3] = {-(kW.w[q][p][0] * wf), -(kW.w[q][p][1] * wf),
                              -(kW.w[q][p][2] * wf)};
        bwd2<true>(tb, az[q], fs, rv);
        double* c = &s_carry[3 * (3 * q + p)][cl];
        P[0][0][q][p] = c[0] + rx[0];
        P[0][1][q][p] = c[64] + ry[0];
        P[0][2][q][p] = c[128] + rv[0];
        P[1][0][q][p] = rx[1];
        P[1][1][q][p] = ry[1];
        P[1][2][q][p] = rv[1];
        c[0] = rx[2];
        c[64] = ry[2];
        c[128] = rv[2];
      }
      __builtin_amdgcn_sched_barrier(0);  // (one q2 at a time: registers)
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // back along y: rows 2 ey + j
      double cxq[2][3], c0q[2][3];  // [j][q1]
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        double rx[3], rv[3];
        bwd(tb, P[k][0][q], rx);
        bwd2<true>(tb, P[k][1][q], P[k][2][q], rv);
        cxq[0][q] = rx[0] + __shfl_up(rx[2], 8);
        c0q[0][q] = rv[0] + __shfl_up(rv[2], 8);
        cxq[1][q] = rx[1];
        c0q[1][q] = rv[1];
      }
      // and along x
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        double r[3];
        bwd2<false>(tb, cxq[j], c0q[j], r);
        r[0] += dpp_move<kDppShr1>(r[2]);
        const int Y = 2 * ey + j, Z = 2 * z + k;
        if (z >= z0 && own && Y < N1 && Z < N2) {
          const long row = 2 * ex + (long)N0 * (Y + (long)N1 * Z);
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            if (2 * ex + i >= N0) continue;
            const bool fx = fixed[row + i] != 0;
            if (add) {
              if (!fx) res[row + i] -= r[i];
            } else {
              res[row + i] = fx ? 0.0 : -r[i];
            }
          }
        }
      }
    }
  }
}

void launch_q2res(Ctx& c, AsmArgs& a) {
  const int tx = (c.mesh.nel[0] + 7) / 7, ty = (c.mesh.nel[1] + 7) / 7, nb = c.mesh.nel[2] + 1;
  // Layers per walk.  A walk repeats the layer before it; the device runs 2,048
  // wavefronts at a time, and where they are 1,024 or fewer a layer takes about
  // three quarters as long.  us by layers: 96^3 3 162, 4 157, 5 148, 7 161, 10
  // 141, 13 166; 64^3 2 68, 3 71, 4 64, 5 70, 7 74, 10 85; 48^3 2 36, 3 36, 5 44;
  // 16^3 2 18, 4 29.
  int best = 1;
  double cost = 1e300;
  for (int s : {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 16, 24, 32, 48}) {
    const long waves = (long)tx * ty * ((nb + s - 1) / s);
    const double t = (waves <= 1024 ? 0.75 : (double)((waves + 2047) / 2048)) * (std::min(s, nb) + 1);
    if (t < cost) best = s, cost = t;
    if (s >= nb) break;
  }
  a.gpb = best;
  ScopedPhase ph(c.prof, "k_q2res", c.stream);
  hipLaunchKernelGGL(k_q2res, dim3((unsigned)(tx * ty * ((nb + best - 1) / best))), dim3(64), 0, c.stream, a, tx, ty);
  MHX_HIP(hipGetLastError());
}

}  // namespace mhx
