// amg.hip — smoothed-aggregation algebraic multigrid on the node lattice
// (CDNA4, gfx950): hierarchy set-up on the device and the V-cycle used as a
// Krylov preconditioner.
//
// Replaces LinearAlgebraInterface::buildAMGPreconditioner
// (linearAlgebraInterface_solvers.hpp:201-253), which hands the Jacobian to
// MueLu::CreateTpetraPreconditioner with "multigrid algorithm" sa,
// "aggregation: type" uncoupled (drop scheme classical, nothing dropped),
// "smoother: type" CHEBYSHEV of degree 2 with eigenvalue ratio 7 and a zero
// starting solution, "coarse: max size" 500, no repartitioning, no reuse.
// MueLu (Trilinos) is not in the reference tree.  What is kept is the
// published smoothed-aggregation method (Vanek, Mandel, Brezina, Computing
// 56 (1996)) with MueLu's defaults for what the reference leaves unset:
//   - tentative prolongator T: the near-null space (one constant vector per
//     field, zero on strong-Dirichlet rows) restricted to each aggregate and
//     orthonormalised, which for one column per field is a normalisation;
//     the coarse near-null space is the column norm;
//   - P = (I - omega D^-1 A) T with omega = (4/3) / lambda, lambda the
//     10-step power-iteration estimate of rho(D^-1 A);
//   - R = P^T and A_c = R A P;
//   - Chebyshev smoothing on D^-1 A over [lmax / 7, lmax], lmax = 1.1 lambda,
//     before and after the coarse correction; V-cycle; the coarsest level
//     (at most 500 rows, or after 10 levels) is solved with its dense inverse.
// The aggregation differs from MueLu's greedy one in form, not in kind: on a
// lattice, uncoupled aggregation builds each aggregate from a root and its
// graph neighbours, i.e. (2r+1)^d node blocks for a stencil of reach r.  Here
// the aggregates ARE those lattice blocks (the last block along an axis takes
// the remainder), so every pattern of the hierarchy is a separable box known
// in closed form, and the Galerkin products need no hashing or sorting: each
// row accumulates into a fixed slot box in LDS, in a fixed order, so the
// hierarchy is bit-reproducible.
#include <algorithm>
#include <climits>
#include <cmath>
#include <memory>
#include <type_traits>

#include "lattice.hpp"
#include "lattice_product.hpp"
#include "mhx_internal.hpp"

namespace mhx {

constexpr int kAmgMaxLevels = 10;      // MueLu "max levels"
// MueLu's "coarse: max size" is 500 with a sparse direct coarse solver; the
// coarsest solve here is a dense inverse built by one workgroup in O(n^3), so
// the hierarchy coarsens on until at most 128 rows remain (one level more at
// most, since a lattice level shrinks 27x or more per step in 3-D)
constexpr long kAmgCoarseMax = 128;
constexpr long kAmgDenseMax = 512;     // Gauss-Jordan kernel limit (2n columns <= 1024 threads)
constexpr int kAmgPowerIters = 10;     // "sa: eigenvalue estimate num iterations"
constexpr double kAmgDamping = 4.0 / 3.0;
constexpr double kChebRatio = 7.0;     // "chebyshev: ratio eigenvalue"
constexpr double kChebBoost = 1.1;     // Ifpack2 Chebyshev boost of the estimate
constexpr int kAmgMaxFields = 4;
// smoothers: Chebyshev(2) on D^-1 A (the reference's MueLu setting), or
// damped sweeps of nodal block Jacobi (the nf x nf block of each node
// inverted), for coupled multi-field systems whose point diagonal does not
// bound the spectrum (stabilised Navier-Stokes).  On the developed 48^3 and
// 64^3 cavity flows damping above 0.5 makes the cycle diverge; three sweeps
// at 0.4 is the default.
constexpr int kSmootherChebyshev = 0, kSmootherBlockJacobi = 1, kSmootherBlockGaussSeidel = 2;
constexpr double kBjOmega = 0.4;  // defaults; options amg.sweeps and amg.omega_pct
constexpr int kBjSweeps = 3;
constexpr int kAmgBlk = 128;           // threads per workgroup of the set-up kernels

// ---------------------------------------------------------------------------
// lattice axis tables of one level.  Node p of an axis of n nodes lies in
// aggregate agg(p) = min(p / b, na - 1), b = 2r + 1, na = max(1, n / b).  The
// prolongator row of p spans aggregates plo(p) .. plo(p) + pext(p) - 1 (at most
// 2), the row of A P spans aplo(p) .. + apext(p) - 1 (at most 3), the
// restriction row of aggregate I spans fine nodes rlo(I) .. + rext(I) - 1, and
// the coarse operator row of I spans clo(I) .. + cext(I) - 1 (reach rc).  The
// s* arrays are prefix sums of the extents (closed-form row pointers).
// ---------------------------------------------------------------------------
enum AxisTable { kAgg, kPlo, kPext, kSp, kAplo, kApext, kRlo, kRext, kSr, kClo, kCext, kSc, kNumTables };

struct AxisDev {
  const int32_t* t[kNumTables];
  int n, na, b;
};
struct Geo {
  AxisDev ax[3];
  int nf;
};

struct AxisHost {
  int n = 1, na = 1, b = 1;
  std::vector<int32_t> t[kNumTables];
};

static void make_axis(AxisHost& a, int n, int r, int rc) {
  a.n = n;
  a.b = 2 * r + 1;
  a.na = std::max(1, n / a.b);
  const int b = a.b, na = a.na;
  for (auto& v : a.t) v.clear();
  auto& agg = a.t[kAgg];
  agg.resize(n);
  for (int p = 0; p < n; ++p) agg[p] = std::min(p / b, na - 1);
  a.t[kPlo].resize(n); a.t[kPext].resize(n); a.t[kAplo].resize(n); a.t[kApext].resize(n);
  a.t[kSp].assign(n + 1, 0);
  for (int p = 0; p < n; ++p) {
    const int lo = agg[std::max(0, p - r)];
    a.t[kPlo][p] = lo;
    a.t[kPext][p] = std::min(lo + 1, na - 1) - lo + 1;
    const int alo = agg[std::max(0, p - 2 * r)];
    a.t[kAplo][p] = alo;
    a.t[kApext][p] = std::min(alo + 2, na - 1) - alo + 1;
    a.t[kSp][p + 1] = a.t[kSp][p] + a.t[kPext][p];
  }
  std::vector<int> rlo(na, INT_MAX), rhi(na, -1);
  for (int p = 0; p < n; ++p)
    for (int I = a.t[kPlo][p]; I < a.t[kPlo][p] + a.t[kPext][p]; ++I) {
      rlo[I] = std::min(rlo[I], p);
      rhi[I] = std::max(rhi[I], p);
    }
  a.t[kRlo].resize(na); a.t[kRext].resize(na); a.t[kClo].resize(na); a.t[kCext].resize(na);
  a.t[kSr].assign(na + 1, 0);
  a.t[kSc].assign(na + 1, 0);
  for (int I = 0; I < na; ++I) {
    if (rhi[I] < 0) throw Error{MHX_ERR_ARG, "AMG: aggregate outside every prolongator row"};
    a.t[kRlo][I] = rlo[I];
    a.t[kRext][I] = rhi[I] - rlo[I] + 1;
    a.t[kSr][I + 1] = a.t[kSr][I] + a.t[kRext][I];
    a.t[kClo][I] = std::max(0, I - rc);
    a.t[kCext][I] = std::min(na - 1, I + rc) - a.t[kClo][I] + 1;
    a.t[kSc][I + 1] = a.t[kSc][I] + a.t[kCext][I];
  }
}

// offset of the first entry of node (x,y,z) in a separable box pattern with
// per-axis extents E and prefix sums S over a lattice of N nodes, nrnc =
// (rows per node) x (columns per box cell)
__device__ __forceinline__ long box_node_base(const int32_t* Sx, const int32_t* Sy, const int32_t* Sz,
                                              const int32_t* Ey, const int32_t* Ez, int Nx, int Ny, int x, int y,
                                              int z, long nrnc) {
  const long Tx = Sx[Nx], Ty = Sy[Ny];
  return nrnc * ((long)Sz[z] * Ty * Tx + (long)Ez[z] * ((long)Sy[y] * Tx + (long)Ey[y] * Sx[x]));
}

// row pointers of a box pattern: lattice N (per-axis extents table e, prefix
// table s), nf rows per node, nf columns per box cell
__global__ void k_box_rowptr(Geo G, int coarse, int e, int s, long nrows, int32_t* __restrict__ rp) {
  const long row = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (row > nrows) return;
  const AxisDev* A = G.ax;
  const int N0 = coarse ? A[0].na : A[0].n, N1 = coarse ? A[1].na : A[1].n;
  const int nf = G.nf;
  if (row == nrows) {
    const int N2 = coarse ? A[2].na : A[2].n;
    rp[row] = (int32_t)((long)nf * nf * A[0].t[s][N0] * (long)A[1].t[s][N1] * (long)A[2].t[s][N2]);
    return;
  }
  const long node = row / nf;
  const int f = (int)(row - node * nf);
  const int x = (int)(node % N0);
  const long yz = node / N0;
  const int y = (int)(yz % N1), z = (int)(yz / N1);
  const long base = box_node_base(A[0].t[s], A[1].t[s], A[2].t[s], A[1].t[e], A[2].t[e], N0, N1, x, y, z, (long)nf * nf);
  rp[row] = (int32_t)(base + (long)f * A[0].t[e][x] * A[1].t[e][y] * A[2].t[e][z] * nf);
}

// lattice coordinates of a node; node numbers fit 32 bits (the CRS indices
// are int32), and 32-bit unsigned division is several times cheaper on the
// GPU than the 64-bit one
__device__ __forceinline__ void node_xyz(long node, int N0, int N1, int& x, int& y, int& z) {
  const unsigned nd = (unsigned)node, n0 = (unsigned)N0, n1 = (unsigned)N1;
  const unsigned yz = nd / n0;
  x = (int)(nd - yz * n0);
  const unsigned zz = yz / n1;
  y = (int)(yz - zz * n1);
  z = (int)zz;
}

// ---------------------------------------------------------------------------
// set-up kernels (FP64)
// ---------------------------------------------------------------------------
__global__ void k_amg_diag(long n, const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
                           const double* __restrict__ A, double* __restrict__ dinv) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int lo = rp[i], hi = rp[i + 1];
  const int end = hi;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (ci[mid] < i) lo = mid + 1;
    else hi = mid;
  }
  const double d = (lo < end && ci[lo] == i) ? A[lo] : 0.0;
  dinv[i] = d != 0.0 ? 1.0 / d : 0.0;
}

__global__ void k_amg_ns0(long n, const uint8_t* __restrict__ fixed, double* __restrict__ ns) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) ns[i] = fixed && fixed[i] ? 0.0 : 1.0;
}

// power-iteration start vector 0.5 + frac(i * 0.618...), rounded op by op
__global__ void k_amg_start(long n, double* __restrict__ v) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double x = __dmul_rn((double)i, 0.6180339887498949);
  v[i] = __dadd_rn(0.5, __dsub_rn(x, floor(x)));
}


// nrm[(I, f)] = || ns restricted to aggregate I, field f ||
__global__ void k_amg_nrm(Geo G, const double* __restrict__ ns, double* __restrict__ nrm, long ncrows) {
  const long cr = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (cr >= ncrows) return;
  const int nf = G.nf;
  const long I = cr / nf;
  const int f = (int)(cr - I * nf);
  int Ix, Iy, Iz;
  node_xyz(I, G.ax[0].na, G.ax[1].na, Ix, Iy, Iz);
  const int Ic[3] = {Ix, Iy, Iz};
  int lo[3], hi[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    lo[d] = Ic[d] * G.ax[d].b;
    hi[d] = Ic[d] == G.ax[d].na - 1 ? G.ax[d].n - 1 : lo[d] + G.ax[d].b - 1;
  }
  double s = 0.0;
  for (int z = lo[2]; z <= hi[2]; ++z)
    for (int y = lo[1]; y <= hi[1]; ++y)
      for (int x = lo[0]; x <= hi[0]; ++x) {
        const double v = ns[((long)x + (long)G.ax[0].n * ((long)y + (long)G.ax[1].n * z)) * nf + f];
        s = fma(v, v, s);
      }
  nrm[cr] = sqrt(s);
}

// Row of a level's operator in closed form: the box of its column nodes and,
// per axis, where the columns cross into the next aggregate.  Every pattern of
// the hierarchy is such a box (level 0: the context's lattice of order p;
// coarse levels: p = 1 and the reach rc), so the set-up kernels decode an
// entry's column from its position instead of dividing the column index and
// looking the axis tables up per entry.
struct LevelBox {
  int N[3], p, reach;
};
struct RowBox {
  int lo[3], ex, ey;
  float iw, iey, inf;  // reciprocals (exact for these small extents, see LatRow)
  int nf;
  // (x, y, z) and field of entry q
  __device__ __forceinline__ void at(int q, int* c, int& f) const {
    const int w = ex * nf;
    const int run = (int)(((float)q + 0.5f) * iw);
    const int r0 = q - run * w;
    const int iz = (int)(((float)run + 0.5f) * iey);
    const int dx = nf == 1 ? r0 : (int)(((float)r0 + 0.5f) * inf);
    c[0] = lo[0] + dx;
    c[1] = lo[1] + run - iz * ey;
    c[2] = lo[2] + iz;
    f = r0 - dx * nf;
  }
};
__device__ __forceinline__ RowBox row_box(const LevelBox& B, int nf, const int* c) {
  RowBox r;
  int ext[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    int hi;
    if (B.p == 1 || c[a] % B.p == 0) {
      r.lo[a] = max(c[a] - B.reach, 0);
      hi = min(c[a] + B.reach, B.N[a] - 1);
    } else {
      r.lo[a] = c[a] - c[a] % B.p;
      hi = r.lo[a] + B.p;
    }
    ext[a] = B.N[a] > 1 ? hi - r.lo[a] + 1 : 1;
    if (B.N[a] <= 1) r.lo[a] = 0;
  }
  r.ex = ext[0];
  r.ey = ext[1];
  r.nf = nf;
  r.iw = 1.0f / (float)(ext[0] * nf);
  r.iey = 1.0f / (float)ext[1];
  r.inf = 1.0f / (float)nf;
  return r;
}

// lanes that share one row of the set-up kernels: lane l takes the entries l,
// l + kApLanes, ... (coalesced reads of the CRS row) into a box of its own in
// LDS, and the group then sums the boxes slot by slot in lane order, so every
// set-up gives the same bits
constexpr int kApLanes = 8;

// P = (I - omega D^-1 A) T.  The row's box of at most 2x2x2 aggregates x nf
// fields collects sum_j A_ij ns_j; T's normalisation (1 / nrm per aggregate
// and field) is applied to the sums.  (One thread per row walked its CRS row
// alone, every lane in lines of its own: mean over the levels of 48^3 Q2 655
// us, now 271.)
__global__ __launch_bounds__(kAmgBlk) void k_amg_P(Geo G, LevelBox B, long n, const int32_t* __restrict__ rp,
                                                   const double* __restrict__ A, const double* __restrict__ dinv,
                                                   const double* __restrict__ ns, const double* __restrict__ nrm,
                                                   const double* __restrict__ lam, const int32_t* __restrict__ prp,
                                                   int32_t* __restrict__ pci, double* __restrict__ P) {
  constexpr int kSlots = 8 * kAmgMaxFields + 1;
  __shared__ double acc_s[kAmgBlk][kSlots];
  const int l = threadIdx.x % kApLanes;
  const long i = ((long)blockIdx.x * kAmgBlk + threadIdx.x) / kApLanes;
  const bool active = i < n;
  double* acc = acc_s[threadIdx.x];
  const int nf = G.nf;
  int c[3] = {0, 0, 0}, lo[3], e3[3];
  const int own_f = active ? (int)((unsigned)i % (unsigned)nf) : 0;
  if (active) node_xyz((long)((unsigned)i / (unsigned)nf), B.N[0], B.N[1], c[0], c[1], c[2]);
  int thr[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    lo[a] = G.ax[a].t[kPlo][c[a]];
    e3[a] = G.ax[a].t[kPext][c[a]];
    // first node of the second aggregate (the last one takes the remainder)
    thr[a] = lo[a] + 1 < G.ax[a].na ? (lo[a] + 1) * G.ax[a].b : INT_MAX;
  }
  for (int s = 0; s < 8 * nf; ++s) acc[s] = 0.0;
  if (active) {
    const RowBox R = row_box(B, nf, c);
    const int b = rp[i], e = rp[i + 1];
    for (int k = b + l; k < e; k += kApLanes) {
      int x[3], f;
      R.at(k - b, x, f);
      const long j = ((long)x[0] + (long)B.N[0] * (x[1] + (long)B.N[1] * x[2])) * nf + f;
      const int s = (x[0] >= thr[0]) + 2 * (x[1] >= thr[1]) + 4 * (x[2] >= thr[2]);
      double& r = acc[s * nf + f];
      r = fma(A[k], ns[j], r);
    }
  }
  __syncthreads();
  if (!active) return;
  const int g0 = threadIdx.x - l;
  const long base = prp[i];
  const double sc = -(kAmgDamping / *lam) * dinv[i];
  const int cnt = e3[0] * e3[1] * e3[2] * nf;
  const int own = (c[0] >= thr[0]) + 2 * (c[1] >= thr[1]) + 4 * (c[2] >= thr[2]);
  for (int s = l; s < cnt; s += kApLanes) {
    const int g = s % nf, cell = s / nf;
    const int dx = cell % e3[0], dy = (cell / e3[0]) % e3[1], dz = cell / (e3[0] * e3[1]);
    const int slot = dx + 2 * dy + 4 * dz;
    double v = 0.0;
    for (int q = 0; q < kApLanes; ++q) v += acc_s[g0 + q][slot * nf + g];
    const long J = (lo[0] + dx) + (long)G.ax[0].na * ((lo[1] + dy) + (long)G.ax[1].na * (lo[2] + dz));
    const double nv = nrm[J * nf + g];
    double t = sc * v;
    if (slot == own && g == own_f) t += ns[i];
    pci[base + s] = (int32_t)(J * nf + g);
    P[base + s] = nv > 0.0 ? t / nv : 0.0;
  }
}

// R = P^T: one workgroup per coarse row (I, f); its columns are the fine DOFs
// of nodes rlo(I) .. rlo(I)+rext(I)-1 per axis, every field
__global__ __launch_bounds__(kAmgBlk) void k_amg_R(Geo G, const int32_t* __restrict__ prp,
                                                   const double* __restrict__ P, const int32_t* __restrict__ rrp,
                                                   int32_t* __restrict__ rci, double* __restrict__ R) {
  const long cr = blockIdx.x;
  const int nf = G.nf;
  const long I = cr / nf;
  const int f = (int)(cr - I * nf);
  int Ix, Iy, Iz;
  node_xyz(I, G.ax[0].na, G.ax[1].na, Ix, Iy, Iz);
  const int rlx = G.ax[0].t[kRlo][Ix], rly = G.ax[1].t[kRlo][Iy], rlz = G.ax[2].t[kRlo][Iz];
  const int rex = G.ax[0].t[kRext][Ix], rey = G.ax[1].t[kRext][Iy];
  const long base = rrp[cr];
  const int cnt = rrp[cr + 1] - rrp[cr];
  for (int e = threadIdx.x; e < cnt; e += kAmgBlk) {
    const int g = e % nf, cell = e / nf;
    const int x = rlx + cell % rex, y = rly + (cell / rex) % rey, z = rlz + cell / (rex * rey);
    const long node = x + (long)G.ax[0].n * (y + (long)G.ax[1].n * z);
    const long i = node * nf + g;
    // position of (I, f) in P row i
    const int ox = Ix - G.ax[0].t[kPlo][x], oy = Iy - G.ax[1].t[kPlo][y], oz = Iz - G.ax[2].t[kPlo][z];
    const int pex = G.ax[0].t[kPext][x], pey = G.ax[1].t[kPext][y];
    rci[base + e] = (int32_t)i;
    R[base + e] = P[prp[i] + ((oz * pey + oy) * pex + ox) * nf + f];
  }
}

// AP(i, (J, g)) in a dense 3x3x3 aggregate box per (fine row i, coarse field
// g), a group of kApLanes lanes each (see k_amg_P).  A column's first aggregate
// is the row's first or the next one per axis.  (With two index divisions and
// seven table loads per entry: mean over the levels of 48^3 Q2 1,010 us, now
// 455.)
__global__ __launch_bounds__(kAmgBlk) void k_amg_AP(Geo G, LevelBox B, long n, const int32_t* __restrict__ rp,
                                                    const double* __restrict__ A, const int32_t* __restrict__ prp,
                                                    const double* __restrict__ P, double* __restrict__ AP) {
  __shared__ double acc_s[kAmgBlk][28];
  const int nf = G.nf;
  const int l = threadIdx.x % kApLanes;
  const long t = ((long)blockIdx.x * kAmgBlk + threadIdx.x) / kApLanes;
  const bool active = t < n * nf;
  double* acc = acc_s[threadIdx.x];
  for (int s = 0; s < 27; ++s) acc[s] = 0.0;
  const long i = active ? (long)((unsigned long)t / (unsigned)nf) : 0;
  const int g = active ? (int)(t - i * nf) : 0;
  if (active) {
    int c[3];
    node_xyz((long)((unsigned)i / (unsigned)nf), B.N[0], B.N[1], c[0], c[1], c[2]);
    int thr[3], last[3];  // columns whose first aggregate is the row's second one; first aggregate of the last
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int r = (G.ax[a].b - 1) / 2, alo = G.ax[a].t[kAplo][c[a]];
      thr[a] = alo + 1 < G.ax[a].na ? (alo + 1) * G.ax[a].b + r : INT_MAX;
      last[a] = G.ax[a].na - 1 - alo;  // 0, 1: a column there spans one aggregate
    }
    const RowBox R = row_box(B, nf, c);
    const int b = rp[i], e = rp[i + 1];
    for (int k = b + l; k < e; k += kApLanes) {
      int x[3], f;
      R.at(k - b, x, f);
      const long j = ((long)x[0] + (long)B.N[0] * (x[1] + (long)B.N[1] * x[2])) * nf + f;
      const double a = A[k];
      const double* Pj = P + prp[j] + g;
      const int sx = x[0] >= thr[0], sy = x[1] >= thr[1], sz = x[2] >= thr[2];
      const int ex = sx < last[0] ? 2 : 1, ey = sy < last[1] ? 2 : 1, ez = sz < last[2] ? 2 : 1;
      double* o = acc + sx + 3 * sy + 9 * sz;
      if (ex + ey + ez == 6) {
        double pv[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) pv[q] = Pj[q * nf];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          double& r = o[(q & 1) + 3 * ((q >> 1) & 1) + 9 * (q >> 2)];
          r = fma(a, pv[q], r);
        }
      } else {
        for (int dz = 0; dz < ez; ++dz)
          for (int dy = 0; dy < ey; ++dy)
            for (int dx = 0; dx < ex; ++dx) {
              double& r = o[dx + 3 * dy + 9 * dz];
              r = fma(a, Pj[((dz * ey + dy) * ex + dx) * nf], r);
            }
      }
    }
  }
  __syncthreads();
  if (!active) return;
  const int g0 = threadIdx.x - l;  // first lane of the group
  for (int s = l; s < 27; s += kApLanes) {
    double v = 0.0;
    for (int q = 0; q < kApLanes; ++q) v += acc_s[g0 + q][s];
    AP[t * 27 + s] = v;
  }
}

// A_c = R (A P): one workgroup per coarse row (I, f).  The R row is a box of
// fine nodes; groups of 32 lanes take its (y, z) lines in turn, lane s the slot s
// of the nodes' 27-slot AP boxes (a contiguous read per box, at least eight in
// flight), and add into the group's own copy of the coarse row in LDS; the
// copies are summed in group order.  Where a node's AP box starts relative to
// the coarse row's comes from three small tables.  (One thread per coarse entry
// walking every R entry left 27 of 125 threads active and one dependent load in
// flight: mean over the levels of 48^3 Q2 1,185 us; with the tables looked up
// per entry in global memory 724; the two levels of the 32^3 cavity 678 -> 217.)
constexpr int kAcGroups = 8;     // groups of 32 lanes
constexpr int kAcMaxCols = 500;  // 5^3 coarse nodes x 4 fields
constexpr int kAcMaxExt = 64;    // nodes of an R row along an axis
template <int NF>
__global__ __launch_bounds__(32 * kAcGroups) void k_amg_Ac(Geo G, const int32_t* __restrict__ rrp,
                                                           const double* __restrict__ R,
                                                           const double* __restrict__ AP,
                                                           const double* __restrict__ nrm,
                                                           const int32_t* __restrict__ arp,
                                                           int32_t* __restrict__ aci, double* __restrict__ Ac) {
  __shared__ double s_acc[kAcGroups][kAcMaxCols];
  __shared__ int s_alo[3][kAcMaxExt], s_aex[3][kAcMaxExt];
  const long cr = blockIdx.x;
  const long I = cr / NF;
  int Ic[3];
  node_xyz(I, G.ax[0].na, G.ax[1].na, Ic[0], Ic[1], Ic[2]);
  int cl[3], ce[3], rl[3], re[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    cl[a] = G.ax[a].t[kClo][Ic[a]];
    ce[a] = G.ax[a].t[kCext][Ic[a]];
    rl[a] = G.ax[a].t[kRlo][Ic[a]];
    re[a] = G.ax[a].t[kRext][Ic[a]];
    for (int t = threadIdx.x; t < re[a]; t += 32 * kAcGroups) {
      s_alo[a][t] = G.ax[a].t[kAplo][rl[a] + t] - cl[a];
      s_aex[a][t] = G.ax[a].t[kApext][rl[a] + t];
    }
  }
  const long base = arp[cr];
  const int cnt = arp[cr + 1] - arp[cr];
  const int grp = threadIdx.x / 32, s = threadIdx.x % 32;
  const int sx = s % 3, sy = (s / 3) % 3, sz = s / 9;  // s < 27
  double* acc = s_acc[grp];
  for (int k = s; k < cnt; k += 32) acc[k] = 0.0;
  __syncthreads();
  const double* Rr = R + rrp[cr];
  constexpr int UX = NF == 1 ? 8 : (NF == 2 ? 2 : 1);  // nodes of a line in flight
  for (int q = grp; q < re[1] * re[2]; q += kAcGroups) {
    const int ly = q % re[1], lz = q / re[1];
    const int jy = s_alo[1][ly] + sy, jz = s_alo[2][lz] + sz;
    // (the coarse box holds every aggregate that a row of R reaches)
    const bool line = s < 27 && sy < s_aex[1][ly] && sz < s_aex[2][lz] && jy >= 0 && jy < ce[1] && jz >= 0 &&
                      jz < ce[2];
    const int yz = (jz * ce[1] + jy) * ce[0];
    const long node0 = rl[0] + (long)G.ax[0].n * ((rl[1] + ly) + (long)G.ax[1].n * (rl[2] + lz));
    const double* Rl = Rr + (long)q * re[0] * NF;
    for (int x0 = 0; x0 < re[0]; x0 += UX) {
      double v[UX][NF][NF], rv[UX][NF];
      int at[UX];
#pragma unroll
      for (int u = 0; u < UX; ++u) {
        const int x = x0 + u;
        at[u] = -1;
        if (x < re[0]) {
          const int jx = s_alo[0][x] + sx;
          if (line && sx < s_aex[0][x] && jx >= 0 && jx < ce[0]) at[u] = (yz + jx) * NF;
#pragma unroll
          for (int f = 0; f < NF; ++f) rv[u][f] = Rl[x * NF + f];
        }
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int g = 0; g < NF; ++g)
            v[u][f][g] = at[u] >= 0 ? AP[(((node0 + x) * NF + f) * NF + g) * 27 + s] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < UX; ++u) {
        // (a node whose box starts one aggregate on has its coarse entries in
        // other lanes than the node before it: 181 -> 185 us at 48^3 Q2 with
        // the order enforced)
        wave_lds_sync();
        if (at[u] >= 0) {
#pragma unroll
          for (int g = 0; g < NF; ++g) {
            double t = acc[at[u] + g];
#pragma unroll
            for (int f = 0; f < NF; ++f) t = fma(rv[u][f], v[u][f][g], t);
            acc[at[u] + g] = t;
          }
        }
      }
    }
  }
  __syncthreads();
  const int nax = G.ax[0].na, nay = G.ax[1].na;
  for (int e = threadIdx.x; e < cnt; e += 32 * kAcGroups) {
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < kAcGroups; ++q) v += s_acc[q][e];
    const int g = e % NF, cell = e / NF;
    const int jx = cl[0] + cell % ce[0], jy = cl[1] + (cell / ce[0]) % ce[1], jz = cl[2] + cell / (ce[0] * ce[1]);
    const long col = (jx + (long)nax * (jy + (long)nay * jz)) * NF + g;
    aci[base + e] = (int32_t)col;
    // an aggregate whose near-null space vanished (all its nodes strong
    // Dirichlet) has an empty prolongator column: an identity row keeps A_c
    // invertible without coupling it to anything
    Ac[base + e] = (col == cr && nrm[cr] == 0.0) ? 1.0 : v;
  }
}

// dense [A | I] of the coarsest level from its CRS
__global__ void k_amg_dense(long n, const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
                            const double* __restrict__ A, double* __restrict__ M) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double* row = M + i * 2 * n;
  for (long j = 0; j < 2 * n; ++j) row[j] = (j - n == i) ? 1.0 : 0.0;
  for (int k = rp[i]; k < rp[i + 1]; ++k) row[ci[k]] += A[k];
}

// Gauss-Jordan with partial pivoting on [A | I] (n x 2n, row-major) in one
// workgroup; afterwards the right half holds A^-1.  F: n factors of scratch.
__global__ __launch_bounds__(1024) void k_amg_gauss_jordan(int n, double* __restrict__ M, double* __restrict__ F,
                                                           int* __restrict__ err) {
  __shared__ double sv[1024];
  __shared__ int si[1024];
  const int t = threadIdx.x, w = 2 * n;
  for (int col = 0; col < n; ++col) {
    double best = -1.0;
    int bi = col;
    for (int r = col + t; r < n; r += 1024) {
      const double v = fabs(M[(long)r * w + col]);
      if (v > best) {
        best = v;
        bi = r;
      }
    }
    sv[t] = best;
    si[t] = bi;
    __syncthreads();
    for (int s = 512; s > 0; s >>= 1) {
      if (t < s && (sv[t + s] > sv[t] || (sv[t + s] == sv[t] && si[t + s] < si[t]))) {
        sv[t] = sv[t + s];
        si[t] = si[t + s];
      }
      __syncthreads();
    }
    const int pr = si[0];
    const double pmax = sv[0];
    __syncthreads();
    if (!(pmax > 0.0)) {
      if (t == 0) atomicOr(err, 4);
      return;  // uniform across the workgroup
    }
    if (pr != col)
      for (int j = t; j < w; j += 1024) {
        const double a = M[(long)pr * w + j];
        M[(long)pr * w + j] = M[(long)col * w + j];
        M[(long)col * w + j] = a;
      }
    __syncthreads();
    const double inv = 1.0 / M[(long)col * w + col];
    __syncthreads();
    for (int j = t; j < w; j += 1024) M[(long)col * w + j] *= inv;
    for (int r = t; r < n; r += 1024) F[r] = r == col ? 0.0 : M[(long)r * w + col];
    __syncthreads();
    // thread t owns column t (w <= 1024); left-half columns before the pivot
    // are already unit vectors with a zero in the pivot row, so they stay
    if (t < w && (t >= col)) {
      const double pc = M[(long)col * w + t];
      if (pc != 0.0)
        for (int r = 0; r < n; ++r)
          if (r != col) M[(long)r * w + t] = fma(-F[r], pc, M[(long)r * w + t]);
    }
    __syncthreads();
  }
}

// Inverse of a dense matrix of at most 128 rows in one workgroup, in place in
// registers: thread (ti, tj) of 32 x 32 holds the entries (ti + 32 a, tj +
// 32 b).  Gauss-Jordan with partial pivoting; the pivot row stays where it is
// (rows are marked as used) and the permutation is applied on the way out:
// with p_k the pivot row of column k, (A^-1)(k, p_j) = M(p_k, j).  Per column
// one wavefront finds the pivot and two 128-value vectors cross LDS.  (On an
// n x 2n matrix in global memory: 2,017 us for the 32^3 cavity's, now 271.)
constexpr int kAmgRegInv = 128;
__global__ __launch_bounds__(1024) void k_amg_inverse(int n, const double* __restrict__ M, double* __restrict__ out,
                                                      int* __restrict__ err) {
  __shared__ double s_col[kAmgRegInv], s_row[kAmgRegInv];
  __shared__ int s_piv[kAmgRegInv], s_used[kAmgRegInv], s_p;
  __shared__ double s_inv;
  const int ti = threadIdx.x >> 5, tj = threadIdx.x & 31;
  double m[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int i = ti + 32 * a, j = tj + 32 * b;
      m[a][b] = i < n && j < n ? M[(long)i * 2 * n + j] : 0.0;
    }
  if (threadIdx.x < kAmgRegInv) s_used[threadIdx.x] = 0;
  for (int k = 0; k < n; ++k) {
    const int kb = k >> 5, kt = k & 31;
    if (tj == kt) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
        if (b == kb) {
#pragma unroll
          for (int a = 0; a < 4; ++a) s_col[ti + 32 * a] = m[a][b];
        }
    }
    __syncthreads();
    if (threadIdx.x < 64) {
      double best = -1.0;
      int bi = n;
      for (int i = threadIdx.x; i < n; i += 64) {
        const double v = s_used[i] ? -1.0 : fabs(s_col[i]);
        if (v > best) best = v, bi = i;
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        const double ov = __shfl_xor(best, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (ov > best || (ov == best && oi < bi)) best = ov, bi = oi;
      }
      if (threadIdx.x == 0) {
        const bool ok = best > 0.0;
        s_p = ok ? bi : -1;
        if (ok) {
          s_inv = 1.0 / s_col[bi];
          s_used[bi] = 1;
          s_piv[k] = bi;
        } else {
          atomicOr(err, 4);
        }
      }
    }
    __syncthreads();
    const int p = s_p;
    if (p < 0) return;  // uniform across the workgroup
    const double inv = s_inv;
    // the scaled pivot row (the inverse pivot in column k)
    if (ti == (p & 31)) {
#pragma unroll
      for (int a = 0; a < 4; ++a)
        if (a == (p >> 5)) {
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const double v = tj + 32 * b == k ? inv : m[a][b] * inv;
            m[a][b] = v;
            s_row[tj + 32 * b] = v;
          }
        }
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int i = ti + 32 * a;
      const double f = s_col[i];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int j = tj + 32 * b;
        if (i != p) m[a][b] = j == k ? -f * inv : fma(-f, s_row[j], m[a][b]);
      }
    }
    __syncthreads();  // s_col and s_row are rewritten in the next column
  }
  // row p_k of M is row k of the inverse
  __shared__ int s_of[kAmgRegInv];
  if (threadIdx.x < n) s_of[s_piv[threadIdx.x]] = threadIdx.x;
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int i = ti + 32 * a, j = tj + 32 * b;
      if (i < n && j < n) out[(long)s_of[i] * n + s_piv[j]] = m[a][b];
    }
}

template <class T>
__global__ void k_amg_extract_inv(long n, const double* __restrict__ M, T* __restrict__ out) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * n) return;
  const long r = idx / n, c = idx - r * n;
  out[idx] = (T)M[r * 2 * n + n + c];
}

template <class TI, class TO>
__global__ void k_amg_cast(long n, const TI* __restrict__ a, TO* __restrict__ b) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (TO)a[i];
}

// nodal block inverses: the BS x BS diagonal block of node k (DOFs k*BS ..
// k*BS+BS-1, consecutive columns in every sorted row), Gauss-Jordan with
// partial pivoting in FP64; a zero pivot leaves a zero block (no smoothing of
// that node) instead of Inf
template <int BS>
__global__ void k_amg_block_inv(long nblk, const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                const double* __restrict__ A, double* __restrict__ out) {
  const long blk = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (blk >= nblk) return;
  double M[BS][BS], I[BS][BS];
  const int c0 = (int)(blk * BS);
  for (int i = 0; i < BS; ++i) {
    int lo = rp[c0 + i], hi = rp[c0 + i + 1];
    const int end = hi;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (ci[mid] < c0) lo = mid + 1;
      else hi = mid;
    }
    int k = lo;
    for (int j = 0; j < BS; ++j) {
      const bool hit = k < end && ci[k] == c0 + j;
      M[i][j] = hit ? A[k] : 0.0;
      k += hit;
      I[i][j] = i == j ? 1.0 : 0.0;
    }
  }
  bool ok = true;
  for (int col = 0; col < BS; ++col) {
    int piv = col;
    double best = fabs(M[col][col]);
    for (int r = col + 1; r < BS; ++r)
      if (fabs(M[r][col]) > best) {
        best = fabs(M[r][col]);
        piv = r;
      }
    if (!(best > 0.0)) {
      ok = false;
      break;
    }
    if (piv != col)
      for (int j = 0; j < BS; ++j) {
        double t = M[col][j]; M[col][j] = M[piv][j]; M[piv][j] = t;
        t = I[col][j]; I[col][j] = I[piv][j]; I[piv][j] = t;
      }
    const double d = 1.0 / M[col][col];
    for (int j = 0; j < BS; ++j) {
      M[col][j] *= d;
      I[col][j] *= d;
    }
    for (int r = 0; r < BS; ++r) {
      if (r == col) continue;
      const double f = M[r][col];
      for (int j = 0; j < BS; ++j) {
        M[r][j] = fma(-f, M[col][j], M[r][j]);
        I[r][j] = fma(-f, I[col][j], I[r][j]);
      }
    }
  }
  for (int i = 0; i < BS; ++i)
    for (int j = 0; j < BS; ++j) out[blk * BS * BS + i * BS + j] = ok ? I[i][j] : 0.0;
}

// xout = (zero_x ? 0 : xin) + omega Binv r, one DOF per thread (in place allowed)
template <class T>
__global__ void k_amg_bj(long n, int nf, const T* __restrict__ binv, const T* __restrict__ r, const T* xin, T* xout,
                         double omega, int zero_x) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long node = (long)((unsigned)i / (unsigned)nf);  // rows fit 32 bits
  const int f = (int)(i - node * nf);
  const T* row = binv + node * nf * nf + f * nf;
  const T* rb = r + node * nf;
  double s = 0.0;
  for (int g = 0; g < nf; ++g) s = fma((double)row[g], (double)rb[g], s);
  xout[i] = (T)((zero_x ? 0.0 : (double)xin[i]) + omega * s);
}

// ---------------------------------------------------------------------------
// V-cycle kernels (T = double or float; sums in FP64)
// ---------------------------------------------------------------------------
template <int LANES, class T, class CI>
__device__ __forceinline__ double row_dot(const int32_t* __restrict__ rp, CI ci, const T* __restrict__ A,
                                          const T* __restrict__ x, long row, int l) {
  const int e = rp[row + 1];
  double acc = 0.0;
  int k = rp[row] + l;
  for (; k + 3 * LANES < e; k += 4 * LANES) {
    T av[4];
    int cv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      av[u] = A[k + u * LANES];
      cv[u] = ci(k + u * LANES);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) acc = fma((double)av[u], (double)x[cv[u]], acc);
  }
  for (; k < e; k += LANES) acc = fma((double)A[k], (double)x[ci(k)], acc);
#pragma unroll
  for (int off = LANES / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, LANES);
  return acc;
}

// LAT: the level-0 operator in the context's lattice pattern, columns from its
// closed form instead of ci (same entries, same order, same sums)
template <bool LAT>
__device__ __forceinline__ auto level_cols(const BoxMesh& m, const int32_t* __restrict__ rp,
                                           const int32_t* __restrict__ ci, long row) {
  if constexpr (LAT) return LatCols{lat_row(m, row), rp[row]};
  else return CsrCols{ci};
}

// The row ends of the level kernels: what happens with (A x)_row.
// w = s * D^-1 A v, s = *sp
struct DinvRow {
  const double* __restrict__ dinv;
  const double* __restrict__ sp;
  double* __restrict__ w;
  struct Pre {
    double s;
  };
  __device__ __forceinline__ Pre load(long row) const { return {*sp * dinv[row]}; }
  __device__ __forceinline__ void operator()(long row, double ax, Pre p) const { w[row] = p.s * ax; }
};
// d = alpha d + beta D^-1 (b - A xin), xout = xin + d (xin = 0 when zero_x)
template <class T>
struct ChebRow {
  const T* __restrict__ b;
  const T* __restrict__ xin;
  T* __restrict__ xout;
  T* __restrict__ d;
  const T* __restrict__ dinv;
  double alpha, beta;
  int zero_x;
  struct Pre {
    T b, x, d, dinv;
  };
  __device__ __forceinline__ Pre load(long row) const {
    return {b[row], zero_x ? (T)0 : xin[row], alpha != 0.0 ? d[row] : (T)0, dinv[row]};
  }
  __device__ __forceinline__ void operator()(long row, double ax, const Pre& p) const {
    const double r = (double)p.b - ax;
    const double dn = (alpha != 0.0 ? alpha * (double)p.d : 0.0) + beta * (double)p.dinv * r;
    d[row] = (T)dn;
    xout[row] = (T)((double)p.x + dn);
  }
};
// r = b - A x
template <class T>
struct ResidRow {
  const T* __restrict__ b;
  T* __restrict__ r;
  struct Pre {
    T b;
  };
  __device__ __forceinline__ Pre load(long row) const { return {b[row]}; }
  __device__ __forceinline__ void operator()(long row, double ax, Pre p) const { r[row] = (T)((double)p.b - ax); }
};

// the same ends, and the nodal block-Jacobi update, for four unknowns per node
// (k_node4_product)
struct DinvNode {
  DinvRow r;
  using Pre = DinvRow::Pre;
  __device__ __forceinline__ Pre load(unsigned, int, int, unsigned row) const { return r.load(row); }
  __device__ __forceinline__ void operator()(bool act, unsigned, int, int d, unsigned row, double ax, Pre p) const {
    if (act && d == 0) r(row, ax, p);
  }
};
template <class T>
struct ResidNode {
  ResidRow<T> r;
  using Pre = typename ResidRow<T>::Pre;
  __device__ __forceinline__ Pre load(unsigned, int, int, unsigned row) const { return r.load(row); }
  __device__ __forceinline__ void operator()(bool act, unsigned, int, int d, unsigned row, double ax, Pre p) const {
    if (act && d == 0) r(row, ax, p);
  }
};
// xout = xin + omega Binv (b - A xin)
template <class T>
struct BjNode {
  const T* __restrict__ binv;
  const T* __restrict__ b;
  const T* __restrict__ xin;
  T* __restrict__ xout;
  double omega;
  struct Pre {
    T b, x, binv;
  };
  __device__ __forceinline__ Pre load(unsigned node, int f, int d, unsigned row) const {
    return {b[row], xin[row], binv[16 * node + 4 * f + d]};
  }
  __device__ __forceinline__ void operator()(bool act, unsigned, int, int d, unsigned row, double ax,
                                             const Pre& p) const {
    // lane (f, d): the residual of field d, from the first lane of its quad
    const double r = (double)p.b - ax;
    const int lane = threadIdx.x & 63;
    double v = (double)p.binv * __shfl(r, (lane & ~15) + 4 * d, 64);
    v += dpp_move<kDppXor1>(v);
    v += dpp_move<kDppXor2>(v);
    if (act && d == 0) xout[row] = (T)((double)p.x + omega * v);
  }
};

// w = s * D^-1 A v  (s = *sp, on the device: the scale applied to v, so v
// need not be normalised in place)
template <int LANES, bool LAT>
__global__ __launch_bounds__(256) void k_amg_dinv_spmv(BoxMesh m, long n, const int32_t* __restrict__ rp,
                                                       const int32_t* __restrict__ ci, const double* __restrict__ A,
                                                       const double* __restrict__ v, DinvRow end) {
  const long row = ((long)blockIdx.x * blockDim.x + threadIdx.x) / LANES;
  const int l = threadIdx.x % LANES;
  if (row >= n) return;
  const double acc = row_dot<LANES, double>(rp, level_cols<LAT>(m, rp, ci, row), A, v, row, l);
  if (l == 0) end(row, acc, end.load(row));
}

// scalar steps of the power iteration, one thread; st = (s, lambda, stopped).
// phase 0: s = 1 / sqrt(v.v); 1: lambda = s (v.w), then s = 1 / |w| unless
// |w| is zero or not finite, which stops the iteration (later steps leave
// lambda alone); 2: lambda = 1 where it is not a finite positive number.
__global__ void k_amg_power(int phase, const double* __restrict__ d0, const double* __restrict__ d1,
                            double* __restrict__ st) {
  if (phase == 0) {
    st[0] = 1.0 / sqrt(*d0);
    st[1] = 1.0;
    st[2] = 0.0;
  } else if (phase == 1) {
    if (st[2] != 0.0) return;
    st[1] = st[0] * *d0;
    const double wn = sqrt(*d1);
    if (!(wn > 0.0) || !isfinite(wn)) st[2] = 1.0;
    else st[0] = 1.0 / wn;
  } else {
    const double lam = st[1];
    st[1] = (isfinite(lam) && lam > 0.0) ? lam : 1.0;
  }
}

// one Chebyshev step (A xin skipped when zero_x)
template <int LANES, bool LAT, class T>
__global__ __launch_bounds__(256) void k_amg_cheb(BoxMesh m, long n, const int32_t* __restrict__ rp,
                                                  const int32_t* __restrict__ ci, const T* __restrict__ A,
                                                  ChebRow<T> end) {
  const long row = ((long)blockIdx.x * blockDim.x + threadIdx.x) / LANES;
  const int l = threadIdx.x % LANES;
  if (row >= n) return;
  const double ax =
      end.zero_x ? 0.0 : row_dot<LANES, T>(rp, level_cols<LAT>(m, rp, ci, row), A, end.xin, row, l);
  if (l == 0) end(row, ax, end.load(row));
}

template <int LANES, bool LAT, class T>
__global__ __launch_bounds__(256) void k_amg_resid(BoxMesh m, long n, const int32_t* __restrict__ rp,
                                                   const int32_t* __restrict__ ci, const T* __restrict__ A,
                                                   const T* __restrict__ x, ResidRow<T> end) {
  const long row = ((long)blockIdx.x * blockDim.x + threadIdx.x) / LANES;
  const int l = threadIdx.x % LANES;
  if (row >= n) return;
  const double ax = row_dot<LANES, T>(rp, level_cols<LAT>(m, rp, ci, row), A, x, row, l);
  if (l == 0) end(row, ax, end.load(row));
}

// One colour of a multicolour nodal block Gauss-Seidel sweep: for every node
// of the colour, x_node += Binv_node (b - A x)_node.  Colour (cx, cy, cz) of
// stride s holds the nodes whose lattice coordinates are congruent to it
// modulo s; with s = reach + 1 no two nodes of a colour share a matrix entry,
// so the in-place update is race free.  A group of NFP * LANES lanes (NFP = nf
// rounded up to a power of two, groups never straddle a wavefront) owns a
// node, LANES lanes per row; the rows' residuals meet through wavefront
// shuffles, which every lane executes.
template <int LANES, int NFP, class T>
__global__ __launch_bounds__(256) void k_amg_gs(long ncol, int nf, int s, int cx, int cy, int cz, long cntx, long cnty,
                                                long Nx, long Ny, const int32_t* __restrict__ rp,
                                                const int32_t* __restrict__ ci, const T* __restrict__ A,
                                                const T* __restrict__ binv, const T* __restrict__ b, T* x) {
  static_assert(NFP * LANES <= 64 && 64 % (NFP * LANES) == 0, "node group must tile a wavefront");
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long t = gid / (NFP * LANES);
  const int within = (int)(gid % (NFP * LANES));
  const int f = within / LANES, l = within % LANES;
  const bool active = t < ncol && f < nf;
  long node = 0, row = 0;
  double res = 0.0;
  if (active) {
    // node numbers fit 32 bits: 32-bit unsigned divisions
    const unsigned tu = (unsigned)t, q = tu / (unsigned)cntx, qz = q / (unsigned)cnty;
    const long a = (long)(tu - q * (unsigned)cntx), qy = (long)(q - qz * (unsigned)cnty);
    node = (cx + s * a) + Nx * ((cy + s * qy) + Ny * (cz + s * (long)qz));
    row = node * nf + f;
    res = (double)b[row] - row_dot<LANES, T>(rp, CsrCols{ci}, A, x, row, l);
  }
  const int base = (int)(threadIdx.x & 63) - within;
  double upd = 0.0;
#pragma unroll
  for (int g = 0; g < NFP; ++g) {
    const double rg = __shfl(res, base + g * LANES, 64);
    if (active && g < nf) upd = fma((double)binv[(node * nf + f) * nf + g], rg, upd);
  }
  if (active && l == 0) x[row] = (T)((double)x[row] + upd);
}

template <class T>
__global__ void k_amg_fill0(long n, T* x) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = (T)0;
}

// y = M x, or y = y0 + M x (y0 may be y)
template <int LANES, class T>
__global__ __launch_bounds__(256) void k_amg_spmv(long n, const int32_t* __restrict__ rp,
                                                  const int32_t* __restrict__ ci, const T* __restrict__ M,
                                                  const T* __restrict__ x, const T* y0, T* y) {
  const long row = ((long)blockIdx.x * blockDim.x + threadIdx.x) / LANES;
  const int l = threadIdx.x % LANES;
  if (row >= n) return;
  const double v = row_dot<LANES, T>(rp, CsrCols{ci}, M, x, row, l);
  if (l == 0) y[row] = (T)(y0 ? (double)y0[row] + v : v);
}

// x = Cinv b, one wavefront per row of the dense coarsest inverse.  The
// inverse stays FP64 in both precisions: in FP32 its rounding error would be
// amplified by the condition number of the coarsest operator.
template <class T>
__global__ __launch_bounds__(256) void k_amg_gemv(long n, const double* __restrict__ Cinv, const T* __restrict__ b,
                                                  T* __restrict__ x) {
  const long row = ((long)blockIdx.x * blockDim.x + threadIdx.x) / 64;
  const int l = threadIdx.x % 64;
  if (row >= n) return;
  double acc = 0.0;
  for (long j = l; j < n; j += 64) acc = fma((double)Cinv[row * n + j], (double)b[j], acc);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (l == 0) x[row] = (T)acc;
}

// ---------------------------------------------------------------------------
// hierarchy
// ---------------------------------------------------------------------------
template <class T>
struct AmgVals {
  DevBuf<T> A, dinv, P, R, cinv, binv;
  DevBuf<T> x, t, b, r, d;  // level work vectors
};

struct AmgLevel {
  long n = 0;            // rows (nodes x fields)
  int N[3] = {1, 1, 1};  // node lattice
  int reach = 1;
  int lanes = 4, plane = 4, rlane = 4;  // lanes per row: A, P, R
  const int32_t* rp = nullptr;  // level 0: the context's pattern
  const int32_t* ci = nullptr;
  DevBuf<int32_t> rp_own, ci_own;
  DevBuf<double> A, dinv, ns;
  DevBuf<int32_t> prp, pci, rrp, rci, tab;
  DevBuf<double> P, R;
  DevBuf<double> binv;  // nodal nf x nf diagonal-block inverses (block-Jacobi smoother)
  bool lat = false;     // level 0 in the context's lattice pattern: closed-form columns
  // products of lattice_product.hpp: order 2 (level 0), four unknowns per node
  // (every level; colidx: level 0 with the index stream)
  bool q2 = false, node4 = false, colidx = false;
  double lambda = 1.0;
  AmgVals<float> f32;
  AmgVals<double> f64;  // FP64 work vectors (values live in A/P/R above)
};

struct Amg {
  std::vector<std::unique_ptr<AmgLevel>> lv;
  DevBuf<double> cinv;    // dense inverse of the coarsest operator (FP64 in both precisions)
  DevBuf<double> scratch;  // set-up temporaries
  DevBuf<int> err;
  // power iterations on the device: two inner-product slots, then per level
  // (s, lambda, stopped, -)
  DevBuf<double> pw;
  const double* A0 = nullptr;  // level-0 operator of the last set-up
  bool fp32 = false;
  int smoother = kSmootherChebyshev;
  int sweeps = kBjSweeps;   // block-Jacobi sweeps before and after the coarse correction
  double omega = kBjOmega;  // block-Jacobi damping
  int nf = 1;
  bool built = false;  // a set-up is complete
  int64_t setup_count = 0;
  int64_t reuse_count = 0;  // set-ups answered by refreshing the fine level only
};

static int lanes_for(double avg) {
  int l = 4;
  while (l < 64 && l * 14 < avg) l *= 2;
  return l;
}

static dim3 g1(long n, int b = 256) { return dim3((unsigned)((n + b - 1) / b)); }

template <class K>
static void by_lanes(int lanes, K&& k) {
  switch (lanes) {
    case 4: k(std::integral_constant<int, 4>{}); break;
    case 8: k(std::integral_constant<int, 8>{}); break;
    case 16: k(std::integral_constant<int, 16>{}); break;
    case 32: k(std::integral_constant<int, 32>{}); break;
    default: k(std::integral_constant<int, 64>{}); break;
  }
}

template <class F>
static void by_lat(bool lat, F&& f) {
  if (lat) f(std::true_type{});
  else f(std::false_type{});
}

static Geo upload_geo(Ctx& c, AmgLevel& L, const AxisHost* ax, int nf) {
  size_t total = 0;
  for (int d = 0; d < 3; ++d)
    for (int k = 0; k < kNumTables; ++k) total += ax[d].t[k].size();
  L.tab.alloc(total);
  std::vector<int32_t> h(total);
  Geo G{};
  size_t off = 0;
  for (int d = 0; d < 3; ++d) {
    G.ax[d].n = ax[d].n;
    G.ax[d].na = ax[d].na;
    G.ax[d].b = ax[d].b;
    for (int k = 0; k < kNumTables; ++k) {
      std::copy(ax[d].t[k].begin(), ax[d].t[k].end(), h.begin() + off);
      G.ax[d].t[k] = L.tab.p + off;
      off += ax[d].t[k].size();
    }
  }
  MHX_HIP(hipMemcpyAsync(L.tab.p, h.data(), total * sizeof(int32_t), hipMemcpyHostToDevice, c.stream));
  G.nf = nf;
  return G;
}

// the set-up's one host synchronisation: its error bits (4: singular coarsest
// operator) and the lambda of each of the first n_smoothed levels
static void finish_setup(Ctx& c, Amg& H, int n_smoothed) {
  int e = 0;
  std::vector<double> st(2 + 4 * (size_t)n_smoothed);
  MHX_HIP(hipMemcpyAsync(&e, H.err.p, sizeof(int), hipMemcpyDeviceToHost, c.stream));
  if (n_smoothed > 0)
    MHX_HIP(hipMemcpyAsync(st.data(), H.pw.p, st.size() * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  MHX_HIP(hipStreamSynchronize(c.stream));
  for (int l = 0; l < n_smoothed; ++l) H.lv[l]->lambda = st[2 + 4 * l + 1];
  if (e & 4) throw Error{MHX_ERR_NONFINITE, "AMG: singular coarsest operator"};
}

// lambda ~ rho(D^-1 A) by power iteration from a fixed start vector,
// entirely on the stream: the scale s and the estimate stay on the device
// (st = (s, lambda, stopped)), and the host reads every level's lambda once,
// at the end of the set-up.  The steps are the host form's, in the same
// floating-point operations: lambda = s (v . D^-1 A s v), s = 1 / |w|.
static void power_estimate(Ctx& c, AmgLevel& L, const double* A, double* v, double* w, double* slots,
                           double* st) {
  const long n = L.n;
  hipLaunchKernelGGL(k_amg_start, g1(n), dim3(256), 0, c.stream, n, v);
  MHX_HIP(hipGetLastError());
  dot_dev(c, v, v, n, slots);
  hipLaunchKernelGGL(k_amg_power, dim3(1), dim3(1), 0, c.stream, 0, slots, slots, st);
  for (int it = 0; it < kAmgPowerIters; ++it) {
    const DinvRow end{L.dinv.p, st, w};
    if (L.q2) {
      q2_product<double>(c, A, v, end);
    } else if (L.node4) {
      node4_product<double>(c, L.N, L.rp, L.ci, L.colidx, A, v, DinvNode{end});
    } else {
      by_lanes(L.lanes, [&](auto LN) {
        by_lat(L.lat, [&](auto LT) {
          hipLaunchKernelGGL((k_amg_dinv_spmv<decltype(LN)::value, decltype(LT)::value>), g1(n * LN), dim3(256), 0,
                             c.stream, c.mesh, n, L.rp, L.ci, A, v, end);
        });
      });
    }
    MHX_HIP(hipGetLastError());
    dot_dev(c, v, w, n, slots);
    dot_dev(c, w, w, n, slots + 1);
    hipLaunchKernelGGL(k_amg_power, dim3(1), dim3(1), 0, c.stream, 1, slots, slots + 1, st);
    std::swap(v, w);
  }
  hipLaunchKernelGGL(k_amg_power, dim3(1), dim3(1), 0, c.stream, 2, slots, slots, st);
  MHX_HIP(hipGetLastError());
}

void amg_setup(Ctx& c, const double* A, bool fp32) {
  ScopedPhase ph(c.prof, "LinearAlgebraInterface::buildAMGPreconditioner", c.stream);
  if (!c.amg) c.amg = std::make_shared<Amg>();
  Amg& H = *c.amg;
  const int nf = c.nfield;
  MHX_REQUIRE(nf >= 1 && nf <= kAmgMaxFields, MHX_ERR_UNSUPPORTED, "AMG: at most 4 unknowns per node");
  // automatic choice: Chebyshev on the point diagonal for one unknown per
  // node, nodal block Jacobi for coupled fields
  const int smoother = c.amg_smoother >= 0 ? c.amg_smoother : (nf > 1 ? kSmootherBlockJacobi : kSmootherChebyshev);
  // reuse (MueLu "reuse: full" in kind): keep the coarse levels of the last
  // set-up and refresh only what the fine-level smoother reads from the new
  // operator (its diagonal, or its nodal block inverses); the fine operator
  // itself is the new one, passed to every V-cycle
  if (c.amg_reuse && H.built && H.fp32 == fp32 && H.nf == nf && H.smoother == smoother &&
      !H.lv.empty() && H.lv[0]->n == c.mesh.ndof) {
    AmgLevel& L0 = *H.lv[0];
    H.A0 = A;
    // cycle parameters are read per V-cycle: take the current options
    H.sweeps = c.amg_sweeps;
    H.omega = c.amg_omega_pct * 0.01;
    hipLaunchKernelGGL(k_amg_diag, g1(L0.n), dim3(256), 0, c.stream, L0.n, L0.rp, L0.ci, A, L0.dinv.p);
    if (H.smoother != kSmootherChebyshev && H.lv.size() > 1) {
      const long nblk = L0.n / nf;
      switch (nf) {
        case 1: hipLaunchKernelGGL(k_amg_block_inv<1>, g1(nblk), dim3(256), 0, c.stream, nblk, L0.rp, L0.ci, A, L0.binv.p); break;
        case 2: hipLaunchKernelGGL(k_amg_block_inv<2>, g1(nblk), dim3(256), 0, c.stream, nblk, L0.rp, L0.ci, A, L0.binv.p); break;
        case 3: hipLaunchKernelGGL(k_amg_block_inv<3>, g1(nblk), dim3(256), 0, c.stream, nblk, L0.rp, L0.ci, A, L0.binv.p); break;
        default: hipLaunchKernelGGL(k_amg_block_inv<4>, g1(nblk), dim3(256), 0, c.stream, nblk, L0.rp, L0.ci, A, L0.binv.p); break;
      }
    }
    if (fp32) {
      hipLaunchKernelGGL((k_amg_cast<double, float>), g1(L0.n), dim3(256), 0, c.stream, L0.n, L0.dinv.p,
                         L0.f32.dinv.p);
      if (H.smoother != kSmootherChebyshev && H.lv.size() > 1)
        hipLaunchKernelGGL((k_amg_cast<double, float>), g1((long)L0.binv.n), dim3(256), 0, c.stream,
                           (long)L0.binv.n, L0.binv.p, L0.f32.binv.p);
    }
    MHX_HIP(hipGetLastError());
    ++H.reuse_count;
    return;
  }
  H.err.alloc(1);
  H.pw.alloc(2 + 4 * kAmgMaxLevels);
  MHX_HIP(hipMemsetAsync(H.err.p, 0, sizeof(int), c.stream));
  H.A0 = A;
  H.fp32 = fp32;
  H.smoother = smoother;
  H.sweeps = c.amg_sweeps;
  H.omega = c.amg_omega_pct * 0.01;
  H.nf = nf;
  ++H.setup_count;
  H.built = false;  // (until the end: a set-up that fails leaves nothing to reuse)

  // level 0: the context's lattice and pattern
  int nlev = 0;
  auto next_level = [&]() -> AmgLevel& {
    if ((int)H.lv.size() <= nlev) H.lv.emplace_back(new AmgLevel());
    return *H.lv[nlev++];
  };
  AmgLevel* L = &next_level();
  L->n = c.mesh.ndof;
  for (int d = 0; d < 3; ++d) L->N[d] = d < c.mesh.dim ? c.mesh.nn[d] : 1;
  L->reach = c.mesh.p;
  L->rp = c.rowptr.p;
  L->ci = c.colidx.p;
  L->lanes = c.spmv_lanes;
  L->lat = c.lattice_cols != 0;
  L->q2 = q2_product_applies(c);
  L->node4 = node4_product_applies(c);
  L->colidx = !L->lat;
  L->dinv.alloc(L->n);
  L->ns.alloc(L->n);
  hipLaunchKernelGGL(k_amg_diag, g1(L->n), dim3(256), 0, c.stream, L->n, L->rp, L->ci, A, L->dinv.p);
  hipLaunchKernelGGL(k_amg_ns0, g1(L->n), dim3(256), 0, c.stream, L->n, c.fixed.p, L->ns.p);
  MHX_HIP(hipGetLastError());
  const double* Acur = A;

  while (L->n > kAmgCoarseMax && nlev < kAmgMaxLevels) {
    const int r = std::max(1, L->reach);
    const int b = 2 * r + 1;
    const int rc = (3 * r - 1) / b + 1;
    AxisHost ax[3];
    for (int d = 0; d < 3; ++d) make_axis(ax[d], L->N[d], r, rc);
    const long ncn = (long)ax[0].na * ax[1].na * ax[2].na;
    const long nc = ncn * nf;
    if (nc >= L->n) break;  // no coarsening left
    Geo G = upload_geo(c, *L, ax, nf);
    const long n = L->n;
    // lambda (on the device; omega = damping / lambda is formed by k_amg_P)
    H.scratch.alloc(std::max<size_t>(H.scratch.n, (size_t)2 * n));
    double* st = H.pw.p + 2 + 4 * (nlev - 1);
    power_estimate(c, *L, Acur, H.scratch.p, H.scratch.p + n, H.pw.p, st);
    // next level's near-null space = aggregate norms
    AmgLevel& C = next_level();
    L = H.lv[nlev - 2].get();  // the vector may have grown
    C.n = nc;
    for (int d = 0; d < 3; ++d) C.N[d] = ax[d].na;
    C.reach = rc;
    C.node4 = L->node4 && rc == 1;
    C.q2 = C.lat = C.colidx = false;
    C.ns.alloc(nc);
    hipLaunchKernelGGL(k_amg_nrm, g1(nc), dim3(256), 0, c.stream, G, L->ns.p, C.ns.p, nc);
    // P
    const long p_nnz = (long)nf * nf * ax[0].t[kSp][ax[0].n] * (long)ax[1].t[kSp][ax[1].n] * ax[2].t[kSp][ax[2].n];
    const long r_nnz = (long)nf * nf * ax[0].t[kSr][ax[0].na] * (long)ax[1].t[kSr][ax[1].na] * ax[2].t[kSr][ax[2].na];
    const long a_nnz = (long)nf * nf * ax[0].t[kSc][ax[0].na] * (long)ax[1].t[kSc][ax[1].na] * ax[2].t[kSc][ax[2].na];
    MHX_REQUIRE(p_nnz < INT_MAX && r_nnz < INT_MAX && a_nnz < INT_MAX, MHX_ERR_UNSUPPORTED,
                "AMG: transfer operator exceeds 32-bit indexing");
    L->prp.alloc(n + 1);
    L->pci.alloc(p_nnz);
    L->P.alloc(p_nnz);
    hipLaunchKernelGGL(k_box_rowptr, g1(n + 1), dim3(256), 0, c.stream, G, 0, (int)kPext, (int)kSp, n, L->prp.p);
    const LevelBox box{{L->N[0], L->N[1], L->N[2]}, nlev == 2 ? c.mesh.p : 1, L->reach};
    hipLaunchKernelGGL(k_amg_P, g1(n * kApLanes, kAmgBlk), dim3(kAmgBlk), 0, c.stream, G, box, n, L->rp, Acur,
                       L->dinv.p, L->ns.p, C.ns.p, st + 1, L->prp.p, L->pci.p, L->P.p);
    // R = P^T
    L->rrp.alloc(nc + 1);
    L->rci.alloc(r_nnz);
    L->R.alloc(r_nnz);
    hipLaunchKernelGGL(k_box_rowptr, g1(nc + 1), dim3(256), 0, c.stream, G, 1, (int)kRext, (int)kSr, nc, L->rrp.p);
    hipLaunchKernelGGL(k_amg_R, dim3((unsigned)nc), dim3(kAmgBlk), 0, c.stream, G, L->prp.p, L->P.p, L->rrp.p,
                       L->rci.p, L->R.p);
    // A P (dense 27-slot boxes), then A_c = R (A P)
    H.scratch.alloc(std::max<size_t>(H.scratch.n, (size_t)n * nf * 27));
    hipLaunchKernelGGL(k_amg_AP, g1(n * nf * kApLanes, kAmgBlk), dim3(kAmgBlk), 0, c.stream, G, box, n, L->rp, Acur,
                       L->prp.p, L->P.p, H.scratch.p);
    C.rp_own.alloc(nc + 1);
    C.ci_own.alloc(a_nnz);
    C.A.alloc(a_nnz);
    hipLaunchKernelGGL(k_box_rowptr, g1(nc + 1), dim3(256), 0, c.stream, G, 1, (int)kCext, (int)kSc, nc,
                       C.rp_own.p);
    for (int d = 0; d < 3; ++d) {
      const auto& rx = ax[d].t[kRext];
      const auto& cx = ax[d].t[kCext];
      MHX_REQUIRE(*std::max_element(rx.begin(), rx.end()) <= kAcMaxExt, MHX_ERR_UNSUPPORTED,
                  "AMG: restriction row longer than the Galerkin kernel's");
      MHX_REQUIRE(*std::max_element(cx.begin(), cx.end()) <= 5, MHX_ERR_UNSUPPORTED,
                  "AMG: coarse operator row wider than the Galerkin kernel's");
    }
    auto galerkin = [&](auto F) {
      hipLaunchKernelGGL((k_amg_Ac<decltype(F)::value>), dim3((unsigned)nc), dim3(32 * kAcGroups), 0, c.stream, G,
                         L->rrp.p, L->R.p, H.scratch.p, C.ns.p, C.rp_own.p, C.ci_own.p, C.A.p);
    };
    switch (nf) {
      case 1: galerkin(std::integral_constant<int, 1>{}); break;
      case 2: galerkin(std::integral_constant<int, 2>{}); break;
      case 3: galerkin(std::integral_constant<int, 3>{}); break;
      default: galerkin(std::integral_constant<int, 4>{}); break;
    }
    MHX_HIP(hipGetLastError());
    L->plane = lanes_for((double)p_nnz / (double)n);
    L->rlane = lanes_for((double)r_nnz / (double)nc);
    C.rp = C.rp_own.p;
    C.ci = C.ci_own.p;
    C.lanes = lanes_for((double)a_nnz / (double)nc);
    C.dinv.alloc(nc);
    hipLaunchKernelGGL(k_amg_diag, g1(nc), dim3(256), 0, c.stream, nc, C.rp, C.ci, C.A.p, C.dinv.p);
    MHX_HIP(hipGetLastError());
    Acur = C.A.p;
    L = &C;
  }
  H.lv.resize(nlev);
  // coarsest: dense inverse
  {
    AmgLevel& Z = *H.lv.back();
    const long n = Z.n;
    MHX_REQUIRE(n <= kAmgDenseMax, MHX_ERR_UNSUPPORTED, "AMG: coarsest level too large for the dense solve");
    H.scratch.alloc(std::max<size_t>(H.scratch.n, (size_t)2 * n * n + n));
    hipLaunchKernelGGL(k_amg_dense, g1(n), dim3(256), 0, c.stream, n, Z.rp, Z.ci, Acur, H.scratch.p);
    H.cinv.alloc(n * n);
    if (n <= kAmgRegInv) {
      hipLaunchKernelGGL(k_amg_inverse, dim3(1), dim3(1024), 0, c.stream, (int)n, H.scratch.p, H.cinv.p, H.err.p);
    } else {
      hipLaunchKernelGGL(k_amg_gauss_jordan, dim3(1), dim3(1024), 0, c.stream, (int)n, H.scratch.p,
                         H.scratch.p + 2 * n * n, H.err.p);
      hipLaunchKernelGGL(k_amg_extract_inv<double>, g1(n * n), dim3(256), 0, c.stream, n, H.scratch.p, H.cinv.p);
    }
    MHX_HIP(hipGetLastError());
    finish_setup(c, H, nlev - 1);
  }
  // block-Jacobi smoother: nodal block inverses of every smoothed level
  if (H.smoother != kSmootherChebyshev) {
    for (int l = 0; l + 1 < nlev; ++l) {
      AmgLevel& V = *H.lv[l];
      const long nblk = V.n / nf;
      V.binv.alloc((size_t)nblk * nf * nf);
      const double* Al = l ? V.A.p : A;
      switch (nf) {
        case 1: hipLaunchKernelGGL(k_amg_block_inv<1>, g1(nblk), dim3(256), 0, c.stream, nblk, V.rp, V.ci, Al, V.binv.p); break;
        case 2: hipLaunchKernelGGL(k_amg_block_inv<2>, g1(nblk), dim3(256), 0, c.stream, nblk, V.rp, V.ci, Al, V.binv.p); break;
        case 3: hipLaunchKernelGGL(k_amg_block_inv<3>, g1(nblk), dim3(256), 0, c.stream, nblk, V.rp, V.ci, Al, V.binv.p); break;
        default: hipLaunchKernelGGL(k_amg_block_inv<4>, g1(nblk), dim3(256), 0, c.stream, nblk, V.rp, V.ci, Al, V.binv.p); break;
      }
    }
  }
  // FP32 copies of the operators
  for (int l = 0; l < nlev; ++l) {
    AmgLevel& V = *H.lv[l];
    const bool last = l == nlev - 1;
    auto vecs = [&](auto& W) {
      W.x.alloc(V.n); W.t.alloc(V.n); W.b.alloc(V.n); W.r.alloc(V.n); W.d.alloc(V.n);
    };
    if (fp32) {
      vecs(V.f32);
      auto cast = [&](const double* s, DevBuf<float>& d, long m) {
        d.alloc(m);
        hipLaunchKernelGGL((k_amg_cast<double, float>), g1(m), dim3(256), 0, c.stream, m, s, d.p);
      };
      cast(V.dinv.p, V.f32.dinv, V.n);
      if (H.smoother != kSmootherChebyshev && !last) cast(V.binv.p, V.f32.binv, V.binv.n);
      if (l > 0) cast(V.A.p, V.f32.A, V.A.n);
      if (!last) {
        cast(V.P.p, V.f32.P, V.P.n);
        cast(V.R.p, V.f32.R, V.R.n);
      }
    } else {
      vecs(V.f64);
    }
  }
  MHX_HIP(hipGetLastError());
  H.built = true;
}

// Chebyshev coefficients of one level (Ifpack2's three-term recurrence)
struct Cheb {
  double inv_theta, a2, b2;
};
static Cheb cheb_coef(double lambda) {
  const double lmax = kChebBoost * lambda, lmin = lmax / kChebRatio;
  const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin);
  const double sigma = theta / delta, rho0 = 1.0 / sigma, rho1 = 1.0 / (2.0 * sigma - rho0);
  return Cheb{1.0 / theta, rho1 * rho0, 2.0 * rho1 / delta};
}

template <class T>
struct LvView {
  const T *A, *dinv, *P, *R, *binv;
  T *x, *t, *b, *r, *d;
};

template <class T>
static LvView<T> view(Amg& H, int l, const T* A0);
template <>
LvView<double> view<double>(Amg& H, int l, const double* A0) {
  AmgLevel& V = *H.lv[l];
  return {l ? V.A.p : A0, V.dinv.p, V.P.p, V.R.p, V.binv.p, V.f64.x.p, V.f64.t.p, V.f64.b.p, V.f64.r.p, V.f64.d.p};
}
template <>
LvView<float> view<float>(Amg& H, int l, const float* A0) {
  AmgLevel& V = *H.lv[l];
  return {l ? V.f32.A.p : A0, V.f32.dinv.p, V.f32.P.p, V.f32.R.p, V.f32.binv.p, V.f32.x.p, V.f32.t.p, V.f32.b.p,
          V.f32.r.p, V.f32.d.p};
}

template <class T>
static void cheb_step(Ctx& c, AmgLevel& V, const LvView<T>& W, const T* b, const T* xin, T* xout, double alpha,
                      double beta, int zero_x) {
  const ChebRow<T> end{b, xin, xout, W.d, W.dinv, alpha, beta, zero_x};
  if (V.q2 && !zero_x) {
    q2_product<double>(c, W.A, xin, end);
    return;
  }
  by_lanes(zero_x ? 4 : V.lanes, [&](auto LN) {
    by_lat(V.lat, [&](auto LT) {
      constexpr int K = decltype(LN)::value;
      constexpr bool LAT = decltype(LT)::value;
      hipLaunchKernelGGL((k_amg_cheb<K, LAT, T>), g1(V.n * K), dim3(256), 0, c.stream, c.mesh, V.n, V.rp, V.ci, W.A,
                         end);
    });
  });
}

// r = b - A x on one level
template <class T>
static void level_resid(Ctx& c, AmgLevel& V, const LvView<T>& W, const T* b, const T* x, T* r) {
  const ResidRow<T> end{b, r};
  if (V.q2) {
    q2_product<double>(c, W.A, x, end);
    return;
  }
  if (V.node4) {
    node4_product<T>(c, V.N, V.rp, V.ci, V.colidx, W.A, x, ResidNode<T>{end});
    return;
  }
  by_lanes(V.lanes, [&](auto LN) {
    by_lat(V.lat, [&](auto LT) {
      constexpr int K = decltype(LN)::value;
      constexpr bool LAT = decltype(LT)::value;
      hipLaunchKernelGGL((k_amg_resid<K, LAT, T>), g1(V.n * K), dim3(256), 0, c.stream, c.mesh, V.n, V.rp, V.ci,
                         W.A, x, end);
    });
  });
}

// Damped nodal block-Jacobi sweeps: x <- x + omega Binv (b - A x); with zero_x
// the first sweep starts from x = 0 and needs no residual.  With four unknowns
// per node a sweep is one launch from one vector into the other: the starting
// iterate is expected where bj_start says (x or W.t), and the last sweep ends
// in x.
template <class T>
static T* bj_start(const Amg& H, const AmgLevel& V, const LvView<T>& W, T* x, int zero_x) {
  const int fused = H.sweeps - (zero_x ? 1 : 0);
  return V.node4 && (fused & 1) ? W.t : x;
}
template <class T>
static void bj_smooth(Ctx& c, Amg& H, AmgLevel& V, const LvView<T>& W, const T* b, T* x, int zero_x) {
  T* cur = bj_start<T>(H, V, W, x, zero_x);
  for (int s = 0; s < H.sweeps; ++s) {
    const bool zero = zero_x && s == 0;
    if (!zero && V.node4) {
      T* nxt = cur == x ? W.t : x;
      node4_product<T>(c, V.N, V.rp, V.ci, V.colidx, W.A, cur, BjNode<T>{W.binv, b, cur, nxt, H.omega});
      cur = nxt;
      continue;
    }
    const T* r = b;
    if (!zero) {
      level_resid<T>(c, V, W, b, cur, W.t);
      r = W.t;
    }
    hipLaunchKernelGGL(k_amg_bj<T>, g1(V.n), dim3(256), 0, c.stream, V.n, H.nf, W.binv, r, cur, cur, H.omega,
                       (int)zero);
  }
}

// one multicolour block Gauss-Seidel sweep over the (reach+1)^d colours of
// the level's node lattice, in lexicographic colour order or its reverse
template <class T>
static void gs_sweep(Ctx& c, Amg& H, AmgLevel& V, const LvView<T>& W, const T* b, T* x, bool forward) {
  const int nf = H.nf;
  const int nfp = nf == 1 ? 1 : nf == 2 ? 2 : 4;
  const int s = std::max(1, V.reach) + 1;
  int nc[3];
  for (int d = 0; d < 3; ++d) nc[d] = V.N[d] > 1 ? s : 1;
  const int ncolour = nc[0] * nc[1] * nc[2];
  const int lanes = std::min(V.lanes, 64 / nfp);
  for (int k = 0; k < ncolour; ++k) {
    const int col = forward ? k : ncolour - 1 - k;
    const int cx = col % nc[0], cy = (col / nc[0]) % nc[1], cz = col / (nc[0] * nc[1]);
    const int co[3] = {cx, cy, cz};
    long cnt[3];
    for (int d = 0; d < 3; ++d) cnt[d] = V.N[d] > co[d] ? (V.N[d] - co[d] + s - 1) / s : 0;
    const long ncol = cnt[0] * cnt[1] * cnt[2];
    if (!ncol) continue;
    by_lanes(lanes, [&](auto LN) {
      constexpr int K = decltype(LN)::value;
      auto go = [&](auto NP) {
        constexpr int F = decltype(NP)::value;
        if constexpr (K * F <= 64)
          hipLaunchKernelGGL((k_amg_gs<K, F, T>), g1(ncol * K * F), dim3(256), 0, c.stream, ncol, nf, s, cx, cy, cz,
                             cnt[0], cnt[1], (long)V.N[0], (long)V.N[1], V.rp, V.ci, W.A, W.binv, b, x);
        else
          throw Error{MHX_ERR_STATE, "AMG Gauss-Seidel: node group wider than a wavefront"};
      };
      if (nfp == 1) go(std::integral_constant<int, 1>{});
      else if (nfp == 2) go(std::integral_constant<int, 2>{});
      else go(std::integral_constant<int, 4>{});
    });
  }
}

template <class T>
static void vcycle(Ctx& c, Amg& H, const T* A0, const double* cinv, const T* v, T* out) {
  const int nl = (int)H.lv.size();
  // downward: pre-smooth (zero start), residual, restrict
  for (int l = 0; l < nl - 1; ++l) {
    AmgLevel& V = *H.lv[l];
    const LvView<T> W = view<T>(H, l, A0);
    const T* b = l ? W.b : v;
    T* x = l ? W.x : out;
    if (H.smoother == kSmootherBlockJacobi) {
      bj_smooth<T>(c, H, V, W, b, x, 1);
    } else if (H.smoother == kSmootherBlockGaussSeidel) {
      hipLaunchKernelGGL(k_amg_fill0<T>, g1(V.n), dim3(256), 0, c.stream, V.n, x);
      gs_sweep<T>(c, H, V, W, b, x, true);
    } else {
      const Cheb k = cheb_coef(V.lambda);
      cheb_step<T>(c, V, W, b, x, W.t, 0.0, k.inv_theta, 1);
      cheb_step<T>(c, V, W, b, W.t, x, k.a2, k.b2, 0);
    }
    level_resid<T>(c, V, W, b, x, W.r);
    const LvView<T> Wc = view<T>(H, l + 1, A0);
    const long nc = H.lv[l + 1]->n;
    by_lanes(V.rlane, [&](auto LN) {
      constexpr int K = decltype(LN)::value;
      hipLaunchKernelGGL((k_amg_spmv<K, T>), g1(nc * K), dim3(256), 0, c.stream, nc, V.rrp.p, V.rci.p, W.R, W.r,
                         (const T*)nullptr, Wc.b);
    });
  }
  // coarsest
  {
    AmgLevel& Z = *H.lv[nl - 1];
    const LvView<T> W = view<T>(H, nl - 1, A0);
    const T* b = nl > 1 ? W.b : v;
    T* x = nl > 1 ? W.x : out;
    hipLaunchKernelGGL(k_amg_gemv<T>, g1(Z.n * 64), dim3(256), 0, c.stream, Z.n, cinv, b, x);
  }
  // upward: prolong-add, post-smooth
  for (int l = nl - 2; l >= 0; --l) {
    AmgLevel& V = *H.lv[l];
    const LvView<T> W = view<T>(H, l, A0);
    const T* b = l ? W.b : v;
    T* x = l ? W.x : out;
    const LvView<T> Wc = view<T>(H, l + 1, A0);
    by_lanes(V.plane, [&](auto LN) {
      constexpr int K = decltype(LN)::value;
      hipLaunchKernelGGL((k_amg_spmv<K, T>), g1(V.n * K), dim3(256), 0, c.stream, V.n, V.prp.p, V.pci.p, W.P, Wc.x,
                         x, H.smoother == kSmootherBlockJacobi ? bj_start<T>(H, V, W, x, 0) : x);
    });
    if (H.smoother == kSmootherBlockJacobi) {
      bj_smooth<T>(c, H, V, W, b, x, 0);
    } else if (H.smoother == kSmootherBlockGaussSeidel) {
      gs_sweep<T>(c, H, V, W, b, x, false);
    } else {
      const Cheb k = cheb_coef(V.lambda);
      cheb_step<T>(c, V, W, b, x, W.t, 0.0, k.inv_theta, 0);
      cheb_step<T>(c, V, W, b, W.t, x, k.a2, k.b2, 0);
    }
  }
  MHX_HIP(hipGetLastError());
}

void amg_apply(Ctx& c, const double* A, const double* v, double* out) {
  MHX_REQUIRE(c.amg && !c.amg->lv.empty() && !c.amg->fp32, MHX_ERR_STATE, "AMG: no FP64 hierarchy");
  ScopedPhase ph(c.prof, "MueLu::Hierarchy::Iterate", c.stream);
  vcycle<double>(c, *c.amg, A, c.amg->cinv.p, v, out);
}
void amg_apply(Ctx& c, const float* A, const float* v, float* out) {
  MHX_REQUIRE(c.amg && !c.amg->lv.empty() && c.amg->fp32, MHX_ERR_STATE, "AMG: no FP32 hierarchy");
  ScopedPhase ph(c.prof, "MueLu::Hierarchy::Iterate", c.stream);
  vcycle<float>(c, *c.amg, A, c.amg->cinv.p, v, out);
}

int amg_levels(const Ctx& c) { return c.amg ? (int)c.amg->lv.size() : 0; }

// sizes (rows, cols, nnz) of one operator of the hierarchy; copies it to the
// host arrays that are not null.  which: 0 = A_l, 1 = P_l, 2 = R_l, 3 = the
// coarsest dense inverse (row-major, rows = cols = its size).
void amg_download(Ctx& c, int level, int which, int64_t* rows, int64_t* cols, int64_t* nnz, int32_t* rp, int32_t* ci,
                  double* vals) {
  MHX_REQUIRE(c.amg && level >= 0 && level < (int)c.amg->lv.size(), MHX_ERR_ARG, "AMG: no such level");
  Amg& H = *c.amg;
  AmgLevel& V = *H.lv[level];
  const bool last = level == (int)H.lv.size() - 1;
  const int32_t *prp = nullptr, *pci = nullptr;
  const double* pv = nullptr;
  long nr = 0, nc = 0, nz = 0;
  if (which == 0) {
    prp = V.rp; pci = V.ci; pv = level ? V.A.p : H.A0;
    nr = nc = V.n;
  } else if (which == 1 || which == 2) {
    MHX_REQUIRE(!last, MHX_ERR_ARG, "AMG: the coarsest level has no transfer operators");
    const long m = H.lv[level + 1]->n;
    if (which == 1) { prp = V.prp.p; pci = V.pci.p; pv = V.P.p; nr = V.n; nc = m; }
    else { prp = V.rrp.p; pci = V.rci.p; pv = V.R.p; nr = m; nc = V.n; }
  } else if (which == 3) {
    MHX_REQUIRE(last, MHX_ERR_ARG, "AMG: the dense inverse belongs to the coarsest level");
    nr = nc = V.n;
    nz = V.n * V.n;
  } else {
    throw Error{MHX_ERR_ARG, "AMG: unknown operator"};
  }
  if (which != 3) {
    int32_t last_rp = 0;
    MHX_HIP(hipMemcpyAsync(&last_rp, prp + nr, sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
    MHX_HIP(hipStreamSynchronize(c.stream));
    nz = last_rp;
    if (rp) MHX_HIP(hipMemcpyAsync(rp, prp, (nr + 1) * sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
    if (ci) MHX_HIP(hipMemcpyAsync(ci, pci, nz * sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
    if (vals) MHX_HIP(hipMemcpyAsync(vals, pv, nz * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  } else if (vals) {
    MHX_HIP(hipMemcpyAsync(vals, H.cinv.p, nz * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  }
  MHX_HIP(hipStreamSynchronize(c.stream));
  if (rows) *rows = nr;
  if (cols) *cols = nc;
  if (nnz) *nnz = nz;
}

double amg_lambda(const Ctx& c, int level) {
  return (c.amg && level >= 0 && level < (int)c.amg->lv.size()) ? c.amg->lv[level]->lambda : 0.0;
}

}  // namespace mhx
