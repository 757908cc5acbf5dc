// assemble_elem.hip — thermal assembly of small and general meshes in two
// launches, CDNA4 (gfx950): k_thermal writes the element matrices and residuals
// to scratch memory, and k_gather_rows sums them into the CRS rows
// (assemblyManager_scatter.hpp:164-278 turned round: each entry collects its
// at most 2^dim contributions).
//
// What it is for.  Element colouring needs 2^dim launches that depend on each
// other, each with 1/2^dim of the elements, and re-reads what earlier colours
// wrote.  On small meshes the launches' latency is all there is (64^2 Q1, four
// launches: 26.3 us); on larger ones the read-backs and the uncoalesced
// element-wise stores cost more than a round trip of the element matrices
// through the cache.  The gather writes every entry once, in CRS order, in the
// same fixed order of contributions on every run; Dirichlet rows become e_d
// (scatter.hpp:208,253; constraints.hpp:125-141) in the same pass.
//
// The gather is bound by load latency on small meshes and by its instructions
// and the traffic of the element matrices on large ones.  A row collects whole
// rows of its elements' matrices in an LDS image: every value is loaded once,
// coalesced, with one address per element.  A lane per CRS entry that fetches
// the entry's at most 2^dim values (mostly repeats, an address each) took 385 us
// at 40^3 Q2, this 216.

#include "thermal_kernel.hpp"

namespace mhx {

namespace {

// A row (node) of the lattice and the at most 2^DIM elements around it in the
// order of the element colours: per axis the even one of two first.  Offsets
// are 32-bit (the rule below bounds the scratch memory).
template <int DIM, int P>
struct RowElems {
  static constexpr int P1 = P + 1;
  int c[3], lo[3], len[3];
  int el[3][2], il[3][2], po[3][2];  // per axis and turn: element, local node, first column in the row
  bool two[3];
  __device__ __forceinline__ RowElems(const BoxMesh& m, unsigned row) {
    const unsigned yz = row / (unsigned)m.nn[0];
    c[0] = (int)(row - yz * (unsigned)m.nn[0]);
    c[2] = DIM == 3 ? (int)(yz / (unsigned)m.nn[1]) : 0;
    c[1] = (int)(yz - (unsigned)c[2] * (unsigned)m.nn[1]);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (d >= DIM) {
        el[d][0] = el[d][1] = il[d][0] = il[d][1] = po[d][0] = po[d][1] = lo[d] = 0;
        len[d] = 1;
        two[d] = false;
        continue;
      }
      const int e = c[d] / P;
      const int elo = c[d] % P == 0 && e > 0 ? e - 1 : e, ehi = min(e, m.nel[d] - 1);
      two[d] = elo != ehi;
      lo[d] = P * elo;
      len[d] = P * (ehi - elo + 1) + 1;
      el[d][0] = two[d] && (elo & 1) ? ehi : elo;
      el[d][1] = elo + ehi - el[d][0];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        il[d][t] = c[d] - P * el[d][t];
        po[d][t] = P * (el[d][t] - elo);
      }
    }
  }
  __device__ __forceinline__ bool has(int k) const {
    return !((k & 1 && !two[0]) || (k & 2 && !two[1]) || (k & 4 && !two[2]));
  }
  __device__ __forceinline__ unsigned elem(const BoxMesh& m, int k) const {
    return (unsigned)(el[0][k & 1] + m.nel[0] * (el[1][k >> 1 & 1] + m.nel[1] * el[2][k >> 2 & 1]));
  }
  __device__ __forceinline__ unsigned local(int k) const {
    return (unsigned)(il[0][k & 1] + P1 * (il[1][k >> 1 & 1] + P1 * il[2][k >> 2 & 1]));
  }
};

// the residual of row r from its elements' parts
template <int DIM, int P>
__device__ __forceinline__ void gather_residual(const AsmArgs& a, unsigned row, const RowElems<DIM, P>& r, bool fixed) {
  constexpr int NB = ipow(P + 1, DIM);
  const bool add = a.first_touch == 0;
  double w[1 << DIM], v = add ? a.res[row] : 0.0;
#pragma unroll
  for (int k = 0; k < 1 << DIM; ++k) w[k] = a.rscr[r.elem(a.m, k) * (unsigned)NB + r.local(k)];
#pragma unroll
  for (int k = 0; k < 1 << DIM; ++k) v = r.has(k) ? v - w[k] : v;
  if (!fixed) a.res[row] = v;
  else if (!add) a.res[row] = 0.0;
}

}  // namespace

// L lanes per row: lane l takes column l of each element's row, and the
// elements are added one after the other into the row's image in LDS, which
// leaves in CRS order.
template <int DIM, int P, int L>
__global__ __launch_bounds__(256) void k_gather_rows(AsmArgs a) {
  constexpr int P1 = P + 1, NB = ipow(P1, DIM), G = 256 / L, ROW = ipow(2 * P + 1, DIM);
  static_assert(NB <= L && L <= 64, "one column of an element's row per lane");
  __shared__ double s_img[G][ROW];
  const int g = threadIdx.x / L, l = threadIdx.x % L;
  const unsigned row = blockIdx.x * (unsigned)G + g;
  if (row >= (unsigned)a.m.ndof) return;
  const RowElems<DIM, P> r(a.m, row);
  const bool fixed = a.fixed[row] != 0, add = a.first_touch == 0;
  const int b = a.rowptr[row], n = r.len[0] * r.len[1] * r.len[2];
  const unsigned col = min(l, NB - 1);
  double w[1 << DIM];
#pragma unroll
  for (int k = 0; k < 1 << DIM; ++k)
    if (__any(r.has(k))) w[k] = a.escr[(r.elem(a.m, k) * (unsigned)NB + r.local(k)) * (unsigned)NB + col];
  double* img = s_img[g];
  for (int q = l; q < n; q += L) img[q] = add ? a.jac[b + q] : 0.0;
  const int j0 = l % P1, j1 = (l / P1) % P1, j2 = DIM == 3 ? l / (P1 * P1) : 0;
#pragma unroll
  for (int k = 0; k < 1 << DIM; ++k)
    if (__any(r.has(k))) {
      wave_lds_sync();
      if (r.has(k) && l < NB)
        img[j0 + r.po[0][k & 1] + r.len[0] * (j1 + r.po[1][k >> 1 & 1] + r.len[1] * (j2 + r.po[2][k >> 2 & 1]))] += w[k];
    }
  wave_lds_sync();
  if (!fixed) {
    for (int q = l; q < n; q += L) a.jac[b + q] = img[q];
  } else if (!add) {  // (accumulating, the caller sets the diagonal afterwards)
    const int dg = r.c[0] - r.lo[0] + r.len[0] * (r.c[1] - r.lo[1] + r.len[1] * (r.c[2] - r.lo[2]));
    for (int q = l; q < n; q += L) a.jac[b + q] = q == dg ? 1.0 : 0.0;
  }
  if (a.res && l == 0) gather_residual<DIM, P>(a, row, r, fixed);
}

// the residual alone: a row per lane
template <int DIM, int P>
__global__ __launch_bounds__(256) void k_gather_res(AsmArgs a) {
  const unsigned row = blockIdx.x * 256u + threadIdx.x;
  if (row >= (unsigned)a.m.ndof) return;
  gather_residual<DIM, P>(a, row, RowElems<DIM, P>(a.m, row), a.fixed[row] != 0);
}

namespace {

template <int DIM, int P, int NQ1>
void launch_store(Ctx& c, AsmArgs& a, bool jac) {
  using C = Cfg<DIM, P, NQ1>;
  a.gpb = C::GPB;
  {
    ScopedPhase ph(c.prof, jac ? "k_thermal<jacres>" : "k_thermal<res>", c.stream);
    const dim3 grid((unsigned)((c.mesh.ne + C::GPB - 1) / C::GPB)), block(C::BLOCK);
    if (jac) hipLaunchKernelGGL((k_thermal<DIM, P, NQ1, true, kElementStore>), grid, block, 0, c.stream, a);
    else hipLaunchKernelGGL((k_thermal<DIM, P, NQ1, false, kElementStore>), grid, block, 0, c.stream, a);
    MHX_HIP(hipGetLastError());
  }
  ScopedPhase ph(c.prof, "k_gather_rows", c.stream);
  const long nr = c.mesh.ndof;
  if (!jac) {
    hipLaunchKernelGGL((k_gather_res<DIM, P>), dim3((unsigned)((nr + 255) / 256)), dim3(256), 0, c.stream, a);
  } else {
    constexpr int NB = ipow(P + 1, DIM), L = NB <= 4 ? 4 : NB <= 8 ? 8 : NB <= 16 ? 16 : NB <= 32 ? 32 : 64;
    hipLaunchKernelGGL((k_gather_rows<DIM, P, L>), dim3((unsigned)((nr * L + 255) / 256)), dim3(256), 0, c.stream, a);
  }
  MHX_HIP(hipGetLastError());
}

using Launcher = void (*)(Ctx&, AsmArgs&, bool);
struct Entry {
  int dim, p, nq1;
  Launcher f;
};
const Entry kStoreTable[] = {
    {2, 1, 1, launch_store<2, 1, 1>}, {2, 1, 2, launch_store<2, 1, 2>}, {2, 1, 3, launch_store<2, 1, 3>},
    {2, 2, 2, launch_store<2, 2, 2>}, {2, 2, 3, launch_store<2, 2, 3>}, {2, 2, 4, launch_store<2, 2, 4>},
    {2, 3, 3, launch_store<2, 3, 3>}, {2, 3, 4, launch_store<2, 3, 4>}, {2, 4, 4, launch_store<2, 4, 4>},
    {2, 4, 5, launch_store<2, 4, 5>}, {2, 5, 6, launch_store<2, 5, 6>}, {2, 6, 7, launch_store<2, 6, 7>},
    {3, 1, 1, launch_store<3, 1, 1>}, {3, 1, 2, launch_store<3, 1, 2>}, {3, 1, 3, launch_store<3, 1, 3>},
    {3, 2, 2, launch_store<3, 2, 2>}, {3, 2, 3, launch_store<3, 2, 3>}, {3, 2, 4, launch_store<3, 2, 4>},
};

}  // namespace

// The two launches against the 2^dim launches of element colouring (us, residual
// + Jacobian, colouring / here):
//   2-D Q1 64^2 23.3/10.5, 256^2 31/26, 1024^2 (128 MiB) 258/208
//   2-D Q2 64^2 36/11, 192^2 55/42, 256^2 (41 MiB) 68/64, 384^2 141/123
//   2-D Q3 64^2 47/21, 128^2 60/49; Q4 64^2 77/37, 96^2 88/69; Q6 32^2 261/69
//   3-D Q1 16^3 77/12, 32^3 81/37, 64^3 (128 MiB) 360/192
//   3-D Q2, three points per axis: 8^3 168/21, 16^3 169/42, 24^3 (77 MiB)
//     176/96, 32^3 (182 MiB) 243/213, 40^3 (356 MiB) 473/429
// The gain shrinks as the round trip of the element matrices leaves the caches.
// No size measured was slower here: the line bounds the memory.  Past the
// largest size measured the scratch memory (1.35 times the Jacobian in
// 3-D Q2) is not spent.  It is allocated with the context, so no assembly
// allocates, given back when an option or a time state takes the assembly
// elsewhere, and for a solve that would otherwise run out of memory.
int64_t element_store_doubles(const mhx_problem_desc& d) {
  if (d.physics != MHX_PHYS_THERMAL || d.n_functions > 0) return 0;
  // boxes at three points per axis: the row-owned kernel (assemble_q2box.hip)
  if (d.dim == 3 && d.order == 2 && d.quadrature / 2 + 1 == 3 && d.perturb == 0.0) return 0;
  const double cap = 384.0 * (1 << 20);
  int64_t nb = 1;
  double n = 1.0;
  for (int a = 0; a < d.dim; ++a) {
    nb *= d.order + 1;
    n *= a == 0 ? d.nx : a == 1 ? d.ny : d.nz;
  }
  return n * (double)(nb * nb) * 8.0 <= cap ? (int64_t)n * nb * nb : 0;
}

int64_t element_store_bytes(const mhx_problem_desc& d) {
  const int64_t n = element_store_doubles(d);
  const int p1 = d.order + 1;
  return 8 * n + 8 * n / (d.dim == 3 ? p1 * p1 * p1 : p1 * p1);
}

bool element_store_release(Ctx& c) {
  if (!c.escr.p || c.store_captured) return false;
  (void)hipStreamSynchronize(c.stream);
  c.escr.release();
  c.rscr.release();
  return true;
}

void element_store_fit(Ctx& c) {
  const int64_t n = c.store_on && c.scatter_mode == kElementColouring && c.bdf_order == 0 && !c.xh.active
                        ? element_store_doubles(c.desc)
                        : 0;
  if (!n) {
    (void)element_store_release(c);
  } else if (!c.escr.p) {
    try {
      c.rscr.alloc((size_t)c.mesh.ne * c.nb);
      c.escr.alloc((size_t)n);
    } catch (const Error&) {  // no room: element colouring
      (void)hipGetLastError();
      c.rscr.release();
    }
  }
}

void launch_element_store(Ctx& c, AsmArgs& a, bool jac) {
  if (!c.store_captured) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c.stream, &cap) != hipSuccess) (void)hipGetLastError();
    c.store_captured = cap != hipStreamCaptureStatusNone;
  }
  a.escr = c.escr.p;
  a.rscr = c.rscr.p;
  a.blocked = 0;
  a.nsub = 1;
  for (const Entry& en : kStoreTable)
    if (en.dim == c.mesh.dim && en.p == c.mesh.p && en.nq1 == c.mesh.nq1) {
      en.f(c, a, jac);
      return;
    }
  throw Error{MHX_ERR_UNSUPPORTED, "no kernel built for this dim/order/quadrature"};
}

}  // namespace mhx
