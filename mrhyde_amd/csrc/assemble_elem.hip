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
// The gather is bound by load latency on small meshes and by the traffic of
// the element matrices on large ones.  Its 2^dim loads per entry are issued
// together whether or not the entry has that many contributions: 64^2 Q1
// 10.3 us with a loop over the contributions, 9.8 us so; Q2 hexes 16^3 55.6
// and 51.7 us.

#include "thermal_kernel.hpp"

namespace mhx {

// LANES lanes walk the entries of one row; the last one sums its residual.
template <int DIM, int P, int LANES>
__global__ __launch_bounds__(256) void k_gather_rows(AsmArgs a) {
  constexpr int P1 = P + 1, NB = ipow(P1, DIM);
  const unsigned row = (blockIdx.x * 256u + threadIdx.x) / LANES;
  const int l = threadIdx.x % LANES;
  if (row >= (unsigned)a.m.ndof) return;
  int c[3];
  {
    const unsigned yz = row / (unsigned)a.m.nn[0];
    c[0] = (int)(row - yz * (unsigned)a.m.nn[0]);
    c[2] = DIM == 3 ? (int)(yz / (unsigned)a.m.nn[1]) : 0;
    c[1] = (int)(yz - (unsigned)c[2] * (unsigned)a.m.nn[1]);
  }
  // the row's elements per axis (elo .. ehi) and columns (lo, len)
  int elo[3] = {0, 0, 0}, ehi[3] = {0, 0, 0}, lo[3] = {0, 0, 0}, len[3] = {1, 1, 1};
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const int e = c[d] / P;
    elo[d] = c[d] % P == 0 && e > 0 ? e - 1 : e;
    ehi[d] = min(e, a.m.nel[d] - 1);
    lo[d] = P * elo[d];
    len[d] = P * (ehi[d] - elo[d] + 1) + 1;
  }
  const bool fixed = a.fixed[row] != 0, add = a.first_touch == 0;
  if (fixed && add) return;  // the caller's rows; the diagonal is set afterwards
  if (a.jac) {
    const int b = a.rowptr[row], n = len[0] * len[1] * len[2];
    const float iw = 1.0f / (float)len[0], iy = 1.0f / (float)len[1];
    for (int q = l; q < n; q += LANES) {
      // (float reciprocals are exact for these extents, see LatRow)
      const int run = (int)(((float)q + 0.5f) * iw);
      const int rz = DIM == 3 ? (int)(((float)run + 0.5f) * iy) : 0;
      const int j[3] = {lo[0] + q - run * len[0], lo[1] + run - rz * len[1], lo[2] + rz};
      double* o = a.jac + b + q;
      double v = add ? *o : 0.0;
      if (fixed) {
        v = j[0] == c[0] && j[1] == c[1] && (DIM == 2 || j[2] == c[2]) ? 1.0 : 0.0;
      } else {
        // per axis the offset of the first element that holds both nodes (the
        // even one of two) and the step to the second: 0 where there is none.
        // All 2^dim loads are issued together (those without an element repeat
        // an address), then summed in the order of the element colours, so the
        // sums are those of element colouring to the bit.
        long off[3], step[3];
#pragma unroll
        for (int d = 0, es = 1, ns = 1; d < 3; ++d, ns *= P1) {
          const bool two = elo[d] != ehi[d] && j[d] == c[d];
          const int hi = two ? elo[d] & 1 : (int)(j[d] > c[d]);  // start at the high element
          const int f = hi ? ehi[d] : elo[d];
          off[d] = (long)es * f * (NB * NB) + ns * ((c[d] - P * f) * NB + (j[d] - P * f));
          step[d] = two ? (long)es * (NB * NB) - ns * (P * NB + P) : 0;
          if (hi) step[d] = -step[d];
          if (DIM == 2 && d == 2) off[d] = step[d] = 0;
          es *= a.m.nel[d];
        }
        const double* E = a.escr + (off[0] + off[1] + off[2]);
        double w[1 << DIM];
#pragma unroll
        for (int k = 0; k < 1 << DIM; ++k)
          w[k] = E[(k & 1 ? step[0] : 0) + (k & 2 ? step[1] : 0) + (k & 4 ? step[2] : 0)];
#pragma unroll
        for (int k = 0; k < 1 << DIM; ++k)
          if (!((k & 1 && !step[0]) || (k & 2 && !step[1]) || (k & 4 && !step[2]))) v += w[k];
      }
      *o = v;
    }
  }
  if (a.res && l == LANES - 1) {
    double v = add ? a.res[row] : 0.0;
    if (!fixed)
      for (int k = 0; k < 1 << DIM; ++k) {
        // colour order: the even element of two first
        int ee[3];
        bool in = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int kd = (k >> d) & 1;
          in = in && !(kd && elo[d] == ehi[d]);
          ee[d] = kd ^ (elo[d] != ehi[d] ? elo[d] & 1 : 0) ? ehi[d] : elo[d];
        }
        if (!in) continue;
        const int ex = ee[0], ey = ee[1], ez = ee[2];
        const long e = ex + (long)a.m.nel[0] * (ey + (long)a.m.nel[1] * ez);
        int il = (c[0] - P * ex) + P1 * (c[1] - P * ey);
        if constexpr (DIM == 3) il += P1 * P1 * (c[2] - P * ez);
        v -= a.rscr[e * NB + il];
      }
    a.res[row] = v;
  }
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
  // lanes per row: an interior row of the order has 9 (2-D Q1) to 27 or more entries
  constexpr int L = ipow(P + 1, DIM) <= 9 ? 8 : 32;
  hipLaunchKernelGGL((k_gather_rows<DIM, P, L>), dim3((unsigned)((c.mesh.ndof * L + 255) / 256)), dim3(256), 0,
                     c.stream, a);
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

// Where the two launches beat the 2^dim launches of element colouring
// (us, residual + Jacobian, colouring / here):
//   2-D Q1 64^2 23.6/9.8, 256^2 31/24, 1024^2 (128 MiB) 257/240
//   3-D Q1 16^3 77/15, 32^3 81/44, 64^3 (128 MiB) 360/213
//   2-D Q2 64^2 36/14, 192^2 (23 MiB) 54/45, 256^2 (41 MiB) 68/68
//   2-D Q3 64^2 48/25, 96^2 (18 MiB) 57/46, 128^2 (32 MiB) 60/66
//   2-D Q4 64^2 (20 MiB) 77/43; Q6 32^2 (19 MiB) 260/71
//   3-D Q2, three points per axis: 8^3 168/24, 16^3 169/52, 24^3 (77 MiB)
//     176/121, 32^3 (182 MiB) 244/272, 40^3 (356 MiB) 473/592
// Past these sizes the round trip of the element matrices costs more than the
// colours' launches.  The bound also keeps the scratch memory small; it is
// allocated with the context, so no assembly allocates.
int64_t element_store_doubles(const mhx_problem_desc& d) {
  if (d.physics != MHX_PHYS_THERMAL || d.n_functions > 0) return 0;
  // boxes at three points per axis: the row-owned kernel (assemble_q2box.hip)
  if (d.dim == 3 && d.order == 2 && d.quadrature / 2 + 1 == 3 && d.perturb == 0.0) return 0;
  const double cap = (d.order == 1 ? 128.0 : d.dim == 3 ? 80.0 : 24.0) * (1 << 20);
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

void launch_element_store(Ctx& c, AsmArgs& a, bool jac) {
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
