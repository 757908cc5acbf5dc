// lattice_product.hpp — products with a matrix in the context's lattice
// pattern for one unknown per node and order 2 (Q2 quads and hexes), CDNA4
// (gfx950): y = A x and the fused forms of the Krylov and multigrid loops.
//
// What bounds it.  The values are read once (8 nnz bytes) and everything else
// is small, so the floor is the HBM read rate (6.1 TB/s for a plain read).
// The general product (a lane group per row that finds each entry's column
// and gathers x through the vector cache) spends its time on column arithmetic
// and on the gathers.  Q2 FP64, general -> here: 64^3 343 -> 229 us (3.1 ->
// 4.7 TB/s), 48^3 131 -> 98 us; the Chebyshev step at 48^3 146 -> 100 us, the
// residual 134 -> 99 us.
//
// Layout.  The rows of one lattice line (Y, Z) are contiguous, and the line's
// rows 2e (vertex, 5 columns a run) and 2e + 1 (interior, 3 columns a run)
// have 8 columns between them: a group of eight lanes takes both rows, lane
// l < 5 column l of the vertex row's run, lane l >= 5 column l - 5 of the
// other's.  Run t of both rows is the same column line (y', z'), so a lane
// walks its row with a constant stride, and the x value is at a fixed
// lane offset plus a run offset that is the same for the whole wavefront: no
// column arithmetic.  x comes from a tile of column lines in LDS (about 8
// loads per row instead of one per entry).  Lines on the box boundary have 3 runs along that axis.
// The row sums meet through DPP moves inside the eight lanes.
#pragma once

#include <type_traits>

#include "mhx_internal.hpp"

namespace mhx {

// first entry (per unit run) of row X of an axis of Q2 rows, and its columns:
// 3, 3, 5, 3, 5, 3, ..., 3
__device__ __forceinline__ int q2_prefix(int X) {
  const int e = X >> 1;
  return (X & 1) ? (e == 0 ? 3 : 8 * e + 3) : (e == 0 ? 0 : 8 * e - 2);
}

// v moved by a DPP control inside the wavefront
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
constexpr int kDppXor1 = 0xB1;        // quad_perm [1, 0, 3, 2]
constexpr int kDppXor2 = 0x4E;        // quad_perm [2, 3, 0, 1]
constexpr int kDppHalfMirror = 0x141;  // lane i of each 8 from lane 7 - i

// Tile of a workgroup of four wavefronts: 8 element blocks along x (element
// block e of an axis: rows 2e and 2e + 1), and one (y, z) block in 3-D, one of
// its four row lines per wavefront; two y blocks in 2-D.  A larger tile (16 x
// 2 x 2 blocks, four lines per wavefront in turn) reads x half as often but
// measured 110 against 100 us at 48^3 and the same at 64^3.
template <int DIM>
struct Q2Tile {
  static constexpr int EX = 8, TY = DIM == 3 ? 1 : 2;
  static constexpr int LY = 2 * TY + 3, LZ = DIM == 3 ? 5 : 1;  // column lines
  static constexpr int W = 2 * EX + 4;                          // columns of a line
};

// epi(row, (A x)_row, epi.load(row)) for every row.  Order of the loads: the x
// tile, the row ends' operands, then the wavefront's matrix values, all in
// flight together; the tile goes to LDS when it arrives (the values behind it
// still under way), so a workgroup waits for memory once.  COLIDX: columns from
// the index stream instead of the tile (the same sums in the same order).
template <int DIM, bool COLIDX, class TA, class TX, class ACC, class Epi>
__global__ __launch_bounds__(256) void k_q2_product(BoxMesh m, unsigned nbx, unsigned nby,
                                                    const int32_t* __restrict__ colidx, const TA* __restrict__ A,
                                                    const TX* __restrict__ x, Epi epi) {
  using T = Q2Tile<DIM>;
  constexpr int LY = T::LY, LZ = T::LZ, W = T::W, NT = LZ * LY * W, NTL = (NT + 255) / 256;
  __shared__ ACC s_x[COLIDX ? 1 : NT];
  const unsigned bq = blockIdx.x / nbx;
  const int e0 = (int)(blockIdx.x - bq * nbx) * T::EX;
  const int ey0 = (int)(bq % nby) * T::TY, ez = DIM == 3 ? (int)(bq / nby) : 0;
  const int n0 = m.nel[0], n1 = m.nel[1], n2 = m.nel[2];
  const int N0 = m.nn[0], N1 = m.nn[1], N2 = m.nn[2];
  // (straight-line code from here to the sums: loads with clamped addresses and
  // selects in place of branches, so each wait counts the loads behind it)
  TX xt[NTL];
  bool xin[NTL];
  if constexpr (!COLIDX) {
    const int X0 = 2 * e0 - 2, Y0 = 2 * ey0 - 2, Z0 = DIM == 3 ? 2 * ez - 2 : 0;
#pragma unroll
    for (int i = 0; i < NTL; ++i) {
      const int k = threadIdx.x + 256 * i;
      const int X = X0 + k % W, Y = Y0 + (k / W) % LY, Z = Z0 + k / (W * LY);
      const bool in = k < NT && X >= 0 && X < N0 && Y >= 0 && Y < N1 && Z >= 0 && Z < N2;
      unsigned at = in ? (unsigned)(((long)Z * N1 + Y) * N0 + X) : 0u;
      // (opaque, so that load and select are not folded back into a branch)
      __asm__ volatile("" : "+v"(at));
      xt[i] = x[at];
      xin[i] = in;
    }
  }
  // the tile's values to LDS, and an LDS-only barrier: the matrix values loaded
  // before it stay in flight
  auto fill_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NTL; ++i)
      if (256 * i + 256 <= NT || threadIdx.x + 256 * i < NT) s_x[threadIdx.x + 256 * i] = xin[i] ? (ACC)xt[i] : (ACC)0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  // the wavefront's row line (Y, Z) = (2 ey + jy, 2 ez + jz)
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int jy = wv & 1, jz = DIM == 3 ? wv >> 1 : 0, by = DIM == 3 ? 0 : wv >> 1;
  const int ey = ey0 + by;
  const int Y = 2 * ey + jy, Z = DIM == 3 ? 2 * ez + jz : 0;
  const bool on = Y < N1 && Z < N2;
  const bool y5 = !jy && ey > 0 && ey < n1, z5 = DIM == 3 && !jz && ez > 0 && ez < n2;
  const int EY = y5 ? 5 : 3, EZ = DIM == 3 ? (z5 ? 5 : 3) : 1;
  // first column line relative to the tile
  const int yo = 2 * by + ((y5 || (!jy && ey == n1)) ? 0 : 2);
  const int zo = DIM == 3 ? ((z5 || (!jz && ez == n2)) ? 0 : 2) : 0;
  const unsigned T0 = 8u * n0 + 1, T1 = 8u * n1 + 1;
  const unsigned line = (DIM == 3 ? (unsigned)q2_prefix(Z) * T1 * T0 : 0u) + (unsigned)EZ * (unsigned)q2_prefix(Y) * T0;
  const TA* Al = A + line;
  const int eg = lane >> 3, l = lane & 7;
  const int r = l >= 5;          // 0: vertex row 2e, 1: row 2e + 1
  const int dx = r ? l - 3 : l;  // column 2e - 2 + dx
  const int e = e0 + eg, X = 2 * e + r;
  // lane 3 ends the vertex row, lane 4 the other
  const int Xo = 2 * e + (l == 4);
  const long row = ((long)Z * N1 + Y) * N0 + Xo;
  const bool owner = on && (l == 3 || l == 4) && Xo < N0;
  const typename Epi::Pre pre = epi.load(owner ? row : 0);
  const int dlo = (r || e == 0) ? 2 : 0;
  const unsigned len = (r || e == 0 || e == n0) ? 3u : 5u;
  const bool act = on && X < N0 && dx >= dlo && dx < dlo + (int)len;
  // inactive lanes repeat the line's first entries
  const unsigned vo = act ? (unsigned)(EY * EZ) * (unsigned)q2_prefix(X) + (unsigned)(dx - dlo) : 0u;
  // (a line's entries are within 4 GB: one uniform base, 32-bit lane offsets)
  const unsigned b0 = vo * (unsigned)sizeof(TA), bl = (act ? len : 3u) * (unsigned)sizeof(TA);
  const ACC* sx = s_x + (COLIDX ? 0 : (zo * LY + yo) * W + 2 * eg + dx);
  // values, tile to LDS, barrier, sums: the wavefront's 5 or 3 column lines per axis
  auto sum = [&](auto EYc, auto EZc) __attribute__((always_inline)) {
    constexpr int CY = decltype(EYc)::value, CZ = decltype(EZc)::value;
    TA a[CY * CZ];
#pragma unroll
    for (int t = 0; t < CY * CZ; ++t) a[t] = *(const TA*)((const char*)Al + (size_t)(b0 + t * bl));
    ACC acc = 0;
    if constexpr (COLIDX) {
      const int32_t* cl = colidx + line;
#pragma unroll
      for (int t = 0; t < CY * CZ; ++t) acc = fma((ACC)a[t], (ACC)x[cl[vo + t * (act ? len : 3u)]], acc);
    } else {
      fill_tile();
#pragma unroll
      for (int t = 0; t < CY * CZ; ++t) acc = fma((ACC)a[t], sx[((t / CY) * LY + t % CY) * W], acc);
    }
    return act ? acc : (ACC)0;
  };
  using C1 = std::integral_constant<int, 1>;
  using C3 = std::integral_constant<int, 3>;
  using C5 = std::integral_constant<int, 5>;
  // (every branch passes the one barrier of fill_tile; the branches are uniform
  // in the wavefront)
  ACC acc;
  if (!on) {
    if constexpr (!COLIDX) fill_tile();
    return;
  }
  if constexpr (DIM == 3) {
    if (y5) acc = z5 ? sum(C5{}, C5{}) : sum(C5{}, C3{});
    else acc = z5 ? sum(C3{}, C5{}) : sum(C3{}, C3{});
  } else {
    acc = y5 ? sum(C5{}, C1{}) : sum(C3{}, C1{});
  }
  // lanes 0..4 sum to row 2e (in lane 3), lanes 5..7 to row 2e + 1 (in lane 4)
  const ACC fifth = dpp_move<kDppHalfMirror>(acc);  // lane 3: lane 4's part
  ACC s = l == 4 ? (ACC)0 : acc;
  s += dpp_move<kDppXor1>(s);
  s += dpp_move<kDppXor2>(s);
  if (owner) epi(row, l == 3 ? s + fifth : s, pre);
}

// The order-2 scalar lattice takes this product unless the caller chose
// another number of lanes per row than the context's default.  3-D: see above.
// 2-D, CG + Jacobi us an iteration, general product / this one: 256^2 28.8/25.7,
// 400^2 44.9/38.4, 1000^2 265/198; GMRES the same order (1000^2 785/713); below
// 150^2 the launches are all there is, equal.
inline bool q2_product_applies(const Ctx& c) {
  return c.mesh.p == 2 && c.mesh.nf == 1 && c.spmv_lanes == c.spmv_lanes_default;
}

// epi over the context's rows; ACC: type of the sums
template <class ACC, class TA, class TX, class Epi>
void q2_product(Ctx& c, const TA* A, const TX* x, const Epi& epi) {
  const BoxMesh& m = c.mesh;
  auto go = [&](auto D) {
    constexpr int DIM = decltype(D)::value;
    using T = Q2Tile<DIM>;
    const unsigned nbx = (m.nel[0] + T::EX) / T::EX, nby = (m.nel[1] + T::TY) / T::TY, nbz = DIM == 3 ? m.nel[2] + 1 : 1;
    const dim3 grid(nbx * nby * nbz);
    if (c.lattice_cols)
      hipLaunchKernelGGL((k_q2_product<DIM, false, TA, TX, ACC, Epi>), grid, dim3(256), 0, c.stream, m, nbx, nby,
                         c.colidx.p, A, x, epi);
    else
      hipLaunchKernelGGL((k_q2_product<DIM, true, TA, TX, ACC, Epi>), grid, dim3(256), 0, c.stream, m, nbx, nby,
                         c.colidx.p, A, x, epi);
    MHX_HIP(hipGetLastError());
  };
  if (m.dim == 3) go(std::integral_constant<int, 3>{});
  else go(std::integral_constant<int, 2>{});
}

// ---------------------------------------------------------------------------
// Order-1 hexahedral lattices with four unknowns per node (3-D Navier-Stokes,
// and every coarse level of its multigrid hierarchy: the same 27-node boxes).
//
// Sixteen lanes take a node: lane 4 f + d the row of field f and the column
// node X - 1 + d of each of the nine (y, z) lines, i.e. four consecutive values
// and one node's four unknowns per line, both 16- or 32-byte loads; d = 3 idles
// through the sums.  The four lanes of a row meet by DPP, and the node's four
// row sums sit in one group, so the nodal block-Jacobi update follows in the
// same launch (one lane per entry of the 4 x 4 inverse).  Entry by entry with
// the column found for each, a sweep of the 32^3 FP32 cavity took 15.0 us (the
// residual 11.4 and a launch of 3.6 for the update, mean over the two smoothed
// levels); now 9.1 us.
// ---------------------------------------------------------------------------
struct NodeLattice {
  int N[3];
};

template <class T>
struct alignas(sizeof(T)) Quad {
  T v[4];
};

// end(node, f, d, row, sum): called by the sixteen lanes of every node, sum the
// row's on all four lanes of its quad.  COLIDX: columns from the index stream
// (the same sums in the same order).
template <bool COLIDX, class T, class End>
__global__ __launch_bounds__(256) void k_node4_product(NodeLattice L, long nnode, const int32_t* __restrict__ rp,
                                                       const int32_t* __restrict__ colidx, const T* __restrict__ A,
                                                       const T* __restrict__ x, End end) {
  const unsigned gid = blockIdx.x * 256u + threadIdx.x;
  const unsigned nd = gid >> 4;
  const bool act = nd < (unsigned)nnode;
  const unsigned node = act ? nd : 0u;
  const int f = (threadIdx.x >> 2) & 3, d = threadIdx.x & 3;
  const int N0 = L.N[0], N1 = L.N[1], N2 = L.N[2];
  const unsigned yz = node / (unsigned)N0;
  const int X = (int)(node - yz * (unsigned)N0);
  const int Z = (int)(yz / (unsigned)N1), Y = (int)(yz - (unsigned)Z * (unsigned)N1);
  const unsigned row = 4 * node + f;
  const typename End::Pre pre = end.load(node, f, d, row);
  const unsigned b = (unsigned)rp[row];
  const int dx = d < 3 ? d : 2;
  const bool inner = X > 0 && X < N0 - 1 && Y > 0 && Y < N1 - 1 && Z > 0 && Z < N2 - 1;
  double acc = 0.0;
  auto term = [&](unsigned k, unsigned col) __attribute__((always_inline)) {
    const Quad<T> a = *(const Quad<T>*)(A + k);
    const unsigned j = COLIDX ? (unsigned)colidx[k] : col;
    const Quad<T> v = *(const Quad<T>*)(x + j);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = fma((double)a.v[i], (double)v.v[i], acc);
  };
  if (__all(inner)) {
    // all lines in flight ahead of the sums
    Quad<T> a[9], v[9];
    const unsigned k0 = b + 4 * dx, c0 = 4 * (node - (unsigned)N0 * (1 + (unsigned)N1) - 1 + dx);
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const unsigned k = k0 + 12 * t;
      a[t] = *(const Quad<T>*)(A + k);
      unsigned col;
      if constexpr (COLIDX) col = (unsigned)colidx[k];
      else col = c0 + 4 * (unsigned)N0 * (t % 3 + (unsigned)N1 * (t / 3));
      v[t] = *(const Quad<T>*)(x + col);
    }
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc = fma((double)a[t].v[i], (double)v[t].v[i], acc);
  } else {
    const int x0 = X > 0 ? X - 1 : 0, x1 = X < N0 - 1 ? X + 1 : X, y0 = Y > 0 ? Y - 1 : 0, y1 = Y < N1 - 1 ? Y + 1 : Y,
              z0 = Z > 0 ? Z - 1 : 0, z1 = Z < N2 - 1 ? Z + 1 : Z;
    const int xc = X - 1 + dx;
    const unsigned ex = x1 - x0 + 1;
    if (xc >= x0 && xc <= x1) {
      unsigned k = b + 4 * (unsigned)(xc - x0);
      for (int z = z0; z <= z1; ++z)
        for (int y = y0; y <= y1; ++y, k += 4 * ex) term(k, 4 * (((unsigned)z * N1 + y) * (unsigned)N0 + xc));
    }
  }
  if (d == 3) acc = 0.0;
  acc += dpp_move<kDppXor1>(acc);
  acc += dpp_move<kDppXor2>(acc);
  end(act, node, f, d, row, acc, pre);
}

inline bool node4_product_applies(const Ctx& c) {
  return c.mesh.p == 1 && c.mesh.nf == 4 && c.mesh.dim == 3 && c.spmv_lanes == c.spmv_lanes_default;
}

template <class T, class End>
void node4_product(Ctx& c, const int* N, const int32_t* rp, const int32_t* ci, bool colidx, const T* A, const T* x,
                   const End& end) {
  const NodeLattice L{{N[0], N[1], N[2]}};
  const long nnode = (long)N[0] * N[1] * N[2];
  const dim3 grid((unsigned)((nnode * 16 + 255) / 256));
  if (colidx)
    hipLaunchKernelGGL((k_node4_product<true, T, End>), grid, dim3(256), 0, c.stream, L, nnode, rp, ci, A, x, end);
  else
    hipLaunchKernelGGL((k_node4_product<false, T, End>), grid, dim3(256), 0, c.stream, L, nnode, rp, ci, A, x, end);
  MHX_HIP(hipGetLastError());
}

}  // namespace mhx
