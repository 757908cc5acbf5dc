// lattice_product.hpp — products with a matrix in the context's lattice
// pattern for one unknown per node and order 2 (Q2 quads and hexes), CDNA4
// (gfx950): y = A x and the fused forms of the Krylov and multigrid loops.
//
// What bounds it.  The values are read once (8 nnz bytes) and everything else
// is small, so the floor is the HBM read rate (6.1 TB/s for a plain read).
// The general product (a lane group per row that finds each entry's column
// and gathers x through the vector cache) spends its time on column arithmetic
// and on the gathers.  Q2 FP64, general -> here: 64^3 343 -> 232 us (3.1 ->
// 4.7 TB/s), 48^3 131 -> 101 us; the Chebyshev step at 48^3 146 -> 106 us, the
// residual 134 -> 106 us.
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

// runs of the rows of one line: EY x EZ column lines, vo the lane's first
// entry relative to the line, len its row's columns per run
template <int EY, int EZ, int LY, int W, bool COLIDX, class TA, class TX, class ACC>
__device__ __forceinline__ ACC q2_line_sum(const TA* __restrict__ A, const int32_t* __restrict__ ci,
                                           const TX* __restrict__ x, const ACC* s_x, unsigned vo, unsigned len) {
  constexpr int NR = EY * EZ;
  ACC acc = 0;
  TA a[NR];
  // (a line's entries are within 4 GB: one uniform base, 32-bit lane offsets)
  const unsigned b0 = vo * (unsigned)sizeof(TA), bl = len * (unsigned)sizeof(TA);
#pragma unroll
  for (int t = 0; t < NR; ++t) a[t] = *(const TA*)((const char*)A + (size_t)(b0 + t * bl));
#pragma unroll
  for (int t = 0; t < NR; ++t) {
    ACC xv;
    if constexpr (COLIDX) xv = (ACC)x[ci[vo + t * len]];
    else xv = s_x[((t / EY) * LY + t % EY) * W];
    acc = fma((ACC)a[t], xv, acc);
  }
  return acc;
}

// epi(row, (A x)_row, epi.load(row)) for every row; the row's operands are
// loaded ahead of its sums.  COLIDX: columns from the index stream instead of
// the tile (the same sums in the same order).
template <int DIM, bool COLIDX, class TA, class TX, class ACC, class Epi>
__global__ __launch_bounds__(256) void k_q2_product(BoxMesh m, unsigned nbx, unsigned nby,
                                                    const int32_t* __restrict__ colidx, const TA* __restrict__ A,
                                                    const TX* __restrict__ x, Epi epi) {
  using T = Q2Tile<DIM>;
  constexpr int LY = T::LY, LZ = T::LZ, W = T::W;
  __shared__ ACC s_x[COLIDX ? 1 : LZ * LY * W];
  const unsigned bq = blockIdx.x / nbx;
  const int e0 = (int)(blockIdx.x - bq * nbx) * T::EX;
  const int ey0 = (int)(bq % nby) * T::TY, ez = DIM == 3 ? (int)(bq / nby) : 0;
  const int n0 = m.nel[0], n1 = m.nel[1], n2 = m.nel[2];
  const int N0 = m.nn[0], N1 = m.nn[1], N2 = m.nn[2];
  if constexpr (!COLIDX) {
    const int X0 = 2 * e0 - 2, Y0 = 2 * ey0 - 2, Z0 = DIM == 3 ? 2 * ez - 2 : 0;
    for (int k = threadIdx.x; k < LZ * LY * W; k += 256) {
      const int X = X0 + k % W, Y = Y0 + (k / W) % LY, Z = Z0 + k / (W * LY);
      const bool in = X >= 0 && X < N0 && Y >= 0 && Y < N1 && Z >= 0 && Z < N2;
      s_x[k] = in ? (ACC)x[((long)Z * N1 + Y) * N0 + X] : (ACC)0;
    }
    __syncthreads();
  }
  // the wavefront's row line (Y, Z) = (2 ey + jy, 2 ez + jz)
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int jy = wv & 1, jz = DIM == 3 ? wv >> 1 : 0, by = DIM == 3 ? 0 : wv >> 1;
  const int ey = ey0 + by;
  const int Y = 2 * ey + jy, Z = DIM == 3 ? 2 * ez + jz : 0;
  if (Y >= N1 || Z >= N2) return;
  const bool y5 = !jy && ey > 0 && ey < n1, z5 = DIM == 3 && !jz && ez > 0 && ez < n2;
  const int EY = y5 ? 5 : 3, EZ = DIM == 3 ? (z5 ? 5 : 3) : 1;
  // first column line relative to the tile
  const int yo = 2 * by + ((y5 || (!jy && ey == n1)) ? 0 : 2);
  const int zo = DIM == 3 ? ((z5 || (!jz && ez == n2)) ? 0 : 2) : 0;
  const unsigned T0 = 8u * n0 + 1, T1 = 8u * n1 + 1;
  const unsigned line = (DIM == 3 ? (unsigned)q2_prefix(Z) * T1 * T0 : 0u) + (unsigned)EZ * (unsigned)q2_prefix(Y) * T0;
  const TA* Al = A + line;
  const int32_t* cl = COLIDX ? colidx + line : nullptr;
  const int eg = lane >> 3, l = lane & 7;
  const int r = l >= 5;          // 0: vertex row 2e, 1: row 2e + 1
  const int dx = r ? l - 3 : l;  // column 2e - 2 + dx
  const int e = e0 + eg, X = 2 * e + r;
  // lane 3 ends the vertex row, lane 4 the other
  const int Xo = 2 * e + (l == 4);
  const long row = ((long)Z * N1 + Y) * N0 + Xo;
  const bool owner = (l == 3 || l == 4) && Xo < N0;
  typename Epi::Pre pre{};
  if (owner) pre = epi.load(row);
  const int dlo = (r || e == 0) ? 2 : 0;
  const unsigned len = (r || e == 0 || e == n0) ? 3u : 5u;
  ACC acc = 0;
  if (X < N0 && dx >= dlo && dx < dlo + (int)len) {
    const unsigned vo = (unsigned)(EY * EZ) * (unsigned)q2_prefix(X) + (unsigned)(dx - dlo);
    const ACC* sx = s_x + (COLIDX ? 0 : (zo * LY + yo) * W + 2 * eg + dx);
    if constexpr (DIM == 3) {
      if (y5) {
        if (z5) acc = q2_line_sum<5, 5, LY, W, COLIDX, TA, TX, ACC>(Al, cl, x, sx, vo, len);
        else acc = q2_line_sum<5, 3, LY, W, COLIDX, TA, TX, ACC>(Al, cl, x, sx, vo, len);
      } else {
        if (z5) acc = q2_line_sum<3, 5, LY, W, COLIDX, TA, TX, ACC>(Al, cl, x, sx, vo, len);
        else acc = q2_line_sum<3, 3, LY, W, COLIDX, TA, TX, ACC>(Al, cl, x, sx, vo, len);
      }
    } else {
      if (y5) acc = q2_line_sum<5, 1, LY, W, COLIDX, TA, TX, ACC>(Al, cl, x, sx, vo, len);
      else acc = q2_line_sum<3, 1, LY, W, COLIDX, TA, TX, ACC>(Al, cl, x, sx, vo, len);
    }
  }
  // lanes 0..4 sum to row 2e (in lane 3), lanes 5..7 to row 2e + 1 (in lane 4)
  const ACC fifth = dpp_move<kDppHalfMirror>(acc);  // lane 3: lane 4's part
  ACC s = l == 4 ? (ACC)0 : acc;
  s += dpp_move<kDppXor1>(s);
  s += dpp_move<kDppXor2>(s);
  if (owner) epi(row, l == 3 ? s + fifth : s, pre);
}

// The order-2 scalar lattice takes this product unless the caller chose
// another number of lanes per row than the context's default.
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

}  // namespace mhx
