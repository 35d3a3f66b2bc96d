// Sweeps over the upper triangle of Hermitian matrices (or over full ones), shared by the
// DIA integrators (gfx950). A view V has n (row stride), n_true, herm, spread (how far a
// stencil read may cross the diagonal), nb = ceil(n_true / 64) and total (tiles per
// instance).
#pragma once

#include <hip/hip_runtime.h>

namespace dqh {
namespace tri {

// Tiles of NE rows per wave, 4 waves, 64 columns. Hermitian: the tiles of block rows
// b <= c, with block rows pair and nb - 1 - pair folded into one run of nb + 1 tiles.
// Consecutive workgroups go round-robin over the 8 XCDs; the remap gives every XCD a
// contiguous run, so that the rows neighbouring tiles share stay in one L2. False past
// the end; id numbers the tiles of an instance. round > 0: the tiles past the grid, for grids
// sized for the triangle that may have to cover the full matrix.
__host__ __device__ inline int tiles_of(int nb, bool herm, int ne) { return (herm ? (nb + 1) / 2 * (nb + 1) : nb * nb) * (16 / ne); }
template <int NE, class V>
__device__ __forceinline__ bool tile(const V &v, int &id, int &i0, int &j, int round = 0) {
  constexpr int kSub = 16 / NE;
  const int chunk = (v.total + 7) >> 3;
  const int b = (int)blockIdx.x + round * (int)gridDim.x;
  id = (b & 7) * chunk + (b >> 3);
  if (id >= v.total || (b >> 3) >= chunk) return false;
  const int t = id / kSub, sub = id - t * kSub, nb = v.nb;
  int br, bc;
  if (v.herm) {
    const int pair = t / (nb + 1), c = t - pair * (nb + 1);
    if (c < nb - pair) {
      br = pair;
      bc = pair + c;
    } else {
      br = nb - 1 - pair;
      bc = c - 1;  // br + (c - (nb - pair))
      if (br == pair) br = -1;  // the middle row of an odd nb has no partner
    }
  } else {
    br = t / nb;
    bc = t - br * nb;
  }
  i0 = br < 0 ? -64 : br * 64 + sub * 4 * NE + NE * __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  j = bc * 64 + ((int)threadIdx.x & 63);
  return true;
}
// row m of the tile holds an element that this thread owns
template <class V>
__device__ __forceinline__ bool owned(const V &v, int i, int j) {
  return i >= 0 && i < (int)v.n_true && j < (int)v.n_true && (!v.herm || j >= i);
}
// store x at (i, j), and its conjugate below the diagonal where stencil reads reach
template <class V, class T2>
__device__ __forceinline__ void put(const V &v, T2 *b, int i, int j, T2 x) {
  b[(size_t)i * v.n + j] = x;
  if (v.herm && j > i && j - i <= v.spread) {
    x.y = -x.y;
    b[(size_t)j * v.n + i] = x;
  }
}

// y equals its conjugate transpose at (i, j) up to rounding: 1e-12 of the element and
// 1e-13 of sqrt(|y_ii y_jj|), which bounds the element of a density matrix (what a product
// such as psi psi^dag leaves; FP32 results resolve 6e-8)
__device__ __forceinline__ bool hermitian_at(const double2 *y, int64_t n, int i, int j) {
  const double2 u = y[(int64_t)i * n + j], l = y[(int64_t)j * n + i];
  const double2 a = y[(int64_t)i * n + i], b = y[(int64_t)j * n + j];
  const double tol = 1e-12 * (fabs(u.x) + fabs(u.y)) + 1e-13 * sqrt(fabs(a.x)) * sqrt(fabs(b.x));
  return fabs(u.x - l.x) <= tol && fabs(u.y + l.y) <= tol;
}

}  // namespace tri
}  // namespace dqh
