// tile.h -- several Gauss-Seidel half sweeps of a multigrid level in one launch.
//
// A workgroup loads a box of the level (its region), does S half sweeps on it in LDS, each over one
// layer less than the one before, and stores the part whose values no missing neighbour has reached.
// The layers around that part are computed by several workgroups, to the same bits: a sweep by
// parities gives a cell one value whoever computes it.  Old and new values live in two arrays, since
// other workgroups read what this one replaces.
#pragma once
#include "stencils.h"

namespace lmfhd {

// Regions: 3-D 16 x 16 x 8 cells, 2-D 64 x 32: a pair of cells of either parity a thread, so that
// everything a cell's updates read from memory is in registers before the first of them.  (16^3 cells
// with two pairs a thread: fewer layers computed twice, but 32^3 FP32 6.7 -> 10.3 us.  16 x 8 x 8: a
// little faster where all tiles run at once, 5.6 against 6.4 us at 16^3, but that ends sooner, 32^3
// 9.8 us.)
template <int DM>
struct TileBox {
  static constexpr int RX = DM == 3 ? 16 : 64, RY = DM == 3 ? 16 : 32, RZ = DM == 3 ? 8 : 1;
  static constexpr int BS = RX * RY * RZ / 2;
  static constexpr int LX = RX + 2, LXY = LX * (RY + 2);   // LDS strides: one layer around the region
  static constexpr int LN = LXY * (DM == 3 ? RZ + 2 : 1);
  static constexpr int LO = 1 + LX + (DM == 3 ? LXY : 0);  // the region's first cell
  HD static constexpr int R(int d) { return d == 0 ? RX : (d == 1 ? RY : RZ); }
};
constexpr int TILE_MAX = 256;  // tiles of a launch: one a compute unit
// tiles of a box of n cells for S half sweeps, nt of them along each direction
template <int DM>
inline long tile_count(const int* n, int S, int* nt) {
  long c = 1;
  nt[2] = 1;
  for (int d = 0; d < DM; ++d) {
    const int e = TileBox<DM>::R(d) - 2 * (S - 1);
    nt[d] = (n[d] + e - 1) / e;
    c *= nt[d];
  }
  return c;
}

// v as an index of [0, n): its periodic image, or (walls) marked invalid
HD int tile_wrap(int v, int n, int per, bool& ok) {
  if (per) {
    while (v < 0) v += n;
    while (v >= n) v -= n;
    return v;
  }
  ok = ok && v >= 0 && v < n;
  return v < 0 ? 0 : (v >= n ? n - 1 : v);
}

template <typename T>
struct MacPair {  // a thread's cells, [c] of parity c
  T b[2][6], r[2], dg[2];
  unsigned o[2];  // index in the level's arrays
  int l[2];       // in LDS
  int m[2];       // layers to the nearest side of the region; -1: beyond a wall
};

// S half sweeps of the MAC level starting with parity C0; UP: on phi plus the coarse level's value of
// each cell's parent (the prolongation), else on phi.  From phi to out.
template <typename T, int DM, int S, int C0, int UP>
struct MacTileBlk {
  using B = TileBox<DM>;
  static constexpr int BS = B::BS, M = S - 1;  // M: layers not stored
  Geo g, gc;
  const T* b[3];
  T h2i;
  const T* phi;
  T* out;
  const T* rhs;
  const T* c;
  int nt[3];  // tiles
  HD static int ext(int d) { return B::R(d) - (d < DM ? 2 * M : 0); }
  HD void origin(int blk, int* o) const {
    o[0] = (blk % nt[0]) * ext(0) - M;
    o[1] = (blk / nt[0]) % nt[1] * ext(1) - M;
    o[2] = DM == 3 ? blk / (nt[0] * nt[1]) * ext(2) - M : 0;
  }
  HD T value(int i, int j, int k) const {
    T v = ld(phi, (unsigned)cidx(g, i, j, k));
    if (UP) v += ld(c, (unsigned)cidx(gc, i >> 1, j >> 1, DM == 3 ? k >> 1 : 0));
    return v;
  }
  // LDS element q's value before the first half sweep
  HD T first(const int* o, int q) const {
    const int w = DM == 3 ? q / B::LXY : 0, rem = DM == 3 ? q - w * B::LXY : q;
    const int v = rem / B::LX, u = rem - v * B::LX;
    bool ok = true;
    const int i = tile_wrap(o[0] + u - 1, g.n[0], g.per[0], ok), j = tile_wrap(o[1] + v - 1, g.n[1], g.per[1], ok);
    const int k = DM == 3 ? tile_wrap(o[2] + w - 1, g.n[2], g.per[2], ok) : 0;
    const T x = value(i, j, k);
    return ok ? x : T(0);  // beyond a wall: met by b = 0 only
  }
  HD MacPair<T> pair(const int* o, int t) const {
    MacPair<T> P;
    const int p = t % (B::RX / 2), v = t / (B::RX / 2) % B::RY, w = DM == 3 ? t / (B::RX / 2 * B::RY) : 0;
    bool okr = true;
    const int j = tile_wrap(o[1] + v, g.n[1], g.per[1], okr), k = DM == 3 ? tile_wrap(o[2] + w, g.n[2], g.per[2], okr) : 0;
    int mr = imin(v, B::RY - 1 - v);
    if (DM == 3) mr = imin(mr, imin(w, B::RZ - 1 - w));
    const int s0 = (o[0] + j + k) & 1;  // the region's first cell of the row has this parity (even extents)
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) {
      const int u = 2 * p + (s0 ^ c2);
      bool ok = okr;
      const int i = tile_wrap(o[0] + u, g.n[0], g.per[0], ok);
      P.o[c2] = (unsigned)cidx(g, i, j, k);
      P.l[c2] = u + B::LX * v + (DM == 3 ? B::LXY * w : 0) + B::LO;
      P.m[c2] = ok ? imin(mr, imin(u, B::RX - 1 - u)) : -1;
      P.r[c2] = ld(rhs, P.o[c2]);
      T ds = T(0);
#pragma unroll
      for (int d = 0; d < DM; ++d) {
        P.b[c2][2 * d] = ld(b[d], (unsigned)fidx(g, d, i + (d == 0), j + (d == 1), k + (d == 2)));
        P.b[c2][2 * d + 1] = ld(b[d], (unsigned)fidx(g, d, i, j, k));
        ds += P.b[c2][2 * d] + P.b[c2][2 * d + 1];
      }
      P.dg[c2] = -ds * h2i;
    }
    return P;
  }
  template <int C>
  HD void step(const MacPair<T>& P, T* x, int s) const {  // mac_L's sums
    if (P.m[C] < s) return;
    const T* q = x + P.l[C];
    const T old = q[0];
    T sum = T(0);
#pragma unroll
    for (int d = 0; d < DM; ++d) {
      const int e = d == 0 ? 1 : (d == 1 ? B::LX : B::LXY);
      sum += P.b[C][2 * d] * (q[e] - old) - P.b[C][2 * d + 1] * (old - q[-e]);
    }
    if (P.dg[C] != T(0)) x[P.l[C]] = old + (P.r[C] - sum * h2i) / P.dg[C];
  }
  HD void store(const int* o, const MacPair<T>& P, const T* x, int t) const {
    const int v = t / (B::RX / 2) % B::RY, w = DM == 3 ? t / (B::RX / 2 * B::RY) : 0;
    if (o[1] + v >= g.n[1] || (DM == 3 && o[2] + w >= g.n[2])) return;  // another tile's
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) {
      const int u = P.l[c2] - B::LO - B::LX * v - (DM == 3 ? B::LXY * w : 0);
      if (P.m[c2] >= M && o[0] + u < g.n[0]) st(out, P.o[c2], x[P.l[c2]]);
    }
  }
#ifndef LMFHD_HOST_DEBUG
  __device__ void block(int blk) const {
    __shared__ T x[B::LN];
    int o[3];
    origin(blk, o);
    const int t = threadIdx.x;
    const MacPair<T> P = pair(o, t);
#pragma unroll
    for (int q = 0; q < (B::LN + BS - 1) / BS; ++q)
      if (q * BS + t < B::LN) x[q * BS + t] = first(o, q * BS + t);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (((C0 + s) & 1) == 0) step<0>(P, x, s);
      else step<1>(P, x, s);
      if (s + 1 < S) __syncthreads();
    }
    store(o, P, x, t);
  }
#endif
  void block_host(int blk) const {
    std::vector<T> x(B::LN);
    int o[3];
    origin(blk, o);
    for (int q = 0; q < B::LN; ++q) x[q] = first(o, q);
    for (int s = 0; s < S; ++s)
      for (int t = 0; t < BS; ++t) {
        const MacPair<T> P = pair(o, t);
        if (((C0 + s) & 1) == 0) step<0>(P, x.data(), s);
        else step<1>(P, x.data(), s);
      }
    for (int t = 0; t < BS; ++t) store(o, pair(o, t), x.data(), t);
  }
};

}  // namespace lmfhd
