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

// The same for a staggered level with decoupled components (|VT| = 1): a workgroup takes a tile of one
// component's faces; wall faces are copied.  A periodic direction's faces 0 and n are two faces with
// values of their own (odd coarser levels and callers can give them different ones): 0 and n both read
// n - 1 and 1, n - 1 reads n, 1 reads 0.  Along the component's direction a region is therefore a
// stretch of the sequence .. n - 1, n, 0, 1, .. with the period n + 1, in which n's neighbour and 0's
// lie two places on.  A face can be swept as often as it has places on its way to the layer loaded
// around the region, less one for each n | 0 on that way; a face n whose way is one place (the
// region's last) cannot be swept at all, since the layer holds 0 and not the 1 it reads.  The stored
// part leaves S places on each side along the component's direction, S - 1 along the others (M): of
// the S + 1 places to the layer at most one n | 0 is among them (S <= 4, n + 1 >= 5), so every stored
// face gets its S steps, and what it reads its steps before them.
// The thin side of the region lies along z, for z faces along y; the pairs lie along x, for x faces
// along y (a pair's faces differ in parity, which n and 0 do not).
template <int DM, int A>
struct StagBox {
  static constexpr int RX = DM == 3 ? 16 : 64, RY = DM == 3 ? (A == 2 ? 8 : 16) : 32, RZ = DM == 3 ? (A == 2 ? 16 : 8) : 1;
  static constexpr int LX = RX + 2, LXY = LX * (RY + 2);
  static constexpr int LN = LXY * (DM == 3 ? RZ + 2 : 1);
  static constexpr int LO = 1 + LX + (DM == 3 ? LXY : 0);
  static constexpr int PX = A == 0 ? 1 : 2, PY = A == 0 ? 2 : 1;  // faces of a pair along x, y
  HD static constexpr int R(int d) { return d == 0 ? RX : (d == 1 ? RY : RZ); }
  HD static constexpr int E(int d) { return d == 0 ? 1 : (d == 1 ? LX : LXY); }
  // places at either side not stored after S half sweeps (above)
  HD static constexpr int M(int d, int S) { return d >= DM ? 0 : S - 1 + (d == A); }
};
// tiles of component a's faces for S half sweeps (extents of at least 4: a period holds the layers)
template <int DM, int A>
inline int stag_tile_count(const Geo& g, int S, int* nt) {
  using B = StagBox<DM, A>;
  for (int d = 0; d < 3; ++d) {
    const int e = B::R(d) - 2 * B::M(d, S);
    nt[d] = (fext(g, A, d) + e - 1) / e;
  }
  return nt[0] * nt[1] * nt[2];
}

template <typename T>
struct StagPair {  // a thread's faces, [c] of parity c
  T w[2][6], r[2], dg[2];  // weights of the neighbours (VT = -1): normal +, -, transverse +, -, ...
  unsigned o[2];
  int l[2], m[2];  // in LDS; the last half sweep that may take it (from 0), -1: none, or a wall face
  int fix[2];      // bits 0 .. 3: that transverse neighbour is the face's own reflection; 4, 5: the normal
                   // neighbour +, - lies two places on; 6: stored
};

template <typename T, int VT, int DM, int S, int C0>
struct StagTileBlk {
  static_assert(VT == 1 || VT == -1, "components are coupled for |visc_type| > 1");
  static constexpr int BS = TileBox<DM>::BS;
  Geo g;
  Coefs<T> C;
  const T* phi[3];
  T* out[3];
  const T* rhs[3];
  T omega;
  int nt[3][3], nb[3];  // component's tiles; tiles of the components up to it
  int sp;
  // the face at place v of direction d; cross: the periods below it (faces n | 0 passed)
  template <int A>
  HD int wrap(int d, int v, bool& ok, int* cross = nullptr) const {
    const int n = g.n[d];
    if (d != A) return tile_wrap(v, n, g.per[d], ok);
    if (g.per[d]) {
      int c = 0;
      while (v < 0) v += n + 1, --c;
      while (v > n) v -= n + 1, ++c;
      if (cross) *cross = c;
      return v;
    }
    ok = ok && v >= 0 && v <= n;
    return v < 0 ? 0 : (v > n ? n : v);
  }
  template <int A>
  HD void origin(int blk, int* o) const {
    using B = StagBox<DM, A>;
    const int q = blk / nt[A][0], h = q / nt[A][1];
    const int tl[3] = {blk - q * nt[A][0], q - h * nt[A][1], h};
#pragma unroll
    for (int d = 0; d < 3; ++d) o[d] = tl[d] * (B::R(d) - 2 * B::M(d, S)) - B::M(d, S);
  }
  template <int A>
  HD T first(const int* o, int q) const {
    using B = StagBox<DM, A>;
    const int w = DM == 3 ? q / B::LXY : 0, rem = DM == 3 ? q - w * B::LXY : q;
    const int v = rem / B::LX, u = rem - v * B::LX;
    bool ok = true;
    const int i = wrap<A>(0, o[0] + u - 1, ok), j = wrap<A>(1, o[1] + v - 1, ok), k = DM == 3 ? wrap<A>(2, o[2] + w - 1, ok) : 0;
    return ld(phi[A], lidx(g, A, i, j, k, sp));  // beyond a wall: never met
  }
  template <int A>
  HD StagPair<T> pair(const int* o, int t) const {
    using B = StagBox<DM, A>;
    StagPair<T> P;
    constexpr int hx = B::RX / B::PX, hy = B::RY / B::PY;
    const int w = DM == 3 ? t / (hx * hy) : 0, rem = DM == 3 ? t - w * hx * hy : t;
    const int pv = rem / hx, pu = rem - pv * hx;
    bool okr = true;
    int cr = 0;
    const int k = DM == 3 ? wrap<A>(2, o[2] + w, okr, &cr) : 0;
    const int line = A == 0 ? wrap<A>(0, o[0] + pu, okr, &cr) : wrap<A>(1, o[1] + pv, okr, &cr);  // across the pair
    const int s0 = ((A == 0 ? o[1] : o[0]) + line + k) & 1;
    int tb[2];
    transverse(A, tb[0], tb[1]);
    constexpr int ea0 = A == 0, ea1 = A == 1, ea2 = A == 2;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int u = A == 0 ? pu : 2 * pu + (s0 ^ c), v = A == 0 ? 2 * pv + (s0 ^ c) : pv;
      bool ok = okr;
      const int i = A == 0 ? line : wrap<A>(0, o[0] + u, ok), j = A == 0 ? wrap<A>(1, o[1] + v, ok) : line;
      const int I[3] = {i, j, k}, U[3] = {u, v, w};
      P.o[c] = lidx(g, A, i, j, k, sp);
      P.l[c] = u + B::LX * v + (DM == 3 ? B::LXY * w : 0) + B::LO;
      const bool wall = wall_face(g, A, I[A]);
      int m = 1 << 20, fix = 64;
#pragma unroll
      for (int d = 0; d < DM; ++d) {
        int lo = U[d], hi = B::R(d) - 1 - U[d];
        if (d == A && g.per[d]) {  // each n | 0 on the way to the loaded layer saves a step
          int c0 = 0, c1 = 0;
          bool z = true;
          wrap<A>(d, o[d] - 1, z, &c0);
          wrap<A>(d, o[d] + B::R(d), z, &c1);
          lo -= cr - c0;
          hi -= c1 - cr;
          fix |= (I[d] == g.n[d] ? 16 : 0) | (I[d] == 0 ? 32 : 0);
        }
        m = imin(m, imin(lo, hi));
        const int at = U[d] - B::M(d, S);
        if (at < 0 || at >= B::R(d) - 2 * B::M(d, S) || o[d] + U[d] >= fext(g, A, d)) fix &= ~64;
      }
      P.m[c] = ok && !wall ? m : -1;
      P.r[c] = ld(rhs[A], P.o[c]);
      const T alpha = ld(C.alpha[A], P.o[c]) * C.theta;
      T dsum = T(0);
      if (VT == -1) {
        P.w[c][0] = cc_at(C.beta, g, i, j, k);
        P.w[c][1] = cc_at(C.beta, g, i - ea0, j - ea1, k - ea2);
        dsum = P.w[c][0] + P.w[c][1];
      }
#pragma unroll
      for (int q = 0; q < DM - 1; ++q) {
        const int b = tb[q], eb0 = b == 0, eb1 = b == 1, eb2 = b == 2;
        if (VT == -1) {
          const T* E = C.bed[edge_id(DM, A, b)];
          P.w[c][3 + 2 * q] = ld(E, (unsigned)eidx(g, edge_id(DM, A, b), i, j, k));
          P.w[c][2 + 2 * q] = ld(E, (unsigned)eidx(g, edge_id(DM, A, b), i + eb0, j + eb1, k + eb2));
          dsum += P.w[c][3 + 2 * q] + P.w[c][2 + 2 * q];
        }
        if (!g.per[b]) fix |= (I[b] == g.n[b] - 1 ? 1 << (2 * q) : 0) | (I[b] == 0 ? 2 << (2 * q) : 0);
      }
      P.fix[c] = fix;
      P.dg[c] = VT == -1 ? alpha + dsum * C.dxsqinv : alpha + T(2 * DM) * C.beta[0] * C.dxsqinv;
    }
    return P;
  }
  template <int A, int CL>
  HD void step(const StagPair<T>& P, T* x, int s) const {  // lphi_acc's sums
    using B = StagBox<DM, A>;
    if (P.m[CL] < s) return;
    const int fix = P.fix[CL];
    const T* q = x + P.l[CL];
    const T old = q[0];
    int tb[2];
    transverse(A, tb[0], tb[1]);
    const T np = q[fix & 16 ? 2 * B::E(A) : B::E(A)], nm = q[fix & 32 ? -2 * B::E(A) : -B::E(A)];
    T offs = VT == -1 ? np * P.w[CL][0] + nm * P.w[CL][1] : T(0);
#pragma unroll
    for (int t = 0; t < DM - 1; ++t) {
      const int b = tb[t];
      T xp = q[B::E(b)], xm = q[-B::E(b)];
      if (fix & (1 << (2 * t))) xp = g.shi[b] < 0 ? -old : old;
      if (fix & (2 << (2 * t))) xm = g.slo[b] < 0 ? -old : old;
      if (VT == -1) offs += xp * P.w[CL][2 + 2 * t] + xm * P.w[CL][3 + 2 * t];
      else offs += xp + xm;
    }
    const T L = VT == -1 ? old * P.dg[CL] - offs * C.dxsqinv : old * P.dg[CL] - (np + nm + offs) * C.beta[0] * C.dxsqinv;
    x[P.l[CL]] = old + omega * (P.r[CL] - L) / P.dg[CL];
  }
  template <int A>
  HD void store(const StagPair<T>& P, const T* x) const {
#pragma unroll
    for (int c = 0; c < 2; ++c)
      if (P.fix[c] & 64) st(out[A], P.o[c], x[P.l[c]]);
  }
#ifndef LMFHD_HOST_DEBUG
  template <int A>
  __device__ void comp(int blk, T* x) const {
    using B = StagBox<DM, A>;
    const int t = threadIdx.x;
    int o[3];
    origin<A>(blk, o);
    const StagPair<T> P = pair<A>(o, t);
#pragma unroll
    for (int q = 0; q < (B::LN + BS - 1) / BS; ++q)
      if (q * BS + t < B::LN) x[q * BS + t] = first<A>(o, q * BS + t);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (((C0 + s) & 1) == 0) step<A, 0>(P, x, s);
      else step<A, 1>(P, x, s);
      if (s + 1 < S) __syncthreads();
    }
    store<A>(P, x);
  }
  __device__ void block(int blk) const {
    __shared__ T x[TileBox<DM>::LN];  // the components' boxes are of one size
    if (blk < nb[0]) comp<0>(blk, x);
    else if (DM == 2 || blk < nb[1]) comp<1>(blk - nb[0], x);
    else comp<DM - 1>(blk - nb[1], x);
  }
#endif
  template <int A>
  void comp_host(int blk) const {
    std::vector<T> x(StagBox<DM, A>::LN);
    int o[3];
    origin<A>(blk, o);
    for (int q = 0; q < StagBox<DM, A>::LN; ++q) x[q] = first<A>(o, q);
    for (int s = 0; s < S; ++s)
      for (int t = 0; t < BS; ++t) {
        const StagPair<T> P = pair<A>(o, t);
        if (((C0 + s) & 1) == 0) step<A, 0>(P, x.data(), s);
        else step<A, 1>(P, x.data(), s);
      }
    for (int t = 0; t < BS; ++t) store<A>(pair<A>(o, t), x.data());
  }
  void block_host(int blk) const {
    if (blk < nb[0]) comp_host<0>(blk);
    else if (DM == 2 || blk < nb[1]) comp_host<1>(blk - nb[0]);
    else comp_host<DM - 1>(blk - nb[1]);
  }
};

}  // namespace lmfhd
