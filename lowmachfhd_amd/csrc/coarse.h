// coarse.h -- the multigrids' coarse levels in one workgroup.
//
// The smallest levels of a V-cycle (level l0 and every coarser one) run in one kernel of one
// workgroup, with a barrier where the reference has a pass (stag_mg_solver.f90:323-807).  Every
// face (cell) of a level belongs to one thread, which forms the stencil of its faces once per
// visit of the level -- the neighbours' offsets, the coefficients, the diagonal, the right-hand
// side -- and holds it in registers for all sweeps of that visit; a colour step is then a few LDS
// reads, the sum in the reference's order, a division and a write.  phi, rhs and the residual of
// all these levels live in LDS (the "work" block); the coefficients are read from memory.
//
// What bounds it: the length of the dependent chain between two barriers (one workgroup, most
// levels with fewer faces than threads).  With the stencil formed anew in every phase the chain
// was index arithmetic, about 1.5 us a phase; with it in registers a phase is a few LDS
// latencies.  Measured on MI355X, the V-cycle from 8^3 down to 2^3: staggered, visc_type -1, 73 ->
// 35 us in FP32 and 76 -> 35 us in FP64, visc_type -2 in FP64 152 -> 59 us; MAC 36 -> 20 us.
// Levels just above 8^3 (12^3, 10 x 6 x 7, 2-D 32^2) used to take some 11 launches of about 4.3 us
// each per V-cycle and hierarchy; here they add 10 to 30 us.
//
// A body is written as a sequence of phases, x.each(f): f(tid, st) for every thread on its own
// state st, then a barrier.  The same bodies run on the CPU in the host debug build (HostX).
#pragma once
#include <type_traits>

#include "launch.h"
#include "stencils.h"

namespace lmfhd {

// compile-time dispatch on (visc_type, dm)
template <class F>
void dispatch_vd(int vt, int dm, F&& f) {
#define LMFHD_VD(V, D) f(std::integral_constant<int, V>{}, std::integral_constant<int, D>{})
  if (dm == 3) {
    switch (vt) {
      case -1: LMFHD_VD(-1, 3); break;
      case -2: LMFHD_VD(-2, 3); break;
      case -3: LMFHD_VD(-3, 3); break;
      case 1: LMFHD_VD(1, 3); break;
      case 2: LMFHD_VD(2, 3); break;
      default: LMFHD_VD(3, 3); break;
    }
  } else {
    switch (vt) {
      case -1: LMFHD_VD(-1, 2); break;
      case -2: LMFHD_VD(-2, 2); break;
      case -3: LMFHD_VD(-3, 2); break;
      case 1: LMFHD_VD(1, 2); break;
      case 2: LMFHD_VD(2, 2); break;
      default: LMFHD_VD(3, 2); break;
    }
  }
#undef LMFHD_VD
}

static const int COARSE_MAXL = 16;
static const int COARSE_N = 16;             // largest extent lmfhd_tune.coarse_n may ask for
constexpr int COARSE_THREADS = 1024;        // largest workgroup of the kernels
constexpr unsigned COARSE_LDS = 156u * 1024u;  // LDS of the work block (160 KB per CU, less the mean's few words)
constexpr long COARSE_WORK_MAX = 65536;     // elements: offsets in the work block are held in 16 bits

// Faces (cells) one thread holds in registers.  A workgroup of 1024 threads has 128 VGPRs a
// thread; a slot takes about 14 in FP32, 22 in FP64, six more with the cross terms of
// |visc_type| 2 and 3.
template <typename T>
constexpr int stag_slots_max(int vt) { return (vt == 1 || vt == -1) ? (sizeof(T) == 4 ? 6 : 3) : (sizeof(T) == 4 ? 4 : 2); }
template <typename T>
constexpr int mac_slots_max(int dm) { return sizeof(T) == 4 || dm == 2 ? 4 : 2; }
// Where no level needs more than two slots a thread, the kernel that holds only those runs: a
// single short copy of each step.  A coarse V-cycle runs its code about once, from a cold
// instruction cache, so its length counts.
constexpr int SLOTS_SMALL = 2;

// The argument block as the kernels see it: in the constant address space, so that a field at a
// wave-uniform address is one scalar load (through a plain pointer every field would be a vector
// load of its own after each barrier, since a store in between might alias it)
#ifdef LMFHD_HOST_DEBUG
#define LMFHD_CONST
#else
#define LMFHD_CONST __attribute__((address_space(4)))
#endif
// decode3 / decode_color on a decoder there; decode_color's item u is moved into [0, ..) of the
// array by the caller, and a row's missing last item gives i = nx (the caller's to drop)
template <class D>
HD unsigned cdiv(D& f, unsigned u) {
  const unsigned t = (unsigned)(((unsigned long long)f.m * u) >> 32);
  return (t + u) >> f.l;
}
template <class D>
HD void cdecode3(unsigned u, D& dc, int& i, int& j, int& k) {
  const unsigned r = cdiv(dc.x, u);
  i = (int)(u - r * dc.x.d);
  const unsigned q = cdiv(dc.y, r);
  j = (int)(r - q * dc.y.d);
  k = (int)q;
}
template <class D>
HD void cdecode_color(unsigned u, D& dc, int par, int& i, int& j, int& k) {
  cdecode3(u, dc, i, j, k);
  i = 2 * i + ((par + j + k) & 1);
}

HD int pad64(int n) { return (n + 63) & ~63; }
template <typename V>
HD V sel3(int a, V x, V y, V z) { return a == 0 ? x : (a == 1 ? y : z); }

// ---- staggered multigrid ------------------------------------------------------------------------
// A level's slots: the colour items of every component and parity, each colour padded to a
// multiple of 64, so that a wave holds one colour.  Colours by parity then component where the
// components decouple (|visc_type| 1: one phase per parity), else in the reference's order
// 1 .. 2 dm (component, then parity; one phase each).
template <typename T>
struct StagLevArgs {
  Geo g;
  T dxsqinv;
  int inplace;        // even sizes: no face of a colour reads another, updates in place
  int start[7];       // first slot of each colour, then the number of slots
  int nc[3];          // colour items of component a
  int nx[3], nxy[3];  // strides of component a's arrays
  int off[3];         // element offset of component a within phi, rhs and res alike
  int phi, span;      // work block: phi at phi, rhs at phi + span, res at phi + 2 span
  int fstart[4];      // padded ranges of the components' faces
  int nf[3];          // their numbers
  int enx[3], enxy[3];
  Dec dface[3], dcolor[3];
  const T* alpha[3];
  const T* beta;
  const T* gamma;
  const T* bed[3];
};
template <typename T>
struct StagCoarseArgs {
  int l0, nl, nu_down, nu_up, nu_bottom;
  T omega;
  T* work;  // the work block in device memory
  StagLevArgs<T> L[COARSE_MAXL];
};
// The level table (several KB) exceeds the kernel-argument segment (launch.h), so it lives in
// device memory, written by a completed copy from the host before any kernel reads it.

// the slots of one level: colour starts, padded; returns their number
inline int stag_slots(const Geo& g, int vt, int* start) {
  const bool fused = vt == 1 || vt == -1;
  int s = 0;
  for (int c = 0; c < 2 * g.dm; ++c) {
    const int a = fused ? c % g.dm : c / 2;
    if (start) start[c] = s;
    s += pad64((fext(g, a, 0) + 1) / 2 * fext(g, a, 1) * fext(g, a, 2));
  }
  if (start) start[2 * g.dm] = s;
  return s;
}
// elements of one of a level's three blocks (component arrays on multiples of 64 elements)
inline long stag_span(const Geo& g) {
  long n = 0;
  for (int a = 0; a < g.dm; ++a) n += (fsize(g, a) + 63) / 64 * 64;
  return n;
}

// the stencil of one face in registers
template <typename T, int VT, int DM>
struct StagSlot {
  // bits 0-15: its phi in the work block; 16, 17: kind (0 none, 1 a face to smooth, 2 a wall face,
  // held at zero); 18 + 2 t, 19 + 2 t: ghost sign of the transverse neighbour + / - of direction t
  unsigned m = 0;
  unsigned nb[DM];  // neighbours along the normal, then the transverse directions: + | - << 16
  unsigned xo[VT == 1 || VT == -1 ? 1 : 2 * (DM - 1)];  // cross terms: I | P << 16, M | MP << 16
  T c[VT < 0 ? 2 * DM : 1];  // nI, nM, then eP, eI per transverse direction (visc_type -1: with sign)
  T tI[VT == -3 ? 2 : 1];
  T diag, r;
  HD unsigned o() const { return m & 0xffffu; }
  HD int kind() const { return (int)(m >> 16 & 3u); }
  HD bool neg(int bit) const { return m >> (18 + bit) & 1u; }
};

// slot s of level L: which face, its stencil.  Each neighbour follows vel_at's and cc_at's rules;
// every coefficient and sum is lphi_acc's.  comp, i, j, k: the face.
// Without branches: an item past the colour's end takes item 0's, a row's missing last one its
// neighbour's (loads in bounds), and is dropped by its kind; so the loads of several slots are in
// flight together.
template <typename T, int VT, int DM, class LV>
HD void stag_setup(LV& L, const T* W, int s, int color, StagSlot<T, VT, DM>& S, int& comp, int& i, int& j, int& k) {
  constexpr bool FUSED = VT == 1 || VT == -1;
  const int a = FUSED ? (color >= DM ? color - DM : color) : color >> 1;
  const int par = FUSED ? (color >= DM ? 1 : 0) : color & 1;
  comp = a;
  const int u = s - L.start[color];
  const bool in = u < L.nc[a];
  cdecode_color((unsigned)(in ? u : 0), L.dcolor[a], par, i, j, k);
  const int nx = L.nx[a], nxy = L.nxy[a];
  const bool row = i < nx;
  i = row ? i : nx - 1;
  const int fo = i + nx * j + nxy * k;
  const unsigned o = (unsigned)(L.phi + L.off[a] + fo);
  const int Ia = sel3(a, i, j, k), na = L.g.n[a];
  const bool wall = (Ia == 0 && L.g.wlo[a]) || (Ia == na && L.g.whi[a]);
  unsigned m = o | (in && row ? (wall ? 2u : 1u) : 0u) << 16;
  S.r = W[o + L.span];
  int tb[2];
  tb[0] = a == 0 ? 1 : 0;
  tb[1] = a == 2 ? 1 : 2;
  const int sa = sel3(a, 1, nx, nxy);
  {
    const int up = Ia == na ? 1 : Ia + 1, dn = Ia == 0 ? na - 1 : Ia - 1;
    S.nb[0] = (o + (up - Ia) * sa) | ((o + (dn - Ia) * sa) << 16);
  }
#pragma unroll
  for (int t = 0; t < DM - 1; ++t) {
    const int b = tb[t], n = L.g.n[b], per = L.g.per[b];
    const int v = sel3(b, i, j, k), st = sel3(b, 1, nx, nxy);
    const bool hi = v == n - 1, lo = v == 0;
    const int up = hi ? (per ? 0 : v) : v + 1, dn = lo ? (per ? n - 1 : v) : v - 1;
    S.nb[1 + t] = (o + (up - v) * st) | ((o + (dn - v) * st) << 16);
    m |= (hi && !per && L.g.shi[b] < 0) ? 1u << (18 + 2 * t) : 0u;
    m |= (lo && !per && L.g.slo[b] < 0) ? 2u << (18 + 2 * t) : 0u;
  }
  S.m = m;
  const T alpha = L.alpha[a][fo];
  // the cells on both sides of the face (cc_at)
  const int iI = Ia == na ? 0 : Ia, iM = Ia == 0 ? na - 1 : Ia - 1;
  if constexpr (VT < 0) {
    const int cx = L.g.n[0], cxy = L.g.n[0] * L.g.n[1];
    const int cs = sel3(a, 1, cx, cxy);
    const int cb = i + cx * j + cxy * k - Ia * cs;
    const T bI = L.beta[cb + iI * cs], bM = L.beta[cb + iM * cs];
    T nI, nM;
    if constexpr (VT == -3) {
      const T gI = L.gamma[cb + iI * cs], gM = L.gamma[cb + iM * cs];
      nI = T(4.0 / 3.0) * bI + gI;
      nM = T(4.0 / 3.0) * bM + gM;
      S.tI[0] = -T(2.0 / 3.0) * bI + gI;
      S.tI[1] = -T(2.0 / 3.0) * bM + gM;
    } else if constexpr (VT == -2) {
      nI = T(2) * bI;
      nM = T(2) * bM;
    } else {
      nI = bI;
      nM = bM;
    }
    S.c[0] = nI;
    S.c[1] = nM;
    T dsum = nI + nM;
#pragma unroll
    for (int t = 0; t < DM - 1; ++t) {
      const int b = tb[t], e = edge_id(DM, a, b);
      const int es = sel3(b, 1, L.enx[e], L.enxy[e]);
      const T* E = L.bed[e];
      const int eo = i + L.enx[e] * j + L.enxy[e] * k;
      const T eI = E[eo], eP = E[eo + es];
      dsum += eI + eP;
      if constexpr (VT == -1) {  // the ghost's sign on its coefficient: the same products
        S.c[2 + 2 * t] = S.neg(2 * t) ? -eP : eP;
        S.c[3 + 2 * t] = S.neg(2 * t + 1) ? -eI : eI;
      } else {
        S.c[2 + 2 * t] = eP;
        S.c[3 + 2 * t] = eI;
      }
    }
    S.diag = alpha + dsum * L.dxsqinv;
  } else if constexpr (VT == 1) {
    S.diag = alpha + T(2 * DM) * L.beta[0] * L.dxsqinv;
  } else if constexpr (VT == 2) {
    S.diag = alpha + T(2 * DM + 2) * L.beta[0] * L.dxsqinv;
  } else {
    const T num = DM == 3 ? T(20) : T(14);
    S.diag = alpha + (num * L.beta[0] * T(1.0 / 3.0) + T(2) * L.gamma[0]) * L.dxsqinv;
  }
  if constexpr (!FUSED) {
#pragma unroll
    for (int t = 0; t < DM - 1; ++t) {
      const int b = tb[t];
      const int ba = sel3(a, 1, L.nx[b], L.nxy[b]), bb = sel3(b, 1, L.nx[b], L.nxy[b]);
      const unsigned base = (unsigned)(L.phi + L.off[b] + i + L.nx[b] * j + L.nxy[b] * k - Ia * ba);
      const unsigned oI = base + iI * ba, oM = base + iM * ba;
      S.xo[2 * t] = oI | ((oI + bb) << 16);
      S.xo[2 * t + 1] = oM | ((oM + bb) << 16);
    }
  }
}

// L phi at the slot's face (old: phi there), lphi_acc's sums in its order
template <typename T, int VT, int DM>
HD T stag_slot_L(T dxsqinv, const T* W, const StagSlot<T, VT, DM>& S, T old, T b0, T g0) {
  constexpr bool FUSED = VT == 1 || VT == -1;
  const T pp = W[S.nb[0] & 0xffffu], pm = W[S.nb[0] >> 16];
  T tp[DM - 1], tm[DM - 1];
#pragma unroll
  for (int t = 0; t < DM - 1; ++t) {
    tp[t] = W[S.nb[1 + t] & 0xffffu];
    tm[t] = W[S.nb[1 + t] >> 16];
    if constexpr (VT != -1) {
      tp[t] = S.neg(2 * t) ? -tp[t] : tp[t];
      tm[t] = S.neg(2 * t + 1) ? -tm[t] : tm[t];
    }
  }
  T xI[DM - 1], xP[DM - 1], xM[DM - 1], xMP[DM - 1];
  if constexpr (!FUSED) {
#pragma unroll
    for (int t = 0; t < DM - 1; ++t) {
      xI[t] = W[S.xo[2 * t] & 0xffffu];
      xP[t] = W[S.xo[2 * t] >> 16];
      xM[t] = W[S.xo[2 * t + 1] & 0xffffu];
      xMP[t] = W[S.xo[2 * t + 1] >> 16];
    }
  }
  T cross = T(0);
  if constexpr (VT < 0) {
    T offs = pp * S.c[0] + pm * S.c[1];
#pragma unroll
    for (int t = 0; t < DM - 1; ++t) {
      const T eP = S.c[2 + 2 * t], eI = S.c[3 + 2 * t];
      offs += tp[t] * eP + tm[t] * eI;
      if constexpr (VT == -2) cross += xP[t] * eP - xI[t] * eI - xMP[t] * eP + xM[t] * eI;
      if constexpr (VT == -3)
        cross += xP[t] * (eP + S.tI[0]) - xI[t] * (eI + S.tI[0]) - xMP[t] * (eP + S.tI[1]) + xM[t] * (eI + S.tI[1]);
    }
    return old * S.diag - (offs + cross) * dxsqinv;
  } else {
    const T nsum = pp + pm;
    T tsum = T(0);
#pragma unroll
    for (int t = 0; t < DM - 1; ++t) {
      tsum += tp[t] + tm[t];
      if constexpr (!FUSED) cross += xP[t] - xI[t] - xMP[t] + xM[t];
    }
    if constexpr (VT == 1) return old * S.diag - (nsum + tsum) * b0 * dxsqinv;
    if constexpr (VT == 2) return old * S.diag - (T(2) * nsum + tsum + cross) * b0 * dxsqinv;
    return old * S.diag -
           (nsum * (T(4.0 / 3.0) * b0 + g0) + tsum * b0 + cross * (T(1.0 / 3.0) * b0 + g0)) * dxsqinv;
  }
}

// the prolongation's increment at face (i,j,k) of component a (ProlongCFn's sums in its order)
template <typename T, int DM, class LV>
HD T stag_prolong_add(LV& Lc, const T* W, int a, int i, int j, int k) {
  int tb[2];
  tb[0] = a == 0 ? 1 : 0;
  tb[1] = a == 2 ? 1 : 2;
  const T* P = W + Lc.phi + Lc.off[a];
  const int nx = Lc.nx[a], nxy = Lc.nxy[a];
  const int Ia = sel3(a, i, j, k);
  const bool odd = Ia & 1;
  const int sa = sel3(a, 1, nx, nxy);
  int base = (Ia >> 1) * sa;
  const int step = odd ? sa : 0;  // even faces take no value above
  int d[2] = {0, 0};
  bool neg[2] = {false, false};
#pragma unroll
  for (int t = 0; t < DM - 1; ++t) {
    const int b = tb[t], n = Lc.g.n[b], per = Lc.g.per[b];
    const int v = sel3(b, i, j, k), st = sel3(b, 1, nx, nxy);
    const int c0 = v >> 1, c1 = (v & 1) ? c0 + 1 : c0 - 1;
    const bool hi = c1 >= n, lo = c1 < 0;
    const int w = hi ? (per ? 0 : n - 1) : (lo ? (per ? n - 1 : 0) : c1);
    neg[t] = !per && ((hi && Lc.g.shi[b] < 0) || (lo && Lc.g.slo[b] < 0));
    base += c0 * st;
    d[t] = (w - c0) * st;
  }
  const T p000 = P[base], p100 = P[base + step];
  T p0b0 = P[base + d[0]], p1b0 = P[base + step + d[0]];
  p0b0 = neg[0] ? -p0b0 : p0b0;
  p1b0 = neg[0] ? -p1b0 : p1b0;
  if constexpr (DM == 3) {
    T p00c = P[base + d[1]], p10c = P[base + step + d[1]];
    T p0bc = P[base + d[0] + d[1]], p1bc = P[base + step + d[0] + d[1]];
    p00c = neg[1] ? -p00c : p00c;
    p10c = neg[1] ? -p10c : p10c;
    p0bc = neg[0] != neg[1] ? -p0bc : p0bc;
    p1bc = neg[0] != neg[1] ? -p1bc : p1bc;
    const T se = T(9.0 / 16.0) * p000 + T(3.0 / 16.0) * p0b0 + T(3.0 / 16.0) * p00c + T(1.0 / 16.0) * p0bc;
    const T so = T(9.0 / 32.0) * p000 + T(3.0 / 32.0) * p0b0 + T(3.0 / 32.0) * p00c + T(1.0 / 32.0) * p0bc +
                 T(9.0 / 32.0) * p100 + T(3.0 / 32.0) * p1b0 + T(3.0 / 32.0) * p10c + T(1.0 / 32.0) * p1bc;
    return odd ? so : se;
  } else {
    const T se = T(0.75) * p000 + T(0.25) * p0b0;
    const T so = T(0.375) * p000 + T(0.125) * p0b0 + T(0.375) * p100 + T(0.125) * p1b0;
    return odd ? so : se;
  }
}

// the residual restricted to face (i,j,k) of component a (RestrictFn's sums in its order)
template <typename T, int DM, class LV>
HD T stag_restrict(LV& Lf, LV& Lc, const T* W, int a, int i, int j, int k) {
  const int Ia = sel3(a, i, j, k);
  if ((Ia == 0 && Lc.g.wlo[a]) || (Ia == Lc.g.n[a] && Lc.g.whi[a])) return T(0);
  int tb[2];
  tb[0] = a == 0 ? 1 : 0;
  tb[1] = a == 2 ? 1 : 2;
  const T* R = W + Lf.phi + 2 * Lf.span + Lf.off[a];
  const int nx = Lf.nx[a], nxy = Lf.nxy[a], na = Lf.g.n[a];
  const int sa = sel3(a, 1, nx, nxy);
  const int fa = 2 * Ia, up = fa == na ? 1 : fa + 1, dn = fa == 0 ? na - 1 : fa - 1;
  const int o0 = 2 * (i + nx * j + (DM == 3 ? nxy * k : 0));
  const int s0b = sel3(tb[0], 1, nx, nxy), s1b = DM == 3 ? sel3(tb[1], 1, nx, nxy) : 0;
  const int du = (up - fa) * sa, dd = (dn - fa) * sa;
  T s0 = T(0), sp = T(0), sm = T(0);
#pragma unroll
  for (int q = 0; q < (1 << (DM - 1)); ++q) {
    const int o = o0 + (q & 1) * s0b + ((q >> 1) & 1) * s1b;
    s0 += R[o];
    sp += R[o + du];
    sm += R[o + dd];
  }
  if (DM == 3) return T(0.125) * s0 + T(0.0625) * sp + T(0.0625) * sm;
  return T(0.25) * s0 + T(0.125) * (sp + sm);
}

template <typename T, int VT, int DM, int KM>
struct StagState {
  StagSlot<T, VT, DM> S[KM];
};

// KM: the most slots a thread holds; SMALL: every level fits SLOTS_SMALL (the host's choice)
template <typename T, int VT, int DM, int KM, int SMALL, class AV, class X>
HD void stag_coarse_body(AV& A, T* W, X& x) {
  using Slot = StagSlot<T, VT, DM>;
  using State = StagState<T, VT, DM, KM>;
  constexpr bool FUSED = VT == 1 || VT == -1;
  constexpr int NCOL = 2 * DM;
  constexpr int NPH = FUSED ? 2 : NCOL;
  const int nt = x.threads();
  const int D = A.nl - 1 - A.l0;
  for (int v = 0; v <= 2 * D; ++v) {
    const bool up = v > D;
    const int n = A.l0 + (up ? 2 * D - v : v);
    const int nsw = v < D ? A.nu_down : (up ? A.nu_up : A.nu_bottom);
    auto& L = A.L[n];
    auto& Lc = A.L[up || v < D ? n + 1 : n];  // the next coarser level
    const int nslots = L.start[NCOL];
    const int res = 2 * L.span;
    const bool inplace = L.inplace;
    const T dxsqinv = L.dxsqinv, omega = A.omega;
    T b0 = T(0), g0 = T(0);
    if constexpr (VT > 0) b0 = L.beta[0];
    if constexpr (VT == 3) g0 = L.gamma[0];
    auto color_of = [&](int s) __attribute__((always_inline)) {  // of slot s (one colour per wave)
      int c = 0;
#pragma unroll
      for (int q = 1; q < NCOL; ++q) c += s >= L.start[q] ? 1 : 0;
      return x.uniform(c);
    };
    auto phase_range = [&](int ph, int& p0, int& p1) __attribute__((always_inline)) {
      p0 = FUSED ? (ph == 0 ? 0 : L.start[DM]) : L.start[ph];
      p1 = FUSED ? (ph == 0 ? L.start[DM] : nslots) : L.start[ph + 1];
    };
    auto updated = [&](const Slot& S) __attribute__((always_inline)) {
      const T old = W[S.o()];
      const T Lp = stag_slot_L<T, VT, DM>(dxsqinv, W, S, old, b0, g0);
      return old + omega * (S.r - Lp) / S.diag;
    };
    auto residual = [&](const Slot& S) __attribute__((always_inline)) {
      const T r = S.r - stag_slot_L<T, VT, DM>(dxsqinv, W, S, W[S.o()], b0, g0);
      if (S.kind()) W[S.o() + res] = S.kind() == 1 ? r : T(0);
    };
    auto held = [&](auto Kc) __attribute__((always_inline)) {
      constexpr int K = decltype(Kc)::value;
      // the thread's slots tid, tid + nt, ...: set up, and on the way up the prolongation added
      x.template each<State>([&](int tid, State& st) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < K; ++q) st.S[q].m = 0;
        if (x.uniform(tid & ~63) >= nslots) return;  // a wave without slots leaves the unit to the others
#pragma unroll
        for (int q = 0; q < K; ++q) {
          int a, i, j, k;
          stag_setup<T, VT, DM>(L, W, tid + q * nt, color_of(tid + q * nt), st.S[q], a, i, j, k);
          if (up) {
            const T add = stag_prolong_add<T, DM>(Lc, W, a, i, j, k);
            if (st.S[q].kind() == 1) W[st.S[q].o()] = W[st.S[q].o()] + add;
          }
          if (K > 2) x.fence();
        }
      });
      for (int m = 0; m < nsw; ++m)
        for (int ph = 0; ph < NPH; ++ph) {
          int p0, p1;
          phase_range(ph, p0, p1);
          if (inplace) {
            x.template each<State>([&](int tid, State& st) __attribute__((always_inline)) {
#pragma unroll
              for (int q = 0; q < K; ++q) {
                const int w = x.uniform(tid & ~63) + q * nt;
                if (w >= p0 && w < p1 && st.S[q].kind() == 1) W[st.S[q].o()] = updated(st.S[q]);
              }
            });
            continue;
          }
          // odd sizes: every new value from the old ones (kept in the residual's place), then stored
          for (int step = 0; step < 2; ++step)
            x.template each<State>([&](int tid, State& st) __attribute__((always_inline)) {
#pragma unroll
              for (int q = 0; q < K; ++q) {
                const int w = x.uniform(tid & ~63) + q * nt;
                if (w < p0 || w >= p1 || st.S[q].kind() != 1) continue;
                if (step == 0) W[st.S[q].o() + res] = updated(st.S[q]);
                else W[st.S[q].o()] = W[st.S[q].o() + res];
              }
            });
        }
      if (v < D)
        x.template each<State>([&](int tid, State& st) __attribute__((always_inline)) {
          if (x.uniform(tid & ~63) >= nslots) return;
#pragma unroll
          for (int q = 0; q < K; ++q) {
            residual(st.S[q]);
            if (K > 2) x.fence();
          }
        });
    };
    // more faces than registers: each phase sets up the slots it needs
    auto over = [&](int s0, int s1, const auto& f) __attribute__((always_inline)) {
      x.template each<State>([&](int tid, State&) __attribute__((always_inline)) {
        for (int s = s0 + tid; s < s1; s += nt) {
          Slot S;
          int a, i, j, k;
          stag_setup<T, VT, DM>(L, W, s, color_of(s), S, a, i, j, k);
          f(S, a, i, j, k);
        }
      });
    };
    if constexpr (SMALL) {
      held(std::integral_constant<int, SLOTS_SMALL>{});
    } else if (nslots <= SLOTS_SMALL * nt) {
      held(std::integral_constant<int, SLOTS_SMALL>{});
    } else if (KM > SLOTS_SMALL && nslots <= KM * nt) {
      held(std::integral_constant<int, KM>{});
    } else {
      if (up)
        over(0, nslots, [&](const Slot& S, int a, int i, int j, int k) __attribute__((always_inline)) {
          if (S.kind() == 1) W[S.o()] = W[S.o()] + stag_prolong_add<T, DM>(Lc, W, a, i, j, k);
        });
      for (int m = 0; m < nsw; ++m)
        for (int ph = 0; ph < NPH; ++ph) {
          int p0, p1;
          phase_range(ph, p0, p1);
          for (int step = 0; step < (inplace ? 1 : 2); ++step)
            over(p0, p1, [&](const Slot& S, int, int, int, int) __attribute__((always_inline)) {
              if (S.kind() != 1) return;
              if (step == 1) W[S.o()] = W[S.o() + res];
              else W[S.o() + (inplace ? 0 : res)] = updated(S);
            });
        }
      if (v < D)
        over(0, nslots, [&](const Slot& S, int, int, int, int) __attribute__((always_inline)) { residual(S); });
    }
    if (v < D) {  // the residual restricted; phi of the level below starts from zero
      x.template each<State>([&](int tid, State&) __attribute__((always_inline)) {
        for (int s = tid; s < Lc.fstart[DM]; s += nt) {
          int a = 0;
#pragma unroll
          for (int q = 1; q < DM; ++q) a += s >= Lc.fstart[q] ? 1 : 0;
          a = x.uniform(a);
          const int t = s - Lc.fstart[a];
          if (t >= Lc.nf[a]) continue;  // padding
          int i, j, k;
          cdecode3((unsigned)t, Lc.dface[a], i, j, k);
          const T r = stag_restrict<T, DM>(L, Lc, W, a, i, j, k);
          const int o = Lc.phi + Lc.off[a] + t;
          W[o + Lc.span] = r;
          W[o] = T(0);
        }
      });
    }
  }
}

// ---- MAC multigrid --------------------------------------------------------------------------------
template <typename T>
struct MacLevArgs {
  Geo g;
  T h2i;
  int inplace;
  int half, nc;      // padded slots of one parity, its colour items
  int phi, span;     // work block: phi, rhs at phi + span, residual at phi + 2 span
  int fnx[3], fnxy[3];
  Dec dcell, dcolor;
  const T* b[3];
};
template <typename T>
struct MacCoarseArgs {
  int l0, nl, nu_down, nu_up, nu_bottom;
  T* work;
  MacLevArgs<T> L[COARSE_MAXL];
};
inline int mac_slots(const Geo& g) { return 2 * pad64((g.n[0] + 1) / 2 * g.n[1] * g.n[2]); }
inline long mac_span(const Geo& g) { return (csize(g) + 63) / 64 * 64; }

template <typename T, int DM>
struct MacSlot {
  unsigned m = 0;  // bits 0-15: its phi in the work block; 16: a cell is there
  unsigned nb[DM];
  T bp[DM], bm[DM];
  T diag, r;
  HD unsigned o() const { return m & 0xffffu; }
  HD int kind() const { return (int)(m >> 16); }
};
template <typename T, int DM, class LV>
HD void mac_setup(LV& L, const T* W, int s, int par, MacSlot<T, DM>& S, int& i, int& j, int& k) {
  const int u = s - par * L.half;
  const bool in = u < L.nc;
  cdecode_color((unsigned)(in ? u : 0), L.dcolor, par, i, j, k);
  const bool row = i < L.g.n[0];
  i = row ? i : L.g.n[0] - 1;
  const unsigned o = (unsigned)(L.phi + i + L.g.n[0] * (j + L.g.n[1] * k));
  S.m = o | (in && row ? 1u : 0u) << 16;
  S.r = W[o + L.span];
  const int I[3] = {i, j, k};
  T dsum = T(0);
#pragma unroll
  for (int d = 0; d < DM; ++d) {
    const int n = L.g.n[d], per = L.g.per[d], v = I[d];
    const int st = d == 0 ? 1 : (d == 1 ? L.g.n[0] : L.g.n[0] * L.g.n[1]);
    const int up = v == n - 1 ? (per ? 0 : v) : v + 1, dn = v == 0 ? (per ? n - 1 : v) : v - 1;
    S.nb[d] = (o + (up - v) * st) | ((o + (dn - v) * st) << 16);
    const int fo = i + L.fnx[d] * j + L.fnxy[d] * k, fs = d == 0 ? 1 : (d == 1 ? L.fnx[d] : L.fnxy[d]);
    S.bm[d] = L.b[d][fo];
    S.bp[d] = L.b[d][fo + fs];
    dsum += S.bp[d] + S.bm[d];
  }
  S.diag = -dsum * L.h2i;
}
template <typename T, int DM, class LV>
HD T mac_slot_L(LV& L, const T* W, const MacSlot<T, DM>& S, T pc) {  // mac_L's sums
  T s = T(0);
#pragma unroll
  for (int d = 0; d < DM; ++d) s += S.bp[d] * (W[S.nb[d] & 0xffffu] - pc) - S.bm[d] * (pc - W[S.nb[d] >> 16]);
  return s * L.h2i;
}
template <typename T, int DM, int KM>
struct MacState {
  MacSlot<T, DM> S[KM];
};

template <typename T, int DM, int KM, int SMALL, class AV, class X>
HD void mac_coarse_body(AV& A, T* W, X& x) {
  using Slot = MacSlot<T, DM>;
  using State = MacState<T, DM, KM>;
  const int nt = x.threads();
  const int D = A.nl - 1 - A.l0;
  for (int v = 0; v <= 2 * D; ++v) {
    const bool up = v > D;
    const int n = A.l0 + (up ? 2 * D - v : v);
    const int nsw = v < D ? A.nu_down : (up ? A.nu_up : A.nu_bottom);
    auto& L = A.L[n];
    auto& Lc = A.L[up || v < D ? n + 1 : n];
    const int half = L.half, nslots = 2 * half;
    const int res = 2 * L.span;
    const bool inplace = L.inplace;
    if (v == D) x.mean(W + L.phi + L.span, L.g.n[0] * L.g.n[1] * L.g.n[2]);
    auto updated = [&](const Slot& S) __attribute__((always_inline)) {
      const T old = W[S.o()];
      const T Lp = mac_slot_L<T, DM>(L, W, S, old);
      return S.diag != T(0) ? old + (S.r - Lp) / S.diag : old;
    };
    auto coarse_phi = [&](int i, int j, int k) __attribute__((always_inline)) {
      return W[Lc.phi + (i >> 1) + Lc.g.n[0] * ((j >> 1) + (DM == 3 ? Lc.g.n[1] * (k >> 1) : 0))];
    };
    auto held = [&](auto Kc) __attribute__((always_inline)) {
      constexpr int K = decltype(Kc)::value;
      x.template each<State>([&](int tid, State& st) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < K; ++q) st.S[q].m = 0;
        if (x.uniform(tid & ~63) >= nslots) return;
#pragma unroll
        for (int q = 0; q < K; ++q) {
          const int s = tid + q * nt;
          int i, j, k;
          mac_setup<T, DM>(L, W, s, x.uniform(s >= half ? 1 : 0), st.S[q], i, j, k);
          if (up) {
            const T add = coarse_phi(i, j, k);
            if (st.S[q].kind()) W[st.S[q].o()] = W[st.S[q].o()] + add;
          }
          if (K > 2) x.fence();
        }
      });
      for (int m = 0; m < nsw; ++m)
        for (int ph = 0; ph < 2; ++ph) {
          if (inplace) {
            x.template each<State>([&](int tid, State& st) __attribute__((always_inline)) {
#pragma unroll
              for (int q = 0; q < K; ++q) {
                const int w = x.uniform(tid & ~63) + q * nt;
                if ((w >= half ? 1 : 0) == ph && st.S[q].kind()) W[st.S[q].o()] = updated(st.S[q]);
              }
            });
            continue;
          }
          for (int step = 0; step < 2; ++step)
            x.template each<State>([&](int tid, State& st) __attribute__((always_inline)) {
#pragma unroll
              for (int q = 0; q < K; ++q) {
                const int w = x.uniform(tid & ~63) + q * nt;
                if ((w >= half ? 1 : 0) != ph || !st.S[q].kind()) continue;
                if (step == 0) W[st.S[q].o() + res] = updated(st.S[q]);
                else W[st.S[q].o()] = W[st.S[q].o() + res];
              }
            });
        }
      if (v < D)
        x.template each<State>([&](int tid, State& st) __attribute__((always_inline)) {
          if (x.uniform(tid & ~63) >= nslots) return;
#pragma unroll
          for (int q = 0; q < K; ++q) {
            const T r = st.S[q].r - mac_slot_L<T, DM>(L, W, st.S[q], W[st.S[q].o()]);
            if (st.S[q].kind()) W[st.S[q].o() + res] = r;
          }
        });
    };
    auto over = [&](int s0, int s1, const auto& f) __attribute__((always_inline)) {
      x.template each<State>([&](int tid, State&) __attribute__((always_inline)) {
        for (int s = s0 + tid; s < s1; s += nt) {
          Slot S;
          int i, j, k;
          mac_setup<T, DM>(L, W, s, x.uniform(s >= half ? 1 : 0), S, i, j, k);
          if (S.kind()) f(S, i, j, k);
        }
      });
    };
    if constexpr (SMALL) {
      held(std::integral_constant<int, SLOTS_SMALL>{});
    } else if (nslots <= SLOTS_SMALL * nt) {
      held(std::integral_constant<int, SLOTS_SMALL>{});
    } else if (KM > SLOTS_SMALL && nslots <= KM * nt) {
      held(std::integral_constant<int, KM>{});
    } else {
      if (up)
        over(0, nslots, [&](const Slot& S, int i, int j, int k) __attribute__((always_inline)) {
          W[S.o()] = W[S.o()] + coarse_phi(i, j, k);
        });
      for (int m = 0; m < nsw; ++m)
        for (int ph = 0; ph < 2; ++ph)
          for (int step = 0; step < (inplace ? 1 : 2); ++step)
            over(ph * half, (ph + 1) * half, [&](const Slot& S, int, int, int) __attribute__((always_inline)) {
              if (step == 1) W[S.o()] = W[S.o() + res];
              else W[S.o() + (inplace ? 0 : res)] = updated(S);
            });
      if (v < D)
        over(0, nslots, [&](const Slot& S, int, int, int) __attribute__((always_inline)) {
          W[S.o() + res] = S.r - mac_slot_L<T, DM>(L, W, S, W[S.o()]);
        });
    }
    if (v < D) {  // mean of the children's residuals (MacResidRestrictFn's order)
      x.template each<State>([&](int tid, State&) __attribute__((always_inline)) {
        const T* R = W + L.phi + res;
        const int fx = L.g.n[0], fxy = L.g.n[0] * L.g.n[1];
        const int nc = Lc.g.n[0] * Lc.g.n[1] * Lc.g.n[2];
        for (int t = tid; t < nc; t += nt) {
          int i, j, k;
          cdecode3((unsigned)t, Lc.dcell, i, j, k);
          const int o = 2 * i + fx * 2 * j + (DM == 3 ? fxy * 2 * k : 0);
          T s = T(0);
#pragma unroll
          for (int q = 0; q < (1 << DM); ++q) s += R[o + (q & 1) + ((q >> 1) & 1) * fx + ((q >> 2) & 1) * fxy];
          W[Lc.phi + Lc.span + t] = (DM == 3 ? T(0.125) : T(0.25)) * s;
          W[Lc.phi + t] = T(0);
        }
      });
    }
  }
}

// ---- launch (coarse.hip) ------------------------------------------------------------------------------
// The form of a coarse kernel: on LDS (level l0's phi and rhs copied in, phi out) with at most
// SLOTS_SMALL slots a thread, on LDS with more, or on the work block in device memory
enum class CoarseForm { lds_small, lds, device };
// one V-cycle of levels l0 .. nl - 1 by one workgroup of nt threads (256, 512 or 1024)
template <typename T>
void launch_stag_coarse(hipStream_t s, int vt, int dm, int nt, CoarseForm form, const StagCoarseArgs<T>* A);
template <typename T>
void launch_mac_coarse(hipStream_t s, int dm, int nt, CoarseForm form, const MacCoarseArgs<T>* A);

}  // namespace lmfhd
