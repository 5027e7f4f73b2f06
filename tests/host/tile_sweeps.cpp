// Host run of the staggered tile (lowmachfhd_amd/csrc/tile.h): for every grid and sweep count
//   * no face a tile sweeps reads beyond the layer loaded around its region;
//   * the stored faces hold, to the bit, what the plain half sweeps (GsColorFn) give.
// The two copies of a periodic face start from values of their own.  Prints one line per failure;
// exit status 0 when there is none.  Built by tests/test_tile_host.py.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../lowmachfhd_amd/csrc/tile.h"

using namespace lmfhd;
typedef std::vector<double> Vec;
static int failures = 0;

// faces of component A swept by a tile whose neighbours are not all in the box it loads
template <int VT, int DM, int S, int C0, int A>
static long beyond(const StagTileBlk<double, VT, DM, S, C0>& F, int nblk) {
  using B = StagBox<DM, A>;
  long bad = 0;
  for (int blk = 0; blk < nblk; ++blk) {
    int o[3];
    F.template origin<A>(blk, o);
    for (int t = 0; t < F.BS; ++t) {
      const StagPair<double> P = F.template pair<A>(o, t);
      for (int c = 0; c < 2; ++c) {
        if (P.m[c] < 0) continue;
        const int l = P.l[c] - B::LO;
        const int U[3] = {l % B::LX, l / B::LX % (B::LXY / B::LX), l / B::LXY};
        for (int d = 0; d < DM; ++d) {
          const int up = d == A && (P.fix[c] & 16) ? 2 : 1, dn = d == A && (P.fix[c] & 32) ? 2 : 1;
          if (U[d] + up > B::R(d) || U[d] - dn < -1) ++bad;
        }
      }
    }
  }
  return bad;
}

template <int VT, int DM, int S, int C0>
static void run(const Geo& g, unsigned seed) {
  std::mt19937 gen(seed);
  std::uniform_real_distribution<double> u01(0.5, 1.5), pm(-1.0, 1.0);
  auto field = [&](long n, bool positive) {
    Vec v(n);
    for (double& x : v) x = positive ? u01(gen) : pm(gen);
    return v;
  };
  Vec alpha[3], phi[3], rhs[3], out[3], bed[3];
  const Vec beta = field(csize(g), true);
  StagTileBlk<double, VT, DM, S, C0> F;
  F.g = g;
  F.omega = 1.0;
  F.sp = 0;
  F.C.beta = F.C.gamma = beta.data();
  F.C.dxsqinv = 7.0;
  F.C.theta = 1.0;
  for (int a = 0; a < 3; ++a) {
    const int q = a < DM ? a : DM - 1;
    alpha[a] = field(fsize(g, q), true);
    rhs[a] = field(fsize(g, q), false);
    phi[a] = field(fsize(g, q), false);
    for (long t = 0; t < fsize(g, q); ++t) {  // wall faces are zero
      const int i = (int)(t % fext(g, q, 0)), j = (int)(t / fext(g, q, 0) % fext(g, q, 1)),
                k = (int)(t / fext(g, q, 0) / fext(g, q, 1));
      const int I[3] = {i, j, k};
      if (wall_face(g, q, I[q])) phi[a][t] = 0.0;
    }
    out[a].assign(fsize(g, q), 1e300);
    bed[a] = field(esize(g, DM == 3 ? a : 0), true);
  }
  int nb = 0;
  for (int a = 0; a < 3; ++a) {
    F.C.alpha[a] = alpha[a].data();
    F.C.bed[a] = bed[a].data();
    F.phi[a] = phi[a].data();
    F.out[a] = out[a].data();
    F.rhs[a] = rhs[a].data();
    int cnt = 0;
    if (a == 0) cnt = stag_tile_count<DM, 0>(g, S, F.nt[0]);
    if (a == 1) cnt = stag_tile_count<DM, 1>(g, S, F.nt[1]);
    if constexpr (DM == 3) {
      if (a == 2) cnt = stag_tile_count<DM, 2>(g, S, F.nt[2]);
    }
    F.nb[a] = nb += cnt;
  }
  long bad = beyond<VT, DM, S, C0, 0>(F, F.nb[0]) + beyond<VT, DM, S, C0, 1>(F, F.nb[1] - F.nb[0]);
  if constexpr (DM == 3) bad += beyond<VT, DM, S, C0, 2>(F, F.nb[2] - F.nb[1]);
  auto say = [&](const char* what, long n) {
    ++failures;
    printf("%dx%dx%d per %d%d%d visc_type %d S %d: %ld %s\n", g.n[0], g.n[1], g.n[2], g.per[0], g.per[1], g.per[2], VT,
           S, n, what);
  };
  if (bad) {  // not run: it would read outside the box
    say("reads beyond the loaded layer", bad);
    return;
  }
  for (int blk = 0; blk < nb; ++blk) F.block_host(blk);
  double* p[3] = {phi[0].data(), phi[1].data(), phi[2].data()};
  for (int s = 0; s < S; ++s)
    for (int a = 0; a < DM; ++a) {
      const int nx = fext(g, a, 0), ny = fext(g, a, 1);
      const GsColorFn<double, VT, DM> G{g, F.C, {p[0], p[1], p[2]}, rhs[a].data(), 1.0, a, make_dec_color(nx, ny), (C0 + s) & 1};
      const long n = (long)((nx + 1) / 2) * ny * fext(g, a, 2);
      for (long t = 0; t < n; ++t) G(t);
    }
  long diff = 0;
  for (int a = 0; a < DM; ++a)
    for (long t = 0; t < fsize(g, a); ++t) diff += out[a][t] != phi[a][t];
  if (diff) say("faces differ from the plain sweeps", diff);
}

static Geo geo(int dm, const int* n, const int* per) {
  Geo g{};
  g.dm = dm;
  for (int d = 0; d < 3; ++d) {
    g.n[d] = d < dm ? n[d] : 1;
    g.per[d] = d < dm ? per[d] : 1;
    g.wlo[d] = g.whi[d] = !g.per[d];
    g.slo[d] = g.per[d] ? 0 : -1;
    g.shi[d] = g.per[d] ? 0 : 1;
  }
  return g;
}
template <int DM>
static void all(const Geo& g, unsigned seed) {
  run<-1, DM, 4, 0>(g, seed);
  run<-1, DM, 3, 1>(g, seed);
}

int main() {
  // every even extent along each direction in turn, periodic and between walls, the others a tile's
  // inner size, one place more, and the smallest
  unsigned seed = 0;
  for (int d = 0; d < 3; ++d)
    for (int n = 4; n <= 44; n += 2)
      for (int per = 0; per < 2; ++per) {
        int N[3] = {4, 10, 12}, P[3] = {1, 1, (n / 2) & 1};
        N[d] = n;
        P[d] = per;
        all<3>(geo(3, N, P), ++seed);
      }
  for (int d = 0; d < 2; ++d)
    for (int n = 4; n <= 90; n += 2)
      for (int per = 0; per < 2; ++per) {
        int N[3] = {28, 54, 1}, P[3] = {1, 1, 1};
        N[d] = n;
        P[d] = per;
        all<2>(geo(2, N, P), ++seed);
      }
  const int M[2][3] = {{24, 24, 12}, {12, 22, 32}}, per[3] = {1, 1, 1};
  for (const auto& n : M) all<3>(geo(3, n, per), ++seed), run<1, 3, 3, 1>(geo(3, n, per), seed);
  const int m2[3] = {56, 28, 1};
  all<2>(geo(2, m2, per), ++seed);
  run<1, 2, 4, 0>(geo(2, m2, per), seed);
  printf("%d failures\n", failures);
  return failures != 0;
}
