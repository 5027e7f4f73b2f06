// Host run of the Arnoldi steps of a GMRES cycle (arnoldi, lsq_status, gs_repair of lmfhd.hip) on
// given vectors, past the 15 that the fused sweeps take.  Step `lost` gets a w that lies in the span
// of the basis but for a part of the size of its rounding: the norm by Pythagoras cannot be used
// there and the step is repaired.  Every step is checked for
//   * the repair: asked for at step `lost` and nowhere else;
//   * an orthonormal basis and w = sum_q H(q, i) V_q;
//   * the residual estimate, against the least-squares problem of the columns so far solved anew.
// Prints one line per failure; exit status 0 when there is none.  Built by tests/test_arnoldi_host.py.
#include "../../lowmachfhd_amd/csrc/lmfhd.hip"

#include <random>

namespace lmfhd {
template <typename T>
void launch_stag_coarse(hipStream_t, int, int, int, CoarseForm, const StagCoarseArgs<T>*) { abort(); }
template <typename T>
void launch_mac_coarse(hipStream_t, int, int, CoarseForm, const MacCoarseArgs<T>*) { abort(); }
}  // namespace lmfhd
using namespace lmfhd;

static double dot(Ctx& c, const double* x, const double* y) {
  double s = 0.0;
  for (long e = 0; e < c.vlen; ++e) s += x[e] * c.VL.weight(e) * y[e];
  return s;
}
// min |beta e1 - H y| over y, H of k columns and k + 1 rows: the columns orthonormalised (twice)
static double least_squares(double beta, const std::vector<std::vector<double>>& H) {
  const int k = (int)H.size();
  std::vector<std::vector<double>> Q;
  std::vector<double> r(k + 1, 0.0);
  r[0] = beta;
  auto take = [&](std::vector<double>& v) {
    for (int pass = 0; pass < 2; ++pass)
      for (const auto& q : Q) {
        double d = 0.0;
        for (int e = 0; e <= k; ++e) d += q[e] * v[e];
        for (int e = 0; e <= k; ++e) v[e] -= d * q[e];
      }
  };
  auto norm = [&](const std::vector<double>& v) {
    double s = 0.0;
    for (double x : v) s += x * x;
    return std::sqrt(s);
  };
  for (auto col : H) {
    col.resize(k + 1, 0.0);
    take(col);
    const double n = norm(col);
    for (double& x : col) x /= n;
    Q.push_back(col);
  }
  take(r);
  return norm(r);
}

static int run(int lost, int m) {
  int bad = 0;
  auto say = [&](int i, const char* what, double v) {
    ++bad;
    printf("step %d lost, step %d of %d: %s %.3g\n", lost, i, m, what, v);
  };
  lmfhd_desc d;
  lmfhd_desc_defaults(&d);
  d.dm = 2;
  d.n_cells[0] = d.n_cells[1] = 8;
  d.dx = 0.125;
  for (int k = 0; k < 3; ++k) d.bc_lo[k] = d.bc_hi[k] = -1;
  d.gmres_max_inner = m;
  lmfhd_ctx* x = nullptr;
  if (lmfhd_ctx_create(&d, &x) != LMFHD_OK) {
    printf("no context: %s\n", lmfhd_last_error());
    return 1;
  }
  Ctx& c = x->c;
  std::mt19937 gen(7 + lost);
  std::uniform_real_distribution<double> pm(-1.0, 1.0);
  // vectors within the first `lost` entries up to step `lost`: the basis spans them then
  auto draw = [&](int i, double* w) {
    for (long e = 0; e < c.vlen; ++e) w[e] = (i > lost || e < lost) ? pm(gen) : 0.0;
    if (i == lost) w[lost] = 1e-17;
  };
  draw(0, c.r);
  const double beta = vnorm(c, c.r);
  scale_div(c.s, c.V, c.r, c.s_tmp(), c.vlen);
  lsq_init(c, c.s_tmp(), 0.0, 0.0);
  std::vector<std::vector<double>> H;
  for (int i = 1; i <= m; ++i) {
    draw(i, c.w);
    const std::vector<double> w(c.w, c.w + c.vlen);
    arnoldi(c, c.w, i);
    double st[4];
    lsq_status(c, i, st);
    if ((st[3] != 0.0) != (i == lost)) say(i, "repair flag", st[3]);
    std::vector<double> col(i + 1);
    for (int q = 0; q < i; ++q) col[q] = c.s_h1()[q] + c.s_h2()[q];
    col[i] = c.s_nrm()[0];
    H.push_back(col);
    double e1 = 0.0, e2 = 0.0;
    for (int q = 0; q <= i; ++q)
      e1 = std::max(e1, std::fabs(dot(c, c.V + (long)q * c.vs, c.V + (long)i * c.vs) - (q == i)));
    for (long e = 0; e < c.vlen; ++e) {
      double s = 0.0;
      for (int q = 0; q <= i; ++q) s += col[q] * c.V[(long)q * c.vs + e];
      e2 = std::max(e2, std::fabs(s - w[e]));
    }
    // rounding: some 30 products of unit vectors of 208 entries
    if (!(e1 < 1e-13)) say(i, "products of the basis off by", e1);
    if (!(e2 < 1e-13)) say(i, "w off by", e2);
    const double est = least_squares(beta, H);
    if (!(std::fabs(st[0] - est) < 1e-12 * beta)) say(i, "residual estimate off by", st[0] - est);
  }
  lmfhd_ctx_destroy(x);
  return bad;
}

int main() {
  int bad = 0;
  for (int lost : {2, 9, 14, 15}) bad += run(lost, 20);
  printf("%d failures\n", bad);
  return bad != 0;
}
