// Host-side code of libteuk run under AddressSanitizer and
// UndefinedBehaviorSanitizer (tests/test_host_sanitizers.py builds it with
// g++ -fsanitize=address,undefined and runs it): the grid inversions, the
// coefficient and projection tables, the source preparation and T4
// coefficients, the trajectory generator over steep, fast, near-polar and
// high-spin worldlines, the stage kernels' theta-chunk layout and block
// order, and the tiles of resident stepping.  Every output must be finite; any out-of-bounds
// access or undefined operation aborts the run.
#include <cmath>
#include <cstdio>
#include <vector>

#include "teuk.h"
#include "teuk_internal.h"

namespace {

int failures = 0;

void check_finite(const char *what, const double *v, size_t n) {
  for (size_t i = 0; i < n; i++)
    if (!std::isfinite(v[i])) {
      std::printf("non-finite %s[%zu]\n", what, i);
      failures++;
      return;
    }
}

void grids_and_tables(int N, int M, double xmin, double xmax, double a, double m) {
  using namespace teuk;
  const double dx = (xmax - xmin) / N;
  std::vector<double> x(N), r(N), th(M), xh(N), rh(N);
  host_grid(N, M, xmin, xmax, 1.0, a, x.data(), r.data(), th.data());
  host_grid_half(N, xmin, xmax, 1.0, a, xh.data(), rh.data());
  check_finite("r_c", r.data(), N);
  check_finite("r_h", rh.data(), N);
  std::vector<double> ktab((size_t)kNK * N), rtab((size_t)kNR * M);
  host_coeff_tables(N, M, xmin, xmax, dx, 1.0, a, m, r.data(), th.data(), ktab.data(), rtab.data(), 0.0, false);
  host_coeff_tables(N, M, xmin, xmax, dx, 1.0, a, m, rh.data(), th.data(), ktab.data(), rtab.data(), -0.5, true);
  std::vector<double> w((size_t)7 * 5 * (M / 4) * 3), ph(2 * (size_t)N);
  host_projection_weights(M, m, w.data());
  check_finite("projection weights", w.data(), w.size());
  host_source_phase(N, 1.0, a, m, r.data(), ph.data());
}

void trajectory_and_source(double a, double eta, double iota_deg, double dt_out, double t_final) {
  using namespace teuk;
  const int cap = (int)(t_final / dt_out) + 8;
  std::vector<double> rows((size_t)cap * 10);
  int n = 0;
  const int rc = teuk_traj_plunge(a, eta, iota_deg * M_PI / 180.0, 1.02, dt_out, t_final, 7, rows.data(), cap, &n);
  if (rc != TEUK_OK || n < 2) {
    std::printf("trajectory a=%g eta=%g iota=%g failed (%d)\n", a, eta, iota_deg, rc);
    failures++;
    return;
  }
  check_finite("trajectory", rows.data(), (size_t)n * 10);
  // source preparation and T4 coefficients along the worldline (one row in
  // every 64), on a grid that holds the particle
  Grid g{};
  g.N = 4096;
  g.M = 64;
  g.ptsx = g.ptsy = 128;
  g.xmin = -400.0;
  g.xmax = 1200.0;
  g.dx = (g.xmax - g.xmin) / g.N;
  g.dtheta = 3.14159265358979 / g.M;
  g.dt = 0.5 * g.dx;
  g.mass = 1.0;
  g.a = a;
  g.m = 2.0;
  for (int k = 1; k < n; k += 64) {
    const double *q = &rows[10 * (size_t)k];
    if (!(q[1] > 1.0 + std::sqrt(1.0 - a * a) + 1e-3)) break;   // at the horizon
    SrcStep st{};
    st.timer = q[0];
    st.start = 0.0;
    st.rp = q[1];
    st.tp = q[2];
    st.drdt = q[3];
    st.dthdt = q[4];
    st.dphidt = q[5];
    st.phip = q[6];
    st.E = q[7];
    st.lz = q[8];
    st.Q = q[9];
    SrcPrep prep;
    host_source_prepare(g, st, prep);
    double c[12];
    teuk_t4::t4_coeffs(prep.in, c);
    check_finite("T4 coefficients", c, 12);
  }
}

// The stage kernels' theta chunks (theta_chunks, theta_chunk_b0) cover the
// rows 0 .. M-1 once and compute the rows 3 .. M-4 once, each edge chunk
// holding the two rows it extrapolates from, for every M the solver accepts;
// the single-solve block order (stage_block_tile) visits every (strip,
// block-row) once, in both orders.
void chunk_layout_and_block_order() {
  using namespace teuk;
  for (int M = 16; M <= 1024; M += 8)
    for (int R : {2, 4, 8}) {
      const int nc = theta_chunks(M, R), E = edge_rows(R);
      std::vector<int> spanned(M, 0), computed(M, 0);
      for (int c = 0; c < nc; c++) {
        const bool first = c == 0, last = c == nc - 1;
        const int b0 = theta_chunk_b0(M, R, c), span = (first || last) ? E + 3 : R;
        const int c0 = b0 + (first ? 3 : 0), c1 = b0 + (last ? span - 3 : span);   // computed rows [c0, c1)
        if (b0 < 0 || b0 + span > M) {
          std::printf("chunk %d of M=%d R=%d outside the grid\n", c, M, R);
          failures++;
          continue;
        }
        for (int r = b0; r < b0 + span; r++) spanned[r]++;
        for (int r = c0; r < c1; r++) computed[r]++;
        if ((first && !(c0 <= 3 && 4 < c1)) || (last && !(c0 <= M - 5 && M - 4 < c1))) {
          std::printf("edge chunk %d of M=%d R=%d lacks its extrapolation rows\n", c, M, R);
          failures++;
        }
      }
      for (int r = 0; r < M; r++)
        if (spanned[r] != 1 || computed[r] != (r >= 3 && r < M - 3 ? 1 : 0)) {
          std::printf("row %d of M=%d R=%d: spanned %d, computed %d times\n", r, M, R, spanned[r], computed[r]);
          failures++;
          break;
        }
    }
  for (int S : {1, 2, 3, 5, 8, 12, 16, 24, 40, 64, 256})
    for (int ng = 1; ng <= 40; ng++)
      for (bool edge_first : {false, true}) {
        std::vector<int> seen((size_t)S * ng, 0);
        for (int b = 0; b < S * ng; b++) {
          int strip = -1, grp = -1;
          stage_block_tile(b, S * ng, ng, edge_first, strip, grp);
          if (strip < 0 || strip >= S || grp < 0 || grp >= ng) {
            std::printf("block %d of %dx%d maps outside\n", b, S, ng);
            failures++;
            return;
          }
          seen[(size_t)strip * ng + grp]++;
        }
        for (int v : seen)
          if (v != 1) {
            std::printf("block order %dx%d (edge first %d) is not a permutation\n", S, ng, (int)edge_first);
            failures++;
            break;
          }
      }
}

// Tiles of resident stepping: every column in one block, at least 8 in each
// (edge columns, rho fill), as many threads' columns as the tile has, LDS and
// the borrowed buffers (exchange slots in the two stage buffers of 4 N M
// doubles, flags and constants in the set-up plane) large enough.
void resident_tiles(int cus) {
  using namespace teuk;
  for (int M = 8; M <= 136; M += 8)
    for (int N = 128; N <= 131072; N += (N < 4096 ? 64 : (N < 20000 ? 832 : 4096))) {
      ResShape sh{0, 0, 0};
      const bool ok = resident_shape(N, M, cus, sh);
      if (!ok) {
        if (M >= 16 && M <= 64 && (long long)N * M <= 400000 && cus >= 256) {
          std::printf("no resident tile for %dx%d\n", N, M);
          failures++;
        }
        continue;
      }
      const int rest = N - (sh.B - 1) * sh.C;
      const bool sweep = sh.CP >= 4;
      const int edges = sh.CP == 1 && res_pair(M, sh.C) && sh.C >= 16 ? 16 : 8;   // columns a block publishes
      const size_t xbytes = 2 * (size_t)sh.B * edges * 32 * M, cbytes = sweep ? 24 * (size_t)N * M : 0;
      const size_t NM32 = 32 * (size_t)N * M;
      const bool good = M >= 16 && M <= 128 && sh.B <= cus && sh.C % 8 == 0 && sh.C >= res_least_tile(M, sh.CP) && rest >= 8 && rest <= sh.C &&
                        res_groups(M, sh.CP) >= (sweep ? 4 : 8) && res_groups(M, sh.CP) * sh.CP >= sh.C &&
                        res_lds_bytes(M, sh.C, sh.CP) <= kResLdsMax && xbytes <= (sweep ? NM32 : 2 * NM32) &&
                        cbytes <= NM32 && 128 * (size_t)sh.B + 64 * (size_t)N <= 8 * (size_t)N * M;
      if (!good) {
        std::printf("bad resident tile %dx%d: C %d B %d CP %d\n", N, M, sh.C, sh.B, sh.CP);
        failures++;
      }
    }
}

// Segments of grids beyond the chip: their own columns tile the grid, each
// launch reaches as far beside them as its steps do (or to the grid's edge),
// is one that its kernel takes, and finds room in the borrowed buffers.
void resident_spans(int cus) {
  using namespace teuk;
  int planned = 0;
  for (int M = 8; M <= 136; M += 8)
    for (int N = 1024; N <= 131072; N += (N < 20000 ? 1600 : 5824))
      for (int integ = 0; integ < 2; integ++) {
        const ResSegments r = resident_segments(N, M, integ, cus);
        if (r.spans.empty()) continue;
        planned++;
        const int H = 4 * (integ ? 4 : 3) * r.steps, C = r.sh.C, CP = r.sh.CP, k = (int)r.spans.size();
        bool good = M >= 16 && M <= 128 && r.steps >= 1 && r.steps <= kRing && k >= 2 && k <= kMaxSegments &&
                    r.sh.B <= cus && C % 8 == 0 && C >= res_least_tile(M, CP) && res_groups(M, CP) * CP >= C &&
                    res_lds_bytes(M, C, CP) <= kResLdsMax;
        int at = 0;
        for (int i = 0; i < k; i++) {
          const ResSpan &sp = r.spans[i];
          const int len = sp.s1 - sp.s0, B = (len + C - 1) / C;
          good = good && sp.v0 == at && sp.v1 > sp.v0 && sp.s0 == (sp.v0 > H ? sp.v0 - H : 0) &&
                 sp.s1 == (sp.v1 + H < N ? sp.v1 + H : N) && B <= r.sh.B && len - (B - 1) * C >= 8 && len % 8 == 0 &&
                 sp.flag_blk >= i * r.sh.B && 512LL * B * M + 24LL * len * M <= 32LL * N * M &&
                 128LL * (sp.flag_blk + B) + 16 * kMaxSegments <= 16LL * N;
          at = sp.v1;
        }
        if (!good || at != N) {
          std::printf("bad segments for %dx%d integrator %d on %d CUs\n", N, M, integ, cus);
          failures++;
        }
      }
  if (cus == 256 && planned < 20) {
    std::printf("only %d grids in segments\n", planned);
    failures++;
  }
}

// Launches of a batch: every member that fits on the chip in exactly one, at
// most one block per CU, a tile that its kernel takes for every member.
void resident_batches(int cus) {
  using namespace teuk;
  unsigned long long rng = 12345;
  auto next = [&](int n) { rng = rng * 6364136223846793005ULL + 1442695040888963407ULL; return (int)((rng >> 33) % n); };
  static const int kM[] = {16, 24, 32, 40, 48, 64, 72, 128};
  for (int trial = 0; trial < 300; trial++) {
    std::vector<std::pair<int, int>> shapes;
    const int n = next(24), same = next(3) == 0 ? 8 * (2 + next(8)) : 0;
    for (int i = 0; i < n; i++) shapes.push_back({64 * (2 + next(next(2) ? 300 : 60)), same ? same : kM[next(8)]});
    std::vector<int> seen(n, 0);
    bool good = true;
    for (const ResGroup &g : resident_groups(shapes, cus)) {
      int nb = 0;
      for (size_t m = 0; m < g.members.size(); m++) {
        const int i = g.members[m], C = g.C[m], N = shapes[i].first, M = shapes[i].second;
        const int rest = N - ((N + C - 1) / C - 1) * C;
        seen[i]++;
        nb += (N + C - 1) / C;
        good = good && C >= res_least_tile(M, g.CP) && C % 8 == 0 && rest >= 8 && res_groups(M, g.CP) * g.CP >= C &&
               res_lds_bytes(M, C, g.CP) <= kResLdsMax && g.MT == res_built_rows(M, g.CP);
      }
      good = good && nb <= cus && !g.members.empty();
    }
    for (int i = 0; i < n; i++) {
      ResShape sh;
      good = good && seen[i] == (resident_shape(shapes[i].first, shapes[i].second, cus, sh) ? 1 : 0);
    }
    if (!good) {
      std::printf("bad resident launches for a batch of %d (trial %d, %d CUs)\n", n, trial, cus);
      failures++;
    }
  }
}

// A resident launch's wait in ticks: none for 0, else positive and bounded
// for every number of seconds.
void resident_waits() {
  using namespace teuk;
  const long long most = (long long)(kResWaitMost * 1e8) + 1;
  bool good = res_wait_ticks(0.0) == 0 && res_wait_ticks(0.25) == 25000001 && res_wait_ticks(5e-324) == 1;
  for (double s : {1e-9, 59.9, 60.0, 61.0, 9.3e10, 1e300, (double)INFINITY}) {
    const long long t = res_wait_ticks(s);
    good = good && t >= 1 && t <= most && (s < kResWaitMost || t == most);
  }
  good = good && res_shared_wait({10.0, 2.0, 30.0}) == 2.0 && res_shared_wait({5.0}) == 5.0 &&
         res_shared_wait({kResWait, 0.0}) == 0.0;
  if (!good) {
    std::printf("bad resident wait\n");
    failures++;
  }
}

}  // namespace

int main() {
  resident_waits();
  chunk_layout_and_block_order();
  grids_and_tables(1024, 32, -100.0, 300.0, 0.5, 2.0);
  grids_and_tables(512, 16, -40.0, 60.0, 0.99, -3.0);
  grids_and_tables(256, 64, -50.0, 50.0, 1e-8, 0.0);
  grids_and_tables(256, 16, -100.0, 300.0, 0.0, 1.0);
  const double cases[][3] = {{0.9, 1e-3, 30.0}, {0.0926, 8.4e-3, 85.0}, {0.9366, 7.4e-3, 84.0},
                             {0.99, 1e-2, 60.0}, {0.0, 1e-4, 0.0}, {0.7, 1.3e-3, 0.0}, {0.6, 4.1e-3, 85.0}};
  for (const auto &c : cases) trajectory_and_source(c[0], c[1], c[2], 0.05, 600.0);
  double X, dX;
  for (double L = -40.0; L <= 3.4; L += 0.37)
    if (teuk_ot_transition(L, &X, &dX) != TEUK_OK || !std::isfinite(X) || !std::isfinite(dX)) failures++;
  for (int cus : {256, 64, 8}) {
    resident_tiles(cus);
    resident_spans(cus);
    resident_batches(cus);
  }
  std::printf("host checks: %d failures\n", failures);
  return failures == 0 ? 0 : 1;
}
