// Host-side set-up for libteuk: the compactified grid with its Newton
// inversion r(r*), the -2Y_lm projection weights and the trajectory
// consumption pattern of the reference driver.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "teuk_internal.h"

namespace teuk {

// TD_GPU_code/HighOrder/main.c:79-198 from the rho grid on: Omega(rho) = 1
// inside rin = Xmin + 0.64 (Xmax - Xmin) and 1 - ((rho - rin)/(Xmax + 1e-6 -
// rin))^4 beyond, r* = rho/Omega, then Newton on r*(r) - r* = 0 with
// dr*/dr = (r^2+a^2)/Delta, marching inward from the outer edge with each
// point warm-started from its neighbour.
static void host_radii(int N, const double *x, double xmin, double xmax, double mass, double a, double *r_out) {
  const double rin = xmin + (xmax - xmin) * 0.64;
  const double outer = xmax + 1e-6;
  std::vector<double> target(N);
  for (int l = 0; l < N; l++) {
    const double om = (x[l] < rin) ? 1.0 : 1.0 - std::pow((x[l] - rin) / (outer - rin), 4);
    target[l] = x[l] / om;
  }
  if (mass == 0.0) {
    for (int l = 0; l < N; l++) r_out[l] = target[l];
    return;
  }
  const double disc = std::sqrt(mass * mass - a * a);
  const double rp = mass + disc, rm = mass - disc;
  const double tol = 1e-12;
  double r = target[N - 1];
  for (int l = N - 1; l >= 0; l--) {
    double step_rel, r_new;
    do {
      const double jac = (r * r + a * a - 2.0 * mass * r) / (r * r + a * a);
      double rstar;
      if (mass == a)
        rstar = r + 2.0 * a * std::log(r / a - 1.0) - 2.0 * a * a / (r - a);
      else if (a == 0.0)
        rstar = r + 2.0 * mass * std::log(r / (2.0 * mass) - 1.0);
      else
        rstar = r + (rp * rp + a * a) / (rp - rm) * std::log(r / rp - 1.0) -
                (rm * rm + a * a) / (rp - rm) * std::log(r / rm - 1.0);
      r_new = r + (target[l] - rstar) * jac;
      // Past double resolution of r - r+ the reference iteration hits
      // log(0) and returns NaN for every inner point; clamp to r+ (the
      // r* -> -inf limit) there.  Finite reference results are unchanged.
      if (!(r_new > rp)) {
        r_new = rp;
        r = r_new;
        break;
      }
      step_rel = std::fabs(r_new - r) / r;
      r = r_new;
    } while (step_rel > tol);
    r_out[l] = r_new;
  }
}

// main.c:79-198: rho_l = Xmin + l dx, theta_k = k dtheta and the radii.
void host_grid(int N, int M, double xmin, double xmax, double mass, double a, double *x_c, double *r_c,
               double *theta) {
  const double dx = (xmax - xmin) / N;
  const double dth = kPi15 / M;
  for (int l = 0; l < N; l++) x_c[l] = xmin + (double)l * dx;
  for (int k = 0; k < M; k++) theta[k] = (double)k * dth;
  host_radii(N, x_c, xmin, xmax, mass, a, r_c);
}

// The staggered scheme's half points (TD_GPU_code/Old/kern.cu:93 places
// its half-point coefficients at Xmin + (j - 1/2) dx with radius r_h[j]; Old/
// has no main.c, so r_h is the same inversion at those points).
void host_grid_half(int N, double xmin, double xmax, double mass, double a, double *x_h, double *r_h) {
  const double dx = (xmax - xmin) / N;
  for (int l = 0; l < N; l++) x_h[l] = xmin + ((double)l - 0.5) * dx;
  host_radii(N, x_h, xmin, xmax, mass, a, r_h);
}

static double factorial(double n) {
  double f = 1.0;
  for (double c = 1.0; c <= n; c++) f = f * c;
  return f;
}

// proj.c:16-35: -2Y_lm(theta) (phi part dropped) from the Wigner d-matrix sum.
double host_swsh(double ell, double ml, double the) {
  const double tlo = (ml - 2.0) > 0 ? ml - 2.0 : 0.0;
  const double thi = (ell - 2.0) > (ell + ml) ? ml + ell : ell - 2.0;
  double acc = 0.0;
  for (double t = tlo; t <= thi; t++) {
    double c = std::pow(-1.0, t) *
               std::sqrt(factorial(ell + ml) * factorial(ell - ml) * factorial(ell + 2.0) * factorial(ell - 2.0));
    c = c / (factorial(ell + ml - t) * factorial(ell - 2.0 - t) * factorial(t) * factorial(t + 2.0 - ml));
    acc = acc + c * std::pow(std::cos(the / 2.0), 2.0 * ell + ml - 2.0 - 2.0 * t) *
                    std::pow(std::sin(the / 2.0), 2.0 * t + 2.0 - ml);
  }
  return std::sqrt((2.0 * ell + 1.0) / 4.0 / kPi15) * acc;
}

// Factors of the composite Boole rule of proj.c:47-72 for l = |m| .. |m|+6.
// The reference sum has 5 terms per panel (panel joints appear twice, at
// slightly different accumulated theta), so the table holds one entry per
// term t = 5 i + j, evaluated at grid point 4 i + j (point M repeats M-1,
// proj.c:45): (w_j*4*Pi, sin(theta_t), -2Y_lm(theta_t)), with theta_t
// accumulated exactly as the reference does (4 dtheta i, then += dtheta).
void host_projection_weights(int M, double m, double *w) {
  const double dth = kPi15 / M;
  static const double boole[5] = {7.0, 32.0, 12.0, 32.0, 7.0};
  const int am = std::abs((int)m);
  const int nterm = 5 * (M / 4);
  for (int l = 0; l < 7; l++) {
    double *wl = w + (size_t)l * nterm * 3;
    for (int i = 0; i < M / 4; i++) {
      double th = 4.0 * dth * (double)i;
      for (int j = 0; j < 5; j++) {
        if (j > 0) th += dth;
        double *e = wl + 3 * (5 * i + j);
        e[0] = boole[j] * 4.0 * kPi15;
        e[1] = std::sin(th);
        e[2] = host_swsh((double)(l + am), m, th);
      }
    }
  }
}

// Coefficient fields of kernel_init (kern.cu:110-158) split into what depends
// on the rho column only and what depends on the theta row only.  The layer
// function Omega(rho) and its derivatives (kern.cu:119-127), the compactified
// radius eR = Omega r and the Kerr factors are folded into 12 constants per
// column; the device then needs one division and one square root per point.
// Evaluated with the host libm so that the device assembly reproduces the
// host computation bit for bit.
void host_coeff_tables(int N, int M, double xmin, double xmax, double dx, double mass, double a,
                       double m, const double *r, const double *theta, double *ktab, double *rtab, double shift,
                       bool staggered) {
  const double rin = xmin + (xmax - xmin) * 0.64;
  const double outer = xmax + 1e-6;
  const double spin = a, em = m;
  for (int j = 0; j < N; j++) {
    const double x = xmin + ((double)j + shift) * dx;
    double om = 1.0, om1 = 0.0, om2 = 0.0;
    if (!(x < rin)) {
      om = 1.0 - std::pow((x - rin) / (outer - rin), 4);
      om1 = -4.0 * std::pow(x - rin, 3) / std::pow(outer - rin, 4);
      om2 = -12.0 * std::pow(x - rin, 2) / std::pow(outer - rin, 4);
    }
    const double L = om - x * om1;  // Omega^2 d(r*)/d(rho)
    const double R = om * r[j];     // eR of kern.cu:130
    const double a2 = spin * spin, a4 = a2 * a2;
    const double om_2 = om * om, om3 = om_2 * om, om4 = om_2 * om_2, om5 = om4 * om;
    const double S = R * R + om_2 * a2;
    const double D = R * R - 2.0 * R * mass * om + om_2 * a2;
    const double L2 = L * L, L3 = L2 * L;
    const double R2 = R * R, R3 = R2 * R, R5 = R3 * R2;
    double K[kNK];
    K[kK1] = ((2.0 * L - om_2) * (S * S)) / L2;
    K[kK2] = a2 * D;
    K[kKA] = (2.0 * (L - om_2) * (S * S)) / L2;
    K[kKR] = -((om_2 * (S * S)) / L2);
    K[kKD] = D;
    K[kKBt] = -((om * (R3 * (4.0 * L2 * (R - 3.0 * mass * om) + 2.0 * L * R2 * om1 + R2 * om * om2 * x) +
                       2.0 * R *
                           (L2 * om_2 * (5.0 * R - 4.0 * mass * om) - 3.0 * L3 * (R - 2.0 * mass * om) +
                            2.0 * L * R2 * om_2 * om1 + R2 * om3 * om2 * x) *
                           a2 +
                       (-6.0 * L3 * om_2 + 6.0 * L2 * om4 + 2.0 * L * R * om4 * om1 + R * om5 * om2 * x) * a4)) /
                (L3 * R));
    K[kKBr] = -((om * (R5 * (2.0 * om * om1 - 2.0 * om1 * om1 * x + om * om2 * x) +
                       2.0 * R3 * om_2 * (2.0 * om * om1 - 2.0 * om1 * om1 * x + om * om2 * x) * a2 +
                       om4 * (6.0 * om_2 + 2.0 * om1 * om1 * x * (-R + 3.0 * x) +
                              om * (2.0 * R * om1 - 12.0 * om1 * x + R * om2 * x)) *
                           a4 +
                       2.0 * L2 * R * (2.0 * R3 - 6.0 * R2 * mass * om + 5.0 * R * om_2 * a2 - 4.0 * mass * om3 * a2))) /
                (L3 * R));
    K[kKC0] = (D * (2.0 * R2 + 6.0 * R * mass * om - 6.0 * om_2 * a2)) / R2;
    K[kKI0] = (2.0 * spin * (em * (-(om_2 * S) + L * (R2 + 2.0 * R * mass * om + om_2 * a2)))) / L;
    K[kKI1] = 4.0 * spin * D;
    K[kKBi] = (-2.0 * em * om_2 * spin * S) / L;
    K[kKCi] = (2.0 * em * om * spin * (R2 + 2.0 * R * mass * om - 3.0 * om_2 * a2)) / R;
    for (int i = 0; i < kNK; i++) ktab[(size_t)i * N + j] = K[i];
  }
  for (int k = 0; k < M; k++) {
    const double y = theta[k];
    const double sn = std::sin(y), cs = std::cos(y);
    const double cot = 1.0 / std::tan(y), csc = 1.0 / std::sin(y);
    rtab[k] = sn * sn;
    rtab[M + k] = cs;
    rtab[2 * M + k] = 4.0 * (cot * cot) - 4.0 * em * cot * csc + (em * em) * (csc * csc);
    rtab[3 * M + k] = staggered ? cs / sn : std::tan(0.5 * kPi15 - y);  // Old/kern.cu:241-243, kern.cu:204
  }
}

// kern.cu:2671-2672: the source picks up e^{-i m a/(r+ - r-) ln((r - r+)/(r - r-))},
// evaluated at the grid radius of each column.
void host_source_phase(int N, double mass, double a, double m, const double *r_c, double *phase) {
  const double rpl = mass + std::sqrt(mass * mass - a * a);
  const double rmi = mass - std::sqrt(mass * mass - a * a);
  for (int j = 0; j < N; j++) {
    const double r = r_c[j];
    double arg = 0.0;
    if (a != 0.0) arg = -m * a / (rpl - rmi) * std::log((r - rpl) / (r - rmi));
    phase[j] = std::cos(arg);
    phase[N + j] = std::sin(arg);
  }
}

// kern.cu:1186-1206 and 2673 for one step: the patch origin from the
// particle's tortoise radius and theta, the radial Gaussian width
// wr = 2 dx (1 - r+/r_p), the turn-on (1 - e^{-(t - t0)/25})^4, and the
// transcendental inputs of the T_4 coefficients.  For a = 0 the tortoise
// radius uses its Schwarzschild form (the reference's Kerr form is 0 * inf
// there).
void host_source_prepare(const Grid &g, const SrcStep &st, SrcPrep &out) {
  const double a = g.a, mass = g.mass;
  const double rpl = mass + std::sqrt(mass * mass - a * a);
  const double rmi = mass - std::sqrt(mass * mass - a * a);
  double xp;
  if (a != 0.0)
    xp = st.rp + (rpl * rpl + a * a) / (rpl - rmi) * std::log(st.rp / rpl - 1.0) -
         (rmi * rmi + a * a) / (rpl - rmi) * std::log(st.rp / rmi - 1.0);
  else
    xp = st.rp + 2.0 * mass * std::log(st.rp / (2.0 * mass) - 1.0);
  const int ip = (int)((xp - g.xmin) / g.dx);
  const int it = (int)(st.tp / g.dtheta);
  SrcDev &d = out.dev;
  for (int i = 0; i < 12; i++) d.c[i] = 0.0;
  d.rp = st.rp;
  d.tp = st.tp;
  d.wr = (2.0 * g.dx) * (1.0 - rpl / st.rp);
  d.turnon = std::pow(1.0 - std::exp(-(st.timer - st.start) / 25.0), 4);
  d.ip0 = ip - g.ptsx / 2;
  d.it0 = it - g.ptsy / 2;
  teuk_t4::StepIn &in = out.in;
  in.mass = mass;
  in.a = a;
  in.E = st.E;
  in.lz = st.lz;
  in.nmu = 1.0;  // kern.cu:1190
  in.mm = g.m;
  in.rp = st.rp;
  in.drdt = st.drdt;
  in.d2rdt2 = st.d2rdt2;
  in.dthdt = st.dthdt;
  in.d2thdt2 = st.d2thdt2;
  in.dphidt = st.dphidt;
  in.d2phidt2 = st.d2phidt2;
  in.stp = std::sin(st.tp);
  in.ctp = std::cos(st.tp);
  in.cmphi = std::cos(g.m * st.phip);
  in.smphi = std::sin(g.m * st.phip);
}

// The fewest columns per block (a multiple of 8, so that the last block holds
// at least 8 too: its edge columns and what the rho fill reads) that put the
// grid on the chip with one block per CU: the narrowest tiles were the fastest
// at every size (4096x32 RK4: 16 columns 2.5 us a stage, 32 2.9, 64 5.1;
// 2048x64: 8 columns 3.2, 16 3.5, 32 5.3).  A tile that needs more than eight
// columns per thread, or more LDS than a CU has, does not fit; nor does a
// column of more than 128 rows, which must lie within two waves.
bool resident_shape(int N, int M, int cus, ResShape &sh) {
  if (M > 2 * kWave || M < 16 || M % 8 != 0 || N % 8 != 0 || cus < 1) return false;
  const int fit = std::max(8, (((N + cus - 1) / cus) + 7) & ~7);
  for (int CP : kResCP) {
    const int C = std::max(fit, res_least_tile(M, CP));
    if (res_groups(M, CP) * CP < C || res_lds_bytes(M, C, CP) > kResLdsMax) continue;
    sh = ResShape{C, (N + C - 1) / C, CP};
    return true;
  }
  return false;
}

// Measured time of one stage with tiles of kResCP[c] columns per thread (us).
// Columns of 72 to 128 rows take 5.8, 7.9 and 9.5 with 4, 6 and 8, 5 to 8 %
// more than 64 rows' (there are no tiles of 1 or 2): which width is the
// cheapest does not change by it.
static double stage_us(int M, int c) {
  static const double k32[5] = {2.5, 2.9, 5.2, 7.2, 8.9}, k64[5] = {3.2, 3.5, 5.4, 7.6, 8.9};
  return M <= 32 ? k32[c] : k64[c];
}

// The widest tile of CP columns per thread (0: none).
static int widest_tile(int M, int CP) {
  int C = (res_groups(M, CP) * CP) & ~7;
  while (C >= 8 && res_lds_bytes(M, C, CP) > kResLdsMax) C -= 8;
  return C >= res_least_tile(M, CP) ? C : 0;
}

// A launch takes as long as its tiles, whatever they belong to, so members
// share launches, and wide tiles put more of them into one.  For the members
// of each row class (the row counts kernels are built for, others together)
// the tile width with the least sum of stage_us over its launches is taken,
// the launches filled in order of size, and each launch's tiles then narrowed
// as far as the CUs allow.
std::vector<ResGroup> resident_groups(const std::vector<std::pair<int, int>> &shapes, int cus) {
  std::vector<ResGroup> out;
  for (int cls : {32, 64, 128, kAnyTall, 0}) {
    std::vector<int> own;
    int tallest = 0;
    for (size_t i = 0; i < shapes.size(); i++) {
      const int M = shapes[i].second;
      ResShape sh;
      if (res_built_rows(M, 8) != cls || !resident_shape(shapes[i].first, M, cus, sh)) continue;
      own.push_back((int)i);
      tallest = std::max(tallest, M);
    }
    std::stable_sort(own.begin(), own.end(), [&](int x, int y) {
      return (long long)shapes[x].first * shapes[x].second > (long long)shapes[y].first * shapes[y].second;
    });
    // a member's tile of about `want` columns, and its blocks
    auto tile = [&](int i, int CP, int want) {
      const int M = shapes[i].second;
      return std::min(widest_tile(M, CP), std::max(want, res_least_tile(M, CP)));
    };
    auto blocks = [&](int i, int CP, int want) {
      const int C = tile(i, CP, want);
      return C ? (shapes[i].first + C - 1) / C : cus + 1;
    };
    auto total = [&](const std::vector<int> &m, int CP, int want) {
      long long nb = 0;
      for (int i : m) nb += blocks(i, CP, want);
      return nb;
    };
    const int kWide = 1 << 20;
    std::vector<std::vector<int>> best;
    double best_cost = 0.0;
    for (int c = 0; c < 5 && !own.empty(); c++) {
      std::vector<std::vector<int>> bins;
      std::vector<int> used;
      for (int i : own) {
        const int nb = blocks(i, kResCP[c], kWide);
        size_t k = 0;
        while (k < bins.size() && used[k] + nb > cus) k++;
        if (k == bins.size()) {
          bins.push_back({});
          used.push_back(0);
        }
        bins[k].push_back(i);
        used[k] += nb;
      }
      const bool fits = *std::max_element(used.begin(), used.end()) <= cus;
      const double cost = (double)bins.size() * stage_us(tallest, c);
      if (fits && (best.empty() || cost < best_cost)) {
        best = bins;
        best_cost = cost;
      }
    }
    for (std::vector<int> &m : best) {
      ResGroup g;
      g.CP = 8;
      for (int c = 4; c >= 0; c--)
        if (total(m, kResCP[c], kWide) <= cus) g.CP = kResCP[c];
      int want = 8;
      while (total(m, g.CP, want) > cus) want += 8;
      for (int i : m) g.C.push_back(tile(i, g.CP, want));
      g.members = std::move(m);
      g.MT = g.CP >= 4 || cls == 32 || cls == kWave ? cls : 0;   // (res_built_rows of all members)
      out.push_back(g);
    }
  }
  return out;
}

// Tiles of each width and 4 to 32 steps a launch: the segments cover the
// columns beside them that the steps reach (H on each inner side), so fewer
// steps mean less to compute twice and more launches, each about 25 us of
// loads, stores and set-up.  The per-stage kernels take about 19.5 us a stage
// and million points (16 to 23 over 12288x72 ... 65536x96); the plan must beat
// that by a tenth (16384x96: 23.5 us a stage in segments, 25.1 by stages;
// 16384x72, by stages: 20.3).
ResSegments resident_segments(int N, int M, int integrator, int cus) {
  ResSegments best;
  ResShape whole;
  if (M > 2 * kWave || M < 16 || M % 8 != 0 || N % 8 != 0 || cus < 1 || resident_shape(N, M, cus, whole)) return best;
  const int S = integrator == 0 ? 3 : 4;
  double best_cost = 0.9 * S * 19.5e-6 * (double)N * M;
  for (int c = 2; c < 5; c++) {
    const int C = widest_tile(M, kResCP[c]);
    for (int steps = 4; C && steps <= kRing; steps *= 2) {
      const int cap = C * cus, H = 4 * S * steps;
      if (cap <= 2 * H) continue;
      int k = 2;
      while (2LL * (cap - H) + (long long)(k - 2) * (cap - 2 * H) < N) k++;
      const double cost = k * (S * stage_us(M, c) + 25.0 / steps);
      if (k > kMaxSegments || cost >= best_cost) continue;
      const int w = ((N - 2 * H + k - 1) / k + 7) & ~7;   // an inner segment's own columns; the outer ones' are H more
      ResSegments r;
      r.steps = steps;
      bool good = w >= 8;
      int widest = 0;
      for (int i = 0, v0 = 0; i < k && good; i++) {
        const int v1 = i == k - 1 ? N : std::min(N, v0 + w + (i == 0 ? H : 0));
        ResSpan sp{std::max(0, v0 - H), std::min(N, v1 + H), v0, v1, nullptr, nullptr, nullptr, 0};
        widest = std::max(widest, sp.s1 - sp.s0);
        good = v1 > v0 && sp.s1 - sp.s0 <= cap;
        r.spans.push_back(sp);
        v0 = v1;
      }
      const int Cn = std::max(res_least_tile(M, kResCP[c]), (((widest + cus - 1) / cus) + 7) & ~7);
      r.sh = ResShape{Cn, (widest + Cn - 1) / Cn, kResCP[c]};
      for (int i = 0; i < k && good; i++) r.spans[i].flag_blk = i * r.sh.B;
      // the stage buffer that holds exchange slots and coefficient values; the flags' place
      good = good && Cn <= C && 512LL * r.sh.B + 24LL * widest <= 32LL * N &&
             128LL * k * r.sh.B + 16 * kMaxSegments <= 16LL * N;
      if (!good) continue;
      best = r;
      best_cost = cost;
    }
  }
  return best;
}

}  // namespace teuk
