// Host plan of the far field through spherical harmonics (harmonic.hpp): the
// degrees of every radial node and the constant matrices of the transforms.
#pragma once

#include "harmonic.hpp"
#include "numerics.hpp"
#include "runtime.hpp"

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <type_traits>
#include <vector>

namespace glst {

// Truncation: the terms left out of a plane wave over the unit ball sum to at
// most this (a bound that is about a hundred times the error that is met).
// FP32 products round at 6e-8, FP64 at 1e-16.
constexpr double kHarmEps32 = 3e-7;
constexpr double kHarmEps64 = 1e-15;
// Systems with fewer (atom, node) pairs keep the direct sums: those are the
// direct sums' work, while the passes here take 0.2 (mixed) to 0.5 ms (FP64)
// however small the grid.  Measured in us per step, expansion against direct
// sums: mixed 1,000 waters at tol 1e-5 (1.7e8 pairs) 334 to 333, 3,300 at 1e-4
// (2.5e8) 272 to 317, 1,000 at 1e-6 (4e8) 461 to 517; FP64 1,000 at 1e-5 725
// to 749 but 3,300 at 1e-4 525 to 528 and 1,800 at 1e-4 (1.3e8) 479 to 385,
// 5,500 at 1e-4 (4e8) 828 to 858, 1,000 at 1e-6 1,213 to 1,403.
constexpr double kHarmPairs32 = 2e8, kHarmPairs64 = 3e8;
// So do dilute ones: the direct sums cost (atom, node) work, the expansion
// (cell, node) work, whatever the cells hold.  Fewest atoms per cell on grids
// of up to 512 cells, where the direct sums' launches leave the device partly
// idle, and beyond.  Steps in ms, expansion against direct sums, at so many
// atoms per cell: mixed 6^3 cells (tol 1e-6) 0.75 to 0.88 at 10, 8^3 (1e-5)
// 0.70 to 0.84 at 5; 10^3 (1e-4) 0.56 to 0.66 at 22, 15^3 1.24 to 1.27 at 22,
// 1.22 to 1.07 at 12, 1.22 to 0.98 at 6.  FP64 6^3 2.14 to 2.53 at 23 and to
// 1.67 at 10, 8^3 2.31 to 2.82 at 21 and to 2.09 at 11; 10^3 1.39 to 2.05 at
// 39, 1.29 to 1.30 at 22, 15^3 3.63 to 3.51 at 22, 3.60 to 2.31 at 12.
constexpr uint32_t kHarmSmallGrid = 512;
constexpr double kHarmFill32[2] = {0.0, 22.0}, kHarmFill64[2] = {17.0, 24.0};

// j_0(z) .. j_{n-1}(z), z > 0: Miller's backward recurrence j_{m-1} =
// (2m + 1) / z j_m - j_{m+1} from well above max(n, z), normalised by
// sum_m (2m + 1) j_m^2 = 1 and the sign of j_0 = sin z / z (or of j_1 where
// j_0 is small).
inline std::vector<double> spherical_bessel(double z, uint32_t n) {
  const double big = std::max(static_cast<double>(n), z);
  const uint32_t top = static_cast<uint32_t>(big) + 30 +
                       static_cast<uint32_t>(std::sqrt(40.0 * big));
  std::vector<long double> b(top + 2, 0.0L);
  b[top] = 1e-150L;
  for (uint32_t m = top; m >= 1; --m) {
    b[m - 1] = (2.0L * m + 1.0L) / z * b[m] - b[m + 1];
    if (std::fabs(b[m - 1]) > 1e150L)
      for (uint32_t k = m - 1; k <= top; ++k) b[k] *= 1e-150L;
  }
  long double norm = 0.0L;
  for (uint32_t m = 0; m <= top; ++m)
    norm += (2.0L * m + 1.0L) * b[m] * b[m];
  norm = std::sqrt(norm);
  const long double j0 = std::sin(static_cast<long double>(z)) / z;
  const long double j1 =
      (j0 - std::cos(static_cast<long double>(z))) / z;
  const long double lead = std::fabs(j0) > std::fabs(j1) ? j0 * b[0] : j1 * b[1];
  if (lead < 0) norm = -norm;
  std::vector<double> j(n);
  for (uint32_t m = 0; m < n; ++m) j[m] = static_cast<double>(b[m] / norm);
  return j;
}

// Degrees needed at z = kappa rho: the smallest N with
// sum_{n >= N} (2n+3) |j_{n+1}(z)| / z (n+1)(n+2)/2 < eps (the last factor
// bounds sum_l (2l+1) |R_n^l P_l|); kHarmMaxN + 1 if more than the kernels
// hold.
inline uint32_t harm_degree(double z, double eps) {
  constexpr uint32_t kTop = dev::kHarmMaxN + 60;
  const std::vector<double> j = spherical_bessel(z, kTop + 2);
  double tail = 0.0;
  uint32_t N = kTop;
  while (N > 1) {
    const double n = N - 1;
    tail += (2 * n + 3) * std::fabs(j[N]) / z * (n + 1) * (n + 2) / 2;
    if (tail >= eps) break;
    --N;
  }
  return N;
}

struct HarmTables {
  bool ok = false;
  std::vector<dev::HarmRad> rad;
  std::vector<dev::HarmGroup> grp;
  std::vector<uint2> mup;
  std::vector<double> leg, legt, trig, trigt, gam, gamt, jac, rec;
  std::vector<double> leg64, legt64, gam64, gamt64;  // mixed (HarmDev)
  std::vector<uint2> lrow64, mup64;
  std::vector<uint4> lrow;
  std::vector<uint2> pair;  // (degree, order tile)
  std::vector<uint32_t> crow, urow, qoff;
  uint32_t rows = 0;
  std::vector<uint2> unit;  // (radial node, ring tile)
  std::vector<uint32_t> node_of_row;  // node (device order) of a fields' row
  uint32_t N = 0, stride = 0;
  double scale = 0.0, smax = 0.0;
  uint32_t hsteps = 0;
  size_t lds_sf = 0, lds_lr = 0;
  // device bytes at `real` per scalar (a little more, for the boundaries)
  size_t bytes(size_t real) const {
    return (leg.size() + legt.size() + trig.size() + trigt.size() +
            gam.size() + gamt.size() + jac.size() + rec.size()) * real +
           (leg64.size() + legt64.size() + gam64.size() + gamt64.size()) * 8 +
           (lrow64.size() + mup64.size()) * sizeof(uint2) +
           rad.size() * sizeof(rad[0]) + grp.size() * sizeof(grp[0]) +
           (mup.size() + pair.size() + unit.size()) * sizeof(uint2) +
           lrow.size() * sizeof(uint4) + (crow.size() + urow.size()) * 4 +
           (node_of_row.size() + 256) * sizeof(double4) +
           26 * 256;
  }
};

// Tables for a grid of cell edge h, or ok = false where the nodes are not
// those of the product rule or need more degrees than the kernels hold.
inline HarmTables plan_harmonic(const NodeTable &nodes, double h,
                                int spherical_rule, bool single) {
  HarmTables T;
  const size_t ng = nodes.kappa.size();
  if (spherical_rule != 0 || ng == 0) return T;
  const double eps = single ? kHarmEps32 : kHarmEps64;
  // positions are scaled by a power of two, which puts the ball's radius in
  // (0.7, 1.42)
  const double rho = dev::cheb_rho(h);
  T.scale = std::exp2(-std::round(std::log2(rho)));
  const long double rs = static_cast<long double>(rho) * T.scale;
  T.smax = static_cast<double>(rs * rs);
  constexpr long double kPi = 3.14159265358979323846264338327950288L;
  // groups: rings and azimuths of the product rule (numerics.cpp)
  std::vector<std::vector<double>> ring_u(ng);
  for (size_t g = 0; g < ng; ++g) {
    dev::HarmGroup G{};
    G.nr = static_cast<uint32_t>(nodes.kappa[g].size());
    G.node0 = nodes.first[g];
    G.h = nodes.sph_m[g] + 1;
    G.equator = nodes.sph_m[g] % 2 == 0 ? 1u : 0u;
    G.nring = (nodes.sph_m[g] + 2) / 2;
    if (G.h > dev::kHarmMaxH) return T;
    const auto &d = nodes.dirs[g];
    if (d.size() != static_cast<size_t>(G.nring) * 2 * G.h -
                        (G.equator ? G.h : 0u))
      return T;
    for (uint32_t j = 0; j < G.nring; ++j)
      ring_u[g].push_back(
          d[G.equator ? (j ? G.h + 2 * G.h * (j - 1) : 0u) : 2 * G.h * j][2]);
    for (uint32_t i = 0; i < G.nr; ++i) {
      const double z = nodes.kappa[g][i] * rho;
      if (!(z > 0.0)) return T;
      const uint32_t N = harm_degree(z, eps);
      if (N > (single ? dev::kHarmMaxN32 : dev::kHarmMaxN)) return T;
      G.N = std::max(G.N, N);
      T.rad.push_back({N, static_cast<uint32_t>(g), i, 0u});
    }
    T.grp.push_back(G);
    for (uint32_t i = 0; i < G.nr; ++i)
      for (uint32_t j = 0; j < d.size(); ++j)
        T.node_of_row.push_back(G.node0 + j * G.nr + i);
  }
  std::stable_sort(T.rad.begin(), T.rad.end(),
                   [](const dev::HarmRad &a, const dev::HarmRad &b) {
                     return a.N > b.N;
                   });
  T.N = T.rad[0].N;
  for (auto &r : T.rad) {
    r.off = T.stride;
    T.stride += 16 * dev::harm_blocks(r.N);
  }
  const uint32_t N = T.N;
  // The atoms' side runs on monic polynomials: the Legendre part M_l = z
  // M_{l-1} - b s M_{l-2} from M_m = 1, s = |d|^2, whose derivative in z is
  // (l^2 - m^2) / (2l - 1) M_{l-1}, and radial polynomials of leading factor 1
  // in x.  Their normalisations are in the tables of the nodes' side: weight[l]
  // [m] times the Legendre functions there, with the radius of the ball to the
  // power -l, and kap[l][p] times the radial matrices.  Recurrences with
  // leading factors would round these in every step, for all atoms alike.
  T.rec.assign(static_cast<size_t>(N + 8) * 64 * 2, 0.0);
  std::vector<std::vector<long double>> weight(N), ra(N), rb(N);
  {
    long double c = std::sqrt(1.0L / (4.0L * kPi));
    for (uint32_t l = 0; l < N; ++l) {
      weight[l].assign(l + 1, 0.0L);
      ra[l].assign(l + 1, 0.0L);
      rb[l].assign(l + 1, 0.0L);
      if (l == 1) c *= std::sqrt(3.0L);
      if (l > 1) c *= std::sqrt((2.0L * l + 1.0L) / (2.0L * l));
      weight[l][l] = c;
      for (uint32_t m = 0; m < l; ++m) {
        const long double L = l, M = m, d = L * L - M * M;
        ra[l][m] = std::sqrt((4 * L * L - 1) / d);
        if (l > m + 1)
          rb[l][m] = std::sqrt((2 * L + 1) * (L + M - 1) * (L - M - 1) /
                               ((2 * L - 3) * d));
        weight[l][m] = weight[l - 1][m] * ra[l][m];
        double *r = &T.rec[(static_cast<size_t>(l) * 64 + m) * 2];
        r[0] = l > m + 1 ? static_cast<double>(((L - 1) * (L - 1) - M * M) /
                                               (4 * (L - 1) * (L - 1) - 1))
                         : 0.0;
        r[1] = static_cast<double>(d / (2 * L - 1));
      }
    }
  }
  // rows of the radial polynomials, and of the moments: per order tile, its
  // degrees in turn
  T.crow.push_back(0);
  T.urow.push_back(0);
  for (uint32_t l = 0; l < N; ++l) {
    T.crow.push_back(T.crow[l] + 4 * dev::harm_psteps(l, N));
    T.urow.push_back(T.urow[l] + (l + 1) * dev::harm_psteps(l, N));
  }
  for (uint32_t t = 0; 8 * t < N; ++t) {
    T.qoff.push_back(T.rows - T.crow[8 * t]);
    T.rows += T.crow[N] - T.crow[8 * t];
    for (uint32_t l = 8 * t; l < N; ++l) T.pair.push_back(make_uint2(l, t));
  }
  // radial polynomials P_p^(0, l+1/2)(x), x = 2 t^2 - 1, scaled to leading
  // factor 1: row p gives (x + c1) v_{p-1} - c2 v_{p-2}
  T.jac.assign(static_cast<size_t>(T.crow[N]) * 2, 0.0);
  std::vector<std::vector<long double>> kap(N);
  for (uint32_t l = 0; l < N; ++l) {
    const long double be = l + 0.5L;
    auto coef = [](long double al, long double b, uint32_t k, long double *c) {
      // P_k = (c0 x + c1) P_{k-1} - c2 P_{k-2}
      if (k == 1) {
        c[0] = (al + b + 2) / 2;
        c[1] = (al - b) / 2;
        c[2] = 0;
        return;
      }
      const long double s = 2 * k + al + b, a = 2 * k * (k + al + b) * (s - 2);
      c[0] = (s - 1) * s * (s - 2) / a;
      c[1] = (s - 1) * (al * al - b * b) / a;
      c[2] = 2 * (k + al - 1) * (k + b - 1) * s / a;
    };
    kap[l].assign(1, 1.0L);
    long double c[3], last = 1.0L;
    for (uint32_t p = 1; p < 4 * dev::harm_psteps(l, N); ++p) {
      double *J = &T.jac[(static_cast<size_t>(T.crow[l]) + p) * 2];
      coef(0, be, p, c);
      J[0] = static_cast<double>(c[1] / c[0]);
      J[1] = static_cast<double>(c[2] / (c[0] * last));
      last = c[0];
      kap[l].push_back(kap[l].back() * c[0]);
    }
  }
  // radial matrices: gam_l[i][p] = 4 pi (-1)^p (2n+3) j_{n+1}(z_i) / z_i
  const uint32_t nrad = static_cast<uint32_t>(T.rad.size());
  std::vector<std::vector<long double>> gn(nrad);
  for (uint32_t i = 0; i < nrad; ++i) {
    const double z = nodes.kappa[T.rad[i].group][T.rad[i].idx] * rho;
    const std::vector<double> j = spherical_bessel(z, T.rad[i].N + 2);
    for (uint32_t n = 0; n < T.rad[i].N; ++n)
      gn[i].push_back(4 * kPi * (2.0L * n + 3) * j[n + 1] / z);
  }
  auto gamma = [&](uint32_t i, uint32_t l, uint32_t p) {
    const uint32_t n = l + 2 * p;
    if (i >= nrad || n >= T.rad[i].N) return 0.0;
    const double v = static_cast<double>(gn[i][n] * kap[l][p]);
    return p % 2 ? -v : v;
  };
  // row R of a chained FP32 product stands for index 4 (R % 4) + R / 4
  // (Harm<float>::perm)
  auto radial = [&](uint32_t l, bool fp32, std::vector<double> &gam,
                    std::vector<double> &gamt) {
    auto perm = [&](uint32_t R) { return fp32 ? 4 * (R & 3u) + (R >> 2) : R; };
    const uint32_t PK = dev::harm_psteps(l, N);
    uint32_t above = 0;  // radial nodes with more than l degrees
    while (above < nrad && T.rad[above].N > l) ++above;
    for (uint32_t i0 = 0; i0 < above; i0 += 16)
      for (uint32_t k = 0; k < PK; ++k)
        for (uint32_t a = 0; a < 64; ++a)
          gam.push_back(gamma(i0 + a % 16, l, 4 * k + a / 16));
    for (uint32_t i0 = 0; i0 < above; i0 += 4)
      for (uint32_t t = 0; t < (PK > 4 ? 2u : 1u); ++t)
        for (uint32_t a = 0; a < 64; ++a)
          gamt.push_back(gamma(i0 + a / 16, l, 16 * t + perm(a % 16)));
    return above;
  };
  auto at = [](const std::vector<double> &v) {
    return static_cast<uint32_t>(v.size() / 64);
  };
  for (uint32_t l = 0; l < N; ++l) {
    uint4 r = make_uint4(at(T.gam), at(T.gamt), 0, 0);
    r.z = radial(l, single, T.gam, T.gamt);
    T.lrow.push_back(r);
    if (single && l < dev::kHarmExactL) {
      T.lrow64.push_back(make_uint2(at(T.gam64), at(T.gamt64)));
      radial(l, false, T.gam64, T.gamt64);
    }
  }
  // Legendre functions on the rings and Fourier matrices
  uint32_t hmax = 0;  // (one launch for all groups)
  for (size_t g = 0; g < ng; ++g) {
    dev::HarmGroup &G = T.grp[g];
    G.mup = static_cast<uint32_t>(T.mup.size());
    G.leg = at(T.leg);
    G.legt = at(T.legt);
    G.legt_k = std::max<uint32_t>(4, (G.nring + 3) / 4);
    const uint32_t nrt = (G.nring + 15) / 16;
    // pl[ring][mu][l], with the sign of (-i)^l: even degrees give the real
    // part, odd ones the imaginary part
    std::vector<double> pl(static_cast<size_t>(G.nring) * G.N * G.N, 0.0);
    std::vector<long double> rsl(G.N, 1.0L);  // rs^-l
    for (uint32_t l = 1; l < G.N; ++l) rsl[l] = rsl[l - 1] / rs;
    for (uint32_t j = 0; j < G.nring; ++j) {
      const long double u = ring_u[g][j];
      const long double st = std::sqrt((1 - u) * (1 + u));
      long double stm = 1.0L;  // st^m
      for (uint32_t m = 0; m < G.N; ++m, stm *= st) {
        long double p1 = weight[m][m] * stm;
        long double p2 = 0;
        for (uint32_t l = m; l < G.N; ++l) {
          if (l > m) {
            const long double p = ra[l][m] * u * p1 - rb[l][m] * p2;
            p2 = p1;
            p1 = p;
          }
          const bool neg = l % 2 == 0 ? (l / 2) % 2 == 1 : ((l - 1) / 2) % 2 == 0;
          pl[(static_cast<size_t>(j) * G.N + m) * G.N + l] =
              static_cast<double>((neg ? -p1 : p1) * weight[l][m] *
                                  rsl[l]);
        }
      }
    }
    auto P = [&](uint32_t j, uint32_t m, uint32_t l) {
      return j < G.nring && l < G.N
                 ? pl[(static_cast<size_t>(j) * G.N + m) * G.N + l]
                 : 0.0;
    };
    // orders below `orders` of every ring tile; returns the length of one
    auto legendre = [&](uint32_t orders, std::vector<double> &leg,
                        std::vector<double> &legt, std::vector<uint2> &off) {
      std::vector<double> one;  // one ring tile
      const uint32_t base = at(legt);
      for (uint32_t rt = 0; rt < nrt; ++rt) {
        one.clear();
        for (uint32_t m = 0; m < orders; ++m)
          for (uint32_t par = 0; par < 2; ++par) {
            const uint32_t l0 = m + ((m ^ par) & 1u);
            const uint32_t n = l0 < G.N ? (G.N - l0 + 1) / 2 : 0u;
            if (rt == 0) off.push_back(make_uint2(at(one), at(legt) - base));
            for (uint32_t k = 0; k < n; k += 4)
              for (uint32_t a = 0; a < 64; ++a)
                one.push_back(P(16 * rt + a % 16, m, l0 + 2 * (k + a / 16)));
            if (rt == 0)
              for (uint32_t i0 = 0; i0 < n; i0 += 16)
                for (uint32_t ks = 0; ks < G.legt_k; ++ks)
                  for (uint32_t a = 0; a < 64; ++a)
                    legt.push_back(
                        P(4 * ks + a / 16, m, l0 + 2 * (i0 + a % 16)));
          }
        leg.insert(leg.end(), one.begin(), one.end());
      }
      return at(one);
    };
    G.leg_n = legendre(G.N, T.leg, T.legt, T.mup);
    if (single) {
      G.mup64 = static_cast<uint32_t>(T.mup64.size());
      G.leg64 = at(T.leg64);
      G.legt64 = at(T.legt64);
      G.leg64_n = legendre(dev::kHarmExactMu, T.leg64, T.legt64, T.mup64);
    }
    std::vector<double> ct(2 * G.h), sn(2 * G.h);
    for (uint32_t k = 0; k < 2 * G.h; ++k) {
      ct[k] = static_cast<double>(std::cos(kPi * k / G.h));
      sn[k] = static_cast<double>(std::sin(kPi * k / G.h));
    }
    // cosine or sine of order 2 m + set at azimuth pi k / h, k <= h / 2
    auto mode = [&](uint32_t k, uint32_t m, uint32_t set, uint32_t cs) {
      const uint32_t mu = 2 * m + set;
      if (2 * k > G.h || mu >= G.N) return 0.0;
      const uint32_t a = mu * k % (2 * G.h);
      return cs ? sn[a] : ct[a];
    };
    G.trig = static_cast<uint32_t>(T.trig.size() / 64);
    G.trig_k = ((G.N + 1) / 2 + 3) / 4;
    G.trig_t = (G.h / 2 + 16) / 16;
    for (uint32_t pt = 0; pt < G.trig_t; ++pt)
      for (uint32_t cs = 0; cs < 2; ++cs)
        for (uint32_t set = 0; set < 2; ++set)
          for (uint32_t k = 0; k < G.trig_k; ++k)
            for (uint32_t a = 0; a < 64; ++a)
              T.trig.push_back(
                  mode(16 * pt + a % 16, 4 * k + a / 16, set, cs));
    G.trigt = static_cast<uint32_t>(T.trigt.size() / 64);
    G.trigt_m = (G.trig_k + 3) / 4;
    G.trigt_k = (G.h / 2 + 4) / 4;
    T.hsteps = std::max(T.hsteps, G.trigt_k);
    hmax = std::max(hmax, G.h);
    for (uint32_t set = 0; set < 2; ++set)
      for (uint32_t cs = 0; cs < 2; ++cs)
        for (uint32_t mt = 0; mt < G.trigt_m; ++mt)
          for (uint32_t k = 0; k < G.trigt_k; ++k)
            for (uint32_t a = 0; a < 64; ++a)
              T.trigt.push_back(
                  mode(4 * k + a / 16, 16 * mt + a % 16, set, cs));
  }
  for (uint32_t i = 0; i < nrad; ++i) {
    const dev::HarmGroup &G = T.grp[T.rad[i].group];
    for (uint32_t rt = 0; rt < (G.nring + 15) / 16; ++rt)
      T.unit.push_back(make_uint2(i, rt));
    T.lds_sf = std::max(T.lds_sf, single
                                      ? dev::harm_lds_sf<float>(T.rad[i].N, hmax)
                                      : dev::harm_lds_sf<double>(T.rad[i].N, hmax));
    T.lds_lr = std::max(
        T.lds_lr, single
                      ? dev::harm_lds_lr<float>(T.rad[i].N, hmax, G.nring)
                      : dev::harm_lds_lr<double>(T.rad[i].N, hmax, G.nring));
  }
  // the kernels load whole groups of steps
  for (auto *t : {&T.leg, &T.legt, &T.gam, &T.gamt, &T.leg64, &T.legt64,
                  &T.gam64, &T.gamt64})
    t->resize(t->size() + 8 * 64, 0.0);
  T.ok = true;
  return T;
}

inline bool harm_worth(uint32_t natom, uint32_t ncell, uint32_t K,
                       bool single) {
  const double fill =
      (single ? kHarmFill32 : kHarmFill64)[ncell > kHarmSmallGrid];
  return static_cast<double>(natom) * K >=
             (single ? kHarmPairs32 : kHarmPairs64) &&
         natom >= fill * ncell;
}

// Whether the shell sums of node-major fields run on tables no worse than
// those of the direct sums' fields: not where only they need the FP64 tables
// in global memory, because the node-major matrix-core kernel takes z slices
// too (mixed grids of up to 16 x 16 cells whose long axis in z leaves no room
// in LDS).  345,000 charges on 16 x 16 x 33 cells: shell sums 10.8 ms against
// 1.8 on the matrix cores, steps 13.8 against 5.0, and 2.5 GB of tables.  Up
// to 32 cells in z the tables fit in LDS and the expansion keeps its gain
// (251,000 charges on 16 x 16 x 24: 3.13 ms against 3.52).
inline bool harm_shell_sums(bool mixed, int rmt_shape,
                            const dev::GridShape &g, size_t lds_limit) {
  auto path = [&](bool nm) {
    return dev::rmt_path(mixed, rmt_shape, g, lds_limit, nm);
  };
  return path(true) == path(false) || path(true) != dev::RmtPath::kGlobal;
}

// Launch sizes for a system of natom atoms in ncell cells; nrad 0 where a
// kernel's LDS does not fit.
inline dev::HarmPlanDev harm_fit(const HarmTables &t, bool single,
                                 size_t lds_limit, uint32_t natom,
                                 uint32_t ncell) {
  dev::HarmPlanDev plan;
  plan.nrad = static_cast<uint32_t>(t.rad.size());
  plan.nunit = static_cast<uint32_t>(t.unit.size());
  plan.hsteps = t.hsteps;
  // room for most cells in one pass, within the LDS and the registers
  const double mean = static_cast<double>(natom) / ncell;
  auto lds = [&](uint32_t ks) {
    return single ? dev::harm_lds_moments<float>(t.N, ks)
                  : dev::harm_lds_moments<double>(t.N, ks);
  };
  plan.ksteps = single ? 16 : mean > 75.0 ? 32 : mean > 48.0 ? 24 : 16;
  while (plan.ksteps > 16 && lds(plan.ksteps) > lds_limit) plan.ksteps -= 8;
  while (plan.nset < 8 && 64.0 * plan.nset < 1.2 * mean) ++plan.nset;
  plan.lds_moments = lds(plan.ksteps);
  plan.lds_sf = t.lds_sf;
  plan.lds_lr = t.lds_lr;
  if (std::max(std::max(plan.lds_moments, plan.lds_sf), plan.lds_lr) >
      lds_limit)
    plan.nrad = 0;
  return plan;
}
// Scalars of the coefficients and of the moments of ncell cells.
inline size_t harm_coef_len(const HarmTables &t, uint32_t ncell) {
  return static_cast<size_t>((ncell + dev::kHarmCells - 1) / dev::kHarmCells) *
         dev::kHarmCells * t.stride;
}
inline size_t harm_mom_len(const HarmTables &t, uint32_t ncell) {
  return (static_cast<size_t>(ncell) * t.rows + 64) * 16;
}

// A plan's tables on the device.
class HarmDevice {
 public:
  bool ok() const { return buf_.bytes() > 0; }
  size_t device_bytes() const { return buf_.bytes(); }
  const uint2 *unit = nullptr;  // HarmPlanDev::unit
  const double4 *k64 = nullptr;  // the nodes in the order of the fields' rows
  template <typename T>
  const dev::HarmDev<T> &dev() const;
  void release() { buf_.release(); }

  void upload(const HarmTables &t, bool single,
              const std::vector<double4> &nodes) {
    // one buffer, every table on a 256-byte boundary
    const size_t room = t.bytes(single ? 4 : 8) + nodes.size() * sizeof(double4);
    const std::unique_ptr<char[]> host(new char[room]);  // (not cleared)
    size_t size = 0;
    auto place = [&](size_t bytes) {
      const size_t at = (size + 255) / 256 * 256;
      size = at + bytes;
      return at;
    };
    auto raw = [&](const void *p, size_t bytes) {
      const size_t at = place(bytes);
      if (bytes) std::memcpy(host.get() + at, p, bytes);
      return at;
    };
    auto real = [&](const std::vector<double> &v) {
      if (!single) return raw(v.data(), v.size() * 8);
      const size_t at = place(v.size() * 4);
      float *f = reinterpret_cast<float *>(host.get() + at);
      for (size_t i = 0; i < v.size(); ++i) f[i] = static_cast<float>(v[i]);
      return at;
    };
    const size_t rad = raw(t.rad.data(), t.rad.size() * sizeof(t.rad[0]));
    const size_t grp = raw(t.grp.data(), t.grp.size() * sizeof(t.grp[0]));
    const size_t mup = raw(t.mup.data(), t.mup.size() * sizeof(uint2));
    const size_t lrow = raw(t.lrow.data(), t.lrow.size() * sizeof(uint4));
    const size_t pair = raw(t.pair.data(), t.pair.size() * sizeof(uint2));
    const size_t crow = raw(t.crow.data(), t.crow.size() * 4);
    const size_t urow = raw(t.urow.data(), t.urow.size() * 4);
    const size_t kat = place(nodes.size() * sizeof(double4));
    double4 *k = reinterpret_cast<double4 *>(host.get() + kat);
    for (size_t r = 0; r < nodes.size(); ++r)
      k[r] = nodes[r < t.node_of_row.size() ? t.node_of_row[r] : r];
    const size_t units = raw(t.unit.data(), t.unit.size() * sizeof(uint2));
    const size_t leg = real(t.leg), legt = real(t.legt);
    const size_t trig = real(t.trig), trigt = real(t.trigt);
    const size_t gam = real(t.gam), gamt = real(t.gamt);
    const size_t jac = real(t.jac), rec = real(t.rec);
    auto fp64 = [&](const std::vector<double> &v) {
      return raw(v.data(), v.size() * 8);
    };
    const size_t leg64 = fp64(t.leg64), legt64 = fp64(t.legt64);
    const size_t gam64 = fp64(t.gam64), gamt64 = fp64(t.gamt64);
    const size_t lrow64 = raw(t.lrow64.data(), t.lrow64.size() * sizeof(uint2));
    const size_t mup64 = raw(t.mup64.data(), t.mup64.size() * sizeof(uint2));
    buf_.resize(size);
    GLST_HIP(hipMemcpy(buf_.as<void>(), host.get(), size,
                       hipMemcpyHostToDevice));
    auto fill = [&](auto &d) {
      using T = std::remove_const_t<std::remove_reference_t<decltype(*d.leg)>>;
      const char *b = buf_.as<char>();
      auto at = [&](size_t o) { return reinterpret_cast<const T *>(b + o); };
      d.rad = reinterpret_cast<const dev::HarmRad *>(b + rad);
      d.grp = reinterpret_cast<const dev::HarmGroup *>(b + grp);
      d.mup = reinterpret_cast<const uint2 *>(b + mup);
      d.lrow = reinterpret_cast<const uint4 *>(b + lrow);
      d.pair = reinterpret_cast<const uint2 *>(b + pair);
      d.crow = reinterpret_cast<const uint32_t *>(b + crow);
      d.urow = reinterpret_cast<const uint32_t *>(b + urow);
      d.leg = at(leg);
      d.legt = at(legt);
      d.trig = at(trig);
      d.trigt = at(trigt);
      d.gam = at(gam);
      d.gamt = at(gamt);
      d.jac = at(jac);
      d.rec = at(rec);
      d.leg64 = reinterpret_cast<const double *>(b + leg64);
      d.legt64 = reinterpret_cast<const double *>(b + legt64);
      d.gam64 = reinterpret_cast<const double *>(b + gam64);
      d.gamt64 = reinterpret_cast<const double *>(b + gamt64);
      d.lrow64 = reinterpret_cast<const uint2 *>(b + lrow64);
      d.mup64 = reinterpret_cast<const uint2 *>(b + mup64);
      d.nrad = static_cast<uint32_t>(t.rad.size());
      d.N = t.N;
      d.stride = t.stride;
      d.npair = static_cast<uint32_t>(t.pair.size());
      d.rows = t.rows;
      d.jrows = t.crow.back();
      d.ustride = 8 * t.urow.back();
      std::copy(t.qoff.begin(), t.qoff.end(), d.qoff);
      d.scale = t.scale;
      d.smax = t.smax;
      d.xk = 2.0 / t.smax;
      unit = reinterpret_cast<const uint2 *>(b + units);
      k64 = reinterpret_cast<const double4 *>(b + kat);
    };
    if (single)
      fill(f_);
    else
      fill(d_);
  }

 private:
  DeviceBuffer buf_;
  dev::HarmDev<float> f_{};
  dev::HarmDev<double> d_{};
};
template <>
inline const dev::HarmDev<float> &HarmDevice::dev<float>() const {
  return f_;
}
template <>
inline const dev::HarmDev<double> &HarmDevice::dev<double>() const {
  return d_;
}

}  // namespace glst
