// Host check of the far field's harmonic tables (harmonic_plan.hpp): at random
// points of a cell's ball, a plane wave of every radial node at directions of
// the upper half sphere, put together from the tables (recurrences of the
// Legendre and radial parts, radial, Legendre and Fourier matrices), against
// cos and sin of the phase; and every offset against its table's length.
// Usage: harm_check <0 mixed, 1 FP64> <bx> <by> <bz> <rcut> <tol>
#include "harmonic_plan.hpp"

#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>

namespace glst {
std::string tdesign_dir() { return ""; }
namespace dev {
// (the launches' LDS sizes, which the plan only passes on)
template <typename T>
size_t harm_lds_sf(uint32_t, uint32_t) { return 0; }
template <typename T>
size_t harm_lds_lr(uint32_t, uint32_t, uint32_t) { return 0; }
template size_t harm_lds_sf<float>(uint32_t, uint32_t);
template size_t harm_lds_sf<double>(uint32_t, uint32_t);
template size_t harm_lds_lr<float>(uint32_t, uint32_t, uint32_t);
template size_t harm_lds_lr<double>(uint32_t, uint32_t, uint32_t);
}  // namespace dev
}  // namespace glst

int main(int argc, char **argv) {
  using namespace glst;
  if (argc < 7) return 2;
  const int ct = std::atoi(argv[1]) ? GLST_CT_DOUBLE : GLST_CT_FLOAT;
  const SystemSetup S =
      setup_system(ct, std::atof(argv[2]), std::atof(argv[3]),
                   std::atof(argv[4]), std::atof(argv[5]), std::atof(argv[6]));
  const bool single = ct == GLST_CT_FLOAT;
  const HarmTables T =
      plan_harmonic(S.nodes, S.grid.h, S.spherical_rule, single);
  if (!T.ok) {
    std::printf("no plan\n");
    return 0;
  }
  const uint32_t N = T.N;
  std::mt19937_64 rng(5);
  std::uniform_real_distribution<double> uni(-1.0, 1.0);
  const double rho = dev::cheb_rho(S.grid.h);
  double worst = 0.0;
  long failures = 0, checks = 0;
  for (int point = 0; point < 6; ++point) {
    double d[3], r2;
    do {
      r2 = 0.0;
      for (double &x : d) {
        x = uni(rng) * rho;
        r2 += x * x;
      }
    } while (r2 > rho * rho);
    if (point == 0) d[0] = d[1] = d[2] = 0.0;
    if (point == 1) {  // on the surface
      const double f = rho / std::sqrt(r2);
      for (double &x : d) x *= f;
    }
    const double x = d[0] * T.scale, y = d[1] * T.scale, z = d[2] * T.scale;
    const double s = x * x + y * y + z * z, t = 2.0 * s / T.smax - 1.0;
    // moments of a unit charge: q[l][p][mu][cs]
    std::vector<std::vector<double>> R(N), M(N);
    std::vector<double> xc(N), xs(N);
    double re = 1.0, im = 0.0;
    for (uint32_t m = 0; m < N; ++m) {
      xc[m] = re;
      xs[m] = im;
      const double nr = re * x - im * y;
      im = re * y + im * x;
      re = nr;
    }
    for (uint32_t l = 0; l < N; ++l) {
      const uint32_t np = 4 * dev::harm_psteps(l, N);
      for (uint32_t p = 0; p < np; ++p) {
        const double *J = &T.jac[(static_cast<size_t>(T.crow[l]) + p) * 2];
        R[l].push_back(p == 0 ? 1.0
                              : (t + J[0]) * R[l][p - 1] -
                                    (p > 1 ? J[1] * R[l][p - 2] : 0.0));
      }
      for (uint32_t m = 0; m <= l; ++m) {
        const double b = T.rec[(static_cast<size_t>(l) * 64 + m) * 2];
        const double p1 = l > m ? M[l - 1][m] : 0.0;
        const double p2 = l > m + 1 ? M[l - 2][m] : 0.0;
        M[l].push_back(l == m ? 1.0 : z * p1 - b * s * p2);
      }
    }
    for (uint32_t i = 0; i < T.rad.size(); ++i) {
      const dev::HarmRad &ri = T.rad[i];
      const dev::HarmGroup &G = T.grp[ri.group];
      if (ri.off + 16 * dev::harm_blocks(ri.N) > T.stride) ++failures;
      // radial matrix times radial values, per degree
      std::vector<double> B(ri.N);
      for (uint32_t l = 0; l < ri.N; ++l) {
        const uint32_t PK = dev::harm_psteps(l, N);
        if (i >= T.lrow[l].z) ++failures;
        for (uint32_t p = 0; p < 4 * PK; ++p) {
          const size_t at =
              (T.lrow[l].x + static_cast<size_t>(i / 16) * PK + p / 4) * 64 +
              (p % 4) * 16 + i % 16;
          B[l] += T.gam[at] * R[l][p];
        }
      }
      for (uint32_t j = 0; j < G.nring; j += 1 + G.nring / 4)
        for (uint32_t k = 0; k < G.h; k += 1 + G.h / 3) {
          double sr = 0.0, si = 0.0;
          for (uint32_t m = 0; m < ri.N; ++m)
            for (uint32_t par = 0; par < 2; ++par) {
              const uint32_t l0 = m + ((m ^ par) & 1u);
              const uint2 o = T.mup[G.mup + 2 * m + par];
              // azimuths past pi / 2 through the one at pi - phi: the cosine
              // changes sign for odd orders, the sine for even ones
              const uint32_t kk2 = 2 * k > G.h ? G.h - k : k;
              const double sg[2] = {kk2 != k && m % 2 ? -1.0 : 1.0,
                                    kk2 != k && m % 2 == 0 ? -1.0 : 1.0};
              auto mode = [&](size_t c) {
                const size_t ft =
                    G.trig +
                    ((static_cast<size_t>(kk2 / 16) * 2 + c) * 2 + m % 2) *
                        G.trig_k;
                return sg[c] * T.trig[(ft + m / 2 / 4) * 64 +
                                      (m / 2 % 4) * 16 + kk2 % 16];
              };
              const double az = mode(0) * xc[m] + mode(1) * xs[m];
              double sum = 0.0;
              for (uint32_t l = l0, kk = 0; l < ri.N; l += 2, ++kk)
                sum += T.leg[(G.leg + static_cast<size_t>(j / 16) * G.leg_n +
                              o.x + kk / 4) * 64 +
                             (kk % 4) * 16 + j % 16] *
                       B[l] * M[l][m];
              (par ? si : sr) += sum * az;
            }
          const uint32_t dir =
              (G.equator ? (j ? G.h + 2 * G.h * (j - 1) : 0u) : 2 * G.h * j) +
              k;
          const auto &u = S.nodes.dirs[ri.group][dir];
          const double ph = S.nodes.kappa[ri.group][ri.idx] *
                            (u[0] * d[0] + u[1] * d[1] + u[2] * d[2]);
          worst = std::max(worst, std::fabs(sr - std::cos(ph)));
          worst = std::max(worst, std::fabs(si + std::sin(ph)));
          ++checks;
        }
    }
  }
  for (uint32_t l = 0; l < N; ++l)
    if (T.urow[l + 1] - T.urow[l] != (l + 1) * dev::harm_psteps(l, N))
      ++failures;
  std::printf("N %u checks %ld failures %ld worst %.3e\n", N, checks, failures,
              worst);
  return failures ? 1 : 0;
}
