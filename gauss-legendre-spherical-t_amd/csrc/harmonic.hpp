// The far field through spherical harmonics of the cells.
//
// Around a cell's centre (d = rho t u, |t| <= 1, u a unit vector) a plane wave
// of a direction s and magnitude kappa, z = kappa rho, is
//   exp(-i kappa s.d) = 4 pi sum_n (-i)^n (2n+3) j_{n+1}(z) / z
//                       sum_{l <= n, l = n mod 2} R_n^l(t) sum_mu Y_lmu(u) Y_lmu(s)
// with the real spherical harmonics Y and the radial polynomials of the ball
// R_n^l(t) = t^l P_p^(0, l+1/2)(2 t^2 - 1), n = l + 2 p (the Rayleigh
// expansion with j_l(z t) expanded in R_n^l).  So one set of moments
// sum_j q_j R_n^l Y_lmu of a cell's atoms gives its structure factors at
// every node of every alpha group, and one expansion of the remote sums gives
// the potential and its gradient at every atom: the (atom, node) work of the
// direct sums becomes (cell, node) work.  The nodes of the product rule lie
// on rings of constant polar angle with equispaced azimuths, so the step
// between harmonics and directions is a Legendre product per azimuthal order
// and a Fourier product per ring.  All of it is small dense products on the
// matrix cores, in the precision of the calculation type.
//
// The expansion of radial node i stops at the degree N_i - 1 (harm_degree);
// the radial nodes of all groups are sorted by falling N_i.
//
// Fields of this path are node-major: S and R hold a row of `ncp` cells for
// every node (mixed: (re, im) pairs; FP64: the row of real parts, then the
// row of imaginary parts).  The rows of a group run over its directions for
// each radial node in turn (elsewhere: over the radial nodes for each
// direction), so that a workgroup, which holds one radial node, meets adjacent
// rows: at 1.0M charges, where they were 1.2 MB apart, S took 3,938 us and the
// way back 2,599; the nodes' table of this path is in the same order.  S = sum_j q_j exp(-i k.d_j) around the cell
// centre, R = V = exp(+i k.c) R_c(k).
#pragma once

#include "kernels.hpp"

#include <hip/hip_runtime.h>
#include <cstdint>

namespace glst {
namespace dev {

constexpr uint32_t kHarmMaxN = 56;   // expansion degrees 0 .. N - 1
constexpr uint32_t kHarmMaxN32 = 40; // in FP32 (reached at phases of 20 radians)
constexpr uint32_t kHarmMaxH = 63;   // half azimuths of a ring (reached with
                                     // 56 degrees; more need more)
constexpr uint32_t kHarmCells = 8;   // cells per tile of the transforms
constexpr uint32_t kHarmMu = 8;      // azimuthal orders per tile of 16 columns

// The coefficients of one radial node (N degrees): blocks of 16 columns (the
// cosine and sine of orders mu = 8 t .. 8 t + 7), for t = 0, 1, ... the
// degrees l = 8 t .. N - 1.  Columns hold the eight cells of a tile side by
// side: scalar (tile * stride + off_i + 16 block + column) * 8 + cell.  The
// moments of a cell, and the coefficients contracted over the radial nodes,
// are rows of 16 columns: row qoff[t] + crow[l] + p of its `rows` rows.
__host__ __device__ inline uint32_t harm_block(uint32_t t, uint32_t l,
                                               uint32_t N) {
  return t * N - 4 * t * (t - 1) + (l - 8 * t);
}
__host__ __device__ inline uint32_t harm_blocks(uint32_t N) {
  const uint32_t nt = (N + 7) / 8;
  return nt * N - 4 * nt * (nt - 1);
}
// radial polynomials of degree l below N, padded to a multiple of four
__host__ __device__ inline uint32_t harm_psteps(uint32_t l, uint32_t N) {
  return ((N - 1 - l) / 2 + 4) / 4;
}

// Mixed path: the products of the lowest degrees (radial) and orders (Legendre)
// that are formed in FP64, from FP32 operands and FP64 tables, and stored in
// FP32.  Their rounding is common to all directions of a radial node (degree
// 0) or all azimuths of a ring (order 0) and so does not average out: with FP32
// products it was nearly all of the far field's error, whose rms over 15 water
// boxes was 3.2e-7 in the forces and 2.9e-7 in the energies against 2.6e-7 and
// 1.4e-7 of the direct sums, and is 2.0e-7 and 1.3e-7.
constexpr uint32_t kHarmExactL = 4, kHarmExactMu = 2;

// One radial node.
struct HarmRad {
  uint32_t N;      // degrees
  uint32_t group;  // alpha group
  uint32_t idx;    // radial index inside the group
  uint32_t off;    // first scalar in a cell's coefficient record
};

// One alpha group.  Table offsets count operands of one matrix instruction
// (64 values, one per lane).
struct HarmGroup {
  uint32_t nr, node0;  // radial nodes, first device node
  uint32_t h;          // half the azimuths of a ring
  uint32_t nring;      // rings of the upper half sphere
  uint32_t equator;    // 1: ring 0 is the equator (h azimuths only)
  uint32_t N;          // largest N_i of the group
  uint32_t mup;        // first (mu, parity) entry of HarmDev::mup
  uint32_t leg, leg_n;    // Legendre, degrees -> rings: per ring tile of 16
  uint32_t legt, legt_k;  // rings -> degrees; steps over the rings
  // Fourier, azimuths up to pi / 2: orders -> azimuths [tile][cs][set][step]
  // (cs 0: cosines, 1: sines), trig_t tiles, and back [set][cs][tile][step]
  uint32_t trig, trig_k, trig_t;
  uint32_t trigt, trigt_m, trigt_k;
  // the FP64 copies of leg and legt for the orders below kHarmExactMu, and
  // their offsets, four (order, parity) entries of HarmDev::mup64
  uint32_t leg64, leg64_n, legt64, mup64;
};

// directions of a group
__host__ __device__ inline uint32_t harm_dirs(const HarmGroup &g) {
  return g.nring * 2 * g.h - (g.equator ? g.h : 0u);
}

// Expansion tables on the device (T: the calculation type).
template <typename T>
struct HarmDev {
  const HarmRad *rad;     // nrad radial nodes, N falling
  const HarmGroup *grp;
  const uint2 *mup;       // per (group, mu, parity): offsets into leg, legt
  const T *leg, *legt, *trig, *trigt;
  const T *gam, *gamt;    // radial matrices: moments -> radial nodes and back
  const uint4 *lrow;      // per degree l: gam, gamt offsets, radial nodes with
                          // N_i > l
  // mixed: FP64 tables of the low degrees and orders; offsets by degree into
  // gam64 and gamt64, by (group, order, parity) into leg64 and legt64
  const double *leg64, *legt64, *gam64, *gamt64;
  const uint2 *lrow64, *mup64;
  const uint2 *pair;      // npair (degree, order tile) pairs
  const uint32_t *crow;   // rows of the degrees below l
  const uint32_t *urow;   // groups of the contracted coefficients below l
  const T *jac;           // per row crow[l] + p (jrows of them): the constants
                          // c1, c2 of the radial polynomials' recurrence
  const T *rec;           // per (l, mu): b, e of the Legendre recurrence
  uint32_t nrad, N, stride, npair, rows, jrows, ustride;
  uint32_t qoff[8];       // per order tile
  // positions are held in units of 1 / scale, a power of two near 1 / rho (so
  // they keep the bits of the record): smax = (rho scale)^2, xk = 2 / smax
  double scale, smax, xk;
};

// Everything a launch needs: units of the transforms are (radial node, ring
// tile) forward and radial nodes backward, times the tiles of kHarmCells
// cells.
struct HarmPlanDev {
  uint32_t nrad = 0, nunit = 0;
  uint32_t ksteps = 16;  // steps of four atoms per pass of the moments
  uint32_t nset = 1;     // workgroups (of 64 atoms a time) per cell, evaluation
  uint32_t hsteps = 0;   // largest HarmGroup::trigt_k
  size_t lds_moments = 0, lds_sf = 0, lds_lr = 0;
  const uint2 *unit = nullptr;
};

// Dynamic LDS of the kernels: the moments of a plan of N degrees; sf and lr for
// one radial node of N degrees in a group with h half azimuths and nring rings.
template <typename T>
size_t harm_lds_moments(uint32_t N, uint32_t ksteps);
template <typename T>
size_t harm_lds_sf(uint32_t N, uint32_t h);
template <typename T>
size_t harm_lds_lr(uint32_t N, uint32_t h, uint32_t nring);

template <typename T>
void harm_moments(const HarmPlanDev &P, const HarmDev<T> &H, const void *atoms,
                  const uint32_t *start, const GridShape &g, T *mom, T *coef,
                  uint32_t *outside, hipStream_t s);
template <typename T>
void harm_sf(const HarmPlanDev &P, const HarmDev<T> &H, const void *atoms,
             const uint32_t *start, const double4 *k64, const GridShape &g,
             const T *coef, const uint32_t *outside, T *S, hipStream_t s);
template <typename T>
void harm_lr(const HarmPlanDev &P, const HarmDev<T> &H, const GridShape &g,
             const T *R, T *coef, T *mom, hipStream_t s);
template <typename T>
void harm_eval(const HarmPlanDev &P, const HarmDev<T> &H, const void *atoms,
               const uint32_t *start, const double4 *k64, uint32_t K,
               const GridShape &g, const T *mom, const T *R,
               const uint32_t *outside, T *coef, double4 *out, hipStream_t s);
// Once per process and device (see prepare_kernels).
void prepare_harmonic(size_t lds_limit);

}  // namespace dev
}  // namespace glst
