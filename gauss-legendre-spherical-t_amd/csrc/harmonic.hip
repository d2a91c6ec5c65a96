// Kernels of the far field through spherical harmonics (harmonic.hpp), for
// gfx950.  Four kernels: moments of a cell's atoms -> coefficients of every
// radial node (harm_moments), coefficients -> S at the nodes (harm_sf),
// remote sums -> coefficients (harm_lr), coefficients -> fields at the atoms
// (harm_eval).  The dense products of the first three are
// v_mfma_f32_16x16x4f32 or v_mfma_f64_16x16x4f64.
//
// Times below are of the 288,000-charge box at tol 1e-4 (3,375 cells of 85
// atoms, 27,453 nodes, 53 radial nodes, N = 26 mixed and 37 FP64), mixed and
// FP64.  The direct sums that these passes replace took 724 and 9,160 us (S)
// and 1,873 and 10,153 us (back-projection); S and R are 0.74 and 1.48 GB
// each, 0.15 and 0.29 ms at the 5.1 TB/s of a large copy.
//
// Operand layouts for lane l (c = l % 16, g = l / 16): A[c][g], B[g][c];
// accumulator register r holds D[4g + r][c] in FP32 and D[g + 4r][c] in FP64
// (both checked on the GPU).  Where an accumulator is the B operand of a
// following product, register r is step r of it: its rows are numbered so
// that step r covers the indices 4r .. 4r + 3 (harm_perm).
#include "harmonic.hpp"

#include <algorithm>
#include <type_traits>

namespace glst {
namespace dev {
namespace {

typedef float harm_f4 __attribute__((ext_vector_type(4)));
typedef double harm_d4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Harm;
template <>
struct Harm<float> {
  using v4 = harm_f4;
  static __device__ __forceinline__ v4 mfma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // row of the accumulator in register r of lane group g
  static __device__ __forceinline__ uint32_t row(uint32_t g, uint32_t r) {
    return 4 * g + r;
  }
  // the index that row R of a chained product stands for
  static __device__ __forceinline__ uint32_t perm(uint32_t R) {
    return 4 * (R & 3u) + (R >> 2);
  }
};
template <>
struct Harm<double> {
  using v4 = harm_d4;
  static __device__ __forceinline__ v4 mfma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t row(uint32_t g, uint32_t r) {
    return g + 4 * r;
  }
  static __device__ __forceinline__ uint32_t perm(uint32_t R) { return R; }
};

__device__ __forceinline__ float harm_fma(float a, float b, float c) {
  return fmaf(a, b, c);
}
__device__ __forceinline__ double harm_fma(double a, double b, double c) {
  return fma(a, b, c);
}

// An atom around its cell's centre, in units of 1 / scale: position, square,
// argument of the radial polynomials x = 2 t^2 - 1, charge, and whether it
// lies outside the ball.  The squares are formed in FP64 (an FP32 one would
// move the atom, for all directions alike), by the same operations in every
// kernel, so that all agree on which atoms lie outside.
template <typename T>
struct HarmAtom {
  T x, y, z, s, t, q;
  bool out;
};
// An atom's offset from its cell's centre and its charge in FP64.
struct HarmOffset {
  double x, y, z, q;
};
template <typename T>
struct HarmRecord;
template <>
struct HarmRecord<float> {
  using type = float4;
};
template <>
struct HarmRecord<double> {
  using type = double4;
};

struct HarmCentre {
  double x, y, z;
};
__device__ __forceinline__ HarmOffset harm_offset(const float4 *atoms,
                                                  uint32_t i, HarmCentre) {
  const float4 a = atoms[i];
  return {a.x, a.y, a.z, a.w};
}
__device__ __forceinline__ HarmOffset harm_offset(const double4 *atoms,
                                                  uint32_t i, HarmCentre c) {
  const double4 a = atoms[i];
  return {a.x - c.x, a.y - c.y, a.z - c.z, a.w};
}
template <typename T>
__device__ __forceinline__ HarmAtom<T> harm_atom(
    const HarmDev<T> &H, const typename HarmRecord<T>::type *atoms, uint32_t i,
    HarmCentre c) {
#pragma clang fp contract(off)
  const HarmOffset d = harm_offset(atoms, i, c);
  const double x = d.x * H.scale, y = d.y * H.scale, z = d.z * H.scale;
  const double s = x * x + y * y + z * z;
  HarmAtom<T> o = {};
  o.q = static_cast<T>(d.q);
  o.out = s > H.smax;
  if (!o.out) {
    o.x = static_cast<T>(x);
    o.y = static_cast<T>(y);
    o.z = static_cast<T>(z);
    o.s = static_cast<T>(s);
    o.t = static_cast<T>(s * H.xk - 1.0);
  }
  return o;
}
__device__ __forceinline__ HarmCentre harm_centre(uint32_t cell, uint32_t ny,
                                                  uint32_t nz, double h) {
  HarmCentre c;
  c.x = (static_cast<double>(cell / (ny * nz)) + 0.5) * h;
  c.y = (static_cast<double>((cell / nz) % ny) + 0.5) * h;
  c.z = (static_cast<double>(cell % nz) + 0.5) * h;
  return c;
}

// One wave: the atoms of [a0, a0 + na) outside the ball, in order, into list[1]
// ...; their number into list[0].  na <= 64.
template <typename T>
__device__ __forceinline__ void harm_list_outside(
    const HarmDev<T> &H, const typename HarmRecord<T>::type *atoms, uint32_t a0,
    uint32_t na, const HarmCentre &cc, uint32_t *list) {
  const uint32_t lane = threadIdx.x & 63u;
  const bool out = lane < na && harm_atom(H, atoms, a0 + lane, cc).out;
  const unsigned long long mask = __ballot(out);
  if (out) list[1 + __popcll(mask & ((1ull << lane) - 1))] = a0 + lane;
  if (lane == 0) list[0] = static_cast<uint32_t>(__popcll(mask));
}
// Workgroup barrier for data in LDS: waits for the LDS operations only, so that
// loads issued ahead and stores stay in flight (__syncthreads drains them).
__device__ __forceinline__ void harm_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// The scalar at byte `off` of the `bytes` from a base uniform over the wave, or
// zero past them: the buffer's own range check takes the place of a compare,
// a clamped address and a select per load.
template <typename T>
__device__ __forceinline__ T harm_ranged(const T *base, uint32_t bytes,
                                         uint32_t off) {
  const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(base), 0,
                                                   bytes, 0x00020000);
  if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(
        T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  else
    return __builtin_bit_cast(
        T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
// p[byte offset], the base uniform over the wave
template <typename T>
__device__ __forceinline__ T harm_at_byte(const T *p, uint32_t off) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + off);
}


// ---------------------------------------------------------------------------
// moments of the atoms -> coefficients of the radial nodes

// Radial values of one degree l at one atom: rows p of `tab` (pitch AS) get
// scale R_{l,p} at x, for p < 4 PK.  J: the recurrence constants of the degree
// (staged in LDS, two scalars per p).
template <typename T>
__device__ __forceinline__ void harm_radial(const T *J, T x, T scale,
                                            uint32_t PK, T *tab, uint32_t AS) {
  T v1 = scale, v2 = T(0);
  tab[0] = scale;
#pragma unroll
  for (uint32_t u = 1; u < 4; ++u) {
    const T v = harm_fma(x + J[2 * u], v1, -J[2 * u + 1] * v2);
    tab[u * AS] = v;
    v2 = v1;
    v1 = v;
  }
  for (uint32_t k = 1; k < PK; ++k) {
    J += 8;
    tab += 4 * AS;
    T c[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) c[u] = J[u];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
      const T v = harm_fma(x + c[2 * u], v1, -c[2 * u + 1] * v2);
      tab[u * AS] = v;
      v2 = v1;
      v1 = v;
    }
  }
}
// Stages `n` scalars of a constant table.
template <typename T>
__device__ __forceinline__ void harm_stage(T *dst, const T *src, uint32_t n) {
  for (uint32_t e = threadIdx.x; e < n; e += blockDim.x) dst[e] = src[e];
}

// degrees per round of the radial tables
template <typename T>
constexpr uint32_t harm_lb() {
  return sizeof(T) == 4 ? 4 : 2;
}
constexpr uint32_t kHarmBlock = 512;  // threads of the transform kernels

template <int V>
struct HarmInt {
  static constexpr int value = V;
};
// f(HarmInt<n>) for the uniform n in 1 .. MAX: the inner loops have constant
// lengths (conditional steps would copy the accumulators at every branch)
template <int MAX, class F>
void harm_host_switch(uint32_t n, F f) {
  if constexpr (MAX <= 1) {
    f(HarmInt<1>{});
  } else {
    if (n >= static_cast<uint32_t>(MAX))
      f(HarmInt<MAX>{});
    else
      harm_host_switch<MAX - 1>(n, f);
  }
}
template <int MAX, class F>
__device__ __forceinline__ void harm_switch(uint32_t n, F f) {
  if constexpr (MAX <= 1) {
    f(HarmInt<1>{});
  } else {
    if (n >= static_cast<uint32_t>(MAX))
      f(HarmInt<MAX>{});
    else
      harm_switch<MAX - 1>(n, f);
  }
}

// One workgroup per cell, wave t on the azimuthal orders 8 t .. 8 t + 7.  A
// wave walks the degrees l of its tile: lane (c, g) carries the solid harmonic
// of column c (order, cosine or sine) at the atoms 4k + g through the
// recurrence in l, and
//   Q[p][column] = sum_atoms (q R_{l,p}) Y        (steps of four atoms)
// is one product per degree.  The radial values of LB degrees at a time are
// tabulated in LDS by all waves; the recurrence constants of a round are
// loaded during the one before and go through LDS too (a load inside the loop
// over the degrees would wait for the stores before it).  Cells of more than
// 4 KS atoms take several passes that add up in `mom`.  The mixed path sums the
// degrees below kHarmExactL in FP64: the terms of a cell's low moments mostly
// cancel, and the rest is common to all nodes.  345 and 1,637 us
// (336 with all sums in FP32, 422 and 1,560 with the constants loaded per degree), bound by the latency
// of the LDS reads between the products: 59 % of the wave cycles wait.  FP32
// takes 64 atoms a pass (more registers leave fewer waves: 388 us at 128),
// FP64 up to 128 (1,880 us at 64).
template <typename T, int KS>
__device__ __forceinline__ void harm_moments_body(
    const HarmDev<T> &H, const typename HarmRecord<T>::type *atoms,
    const uint32_t *start, uint32_t ny, uint32_t nz, double h, uint32_t cell,
    uint32_t turn, T *mom, uint32_t *outside, char *smem) {
  using M = Harm<T>;
  using v4 = typename M::v4;
  constexpr uint32_t CH = 4 * KS, AS = CH + 4, LB = harm_lb<T>();
  const uint32_t tid = threadIdx.x, nth = blockDim.x, nwave = nth >> 6;
  const uint32_t lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the tiles' lengths differ: the first one is another wave (another SIMD)
  // from workgroup to workgroup
  const uint32_t t = (wave + turn) % nwave;
  const uint32_t c16 = lane & 15u, g = lane >> 4;
  const uint32_t N = H.N;
  const uint32_t prow = 4 * harm_psteps(0, N);
  T *xs = reinterpret_cast<T *>(smem);
  T *ys = xs + CH, *zs = ys + CH;  // zs: (z, s) pairs
  T *ts = zs + 2 * CH, *qs = ts + CH;
  // radial tables [LB][prow][AS]; first the powers [16 nt][AS]
  T *zt = qs + CH;
  const uint32_t trow = LB * prow > 16 * nwave ? LB * prow : 16 * nwave;
  T *rec = zt + trow * AS;             // [LB][8 nt]
  T *jac = rec + LB * 8 * nwave;       // [crow[N]][2]
  const uint32_t jrows = H.jrows;
  uint32_t *flag = reinterpret_cast<uint32_t *>(jac + 2 * jrows);
  if (tid == 0) *flag = 0u;
  harm_stage(jac, H.jac, 2 * jrows);
  const uint32_t a0 = start[cell], na = start[cell + 1] - a0;
  const HarmCentre cc = harm_centre(cell, ny, nz, h);
  T *out = mom + static_cast<size_t>(cell) * H.rows * 16;
  const uint32_t pr = M::perm(c16);  // radial index of this lane's A row
  const uint32_t row0 = (pr < prow ? pr : prow - 1) * AS + g;
  const uint32_t row1 = (16 + pr < prow ? 16 + pr : prow - 1) * AS + g;
  const uint32_t low0 = (c16 < prow ? c16 : prow - 1) * AS + g;
  const uint32_t low1 = (16 + c16 < prow ? 16 + c16 : prow - 1) * AS + g;
  const uint32_t mu = 8 * t + (c16 >> 1);
  for (uint32_t p0 = 0; p0 == 0 || p0 < na; p0 += CH) {
    const uint32_t cnt = na - p0 < CH ? na - p0 : CH;
    harm_barrier();
    for (uint32_t e = tid; e < CH; e += nth) {
      HarmAtom<T> a = {};
      if (e < cnt) {
        a = harm_atom(H, atoms, a0 + p0 + e, cc);
        if (a.out) {
          *flag = 1u;
          a.q = T(0);
        }
      }
      xs[e] = a.x;
      ys[e] = a.y;
      zs[2 * e] = a.z;
      zs[2 * e + 1] = a.s;
      ts[e] = a.t;
      qs[e] = a.q;
    }
    harm_barrier();
    // groups of four steps of four atoms (the staged atoms past cnt are zero)
    const uint32_t ng = cnt ? (cnt + 31) / 32 * 2 : 2u;
    // (x + i y)^mu of every atom, mu < 8 nt, for the start values
    for (uint32_t e = tid; e < 16 * ng; e += nth) {
      const T X = xs[e], Y = ys[e];
      T re = T(1), im = T(0);
      for (uint32_t m = 0; m < 8 * nwave; ++m) {
        zt[(2 * m) * AS + e] = re;
        zt[(2 * m + 1) * AS + e] = im;
        const T nr = re * X - im * Y;
        im = re * Y + im * X;
        re = nr;
      }
    }
    harm_barrier();
    harm_switch<KS / 8>((ng + 1) / 2, [&](auto half) {
      constexpr int NK = 8 * decltype(half)::value;  // steps of four atoms
      T Y1[NK], Y2[NK];
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        Y1[k] = zt[(2 * mu + (c16 & 1u)) * AS + 4 * k + g];
        Y2[k] = T(0);
      }
      harm_barrier();
      // recurrence constants: thread e holds scalar e of a round's
      // [LB][8 nt] (whole rounds are allocated)
      const uint32_t rl = tid / (8 * nwave), rm = tid - rl * 8 * nwave;
      const T *rc = H.rec + (static_cast<size_t>(rl) * 64 + rm) * 2;
      T rnext = rl < LB ? rc[0] : T(0);
      T *o = out + (H.qoff[t] + H.crow[8 * t]) * 16 + lane;
      // one degree: PT row tiles of radial polynomials, LOW: the sums in FP64
      // A: Y of the degree before; B: of the one before that, then of this
      auto degree = [&](auto tiles, auto low, uint32_t l, T(&A)[NK],
                        T(&B)[NK]) {
        constexpr int PT = decltype(tiles)::value;
        constexpr bool LOW = decltype(low)::value != 0;
        const uint32_t PK = harm_psteps(l, N);
        const T *zl = zt + (l % LB) * prow * AS;
        const T rb = rec[(l % LB) * 8 * nwave + mu];
        const T ra = l > mu ? T(1) : T(0), one = T(1) - ra;
        // (partial sums: the rounding of a sum grows with its length)
        constexpr int NA = sizeof(T) == 4 && !LOW ? 4 / PT : 1;
        using S = std::conditional_t<LOW, double, T>;
        using MS = Harm<S>;
        using s4 = typename MS::v4;
        s4 a0s[NA], a1s[NA];
#pragma unroll
        for (int i = 0; i < NA; ++i)
          a0s[i] = a1s[i] = s4{S(0), S(0), S(0), S(0)};
#pragma unroll
        for (int k = 0; k < NK; ++k) {
          const T z = zs[2 * (4 * k + g)], s = zs[2 * (4 * k + g) + 1];
          const T y = harm_fma(harm_fma(ra, z, one), A[k], -(rb * s) * B[k]);
          B[k] = y;
          a0s[k % NA] = MS::mfma(static_cast<S>(zl[(LOW ? low0 : row0) + 4 * k]),
                                 static_cast<S>(y), a0s[k % NA]);
          if (PT > 1)
            a1s[k % NA] = MS::mfma(static_cast<S>(zl[(LOW ? low1 : row1) + 4 * k]),
                                   static_cast<S>(y), a1s[k % NA]);
        }
#pragma unroll
        for (int w = NA / 2; w > 0; w /= 2)
#pragma unroll
          for (int i = 0; i < w; ++i) {
            a0s[i] += a0s[i + w];
            if (PT > 1) a1s[i] += a1s[i + w];
          }
        v4 acc0, acc1;
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
          acc0[r] = static_cast<T>(a0s[0][r]);
          acc1[r] = static_cast<T>(a1s[0][r]);
        }
        // orders above the degree are zero; register r holds the rows
        // p = 4 r + g
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
          acc0[r] = mu > l ? T(0) : acc0[r];
          if (PT > 1) acc1[r] = mu > l ? T(0) : acc1[r];
        }
        if (p0 == 0) {
#pragma unroll
          for (uint32_t r = 0; r < 4 * PT; ++r)
            if (r < PK) o[r * 64] = r < 4 ? acc0[r & 3u] : acc1[r & 3u];
        } else {
          for (uint32_t r = 0; r < PK; ++r) {
            const v4 a = r < 4 ? acc0 : acc1;
            o[r * 64] += (r & 3u) == 0   ? a[0]
                         : (r & 3u) == 1 ? a[1]
                         : (r & 3u) == 2 ? a[2]
                                         : a[3];
          }
        }
        o += PK * 64;
      };
      for (uint32_t l0 = 0; l0 < N; l0 += LB) {
        const uint32_t nl = N - l0 < LB ? N - l0 : LB;
        const uint32_t nch = (16 * ng + 63) / 64;
        if (rl < LB) {
          rec[tid] = rnext;
          rc += LB * 64 * 2;
          rnext = rc[0];
        }
        for (uint32_t e = wave; e < nl * nch; e += nwave) {
          const uint32_t ch = e / nl, l = l0 + (e - ch * nl);
          const uint32_t a = ch * 64 + lane;
          if (a < 16 * ng)
            harm_radial(jac + 2 * H.crow[l],
                        ts[a], qs[a], harm_psteps(l, N), zt + (l - l0) * prow * AS + a, AS);
        }
        harm_barrier();
        for (uint32_t l = l0 < 8 * t ? 8 * t : l0; l < l0 + nl; l += 2) {
          auto one = [&](uint32_t d, T(&A)[NK], T(&B)[NK]) {
            if (sizeof(T) == 4 && d < kHarmExactL) {
              if (harm_psteps(d, N) > 4)
                degree(HarmInt<2>{}, HarmInt<1>{}, d, A, B);
              else
                degree(HarmInt<1>{}, HarmInt<1>{}, d, A, B);
            } else if (harm_psteps(d, N) > 4) {
              degree(HarmInt<2>{}, HarmInt<0>{}, d, A, B);
            } else {
              degree(HarmInt<1>{}, HarmInt<0>{}, d, A, B);
            }
          };
          one(l, Y1, Y2);
          if (l + 1 < N) one(l + 1, Y2, Y1);
        }
        harm_barrier();
      }
    });
  }
  if (tid == 0) outside[cell] = *flag;
}

template <typename T, int KS>
__global__ __launch_bounds__(512) void harm_moments_kernel(
    HarmDev<T> H, const typename HarmRecord<T>::type *__restrict__ atoms,
    const uint32_t *__restrict__ start, uint32_t ny, uint32_t nz, double h,
    T *__restrict__ mom, uint32_t *__restrict__ outside) {
  extern __shared__ char harm_smem[];
  const uint32_t nb = gridDim.x, b = blockIdx.x;
  const uint32_t q = nb >> 3, r = nb & 7u, x = b & 7u;
  const uint32_t cell = x * q + (x < r ? x : r) + (b >> 3);
  harm_moments_body<T, KS>(H, atoms, start, ny, nz, h, cell,
                           (b >> 3) + (b >> 8), mom, outside,
                           harm_smem);
}

// ---------------------------------------------------------------------------
// moments <-> coefficients of the radial nodes

// most steps over the radial polynomials of a degree
template <typename T>
constexpr int harm_max_psteps() {
  return static_cast<int>(
      (((sizeof(T) == 4 ? kHarmMaxN32 : kHarmMaxN) - 1) / 2 + 4) / 4);
}

// One wave: degree l and order tile t of the eight cells of a tile.  Forward:
// B_i = sum_p gam_l[i][p] Q[p] for the radial nodes with more than l degrees,
// the moments in registers for all eight cells; a lane ends with the eight
// cells' values of one (node, column), adjacent in the coefficients.  74 and
// 369 us forward, 107 and 286 us backward: memory traffic of the coefficients
// (0.25 and 1.0 GB), behind which the FP64 products of the mixed path's low
// degrees (see kHarmExactL) cost nothing.
// CT: the type of the products; with FP64 products of FP32 data (the low
// degrees) four cells at a time, so that the registers stay those of the rest.
template <typename T, typename CT>
__device__ __forceinline__ void harm_forward_wave(const HarmDev<T> &H,
                                                  uint32_t ncell, uint32_t tile,
                                                  uint32_t l, uint32_t t,
                                                  const T *mom, T *coef) {
  using M = Harm<CT>;
  using v4 = typename M::v4;
  using o4 = typename Harm<T>::v4;
  constexpr int MAXPK = harm_max_psteps<T>();
  constexpr bool LOW = sizeof(CT) != sizeof(T);
  constexpr uint32_t NC = LOW ? 4 : 8;
  const uint32_t lane = threadIdx.x & 63u, c16 = lane & 15u, g = lane >> 4;
  const uint4 lr = H.lrow[l];
  const size_t cs = static_cast<size_t>(H.rows) * 16;
  const T *Q = mom + static_cast<size_t>(H.qoff[t] + H.crow[l]) * 16 + lane;
  T *out = coef + static_cast<size_t>(tile) * H.stride * 8;
  const CT *gam;
  if constexpr (LOW)
    gam = H.gam64 + static_cast<size_t>(H.lrow64[l].x) * 64 + lane;
  else
    gam = H.gam + static_cast<size_t>(lr.x) * 64 + lane;
  harm_switch<MAXPK>(harm_psteps(l, H.N), [&](auto steps) {
    constexpr int PK = decltype(steps)::value;
#pragma unroll 1
    for (uint32_t c0 = 0; c0 < 8; c0 += NC) {
      CT q[NC][PK];
#pragma unroll
      for (uint32_t c = 0; c < NC; ++c) {
        const uint32_t k = tile * 8 + c0 + c;
        const T *p = Q + (k < ncell ? k : ncell - 1) * cs;
#pragma unroll
        for (int r = 0; r < PK; ++r) q[c][r] = p[r * 64];
      }
      const CT *G = gam;
      CT gm[PK];
#pragma unroll
      for (int r = 0; r < PK; ++r) gm[r] = G[r * 64];
      for (uint32_t i0 = 0; i0 < lr.z; i0 += 16) {
        CT gx[PK];
#pragma unroll
        for (int r = 0; r < PK; ++r) gx[r] = gm[r];
        G += PK * 64;  // (the table has room for one more load)
#pragma unroll
        for (int r = 0; r < PK; ++r) gm[r] = G[r * 64];
        HarmRad ri[4];
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
          const uint32_t i = i0 + M::row(g, r);
          ri[r] = H.rad[i < H.nrad ? i : H.nrad - 1];
        }
        v4 d[NC];
#pragma unroll
        for (uint32_t c = 0; c < NC; ++c)
          d[c] = v4{CT(0), CT(0), CT(0), CT(0)};
#pragma unroll
        for (int r = 0; r < PK; ++r)
#pragma unroll
          for (uint32_t c = 0; c < NC; ++c)
            d[c] = M::mfma(gx[r], q[c][r], d[c]);
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r)
          if (i0 + M::row(g, r) < lr.z) {
            T *o = out +
                   (ri[r].off + harm_block(t, l, ri[r].N) * 16 + c16) * 8 + c0;
#pragma unroll
            for (uint32_t c = 0; c < NC; c += 4)
              *reinterpret_cast<o4 *>(o + c) =
                  o4{static_cast<T>(d[c][r]), static_cast<T>(d[c + 1][r]),
                     static_cast<T>(d[c + 2][r]), static_cast<T>(d[c + 3][r])};
          }
      }
    }
  });
}

// Backward: U[p] = sum_i gam_l[i][p] C_i, per (l, order) the pairs (cosine,
// sine) of the rows p side by side.
template <typename T, typename CT>
__device__ __forceinline__ void harm_backward_wave(const HarmDev<T> &H,
                                                   uint32_t ncell,
                                                   uint32_t tile, uint32_t l,
                                                   uint32_t t, const T *coef,
                                                   T *mom) {
  using M = Harm<CT>;
  using v4 = typename M::v4;
  using i4 = typename Harm<T>::v4;
  constexpr bool LOW = sizeof(CT) != sizeof(T);
  constexpr uint32_t NC = LOW ? 4 : 8;
  const uint32_t lane = threadIdx.x & 63u, c16 = lane & 15u, g = lane >> 4;
  const uint32_t PK = harm_psteps(l, H.N);
  const uint4 lr = H.lrow[l];
  const uint32_t mu = 8 * t + (c16 >> 1);
  const CT *gamt;
  if constexpr (LOW)
    gamt = H.gamt64 + static_cast<size_t>(H.lrow64[l].y) * 64 + lane;
  else
    gamt = H.gamt + static_cast<size_t>(lr.y) * 64 + lane;
  const T *in = coef + static_cast<size_t>(tile) * H.stride * 8 + c16 * 8;
  T *o = mom + 8 * (H.urow[l] + mu * PK) + 2 * g + (c16 & 1u);
  harm_switch<2>(PK > 4 ? 2u : 1u, [&](auto tiles) {
    constexpr int PT = decltype(tiles)::value;
#pragma unroll 1
    for (uint32_t c0 = 0; c0 < 8; c0 += NC) {
      const CT *G = gamt;
      v4 d[PT][NC];
#pragma unroll
      for (int p = 0; p < PT; ++p)
#pragma unroll
        for (uint32_t c = 0; c < NC; ++c)
          d[p][c] = v4{CT(0), CT(0), CT(0), CT(0)};
      // four radial nodes a step, two steps in flight; nodes past the last
      // have zero factors and repeat it
      for (uint32_t i0 = 0; i0 < lr.z; i0 += 8) {
        i4 b[2][NC / 4];
        CT ga[2][PT];
#pragma unroll
        for (uint32_t u = 0; u < 2; ++u) {
          const uint32_t i = i0 + 4 * u + g;
          const HarmRad ri = H.rad[i < lr.z ? i : lr.z - 1];
          const i4 *p = reinterpret_cast<const i4 *>(
              in + (ri.off + harm_block(t, l, ri.N) * 16) * 8 + c0);
#pragma unroll
          for (uint32_t c = 0; c < NC / 4; ++c) b[u][c] = p[c];
#pragma unroll
          for (int p2 = 0; p2 < PT; ++p2) {
            const CT x = G[(u * PT + p2) * 64];
            ga[u][p2] = i0 + 4 * u < lr.z ? x : CT(0);
          }
        }
        G += 2 * PT * 64;
#pragma unroll
        for (uint32_t u = 0; u < 2; ++u)
#pragma unroll
          for (int p = 0; p < PT; ++p)
#pragma unroll
            for (uint32_t c = 0; c < NC; ++c)
              d[p][c] = M::mfma(ga[u][p], static_cast<CT>(b[u][c >> 2][c & 3u]),
                                d[p][c]);
      }
#pragma unroll
      for (uint32_t c = 0; c < NC; ++c) {
        if (tile * 8 + c0 + c >= ncell) break;
        T *p = o + static_cast<size_t>(tile * 8 + c0 + c) * H.ustride;
#pragma unroll
        for (uint32_t r = 0; r < 4 * PT; ++r)
          if (r < PK && mu <= l) p[r * 8] = static_cast<T>(d[r >> 2][c][r & 3u]);
      }
    }
  });
}

// Wave w of a launch: tile w / (pairs) and the (l, t) pair w % pairs of the
// plan.
template <typename T, bool BACK>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 4 : 2) void harm_radial_kernel(
    HarmDev<T> H, uint32_t ncell, uint32_t nwave, const T *__restrict__ in,
    T *__restrict__ out) {
  const uint32_t nb = gridDim.x, b = blockIdx.x;
  const uint32_t q = nb >> 3, r = nb & 7u, x = b & 7u;
  const uint32_t w =
      (x * q + (x < r ? x : r) + (b >> 3)) * 4 +
      __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (w >= nwave) return;
  const uint32_t tile = w / H.npair;
  const uint2 lt = H.pair[w - tile * H.npair];
  if (sizeof(T) == 4 && lt.x < kHarmExactL) {
    if (BACK)
      harm_backward_wave<T, double>(H, ncell, tile, lt.x, lt.y, in, out);
    else
      harm_forward_wave<T, double>(H, ncell, tile, lt.x, lt.y, in, out);
  } else if (BACK) {
    harm_backward_wave<T, T>(H, ncell, tile, lt.x, lt.y, in, out);
  } else {
    harm_forward_wave<T, T>(H, ncell, tile, lt.x, lt.y, in, out);
  }
}

// ---------------------------------------------------------------------------
// coefficients -> structure factors (397 and 943 us; mixed 374 with the lowest
// orders in FP32 too, before that 400 and 1,131 with the
// azimuths up to pi summed one by one, 415 and 1,194 before that with a select
// per coefficient; the workgroups' phases between barriers, two to three
// workgroups per CU, against 0.15 and 0.29 ms of stores)

// Which (unit, cell tile) a workgroup serves.  With many tiles every XCD
// (workgroups b with b % 8 == x) owns a contiguous range of them and takes
// it unit by unit: neighbouring tiles, which share lines of S, run there at
// the same time, and every XCD has all the units.
__device__ __forceinline__ bool harm_place(uint32_t b, uint32_t ntile,
                                           uint32_t nunit, uint32_t &unit,
                                           uint32_t &tile) {
  if (ntile < 64) {
    unit = b / ntile;
    tile = b - unit * ntile;
    return unit < nunit;
  }
  const uint32_t x = b & 7u, i = b >> 3, q = ntile >> 3, r = ntile & 7u;
  const uint32_t n = q + (x < r ? 1u : 0u);
  unit = i / n;
  tile = x * q + (x < r ? x : r) + (i - unit * n);
  return unit < nunit;
}
uint32_t harm_grid(uint32_t ntile, uint32_t nunit) {
  if (ntile < 64) return ntile * nunit;
  return 8 * nunit * ((ntile + 7) / 8);
}

// Steps of four over the orders of one set (even or odd azimuthal orders).
__host__ __device__ inline uint32_t harm_order_steps(uint32_t N) {
  return ((N + 1) / 2 + 3) / 4;
}

// One unit: eight cells, one radial node, a tile of 16 rings.  Even and odd
// orders take turns: (1) Legendre: per order, the rings' Fourier coefficients
// of Re (even degrees) and Im (odd degrees) into LDS; columns are (cosine or
// sine, cell); a wave's next order is loaded while it works on one.  (2)
// Fourier: per ring (wave and wave + 8 in FP32), the sums C over the cosines
// and Z over the sines at NPT tiles of azimuths phi in 0 .. pi / 2, in
// registers, which give those at pi - phi too (C - Z for even, Z - C for odd
// orders); the values at phi and phi + pi are the even sum plus and minus the
// odd one.  Columns are (cell, Re or Im) in FP32; in FP64 Re and Im take turns
// and the columns are (ring of a pair, cell).
template <typename T, int NPT>
__device__ __forceinline__ void harm_sf_body(
    const HarmDev<T> &H, const typename HarmRecord<T>::type *atoms,
    const uint32_t *start, const double4 *k64, uint32_t ny, uint32_t nz,
    double h, uint32_t ncell, const HarmRad &rad, const HarmGroup &gr,
    uint32_t rt, uint32_t tile, const T *coef, const uint32_t *outside, T *S,
    char *smem) {
  using M = Harm<T>;
  using v4 = typename M::v4;
  constexpr bool F = sizeof(T) == 4;
  constexpr uint32_t NW = kHarmBlock / 64;
  constexpr int NR = F ? 2 : 1;  // rows of (2) per wave
  constexpr int NP = F ? 2 : 1;  // parities per pass of (1)
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t c16 = lane & 15u, g = lane >> 4;
  // a ring's cosines, then its sines (other banks), in steps of four orders
  const uint32_t N = rad.N, KC = harm_order_steps(N), MH = 4 * KC;
  const uint32_t sines = MH * 16 + 16, RS = 2 * MH * 16 + 24;
  const uint32_t nd = harm_dirs(gr);
  const uint32_t nrow = F ? 16u : 8u;
  T *Gm = reinterpret_cast<T *>(smem);
  T *tr = Gm + nrow * RS;
  const uint32_t cell0 = tile * kHarmCells;
  const uint32_t ncp = harm_row(ncell);
  // columns of (1): the cosines of the eight cells, then the sines
  const uint32_t c8 = c16 & 7u, cs = c16 >> 3;
  const T *cf = coef + (static_cast<size_t>(tile) * H.stride + rad.off) * 8;
  constexpr uint32_t kRow = 256 * sizeof(T);  // from a degree to the next but one
  const uint32_t brow = g * kRow + c16 * sizeof(T);
  const T *leg = H.leg + (static_cast<size_t>(gr.leg) + rt * gr.leg_n) * 64 + lane;
  // the FP64 factors of the sets' lowest orders (mixed, the last two waves)
  const bool low = F && wave >= NW - 2;
  uint32_t at64[2] = {0u, 0u};
  if (low) {
#pragma unroll
    for (uint32_t set = 0; set < 2; ++set)
      at64[set] = gr.leg64 + rt * gr.leg64_n +
                  H.mup64[gr.mup64 + 2 * set + wave - (NW - 2)].x;
  }
  for (uint32_t pass = 0; pass < (F ? 1u : 2u); ++pass) {
    v4 E[2][NR][NPT];
#pragma unroll
    for (uint32_t set = 0; set < 2; ++set) {
      // the Fourier matrix of the set, as far as this node's degrees go
      for (uint32_t e = wave; e < 2 * NPT * KC; e += NW) {
        const uint32_t pc = e / KC, ks = e - pc * KC;  // pc: 2 pt + cs
        const uint32_t from = pc < 2 * gr.trig_t ? pc : pc & 1u;
        tr[e * 64 + lane] =
            H.trig[(static_cast<size_t>(gr.trig) +
                    (2 * from + set) * gr.trig_k + ks) * 64 + lane];
      }
      // (1) degrees l0, l0 + 2, ... of a parity: the first 16 in flight
      T la[NP][4], lb[NP][4];
      auto degrees = [&](uint32_t mu, uint32_t par, uint32_t &l0) {
        l0 = mu + ((mu ^ par) & 1u);
        return l0 < N ? (N - l0 + 1) / 2 : 0u;
      };
      auto fetch = [&](uint32_t mu) {
#pragma unroll
        for (uint32_t pp = 0; pp < NP; ++pp) {
          const uint32_t par = F ? pp : pass;
          uint32_t l0;
          const uint32_t n = degrees(mu, par, l0);
          const T *A = leg + H.mup[gr.mup + 2 * mu + par].x * 64;
          const T *B = cf + (n ? harm_block(mu >> 3, l0, N) * 16 +
                                     2 * (mu & 7u) : 0u) * 8;
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u) {
            la[pp][u] = A[u * 64];  // (the table ends with four more steps)
            lb[pp][u] = harm_ranged(B, n * kRow, brow + 4 * u * kRow);
          }
        }
      };
      // the lowest order of the set (mixed): the same products in FP64, by
      // the last two waves, which have fewer orders than the first ones
      const uint32_t m0 = F && wave == 0 ? NW : wave;
      if (2 * m0 + set < N) fetch(2 * m0 + set);
      if (low) {
        const uint32_t par = wave - (NW - 2);
        uint32_t l0;
        const uint32_t n = degrees(set, par, l0);
        const double *A = H.leg64 + static_cast<size_t>(at64[set]) * 64 + lane;
        const T *B = cf + (n ? harm_block(0, l0, N) * 16 + 2 * set : 0u) * 8;
        harm_d4 acc = {0.0, 0.0, 0.0, 0.0};
        for (uint32_t k = 0; k < n; k += 16) {
          double x[4];
          T y[4];
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u) {
            x[u] = A[(k + 4 * u) * 16];  // (four more steps in the table)
            y[u] = harm_ranged(B, n * kRow, brow + (k + 4 * u) * kRow);
          }
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u)
            acc = Harm<double>::mfma(x[u], static_cast<double>(y[u]), acc);
        }
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r)
          Gm[Harm<double>::row(g, r) * RS + cs * sines + c8 * 2 + par] =
              static_cast<T>(acc[r]);
      }
      for (uint32_t m = m0; m < MH; m += NW) {
        const uint32_t mu = 2 * m + set;
        const uint32_t mode = cs * sines + m * 16;
        v4 acc[NP];
#pragma unroll
        for (uint32_t pp = 0; pp < NP; ++pp)
          acc[pp] = v4{T(0), T(0), T(0), T(0)};
        if (mu < N) {
          T xa[NP][4], xb[NP][4];
#pragma unroll
          for (uint32_t pp = 0; pp < NP; ++pp)
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
              xa[pp][u] = la[pp][u];
              xb[pp][u] = lb[pp][u];
            }
          if (mu + 2 * NW < N) fetch(mu + 2 * NW);
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u)
#pragma unroll
            for (uint32_t pp = 0; pp < NP; ++pp)
              acc[pp] = M::mfma(xa[pp][u], xb[pp][u], acc[pp]);
#pragma unroll
          for (uint32_t pp = 0; pp < NP; ++pp) {
            const uint32_t par = F ? pp : pass;
            uint32_t l0;
            const uint32_t n = degrees(mu, par, l0);
            if (n > 16) {
              const T *A = leg + H.mup[gr.mup + 2 * mu + par].x * 64;
              const T *B =
                  cf + (harm_block(mu >> 3, l0, N) * 16 + 2 * (mu & 7u)) * 8;
              for (uint32_t k = 16; k < n; k += 4)
                acc[pp] = M::mfma(
                    A[k * 16], harm_ranged(B, n * kRow, brow + k * kRow),
                    acc[pp]);
            }
          }
        }
#pragma unroll
        for (uint32_t pp = 0; pp < NP; ++pp)
#pragma unroll
          for (uint32_t r = 0; r < 4; ++r) {
            const uint32_t ring = M::row(g, r);
            if (F)
              Gm[ring * RS + mode + c8 * 2 + pp] = acc[pp][r];
            else
              Gm[(ring >> 1) * RS + mode + (ring & 1u) * 8 + c8] = acc[pp][r];
          }
      }
      harm_barrier();
      // (2)
      v4 X[2][NR][NPT];  // cosines, sines
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int u = 0; u < NR; ++u)
#pragma unroll
          for (int pt = 0; pt < NPT; ++pt)
            X[c][u][pt] = v4{T(0), T(0), T(0), T(0)};
      const T *At = tr + lane, *Bt = Gm + wave * RS + lane;
      // (a wave whose first row is past the rings has nothing to do)
      const bool some = 16 * rt + (F ? wave : 2 * wave) < gr.nring;
#pragma unroll 2
      for (uint32_t ks = 0; some && ks < KC; ++ks) {
        T a[2][NPT], b[2][NR];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
          for (int pt = 0; pt < NPT; ++pt)
            a[c][pt] = At[((2 * pt + c) * KC + ks) * 64];
#pragma unroll
          for (int u = 0; u < NR; ++u)
            b[c][u] = Bt[u * NW * RS + c * sines + ks * 64];
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int u = 0; u < NR; ++u)
#pragma unroll
            for (int pt = 0; pt < NPT; ++pt)
              X[c][u][pt] = M::mfma(a[c][pt], b[c][u], X[c][u][pt]);
      }
      harm_barrier();
      if (set == 0) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int u = 0; u < NR; ++u)
#pragma unroll
            for (int pt = 0; pt < NPT; ++pt) E[c][u][pt] = X[c][u][pt];
      } else {
        // bytes of an azimuth: a ring's offsets fit 32 bits
        const uint32_t az =
            static_cast<uint32_t>(2 * ncp * sizeof(T));
#pragma unroll
        for (int u = 0; u < NR; ++u) {
          const uint32_t row = wave + u * NW;
          const uint32_t ring0 = 16 * rt + (F ? row : 2 * row);
          if (ring0 >= gr.nring) continue;
          const uint32_t dir0 =
              gr.equator ? (ring0 ? gr.h + 2 * gr.h * (ring0 - 1) : 0u)
                         : 2 * gr.h * ring0;
          char *base = reinterpret_cast<char *>(
              S + harm_slot<T>(gr.node0 + rad.idx * nd + dir0, cell0,
                               F ? 0u : pass, ncp));
          bool eq = gr.equator && ring0 == 0, on = true;
          uint32_t off = c16 * 4;
          if (!F) {  // lanes 8 .. 15 of a row: the next ring
            const bool next = c16 >> 3;
            off = (c16 & 7u) * 8 + (next ? (eq ? gr.h : 2 * gr.h) * az : 0u);
            on = !next || ring0 + 1 < gr.nring;
            eq = eq && !next;
          }
#pragma unroll
          for (int pt = 0; pt < NPT; ++pt)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
              const uint32_t phi = 16 * pt + M::row(g, r);
              const T ec = E[0][u][pt][r], es = E[1][u][pt][r];
              const T oc = X[0][u][pt][r], os = X[1][u][pt][r];
              auto put = [&](uint32_t k, T e, T o) {
                const uint32_t oa = off + k * az;
                *reinterpret_cast<T *>(base + oa) = e + o;
                if (!eq) *reinterpret_cast<T *>(base + oa + gr.h * az) = e - o;
              };
              if (2 * phi <= gr.h && on) put(phi, ec + es, oc + os);
              if (phi > 0 && 2 * phi < gr.h && on)
                put(gr.h - phi, ec - es, os - oc);
            }
        }
      }
    }
  }
  uint32_t any = 0;
  for (uint32_t c = 0; c < kHarmCells; ++c)
    if (cell0 + c < ncell) any |= outside[cell0 + c];
  if (!any) return;
  // atoms outside the unit ball: their terms one by one, 64 atoms of every cell
  // at a time (wave c lists those of cell c)
  uint32_t *list = reinterpret_cast<uint32_t *>(smem);
  const uint32_t d0 = rt ? 32 * gr.h * rt - (gr.equator ? gr.h : 0u) : 0u;
  const uint32_t d1 =
      32 * gr.h * (rt + 1) - (gr.equator ? gr.h : 0u) < nd
          ? 32 * gr.h * (rt + 1) - (gr.equator ? gr.h : 0u)
          : nd;
  uint32_t most = 0;
  for (uint32_t c = 0; c < kHarmCells; ++c)
    if (cell0 + c < ncell && outside[cell0 + c]) {
      const uint32_t n = start[cell0 + c + 1] - start[cell0 + c];
      most = n > most ? n : most;
    }
  for (uint32_t p0 = 0; p0 < most; p0 += 64) {
    __syncthreads();
    for (uint32_t c = wave; c < kHarmCells; c += NW) {
      uint32_t n = 0;
      if (cell0 + c < ncell && outside[cell0 + c])
        n = start[cell0 + c + 1] - start[cell0 + c];
      n = n > p0 ? n - p0 : 0u;
      harm_list_outside(H, atoms, n ? start[cell0 + c] + p0 : 0u,
                        n < 64 ? n : 64u, harm_centre(cell0 + c, ny, nz, h),
                        list + 65 * c);
    }
    __syncthreads();
    for (uint32_t e = tid; e < (d1 - d0) * kHarmCells; e += kHarmBlock) {
      const uint32_t c = e & (kHarmCells - 1), cell = cell0 + c;
      const uint32_t n = list[65 * c];
      if (n == 0) continue;
      const uint32_t node = gr.node0 + rad.idx * nd + d0 + e / kHarmCells;
      const double4 k = k64[node];
      const HarmCentre cc = harm_centre(cell, ny, nz, h);
      double re = 0.0, im = 0.0;
      for (uint32_t q = 0; q < n; ++q) {
        const HarmOffset d = harm_offset(atoms, list[65 * c + 1 + q], cc);
        const double ph = k.x * d.x + k.y * d.y + k.z * d.z;
        re += d.q * cos(ph);
        im -= d.q * sin(ph);
      }
      T *sr = S + harm_slot<T>(node, cell, 0, ncp);
      T *si = S + harm_slot<T>(node, cell, 1, ncp);
      *sr += static_cast<T>(re);
      *si += static_cast<T>(im);
    }
  }
}

template <typename T, int NPT>
__global__ __launch_bounds__(kHarmBlock) void harm_sf_kernel(
    HarmDev<T> H, const uint2 *__restrict__ units, uint32_t nunit,
    const typename HarmRecord<T>::type *__restrict__ atoms,
    const uint32_t *__restrict__ start, const double4 *__restrict__ k64,
    uint32_t ny, uint32_t nz, double h, uint32_t ncell,
    const T *__restrict__ coef, const uint32_t *__restrict__ outside,
    T *__restrict__ S) {
  extern __shared__ char harm_smem[];
  uint32_t unit, tile;
  if (!harm_place(blockIdx.x, (ncell + kHarmCells - 1) / kHarmCells, nunit,
                  unit, tile))
    return;
  const uint2 u = units[unit];
  const HarmRad rad = H.rad[u.x];
  const HarmGroup gr = H.grp[rad.group];
  // tiles of 16 azimuths up to pi / 2
  harm_switch<NPT>(gr.trig_t, [&](auto npt) {
    harm_sf_body<T, decltype(npt)::value>(H, atoms, start, k64, ny, nz, h,
                                          ncell, rad, gr, u.y, tile, coef,
                                          outside, S, harm_smem);
  });
}

// ---------------------------------------------------------------------------
// remote sums -> coefficients (436 and 1,162 us; mixed 420 with the lowest
// orders in FP32 too, before that 438 and 1,311 with the azimuths
// up to pi summed one by one and every group in the registers of the largest;
// reads R once, 0.15 and 0.29 ms, all loads of a workgroup in flight, then the
// phases between barriers as in harm_sf)

// One unit: eight cells, one radial node, all rings; the transpose of
// harm_sf_body.  Every wave first loads its rings' values, all loads in
// flight at once (RW rows of 4 HK values per lane; FP64 rows are pairs of
// rings, and Re and Im take turns).  Even and odd orders take turns, so that
// all the rings' Fourier sums of one set fit in LDS: (1) per ring, f =
// V(phi) +- V(phi + pi), and f(phi) +- f(pi - phi) summed over the azimuths up
// to pi / 2 against the cosines and, with the other sign, the sines;
// (2) per order and parity, the sums over the rings against the Legendre
// functions, stored as the cells' coefficients.  The mixed path keeps the ring
// sums of each set's lowest order apart (`low`) and sums them over the rings in
// FP64 at the end, when the registers of the loaded values are free (inside
// the loop over the sets it spilled 120 of them: 3,824 against 4,461 us for
// the way back at 1.0M charges).
constexpr uint32_t kHarmLowRow = 40;  // scalars of a ring
template <typename T, int RW, int HK, int MT>
__device__ __forceinline__ void harm_lr_body(
    const HarmDev<T> &H, uint32_t ncell, const HarmRad &rad,
    const HarmGroup &gr, uint32_t tile, const T *R, T *coef, char *smem) {
  using M = Harm<T>;
  using v4 = typename M::v4;
  constexpr bool F = sizeof(T) == 4;
  constexpr uint32_t NW = kHarmBlock / 64;
  constexpr int NP = F ? 2 : 1;  // parities per pass of (2)
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t c16 = lane & 15u, g = lane >> 4;
  const uint32_t N = rad.N, MS = 8 * harm_order_steps(N);
  const uint32_t RS = MS * 16 + 8;
  const uint32_t hk = gr.trigt_k;
  const uint32_t nrow = F ? 4 * gr.legt_k : 2 * gr.legt_k;  // padded rings
  T *Gm = reinterpret_cast<T *>(smem);
  T *low = Gm + nrow * RS;  // mixed: [set][ring], the set's lowest order
  T *tr = low + (F ? 2 * nrow * kHarmLowRow : 0u);
  const uint32_t cell0 = tile * kHarmCells;
  const uint32_t ncp = harm_row(ncell);
  // columns of (2): the cosines of the eight cells, then the sines
  const uint32_t c8 = c16 & 7u, cs = c16 >> 3;
  T *cf = coef + (static_cast<size_t>(tile) * H.stride + rad.off) * 8 + c16;
  const T *legt = H.legt + static_cast<size_t>(gr.legt) * 64 + lane;
  // bytes of an azimuth: a row's offsets stay below 4 h of them (32 bits)
  const uint32_t az = static_cast<uint32_t>(2 * ncp * sizeof(T));
  const uint32_t nd = harm_dirs(gr);
  // the FP64 factors of a set's lowest order, waves (set, parity)
  // (asked for ahead of the last phase, except where the registers are held
  // to most waves)
  constexpr bool PRE = F && RW > 2;
  auto factors64 = [&] {
    return H.legt64 + lane +
           (static_cast<size_t>(gr.legt64) + H.mup64[gr.mup64 + wave].y) * 64;
  };
  double x64[4] = {};
  for (uint32_t pass = 0; pass < (F ? 1u : 2u); ++pass) {
    // A row past the rings and an azimuth past pi / 2 repeat the last one
    // (their factors are zero); the equator has no second half.  phi = 0 and
    // pi / 2 have no partner at pi - phi.
    T va[RW][HK], vb[RW][HK], wa[RW][HK], wb[RW][HK];
#pragma unroll
    for (int w = 0; w < RW; ++w) {
      const uint32_t ring0 = F ? wave + w * NW : 2 * (wave + w * NW);
      const uint32_t r0 = ring0 < gr.nring ? ring0 : gr.nring - 1;
      const uint32_t dir0 =
          gr.equator ? (r0 ? gr.h + 2 * gr.h * (r0 - 1) : 0u) : 2 * gr.h * r0;
      const T *base = R + harm_slot<T>(gr.node0 + rad.idx * nd + dir0, cell0,
                                       F ? 0u : pass, ncp);
      const bool eq = gr.equator && r0 == 0;
      uint32_t off = c16 * 4, second = eq ? 0u : gr.h * az;
      if (!F) {  // lanes 8 .. 15 of a row: the next ring
        const bool next = (c16 >> 3) && r0 + 1 < gr.nring;
        off = (c16 & 7u) * 8 + (next ? (eq ? gr.h : 2 * gr.h) * az : 0u);
        if (next) second = gr.h * az;
      }
#pragma unroll
      for (int ks = 0; ks < HK; ++ks) {
        const uint32_t k = 4 * ks + g < gr.h / 2 ? 4 * ks + g : gr.h / 2;
        const bool two = k > 0 && 2 * k < gr.h;
        const uint32_t o = off + k * az;
        const uint32_t p = off + (two ? gr.h - k : k) * az;
        va[w][ks] = harm_at_byte(base, o);
        vb[w][ks] = harm_at_byte(base, o + second);
        const T x = harm_at_byte(base, p), y = harm_at_byte(base, p + second);
        wa[w][ks] = two ? x : T(0);
        wb[w][ks] = two ? y : T(0);
      }
    }
    if (pass == 0) {
      for (uint32_t e = wave; e < 4 * MT * HK; e += NW) {
        const uint32_t sm = e / HK, ks = e - sm * HK;
        const uint32_t sc = sm / MT, mt = sm - sc * MT;  // sc: 2 set + cs
        const T x = H.trigt[(static_cast<size_t>(gr.trigt) +
                             (sc * gr.trigt_m + mt) * hk +
                             (ks < hk ? ks : 0u)) * 64 + lane];
        tr[e * 64 + lane] = ks < hk ? x : T(0);
      }
      harm_barrier();
    }
    for (uint32_t set = 0; set < 2; ++set) {
      T la[NP][4];
      auto fetch = [&](uint32_t mu) {
#pragma unroll
        for (uint32_t pp = 0; pp < NP; ++pp) {
          const T *A = legt + H.mup[gr.mup + 2 * mu + (F ? pp : pass)].y * 64;
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u) la[pp][u] = A[u * 64];
        }
      };
      // (mixed: the lowest order comes last, in FP64)
      const uint32_t m0 = F && wave == 0 ? NW : wave;
      if (2 * m0 + set < N) fetch(2 * m0 + set);
      // (1)
#pragma unroll
      for (int w = 0; w < RW; ++w) {
        const uint32_t row = wave + w * NW;
        const uint32_t ring = F ? row : 2 * row + (c16 >> 3);
        const T half2 = gr.equator && ring == 0 ? T(0) : set ? T(-1) : T(1);
        v4 acc[2][MT];  // cosines, sines
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[0][m] = acc[1][m] = v4{T(0), T(0), T(0), T(0)};
        const T *At = tr + 2 * set * MT * HK * 64 + lane;
#pragma unroll
        for (int ks = 0; ks < HK; ++ks) {
          const T f = harm_fma(half2, vb[w][ks], va[w][ks]);
          const T b = harm_fma(half2, wb[w][ks], wa[w][ks]);
          const T v[2] = {set ? f - b : f + b, set ? f + b : f - b};
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int m = 0; m < MT; ++m)
              acc[c][m] =
                  M::mfma(At[((c * MT + m) * HK + ks) * 64], v[c], acc[c][m]);
        }
        if (row < nrow) {
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
              for (uint32_t r = 0; r < 4; ++r) {
                const uint32_t mode = 2 * (16 * m + M::row(g, r)) + c;
                uint32_t to = row * RS + mode * 16 + c16;
                if (F && m == 0 && r == 0 && g == 0)  // order `set`
                  to = (nrow * RS + (set * nrow + row) * kHarmLowRow) +
                       c * 16 + c16;
                if (mode < MS) Gm[to] = acc[c][m][r];
              }
        }
      }
      harm_barrier();
      // (2)
      if (PRE && set == 1 && wave < 4) {
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) x64[u] = factors64()[u * 64];
      }
      for (uint32_t m = m0; 2 * m + set < N; m += NW) {
        const uint32_t mu = 2 * m + set;
        const uint32_t mode = 2 * m + cs;
        T xa[NP][4];
#pragma unroll
        for (uint32_t pp = 0; pp < NP; ++pp)
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u) xa[pp][u] = la[pp][u];
        if (mu + 2 * NW < N) fetch(mu + 2 * NW);
        auto ring_sum = [&](uint32_t ks, uint32_t par) {
          const uint32_t ring = 4 * ks + g;
          return F ? Gm[ring * RS + mode * 16 + c8 * 2 + par]
                   : Gm[(ring >> 1) * RS + mode * 16 + (ring & 1u) * 8 + c8];
        };
        v4 acc[NP];
#pragma unroll
        for (uint32_t pp = 0; pp < NP; ++pp)
          acc[pp] = v4{T(0), T(0), T(0), T(0)};
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
#pragma unroll
          for (uint32_t pp = 0; pp < NP; ++pp)
            acc[pp] = M::mfma(xa[pp][u], ring_sum(u, F ? pp : pass), acc[pp]);
#pragma unroll
        for (uint32_t pp = 0; pp < NP; ++pp) {
          const uint32_t par = F ? pp : pass;
          const uint32_t l0 = mu + ((mu ^ par) & 1u);
          if (l0 >= N) continue;
          const uint32_t n = (N - l0 + 1) / 2;
          const T *A = legt + H.mup[gr.mup + 2 * mu + par].y * 64;
          T *o = cf + (harm_block(mu >> 3, l0, N) * 16 + 2 * (mu & 7u)) * 8;
          // rings past the first 16, degrees past the first 16 of a parity
          for (uint32_t k = 4; k < gr.legt_k; ++k)
            acc[pp] = M::mfma(A[k * 64], ring_sum(k, par), acc[pp]);
#pragma unroll
          for (uint32_t r = 0; r < 4; ++r) {
            const uint32_t i = M::row(g, r);
            if (i < n) o[i * 256] = acc[pp][r];
          }
          for (uint32_t i0 = 16; i0 < n; i0 += 16) {
            A += gr.legt_k * 64;
            v4 more = {T(0), T(0), T(0), T(0)};
            for (uint32_t k = 0; k < gr.legt_k; ++k)
              more = M::mfma(A[k * 64], ring_sum(k, par), more);
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
              const uint32_t i = i0 + M::row(g, r);
              if (i < n) o[i * 256] = more[r];
            }
          }
        }
      }
      harm_barrier();
    }
  }
  if constexpr (F) {
    // (2) of the lowest order of each set in FP64, wave (set, parity)
    const uint32_t set = wave >> 1, par = wave & 1u;
    const uint32_t l0 = set + ((set ^ par) & 1u);
    if (set < 2 && l0 < N) {
      const uint32_t n = (N - l0 + 1) / 2;
      const double *A = factors64();
      const T *sums = low + set * nrow * kHarmLowRow + cs * 16 + c8 * 2 + par;
      T *o = cf + (harm_block(0, l0, N) * 16 + 2 * set) * 8;
      for (uint32_t i0 = 0; i0 < n; i0 += 16) {
        harm_d4 acc = {0.0, 0.0, 0.0, 0.0};
        for (uint32_t k = 0; k < gr.legt_k; k += 4) {
          if (!PRE || i0 + k > 0) {
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u)
              x64[u] = A[(k + u < gr.legt_k ? k + u : k) * 64];
          }
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u)
            if (k + u < gr.legt_k)
              acc = Harm<double>::mfma(
                  x64[u],
                  static_cast<double>(sums[(4 * (k + u) + g) * kHarmLowRow]),
                  acc);
        }
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
          const uint32_t i = i0 + Harm<double>::row(g, r);
          if (i < n) o[i * 256] = static_cast<T>(acc[r]);
        }
        A += gr.legt_k * 64;
      }
    }
  }
}

// Classes of groups by the steps of four azimuths up to pi / 2, which bound the
// rings too: rows per wave, and steps, of class c.
template <typename T>
constexpr int harm_lr_rows(int c) {
  return sizeof(T) == 4 ? c + 1 : c == 1 ? 1 : 2;
}
constexpr int harm_lr_steps(int c) { return c == 1 ? 4 : c == 2 ? 6 : 8; }
__host__ __device__ constexpr int harm_lr_class(uint32_t hk) {
  return hk <= 4 ? 1 : hk <= 6 ? 2 : 3;
}
// Waves per SIMD the registers are held to: two workgroups per CU pay for the
// spills of the mixed class 2 (181 to 118 us at 10,000 waters, 2.55 to 1.70 ms
// at 1.0M charges) and the FP64 class 1 (1,288 to 1,162 us at 288,000
// charges), not for those of the others (FP64 class 2 410 to 828 us).
template <typename T>
constexpr int harm_lr_waves(int c) {
  return sizeof(T) == 4 ? (c == 1 ? 5 : c == 2 ? 4 : 2) : (c == 1 ? 4 : 2);
}
// C: the largest class of the plan's groups.
template <typename T, int C>
__global__ __launch_bounds__(kHarmBlock, harm_lr_waves<T>(C)) void harm_lr_kernel(
    HarmDev<T> H, uint32_t ncell, const T *__restrict__ R,
    T *__restrict__ coef) {
  extern __shared__ char harm_smem[];
  uint32_t unit, tile;
  if (!harm_place(blockIdx.x, (ncell + kHarmCells - 1) / kHarmCells, H.nrad,
                  unit, tile))
    return;
  const HarmRad rad = H.rad[unit];
  const HarmGroup gr = H.grp[rad.group];
  harm_switch<C>(harm_lr_class(gr.trigt_k), [&](auto cls) {
    constexpr int c = decltype(cls)::value;
    constexpr int RW = harm_lr_rows<T>(c), HK = harm_lr_steps(c), LK = HK - 1;
    // tiles of 16 orders of a set
    harm_switch<2>((harm_order_steps(rad.N) + 3) / 4, [&](auto mt) {
      constexpr int MT = decltype(mt)::value;
      if (gr.trigt_k <= LK)
        harm_lr_body<T, RW, LK, MT>(H, ncell, rad, gr, tile, R, coef,
                                    harm_smem);
      else
        harm_lr_body<T, RW, HK, MT>(H, ncell, rad, gr, tile, R, coef,
                                    harm_smem);
    });
  });
}

// ---------------------------------------------------------------------------
// coefficients -> energies and forces

// Fields of the atoms outside their cell's ball: the direct sums over the nodes,
// four atoms and four nodes at a time (the nodes' remote sums lie rows apart),
// before the evaluation.  The nodes of a cell are shared out to kHarmSlices
// workgroups: workgroup b takes slice j of cell b - j, so that the grid stays
// one workgroup per cell and most find nothing to do.  The slices' sums go to
// the cell's coefficients, which are free by then, and the evaluation adds them
// up; a cell of more atoms than fit there is left to one workgroup, which
// stores the fields itself.  With an atom beyond the box's corner, an FP64 step
// of 2,000 waters at rcut 8, tol 1e-6 takes 2.38 ms, 2.94 with one workgroup for
// all nodes of a cell, 2.73 with direct sums for all (1.83 without that atom).
constexpr uint32_t kHarmSlices = 16;
template <typename T>
__device__ __forceinline__ bool harm_sliced(const HarmDev<T> &H, uint32_t na) {
  return na * kHarmSlices * sizeof(double4) <= H.stride * sizeof(T);
}
// [atom of the cell][slice]
template <typename T>
__device__ __forceinline__ double4 *harm_slices(const HarmDev<T> &H, T *coef,
                                                uint32_t cell) {
  return reinterpret_cast<double4 *>(coef + static_cast<size_t>(cell) * H.stride);
}
template <typename T>
__global__ __launch_bounds__(kHarmBlock) void harm_outside_kernel(
    HarmDev<T> H, const typename HarmRecord<T>::type *__restrict__ atoms,
    const uint32_t *__restrict__ start, const double4 *__restrict__ k64,
    uint32_t K, uint32_t ny, uint32_t nz, double h, uint32_t ncell,
    const T *__restrict__ R, const uint32_t *__restrict__ outside,
    T *__restrict__ coef, double4 *__restrict__ out) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  // (a far field has at least 27 cells, more than the slices)
  auto cell_of = [&](uint32_t j) {
    return blockIdx.x < j ? blockIdx.x + ncell - j : blockIdx.x - j;
  };
  unsigned long long todo =
      __ballot(lane < kHarmSlices && outside[cell_of(lane % kHarmSlices)]);
  if (!todo) return;
  __shared__ uint32_t list[65];
  __shared__ double red[kHarmBlock / 64][16];
  const uint32_t ncp = harm_row(ncell);
  for (; todo; todo &= todo - 1) {
    const uint32_t slice = static_cast<uint32_t>(__ffsll(todo)) - 1;
    const uint32_t cell = cell_of(slice);
    const uint32_t a0 = start[cell], na = start[cell + 1] - a0;
    const bool sliced = harm_sliced(H, na);
    if (!sliced && slice > 0) continue;
    const uint32_t per = sliced ? (K + kHarmSlices - 1) / kHarmSlices : K;
    const uint32_t k0 = slice * per < K ? slice * per : K;
    const uint32_t k1 = k0 + per < K ? k0 + per : K;
    const HarmCentre cc = harm_centre(cell, ny, nz, h);
    for (uint32_t p0 = 0; p0 < na; p0 += 64) {
      __syncthreads();
      if (wave == 0)
        harm_list_outside(H, atoms, a0 + p0, na - p0 < 64 ? na - p0 : 64u, cc,
                          list);
      __syncthreads();
      const uint32_t cnt = list[0];
      for (uint32_t q0 = 0; q0 < cnt; q0 += 4) {
        HarmOffset a[4];
        double v[16];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q)
          a[q] = harm_offset(atoms, list[1 + (q0 + q < cnt ? q0 + q : q0)], cc);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = 0.0;
        for (uint32_t n0 = k0 + tid; n0 < k1; n0 += 4 * kHarmBlock) {
          double4 k[4];
          double vr[4], vi[4];
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t n = n0 + u * kHarmBlock;
            const uint32_t m = n < k1 ? n : n0;
            k[u] = k64[m];
            vr[u] = R[harm_slot<T>(m, cell, 0, ncp)];
            vi[u] = R[harm_slot<T>(m, cell, 1, ncp)];
            if (n >= k1) vr[u] = vi[u] = 0.0;
          }
#pragma unroll
          for (uint32_t q = 0; q < 4; ++q) {
            if (q0 + q >= cnt) break;  // uniform
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
              const double ph =
                  k[u].x * a[q].x + k[u].y * a[q].y + k[u].z * a[q].z;
              const double c = cos(ph), s = sin(ph);
              const double b = c * vi[u] + s * vr[u];
              v[4 * q] += k[u].x * b;
              v[4 * q + 1] += k[u].y * b;
              v[4 * q + 2] += k[u].z * b;
              v[4 * q + 3] += c * vr[u] - s * vi[u];
            }
          }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          for (int o = 32; o > 0; o >>= 1) v[i] += __shfl_xor(v[i], o, 64);
          if (lane == 0) red[wave][i] = v[i];
        }
        __syncthreads();
        if (tid < 4 && q0 + tid < cnt) {
          double t[4] = {0.0, 0.0, 0.0, 0.0};
          for (uint32_t w = 0; w < kHarmBlock / 64; ++w)
            for (uint32_t d = 0; d < 4; ++d) t[d] += red[w][4 * tid + d];
          const uint32_t i = list[1 + q0 + tid];
          if (sliced) {
            harm_slices(H, coef, cell)[(i - a0) * kHarmSlices + slice] =
                make_double4(t[0], t[1], t[2], t[3]);
          } else {
            const double q = harm_offset(atoms, i, cc).q;
            out[i] = make_double4(q * t[0], q * t[1], q * t[2], q * t[3]);
          }
        }
        __syncthreads();
      }
    }
  }
}

// Uniform loads of constant data.
template <typename T>
using HarmConst = const __attribute__((address_space(4))) T;
template <typename T>
__device__ __forceinline__ HarmConst<T> *harm_const(const T *p) {
  return reinterpret_cast<HarmConst<T> *>(reinterpret_cast<uintptr_t>(p));
}

// One workgroup per cell and 64 of its atoms at a time, a lane per atom.  Wave
// w takes the azimuthal orders w, 2W - 1 - w, 2W + w, ... (W waves: their
// lengths N - mu add up to nearly the same everywhere), at most MO of them,
// and walks the degrees l: the radial values R_{l,p} and their derivatives in
// registers, then per order the sums F = sum_p R U, F' = sum_p R' U over the
// contracted coefficients and the recurrences of the Legendre part M_l and of
// its derivative in s.  The coefficients are the same for all lanes and come as
// scalar operands; one vector load per 128-byte line at the start brings them
// into the L2 cache, where the scalar loads find them.  The terms of a degree,
// then the waves, meet in FP64.
template <typename T, int W, int MO, int PM>
__device__ __forceinline__ void harm_eval_body(
    const HarmDev<T> &H, const typename HarmRecord<T>::type *atoms, uint32_t a0,
    uint32_t na, const HarmCentre &cc, const T *U, const double4 *slices,
    double4 *out, double *red) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t N = H.N;
  HarmAtom<T> a = {};
  if (lane < na) a = harm_atom(H, atoms, a0 + lane, cc);
  uint32_t mu[MO];
  // (x + i y)^mu and ^(mu - 1); M and dM/ds of the last two degrees
  T xc[MO], xs[MO], yc[MO], ys[MO], P1[MO], P2[MO], D1[MO], D2[MO];
  {
    T re = T(1), im = T(0), r1 = T(0), i1 = T(0);
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < MO; ++i) {
      mu[i] = i * W + (i & 1 ? W - 1 - wave : wave);
      for (; m < mu[i] && m < N; ++m) {
        r1 = re;
        i1 = im;
        re = r1 * a.x - i1 * a.y;
        im = r1 * a.y + i1 * a.x;
      }
      xc[i] = re;
      xs[i] = im;
      yc[i] = r1 * static_cast<T>(mu[i]);
      ys[i] = i1 * static_cast<T>(mu[i]);
      P1[i] = P2[i] = D1[i] = D2[i] = T(0);
    }
  }
  double E = 0.0, A1 = 0.0, A2 = 0.0, Gz = 0.0, Hx = 0.0, Hy = 0.0;
  HarmConst<uint32_t> *urow = harm_const(H.urow);
  for (uint32_t l = wave; l < N; ++l) {
    HarmConst<T> *J = harm_const(H.jac + 2 * H.crow[l]);
    HarmConst<T> *rec = harm_const(H.rec + 128 * l);
    const T *Ul = U + 8 * urow[l];
    T e = T(0), f1 = T(0), f2 = T(0), gz = T(0), hx = T(0), hy = T(0);
    const uint32_t PKl = harm_psteps(l, N);
    harm_switch<PM>(PKl, [&](auto steps) {
      constexpr int PK = decltype(steps)::value;
      T R[4 * PK], Q[4 * PK];  // R_{l,p}, dR_{l,p}/dx
      R[0] = T(1);
      Q[0] = T(0);
      R[1] = a.t + J[2];
      Q[1] = T(1);
#pragma unroll
      for (int p = 2; p < 4 * PK; ++p) {
        const T v = a.t + J[2 * p], c2 = J[2 * p + 1];
        R[p] = harm_fma(v, R[p - 1], -c2 * R[p - 2]);
        Q[p] = harm_fma(v, Q[p - 1], harm_fma(-c2, Q[p - 2], R[p - 1]));
      }
#pragma unroll
      for (int i = 0; i < MO; ++i)
        if (mu[i] <= l) {  // uniform
          HarmConst<T> *u = harm_const(Ul + 8 * mu[i] * PK);
          const T b = rec[2 * mu[i]], ez = rec[2 * mu[i] + 1];
          T Fc = u[0], Fs = u[1], Gc = T(0), Gs = T(0);
#pragma unroll
          for (int p = 1; p < 4 * PK; ++p) {
            Fc = harm_fma(R[p], u[2 * p], Fc);
            Fs = harm_fma(R[p], u[2 * p + 1], Fs);
            Gc = harm_fma(Q[p], u[2 * p], Gc);
            Gs = harm_fma(Q[p], u[2 * p + 1], Gs);
          }
          const T one = mu[i] == l ? T(1) : T(0);
          const T m = harm_fma(-(b * a.s), P2[i],
                               harm_fma(a.z, P1[i], one));
          const T d = harm_fma(-b, harm_fma(a.s, D2[i], P2[i]), a.z * D1[i]);
          const T F = harm_fma(Fc, xc[i], Fs * xs[i]);
          const T G = harm_fma(Gc, xc[i], Gs * xs[i]);
          const T hc = harm_fma(Fc, yc[i], Fs * ys[i]);
          const T hs = harm_fma(Fs, yc[i], -Fc * ys[i]);
          gz = harm_fma(ez * P1[i], F, gz);
          e = harm_fma(m, F, e);
          f1 = harm_fma(m, G, f1);
          f2 = harm_fma(d, F, f2);
          hx = harm_fma(m, hc, hx);
          hy = harm_fma(m, hs, hy);
          P2[i] = P1[i];
          P1[i] = m;
          D2[i] = D1[i];
          D1[i] = d;
        }
    });
    E += static_cast<double>(e);
    A1 += static_cast<double>(f1);
    A2 += static_cast<double>(f2);
    Gz += static_cast<double>(gz);
    Hx += static_cast<double>(hx);
    Hy += static_cast<double>(hy);
  }
  // s = x^2 + y^2 + z^2; the derivative of M in z is the full one
  A1 *= H.xk;
  double v[4] = {2.0 * (A1 + A2) * static_cast<double>(a.x) + Hx,
                 2.0 * (A1 + A2) * static_cast<double>(a.y) + Hy,
                 2.0 * A1 * static_cast<double>(a.z) + Gz, E};
  // [wave][component][lane]
#pragma unroll
  for (int d = 0; d < 4; ++d) red[(4 * wave + d) * 64 + lane] = v[d];
  harm_barrier();
  if (threadIdx.x < 64 && lane < na) {
#pragma unroll
    for (int w = 1; w < W; ++w)
#pragma unroll
      for (int d = 0; d < 4; ++d) v[d] += red[(4 * w + d) * 64 + lane];
    const double q = a.q;
    double f = -q * H.scale;
    if (a.out && slices) {  // (the sums over the nodes)
      f = q;
#pragma unroll
      for (int d = 0; d < 4; ++d) v[d] = 0.0;
#pragma unroll 1
      for (uint32_t j = 0; j < kHarmSlices; ++j) {
        const double4 t = slices[lane * kHarmSlices + j];
        v[0] += t.x;
        v[1] += t.y;
        v[2] += t.z;
        v[3] += t.w;
      }
    }
    if (!a.out || slices)
      out[a0 + lane] = make_double4(f * v[0], f * v[1], f * v[2], q * v[3]);
  }
  harm_barrier();
}

// Workgroup w: set w % nset of 64 atoms of cell w / nset, then every nset-th.
// 400 and 1,545 us (products on the matrix cores over LDS tables of the radial
// values: 835 and 2,764; without the first touch of the lines 497 and 2,947),
// bound by vector instructions: 22 per (degree, order) beyond the sums, and
// each wave forms the radial values anew.
template <typename T, int W, int MO, int PM>
__global__ __launch_bounds__(64 * W) void harm_eval_kernel(
    HarmDev<T> H, const typename HarmRecord<T>::type *__restrict__ atoms,
    const uint32_t *__restrict__ start, uint32_t ny, uint32_t nz, double h,
    uint32_t nset, const T *__restrict__ mom, T *__restrict__ coef,
    double4 *__restrict__ out) {
  __shared__ double red[W * 256];
  const uint32_t nb = gridDim.x, b = blockIdx.x;
  const uint32_t q = nb >> 3, r = nb & 7u, x = b & 7u;
  const uint32_t w = x * q + (x < r ? x : r) + (b >> 3);
  const uint32_t cell = w / nset, set = w - cell * nset;
  const uint32_t a0 = start[cell], na = start[cell + 1] - a0;
  const HarmCentre cc = harm_centre(cell, ny, nz, h);
  const T *U = mom + static_cast<size_t>(cell) * H.ustride;
  T touch[2] = {T(0), T(0)};
  constexpr uint32_t line = 128 / sizeof(T);
#pragma unroll
  for (uint32_t i = 0; i < 2; ++i) {
    const uint32_t e = (threadIdx.x + i * 64 * W) * line;
    if (e < H.ustride) touch[i] = U[e];
  }
  for (uint32_t p0 = 64 * set; p0 < na; p0 += 64 * nset) {
    const uint32_t cnt = na - p0 < 64 ? na - p0 : 64u;
    const double4 *slices =
        harm_sliced(H, na) ? harm_slices(H, coef, cell) + p0 * kHarmSlices
                           : nullptr;
    harm_eval_body<T, W, MO, PM>(H, atoms, a0 + p0, cnt, cc, U, slices, out,
                                 red);
  }
  asm volatile("" ::"v"(touch[0]), "v"(touch[1]));
}

}  // namespace

// ---------------------------------------------------------------------------
// launchers

void prepare_harmonic(size_t lds_limit) {
  const int n = static_cast<int>(lds_limit);
  auto allow = [&](auto *k) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                              hipFuncAttributeMaxDynamicSharedMemorySize, n);
  };
  allow(harm_moments_kernel<float, 16>);
  allow(harm_moments_kernel<double, 16>);
  allow(harm_moments_kernel<double, 24>);
  allow(harm_moments_kernel<double, 32>);
  allow(harm_sf_kernel<float, 1>);
  allow(harm_sf_kernel<float, 2>);
  allow(harm_sf_kernel<double, 1>);
  allow(harm_sf_kernel<double, 2>);
  allow(harm_lr_kernel<float, 1>);
  allow(harm_lr_kernel<float, 2>);
  allow(harm_lr_kernel<float, 3>);
  allow(harm_lr_kernel<double, 1>);
  allow(harm_lr_kernel<double, 2>);
  allow(harm_lr_kernel<double, 3>);
}

template <typename T>
size_t harm_lds_moments(uint32_t N, uint32_t ksteps) {
  const size_t prow = 4 * harm_psteps(0, N), nt = (N + 7) / 8;
  const size_t ch = 4 * ksteps;
  uint32_t jrows = 0;
  for (uint32_t l = 0; l < N; ++l) jrows += 4 * harm_psteps(l, N);
  return (6 * ch + std::max<size_t>(harm_lb<T>() * prow, 16 * nt) * (ch + 4) +
          harm_lb<T>() * 8 * nt + 2 * jrows) * sizeof(T) + 8;
}
template <typename T>
size_t harm_lds_sf(uint32_t N, uint32_t h) {
  const size_t KC = harm_order_steps(N), npt = (h / 2 + 16) / 16;
  return ((sizeof(T) == 4 ? 16 : 8) * (128 * KC + 24) + 2 * npt * KC * 64) *
         sizeof(T);
}
template <typename T>
size_t harm_lds_lr(uint32_t N, uint32_t h, uint32_t nring) {
  const size_t KC = harm_order_steps(N);
  const size_t lk = std::max<size_t>(4, (nring + 3) / 4);
  const size_t top = harm_lr_steps(harm_lr_class((h / 2 + 4) / 4));
  return ((sizeof(T) == 4 ? 4 : 2) * lk * (128 * KC + 8) +
          (sizeof(T) == 4 ? 2 * 4 * lk * kHarmLowRow : 0) +
          4 * ((KC + 3) / 4) * top * 64) *
         sizeof(T);
}
template size_t harm_lds_moments<float>(uint32_t, uint32_t);
template size_t harm_lds_moments<double>(uint32_t, uint32_t);
template size_t harm_lds_sf<float>(uint32_t, uint32_t);
template size_t harm_lds_sf<double>(uint32_t, uint32_t);
template size_t harm_lds_lr<float>(uint32_t, uint32_t, uint32_t);
template size_t harm_lds_lr<double>(uint32_t, uint32_t, uint32_t);

template <typename T>
void harm_moments(const HarmPlanDev &P, const HarmDev<T> &H, const void *atoms,
                  const uint32_t *start, const GridShape &g, T *mom, T *coef,
                  uint32_t *outside, hipStream_t s) {
  auto *at = static_cast<const typename HarmRecord<T>::type *>(atoms);
  const uint32_t block = 64 * ((H.N + 7) / 8);
  auto go = [&](auto *kernel) {
    kernel<<<g.ncell, block, P.lds_moments, s>>>(H, at, start, g.ny, g.nz, g.h,
                                                 mom, outside);
  };
  if constexpr (sizeof(T) == 4) {
    go(harm_moments_kernel<T, 16>);
  } else {
    if (P.ksteps <= 16)
      go(harm_moments_kernel<T, 16>);
    else if (P.ksteps <= 24)
      go(harm_moments_kernel<T, 24>);
    else
      go(harm_moments_kernel<T, 32>);
  }
  const uint32_t nw = (g.ncell + kHarmCells - 1) / kHarmCells * H.npair;
  harm_radial_kernel<T, false>
      <<<(nw + 3) / 4, 256, 0, s>>>(H, g.ncell, nw, mom, coef);
}

template <typename T>
void harm_sf(const HarmPlanDev &P, const HarmDev<T> &H, const void *atoms,
             const uint32_t *start, const double4 *k64, const GridShape &g,
             const T *coef, const uint32_t *outside, T *S, hipStream_t s) {
  const uint32_t nt = (g.ncell + kHarmCells - 1) / kHarmCells;
  auto go = [&](auto *kernel) {
    kernel<<<harm_grid(nt, P.nunit), kHarmBlock, P.lds_sf, s>>>(
        H, P.unit, P.nunit,
        static_cast<const typename HarmRecord<T>::type *>(atoms), start, k64,
        g.ny, g.nz, g.h, g.ncell, coef, outside, S);
  };
  if (P.hsteps <= 4)
    go(harm_sf_kernel<T, 1>);
  else
    go(harm_sf_kernel<T, 2>);
}

template <typename T>
void harm_lr(const HarmPlanDev &P, const HarmDev<T> &H, const GridShape &g,
             const T *R, T *coef, T *mom, hipStream_t s) {
  const uint32_t nt = (g.ncell + kHarmCells - 1) / kHarmCells;
  auto go = [&](auto *kernel) {
    kernel<<<harm_grid(nt, H.nrad), kHarmBlock, P.lds_lr, s>>>(H, g.ncell, R,
                                                               coef);
  };
  const int c = harm_lr_class(P.hsteps);
  if (c == 1)
    go(harm_lr_kernel<T, 1>);
  else if (c == 2)
    go(harm_lr_kernel<T, 2>);
  else
    go(harm_lr_kernel<T, 3>);
  const uint32_t nw = nt * H.npair;
  harm_radial_kernel<T, true>
      <<<(nw + 3) / 4, 256, 0, s>>>(H, g.ncell, nw, coef, mom);
}

template <typename T>
void harm_eval(const HarmPlanDev &P, const HarmDev<T> &H, const void *atoms,
               const uint32_t *start, const double4 *k64, uint32_t K,
               const GridShape &g, const T *mom, const T *R,
               const uint32_t *outside, T *coef, double4 *out, hipStream_t s) {
  auto *at = static_cast<const typename HarmRecord<T>::type *>(atoms);
  const uint32_t ps = harm_psteps(0, H.N);
  auto go = [&](auto waves, auto orders, auto steps) {
    constexpr int W = decltype(waves)::value, MO = decltype(orders)::value;
    harm_eval_kernel<T, W, MO, decltype(steps)::value>
        <<<g.ncell * P.nset, 64 * W, 0, s>>>(
            H, at, start, g.ny, g.nz, g.h, P.nset, mom, coef, out);
  };
  harm_outside_kernel<T><<<g.ncell, kHarmBlock, 0, s>>>(
      H, at, start, k64, K, g.ny, g.nz, g.h, g.ncell, R, outside, coef, out);
  // W MO >= N (N <= 8 ps).  FP32: four waves of twice the orders form the
  // radial values half as often (400 against 439 us at 3,375 cells), eight
  // fill the device on smaller grids (69 against 102 us at 64 cells, 87
  // against 106 at 512, two workgroups each)
  if constexpr (sizeof(T) == 4) {
    if (g.ncell * P.nset >= 2048) {
      harm_host_switch<5>(ps, [&](auto k) {
        constexpr int PM = decltype(k)::value;
        if (H.N <= 8 * PM - 4)
          go(HarmInt<4>{}, HarmInt<2 * PM - 1>{}, k);
        else
          go(HarmInt<4>{}, HarmInt<2 * PM>{}, k);
      });
      return;
    }
  }
  harm_host_switch<sizeof(T) == 4 ? 5 : 7>(
      ps, [&](auto k) { go(HarmInt<8>{}, k, k); });
}

#define GLST_HARM(T)                                                          \
  template void harm_moments<T>(const HarmPlanDev &, const HarmDev<T> &,      \
                                const void *, const uint32_t *,               \
                                const GridShape &, T *, T *, uint32_t *,      \
                                hipStream_t);                                 \
  template void harm_sf<T>(const HarmPlanDev &, const HarmDev<T> &,           \
                           const void *, const uint32_t *, const double4 *,   \
                           const GridShape &, const T *, const uint32_t *,    \
                           T *, hipStream_t);                                 \
  template void harm_lr<T>(const HarmPlanDev &, const HarmDev<T> &,           \
                           const GridShape &, const T *, T *, T *,            \
                           hipStream_t);                                      \
  template void harm_eval<T>(const HarmPlanDev &, const HarmDev<T> &,         \
                             const void *, const uint32_t *, const double4 *, \
                             uint32_t, const GridShape &, const T *,          \
                             const T *, const uint32_t *, T *, double4 *,     \
                             hipStream_t);
GLST_HARM(float)
GLST_HARM(double)
#undef GLST_HARM

}  // namespace dev
}  // namespace glst
