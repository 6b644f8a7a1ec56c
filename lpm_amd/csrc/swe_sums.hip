// Sphere shallow-water direct sums for gfx950: velocity from relative
// vorticity and divergence, the velocity-gradient double dot
// grad(u):grad(u)^T, and the PSE surface Laplacian, per target.  Replaces
// SphereVertexSums / SphereFaceSums with SphereSweDirectSumReducer and
// sphere_swe_velocity_sums (src/lpm_swe_kernels.hpp:334-362, 578-619,
// 723-780, 877-930) plus the Gaussian PSE Laplacian of LaplacianReducer
// (src/lpm_pse.hpp:157-203) on chord distances.
//
// Per pair (target x, source y) with t = x.y, D = 1 - t + eps^2,
// a = zeta A / 4pi, b = sigma A / 4pi and g = y - t x (= (I - x x^T) y):
//   alpha = a / D, beta = b / D, a' = alpha / D, b' = beta / D.
// The reference's 12-tuple sums factor into per-target accumulators
//   Vy = sum alpha y,  Gd = sum a' g g^T,  Vg = sum beta g,
//   Bt = sum beta t,   Gs = sum b' g g^T,
// and the finalisation applies the target-only factors once:
//   u  = -x cross Vy - Vg
//   Mz = E(Vy) + [x]x Gd - (x cross Vy) x^T        (E_ab = e_abc v_c)
//   Ms = Bt (I - x x^T) + x Vg^T - Gs
//   M  = Mz + Ms  (the reference's packed gradient, whose vorticity part
//                  carries grad_kzeta's opposite sign convention)
//   ddot = sum_ab M_ab M_ba.
// These are identities of the pair sums for any x (no |x| = 1 needed):
// with d = y - x and delta = 1 - t, d + delta x = g, x cross d = x cross g,
// d - eps^2 x = g - D x and a' D = alpha, so the vorticity gradient
// sum a' (x cross d)(d - eps^2 x)^T is [x]x Gd - (x cross Vy) x^T, and the
// divergence terms sum b' (d + delta x)(d + delta x)^T, sum beta (d + delta
// x) and sum beta (1 - delta) are Gs, Vg and Bt.  Per pair that is 17 FMAs
// of accumulation and one reciprocal (shared by four pairs in FP64).
// The PSE Laplacian sum_j (s_j - s_i) A_j (4/pi) exp(-|x-y|^2/e^2) / e^4 over
// x.y > 0 is accumulated as L = sum A eta (s_j - s_i) in FP64 by both
// kernels (a second difference: its first-order terms cancel by symmetry,
// which FP32 sums cannot resolve).  Source tiles whose bounding sphere lies
// beyond sqrt(kPseCut) e of every target of a wave are skipped, and so are
// the pairs beyond that radius in the others (their terms are below
// exp(-kPseCut) relative), so the PSE work covers a few percent of the pairs.
#include <hip/hip_runtime.h>

#include <type_traits>

#include <algorithm>
#include <cmath>

#include "internal.hpp"

namespace lpm_amd {

namespace {

constexpr double kInv4Pi = 0.079577471545947667884441881686257181;
constexpr double k4OverPi = 1.2732395447351626861510701069801148;
constexpr int kSweTile = 256;
// mixed kernel: source tiles this many bounding radii from a target of the
// wave (centre = the tile's first source) take the FP64 pair loop
constexpr double kSweNearFp64 = 2.0;
constexpr double kPseCut = 50.0;  // exp(-50) ~ 2e-22

struct SweSrc {
  double4 p;  // y0, y1, y2, a = zeta A / 4pi
  double4 q;  // b = sigma A / 4pi, A, s, 0
};

// Bounding sphere (centroid, radius^2) of a wave's run of 64 sources, the first
// n of them real (zero records pad the last run).
__device__ __forceinline__ void swe_run_sphere(const double4& y, int n,
                                               double4* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const bool real = lane < n;
  double v[3] = {y.x, y.y, y.z};
#pragma unroll
  for (int k = 0; k < 3; ++k)
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
  const double m = 1.0 / min(64, n);
  const double c0 = v[0] * m, c1 = v[1] * m, c2 = v[2] * m;
  const double a = y.x - c0, b = y.y - c1, e = y.z - c2;
  double r2 = real ? a * a + b * b + e * e : 0.0;
  for (int off = 32; off > 0; off >>= 1) r2 = fmax(r2, __shfl_xor(r2, off, 64));
  if (lane == 0) *out = make_double4(c0, c1, c2, r2);
}

// Packs the undivided faces; with `runs` also the bounding sphere of each run
// of 64.
__global__ __launch_bounds__(256) void swe_pack_kernel(
    const double* __restrict__ sx, int64_t es, int64_t cs,
    const double* __restrict__ zeta, const double* __restrict__ sigma,
    const double* __restrict__ area, const double* __restrict__ surf,
    const int32_t* __restrict__ inv, const int32_t* __restrict__ count,
    int64_t n_pad, SweSrc* __restrict__ out, double4* __restrict__ runs) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (r >= n_pad) return;
  SweSrc s;
  s.p = make_double4(0.0, 0.0, 0.0, 0.0);
  s.q = make_double4(0.0, 0.0, 0.0, 0.0);
  const int64_t n = *count;
  if (r < n) {
    // zero records pad the last tile: kernels may read whole tiles
    const int64_t i = inv ? inv[r] : r;
    const double* p = sx + i * es;
    const double A = area[i];
    s.p = make_double4(p[0], p[cs], p[2 * cs], zeta[i] * A * kInv4Pi);
    s.q = make_double4(sigma[i] * A * kInv4Pi, A, surf ? surf[i] : 0.0, 0.0);
  }
  out[r] = s;
  // n_pad is a multiple of 256, so whole waves get here
  const int64_t left = n - r / 64 * 64;
  if (runs && left > 0)
    swe_run_sphere(s.p, static_cast<int>(min(left, int64_t(64))), runs + r / 64);
}

// Bounding sphere of each packing tile: centre = first source, radius^2 =
// max |y - c|^2 (for PSE culling); w holds radius^2.
__global__ __launch_bounds__(kSweTile) void swe_tile_bounds_kernel(
    const SweSrc* __restrict__ src, const int32_t* __restrict__ count,
    double4* __restrict__ bounds) {
  __shared__ double red[kSweTile / 64];
  const int n = *count;
  const int j0 = blockIdx.x * kSweTile;
  if (j0 >= n) return;
  const double4 c = src[j0].p;
  const int j = j0 + threadIdx.x;
  double r2 = 0.0;
  if (j < n) {
    const double4 y = src[j].p;
    const double a = y.x - c.x, b = y.y - c.y, e = y.z - c.z;
    r2 = a * a + b * b + e * e;
  }
  for (int off = 32; off > 0; off >>= 1) r2 = fmax(r2, __shfl_down(r2, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = r2;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = 0.0;
    for (int w = 0; w < kSweTile / 64; ++w) m = fmax(m, red[w]);
    bounds[blockIdx.x] = make_double4(c.x, c.y, c.z, m);
  }
}

template <int NR>
__device__ __forceinline__ double rcp_nr(double d) {
  double r = __builtin_amdgcn_rcp(d);
#pragma unroll
  for (int it = 0; it < NR; ++it) {
    const double e = __builtin_fma(-d, r, 1.0);
    r = __builtin_fma(r, e, r);
  }
  return r;
}

// x.y > 0 evaluated with the reference's rounding, ((x0 y0 + x1 y1) + x2 y2)
// without contraction, so that points on the cut (x.y = 0 in exact
// arithmetic, common on the cubed sphere) are classified identically.
// __dmul_rn / __dadd_rn are plain * and + in this toolchain and would still
// be fused into FMAs; the pragma keeps three multiplies and two adds.
__device__ __forceinline__ bool hemisphere(const double* x, const double4& y) {
#pragma clang fp contract(off)
  const double t = (x[0] * y.x + x[1] * y.y) + x[2] * y.z;
  return t > 0.0;
}

// exp(-z) for 0 <= z: exp(-z) = 2^-n exp(n ln 2 - z) with n the integer
// nearest z / ln 2, the second factor by the polynomial that interpolates exp
// at the 12 Chebyshev nodes of [-ln 2 / 2, ln 2 / 2] (1.6e-17 relative as
// rounded to these coefficients).  17 operations without a branch; the library
// function handles every argument, twice as many with the constants' moves.
__device__ __forceinline__ double exp_neg(double z) {
  const double n = __builtin_rint(z * 0x1.71547652b82fep+0);
  const double r = __builtin_fma(
      n, 0x1.abc9e3b39803fp-56, __builtin_fma(n, 0x1.62e42fefa39efp-1, -z));
  double p = 0x1.af632a0f7e2cep-26;
  p = __builtin_fma(p, r, 0x1.28b4101c77212p-22);
  p = __builtin_fma(p, r, 0x1.71ddf56d8deb5p-19);
  p = __builtin_fma(p, r, 0x1.a01991a10d9aep-16);
  p = __builtin_fma(p, r, 0x1.a01a01b1461c5p-13);
  p = __builtin_fma(p, r, 0x1.6c16c1880029fp-10);
  p = __builtin_fma(p, r, 0x1.111111110f21ep-7);
  p = __builtin_fma(p, r, 0x1.555555554f0bap-5);
  p = __builtin_fma(p, r, 0x1.555555555555ap-3);
  p = __builtin_fma(p, r, 0x1.0000000000011p-1);
  p = __builtin_fma(p, r, 1.0);
  p = __builtin_fma(p, r, 1.0);
  return __builtin_amdgcn_ldexp(p, -static_cast<int>(n));
}

// PSE term of one source (y, area A, surface s_y) at squared distance rho2 of
// target x with surface s_i, added to L: only pairs within the Gaussian's
// cut-off radius (rho^2 < pse_cut2); the others are below exp(-kPseCut)
// relative.  Every lane computes the exponential: where one target is near
// most are, and a divergent branch costs more than the rest of them.  HEMI:
// also x.y > 0.
template <bool HEMI>
__device__ __forceinline__ void swe_pse_pair(double& L, const double4& y,
                                             double A, double s_y,
                                             const double* x, double s_i,
                                             double rho2, double inv_pse_e2,
                                             double pse_cut2) {
  const bool in = rho2 < pse_cut2;
  double eta = exp_neg(in ? rho2 * inv_pse_e2 : 0.0) * A;
  double ds = s_y - s_i;
  if (HEMI && !hemisphere(x, y)) eta = 0.0;
  if (!in) eta = ds = 0.0;
  L = fma(eta, ds, L);
}

__device__ __forceinline__ double swe_rho2(const double* x, const double4& y) {
  const double d0 = y.x - x[0], d1 = y.y - x[1], d2 = y.z - x[2];
  return d0 * d0 + d1 * d1 + d2 * d2;
}

// Whether the cut-off implies x.y > 0 for every target of the wave: x.y >= |x|
// (|x| - rho), so where rho^2 < cut^2 < |x|^2.  On the unit sphere, a cut-off
// radius below 1.
__device__ __forceinline__ bool swe_pse_inside(const double* x,
                                               double pse_cut2) {
  return !__ballot(!(x[0] * x[0] + x[1] * x[1] + x[2] * x[2] >
                     1.000001 * pse_cut2));
}

// PSE terms of one tile (cnt sources, any record up to a multiple of 4).
__device__ __forceinline__ void swe_pse_tile(const SweSrc* tile, int cnt,
                                             const double* x, double s_i,
                                             double inv_pse_e2,
                                             double pse_cut2, double& L) {
  auto sum = [&](auto hemi) {
    for (int j = 0; j < cnt; j += 4)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double4 y = tile[j + k].p;
        const double cut2 = j + k < cnt ? pse_cut2 : -1.0;
        const double rho2 = swe_rho2(x, y);
        if (!__ballot(rho2 < cut2)) continue;
        const double4 q = tile[j + k].q;
        swe_pse_pair<decltype(hemi)::value>(L, y, q.y, q.z, x, s_i, rho2,
                                            inv_pse_e2, cut2);
      }
  };
  if (swe_pse_inside(x, pse_cut2))
    sum(std::false_type{});
  else
    sum(std::true_type{});
}

// p[t] through vector loads (the index is held in a vector register), so
// that a load issued one iteration ahead is waited for in order.
__device__ __forceinline__ double4 vload(const double4* p, int t) {
  int v = t;
  asm volatile("" : "+v"(v));
  return p[v];
}

struct SweSeg {
  const double* x;
  int64_t es, cs, n;
  const int32_t* index;
  const int32_t* d_n;
  const int32_t* self_rank;
  int self_identity;
  int nblocks;
  const double* surf;  // target surface (PSE)
  double* out_u;
  int64_t oes, ocs;
  double* out_ddot;
  double* out_laps;
  int64_t slot_base;  // slot c is target index[c] or slot_base + c
  int32_t rank_base;  // self = self_rank[i] - rank_base
  double* part;     // chunk sums, row r of chunk k of slot c: wave-split
  int64_t pstride;  // part[(20 k + r) * pstride + c], far sums (18 k + r)
};

// Target of slot c and its own source (-1: none) as in the BVE kernels.
__device__ __forceinline__ int64_t swe_target(const SweSeg& sg, int64_t c,
                                              bool in) {
  return in ? (sg.index ? sg.index[c] : sg.slot_base + c) : sg.slot_base;
}
__device__ __forceinline__ int swe_self(const SweSeg& sg, int64_t c,
                                        int64_t i, bool in, int skip_self) {
  if (!in || !skip_self) return -1;
  if (sg.self_rank) {
    const int r = sg.self_rank[i];
    return r < 0 ? -1 : r - sg.rank_base;
  }
  return sg.self_identity ? static_cast<int>(c) : -1;
}

// FP64 accumulators of one target (see the file comment); Gd and Gs hold
// the symmetric matrices as xx, xy, xz, yy, yz, zz.
struct SweAcc {
  double Vy[3], Gd[6], Vg[3], Bt, Gs[6];
  double L1;  // PSE sum
  __device__ void zero() {
    Bt = L1 = 0.0;
    for (int k = 0; k < 3; ++k) Vy[k] = Vg[k] = 0.0;
    for (int k = 0; k < 6; ++k) Gd[k] = Gs[k] = 0.0;
  }
};

// FP32 partials of one source tile: Vy is carried as A0 = sum alpha and
// Vd = sum alpha d with d = y - x (Vy = x A0 + Vd), which keeps the
// tile-relative precision of d.
struct SweAcc32 {
  float A0, Vd[3], Gd[6], Vg[3], Bt, Gs[6];
  __device__ void zero() {
    A0 = Bt = 0.0f;
    for (int k = 0; k < 3; ++k) Vd[k] = Vg[k] = 0.0f;
    for (int k = 0; k < 6; ++k) Gd[k] = Gs[k] = 0.0f;
  }
};

// Gd += ap g g^T, Vg += be g, Bt += be t, Gs += bp g g^T.
template <typename T, typename Acc>
__device__ __forceinline__ void swe_pair_g(Acc& acc, const T g0, const T g1,
                                           const T g2, const T t, const T be,
                                           const T ap, const T bp) {
  const T e0 = ap * g0, e1 = ap * g1, e2 = ap * g2;
  acc.Gd[0] = fma(e0, g0, acc.Gd[0]);
  acc.Gd[1] = fma(e0, g1, acc.Gd[1]);
  acc.Gd[2] = fma(e0, g2, acc.Gd[2]);
  acc.Gd[3] = fma(e1, g1, acc.Gd[3]);
  acc.Gd[4] = fma(e1, g2, acc.Gd[4]);
  acc.Gd[5] = fma(e2, g2, acc.Gd[5]);
  acc.Vg[0] = fma(be, g0, acc.Vg[0]);
  acc.Vg[1] = fma(be, g1, acc.Vg[1]);
  acc.Vg[2] = fma(be, g2, acc.Vg[2]);
  acc.Bt = fma(be, t, acc.Bt);
  const T f0 = bp * g0, f1 = bp * g1, f2 = bp * g2;
  acc.Gs[0] = fma(f0, g0, acc.Gs[0]);
  acc.Gs[1] = fma(f0, g1, acc.Gs[1]);
  acc.Gs[2] = fma(f0, g2, acc.Gs[2]);
  acc.Gs[3] = fma(f1, g1, acc.Gs[3]);
  acc.Gs[4] = fma(f1, g2, acc.Gs[4]);
  acc.Gs[5] = fma(f2, g2, acc.Gs[5]);
}

// FP64 pair: source y, t = x.y, r = 1 / D.
__device__ __forceinline__ void swe_pair_f64(SweAcc& acc, const double4& y,
                                             const double t, const double r,
                                             const double b, const double* x) {
  const double al = y.w * r, be = b * r;
  const double ap = al * r, bp = be * r;
  acc.Vy[0] = fma(al, y.x, acc.Vy[0]);
  acc.Vy[1] = fma(al, y.y, acc.Vy[1]);
  acc.Vy[2] = fma(al, y.z, acc.Vy[2]);
  const double g0 = fma(-t, x[0], y.x), g1 = fma(-t, x[1], y.y),
               g2 = fma(-t, x[2], y.z);
  swe_pair_g<double>(acc, g0, g1, g2, t, be, ap, bp);
}

// FP32 pair on tile-relative offsets: d = y - x, rho2 = |d|^2 (= 2 delta on
// the unit sphere), r = 1 / D; xh = x / 2, so g = d + delta x = d + rho2 xh
// and t = 1 - delta.
__device__ __forceinline__ void swe_pair_f32(SweAcc32& acc, const float d0,
                                             const float d1, const float d2,
                                             const float rho2, const float r,
                                             const float a, const float b,
                                             const float* xh) {
  const float al = a * r, be = b * r;
  const float ap = al * r, bp = be * r;
  acc.A0 += al;
  acc.Vd[0] = fmaf(al, d0, acc.Vd[0]);
  acc.Vd[1] = fmaf(al, d1, acc.Vd[1]);
  acc.Vd[2] = fmaf(al, d2, acc.Vd[2]);
  const float g0 = fmaf(rho2, xh[0], d0), g1 = fmaf(rho2, xh[1], d1),
              g2 = fmaf(rho2, xh[2], d2);
  const float t = fmaf(-0.5f, rho2, 1.0f);
  swe_pair_g<float>(acc, g0, g1, g2, t, be, ap, bp);
}

// Adds one tile's FP32 partials to the FP64 accumulators of target x.
__device__ __forceinline__ void swe_carry(SweAcc& acc, const SweAcc32& p,
                                          const double* x) {
  for (int k = 0; k < 3; ++k) {
    acc.Vy[k] += fma(x[k], static_cast<double>(p.A0),
                     static_cast<double>(p.Vd[k]));
    acc.Vg[k] += p.Vg[k];
  }
  acc.Bt += p.Bt;
  for (int k = 0; k < 6; ++k) {
    acc.Gd[k] += p.Gd[k];
    acc.Gs[k] += p.Gs[k];
  }
}

__device__ __forceinline__ void sym(const double* Y, double (*m)[3]) {
  m[0][0] = Y[0];
  m[0][1] = m[1][0] = Y[1];
  m[0][2] = m[2][0] = Y[2];
  m[1][1] = Y[3];
  m[1][2] = m[2][1] = Y[4];
  m[2][2] = Y[5];
}

// u, ddot and the Laplacian from the accumulators of target x.
__device__ __forceinline__ void swe_finalize(const SweAcc& A, const double* x,
                                             double pse_scale, double* u,
                                             double* ddot, double* laps) {
  const double* V = A.Vy;
  const double xv[3] = {x[1] * V[2] - x[2] * V[1], x[2] * V[0] - x[0] * V[2],
                        x[0] * V[1] - x[1] * V[0]};
  u[0] = -xv[0] - A.Vg[0];
  u[1] = -xv[1] - A.Vg[1];
  u[2] = -xv[2] - A.Vg[2];

  double Gd[3][3], Gs[3][3];
  sym(A.Gd, Gd);
  sym(A.Gs, Gs);
  // [x]x Gd: row a = (x cross column)_a
  double M[3][3];
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    M[0][b] = x[1] * Gd[2][b] - x[2] * Gd[1][b];
    M[1][b] = x[2] * Gd[0][b] - x[0] * Gd[2][b];
    M[2][b] = x[0] * Gd[1][b] - x[1] * Gd[0][b];
  }
  // E(Vy): [[0, v2, -v1], [-v2, 0, v0], [v1, -v0, 0]]
  M[0][1] += V[2];
  M[0][2] -= V[1];
  M[1][0] -= V[2];
  M[1][2] += V[0];
  M[2][0] += V[1];
  M[2][1] -= V[0];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      const double P = (a == b ? 1.0 : 0.0) - x[a] * x[b];
      M[a][b] += A.Bt * P + x[a] * A.Vg[b] - Gs[a][b] - xv[a] * x[b];
    }
  double dd = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) dd += M[a][b] * M[b][a];
  *ddot = dd;
  *laps = pse_scale * A.L1;
}

// FP64 pair terms of one LDS tile (cnt sources, zero padding up to a
// multiple of SHARE) for target x; `self` is the target's own source in tile
// numbering (outside [0, cnt): none) and any_self says whether some lane of
// the wave has one here.  Without, SHARE sources share one reciprocal,
// e.g. 1/D_a = D_b (D_c D_d) / (D_a D_b D_c D_d).
__device__ __forceinline__ double swe_t(const double* x, const double4& y) {
  return fma(x[2], y.z, fma(x[1], y.y, x[0] * y.x));
}

template <int SHARE = 4>
__device__ __forceinline__ void swe_tile_f64(SweAcc& acc, const SweSrc* tile,
                                             int cnt, const double* x,
                                             double eps2, int self,
                                             bool any_self) {
  static_assert(SHARE == 2 || SHARE == 4, "two or four pairs per reciprocal");
  if (any_self) {
    for (int jj = 0; jj < cnt; ++jj) {
      const double4 yp = tile[jj].p;
      const double t = swe_t(x, yp);
      double r = rcp_nr<1>((1.0 - t) + eps2);
      if (jj == self) r = 0.0;
      swe_pair_f64(acc, yp, t, r, tile[jj].q.x, x);
    }
  } else if (SHARE == 2) {
    for (int jj = 0; jj < cnt; jj += 2) {
      const double4 ya = tile[jj].p, yb = tile[jj + 1].p;
      const double ta = swe_t(x, ya), tb = swe_t(x, yb);
      const double Da = (1.0 - ta) + eps2, Db = (1.0 - tb) + eps2;
      const double r = rcp_nr<1>(Da * Db);
      swe_pair_f64(acc, ya, ta, Db * r, tile[jj].q.x, x);
      swe_pair_f64(acc, yb, tb, Da * r, tile[jj + 1].q.x, x);
    }
  } else {
    for (int jj = 0; jj < cnt; jj += 4) {
      const double4 ya = tile[jj].p, yb = tile[jj + 1].p;
      const double4 yc = tile[jj + 2].p, yd = tile[jj + 3].p;
      const double ta = swe_t(x, ya), tb = swe_t(x, yb);
      const double tc = swe_t(x, yc), td = swe_t(x, yd);
      const double Da = (1.0 - ta) + eps2, Db = (1.0 - tb) + eps2;
      const double Dc = (1.0 - tc) + eps2, Dd = (1.0 - td) + eps2;
      const double pab = Da * Db, pcd = Dc * Dd;
      const double r = rcp_nr<1>(pab * pcd);
      const double rab = pcd * r, rcd = pab * r;
      swe_pair_f64(acc, ya, ta, Db * rab, tile[jj].q.x, x);
      swe_pair_f64(acc, yb, tb, Da * rab, tile[jj + 1].q.x, x);
      swe_pair_f64(acc, yc, tc, Dd * rcd, tile[jj + 2].q.x, x);
      swe_pair_f64(acc, yd, td, Dc * rcd, tile[jj + 3].q.x, x);
    }
  }
}

constexpr double kSweMfNear = 3.0;
constexpr int kSweMfSub = 64;                     // sources per sub-tile
constexpr int kSweMfNsub = kSweTile / kSweMfSub;  // sub-tiles per tile

// Whether target x lies within kSweMfNear radii of the centroid of a tile
// or sub-tile (c.w = radius^2): the near / far split of the matrix-core
// kernels.  Contraction is off so that every kernel rounds it alike: both
// passes classify every tile and sub-tile, and must agree.
__device__ __forceinline__ bool swe_mf_near(const double* x, const double4& c) {
#pragma clang fp contract(off)
  const double e0 = x[0] - c.x, e1 = x[1] - c.y, e2 = x[2] - c.z;
  return (e0 * e0 + e1 * e1) + e2 * e2 <= (kSweMfNear * kSweMfNear) * c.w;
}
constexpr int kSweMfR1 = 6;   // set-1 feature rows
constexpr int kSweMfR2 = 12;  // set-2 feature rows
constexpr int kSweMfKb = kSweTile / 32;
constexpr int kSweMfFr = kSweMfKb * 2 * 4 * kSweMfR1;   // uint4 per tile
constexpr int kSweMfFr2 = kSweMfKb * 2 * 4 * kSweMfR2;  // uint4 per tile
// Offsets of a tile's fields in its record (uint4), and the record's length.
constexpr int kSweMfYas = kSweTile;
constexpr int kSweMfFrAt = 2 * kSweTile;
constexpr int kSweMfFr2At = kSweMfFrAt + kSweMfFr;
constexpr int kSweMfFsAt = kSweMfFr2At + kSweMfFr2;
constexpr int kSweMfRec = kSweMfFsAt + 16;
constexpr int64_t kSweMfTileBytes = 32 + 32 * kSweMfNsub + 16 * kSweMfRec;

// Matrix-core records of consecutive tiles (see the matrix-core section).
struct SweMfTiles {
  double4* cen;   // per tile: centroid, radius^2
  double4* scen;  // per sub-tile: centroid, radius^2 (-1: no sources)
  uint4* rec;     // kSweMfRec per tile
  // the records of tiles t0 and later
  __host__ __device__ SweMfTiles from(int64_t t0) const {
    return SweMfTiles{cen + t0, scen + kSweMfNsub * t0, rec + kSweMfRec * t0};
  }
};

// ----------------------------------------------------------- FP64 kernel --
// One target per lane; sources staged through LDS.  PSE terms are evaluated
// only for tiles near some target of the wave.
// Parameters shared by every target of a launch.
struct SweParams {
  double eps2, inv_pse_e2, pse_cut2;
  int do_pse, skip_self;
  SweMfTiles mf{};  // matrix-core variants: the tile records
  int C = 1;        // the source chunks of their far pass
  int rows = 1;     // and the chunk sums stored per target: C, or 1
};

// Block `blk` of segment `sg` against nsrc packed sources (bounds: their
// tile bounding spheres).  Every thread of the block calls it.
template <int BLOCK, int SHARE>
__device__ __forceinline__ void swe_f64_block(
    const SweSrc* __restrict__ src, const double4* __restrict__ bounds,
    int nsrc, const SweSeg& sg, int blk, const SweParams& P, SweSrc* tile) {
  const double eps2 = P.eps2, inv_pse_e2 = P.inv_pse_e2;
  const double pse_cut2 = P.pse_cut2;
  const int do_pse = P.do_pse;
  const int64_t n_live = sg.d_n ? *sg.d_n : sg.n;
  const int64_t c = static_cast<int64_t>(blk) * BLOCK + threadIdx.x;
  if (static_cast<int64_t>(blk) * BLOCK >= n_live) return;
  const bool in = c < n_live;
  const int64_t i = swe_target(sg, c, in);
  const double* px = sg.x + i * sg.es;
  const double x[3] = {px[0], px[sg.cs], px[2 * sg.cs]};
  const double s_i = (do_pse && sg.surf) ? sg.surf[i] : 0.0;
  const int self = swe_self(sg, c, i, in, P.skip_self);

  SweAcc acc;
  acc.zero();
  for (int j0 = 0; j0 < nsrc; j0 += kSweTile) {
    __syncthreads();
    for (int t = threadIdx.x; t < kSweTile; t += BLOCK) {
      const int j = j0 + t;
      if (j < nsrc) {
        tile[t] = src[j];
      } else {
        tile[t].p = make_double4(0.0, 0.0, 0.0, 0.0);
        tile[t].q = make_double4(0.0, 0.0, 0.0, 0.0);
      }
    }
    __syncthreads();
    const int cnt = min(kSweTile, nsrc - j0);
    const bool diag = static_cast<unsigned>(self - j0) <
                      static_cast<unsigned>(cnt);
    swe_tile_f64<SHARE>(acc, tile, cnt, x, eps2, self - j0,
                        __ballot(diag) != 0);
    if (do_pse) {
      // wave-uniform test: is any target of the wave near this tile?
      const double4 bd = bounds[j0 / kSweTile];
      const double e0 = x[0] - bd.x, e1 = x[1] - bd.y, e2 = x[2] - bd.z;
      const double dist2 = e0 * e0 + e1 * e1 + e2 * e2;
      const double rr = sqrt(bd.w) + sqrt(pse_cut2);
      const bool near = in && dist2 <= rr * rr;
      if (__ballot(near)) {
        swe_pse_tile(tile, cnt, x, s_i, inv_pse_e2, pse_cut2, acc.L1);
      }
    }
  }
  if (!in) return;
  double u[3], dd, lap;
  swe_finalize(acc, x, k4OverPi * inv_pse_e2 * inv_pse_e2, u, &dd, &lap);
  if (sg.out_u) {
    double* o = sg.out_u + i * sg.oes;
    o[0] = u[0];
    o[sg.ocs] = u[1];
    o[2 * sg.ocs] = u[2];
  }
  if (sg.out_ddot) sg.out_ddot[i] = dd;
  if (sg.out_laps && do_pse) sg.out_laps[i] = lap;
}

// SHARE: pairs per FP64 reciprocal; MINW: minimum waves per SIMD asked of
// the register allocator.
template <int BLOCK, int SHARE, int MINW>
__global__ __launch_bounds__(BLOCK, MINW) void swe_f64_kernel(
    const SweSrc* __restrict__ src, const double4* __restrict__ bounds,
    const int32_t* __restrict__ count, SweSeg s0, SweSeg s1, SweParams P) {
  __shared__ SweSrc tile[kSweTile];
  const bool first = static_cast<int>(blockIdx.x) < s0.nblocks;
  const SweSeg& sg = first ? s0 : s1;
  const int blk = first ? blockIdx.x : blockIdx.x - s0.nblocks;
  swe_f64_block<BLOCK, SHARE>(src, bounds, *count, sg, blk, P, tile);
}

// ------------------------------------------------------- FP64 wave split --
// A block of eight waves owns 64 targets, one per lane, and one of C chunks of
// the sources; wave w sums the w-th eighth of the chunk and the eight sums are
// added in a fixed tree through LDS.  Sources are read at wave-uniform
// addresses, so each 64-byte record arrives through the scalar cache in SGPRs
// and enters the FMAs as their scalar operand (no LDS staging, no barriers in
// the loop); four pairs share one reciprocal.  The 64-target block with all
// sources of its target in one wave that this replaces left 38 blocks for
// 7,682 targets (1,183 us for 5,120 sources).
// What bounds it: FP64 issue, about 40 operations per pair, and the
// exponentials of the PSE terms.  The sums depend on C and the source count
// alone, not on whether a block takes one chunk or all of them.
constexpr int kSweWaves = 8;
constexpr int kSweRows = 20;  // values of SweAcc

// Visits the values of an accumulator in a fixed order.
template <typename F>
__device__ __forceinline__ void swe_rows(SweAcc& a, F&& f) {
  int r = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) f(r++, a.Vy[k]);
#pragma unroll
  for (int k = 0; k < 6; ++k) f(r++, a.Gd[k]);
#pragma unroll
  for (int k = 0; k < 3; ++k) f(r++, a.Vg[k]);
  f(r++, a.Bt);
#pragma unroll
  for (int k = 0; k < 6; ++k) f(r++, a.Gs[k]);
  f(r++, a.L1);
}

// Sources [j0, j1) (multiples of four; zero records pad the last) of the
// packed records at src against target x.  CHECK drops source `self`.
template <bool CHECK>
__device__ __forceinline__ void swe_wave_pairs(SweAcc& acc,
                                               const double* __restrict__ src,
                                               int j0, int j1, const double* x,
                                               double eps2, int self) {
#pragma unroll 1
  for (int j = j0; j < j1; j += 4) {
    const double* p = src + static_cast<int64_t>(j) * 8;
    double y[4][5];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int e = 0; e < 5; ++e) y[k][e] = p[8 * k + e];
    double t[4], D[4], r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      t[k] = fma(x[2], y[k][2], fma(x[1], y[k][1], x[0] * y[k][0]));
      D[k] = (1.0 - t[k]) + eps2;
      if (CHECK && j + k == self) D[k] = 1.0;
    }
    const double pab = D[0] * D[1], pcd = D[2] * D[3];
    const double q = rcp_nr<1>(pab * pcd);
    const double rab = pcd * q, rcd = pab * q;
    r[0] = D[1] * rab;
    r[1] = D[0] * rab;
    r[2] = D[3] * rcd;
    r[3] = D[2] * rcd;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (CHECK && j + k == self) r[k] = 0.0;
      swe_pair_f64(acc, make_double4(y[k][0], y[k][1], y[k][2], y[k][3]), t[k],
                   r[k], y[k][4], x);
    }
  }
}

// PSE terms of sources [j0, j1) of n, j0 and j1 multiples of four.
__device__ __forceinline__ double swe_wave_pse(const double* __restrict__ src,
                                               int j0, int j1, int n,
                                               const double* x, double s_i,
                                               double inv_pse_e2,
                                               double pse_cut2) {
  double L = 0.0;
  auto sum = [&](auto hemi) {
#pragma unroll 1
    for (int j = j0; j < j1; j += 4) {
      const double* p = src + static_cast<int64_t>(j) * 8;
      double4 y[4];
      double rho2[4], cut2[4];
      bool any = false;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        y[k] = make_double4(p[8 * k], p[8 * k + 1], p[8 * k + 2], 0.0);
        rho2[k] = swe_rho2(x, y[k]);
        cut2[k] = j + k < n ? pse_cut2 : -1.0;
        any |= rho2[k] < cut2[k];
      }
      if (!__ballot(any)) continue;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        swe_pse_pair<decltype(hemi)::value>(L, y[k], p[8 * k + 5], p[8 * k + 6],
                                            x, s_i, rho2[k], inv_pse_e2, cut2[k]);
    }
  };
  if (swe_pse_inside(x, pse_cut2))
    sum(std::false_type{});
  else
    sum(std::true_type{});
  return L;
}

// Outputs of target i at x from its sums.
__device__ __forceinline__ void swe_store(const SweSeg& sg, int64_t i,
                                          const SweAcc& acc, const double* x,
                                          const SweParams& P) {
  double u[3], dd, lap;
  swe_finalize(acc, x, k4OverPi * P.inv_pse_e2 * P.inv_pse_e2, u, &dd, &lap);
  if (sg.out_u) {
    double* o = sg.out_u + i * sg.oes;
    o[0] = u[0];
    o[sg.ocs] = u[1];
    o[2 * sg.ocs] = u[2];
  }
  if (sg.out_ddot) sg.out_ddot[i] = dd;
  if (sg.out_laps && P.do_pse) sg.out_laps[i] = lap;
}

// Targets of block `blk` of segment sg against chunk `chunk` of C (SPLIT: the
// sums go to sg.part[(20 chunk + row) pstride + slot]) or against every chunk
// in order (the outputs are written).  sub: bounding sphere (centroid,
// radius^2) per 64 sources.  Every thread of the 512 calls it.
template <bool SPLIT>
__device__ __forceinline__ void swe_wave_block(
    const double* __restrict__ src, const double4* __restrict__ sub, int nsrc,
    const SweSeg& sg, int blk, int chunk, int C, const SweParams& P,
    double (*red)[kSweRows][64]) {
  const int64_t n_live = sg.d_n ? *sg.d_n : sg.n;
  const int64_t c0 = static_cast<int64_t>(blk) * 64;
  if (c0 >= n_live) return;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t c = c0 + lane;
  const bool in = c < n_live;
  const int64_t i = swe_target(sg, c, in);
  const double* px = sg.x + i * sg.es;
  const double x[3] = {px[0], px[sg.cs], px[2 * sg.cs]};
  const double s_i = (P.do_pse && sg.surf) ? sg.surf[i] : 0.0;
  const int self = swe_self(sg, c, i, in, P.skip_self);
  // range of the wave's own sources, the same in every lane
  int lo = self >= 0 ? self : 0x7fffffff, hi = self;
  for (int off = 32; off > 0; off >>= 1) {
    lo = min(lo, __shfl_xor(lo, off, 64));
    hi = max(hi, __shfl_xor(hi, off, 64));
  }
  lo = __builtin_amdgcn_readfirstlane(lo);
  hi = __builtin_amdgcn_readfirstlane(hi);
  const double rcut = sqrt(P.pse_cut2);
  const int nq = (nsrc + 3) / 4;
  SweAcc tot;
  if constexpr (!SPLIT) tot.zero();
#pragma unroll 1
  for (int k = SPLIT ? chunk : 0; k < (SPLIT ? chunk + 1 : C); ++k) {
    const int64_t seg = static_cast<int64_t>(kSweWaves) * k + w;
    const int64_t nseg = static_cast<int64_t>(kSweWaves) * C;
    const int a = 4 * static_cast<int>(nq * seg / nseg);
    const int b = 4 * static_cast<int>(nq * (seg + 1) / nseg);
    SweAcc acc;
    acc.zero();
#pragma unroll 1
    for (int j = a; j < b;) {
      const int e = min((j / 64 + 1) * 64, b);
      if (lo < e && hi >= j)
        swe_wave_pairs<true>(acc, src, j, e, x, P.eps2, self);
      else
        swe_wave_pairs<false>(acc, src, j, e, x, P.eps2, -1);
      if (P.do_pse) {
        // wave-uniform test: is any target of the wave near these sources?
        const double4 bd = sub[j / 64];
        const double p0 = x[0] - bd.x, p1 = x[1] - bd.y, p2 = x[2] - bd.z;
        const double rr = sqrt(bd.w) + rcut;
        if (__ballot(in && p0 * p0 + p1 * p1 + p2 * p2 <= rr * rr))
          acc.L1 += swe_wave_pse(src, j, e, nsrc, x, s_i, P.inv_pse_e2,
                                 P.pse_cut2);
      }
      j = e;
    }
    // sums of the eight waves: (w, w + 4), then (w, w + 2), then (0, 1)
#pragma unroll 1
    for (int half = kSweWaves / 2; half > 0; half >>= 1) {
      __syncthreads();  // the previous values are read
      if (w >= half && w < 2 * half)
        swe_rows(acc, [&](int r, double& v) { red[w - half][r][lane] = v; });
      __syncthreads();
      if (w < half)
        swe_rows(acc, [&](int r, double& v) { v += red[w][r][lane]; });
    }
    if (w == 0) {
      if constexpr (SPLIT) {
        if (in)
          swe_rows(acc, [&](int r, double& v) {
            sg.part[(kSweRows * static_cast<int64_t>(k) + r) * sg.pstride + c] = v;
          });
      } else {
        double v[kSweRows];
        swe_rows(acc, [&](int r, double& q) { v[r] = q; });
        swe_rows(tot, [&](int r, double& q) { q += v[r]; });
      }
    }
  }
  if constexpr (!SPLIT)
    if (w == 0 && in) swe_store(sg, i, tot, x, P);
}

// Sums of slot c of sg from its C chunks, added in chunk order, and outputs.
__device__ __forceinline__ void swe_wave_reduce(const SweSeg& sg, int64_t c,
                                                int C, const SweParams& P) {
  const int64_t n_live = sg.d_n ? *sg.d_n : sg.n;
  if (c >= n_live) return;
  const int64_t i = swe_target(sg, c, true);
  SweAcc acc;
  acc.zero();
  const double* q = sg.part + c;
#pragma unroll 4
  for (int k = 0; k < C; ++k)
    swe_rows(acc, [&](int r, double& v) {
      v += q[(kSweRows * static_cast<int64_t>(k) + r) * sg.pstride];
    });
  const double* px = sg.x + i * sg.es;
  const double x[3] = {px[0], px[sg.cs], px[2 * sg.cs]};
  swe_store(sg, i, acc, x, P);
}

template <bool SPLIT>
__global__ __launch_bounds__(64 * kSweWaves, 4) void swe_wave_kernel(
    const double* __restrict__ src, const double4* __restrict__ sub,
    const int32_t* __restrict__ count, SweSeg s0, SweSeg s1, SweParams P,
    int C) {
  __shared__ double red[kSweWaves / 2][kSweRows][64];
  const int b = SPLIT ? flat_block() / C : flat_block();
  const int k = SPLIT ? flat_block() % C : 0;
  const bool first = b < s0.nblocks;
  const SweSeg& sg = first ? s0 : s1;
  const int blk = first ? b : b - s0.nblocks;
  swe_wave_block<SPLIT>(src, sub, *count, sg, blk, k, C, P, red);
}

__global__ __launch_bounds__(64) void swe_wave_reduce_kernel(SweSeg s0,
                                                             SweSeg s1,
                                                             SweParams P,
                                                             int C) {
  const int64_t g = static_cast<int64_t>(blockIdx.x) * 64 + threadIdx.x;
  const bool first = g < s0.n;
  const SweSeg& sg = first ? s0 : s1;
  swe_wave_reduce(sg, first ? g : g - s0.n, C, P);
}

// ---------------------------------------------------------- mixed kernel --
// FP32 pair arithmetic on tile-relative coordinates (d formed from offsets
// to the tile's FP64 centre, delta = |d|^2 / 2); FP32 partial sums per
// source tile are carried into FP64 accumulators.
struct F4x2 {
  float4 p;  // y - c (3), a
  float4 q;  // b, A, 0, 0
};

// As swe_f64_block with FP32 pair arithmetic; tile64 is the FP64 copy of
// the LDS tile for the PSE terms.
template <int BLOCK>
__device__ __forceinline__ void swe_mixed_block(
    const SweSrc* __restrict__ src, const double4* __restrict__ bounds,
    int nsrc, const SweSeg& sg, int blk, const SweParams& P, F4x2* tile,
    SweSrc* tile64) {
  const double eps2 = P.eps2, inv_pse_e2 = P.inv_pse_e2;
  const double pse_cut2 = P.pse_cut2;
  const int do_pse = P.do_pse;
  const int64_t n_live = sg.d_n ? *sg.d_n : sg.n;
  const int64_t c = static_cast<int64_t>(blk) * BLOCK + threadIdx.x;
  if (static_cast<int64_t>(blk) * BLOCK >= n_live) return;
  const bool in = c < n_live;
  const int64_t i = swe_target(sg, c, in);
  const double* px = sg.x + i * sg.es;
  const double x[3] = {px[0], px[sg.cs], px[2 * sg.cs]};
  const double s_i = (do_pse && sg.surf) ? sg.surf[i] : 0.0;
  const int self = swe_self(sg, c, i, in, P.skip_self);
  const float e2f = static_cast<float>(eps2);

  SweAcc acc;
  acc.zero();
  for (int j0 = 0; j0 < nsrc; j0 += kSweTile) {
    const double4 bd = bounds[j0 / kSweTile];
    __syncthreads();
    for (int t = threadIdx.x; t < kSweTile; t += BLOCK) {
      const int j = j0 + t;
      F4x2 z;
      if (j < nsrc) {
        const SweSrc sj = src[j];
        z.p = make_float4(static_cast<float>(sj.p.x - bd.x),
                          static_cast<float>(sj.p.y - bd.y),
                          static_cast<float>(sj.p.z - bd.z),
                          static_cast<float>(sj.p.w));
        z.q = make_float4(static_cast<float>(sj.q.x),
                          static_cast<float>(sj.q.y), 0.0f, 0.0f);
        tile64[t] = sj;
      } else {
        z.p = make_float4(8.0f, 8.0f, 8.0f, 0.0f);
        z.q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        tile64[t].p = make_double4(0.0, 0.0, 0.0, 0.0);
        tile64[t].q = make_double4(0.0, 0.0, 0.0, 0.0);
      }
      tile[t] = z;
    }
    __syncthreads();
    const float xr[3] = {static_cast<float>(x[0] - bd.x),
                         static_cast<float>(x[1] - bd.y),
                         static_cast<float>(x[2] - bd.z)};
    const int cnt = min(kSweTile, nsrc - j0);
    const bool diag = static_cast<unsigned>(self - j0) <
                      static_cast<unsigned>(cnt);
    const double g0 = x[0] - bd.x, g1 = x[1] - bd.y, g2 = x[2] - bd.z;
    // tiles within kSweNearFp64 bounding radii of some target of the wave
    // hold the largest pair terms of grad u, whose assembly cancels: those
    // run in FP64 straight into the FP64 accumulators
    if (__ballot(in && g0 * g0 + g1 * g1 + g2 * g2 <=
                           kSweNearFp64 * kSweNearFp64 * bd.w)) {
      swe_tile_f64<2>(acc, tile64, cnt, x, eps2, self - j0,
                      __ballot(diag) != 0);
    } else {
      SweAcc32 p;
      p.zero();
      const float xh[3] = {0.5f * static_cast<float>(x[0]),
                           0.5f * static_cast<float>(x[1]),
                           0.5f * static_cast<float>(x[2])};
      // the per-pair self test only in tiles holding some lane's own source;
      // the padding sources (far away, zero strengths) add nothing, so the
      // loop runs to a multiple of four and unrolls
      const int cnt4 = (cnt + 3) & ~3;
      auto pairs = [&](auto check) {
#pragma unroll 4
        for (int jj = 0; jj < cnt4; ++jj) {
          const float4 yp = tile[jj].p;
          const float4 yq = tile[jj].q;
          const float d0 = yp.x - xr[0], d1 = yp.y - xr[1], d2 = yp.z - xr[2];
          const float rho2 = fmaf(d2, d2, fmaf(d1, d1, d0 * d0));
          float r = __builtin_amdgcn_rcpf(fmaf(0.5f, rho2, e2f));
          if (decltype(check)::value && j0 + jj == self) r = 0.0f;
          swe_pair_f32(p, d0, d1, d2, rho2, r, yp.w, yq.x, xh);
        }
      };
      if (__ballot(diag))
        pairs(std::true_type{});
      else
        pairs(std::false_type{});
      // carry the tile's FP32 partials into the FP64 accumulators
      swe_carry(acc, p, x);
    }
    if (do_pse) {
      const double e0 = x[0] - bd.x, e1 = x[1] - bd.y, e2 = x[2] - bd.z;
      const double dist2 = e0 * e0 + e1 * e1 + e2 * e2;
      const double rr = sqrt(bd.w) + sqrt(pse_cut2);
      const bool near = in && dist2 <= rr * rr;
      if (__ballot(near)) {
        // the PSE sum is a second difference whose first-order terms cancel
        // by symmetry; it covers few tiles, so it runs in FP64
        double L = 0.0;
        swe_pse_tile(tile64, cnt, x, s_i, inv_pse_e2, pse_cut2, L);
        acc.L1 += L;
      }
    }
  }
  if (!in) return;
  double u[3], dd, lap;
  swe_finalize(acc, x, k4OverPi * inv_pse_e2 * inv_pse_e2, u, &dd, &lap);
  if (sg.out_u) {
    double* o = sg.out_u + i * sg.oes;
    o[0] = u[0];
    o[sg.ocs] = u[1];
    o[2 * sg.ocs] = u[2];
  }
  if (sg.out_ddot) sg.out_ddot[i] = dd;
  if (sg.out_laps && do_pse) sg.out_laps[i] = lap;
}

// MINW: minimum waves per SIMD asked of the register allocator (the FP64
// accumulators, the FP32 tile partials and the FP64 near-tile and PSE loops
// hold about 170 registers at 3 waves).
template <int BLOCK, int MINW>
__global__ __launch_bounds__(BLOCK, MINW) void swe_mixed_kernel(
    const SweSrc* __restrict__ src, const double4* __restrict__ bounds,
    const int32_t* __restrict__ count, SweSeg s0, SweSeg s1, SweParams P) {
  __shared__ F4x2 tile[kSweTile];
  __shared__ SweSrc tile64[kSweTile];
  const bool first = static_cast<int>(blockIdx.x) < s0.nblocks;
  const SweSeg& sg = first ? s0 : s1;
  const int blk = first ? blockIdx.x : blockIdx.x - s0.nblocks;
  swe_mixed_block<BLOCK>(src, bounds, *count, sg, blk, P, tile, tile64);
}

// ------------------------------------------------ matrix-core far field --
// Mixed precision on the matrix cores, in two passes.  A tile or 64-source
// sub-tile is far from a wave when no target of the wave lies within
// kSweMfNear radii of its centroid c (swe_mf_near).  The first pass sums
// every far tile, and the far sub-tiles of the other tiles, per 32 sources
// and 16 targets in two stages:
//   stage 1 (v_mfma_f32_16x16x4_f32): sigma D for 16 sources x 16 targets,
//     D = |x' - y'|^2 / 2 + eps^2 = |x'|^2 / 2 - x'.y' + |y'|^2 / 2 + eps^2
//     on FP32 offsets x' = x - c, y' = y - c:  A_j = (y'_j, |y'_j|^2 / 2),
//     B_i = sigma (-x'_i, 1), C_i = sigma (|x'_i|^2 / 2 + eps^2);
//   vector ALUs: w = 1 / (sigma D) and w^2, each split into f16 hi + lo;
//   stage 2 (v_mfma_f32_16x16x32_f16): per target, the sums over 32 sources
//     of w times six source features and of w^2 times twelve, as
//     F_hi w_hi + F_lo w_hi + F_hi w_lo (22 significant bits).
// With a = zeta A / 4pi, b = sigma A / 4pi and absolute coordinates y the
// features are
//   set 1 (weight 1 / D):    a y0, a y1, a y2, b y0, b y1, b y2
//   set 2 (weight 1 / D^2):  a y y^T (xx, xy, xz, yy, yz, zz), b y y^T
// and the far sums follow from them by target-only projections
// (g = Q y, Q = I - x x^T):
//   Vy += set 1 rows 0..2;  Vg += Q (rows 3..5);  Bt += x . (rows 3..5);
//   Gd += Q (set 2 rows 0..5) Q;  Gs += Q (rows 6..11) Q.
// The projections are linear, so each lane carries the FP32 sums into FP64
// per tile or sub-tile and the 18 raw sums of every target and source chunk
// go to a workspace; the second pass sums the near sub-tiles in FP64 (and the PSE
// terms), adds the projected far sums of all chunks and writes the outputs.
// Every feature
// row of a tile is scaled by a power of two to a maximum in [2^13, 2^14), and
// sigma, a power of two per 16 targets, bounds w by 2^7 and w^2 by 2^14 from
// the group's smallest D over the (sub-)tile's bounding sphere, so no f16
// operand overflows.  Offsets are taken from the centroid of the tile or
// sub-tile being summed, so the FP32 distance form cancels by at most
// (kSweMfNear + 1)^2 / (kSweMfNear - 1)^2 against its terms.
//
// Tile records (one 256-source tile each):
//   cen        double4  (c, R^2)
//   scen[4]    double4  sub-tile (c_s, r_s^2), r_s^2 = -1 without sources
// and in one piece:
//   ya[256]    float4   (y - c, |y - c|^2 / 2); padding (8, 8, 8, 96)
//   yas[256]   float4   the same relative to the source's sub-tile centroid
//   fr[384]    uint4    set 1, [k-block 8][hi/lo][g 4][row 6] x 8 f16
//   fr2[768]   uint4    set 2, [k-block 8][hi/lo][g 4][row 12] x 8 f16
//   fs[32]     double   inverse row scales: set 1 at 0..5, set 2 at 16..27
//                       (zero for the unused rows)
// Slot i of K-group g in a 32-source k-block is source 4 g + i (i < 4) or
// 16 + 4 g + i - 4: the rows that lane (g, target) holds after stage 1.

// Records of ntile tiles carved from one buffer (kSweMfTileBytes each).
SweMfTiles swe_mf_tiles(void* base, int64_t ntile) {
  unsigned char* p = static_cast<unsigned char*>(base);
  SweMfTiles T;
  T.cen = reinterpret_cast<double4*>(p);
  p += 32 * ntile;
  T.scen = reinterpret_cast<double4*>(p);
  p += 32 * kSweMfNsub * ntile;
  T.rec = reinterpret_cast<uint4*>(p);
  return T;
}

// Block-wide max / sum of v over 256 threads (red: 4 doubles of LDS); every
// thread gets the result.
__device__ __forceinline__ double block_max256(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

__device__ __forceinline__ double block_sum256(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// (y', |y'|^2 / 2) in FP32 for offset e (FP64); q from the rounded offset.
__device__ __forceinline__ float4 swe_mf_offset(double e0, double e1,
                                                double e2) {
  const float f0 = static_cast<float>(e0), f1 = static_cast<float>(e1),
              f2 = static_cast<float>(e2);
  const double q = static_cast<double>(f0) * f0 +
                   static_cast<double>(f1) * f1 + static_cast<double>(f2) * f2;
  return make_float4(f0, f1, f2, static_cast<float>(0.5 * q));
}

// The records of one tile from its cnt (> 0) packed sources at src; a block
// of 256 threads, thread jj takes source jj (wave s: sub-tile s).
__device__ __forceinline__ void swe_mf_pack_tile(const SweSrc* __restrict__ src,
                                                 int cnt, const SweMfTiles& T) {
  __shared__ double red[4];
  __shared__ double scale[32];
  const int jj = threadIdx.x;
  const bool real = jj < cnt;
  SweSrc s;
  s.p = make_double4(0.0, 0.0, 0.0, 0.0);
  s.q = make_double4(0.0, 0.0, 0.0, 0.0);
  if (real) s = src[jj];
  const double m = static_cast<double>(cnt);
  const double c0 = block_sum256(s.p.x, red) / m;
  const double c1 = block_sum256(s.p.y, red) / m;
  const double c2 = block_sum256(s.p.z, red) / m;
  const double e0 = s.p.x - c0, e1 = s.p.y - c1, e2 = s.p.z - c2;
  const double R2 = block_max256(real ? e0 * e0 + e1 * e1 + e2 * e2 : 0.0, red);
  if (jj == 0) T.cen[0] = make_double4(c0, c1, c2, R2);
  float4* ya = reinterpret_cast<float4*>(T.rec);
  float4* yas = reinterpret_cast<float4*>(T.rec + kSweMfYas);
  ya[jj] = real ? swe_mf_offset(e0, e1, e2)
                  : make_float4(8.0f, 8.0f, 8.0f, 96.0f);

  // this wave's sub-tile
  const int sub = jj / kSweMfSub;
  const int ns = min(max(cnt - sub * kSweMfSub, 0), kSweMfSub);
  if (ns > 0) {
    const double ms = static_cast<double>(ns);
    const double s0 = wave_sum(s.p.x) / ms, s1 = wave_sum(s.p.y) / ms,
                 s2 = wave_sum(s.p.z) / ms;
    const double f0 = s.p.x - s0, f1 = s.p.y - s1, f2 = s.p.z - s2;
    double r2 = real ? f0 * f0 + f1 * f1 + f2 * f2 : 0.0;
    for (int off = 32; off > 0; off >>= 1) r2 = fmax(r2, __shfl_xor(r2, off, 64));
    if ((jj & 63) == 0) T.scen[sub] = make_double4(s0, s1, s2, r2);
    yas[jj] = real ? swe_mf_offset(f0, f1, f2)
                     : make_float4(8.0f, 8.0f, 8.0f, 96.0f);
  } else {
    if ((jj & 63) == 0) T.scen[sub] = make_double4(0.0, 0.0, 0.0, -1.0);
    yas[jj] = make_float4(8.0f, 8.0f, 8.0f, 96.0f);
  }

  const double y0 = s.p.x, y1 = s.p.y, y2 = s.p.z, a = s.p.w, b = s.q.x;
  double F[kSweMfR1 + kSweMfR2] = {
      a * y0,      a * y1,      a * y2,      b * y0,      b * y1,
      b * y2,      a * y0 * y0, a * y0 * y1, a * y0 * y2, a * y1 * y1,
      a * y1 * y2, a * y2 * y2, b * y0 * y0, b * y0 * y1, b * y0 * y2,
      b * y1 * y1, b * y1 * y2, b * y2 * y2};
  // per-row power-of-two scales: row maximum into [2^13, 2^14)
#pragma unroll
  for (int r = 0; r < kSweMfR1 + kSweMfR2; ++r) {
    const double mx = block_max256(fabs(F[r]), red);
    const int k = mx > 0.0 ? 14 - ilogb(mx) - 1 : 0;
    if (jj == 0) scale[r] = mx > 0.0 ? ldexp(1.0, -k) : 0.0;
    F[r] = ldexp(F[r], k);
  }
  __syncthreads();
  if (jj < 32) {
    double v = 0.0;
    if (jj < kSweMfR1) v = scale[jj];
    if (jj >= 16 && jj < 16 + kSweMfR2) v = scale[kSweMfR1 + jj - 16];
    reinterpret_cast<double*>(T.rec + kSweMfFsAt)[jj] = v;
  }
  // slot (g, i) of k-block kb that holds source jj
  const int kb = jj >> 5, sl = jj & 31;
  const int g = (sl & 15) >> 2, i = (sl & 3) + 4 * (sl >> 4);
  _Float16* h1 = reinterpret_cast<_Float16*>(T.rec + kSweMfFrAt);
  _Float16* h2 = reinterpret_cast<_Float16*>(T.rec + kSweMfFr2At);
#pragma unroll
  for (int r = 0; r < kSweMfR1 + kSweMfR2; ++r) {
    const _Float16 hi = static_cast<_Float16>(static_cast<float>(F[r]));
    const _Float16 lo =
        static_cast<_Float16>(static_cast<float>(F[r] - static_cast<double>(hi)));
    if (r < kSweMfR1) {
      h1[((((kb * 2 + 0) * 4 + g) * kSweMfR1) + r) * 8 + i] = hi;
      h1[((((kb * 2 + 1) * 4 + g) * kSweMfR1) + r) * 8 + i] = lo;
    } else {
      const int r2 = r - kSweMfR1;
      h2[((((kb * 2 + 0) * 4 + g) * kSweMfR2) + r2) * 8 + i] = hi;
      h2[((((kb * 2 + 1) * 4 + g) * kSweMfR2) + r2) * 8 + i] = lo;
    }
  }
}

// One block per tile of the packed sources j < *count.
__global__ __launch_bounds__(256) void swe_mf_pack_kernel(
    const SweSrc* __restrict__ src, const int32_t* __restrict__ count,
    SweMfTiles T) {
  const int n = *count;
  const int j0 = blockIdx.x * kSweTile;
  if (j0 >= n) return;
  swe_mf_pack_tile(src + j0, min(kSweTile, n - j0), T.from(blockIdx.x));
}

typedef float swe_mf4 __attribute__((ext_vector_type(4)));
typedef _Float16 swe_mh8 __attribute__((ext_vector_type(8)));
typedef _Float16 swe_mh2 __attribute__((ext_vector_type(2)));
typedef float swe_mf2 __attribute__((ext_vector_type(2)));

// Two FP32 values into packed f16 hi parts and packed f16 lo parts.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& hi,
                                           uint32_t& lo) {
  const swe_mh2 h = __builtin_convertvector(swe_mf2{a, b}, swe_mh2);
  const swe_mf2 r = {a - static_cast<float>(h[0]), b - static_cast<float>(h[1])};
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, swe_mh2));
}

// x minus the f16 in half H of h, in one v_fma_mix_f32 (x - hi is exact
// when hi is x rounded to f16).
template <int H>
__device__ __forceinline__ float minus_half(float x, uint32_t h) {
  float r;
  if constexpr (H == 0)
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[0,0,1]"
        : "=v"(r) : "v"(x), "v"(h));
  else
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "=v"(r) : "v"(x), "v"(h));
  return r;
}

// split_pair with the differences in v_fma_mix_f32.
__device__ __forceinline__ void split_pair_mix(float a, float b, uint32_t& hi,
                                               uint32_t& lo) {
  hi = __builtin_bit_cast(
      uint32_t, __builtin_convertvector(swe_mf2{a, b}, swe_mh2));
  const swe_mf2 r = {minus_half<0>(a, hi), minus_half<1>(b, hi)};
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, swe_mh2));
}

// Adds Q Y Q (Q = I - x x^T, Y symmetric: xx, xy, xz, yy, yz, zz) to G.
__device__ __forceinline__ void add_qyq(double* G, const double* Y,
                                        const double* x) {
  const double v0 = Y[0] * x[0] + Y[1] * x[1] + Y[2] * x[2];
  const double v1 = Y[1] * x[0] + Y[3] * x[1] + Y[4] * x[2];
  const double v2 = Y[2] * x[0] + Y[4] * x[1] + Y[5] * x[2];
  const double sv = x[0] * v0 + x[1] * v1 + x[2] * v2;
  const double v[3] = {v0, v1, v2};
  const int ia[6] = {0, 0, 0, 1, 1, 2}, ib[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    const int p = ia[e], q = ib[e];
    G[e] += Y[e] - x[p] * v[q] - v[p] * x[q] + sv * x[p] * x[q];
  }
}

// Far sums of k-blocks kb0 .. kb1 - 1 of one tile (its record rec, whose operands
// are fetched a k-block ahead; ya: the record's offsets from the centroid c of
// the tile or sub-tile summed) for the wave's four groups of 16 targets, carried into F1 / F2: lane (g, col)
// holds rows 4 g + v of target 16 G + col.  e is this lane's target minus c,
// dist2 = |e|^2, R2 = the radius^2 around c.
__device__ __forceinline__ void swe_mf_far_tile(
    const uint4* __restrict__ rec, const float* __restrict__ ya, int kb0, int kb1, bool in, double e0,
    double e1, double e2, double dist2, double R2, double eps2, int col, int g,
    double (*F1)[4], double (*F2)[4]) {
  constexpr int NG = 4;
  const float e2f = static_cast<float>(eps2);
  // this lane's target as a stage-1 operand: (-x', 1) and |x'|^2 / 2 +
  // eps^2 (lanes past the end: D = 4 for every source)
  const float xp0 = static_cast<float>(e0), xp1 = static_cast<float>(e1),
              xp2 = static_cast<float>(e2);
  const float own[5] = {
      in ? -xp0 : 0.0f, in ? -xp1 : 0.0f, in ? -xp2 : 0.0f, in ? 1.0f : 0.0f,
      in ? fmaf(0.5f, fmaf(xp2, xp2, fmaf(xp1, xp1, xp0 * xp0)), e2f) : 4.0f};
  // smallest D over the sphere around c in each group of 16 targets (it only
  // sets a power of two with room of four times below the f16 range)
  const float gap = __builtin_amdgcn_sqrtf(static_cast<float>(dist2)) -
                    __builtin_amdgcn_sqrtf(static_cast<float>(R2));
  float dl = in ? fmaf(0.5f * gap, gap, e2f) : 4.0f;
  dl = fmaxf(fminf(dl, 4.0f), 1e-30f);
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) dl = fminf(dl, __shfl_xor(dl, off, 64));
  float sig[NG], Bv[NG], Cv[NG];
#pragma unroll
  for (int G = 0; G < NG; ++G) {
    const float dG = __shfl(dl, 16 * G, 64);
    // sigma dl in [2^-7, 2^-6): w = 1 / (sigma D) <= 2^7
    sig[G] = __builtin_ldexpf(1.0f, -__builtin_amdgcn_frexp_expf(dG) - 6);
    const int from = 16 * G + col;
    const float b0 = __shfl(own[0], from, 64), b1 = __shfl(own[1], from, 64);
    const float b2 = __shfl(own[2], from, 64), b3 = __shfl(own[3], from, 64);
    const float pq = __shfl(own[4], from, 64);
    Bv[G] = sig[G] * (g == 0 ? b0 : g == 1 ? b1 : g == 2 ? b2 : b3);
    Cv[G] = sig[G] * pq;
  }
  swe_mf4 S1[NG], S2[NG];
#pragma unroll
  for (int G = 0; G < NG; ++G) S1[G] = S2[G] = swe_mf4{0.0f, 0.0f, 0.0f, 0.0f};
  // lanes of unused rows repeat the last row: their results are not read
  const uint4* fr = rec + kSweMfFrAt + g * kSweMfR1 + min(col, kSweMfR1 - 1);
  const uint4* fr2 = rec + kSweMfFr2At + g * kSweMfR2 + min(col, kSweMfR2 - 1);
  struct Operands {
    float a0, a1;
    uint4 u1h, u1l, u2h, u2l;
  };
  auto fetch = [&](int kb) {
    Operands o;
    o.a0 = ya[(32 * kb + col) * 4 + g];
    o.a1 = ya[(32 * kb + 16 + col) * 4 + g];
    o.u1h = fr[(kb * 2 + 0) * 4 * kSweMfR1];
    o.u1l = fr[(kb * 2 + 1) * 4 * kSweMfR1];
    o.u2h = fr2[(kb * 2 + 0) * 4 * kSweMfR2];
    o.u2l = fr2[(kb * 2 + 1) * 4 * kSweMfR2];
    return o;
  };
  Operands next = fetch(kb0);
#pragma unroll 1
  for (int kb = kb0; kb < kb1; ++kb) {
    const Operands cur = next;
    next = fetch(min(kb + 1, kb1 - 1));
    const float a0 = cur.a0, a1 = cur.a1;
    const swe_mh8 A1h = __builtin_bit_cast(swe_mh8, cur.u1h);
    const swe_mh8 A1l = __builtin_bit_cast(swe_mh8, cur.u1l);
    const swe_mh8 A2h = __builtin_bit_cast(swe_mh8, cur.u2h);
    const swe_mh8 A2l = __builtin_bit_cast(swe_mh8, cur.u2l);
    swe_mf4 O[NG][2];
#pragma unroll
    for (int G = 0; G < NG; ++G) {
      const swe_mf4 C = {Cv[G], Cv[G], Cv[G], Cv[G]};
      O[G][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, Bv[G], C, 0, 0, 0);
      O[G][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, Bv[G], C, 0, 0, 0);
    }
#pragma unroll
    for (int G = 0; G < NG; ++G) {
      float w[8];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        w[v] = __builtin_amdgcn_rcpf(O[G][0][v]);
        w[4 + v] = __builtin_amdgcn_rcpf(O[G][1][v]);
      }
      uint32_t wh[4], wl[4], vh[4], vl[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        split_pair_mix(w[2 * p], w[2 * p + 1], wh[p], wl[p]);
        split_pair(w[2 * p] * w[2 * p], w[2 * p + 1] * w[2 * p + 1], vh[p],
                   vl[p]);
      }
      const swe_mh8 Wh = __builtin_bit_cast(swe_mh8, make_uint4(wh[0], wh[1], wh[2], wh[3]));
      const swe_mh8 Wl = __builtin_bit_cast(swe_mh8, make_uint4(wl[0], wl[1], wl[2], wl[3]));
      const swe_mh8 Vh = __builtin_bit_cast(swe_mh8, make_uint4(vh[0], vh[1], vh[2], vh[3]));
      const swe_mh8 Vl = __builtin_bit_cast(swe_mh8, make_uint4(vl[0], vl[1], vl[2], vl[3]));
      S1[G] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A1h, Wh, S1[G], 0, 0, 0);
      S2[G] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2h, Vh, S2[G], 0, 0, 0);
      S1[G] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A1l, Wh, S1[G], 0, 0, 0);
      S2[G] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2l, Vh, S2[G], 0, 0, 0);
      S1[G] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A1h, Wl, S1[G], 0, 0, 0);
      S2[G] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2h, Vl, S2[G], 0, 0, 0);
    }
  }
  // undo the scales into the FP64 sums: w = 1 / (sigma D)
  const double* fs = reinterpret_cast<const double*>(rec + kSweMfFsAt);
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const double s1 = fs[4 * g + v], s2 = fs[16 + 4 * g + v];
#pragma unroll
    for (int G = 0; G < NG; ++G) {
      const double sg1 = static_cast<double>(sig[G]);
      F1[G][v] = fma(static_cast<double>(S1[G][v]), sg1 * s1, F1[G][v]);
      F2[G][v] = fma(static_cast<double>(S2[G][v]), sg1 * sg1 * s2, F2[G][v]);
    }
  }
}

constexpr int kSweMfRows = kSweMfR1 + kSweMfR2;

// Row r of this lane's target's far sums (the target is 16 g + col; row
// 4 q + v of it sits in lane col + 16 q, group g).  Every lane calls it.
__device__ __forceinline__ void swe_mf_gather(double (*F1)[4], double (*F2)[4],
                                              int col, int g, double* R) {
#pragma unroll
  for (int r = 0; r < kSweMfR2; ++r) {
    const int from = col + 16 * (r >> 2), v = r & 3;
    double a1 = 0.0, a2 = 0.0;
#pragma unroll
    for (int G = 0; G < 4; ++G) {
      const double t2 = __shfl(F2[G][v], from, 64);
      if (g == G) a2 = t2;
      if (r < kSweMfR1) {
        const double t1 = __shfl(F1[G][v], from, 64);
        if (g == G) a1 = t1;
      }
    }
    R[kSweMfR1 + r] = a2;
    if (r < kSweMfR1) R[r] = a1;
  }
}

// Adds the projected far sums R (set 1 rows 0..5, set 2 rows 6..17) of
// target x to its accumulators.
__device__ __forceinline__ void swe_mf_add_far(SweAcc& acc, const double* R,
                                               const double* x) {
  acc.Vy[0] += R[0];
  acc.Vy[1] += R[1];
  acc.Vy[2] += R[2];
  const double xs = x[0] * R[3] + x[1] * R[4] + x[2] * R[5];
  acc.Vg[0] += R[3] - xs * x[0];
  acc.Vg[1] += R[4] - xs * x[1];
  acc.Vg[2] += R[5] - xs * x[2];
  acc.Bt += xs;
  add_qyq(acc.Gd, R + kSweMfR1, x);
  add_qyq(acc.Gs, R + kSweMfR1 + 6, x);
}

// First pass: the far tiles, and the far sub-tiles of the others, of each
// wave in source chunk `chunk` of C equal runs of tiles; the 18 raw far sums
// go to rows 18 row .. of sg.part, added to what they hold if `add`.  Each wave
// reads the records of its far tiles from L2 and waits for no other.
//
// What bounds it: per 64 pairs 37 cycles of vector issue (reciprocal 8, f16
// splits of w and w^2 16, products 2, the rest once per tile) and 20 of matrix
// products; at 256 registers two waves of a SIMD overlap little of them (68 %
// and 33 % busy).  Level 6 (1.0e10 pairs): 3.76 ms.  Records staged in LDS by
// the block, a tile ahead, took 3.83 there, and 1.18 ms against 0.85 for eight
// members of 10,700 cubed-sphere faces, most of whose tiles are near: the block
// then copies every record and waits for its slowest wave at each.
template <int BLOCK>
__device__ __forceinline__ void swe_mf_far_block(
    const SweMfTiles& mt, int nsrc, const SweSeg& sg, int blk, int chunk, int C,
    const SweParams& P, int row, bool add) {
  const int64_t n_live = sg.d_n ? *sg.d_n : sg.n;
  const int64_t c = static_cast<int64_t>(blk) * BLOCK + threadIdx.x;
  if (c - (threadIdx.x & 63) >= n_live) return;  // no target in the wave
  const bool in = c < n_live;
  const int64_t i = swe_target(sg, c, in);
  const double* px = sg.x + i * sg.es;
  const double x[3] = {px[0], px[sg.cs], px[2 * sg.cs]};
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  const int ntile = (nsrc + kSweTile - 1) / kSweTile;
  const int t0 = static_cast<int>(static_cast<int64_t>(ntile) * chunk / C);
  const int t1 = static_cast<int>(static_cast<int64_t>(ntile) * (chunk + 1) / C);
  double F1[4][4], F2[4][4];
#pragma unroll
  for (int G = 0; G < 4; ++G)
#pragma unroll
    for (int v = 0; v < 4; ++v) F1[G][v] = F2[G][v] = 0.0;
  if (t0 < t1) {
    double4 cc_next = vload(mt.cen, t0);
#pragma unroll 1
    for (int t = t0; t < t1; ++t) {
      const double4 cc = cc_next;
      cc_next = vload(mt.cen, min(t + 1, t1 - 1));
      const uint4* rec = mt.rec + kSweMfRec * static_cast<int64_t>(t);
      // a far tile is one range of k-blocks; a near tile, its far sub-tiles
      // with offsets from their own centroids
      const bool tile_far = !__ballot(in && swe_mf_near(x, cc));
      const int nrange = tile_far ? 1 : kSweMfNsub;
#pragma unroll 1
      for (int sub = 0; sub < nrange; ++sub) {
        double4 cs = cc;
        const uint4* ya = rec;
        int kb0 = 0, kb1 = kSweMfKb;
        if (!tile_far) {
          cs = mt.scen[kSweMfNsub * static_cast<int64_t>(t) + sub];
          if (cs.w < 0.0 || __ballot(in && swe_mf_near(x, cs))) continue;
          ya += kSweMfYas;
          kb0 = sub * (kSweMfSub / 32);
          kb1 = kb0 + kSweMfSub / 32;
        }
        const double e0 = x[0] - cs.x, e1 = x[1] - cs.y, e2 = x[2] - cs.z;
        swe_mf_far_tile(rec, reinterpret_cast<const float*>(ya), kb0, kb1, in,
                        e0, e1, e2, e0 * e0 + e1 * e1 + e2 * e2, cs.w, P.eps2,
                        col, g, F1, F2);
      }
    }
  }
  double R[kSweMfRows];
  swe_mf_gather(F1, F2, col, g, R);
  if (!in) return;
  double* part = sg.part + kSweMfRows * row * sg.pstride + c;
  for (int r = 0; r < kSweMfRows; ++r) {
    double* p = part + r * sg.pstride;
    *p = add ? *p + R[r] : R[r];
  }
}

// Second pass, four waves of a block on the same 64 targets: wave w scans the
// tiles (the first pass's classification: tile near, then sub-tile near) and
// the PSE range of its targets, stages sub-tile w of each tile it needs into
// its own LDS slice (one record per lane) and sums it in FP64; no barriers
// until the four sums are added in a fixed tree.  Then wave 0 adds the first
// pass's far sums and writes the outputs.  SHARE: pairs per FP64 reciprocal
// without a self pair.  stage: kSweMfSub records of this wave.
// What bounds it: FP64 issue and waits of too few waves: one wave per 64
// targets left 1.1 waves per SIMD on average (level 6: 1.16 ms, now 0.95).
template <int SHARE>
__device__ __forceinline__ void swe_mf_near_block(
    const SweSrc* __restrict__ src, const SweMfTiles& mt, int nsrc,
    const SweSeg& sg, int blk, int rows, const SweParams& P, SweSrc* stage,
    double (*red)[kSweRows][64]) {
  const double eps2 = P.eps2, inv_pse_e2 = P.inv_pse_e2;
  const double pse_cut2 = P.pse_cut2;
  const int do_pse = P.do_pse;
  const int64_t n_live = sg.d_n ? *sg.d_n : sg.n;
  if (static_cast<int64_t>(blk) * 64 >= n_live) return;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t c = static_cast<int64_t>(blk) * 64 + lane;
  const bool in = c < n_live;
  const int64_t i = swe_target(sg, c, in);
  const double* px = sg.x + i * sg.es;
  const double x[3] = {px[0], px[sg.cs], px[2 * sg.cs]};
  const double s_i = (do_pse && sg.surf) ? sg.surf[i] : 0.0;
  const int self = swe_self(sg, c, i, in, P.skip_self);
  const double rcut = sqrt(pse_cut2);
  const int last = max((nsrc + kSweTile - 1) / kSweTile - 1, 0);
  // is x within PSE range of some source in the sphere (c, c.w = r^2)?
  auto pse_near = [&](const double4& s) {
    const double p0 = x[0] - s.x, p1 = x[1] - s.y, p2 = x[2] - s.z;
    const double rr = sqrt(s.w) + rcut;
    return in && p0 * p0 + p1 * p1 + p2 * p2 <= rr * rr;
  };
  SweAcc acc;
  acc.zero();
  double4 cc_next = vload(mt.cen, 0);
  for (int t = 0; t <= last && t * kSweTile < nsrc; ++t) {
    const double4 cc = cc_next;
    cc_next = vload(mt.cen, min(t + 1, last));
    const bool near = __ballot(in && swe_mf_near(x, cc)) != 0;
    const bool pse = do_pse && __ballot(pse_near(cc)) != 0;
    if (!near && !pse) continue;
    const double4 cs = mt.scen[kSweMfNsub * static_cast<int64_t>(t) + w];
    if (cs.w < 0.0) continue;
    const bool nsub = near && __ballot(in && swe_mf_near(x, cs)) != 0;
    const bool psub = pse && __ballot(pse_near(cs)) != 0;
    if (!nsub && !psub) continue;
    const int s0 = t * kSweTile + w * kSweMfSub;
    const int cnt = min(kSweMfSub, nsrc - s0);
    // the previous sub-tile's reads are done before it is overwritten;
    // the writes land before any lane reads (LDS is in order per wave)
    __builtin_amdgcn_wave_barrier();
    stage[lane] = src[s0 + lane];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (nsub) {
      const bool diag =
          static_cast<unsigned>(self - s0) < static_cast<unsigned>(cnt);
      if (__ballot(diag))
        swe_tile_f64<2>(acc, stage, cnt, x, eps2, self - s0, true);
      else
        swe_tile_f64<SHARE>(acc, stage, cnt, x, eps2, -1, false);
    }
    if (psub) {
      double L = 0.0;
      swe_pse_tile(stage, cnt, x, s_i, inv_pse_e2, pse_cut2, L);
      acc.L1 += L;
    }
  }
  // sums of the four waves: (w, w + 2), then (0, 1)
#pragma unroll 1
  for (int half = kSweMfNsub / 2; half > 0; half >>= 1) {
    __syncthreads();  // the previous values are read
    if (w >= half && w < 2 * half)
      swe_rows(acc, [&](int r, double& v) { red[w - half][r][lane] = v; });
    __syncthreads();
    if (w < half)
      swe_rows(acc, [&](int r, double& v) { v += red[w][r][lane]; });
  }
  if (w != 0 || !in) return;
  double R[kSweMfRows];
#pragma unroll
  for (int r = 0; r < kSweMfRows; ++r) R[r] = 0.0;
  for (int k = 0; k < rows; ++k) {
    const double* part = sg.part + kSweMfRows * k * sg.pstride + c;
#pragma unroll
    for (int r = 0; r < kSweMfRows; ++r) R[r] += part[r * sg.pstride];
  }
  swe_mf_add_far(acc, R, x);
  double u[3], dd, lap;
  swe_finalize(acc, x, k4OverPi * inv_pse_e2 * inv_pse_e2, u, &dd, &lap);
  if (sg.out_u) {
    double* o = sg.out_u + i * sg.oes;
    o[0] = u[0];
    o[sg.ocs] = u[1];
    o[2 * sg.ocs] = u[2];
  }
  if (sg.out_ddot) sg.out_ddot[i] = dd;
  if (sg.out_laps && do_pse) sg.out_laps[i] = lap;
}

// MINW: minimum waves per SIMD asked of the register allocator.  With P.rows =
// P.C block b C + k sums chunk k of target block b; with P.rows = 1 (no
// workspace for more) block b sums every chunk in order, to the same bits.
template <int BLOCK, int MINW>
__global__ __launch_bounds__(BLOCK, MINW) void swe_mf_far_kernel(
    const SweSrc* __restrict__, const double4* __restrict__,
    const int32_t* __restrict__ count, SweSeg s0, SweSeg s1, SweParams P) {
  const int b = flat_block() / P.rows;
  const int k0 = flat_block() % P.rows;
  const bool first = b < s0.nblocks;
  const SweSeg& sg = first ? s0 : s1;
  const int blk = first ? b : b - s0.nblocks;
#pragma unroll 1
  for (int k = k0; k < P.C; k += P.rows)
    swe_mf_far_block<BLOCK>(P.mf, *count, sg, blk, k, P.C, P, k0, k != k0);
}

// SHARE: pairs per FP64 reciprocal in near sub-tiles (2 or 4).
// Blocks of 64 targets: nblocks of the segments counts those.
template <int MINW, int SHARE>
__global__ __launch_bounds__(256, MINW) void swe_mf_near_kernel(
    const SweSrc* __restrict__ src, const double4* __restrict__,
    const int32_t* __restrict__ count, SweSeg s0, SweSeg s1, SweParams P) {
  __shared__ SweSrc stage[4 * kSweMfSub];
  __shared__ double red[2][kSweRows][64];
  const int b = flat_block();
  const bool first = b < s0.nblocks;
  const SweSeg& sg = first ? s0 : s1;
  const int blk = first ? b : b - s0.nblocks;
  swe_mf_near_block<SHARE>(src, P.mf, *count, sg, blk, P.rows, P,
                           stage + (threadIdx.x & ~63), red);
}

// ------------------------------------------------------------ ensembles --
// grid (ceil(max member faces / 256), n_members): member m's c-th undivided
// face at packed slot P_m + c; zero sources pad the member's last tile.  With
// `runs` also the bounding sphere of each run of 64 (at packed run P_m / 64 on).
__global__ __launch_bounds__(256) void swe_ens_pack_kernel(
    const double* __restrict__ sx, int64_t es, int64_t cs,
    const double* __restrict__ zeta, const double* __restrict__ sigma,
    const double* __restrict__ area, const double* __restrict__ surf,
    const int32_t* __restrict__ inv, const EnsMember* __restrict__ mem,
    SweSrc* __restrict__ out, double4* __restrict__ runs) {
  const EnsMember M = mem[blockIdx.y];
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int padded = (M.cnt + kSweTile - 1) / kSweTile * kSweTile;
  if (c >= padded) return;
  SweSrc v;
  v.p = make_double4(0.0, 0.0, 0.0, 0.0);
  v.q = make_double4(0.0, 0.0, 0.0, 0.0);
  if (c < M.cnt) {
    const int64_t r = static_cast<int64_t>(M.R) + c;
    const int64_t i = inv ? inv[r] : r;
    const double* p = sx + i * es;
    const double A = area[i];
    v.p = make_double4(p[0], p[cs], p[2 * cs], zeta[i] * A * kInv4Pi);
    v.q = make_double4(sigma[i] * A * kInv4Pi, A, surf ? surf[i] : 0.0, 0.0);
  }
  out[M.P + c] = v;
  // padded is a multiple of 256, so whole waves get here
  const int left = M.cnt - c / 64 * 64;
  if (runs && left > 0)
    swe_run_sphere(v.p, min(left, 64), runs + (M.P + c) / 64);
}

// grid (ceil(max member faces / 256), n_members): bounding sphere of tile t
// of member m over its real sources only.
__global__ __launch_bounds__(kSweTile) void swe_ens_bounds_kernel(
    const SweSrc* __restrict__ src, const EnsMember* __restrict__ mem,
    double4* __restrict__ bounds) {
  __shared__ double red[kSweTile / 64];
  const EnsMember M = mem[blockIdx.y];
  const int j0 = blockIdx.x * kSweTile;
  if (j0 >= M.cnt) return;
  const double4 c = src[M.P + j0].p;
  const int j = j0 + threadIdx.x;
  double r2 = 0.0;
  if (j < M.cnt) {
    const double4 y = src[M.P + j].p;
    const double a = y.x - c.x, b = y.y - c.y, e = y.z - c.z;
    r2 = a * a + b * b + e * e;
  }
  for (int off = 32; off > 0; off >>= 1) r2 = fmax(r2, __shfl_down(r2, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = r2;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = 0.0;
    for (int w = 0; w < kSweTile / 64; ++w) m = fmax(m, red[w]);
    bounds[(M.P + j0) / kSweTile] = make_double4(c.x, c.y, c.z, m);
  }
}

// grid (ceil(max member faces / 256), n_members): the tile records of
// member m (its tiles start at packed tile P_m / 256).
__global__ __launch_bounds__(256) void swe_ens_mf_pack_kernel(
    const SweSrc* __restrict__ src, const EnsMember* __restrict__ mem,
    SweMfTiles T) {
  const EnsMember M = mem[blockIdx.y];
  const int j0 = blockIdx.x * kSweTile;
  if (j0 >= M.cnt) return;
  swe_mf_pack_tile(src + M.P + j0, min(kSweTile, M.cnt - j0),
                   T.from((static_cast<int64_t>(M.P) + j0) / kSweTile));
}

struct SweEnsArgs {
  const EnsMember* mem;
  const int4* items;
  int n_items;
  int32_t* queue;
  SweSeg vert;  // arrays of the vertex targets (x, surf, outputs)
  SweSeg face;  // arrays of the face targets
  const int32_t* rank;
  const int32_t* inv;
  int skip_masked;
  SweParams P;
};

__device__ __forceinline__ SweSeg swe_ens_segment(const SweEnsArgs& A,
                                                  const EnsMember& M, int seg) {
  if (seg == 0) {
    SweSeg sg = A.vert;
    sg.n = M.nv;
    sg.slot_base = M.v0;
    if (A.vert.index) sg.index = A.vert.index + M.v0;
    return sg;
  }
  SweSeg sg = A.face;
  if (A.skip_masked && A.inv) {
    sg.index = A.inv + M.R;
    sg.n = M.cnt;
    sg.self_identity = 1;
  } else {
    sg.n = M.nf;
    sg.slot_base = M.f0;
    if (A.rank) {
      sg.self_rank = A.rank;
      sg.rank_base = M.R;
    } else {
      sg.self_identity = 1;
    }
  }
  return sg;
}

__device__ __forceinline__ int swe_ens_next(const SweEnsArgs& A, int* slot) {
  if (threadIdx.x == 0) *slot = atomicAdd(A.queue, 1);
  __syncthreads();
  const int it = *slot;
  __syncthreads();
  return it;
}

// Chunk sums of segment `seg` of member M: ROWS C rows of its targets.
template <int ROWS = kSweRows>
__device__ __forceinline__ void swe_ens_parts(SweSeg& sg, const EnsMember& M,
                                              int seg, double* part) {
  sg.part = part + ROWS * (M.part0 + (seg == 0 ? 0 : M.C * M.nv));
  sg.pstride = seg == 0 ? M.nv : M.nf;
}

// Wave-split sums of every member: one block per (item, chunk) of A.items, or
// without part one per item, which sums every chunk.
template <bool SPLIT>
__global__ __launch_bounds__(64 * kSweWaves, 4) void swe_ens_wave_kernel(
    const double* __restrict__ src, const double4* __restrict__ sub,
    SweEnsArgs A, double* part) {
  __shared__ double red[kSweWaves / 2][kSweRows][64];
  if (flat_block() >= A.n_items) return;
  const int4 w = A.items[flat_block()];
  const EnsMember M = A.mem[w.x];
  SweSeg sg = swe_ens_segment(A, M, w.y);
  if (SPLIT) swe_ens_parts(sg, M, w.y, part);
  swe_wave_block<SPLIT>(src + static_cast<int64_t>(M.P) * 8, sub + M.P / 64,
                        M.cnt, sg, w.z, w.w, M.C, A.P, red);
}

__global__ __launch_bounds__(64) void swe_ens_wave_reduce_kernel(SweEnsArgs A,
                                                                 double* part) {
  if (flat_block() >= A.n_items) return;
  const int4 w = A.items[flat_block()];
  const EnsMember M = A.mem[w.x];
  SweSeg sg = swe_ens_segment(A, M, w.y);
  swe_ens_parts(sg, M, w.y, part);
  swe_wave_reduce(sg, static_cast<int64_t>(w.z) * 64 + threadIdx.x, M.C, A.P);
}

template <int BLOCK, int SHARE, int MINW>
__global__ __launch_bounds__(BLOCK, MINW) void swe_ens_f64_kernel(
    const SweSrc* __restrict__ src, const double4* __restrict__ bounds,
    SweEnsArgs A) {
  __shared__ SweSrc tile[kSweTile];
  __shared__ int slot;
  for (;;) {
    const int it = swe_ens_next(A, &slot);
    if (it >= A.n_items) break;
    const int4 w = A.items[it];
    const EnsMember M = A.mem[w.x];
    const SweSeg sg = swe_ens_segment(A, M, w.y);
    swe_f64_block<BLOCK, SHARE>(src + M.P, bounds + M.P / kSweTile, M.cnt,
                                sg, w.z, A.P, tile);
  }
}

template <int BLOCK, int MINW>
__global__ __launch_bounds__(BLOCK, MINW) void swe_ens_mixed_kernel(
    const SweSrc* __restrict__ src, const double4* __restrict__ bounds,
    SweEnsArgs A) {
  __shared__ F4x2 tile[kSweTile];
  __shared__ SweSrc tile64[kSweTile];
  __shared__ int slot;
  for (;;) {
    const int it = swe_ens_next(A, &slot);
    if (it >= A.n_items) break;
    const int4 w = A.items[it];
    const EnsMember M = A.mem[w.x];
    const SweSeg sg = swe_ens_segment(A, M, w.y);
    swe_mixed_block<BLOCK>(src + M.P, bounds + M.P / kSweTile, M.cnt, sg, w.z,
                           A.P, tile, tile64);
  }
}

// Far sums of segment `seg` of member M: the rows of its chunks, or with
// A.P.rows = 1 one set per target.
__device__ __forceinline__ void swe_ens_far(SweSeg& sg, const EnsMember& M,
                                            int seg, const SweEnsArgs& A,
                                            double* part) {
  if (A.P.rows == 1) {
    sg.part = part + kSweMfRows * (M.v0 + M.f0 + (seg == 0 ? 0 : M.nv));
    sg.pstride = seg == 0 ? M.nv : M.nf;
  } else {
    swe_ens_parts<kSweMfRows>(sg, M, seg, part);
  }
}

// The two passes of every member: one block per (item, chunk) of A.items, or
// with A.P.rows = 1 one per item, then four of 64 targets per item.
template <int BLOCK, int MINW>
__global__ __launch_bounds__(BLOCK, MINW) void swe_ens_mf_far_kernel(
    SweEnsArgs A, double* part) {
  if (flat_block() >= A.n_items) return;
  const int4 w = A.items[flat_block()];
  const EnsMember M = A.mem[w.x];
  SweSeg sg = swe_ens_segment(A, M, w.y);
  swe_ens_far(sg, M, w.y, A, part);
  const SweMfTiles mt = A.P.mf.from(M.P / kSweTile);
  const int step = A.P.rows == 1 ? 1 : M.C;
#pragma unroll 1
  for (int k = w.w; k < M.C; k += step)
    swe_mf_far_block<BLOCK>(mt, M.cnt, sg, w.z, k, M.C, A.P,
                            A.P.rows == 1 ? 0 : k, k != w.w);
}

template <int MINW, int SHARE>
__global__ __launch_bounds__(256, MINW) void swe_ens_mf_near_kernel(
    const SweSrc* __restrict__ src, SweEnsArgs A, double* part) {
  __shared__ SweSrc stage[4 * kSweMfSub];
  __shared__ double red[2][kSweRows][64];
  if (flat_block() / 4 >= A.n_items) return;
  const int4 w = A.items[flat_block() / 4];
  const EnsMember M = A.mem[w.x];
  SweSeg sg = swe_ens_segment(A, M, w.y);
  swe_ens_far(sg, M, w.y, A, part);
  swe_mf_near_block<SHARE>(src + M.P, A.P.mf.from(M.P / kSweTile), M.cnt, sg,
                           4 * w.z + flat_block() % 4,
                           A.P.rows == 1 ? 1 : M.C, A.P,
                           stage + (threadIdx.x & ~63), red);
}

// ------------------------------------------------------ kernel registry ---
using SweKernel = void (*)(const SweSrc*, const double4*, const int32_t*,
                           SweSeg, SweSeg, SweParams);
using SweEnsKernel = void (*)(const SweSrc*, const double4*, SweEnsArgs);
using SweEnsFarKernel = void (*)(SweEnsArgs, double*);
using SweEnsNearKernel = void (*)(const SweSrc*, SweEnsArgs, double*);
struct SweVariant {
  SweKernel fn;
  SweEnsKernel ens;
  const char* name;
  // matrix-core sums: the far pass, then the near tiles, PSE and outputs
  SweKernel far = nullptr, near = nullptr;
  SweEnsFarKernel ens_far = nullptr;
  SweEnsNearKernel ens_near = nullptr;
  bool wave = false;  // wave-split sums (64 targets per work item)

  bool mf() const { return far != nullptr; }
  EnsChunks chunks() const {
    return wave ? kEnsSwe : mf() ? kEnsSweMixed : kEnsWhole;
  }
};
constexpr int kSweBlock = 256;
// The numbers are kept: programs and tuning tables hold them.
const SweVariant kSweF64Variants[] = {
    {swe_f64_kernel<kSweBlock, 4, 3>, swe_ens_f64_kernel<kSweBlock, 4, 3>,
     "share4_occ3"},
    {swe_f64_kernel<kSweBlock, 4, 4>, swe_ens_f64_kernel<kSweBlock, 4, 4>,
     "share4_occ4"},
    {swe_f64_kernel<kSweBlock, 2, 4>, swe_ens_f64_kernel<kSweBlock, 2, 4>,
     "share2_occ4"},
    {swe_f64_kernel<kSweBlock, 2, 3>, swe_ens_f64_kernel<kSweBlock, 2, 3>,
     "share2_occ3"},
    // 4: the default
    {nullptr, nullptr, "wave8_scalar", nullptr, nullptr, nullptr, nullptr, true},
};
constexpr int kDefaultSweF64 = 4;
const SweVariant kSweMixedVariants[] = {
    // two passes: far tiles and sub-tiles on the matrix cores, then near
    // sub-tiles and PSE terms in FP64 and the outputs
    {nullptr, nullptr, "mfma_f2n3", swe_mf_far_kernel<kSweBlock, 2>,
     swe_mf_near_kernel<3, 4>, swe_ens_mf_far_kernel<kSweBlock, 2>,
     swe_ens_mf_near_kernel<3, 4>},
    {nullptr, nullptr, "mfma_f2n4", swe_mf_far_kernel<kSweBlock, 2>,
     swe_mf_near_kernel<4, 4>, swe_ens_mf_far_kernel<kSweBlock, 2>,
     swe_ens_mf_near_kernel<4, 4>},
    // FP32 pair arithmetic on the vector ALUs
    {swe_mixed_kernel<kSweBlock, 4>, swe_ens_mixed_kernel<kSweBlock, 4>,
     "occ4"},
    {swe_mixed_kernel<kSweBlock, 3>, swe_ens_mixed_kernel<kSweBlock, 3>,
     "occ3"},
    {swe_mixed_kernel<kSweBlock, 2>, swe_ens_mixed_kernel<kSweBlock, 2>,
     "occ2"},
};
constexpr int kNumSweF64 = sizeof(kSweF64Variants) / sizeof(kSweF64Variants[0]);
constexpr int kNumSweMixed =
    sizeof(kSweMixedVariants) / sizeof(kSweMixedVariants[0]);

// Targets enough to fill the device with one wave for all sources of its
// targets, over too few sources to divide among eight waves: share4_occ3 is
// the faster FP64 form, and over a tile's half also faster than the mixed
// passes.  For arbitrary points only (n_src, else -1): a mesh has no such
// sizes, and a member of an ensemble keeps the bits of its problem alone.
// 1e5 and 1e6 targets against 20 and 80 sources: 38, 46 and 84, 237 us, eight
// waves 65, 77 and 452, 542, mixed 72, 93 and 362, 499; 5,000 targets 34 to 38
// in FP64 either way.  1e6 against 320: 857, eight waves 926, mixed 844.
bool swe_few_sources(int64_t n_targets, int64_t n_src, int precision) {
  if (n_src < 0 || n_targets < 32768) return false;
  return n_src <= 128 || (precision == LPM_FP64 &&
                          one_chunk(n_targets, n_src) && n_src <= 512);
}

// Variant of a launch; n_src: its sources where the targets are arbitrary
// points (else -1).
const SweVariant& swe_variant(lpm_ctx* ctx, int precision, int64_t n_targets,
                              int64_t n_src = -1) {
  const int family = precision == LPM_FP64 ? KID_SWE_F64 : KID_SWE_MIXED;
  int v = pick_variant(ctx, family, n_targets, -1);
  if (v < 0) {
    if (swe_few_sources(n_targets, n_src, precision)) return kSweF64Variants[0];
    v = swe_default_variant(family);
  }
  if (precision == LPM_FP64) {
    LPM_ARG_CHECK(v >= 0 && v < kNumSweF64, "variant out of range");
    return kSweF64Variants[v];
  }
  LPM_ARG_CHECK(v >= 0 && v < kNumSweMixed, "variant out of range");
  return kSweMixedVariants[v];
}

// Bytes of chunk sums of a one-problem launch.
size_t swe_part_bytes(const SweVariant& v, int64_t n_targets, int64_t n_src) {
  return sizeof(double) * static_cast<size_t>(n_targets) *
         static_cast<size_t>(
             v.wave ? kSweRows * swe_chunks(n_targets, n_src)
                    : kSweMfRows * swe_mf_chunks(n_targets, n_src));
}

// Far sums of whole blocks: one set per target.
double* swe_far_rows(lpm_ctx* ctx, int64_t n_targets) {
  return static_cast<double*>(ctx->swe_far.ensure(
      sizeof(double) * kSweMfRows * std::max<int64_t>(n_targets, 1)));
}

SweSeg to_seg(const SweTargets& t, int per_block) {
  SweSeg a{};
  a.x = t.base.x.base;
  a.es = t.base.x.es;
  a.cs = t.base.x.cs;
  a.n = t.base.n;
  a.index = t.base.index;
  a.d_n = t.base.d_n;
  a.self_rank = t.base.self_rank;
  a.self_identity = t.base.self_identity ? 1 : 0;
  a.nblocks = static_cast<int>((t.base.n + per_block - 1) / per_block);
  a.surf = t.surf;
  a.out_u = t.base.out.base;
  a.oes = t.base.out.es;
  a.ocs = t.base.out.cs;
  a.out_ddot = t.ddot;
  a.out_laps = t.laps;
  a.pstride = t.base.n;
  return a;
}

}  // namespace

int swe_variant_count(int family) {
  return family == KID_SWE_F64 ? kNumSweF64
                               : (family == KID_SWE_MIXED ? kNumSweMixed : 0);
}

const char* swe_variant_name(int family, int v) {
  if (v < 0 || v >= swe_variant_count(family)) return nullptr;
  return family == KID_SWE_F64 ? kSweF64Variants[v].name
                               : kSweMixedVariants[v].name;
}

int swe_default_variant(int family) {
  return family == KID_SWE_F64 ? kDefaultSweF64 : 0;
}

void swe_feature_workspace(lpm_ctx* ctx, int64_t n_src, int64_t n_targets,
                           int precision) {
  if (precision != LPM_MIXED) return;
  const SweVariant& v = swe_variant(ctx, precision, n_targets);
  if (!v.mf()) return;
  const int64_t ntile = (std::max<int64_t>(n_src, 1) + kSweTile - 1) / kSweTile;
  ctx->swe_feat.ensure(kSweMfTileBytes * ntile);
}

SweBounds swe_bounds(lpm_ctx* ctx, int precision, int64_t n_targets,
                     int64_t n_src) {
  const SweVariant& v = swe_variant(ctx, precision, n_targets, n_src);
  return v.wave ? kSweRunBounds : v.mf() ? kSweNoBounds : kSweTileBounds;
}

void swe_pack_workspace(lpm_ctx* ctx, int64_t n_src) {
  const int64_t ntile = (std::max<int64_t>(n_src, 1) + kSweTile - 1) / kSweTile;
  ctx->swe_packed.ensure(sizeof(SweSrc) * kSweTile * ntile);
  // bounding spheres of the tiles, then of the runs of 64 sources
  ctx->swe_bounds.ensure(sizeof(double4) * (1 + kSweTile / 64) * ntile);
}

void swe_sums_workspace(lpm_ctx* ctx, int64_t n_src, int64_t n_targets,
                        int precision, hipStream_t s) {
  swe_feature_workspace(ctx, n_src, n_targets, precision);
  const SweVariant& v = swe_variant(ctx, precision, n_targets);
  if (!v.wave && !v.mf()) return;
  const bool chunks = v.wave || swe_mf_chunks(n_targets, n_src) > 1;
  const double* part =
      chunks ? chunk_workspace(ctx, swe_part_bytes(v, n_targets, n_src), s)
             : nullptr;
  if (v.mf() && !part) swe_far_rows(ctx, n_targets);
}

SwePacked swe_pack_sources(lpm_ctx* ctx, CrdIn sx, const double* zeta,
                           const double* sigma, const double* area,
                           const double* surf, const RankMap& map,
                           SweBounds bounds, hipStream_t s) {
  SwePacked ps;
  const int64_t n = map.n;
  const int ntile =
      static_cast<int>((std::max<int64_t>(n, 1) + kSweTile - 1) / kSweTile);
  const int64_t cap = static_cast<int64_t>(ntile) * kSweTile;
  swe_pack_workspace(ctx, n);
  SweSrc* p = ctx->swe_packed.as<SweSrc>();
  double4* b = ctx->swe_bounds.as<double4>();
  double4* runs = bounds == kSweRunBounds ? b + ntile : nullptr;
  if (n > 0) {
    swe_pack_kernel<<<ntile, 256, 0, s>>>(sx.base, sx.es, sx.cs, zeta, sigma,
                                           area, surf, map.inv, map.d_count,
                                           cap, p, runs);
    LPM_HIP_CHECK(hipGetLastError());
    if (bounds == kSweTileBounds) {
      swe_tile_bounds_kernel<<<ntile, kSweTile, 0, s>>>(p, map.d_count, b);
      LPM_HIP_CHECK(hipGetLastError());
    }
  }
  ps.data = p;
  ps.bounds = runs ? b + ntile : b;
  ps.count = map.d_count;
  ps.capacity = n;
  return ps;
}

void launch_swe_sums(lpm_ctx* ctx, const SwePacked& src, SweTargets* segs,
                     int nseg, double eps, double pse_eps, int precision,
                     hipStream_t s) {
  LPM_ARG_CHECK(nseg >= 1 && nseg <= 2, "one or two target segments");
  SweTargets empty;
  const SweTargets& t0 = segs[0];
  const SweTargets& t1 = nseg > 1 ? segs[1] : empty;
  const int64_t nt = t0.base.n + t1.base.n;
  if (nt == 0) return;
  const SweVariant& v =
      swe_variant(ctx, precision, nt, nseg == 1 ? src.capacity : -1);
  constexpr int kBlock = 256;
  const int per = v.wave ? 64 : kBlock;
  SweSeg a0 = to_seg(t0, per), a1 = to_seg(t1, per);
  const int64_t grid = static_cast<int64_t>(a0.nblocks) + a1.nblocks;
  const int do_pse = pse_eps > 0 ? 1 : 0;
  const double inv_e2 = do_pse ? 1.0 / (pse_eps * pse_eps) : 0.0;
  const double cut2 = do_pse ? kPseCut * pse_eps * pse_eps : 0.0;
  // SphereFaceSums skips j == i only for the singular kernel (eps == 0)
  const int skip_self = eps == 0.0 ? 1 : 0;
  double pairs = static_cast<double>(t0.base.n + t1.base.n) * src.capacity;
  SweParams P{eps * eps, inv_e2, cut2, do_pse, skip_self};
  if (v.wave) {
    const int C = swe_chunks(nt, src.capacity);
    // one chunk, or no workspace (a caller's capture, no memory): whole blocks
    double* part =
        C > 1 ? chunk_workspace(ctx, swe_part_bytes(v, nt, src.capacity), s)
              : nullptr;
    a0.part = part;
    a1.part = part + (part ? kSweRows * static_cast<int64_t>(C) * a0.n : 0);
    TimedLaunch tl(ctx, KID_SWE_F64, s, pairs);
    hipLaunchKernelGGL(part ? swe_wave_kernel<true> : swe_wave_kernel<false>,
                       launch_grid(grid * (part ? C : 1), 64 * kSweWaves),
                       dim3(64 * kSweWaves), 0, s,
                       static_cast<const double*>(src.data), src.bounds,
                       src.count, a0, a1, P, C);
    LPM_HIP_CHECK(hipGetLastError());
    if (part) {
      swe_wave_reduce_kernel<<<static_cast<unsigned>((nt + 63) / 64), 64, 0,
                               s>>>(a0, a1, P, C);
      LPM_HIP_CHECK(hipGetLastError());
    }
    return;
  }
  if (v.mf()) {
    // the matrix-core records of every source tile
    const int64_t ntile =
        (std::max<int64_t>(src.capacity, 1) + kSweTile - 1) / kSweTile;
    P.mf = swe_mf_tiles(ctx->swe_feat.ensure(kSweMfTileBytes * ntile), ntile);
    swe_mf_pack_kernel<<<static_cast<int>(ntile), 256, 0, s>>>(
        static_cast<const SweSrc*>(src.data), src.count, P.mf);
    LPM_HIP_CHECK(hipGetLastError());
    P.C = swe_mf_chunks(nt, src.capacity);
    // one chunk, or no workspace (a caller's capture, no memory): whole blocks
    double* part =
        P.C > 1 ? chunk_workspace(ctx, swe_part_bytes(v, nt, src.capacity), s)
                : nullptr;
    P.rows = part ? P.C : 1;
    a0.part = part ? part : swe_far_rows(ctx, nt);
    a1.part = a0.part + kSweMfRows * static_cast<int64_t>(P.rows) * a0.n;
    TimedLaunch tl(ctx, KID_SWE_MIXED, s, pairs);
    hipLaunchKernelGGL(v.far, launch_grid(grid * P.rows, kBlock),
                       dim3(kBlock), 0, s, static_cast<const SweSrc*>(src.data),
                       src.bounds, src.count, a0, a1, P);
    LPM_HIP_CHECK(hipGetLastError());
    a0.nblocks = static_cast<int>((a0.n + 63) / 64);
    a1.nblocks = static_cast<int>((a1.n + 63) / 64);
    hipLaunchKernelGGL(v.near,
                       launch_grid(static_cast<int64_t>(a0.nblocks) + a1.nblocks,
                                   256),
                       dim3(256), 0, s,
                       static_cast<const SweSrc*>(src.data), src.bounds,
                       src.count, a0, a1, P);
    LPM_HIP_CHECK(hipGetLastError());
    return;
  }
  TimedLaunch tl(ctx, precision == LPM_FP64 ? KID_SWE_F64 : KID_SWE_MIXED, s,
                 pairs);
  hipLaunchKernelGGL(v.fn, dim3(static_cast<unsigned>(grid)), dim3(kBlock), 0, s,
                     static_cast<const SweSrc*>(src.data), src.bounds,
                     src.count, a0, a1, P);
  LPM_HIP_CHECK(hipGetLastError());
}

// Vertex slot order of the mixed sums: from the members' state positions
// (also for the stage evaluations of a step, whose positions are close).
const int32_t* swe_ens_vertex_order(lpm_ctx* ctx, const EnsembleDesc& d,
                                    const lpm_swe_fields& f, hipStream_t s) {
  return target_order(ctx, CrdIn{f.vert_x, f.vert_x_es, f.vert_x_cs},
                      d.n_verts, d.voff, d.n_members, s);
}

uint64_t swe_ensemble_prepare(lpm_ctx* ctx, const EnsembleDesc& d,
                              const lpm_swe_fields& f, int precision,
                              hipStream_t s) {
  const SweVariant& v = swe_variant(ctx, precision, d.n_verts + d.n_faces);
  const EnsLayout L = ensemble_plan(ctx, d, v.wave ? 64 : 256, v.chunks());
  const int64_t cap = std::max<int64_t>(d.total_padded_upper, kSweTile);
  ctx->swe_packed.ensure(sizeof(SweSrc) * cap);
  ctx->swe_bounds.ensure(sizeof(double4) * 5 * (cap / kSweTile));
  if (v.wave) chunk_workspace(ctx, sizeof(double) * kSweRows * L.parts, s);
  if (v.mf()) {
    ctx->swe_feat.ensure(kSweMfTileBytes * (cap / kSweTile));
    if (!chunk_workspace(ctx, sizeof(double) * kSweMfRows * L.parts, s))
      swe_far_rows(ctx, d.n_verts + d.n_faces);
  }
  if (precision == LPM_MIXED) {
    swe_ens_vertex_order(ctx, d, f, s);
  }
  return L.serial;
}

void swe_ensemble_sums(lpm_ctx* ctx, const EnsembleDesc& d,
                       const lpm_swe_fields& f, CrdIn vx, CrdIn fx,
                       const double* fzeta, const double* fsigma,
                       const double* farea, const RankMap& map, double eps,
                       double pse_eps, int precision, unsigned flags,
                       hipStream_t s) {
  constexpr int kBlock = 256;
  swe_ensemble_prepare(ctx, d, f, precision, s);
  const SweVariant& v = swe_variant(ctx, precision, d.n_verts + d.n_faces);
  const EnsLayout L =
      ensemble_layout(ctx, d, map, v.wave ? 64 : kBlock, s, v.chunks());
  SweSrc* src = ctx->swe_packed.as<SweSrc>();
  double4* bounds = ctx->swe_bounds.as<double4>();
  const dim3 grid2(static_cast<unsigned>((d.max_member_faces + 255) / 256),
                   static_cast<unsigned>(d.n_members));
  swe_ens_pack_kernel<<<grid2, 256, 0, s>>>(fx.base, fx.es, fx.cs, fzeta,
                                             fsigma, farea, f.face_surf,
                                             map.inv, L.mem, src,
                                             v.wave ? bounds : nullptr);
  LPM_HIP_CHECK(hipGetLastError());
  if (!v.wave && !v.mf())
    swe_ens_bounds_kernel<<<grid2, kSweTile, 0, s>>>(src, L.mem, bounds);
  LPM_HIP_CHECK(hipGetLastError());
  if (L.n_items == 0) return;

  SweEnsArgs A{};
  A.mem = L.mem;
  A.items = L.items;
  A.n_items = L.n_items;
  A.queue = L.queue;
  A.vert.x = vx.base;
  A.vert.es = vx.es;
  A.vert.cs = vx.cs;
  A.vert.surf = f.vert_surf;
  A.vert.out_u = f.vert_u;
  A.vert.oes = f.vert_u_es;
  A.vert.ocs = f.vert_u_cs;
  A.vert.out_ddot = f.vert_ddot;
  A.vert.out_laps = f.vert_laps;
  if (precision == LPM_MIXED) A.vert.index = swe_ens_vertex_order(ctx, d, f, s);
  A.face.x = fx.base;
  A.face.es = fx.es;
  A.face.cs = fx.cs;
  A.face.surf = f.face_surf;
  A.face.out_u = f.face_u;
  A.face.oes = f.face_u_es;
  A.face.ocs = f.face_u_cs;
  A.face.out_ddot = f.face_ddot;
  A.face.out_laps = f.face_laps;
  A.rank = map.rank;
  A.inv = map.inv;
  A.skip_masked = (flags & LPM_FLAG_SKIP_MASKED_TARGETS) ? 1 : 0;
  const int do_pse = pse_eps > 0 ? 1 : 0;
  A.P = SweParams{eps * eps, do_pse ? 1.0 / (pse_eps * pse_eps) : 0.0,
                  do_pse ? kPseCut * pse_eps * pse_eps : 0.0, do_pse,
                  eps == 0.0 ? 1 : 0};
  if (v.wave) {
    double* part =
        chunk_workspace(ctx, sizeof(double) * kSweRows * L.parts, s);
    SweEnsArgs B = A;
    if (part) {
      B.items = L.chunk_items;
      B.n_items = L.n_chunk_items;
    }
    TimedLaunch tl(ctx, KID_SWE_F64, s, L.pairs);
    hipLaunchKernelGGL(
        part ? swe_ens_wave_kernel<true> : swe_ens_wave_kernel<false>,
        launch_grid(B.n_items, 64 * kSweWaves), dim3(64 * kSweWaves), 0, s,
        reinterpret_cast<const double*>(src),
        static_cast<const double4*>(bounds), B, part);
    LPM_HIP_CHECK(hipGetLastError());
    if (part) {
      swe_ens_wave_reduce_kernel<<<launch_grid(L.n_items, 64), 64, 0, s>>>(A,
                                                                        part);
      LPM_HIP_CHECK(hipGetLastError());
    }
    return;
  }
  if (v.mf()) {
    const int64_t cap = std::max<int64_t>(d.total_padded_upper, kSweTile);
    A.P.mf = swe_mf_tiles(ctx->swe_feat.as<void>(), cap / kSweTile);
    swe_ens_mf_pack_kernel<<<grid2, 256, 0, s>>>(src, L.mem, A.P.mf);
    LPM_HIP_CHECK(hipGetLastError());
    double* part =
        chunk_workspace(ctx, sizeof(double) * kSweMfRows * L.parts, s);
    A.P.rows = part ? 0 : 1;  // 0: each member's chunks
    SweEnsArgs B = A;
    if (part) {
      B.items = L.chunk_items;
      B.n_items = L.n_chunk_items;
    } else {
      part = swe_far_rows(ctx, d.n_verts + d.n_faces);
    }
    TimedLaunch tl(ctx, KID_SWE_MIXED, s, L.pairs);
    hipLaunchKernelGGL(v.ens_far, launch_grid(B.n_items, kBlock), dim3(kBlock),
                       0, s, B, part);
    LPM_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(v.ens_near,
                       launch_grid(int64_t{4} * L.n_items, 256), dim3(256), 0, s,
                       static_cast<const SweSrc*>(src), A, part);
    LPM_HIP_CHECK(hipGetLastError());
    return;
  }
  const int grid = ensemble_grid(ctx, reinterpret_cast<const void*>(v.ens),
                                 kBlock, L.n_items);
  TimedLaunch tl(ctx, precision == LPM_FP64 ? KID_SWE_F64 : KID_SWE_MIXED, s,
                 L.pairs);
  hipLaunchKernelGGL(v.ens, dim3(grid), dim3(kBlock), 0, s,
                     static_cast<const SweSrc*>(src),
                     static_cast<const double4*>(bounds), A);
  LPM_HIP_CHECK(hipGetLastError());
}

}  // namespace lpm_amd
