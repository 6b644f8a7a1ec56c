// 2-D incompressible flow on the sphere: the fused velocity + stream
// function direct sum of Incompressible2DKernels<SphereGeometry>::kernel_vals
// (src/lpm_incompressible2d_kernels.hpp:35-47) and the Heun RK2 stepper of
// Incompressible2DRK2 (src/lpm_incompressible2d_rk2_impl.hpp:75-172).
//
// The sum shares the BVE prologue (mask scan, packed FP64 sources
// {y, s = -zeta A / 4 pi}) and target segments.  Per pair:
//   arg = 1 - x.y + eps^2,  S += (s / arg) y,  psi += s log(arg),
// and u = x cross S at the end (x cross y / (-4 pi arg) Gamma = x cross
// (s / arg) y).  The table-driven FP64 log (bve_device.hpp) is half of the
// pair cost.
//
// Mixed precision: 1 - x.y = |d|^2 / 2 on the sphere, so arg = |d|^2 / 2 +
// eps^2, with the distances of far tiles from the f16 matrix cores and of near
// ones in FP32 difference form on tile-relative offsets (bve_device.hpp), the
// native FP32 log, and FP32 partials per 256-source tile carried into FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <functional>
#include <sstream>

#include "bve_device.hpp"
#include "internal.hpp"

namespace lpm_amd {
namespace {

// FP64: a block of four waves owns 64 targets and one of C source chunks, as
// the wave-split velocity sums (bve_device.hpp): records {y, s, s y, 0} are
// scalar loads, four pairs share one reciprocal, and the log comes in two
// parts.  What bounds it: FP64 issue, 23 FP64 and 8 32-bit operations and a
// quarter reciprocal per pair (36 and a reciprocal before).

struct Ic2dSum {
  double S[3], K, R;  // sum (s / arg) y, s k, s (rest of the log)
};

// Quads [qa, qb); CHECK drops source self.
template <bool CHECK>
__device__ __forceinline__ void ic2d_quads(const double* __restrict__ rec,
                                           int qa, int qb, const double* x,
                                           double one_e, int self,
                                           const double2* ltab, Ic2dSum& T,
                                           uint32_t& top) {
#pragma unroll 1
  for (int q = qa; q < qb; ++q) {
    const double* p = rec + static_cast<int64_t>(q) * 32;
    double y[4][7];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 7; ++e) y[j][e] = p[8 * j + e];
    double d[4], w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // 1 - x.y + eps^2 as one FMA chain from 1 + eps^2
      d[j] = __builtin_fma(
          -x[2], y[j][2],
          __builtin_fma(-x[1], y[j][1], __builtin_fma(-x[0], y[j][0], one_e)));
      if (CHECK && 4 * q + j == self) d[j] = 1.0;  // log 1 = 0
      top = max(top, log_screen(d[j]));
    }
    const double pab = d[0] * d[1], pcd = d[2] * d[3];
    const double r = rcp_cubic(pab * pcd);
    const double rab = r * pcd, rcd = r * pab;
    w[0] = d[1] * rab;
    w[1] = d[0] * rab;
    w[2] = d[3] * rcd;
    w[3] = d[2] * rcd;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (CHECK && 4 * q + j == self) w[j] = 0.0;
#pragma unroll
      for (int a = 0; a < 3; ++a)
        T.S[a] = __builtin_fma(w[j], y[j][4 + a], T.S[a]);
      double k;
      const double v = log_part(d[j], ltab, k);
      T.K = __builtin_fma(y[j][3], k, T.K);
      T.R = __builtin_fma(y[j][3], v, T.R);
    }
  }
}

// The same, pair by pair with the library log and two Newton steps (zero,
// negative, infinite and NaN arguments: coincident points without smoothing).
__device__ __forceinline__ void ic2d_redo(const double* __restrict__ rec,
                                          int qa, int qb, const double* x,
                                          double one_e, int self, double* S,
                                          double& psi) {
  S[0] = S[1] = S[2] = psi = 0.0;
#pragma unroll 1
  for (int j = 4 * qa; j < 4 * qb; ++j) {
    const double* y = rec + static_cast<int64_t>(j) * 8;
    const double arg = __builtin_fma(
        -x[2], y[2],
        __builtin_fma(-x[1], y[1], __builtin_fma(-x[0], y[0], one_e)));
    const double w = j == self ? 0.0 : rcp_nr<2>(arg);
    const double v = y[3] * log(arg);
    psi += j == self ? 0.0 : v;
#pragma unroll
    for (int a = 0; a < 3; ++a) S[a] = __builtin_fma(w, y[4 + a], S[a]);
  }
}

// With partial sums, block b * C + k sums source chunk k of target block b into
// its four rows; without, block b adds every chunk in order.
__global__ __launch_bounds__(256) void ic2d_f64_kernel(
    const double* __restrict__ rec, const double2* __restrict__ table,
    const int32_t* __restrict__ count, SegArgs s0, SegArgs s1, double eps2,
    int skip_self, int C) {
  __shared__ double2 ltab[kLogTable];
  __shared__ double red[4][4][64];
  const bool split = s0.part != nullptr;
  const int b = split ? flat_block() / C : flat_block();
  const int c0 = split ? flat_block() % C : 0;
  const bool first = b < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? b : b - s0.nblocks;
  const int nq = (*count + 3) / 4;
  const int64_t n_live = sg.d_n ? *sg.d_n : sg.n;
  const int64_t slot0 = static_cast<int64_t>(blk) * 64;
  if (slot0 >= n_live) return;
  load_log_table(table, ltab);
  const double one_e = 1.0 + eps2;
  // smoothing too wide for a shared reciprocal: every tile pair by pair
  const uint32_t screen = eps2 > kMaxShared ? 0u : kLogScreen;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t c = slot0 + lane;
  double x[3];
  int self;
  const int64_t i = lane_target(sg, c, c < n_live, x, &self);
  if (!skip_self) self = -1;
  int lo, hi;
  wave_self_range<1>(&self, &lo, &hi);
  __syncthreads();
  double tot[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
  for (int k = c0; k < (split ? c0 + 1 : C); ++k) {
    int q0, q1;
    wave_range(nq, k, C, w, &q0, &q1);
    double S[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int q = q0; q < q1; q += kWaveTile) {
      const int e = min(q + kWaveTile, q1);
      Ic2dSum T = {{0.0, 0.0, 0.0}, 0.0, 0.0};
      uint32_t top = 0;
      if (lo < 4 * e && hi >= 4 * q)
        ic2d_quads<true>(rec, q, e, x, one_e, self, ltab, T, top);
      else
        ic2d_quads<false>(rec, q, e, x, one_e, self, ltab, T, top);
      double V[4] = {T.S[0], T.S[1], T.S[2], __builtin_fma(T.K, kLn2, T.R)};
      if (__ballot(top >= screen)) {
        double D[3], psi;
        ic2d_redo(rec, q, e, x, one_e, self, D, psi);
        if (top >= screen) {
          V[0] = D[0];
          V[1] = D[1];
          V[2] = D[2];
          V[3] = psi;
        }
      }
#pragma unroll
      for (int a = 0; a < 4; ++a) S[a] += V[a];
    }
    if (k > c0) __syncthreads();  // the previous chunk's sums are read
#pragma unroll
    for (int a = 0; a < 4; ++a) red[w][a][lane] = S[a];
    __syncthreads();
    if (w == 0)
#pragma unroll
      for (int a = 0; a < 4; ++a)
        tot[a] += ((red[0][a][lane] + red[1][a][lane]) + red[2][a][lane]) +
                  red[3][a][lane];
  }
  if (w != 0 || c >= n_live) return;
  if (split) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
      sg.part[(4 * static_cast<int64_t>(c0) + a) * sg.pstride + c] = tot[a];
  } else if (!(sg.skip && sg.skip[i])) {
    if (sg.out) cross_to(x, tot, sg.out + i * sg.oes, sg.ocs);
    if (sg.out_scalar) sg.out_scalar[i] = tot[3];
  }
}

// Mixed: the chunked matrix-core velocity sums (bve_device.hpp) with the
// logarithm of each distance next to its reciprocal.  What bounds it: per 64
// pairs a quarter-rate logarithm (8.7 SIMD-cycles), a multiply and an FMA for
// psi on top of the velocity's 2.25 multiplies and quarter reciprocal, beside
// 8 cycles of weight products on the matrix cores.  Level 6 (1.0e10 pairs):
// 2.9 ms, against 4.2 for the vector form with a reciprocal and a distance in
// difference form per pair.
template <bool EPS>
__global__ __launch_bounds__(256, 4) void ic2d_mixed_kernel(
    Mfma16Src src, const int32_t* __restrict__ count, SegArgs s0, SegArgs s1,
    float e2x2, float e2, int skip_self, int C) {
  __shared__ uint4 la[2 * kPackTile];
  __shared__ float4 lt[kPackTile];
  const bool split = s0.part != nullptr;
  const int b = split ? flat_block() / C : flat_block();
  const int c0 = split ? flat_block() % C : 0;
  const bool first = b < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? b : b - s0.nblocks;
  const int64_t n_live = sg.d_n ? *sg.d_n : sg.n;
  const int64_t c = static_cast<int64_t>(blk) * 256 + threadIdx.x;
  if (static_cast<int64_t>(blk) * 256 >= n_live) return;
  double x[3];
  int self;
  const int64_t i = lane_target(sg, c, c < n_live, x, &self);
  if (!skip_self) self = -1;
  const int64_t ntile = (*count + kPackTile - 1) / kPackTile;
  double tot[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
  for (int k = c0; k < (split ? c0 + 1 : C); ++k) {
    double T[4];
    mfma16_tiles<EPS, 2, 4, true>(
        src, static_cast<int>(ntile * k / C) * kPackTile,
        static_cast<int>(ntile * (k + 1) / C) * kPackTile, x, self, e2x2, la, lt, T, e2);
#pragma unroll
    for (int a = 0; a < 4; ++a) tot[a] += T[a];
  }
  if (c >= n_live) return;
  if (split) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
      sg.part[(4 * static_cast<int64_t>(c0) + a) * sg.pstride + c] = tot[a];
  } else if (!(sg.skip && sg.skip[i])) {
    if (sg.out) cross_to(x, tot, sg.out + i * sg.oes, sg.ocs);
    if (sg.out_scalar) sg.out_scalar[i] = tot[3];
  }
}

// u = x cross (sum of the ks chunk partials of S, in chunk order) and psi
// = the sum of the chunk partials of psi, at every live slot.
__global__ __launch_bounds__(256) void ic2d_split_reduce_kernel(SegArgs s0,
                                                                SegArgs s1,
                                                                int ks) {
  const int64_t g = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const bool first = g < s0.n;
  const SegArgs& sg = pick(s0, s1, first);
  const int64_t c = first ? g : g - s0.n;
  const int64_t n_live = sg.d_n ? *sg.d_n : sg.n;
  if (c >= n_live) return;
  const int64_t i = sg.index ? sg.index[c] : sg.slot_base + c;
  if (sg.skip && sg.skip[i]) return;
  const double* q = sg.part + c;
  double S[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
  for (int k = 0; k < ks; ++k)
#pragma unroll
    for (int a = 0; a < 4; ++a)
      S[a] += q[(4 * static_cast<int64_t>(k) + a) * sg.pstride];
  if (sg.out) {
    const double* p = sg.x + i * sg.es;
    const double x[3] = {p[0], p[sg.cs], p[2 * sg.cs]};
    cross_to(x, S, sg.out + i * sg.oes, sg.ocs);
  }
  if (sg.out_scalar) sg.out_scalar[i] = S[3];
}

// Stage storage of one particle kind (SoA, leading dimension n): x1 (3n),
// z1 (n), xw (3n), zw (n).
struct Ic2dStage {
  double* x1;
  double* z1;
  double* xw;
  double* zw;
  int64_t n;
};

Ic2dStage carve(DevBuf& buf, int64_t n) {
  const int64_t nn = std::max<int64_t>(n, 1);
  double* p = static_cast<double*>(buf.ensure(sizeof(double) * 8 * nn));
  return Ic2dStage{p, p + 3 * nn, p + 4 * nn, p + 7 * nn, n};
}

struct Ic2dArgs {
  double* x;  // state positions (strided)
  int64_t xes, xcs;
  double* zeta;
  const double* u;  // velocity (strided)
  int64_t ues, ucs;
  const uint8_t* skip;
  Ic2dStage st;
  double dt, Omega;
  int renorm;
};

__device__ __forceinline__ void project(double* v) {
  const double r = 1.0 / sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  v[0] *= r;
  v[1] *= r;
  v[2] *= r;
}

// Both kernels: blocks [0, nbv) take the vertices, the rest the faces.
// Stage 1: x1 = dt u, z1 = -2 Omega u_z (a rate), xw = x + dt u,
// zw = zeta + dt z1 (KokkosBlas::scal / update and
// Incompressible2DTendencies of the reference's first stage).
__global__ __launch_bounds__(256) void ic2d_stage1_kernel(Ic2dArgs V, Ic2dArgs F,
                                                          int nbv) {
  const bool vert = static_cast<int>(blockIdx.x) < nbv;
  const Ic2dArgs& A = vert ? V : F;
  const int64_t i =
      static_cast<int64_t>(blockIdx.x - (vert ? 0 : nbv)) * 256 + threadIdx.x;
  const int64_t n = A.st.n;
  if (i >= n) return;
  if (A.skip && A.skip[i]) return;
  const double* ui = A.u + i * A.ues;
  const double* xi = A.x + i * A.xes;
  const double u[3] = {ui[0], ui[A.ucs], ui[2 * A.ucs]};
  double w[3];
  for (int k = 0; k < 3; ++k) {
    A.st.x1[i + k * n] = A.dt * u[k];
    w[k] = xi[k * A.xcs] + A.dt * u[k];
  }
  if (A.renorm) project(w);
  for (int k = 0; k < 3; ++k) A.st.xw[i + k * n] = w[k];
  const double z1 = -2.0 * A.Omega * u[2];
  A.st.z1[i] = z1;
  A.st.zw[i] = A.zeta[i] + A.dt * z1;
}

// Stage 2 and the Heun update: z2 = -2 Omega u2_z;
// zeta += dt/2 z1 + dt/2 z2, x += x1/2 + (dt u2)/2.
__global__ __launch_bounds__(256) void ic2d_update_kernel(Ic2dArgs V, Ic2dArgs F,
                                                          int nbv) {
  const bool vert = static_cast<int>(blockIdx.x) < nbv;
  const Ic2dArgs& A = vert ? V : F;
  const int64_t i =
      static_cast<int64_t>(blockIdx.x - (vert ? 0 : nbv)) * 256 + threadIdx.x;
  const int64_t n = A.st.n;
  if (i >= n) return;
  if (A.skip && A.skip[i]) return;
  const double* ui = A.u + i * A.ues;
  double* xi = A.x + i * A.xes;
  const double u[3] = {ui[0], ui[A.ucs], ui[2 * A.ucs]};
  const double z2 = -2.0 * A.Omega * u[2];
  A.zeta[i] += 0.5 * A.dt * A.st.z1[i] + 0.5 * A.dt * z2;
  double v[3];
  for (int k = 0; k < 3; ++k)
    v[k] = xi[k * A.xcs] + (0.5 * A.st.x1[i + k * n] + 0.5 * (A.dt * u[k]));
  if (A.renorm) project(v);
  for (int k = 0; k < 3; ++k) xi[k * A.xcs] = v[k];
}

inline int nblk(int64_t n) { return static_cast<int>((n + 255) / 256); }

// Source layouts of the sums: records {y, s, s y, 0} in FP64, the f16-split
// matrix-core records in mixed precision.
unsigned ic2d_layouts(int precision) {
  return precision == LPM_MIXED ? kLayoutMfma16 | kLayoutLog : kLayoutRec;
}

// Source chunks per target block.
int ic2d_chunks(int precision, int64_t n_targets, int64_t nsrc_upper) {
  return precision == LPM_MIXED ? mixed_chunks(n_targets, nsrc_upper)
                                : log_chunks(n_targets, nsrc_upper);
}

size_t ic2d_split_bytes(int ks, int64_t n_targets) {
  return ks > 1 ? sizeof(double) * 4 * static_cast<size_t>(ks) *
                      static_cast<size_t>(std::max<int64_t>(n_targets, 1))
                : 0;
}

void launch_ic2d(lpm_ctx* ctx, const PackedSources& src, TargetSeg* segs,
                 int nseg, double eps, bool collocated_skip, int precision,
                 hipStream_t s) {
  TargetSeg empty;
  const TargetSeg& t0 = segs[0];
  const TargetSeg& t1 = nseg > 1 ? segs[1] : empty;
  if (t0.n + t1.n == 0) return;
  const int per = precision == LPM_MIXED ? 256 : 64;  // targets per block
  auto to_args = [per](const TargetSeg& t) {
    SegArgs a{};
    a.x = t.x.base;
    a.es = t.x.es;
    a.cs = t.x.cs;
    a.n = t.n;
    a.index = t.index;
    a.d_n = t.d_n;
    a.self_rank = t.self_rank;
    a.self_identity = t.self_identity ? 1 : 0;
    a.nblocks = static_cast<int>((t.n + per - 1) / per);
    a.skip = t.skip;
    a.out = t.out.base;
    a.oes = t.out.es;
    a.ocs = t.out.cs;
    a.out_scalar = t.out_scalar;
    a.pstride = t.n;
    return a;
  };
  SegArgs a0 = to_args(t0), a1 = to_args(t1);
  const int64_t blocks = static_cast<int64_t>(a0.nblocks) + a1.nblocks;
  const int ks = ic2d_chunks(precision, t0.n + t1.n, src.capacity);
  // no workspace (a caller's capture, no memory): whole blocks, chunk by chunk
  double* part =
      ks > 1 ? chunk_workspace(ctx, ic2d_split_bytes(ks, t0.n + t1.n), s)
             : nullptr;
  if (part) {
    a0.part = part;
    a1.part = part + 4 * static_cast<int64_t>(ks) * t0.n;
  }
  const double pairs = static_cast<double>(t0.n + t1.n) * src.capacity;
  TimedLaunch tl(ctx, KID_IC2D, s, pairs);
  const dim3 grid = launch_grid(blocks * (part ? ks : 1), 256);
  if (precision == LPM_MIXED) {
    LPM_ARG_CHECK(src.mf_a && src.mf_g, "matrix-core layout not packed");
    Mfma16Src m{src.mf_y, src.mf_s,  src.mf_a, src.mf_t32,
                src.mf_c, src.mf_is, src.mf_g};
    hipLaunchKernelGGL(eps > 0 ? ic2d_mixed_kernel<true>
                               : ic2d_mixed_kernel<false>,
                       grid, dim3(256), 0, s, m, src.count, a0, a1,
                       static_cast<float>(2.0 * eps * eps),
                       static_cast<float>(eps * eps), collocated_skip ? 1 : 0,
                       ks);
  } else {
    LPM_ARG_CHECK(src.rec, "records not packed");
    hipLaunchKernelGGL(ic2d_f64_kernel, grid, dim3(256), 0, s, src.rec,
                       ctx->log_table.as<double2>(), src.count, a0, a1,
                       eps * eps, collocated_skip ? 1 : 0, ks);
  }
  LPM_HIP_CHECK(hipGetLastError());
  if (part) {
    const int64_t nt = t0.n + t1.n;
    hipLaunchKernelGGL(ic2d_split_reduce_kernel,
                       dim3(static_cast<unsigned>((nt + 255) / 256)),
                       dim3(256), 0, s, a0, a1, ks);
    LPM_HIP_CHECK(hipGetLastError());
  }
}

// Sums of the fields at positions (vx, fx) with face vorticity fzeta.
void ic2d_eval(lpm_ctx* ctx, const lpm_ic2d_fields& f, CrdIn vx, CrdIn fx,
               const double* fzeta, const RankMap& map, double eps,
               int precision, unsigned flags, hipStream_t s) {
  PackedSources ps = pack_sources(ctx, ic2d_layouts(precision), fx, fzeta,
                                  f.face_area, map, precision, s);
  TargetSeg segs[2];
  segs[0].x = vx;
  segs[0].n = f.n_verts;
  segs[0].out = CrdOut{f.vert_u, f.vert_u_es, f.vert_u_cs};
  segs[0].out_scalar = f.vert_psi;
  segs[1] = face_targets(fx, map, f.face_mask,
                         (flags & LPM_FLAG_SKIP_MASKED_TARGETS) != 0,
                         CrdOut{f.face_u, f.face_u_es, f.face_u_cs},
                         f.face_psi);
  // the self-exclusion of segment 1 applies only when eps == 0
  launch_ic2d(ctx, ps, segs, 2, eps, eps == 0.0, precision, s);
}

void validate(const lpm_ic2d_fields* f) {
  LPM_ARG_CHECK(f, "null fields");
  LPM_ARG_CHECK(f->n_verts >= 0 && f->n_faces > 0, "bad sizes");
  if (f->n_verts > 0)
    LPM_ARG_CHECK(f->vert_x && f->vert_zeta && f->vert_u && f->vert_x_es > 0 &&
                      f->vert_x_cs > 0 && f->vert_u_es > 0 && f->vert_u_cs > 0,
                  "vertex fields incomplete");
  LPM_ARG_CHECK(f->face_x && f->face_zeta && f->face_u && f->face_area &&
                    f->face_x_es > 0 && f->face_x_cs > 0 && f->face_u_es > 0 &&
                    f->face_u_cs > 0,
                "face fields incomplete");
}

void issue_rk2(lpm_ctx* ctx, const lpm_ic2d_fields& f, double dt, double Omega,
               double eps, int precision, unsigned flags, Ic2dStage& V,
               Ic2dStage& F, hipStream_t s) {
  const RankMap map = build_rank(ctx, f.face_mask, f.n_faces, s);
  const uint8_t* fskip =
      (flags & LPM_FLAG_SKIP_MASKED_TARGETS) ? f.face_mask : nullptr;
  const int renorm = (flags & LPM_RK4_RENORMALIZE) ? 1 : 0;
  auto args = [&](bool face) {
    Ic2dArgs a{};
    a.x = face ? f.face_x : f.vert_x;
    a.xes = face ? f.face_x_es : f.vert_x_es;
    a.xcs = face ? f.face_x_cs : f.vert_x_cs;
    a.zeta = face ? f.face_zeta : f.vert_zeta;
    a.u = face ? f.face_u : f.vert_u;
    a.ues = face ? f.face_u_es : f.vert_u_es;
    a.ucs = face ? f.face_u_cs : f.vert_u_cs;
    a.skip = face ? fskip : nullptr;
    a.st = face ? F : V;
    a.dt = dt;
    a.Omega = Omega;
    a.renorm = renorm;
    return a;
  };
  const int nbv = nblk(f.n_verts), nb = nbv + nblk(f.n_faces);
  ic2d_stage1_kernel<<<nb, 256, 0, s>>>(args(false), args(true), nbv);
  LPM_HIP_CHECK(hipGetLastError());
  ic2d_eval(ctx, f, CrdIn{V.xw, 1, V.n}, CrdIn{F.xw, 1, F.n}, F.zw, map, eps,
            precision, flags, s);
  ic2d_update_kernel<<<nb, 256, 0, s>>>(args(false), args(true), nbv);
  LPM_HIP_CHECK(hipGetLastError());
  ic2d_eval(ctx, f, CrdIn{f.vert_x, f.vert_x_es, f.vert_x_cs},
            CrdIn{f.face_x, f.face_x_es, f.face_x_cs}, f.face_zeta, map, eps,
            precision, flags, s);
}

std::string ic2d_key(const lpm_ic2d_fields& f, double dt, double Omega,
                     double eps, int precision, unsigned flags,
                     hipStream_t s) {
  std::ostringstream k;
  k << "ic2d|" << f.n_verts << '|' << f.vert_x << '|' << f.vert_x_es << '|'
    << f.vert_x_cs << '|' << f.vert_zeta << '|' << f.vert_u << '|'
    << f.vert_u_es << '|' << f.vert_u_cs << '|' << f.vert_psi << '|'
    << f.n_faces << '|' << f.face_x << '|' << f.face_x_es << '|'
    << f.face_x_cs << '|' << f.face_zeta << '|' << f.face_u << '|'
    << f.face_u_es << '|' << f.face_u_cs << '|' << f.face_psi << '|'
    << f.face_area << '|' << static_cast<const void*>(f.face_mask) << '|';
  k.precision(17);
  k << dt << '|' << Omega << '|' << eps << '|' << precision << '|' << flags
    << '|' << s;
  return k.str();
}

template <typename F>
int guarded(lpm_ctx* ctx, F&& fn) {
  try {
    fn();
    return LPM_OK;
  } catch (const Error& e) {
    set_error(ctx, e.what());
    return e.code;
  } catch (const std::exception& e) {
    set_error(ctx, e.what());
    return LPM_ERR_INTERNAL;
  }
}

}  // namespace
}  // namespace lpm_amd

using namespace lpm_amd;

extern "C" {

int lpm_ic2d_sums(lpm_ctx* ctx, const double* tgt_x, int64_t tgt_es,
                  int64_t tgt_cs, int64_t n_tgt, const double* src_x,
                  int64_t src_es, int64_t src_cs, const double* src_zeta,
                  const double* src_area, const uint8_t* src_mask,
                  int64_t n_src, int collocated, double eps, int precision,
                  unsigned flags, double* out_u, int64_t out_es,
                  int64_t out_cs, double* out_psi, void* stream) {
  return guarded(ctx, [&] {
    LPM_ARG_CHECK(ctx, "null context");
    LPM_ARG_CHECK(n_tgt >= 0 && n_src >= 0, "negative size");
    LPM_ARG_CHECK(precision == LPM_FP64 || precision == LPM_MIXED,
                  "unknown precision");
    LPM_ARG_CHECK(eps >= 0 && std::isfinite(eps), "eps must be >= 0");
    if (n_tgt > 0) {
      LPM_ARG_CHECK(tgt_x && tgt_es > 0 && tgt_cs > 0, "bad tgt_x");
      LPM_ARG_CHECK(!out_u || (out_es > 0 && out_cs > 0), "bad out_u strides");
    }
    if (n_src > 0) {
      LPM_ARG_CHECK(src_x && src_es > 0 && src_cs > 0, "bad src_x");
      LPM_ARG_CHECK(src_zeta && src_area, "src_zeta/src_area are NULL");
    }
    if (collocated)
      LPM_ARG_CHECK(n_tgt == n_src,
                    "collocated: targets must be the sources (n_tgt == n_src)");
    LPM_HIP_CHECK(hipSetDevice(ctx->device));
    hipStream_t s = as_stream(stream);
    order_stream(ctx, s);
    const RankMap map = build_rank(ctx, src_mask, n_src, s);
    PackedSources ps =
        pack_sources(ctx, ic2d_layouts(precision),
                     CrdIn{src_x, src_es, src_cs}, src_zeta, src_area, map,
                     precision, s);
    TargetSeg t;
    if (collocated) {
      t = face_targets(CrdIn{tgt_x, tgt_es, tgt_cs}, map, src_mask,
                       (flags & LPM_FLAG_SKIP_MASKED_TARGETS) != 0,
                       CrdOut{out_u, out_es, out_cs}, out_psi);
    } else {
      t.x = CrdIn{tgt_x, tgt_es, tgt_cs};
      t.n = n_tgt;
      t.out = CrdOut{out_u, out_es, out_cs};
      t.out_scalar = out_psi;
    }
    launch_ic2d(ctx, ps, &t, 1, eps, collocated && eps == 0.0, precision, s);
    if ((flags & LPM_FLAG_CHECK_FINITE) && out_u)
      check_finite(ctx, out_u, n_tgt, out_es, out_cs, 3, s);
  });
}

int lpm_bve_solve(lpm_ctx* ctx, const double* tgt_x, int64_t tgt_es,
                  int64_t tgt_cs, int64_t n_tgt, const double* src_x,
                  int64_t src_es, int64_t src_cs, const double* src_zeta,
                  const double* src_area, const uint8_t* src_mask,
                  int64_t n_src, int collocated, int precision, unsigned flags,
                  double* out_u, int64_t out_es, int64_t out_cs,
                  double* out_psi, void* stream) {
  // BVEVertexSolve / BVEFaceSolve are the kernel_vals sums without
  // smoothing: one fused pass gives both of their reductions
  return lpm_ic2d_sums(ctx, tgt_x, tgt_es, tgt_cs, n_tgt, src_x, src_es,
                       src_cs, src_zeta, src_area, src_mask, n_src, collocated,
                       0.0, precision, flags, out_u, out_es, out_cs, out_psi,
                       stream);
}

int lpm_ic2d_init_direct_sums(lpm_ctx* ctx, const lpm_ic2d_fields* f,
                              double eps, int precision, unsigned flags,
                              void* stream) {
  return guarded(ctx, [&] {
    LPM_ARG_CHECK(ctx, "null context");
    validate(f);
    LPM_ARG_CHECK(precision == LPM_FP64 || precision == LPM_MIXED,
                  "unknown precision");
    LPM_ARG_CHECK(eps >= 0 && std::isfinite(eps), "eps must be >= 0");
    LPM_HIP_CHECK(hipSetDevice(ctx->device));
    hipStream_t s = as_stream(stream);
    order_stream(ctx, s);
    const RankMap map = build_rank(ctx, f->face_mask, f->n_faces, s);
    ic2d_eval(ctx, *f, CrdIn{f->vert_x, f->vert_x_es, f->vert_x_cs},
              CrdIn{f->face_x, f->face_x_es, f->face_x_cs}, f->face_zeta, map,
              eps, precision, flags, s);
  });
}

int lpm_ic2d_rk2_step(lpm_ctx* ctx, const lpm_ic2d_fields* f, double dt,
                      double Omega, double eps, int precision, unsigned flags,
                      void* stream) {
  return guarded(ctx, [&] {
    LPM_ARG_CHECK(ctx, "null context");
    validate(f);
    LPM_ARG_CHECK(precision == LPM_FP64 || precision == LPM_MIXED,
                  "unknown precision");
    LPM_ARG_CHECK(std::isfinite(dt) && std::isfinite(Omega),
                  "dt and Omega must be finite");
    LPM_ARG_CHECK(eps >= 0 && std::isfinite(eps), "eps must be >= 0");
    LPM_HIP_CHECK(hipSetDevice(ctx->device));
    hipStream_t s = as_stream(stream);
    order_stream(ctx, s);
    Ic2dStage V = carve(ctx->ic2d_v, f->n_verts);
    Ic2dStage F = carve(ctx->ic2d_f, f->n_faces);
    run_maybe_graph(
        ctx, (flags & LPM_RK4_USE_GRAPH) != 0, s,
        [&]() {
          rank_workspace(ctx, f->face_mask, f->n_faces);
          pack_workspace(ctx, f->n_faces, precision);
          // the split workspace of the two evaluations, before any capture
          const int ks =
              ic2d_chunks(precision, f->n_verts + f->n_faces, f->n_faces);
          if (ks > 1)
            chunk_workspace(ctx, ic2d_split_bytes(ks, f->n_verts + f->n_faces),
                            s);
          return ic2d_key(*f, dt, Omega, eps, precision, flags, s);
        },
        [&]() {
          issue_rk2(ctx, *f, dt, Omega, eps, precision, flags, V, F, s);
        });
    if (flags & LPM_FLAG_CHECK_FINITE) {
      check_finite(ctx, f->vert_u, f->n_verts, f->vert_u_es, f->vert_u_cs, 3, s);
      check_finite(ctx, f->face_u, f->n_faces, f->face_u_es, f->face_u_cs, 3, s);
    }
  });
}

}  // extern "C"
