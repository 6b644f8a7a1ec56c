// BVE ensembles: every member's velocity from one launch (and one that adds the
// chunk sums).  The member layout and work plan come from ensemble.hip; a work
// item runs the same block loop (bve_device.hpp) on the same target slots and source tiles
// as a one-member launch, so results agree bit for bit with
// lpm_bve_init_velocity on each member alone.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bve_device.hpp"
#include "internal.hpp"

namespace lpm_amd {
namespace {

struct EnsArgs {
  const EnsMember* mem;
  const int4* items;  // {member, segment (0 vertices, 1 faces), block, 0}
  int n_items;
  int32_t* queue;
  const double* vx;
  int64_t vxes, vxcs;
  double* vu;
  int64_t vues, vucs;
  const double* fx;
  int64_t fxes, fxcs;
  double* fu;
  int64_t fues, fucs;
  const int32_t* rank;  // compacted rank per face (nullptr: no mask)
  const int32_t* inv;   // face per compacted rank (nullptr: no mask)
  int skip_masked;
  const int32_t* vorder;  // vertex slot -> vertex (nullptr: identity)
};

// grid (ceil(max member faces / 256), n_members): packed slot P_m + c holds
// member m's c-th undivided face, or a zero source for the tile padding.
__global__ __launch_bounds__(256) void ens_pack_f64_kernel(
    const double* __restrict__ sx, int64_t es, int64_t cs,
    const double* __restrict__ zeta, const double* __restrict__ area,
    const int32_t* __restrict__ inv, const EnsMember* __restrict__ mem,
    double4* __restrict__ out, double4* __restrict__ out_sy) {
  const EnsMember M = mem[blockIdx.y];
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int padded = (M.cnt + kPackTile - 1) / kPackTile * kPackTile;
  if (c >= padded) return;
  double4 v = make_double4(0.0, 0.0, 0.0, 0.0);
  if (c < M.cnt) {
    const int64_t r = static_cast<int64_t>(M.R) + c;
    const int64_t i = inv ? inv[r] : r;
    const double* p = sx + i * es;
    v = make_double4(p[0], p[cs], p[2 * cs], -zeta[i] * area[i] * kInv4Pi);
  }
  out[M.P + c] = v;
  // {s y, 0} for the kernels that take the weight from it
  if (out_sy) out_sy[M.P + c] = make_double4(v.w * v.x, v.w * v.y, v.w * v.z, 0.0);
}

// Quad records of member m's undivided faces from packed slot P_m on, zero
// records up to a multiple of four; grid as ens_pack_f64_kernel.
__global__ __launch_bounds__(256) void ens_pack_quad_kernel(
    const double* __restrict__ sx, int64_t es, int64_t cs,
    const double* __restrict__ zeta, const double* __restrict__ area,
    const int32_t* __restrict__ inv, const EnsMember* __restrict__ mem,
    double* __restrict__ quad) {
  const EnsMember M = mem[blockIdx.y];
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= (M.cnt + 3) / 4 * 4) return;
  double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (c < M.cnt) {
    const int64_t r = static_cast<int64_t>(M.R) + c;
    const int64_t i = inv ? inv[r] : r;
    const double* p = sx + i * es;
    const double sv = -zeta[i] * area[i] * kInv4Pi;
    for (int a = 0; a < 3; ++a) {
      v[a] = p[a * cs];
      v[3 + a] = sv * v[a];
    }
  }
  double2* o = reinterpret_cast<double2*>(
      quad + (static_cast<int64_t>(M.P) + c) * 6);
  for (int a = 0; a < 3; ++a) o[a] = make_double2(v[2 * a], v[2 * a + 1]);
}

// The matrix-core records of member m's tiles (from packed tile P_m / 256 on);
// grid as ens_pack_f64_kernel, one block per tile.
__global__ __launch_bounds__(kPackTile) void ens_pack_mfma16_kernel(
    const double* __restrict__ sx, int64_t es, int64_t cs,
    const double* __restrict__ zeta, const double* __restrict__ area,
    const int32_t* __restrict__ inv, const EnsMember* __restrict__ mem,
    Mfma16Out o) {
  const EnsMember M = mem[blockIdx.y];
  const int c = blockIdx.x * kPackTile + threadIdx.x;
  if (static_cast<int>(blockIdx.x) * kPackTile >= M.cnt) return;
  double4 y = make_double4(0.0, 0.0, 0.0, 0.0);
  const bool real =
      c < M.cnt && load_source(sx, es, cs, zeta, area, inv,
                               static_cast<int64_t>(M.R) + c, &y);
  mfma16_pack_tile(y, real, M.P / kPackTile + blockIdx.x, o);
}

// Targets of work item segment `seg` of member M, as a SegArgs whose self
// indices count from the member's first packed source.
__device__ __forceinline__ SegArgs ens_segment(const EnsArgs& A,
                                               const EnsMember& M, int seg) {
  SegArgs sg{};
  if (seg == 0) {
    sg.x = A.vx;
    sg.es = A.vxes;
    sg.cs = A.vxcs;
    sg.n = M.nv;
    sg.slot_base = M.v0;
    if (A.vorder) sg.index = A.vorder + M.v0;
    sg.out = A.vu;
    sg.oes = A.vues;
    sg.ocs = A.vucs;
    return sg;
  }
  sg.x = A.fx;
  sg.es = A.fxes;
  sg.cs = A.fxcs;
  sg.out = A.fu;
  sg.oes = A.fues;
  sg.ocs = A.fucs;
  if (A.skip_masked && A.inv) {
    // compacted targets: slot c is the member's c-th undivided face, which
    // is also its c-th packed source
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

// Takes the next work item for the block; every block leaves the loop when
// the queue passes n_items.
__device__ __forceinline__ int ens_next(const EnsArgs& A, int* slot) {
  if (threadIdx.x == 0) *slot = atomicAdd(A.queue, 1);
  __syncthreads();
  const int it = *slot;
  __syncthreads();
  return it;
}

template <int BLOCK, int TPL, int NR, bool PAIR, bool FUSE = false,
          bool QUAD = false, bool SY = false>
__global__ __launch_bounds__(BLOCK) void ens_f64_kernel(
    const double4* __restrict__ src, const double4* __restrict__ src_sy,
    EnsArgs A) {
  constexpr int TILE = 256;
  __shared__ double4 tile[TILE];
  __shared__ double4 tile_sy[SY ? TILE : 1];
  __shared__ int slot;
  for (;;) {
    const int it = ens_next(A, &slot);
    if (it >= A.n_items) break;
    const int4 w = A.items[it];
    const EnsMember M = A.mem[w.x];
    const SegArgs sg = ens_segment(A, M, w.y);
    f64_block<BLOCK, TPL, TILE, false, NR, PAIR, FUSE, QUAD, SY>(
        src + M.P, SY ? src_sy + M.P : nullptr, M.cnt, sg, w.z, 0.0, tile,
        tile_sy);
  }
}

// Chunk partials of segment `seg` of member M: 3 C rows of its targets.
__device__ __forceinline__ void ens_parts(SegArgs& sg, const EnsMember& M,
                                          int seg, double* part) {
  const int64_t n = seg == 0 ? M.nv : M.nf;
  sg.part = part + 3 * (M.part0 + (seg == 0 ? 0 : M.C * M.nv));
  sg.pstride = n;
}

// Wave-split sums (wave_f64_block) of every member: with partial sums (part)
// one block per (item, chunk) of A.items, without one per item, which sums
// every chunk.  Items are ordered by decreasing member size, so the hardware's
// block order does what the persistent kernels' queue does.
template <int TPL>
__global__ __launch_bounds__(256) void ens_wave_f64_kernel(
    const double* __restrict__ quads, EnsArgs A, double* part) {
  __shared__ double red[4][64 * TPL][3];
  if (flat_block() >= A.n_items) return;
  const int4 w = A.items[flat_block()];
  const int c0 = w.w;
  const EnsMember M = A.mem[w.x];
  SegArgs sg = ens_segment(A, M, w.y);
  if (part) ens_parts(sg, M, w.y, part);
  wave_f64_block<TPL, false, true>(quads + static_cast<int64_t>(M.P) * 6, M.cnt,
                                   sg, w.z, c0, part ? c0 + 1 : M.C, M.C, 0.0,
                                   red);
}

// Adds the chunk partials of the PER targets of each work item, one block per
// item.
template <int PER>
__global__ __launch_bounds__(PER) void ens_chunk_reduce_kernel(EnsArgs A,
                                                               double* part) {
  if (flat_block() >= A.n_items) return;
  const int4 w = A.items[flat_block()];
  const EnsMember M = A.mem[w.x];
  SegArgs sg = ens_segment(A, M, w.y);
  ens_parts(sg, M, w.y, part);
  wave_reduce_one(sg, static_cast<int64_t>(w.z) * PER + threadIdx.x, M.C);
}

// Chunked matrix-core sums of every member; blocks as ens_wave_f64_kernel.
__global__ __launch_bounds__(256, 5) void ens_mfma16_chunk_kernel(
    Mfma16Src src, EnsArgs A, double* part) {
  __shared__ uint4 la[2 * kPackTile];
  __shared__ float4 lt[kPackTile];
  if (flat_block() >= A.n_items) return;
  const int4 w = A.items[flat_block()];
  const EnsMember M = A.mem[w.x];
  SegArgs sg = ens_segment(A, M, w.y);
  if (part) ens_parts(sg, M, w.y, part);
  const int t0 = M.P / kPackTile;
  Mfma16Src ms{src.y + M.P, src.s + M.P, src.a + 2 * static_cast<int64_t>(M.P),
               src.t + static_cast<int64_t>(t0) * 1024, src.c + t0,
               src.is + t0, nullptr};
  mfma16_chunks<false>(ms, M.cnt, sg, w.z, w.w, M.C, 0.0f, la, lt);
}

template <int BLOCK, int TPL, bool PAIR>
__global__ __launch_bounds__(BLOCK) void ens_mixed_kernel(
    const float4* __restrict__ src, const double4* __restrict__ centers,
    EnsArgs A) {
  constexpr int TILE = 256;
  __shared__ float4 tile[TILE];
  __shared__ int slot;
  for (;;) {
    const int it = ens_next(A, &slot);
    if (it >= A.n_items) break;
    const int4 w = A.items[it];
    const EnsMember M = A.mem[w.x];
    const SegArgs sg = ens_segment(A, M, w.y);
    mixed_block<BLOCK, TPL, TILE, false, PAIR>(
        src + M.P, centers + M.P / kPackTile, M.cnt, sg, w.z, 0.0f, tile);
  }
}

__global__ __launch_bounds__(256) void ens_mfma_kernel(MfmaSrc src, EnsArgs A) {
  __shared__ float4 ly[kPackTile];
  __shared__ float lq[kPackTile];
  __shared__ float ls[kPackTile];
  __shared__ float4 lt[kPackTile];
  __shared__ int slot;
  for (;;) {
    const int it = ens_next(A, &slot);
    if (it >= A.n_items) break;
    const int4 w = A.items[it];
    const EnsMember M = A.mem[w.x];
    const SegArgs sg = ens_segment(A, M, w.y);
    const int t0 = M.P / kPackTile;
    MfmaSrc ms{src.y + M.P, src.q + M.P, src.s + M.P,
               src.t + static_cast<int64_t>(t0) * 1024, src.c + t0};
    mfma_block<false>(ms, M.cnt, sg, w.z, 0.0f, ly, lq, ls, lt);
  }
}

template <int MINW, int NACC = 1, int RS = 1>
__global__ __launch_bounds__(256, MINW) void ens_mfma16_kernel(Mfma16Src src,
                                                               EnsArgs A) {
  __shared__ uint4 la[2 * kPackTile];
  __shared__ float4 lt[kPackTile];
  __shared__ int slot;
  for (;;) {
    const int it = ens_next(A, &slot);
    if (it >= A.n_items) break;
    const int4 w = A.items[it];
    const EnsMember M = A.mem[w.x];
    const SegArgs sg = ens_segment(A, M, w.y);
    const int t0 = M.P / kPackTile;
    Mfma16Src ms{src.y + M.P, src.s + M.P, src.a + 2 * static_cast<int64_t>(M.P),
                 src.t + static_cast<int64_t>(t0) * 1024, src.c + t0,
                 src.is + t0, nullptr};
    mfma16_block<false, NACC, 1, RS>(ms, M.cnt, sg, w.z, 0.0f, la,
                                     lt);
  }
}

// ------------------------------------------------------ kernel registry ---
// Every variant has a one-problem twin of the same shape in bve_sums.hip.
using EnsF64Fn = void (*)(const double4*, const double4*, EnsArgs);
using EnsMixedFn = void (*)(const float4*, const double4*, EnsArgs);
using EnsMfmaFn = void (*)(MfmaSrc, EnsArgs);
using EnsMfma16Fn = void (*)(Mfma16Src, EnsArgs);

struct EnsVariant {
  EnsF64Fn f64;
  EnsMixedFn mixed;
  int block, tpl;
  const char* name;
  EnsMfmaFn mfma;
  EnsMfma16Fn mfma16;
  bool wave = false;  // wave-split sums: one block per item and chunk
  bool chunked = false;  // chunked matrix-core sums, likewise
  EnsChunks chunks() const {
    return wave ? kEnsWave : chunked ? kEnsMixed : kEnsWhole;
  }
  const void* fn() const {
    return f64 ? reinterpret_cast<const void*>(f64)
           : mixed ? reinterpret_cast<const void*>(mixed)
           : mfma ? reinterpret_cast<const void*>(mfma)
                  : reinterpret_cast<const void*>(mfma16);
  }
};

// Names are "persistent_" and the one-problem variant's, also of the shapes
// whose blocks take one item (and chunk) each: wave4_scalar and
// mfma16_chunked_near3, the defaults.
#define LPM_ENS_F64(B, T, NR, PAIR)                  \
  {ens_f64_kernel<B, T, NR, PAIR>, nullptr, B, T,    \
   "persistent_block" #B "_tpl" #T "_nr" #NR "_pair" #PAIR, nullptr}
#define LPM_ENS_MIXED(B, T, PAIR)                 \
  {nullptr, ens_mixed_kernel<B, T, PAIR>, B, T,   \
   "persistent_block" #B "_tpl" #T "_pair" #PAIR, nullptr}

const EnsVariant kEnsF64[] = {
    LPM_ENS_F64(256, 2, 2, true),  // 0
    LPM_ENS_F64(256, 2, 1, true),  // 1
    LPM_ENS_F64(256, 1, 1, true),  // 2
    LPM_ENS_F64(256, 4, 1, true),  // 3
    LPM_ENS_F64(128, 2, 2, true),  // 4
    {ens_f64_kernel<256, 2, 1, true, true>, nullptr, 256, 2,
     "persistent_block256_tpl2_nr1_pairtrue_fused", nullptr},  // 5
    {ens_f64_kernel<256, 4, 1, true, true>, nullptr, 256, 4,
     "persistent_block256_tpl4_nr1_pairtrue_fused", nullptr},  // 6
    {ens_f64_kernel<256, 4, 1, true, true, true>, nullptr, 256, 4,
     "persistent_block256_tpl4_nr1_quad_fused", nullptr},      // 7
    {ens_f64_kernel<256, 4, 1, true, true, true, true>, nullptr, 256, 4,
     "persistent_block256_tpl4_nr1_quad_fused_sy", nullptr},   // 8: s y packed
    // 9: scalar-loaded sources divided among a block's waves (the default);
    // 64 block / 128 targets per item
    {nullptr, nullptr, 64, 2, "persistent_wave4_scalar", nullptr, nullptr,
     true},
};
const EnsVariant kEnsMixed[] = {
    LPM_ENS_MIXED(256, 2, false),  // 0
    LPM_ENS_MIXED(256, 1, true),   // 1
    LPM_ENS_MIXED(256, 1, false),  // 2
    LPM_ENS_MIXED(256, 2, true),   // 3
    LPM_ENS_MIXED(256, 4, false),  // 4
    LPM_ENS_MIXED(128, 2, true),   // 5
    {nullptr, nullptr, 256, 1, "persistent_mfma_block256_near3",
     ens_mfma_kernel},             // 6: matrix-core far field
    {nullptr, nullptr, 256, 1, "persistent_mfma16_block256_near3", nullptr,
     ens_mfma16_kernel<1>},        // 7: f16-split distance product
    {nullptr, nullptr, 256, 1, "persistent_mfma16_occ5_block256_near3", nullptr,
     ens_mfma16_kernel<5>},        // 8: register budget for 5 waves per SIMD
    {nullptr, nullptr, 256, 1, "persistent_mfma16_occ5_acc2_block256_near3",
     nullptr, ens_mfma16_kernel<5, 2>},  // 9: two weight-product accumulators
    // 10-11: one reciprocal per four distances
    {nullptr, nullptr, 256, 1, "persistent_mfma16_occ5_qrcp_block256_near3",
     nullptr, ens_mfma16_kernel<5, 1, 4>},
    {nullptr, nullptr, 256, 1,
     "persistent_mfma16_occ5_acc2_qrcp_block256_near3", nullptr,
     ens_mfma16_kernel<5, 2, 4>},
    // 12: the sources in chunks by the member's sizes (the default)
    {nullptr, nullptr, 256, 1, "persistent_mfma16_chunked_near3", nullptr,
     nullptr, false, true},
};
constexpr int kNumEnsF64 = sizeof(kEnsF64) / sizeof(kEnsF64[0]);
constexpr int kNumEnsMixed = sizeof(kEnsMixed) / sizeof(kEnsMixed[0]);

const EnsVariant& ens_variant(int family, int v) {
  return family == KID_BVE_ENS_F64 ? kEnsF64[v] : kEnsMixed[v];
}

}  // namespace

int ens_variant_count(int family) {
  return family == KID_BVE_ENS_F64 ? kNumEnsF64 : kNumEnsMixed;
}
const char* ens_variant_name(int family, int v) {
  return ens_variant(family, v).name;
}
// The defaults are the shapes of the one-problem defaults (default_variant).
int ens_default_variant(int family) {
  return family == KID_BVE_ENS_F64 ? 9 : 12;
}

}  // namespace lpm_amd

namespace lpm_amd {

namespace {

const EnsVariant& pick_ens_variant(lpm_ctx* ctx, const EnsembleDesc& d,
                                   int precision) {
  const int family =
      precision == LPM_MIXED ? KID_BVE_ENS_MIXED : KID_BVE_ENS_F64;
  return ens_variant(family,
                     pick_variant(ctx, family, d.n_verts + d.n_faces));
}

void ensure_sources(lpm_ctx* ctx, const EnsembleDesc& d, int precision,
                    bool wave) {
  const int64_t cap = std::max<int64_t>(d.total_padded_upper, kPackTile);
  if (wave) {
    ctx->quad.ensure(sizeof(double) * 6 * cap);
    return;
  }
  ctx->packed64.ensure(sizeof(double4) * cap);
  if (precision == LPM_FP64) ctx->packed64sy.ensure(sizeof(double4) * cap);
  if (precision == LPM_MIXED) {
    ctx->packed32.ensure(sizeof(float4) * cap);
    ctx->centers.ensure(sizeof(double4) * (cap / kPackTile));
    ctx->mf_y.ensure(sizeof(float4) * cap);
    ctx->mf_q.ensure(sizeof(float) * cap);
    ctx->mf_s.ensure(sizeof(float) * cap);
    ctx->mf_t.ensure(sizeof(float) * 4 * cap);
    ctx->mf_c.ensure(sizeof(double4) * (cap / kPackTile));
    ctx->mf_a.ensure(sizeof(uint4) * 2 * cap);
    ctx->mf_t32.ensure(sizeof(float) * 4 * cap);
    ctx->mf_is.ensure(sizeof(double) * (cap / kPackTile));
  }
}

}  // namespace

// Vertex slot order of the mixed sums, from the members' state positions
// (also used for the stage evaluations of a step, whose positions are close).
const int32_t* bve_ens_vertex_order(lpm_ctx* ctx, const EnsembleDesc& d,
                                    const lpm_bve_fields& f, hipStream_t s) {
  return target_order(ctx, CrdIn{f.vert_x, f.vert_x_es, f.vert_x_cs},
                      d.n_verts, d.voff, d.n_members, s);
}

uint64_t ensemble_prepare(lpm_ctx* ctx, const EnsembleDesc& d,
                          const lpm_bve_fields& f, int precision,
                          hipStream_t s) {
  const EnsVariant& v = pick_ens_variant(ctx, d, precision);
  const EnsLayout L = ensemble_plan(ctx, d, v.block * v.tpl, v.chunks());
  ensure_sources(ctx, d, precision, v.wave);
  if (v.wave || v.chunked)
    chunk_workspace(ctx, sizeof(double) * 3 * L.parts, s);
  if (precision == LPM_MIXED) bve_ens_vertex_order(ctx, d, f, s);
  return L.serial;
}

void ensemble_velocity(lpm_ctx* ctx, const EnsembleDesc& d,
                       const lpm_bve_fields& f, CrdIn vx, CrdIn fx,
                       const double* fzeta, const RankMap& map, int precision,
                       unsigned flags, hipStream_t s) {
  const int M = d.n_members;
  const int family =
      precision == LPM_MIXED ? KID_BVE_ENS_MIXED : KID_BVE_ENS_F64;
  const EnsVariant& v = pick_ens_variant(ctx, d, precision);
  ensure_sources(ctx, d, precision, v.wave);
  const EnsLayout L =
      ensemble_layout(ctx, d, map, v.block * v.tpl, s, v.chunks());

  double4* p64 = ctx->packed64.as<double4>();
  double4* psy =
      precision == LPM_FP64 ? ctx->packed64sy.as<double4>() : nullptr;
  const dim3 pgrid(static_cast<unsigned>((d.max_member_faces + 255) / 256),
                   static_cast<unsigned>(M));
  if (v.wave)
    ens_pack_quad_kernel<<<pgrid, 256, 0, s>>>(
        fx.base, fx.es, fx.cs, fzeta, f.face_area, map.inv, L.mem,
        ctx->quad.as<double>());
  else if (v.mfma16 || v.chunked)
    ens_pack_mfma16_kernel<<<pgrid, kPackTile, 0, s>>>(
        fx.base, fx.es, fx.cs, fzeta, f.face_area, map.inv, L.mem,
        Mfma16Out{ctx->mf_y.as<float4>(), ctx->mf_s.as<float>(),
                  ctx->mf_c.as<double4>(), ctx->mf_a.as<uint4>(),
                  ctx->mf_t32.as<float>(), ctx->mf_is.as<double>()});
  else
    ens_pack_f64_kernel<<<pgrid, 256, 0, s>>>(fx.base, fx.es, fx.cs, fzeta,
                                               f.face_area, map.inv, L.mem,
                                               p64, psy);
  LPM_HIP_CHECK(hipGetLastError());

  EnsArgs A{};
  A.mem = L.mem;
  A.items = L.items;
  A.n_items = L.n_items;
  A.queue = L.queue;
  A.vx = vx.base;
  A.vxes = vx.es;
  A.vxcs = vx.cs;
  A.vu = f.vert_u;
  A.vues = f.vert_u_es;
  A.vucs = f.vert_u_cs;
  A.fx = fx.base;
  A.fxes = fx.es;
  A.fxcs = fx.cs;
  A.fu = f.face_u;
  A.fues = f.face_u_es;
  A.fucs = f.face_u_cs;
  A.rank = map.rank;
  A.inv = map.inv;
  A.skip_masked = (flags & LPM_FLAG_SKIP_MASKED_TARGETS) ? 1 : 0;
  if (precision == LPM_MIXED) A.vorder = bve_ens_vertex_order(ctx, d, f, s);
  if (A.n_items == 0) return;
  if (v.wave) {
    constexpr int kTpl = 2;
    LPM_ARG_CHECK(v.block * v.tpl == 64 * kTpl, "wave-split item size");
    // no workspace (a caller's capture, no memory): whole items, same bits
    double* part = chunk_workspace(ctx, sizeof(double) * 3 * L.parts, s);
    EnsArgs B = A;
    if (part) {
      B.items = L.chunk_items;
      B.n_items = L.n_chunk_items;
    }
    TimedLaunch tl(ctx, family, s, L.pairs);
    ens_wave_f64_kernel<kTpl>
        <<<launch_grid(B.n_items, 256), 256, 0, s>>>(
            ctx->quad.as<double>(), B, part);
    LPM_HIP_CHECK(hipGetLastError());
    if (part) {
      ens_chunk_reduce_kernel<64 * kTpl>
          <<<A.n_items, 64 * kTpl, 0, s>>>(A, part);
      LPM_HIP_CHECK(hipGetLastError());
    }
    return;
  }
  const float4* p32 = nullptr;
  const double4* cen = nullptr;
  MfmaSrc ms{};
  Mfma16Src ms16{};
  if (precision == LPM_MIXED) {
    const int ntile = static_cast<int>(d.total_padded_upper / kPackTile);
    p32 = ctx->packed32.as<float4>();
    cen = ctx->centers.as<double4>();
    if (v.mfma16 || v.chunked) {
      ms16 = Mfma16Src{ctx->mf_y.as<float4>(), ctx->mf_s.as<float>(),
                       ctx->mf_a.as<uint4>(), ctx->mf_t32.as<float>(),
                       ctx->mf_c.as<double4>(), ctx->mf_is.as<double>(),
                       nullptr};
    } else if (v.mfma) {
      ms = MfmaSrc{ctx->mf_y.as<float4>(), ctx->mf_q.as<float>(),
                   ctx->mf_s.as<float>(), ctx->mf_t.as<float>(),
                   ctx->mf_c.as<double4>()};
      // member padding is all-zero records, which the packer skips
      pack_mfma_kernel<<<ntile, kPackTile, 0, s>>>(
          p64, L.padded_total, ctx->mf_y.as<float4>(), ctx->mf_q.as<float>(),
          ctx->mf_s.as<float>(), ctx->mf_t.as<float>(),
          ctx->mf_c.as<double4>());
    } else {
      pack_mixed_kernel<<<ntile, kPackTile, 0, s>>>(
          p64, L.padded_total, ctx->packed32.as<float4>(),
          ctx->centers.as<double4>());
    }
    LPM_HIP_CHECK(hipGetLastError());
  }
  if (v.chunked) {
    // no workspace (a caller's capture, no memory): whole items, same bits
    double* part = chunk_workspace(ctx, sizeof(double) * 3 * L.parts, s);
    EnsArgs B = A;
    if (part) {
      B.items = L.chunk_items;
      B.n_items = L.n_chunk_items;
    }
    TimedLaunch tl(ctx, family, s, L.pairs);
    ens_mfma16_chunk_kernel<<<launch_grid(B.n_items, 256), 256, 0, s>>>(
        ms16, B, part);
    LPM_HIP_CHECK(hipGetLastError());
    if (part) {
      ens_chunk_reduce_kernel<256><<<A.n_items, 256, 0, s>>>(A, part);
      LPM_HIP_CHECK(hipGetLastError());
    }
    return;
  }
  const int grid = ensemble_grid(ctx, v.fn(), v.block, A.n_items);
  TimedLaunch tl(ctx, family, s, L.pairs);
  if (v.mfma16)
    hipLaunchKernelGGL(v.mfma16, dim3(grid), dim3(v.block), 0, s, ms16, A);
  else if (v.mfma)
    hipLaunchKernelGGL(v.mfma, dim3(grid), dim3(v.block), 0, s, ms, A);
  else if (precision == LPM_MIXED)
    hipLaunchKernelGGL(v.mixed, dim3(grid), dim3(v.block), 0, s, p32, cen, A);
  else
    hipLaunchKernelGGL(v.f64, dim3(grid), dim3(v.block), 0, s,
                       static_cast<const double4*>(p64),
                       static_cast<const double4*>(psy), A);
  LPM_HIP_CHECK(hipGetLastError());
}

}  // namespace lpm_amd
