// Ensembles of independent problems stored back to back: member offsets,
// work plans and the device member table, shared by the BVE and SWE
// ensemble kernels.
//
// Per evaluation the face mask of the whole ensemble is compacted by the
// scan of a single problem (build_rank); member m's undivided faces are then
// the compacted ranks [R_m, R_m + cnt_m).  Each member's sources are packed
// into their own region starting at P_m, a multiple of the 256-source
// packing tile, so that every member's tiles are exactly those a
// one-member call would build.  A work item is (member, segment, target block)
// or, of sums in chunks, one source chunk of it: a block each, or taken from a
// queue through one atomic counter by the persistent kernels of the other
// variants.  Items are ordered by decreasing member face count, so the largest
// members start first and small ones fill the tail.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "internal.hpp"

// Work list and member table of one offset layout for one target-block
// size.  Rebuilt (and uploaded synchronously) when the offsets change.
struct lpm_ctx::EnsemblePlan {
  std::vector<int64_t> voff, foff;
  int per = 0;
  int n_items = 0;
  double pairs = 0;
  int n_chunk_items = 0;
  int64_t parts = 0;
  uint64_t serial = 0;
  lpm_amd::DevBuf members;  // EnsMember per member
  lpm_amd::DevBuf items;    // int4 per work item
  lpm_amd::DevBuf chunk_items;  // int4 per (item, chunk) of chunked sums
};

namespace lpm_amd {
namespace {

// Undivided faces before face pos (rank: see RankMap; pos < n).
__device__ __forceinline__ int32_t faces_before(const int32_t* rank,
                                                int64_t pos) {
  if (!rank) return static_cast<int32_t>(pos);
  const int32_t r = rank[pos];
  return r < 0 ? -1 - r : r;
}

// cnt_m, R_m and P_m = sum over earlier members of cnt rounded up to the
// packing tile; *padded_total = P after the last member.
__global__ __launch_bounds__(1024) void ens_layout_kernel(
    EnsMember* __restrict__ mem, int n_members,
    const int32_t* __restrict__ rank, const int32_t* __restrict__ count,
    int32_t* __restrict__ padded_total, int32_t* __restrict__ queue) {
  __shared__ int32_t buf[1024];
  __shared__ int32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int m0 = 0; m0 < n_members; m0 += 1024) {
    const int m = m0 + threadIdx.x;
    int R = 0, cnt = 0;
    if (m < n_members) {
      const int64_t f0 = mem[m].f0, f1 = f0 + mem[m].nf;
      R = faces_before(rank, f0);
      cnt = (m + 1 < n_members ? faces_before(rank, f1) : *count) - R;
    }
    const int padded = (cnt + kEnsTile - 1) / kEnsTile * kEnsTile;
    buf[threadIdx.x] = padded;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      const int add = threadIdx.x >= off ? buf[threadIdx.x - off] : 0;
      __syncthreads();
      buf[threadIdx.x] += add;
      __syncthreads();
    }
    if (m < n_members) {
      mem[m].R = R;
      mem[m].cnt = cnt;
      mem[m].P = carry + buf[threadIdx.x] - padded;
    }
    __syncthreads();
    if (threadIdx.x == 1023) carry += buf[1023];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    *padded_total = carry;
    *queue = 0;
  }
}

int member_chunks(EnsChunks kind, int64_t n_targets, int64_t n_src) {
  switch (kind) {
    case kEnsWave: return wave_chunks(n_targets, n_src);
    case kEnsSwe: return swe_chunks(n_targets, n_src);
    case kEnsMixed: return mixed_chunks(n_targets, n_src);
    case kEnsSweMixed: return swe_mf_chunks(n_targets, n_src);
    default: return 1;
  }
}

std::shared_ptr<lpm_ctx::EnsemblePlan> plan_for(lpm_ctx* ctx,
                                                const EnsembleDesc& d,
                                                int per, EnsChunks kind) {
  const int M = d.n_members;
  auto& slot = ctx->ens_plans[{per, kind}];
  if (slot && static_cast<int>(slot->voff.size()) == M + 1 &&
      std::equal(slot->voff.begin(), slot->voff.end(), d.voff) &&
      std::equal(slot->foff.begin(), slot->foff.end(), d.foff))
    return slot;
  auto np = std::make_shared<lpm_ctx::EnsemblePlan>();
  np->voff.assign(d.voff, d.voff + M + 1);
  np->foff.assign(d.foff, d.foff + M + 1);
  np->per = per;
  std::vector<EnsMember> mem(M);
  std::vector<int> order(M);
  for (int m = 0; m < M; ++m) {
    EnsMember& x = mem[m];
    x.v0 = np->voff[m];
    x.nv = np->voff[m + 1] - np->voff[m];
    x.f0 = np->foff[m];
    x.nf = np->foff[m + 1] - np->foff[m];
    x.R = x.cnt = x.P = 0;
    x.C = member_chunks(kind, x.nv + x.nf, x.nf);
    x.part0 = np->parts;
    np->parts += x.C * (x.nv + x.nf);
    np->pairs += static_cast<double>(x.nv + x.nf) * static_cast<double>(x.nf);
    order[m] = m;
  }
  std::stable_sort(order.begin(), order.end(),
                   [&](int a, int b) { return mem[a].nf > mem[b].nf; });
  std::vector<int4> w, wc;
  for (int m : order) {
    for (int seg = 0; seg < 2; ++seg) {
      const int64_t n = seg == 0 ? mem[m].nv : mem[m].nf;
      for (int64_t b = 0; b < (n + per - 1) / per; ++b) {
        w.push_back(make_int4(m, seg, static_cast<int>(b), 0));
        for (int k = 0; kind != kEnsWhole && k < mem[m].C; ++k)
          wc.push_back(make_int4(m, seg, static_cast<int>(b), k));
      }
    }
  }
  LPM_ARG_CHECK(std::max(w.size(), wc.size()) < (size_t(1) << 31),
                "too many work items");
  np->n_items = static_cast<int>(w.size());
  np->n_chunk_items = static_cast<int>(wc.size());
  np->members.kept = np->items.kept = np->chunk_items.kept = &ctx->kept;
  void* dm = np->members.ensure(sizeof(EnsMember) * M);
  void* di = np->items.ensure(sizeof(int4) * std::max<size_t>(w.size(), 1));
  LPM_HIP_CHECK(hipMemcpy(dm, mem.data(), sizeof(EnsMember) * M,
                          hipMemcpyHostToDevice));
  if (!w.empty())
    LPM_HIP_CHECK(hipMemcpy(di, w.data(), sizeof(int4) * w.size(),
                            hipMemcpyHostToDevice));
  if (!wc.empty()) {
    void* dc = np->chunk_items.ensure(sizeof(int4) * wc.size());
    LPM_HIP_CHECK(hipMemcpy(dc, wc.data(), sizeof(int4) * wc.size(),
                            hipMemcpyHostToDevice));
  }
  np->serial = ++ctx->ens_plan_serial;
  slot = np;
  return slot;
}

}  // namespace

EnsembleDesc validate_members(int32_t n_members, const int64_t* voff,
                              const int64_t* foff, int64_t n_verts,
                              int64_t n_faces) {
  const int M = n_members;
  LPM_ARG_CHECK(M >= 1 && M <= 65535, "n_members must be in [1, 65535]");
  LPM_ARG_CHECK(voff && foff, "null member offsets");
  LPM_ARG_CHECK(voff[0] == 0 && foff[0] == 0, "member offsets must start at 0");
  LPM_ARG_CHECK(voff[M] == n_verts,
                "vert_offsets[n_members] must equal n_verts");
  LPM_ARG_CHECK(foff[M] == n_faces,
                "face_offsets[n_members] must equal n_faces");
  EnsembleDesc d;
  d.n_members = M;
  d.voff = voff;
  d.foff = foff;
  d.n_verts = n_verts;
  d.n_faces = n_faces;
  for (int m = 0; m < M; ++m) {
    const int64_t nv = voff[m + 1] - voff[m];
    const int64_t nf = foff[m + 1] - foff[m];
    LPM_ARG_CHECK(nv >= 0, "vert_offsets must be nondecreasing");
    LPM_ARG_CHECK(nf >= 1, "every member needs at least one face");
    d.max_member_faces = std::max(d.max_member_faces, nf);
    d.total_padded_upper += (nf + kEnsTile - 1) / kEnsTile * kEnsTile;
  }
  LPM_ARG_CHECK(d.total_padded_upper < (int64_t(1) << 31),
                "ensemble too large for 32-bit packed indices");
  return d;
}

EnsLayout ensemble_plan(lpm_ctx* ctx, const EnsembleDesc& d, int per,
                        EnsChunks chunks) {
  auto p = plan_for(ctx, d, per, chunks);
  int32_t* q = static_cast<int32_t*>(ctx->ens_queue.ensure(sizeof(int32_t) * 2));
  EnsLayout L;
  L.mem = p->members.as<EnsMember>();
  L.items = p->items.as<int4>();
  L.n_items = p->n_items;
  L.queue = q;
  L.padded_total = q + 1;
  L.pairs = p->pairs;
  L.chunk_items = p->chunk_items.as<int4>();
  L.n_chunk_items = p->n_chunk_items;
  L.parts = p->parts;
  L.serial = p->serial;
  return L;
}

EnsLayout ensemble_layout(lpm_ctx* ctx, const EnsembleDesc& d,
                          const RankMap& map, int per, hipStream_t s,
                          EnsChunks chunks) {
  EnsLayout L = ensemble_plan(ctx, d, per, chunks);
  const int M = d.n_members;
  ens_layout_kernel<<<1, 1024, 0, s>>>(L.mem, M, map.rank, map.d_count,
                                       L.padded_total, L.queue);
  LPM_HIP_CHECK(hipGetLastError());
  return L;
}

int ensemble_grid(lpm_ctx* ctx, const void* kernel, int block, int n_items) {
  int per_cu = 0;
  LPM_HIP_CHECK(
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0));
  const int resident = std::max(1, per_cu) * std::max(1, ctx->num_cus);
  return std::max(1, std::min(resident, n_items));
}

}  // namespace lpm_amd
