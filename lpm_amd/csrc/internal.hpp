// Internal declarations shared by the HIP translation units of
// liblpm_mi355x.so.  Not part of the ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <functional>
#include <map>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "launch_grid.hpp"
#include "lpm_mi355x.h"

namespace lpm_amd {

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define LPM_HIP_CHECK(expr)                                                 \
  do {                                                                      \
    hipError_t lpm_e_ = (expr);                                             \
    if (lpm_e_ != hipSuccess)                                               \
      throw ::lpm_amd::Error(LPM_ERR_HIP, std::string(#expr) + " failed: " + \
                                              hipGetErrorString(lpm_e_));   \
  } while (0)

#define LPM_ARG_CHECK(cond, msg)                                  \
  do {                                                            \
    if (!(cond)) throw ::lpm_amd::Error(LPM_ERR_ARG, (msg));      \
  } while (0)

// Incremented whenever any workspace is allocated or outgrown; captured graphs
// record it and are re-captured when it changed, so that a replay never
// touches freed workspace memory.
extern std::atomic<uint64_t> g_workspace_epoch;

// Memory that a graph of the caller may still use: a call recorded by the
// caller's own capture leaves the addresses of the context's buffers in a graph
// that the library never sees.  So an outgrown buffer that such a call may have
// recorded is kept until the context ends.
struct KeptMemory {
  uint64_t serial = 0;  // odd during a recorded call, of its own for each
  std::vector<void*> ptrs;
  ~KeptMemory();
  void call(bool captured) {
    if ((serial & 1) != captured) ++serial;
    else if (captured) serial += 2;
  }
  // of a buffer allocated at serial `born`
  bool recorded(uint64_t born) const { return (born & 1) || serial > born; }
};

// Grow-only device buffer owned by a context.
struct DevBuf {
  void* ptr = nullptr;
  size_t bytes = 0;
  KeptMemory* kept = nullptr;  // its context's (null: never recorded)
  uint64_t born = 0;           // kept->serial when allocated
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf();
  void* ensure(size_t nbytes);  // reallocates (contents lost) when too small
  hipError_t release();         // frees or keeps the memory
  template <typename T>
  T* as() const {
    return static_cast<T*>(ptr);
  }
};

// Strided coordinate/vector arrays: element (i, k) at base[i*es + k*cs].
struct CrdIn {
  const double* base;
  int64_t es, cs;
};
struct CrdOut {
  double* base;
  int64_t es, cs;
};

// Elements per block of the mask scan.
constexpr int kMaskScanChunk = 1024;

// Compaction of a face mask: rank[i] = packed index of face i, or -1 - (number
// of undivided faces before it) if divided; inv[r] = face of packed index r,
// *d_count = number packed.
// With no mask, rank and inv are the identity and not materialised.
struct RankMap {
  const int32_t* rank = nullptr;
  const int32_t* inv = nullptr;
  const int32_t* d_count = nullptr;
  int64_t n = 0;
};

// A target set of one direct-sum launch.  Thread slot c (0 <= c < n, or
// < *d_n when d_n is set) evaluates target i = index ? index[c] : c.
struct TargetSeg {
  CrdIn x{nullptr, 0, 0};
  int64_t n = 0;
  const int32_t* index = nullptr;      // slot -> target (compacted targets)
  const int32_t* d_n = nullptr;        // device count of live slots
  const int32_t* self_rank = nullptr;  // collocated: packed index of target
                                       // i's own source, < 0 if none
  bool self_identity = false;          // collocated: self = slot c
  const uint8_t* skip = nullptr;       // targets to leave untouched
  bool mesh = false;                   // points of the sources' mesh, in its
                                       // order (else: arbitrary points)
  CrdOut out{nullptr, 0, 0};           // velocity output
  double* out_scalar = nullptr;        // stream-function output
};

// Sources after the prologue: undivided faces, compacted and packed.
struct PackedSources {
  const void* data = nullptr;      // double4 {x,y,z,s} (FP64) or float4
                                   // {x',y',z',2s} tile-relative (mixed)
  const double4* centers = nullptr; // mixed: tile centres (x, y, z, -)
  const double4* sy = nullptr;     // FP64: {s y, 0} per source
  const int32_t* count = nullptr;  // device: number of packed sources
  int64_t capacity = 0;            // host upper bound (n stored faces)
  // mixed: matrix-core layout (see bve_device.hpp)
  const float4* mf_y = nullptr;
  const float* mf_q = nullptr;
  const float* mf_s = nullptr;
  const float* mf_t = nullptr;
  const double4* mf_c = nullptr;
  // mixed: f16 hi/lo distance operands and the 32x32 weight operand
  const uint4* mf_a = nullptr;
  const float* mf_t32 = nullptr;
  const double* mf_is = nullptr;
  const double4* mf_g = nullptr;   // per-tile terms of sums with a logarithm
  const double* quad = nullptr;    // FP64 quad records (see bve_device.hpp)
  const double* rec = nullptr;     // FP64 records {y, s, s y, 0}
};

// Kernel timing records (HIP events around direct-sum launches).
enum KernelId : int {
  KID_BVE_VEL_F64 = 0,
  KID_BVE_VEL_MIXED = 1,
  KID_BVE_PSI = 2,
  KID_SWE_F64 = 3,
  KID_SWE_MIXED = 4,
  KID_BVE_ENS_F64 = 5,
  KID_BVE_ENS_MIXED = 6,
  KID_IC2D = 7,
  KID_COUNT = 8
};

struct TimingRec {
  std::vector<std::pair<hipEvent_t, hipEvent_t>> pending;
  double total_ms = 0;
  int64_t launches = 0;
  double pairs = 0;
};

// Launch configuration of the tiled direct-sum kernels.
struct VelConfig {
  int variant = 0;  // index into the compiled kernel table
};

}  // namespace lpm_amd

struct lpm_ctx {
  int device = 0;
  std::string last_error;
  int num_cus = 0;
  std::string arch;

  lpm_amd::KeptMemory kept;  // before the buffers, which end first

  // prologue workspaces
  lpm_amd::DevBuf rank;         // int32 per stored face
  lpm_amd::DevBuf inv;          // int32 per stored face (packed -> face)
  lpm_amd::DevBuf block_counts; // int32 per scan block (+1 total)
  lpm_amd::DevBuf packed64;     // double4 per source
  lpm_amd::DevBuf packed64sy;   // double4 {s y, 0} per source (FP64)
  lpm_amd::DevBuf quad;         // FP64 quad records (192 B per four sources)
                                // or records (64 B per source)
  lpm_amd::DevBuf log_table;    // table of the FP64 logarithm
  lpm_amd::DevBuf split_part;   // chunk partials of source-split sums
  lpm_amd::DevBuf packed32;     // float4 per source (mixed)
  lpm_amd::DevBuf centers;      // double4 per tile (mixed)
  lpm_amd::DevBuf mf_y, mf_q, mf_s, mf_t, mf_c;  // matrix-core layout (mixed)
  lpm_amd::DevBuf mf_a, mf_t32, mf_is, mf_g;    // f16-split layout (mixed)
  lpm_amd::DevBuf flag;         // int32 non-finite flag
  lpm_amd::DevBuf diag;         // error-norm partial sums
  lpm_amd::DevBuf count_ident;  // int32 count when no mask

  lpm_amd::DevBuf swe_packed;   // SWE sources (64 B each)
  lpm_amd::DevBuf swe_bounds;   // SWE tile bounding spheres
  lpm_amd::DevBuf swe_feat;     // SWE matrix-core tile records
  lpm_amd::DevBuf swe_far;      // SWE far sums without chunks (18 per target)

  // ensemble work plans (keyed by targets per work item and chunking) and
  // scratch
  struct EnsemblePlan;
  std::map<std::pair<int, int>, std::shared_ptr<EnsemblePlan>> ens_plans;
  uint64_t ens_plan_serial = 0;
  lpm_amd::DevBuf ens_queue;    // int32 work-queue head, padded total

  // RK4 stage buffers
  lpm_amd::DevBuf rk_v, rk_f;   // BVE vertex / face stage storage
  lpm_amd::DevBuf swe_v, swe_f; // SWE vertex / face stage storage
  lpm_amd::DevBuf ic2d_v, ic2d_f; // Incompressible2D RK2 stage storage

  // timing
  bool timing = false;
  lpm_amd::TimingRec timing_rec[lpm_amd::KID_COUNT];
  std::vector<hipEvent_t> event_pool;

  // graph cache for RK4 steps
  struct GraphEntry;
  std::map<std::string, std::shared_ptr<GraphEntry>> graphs;
  uint64_t graph_clock = 0;  // LRU stamps of the graph cache

  // stream of the last call that used the context's workspaces, and the
  // event that orders a call on another stream after it
  hipStream_t last_stream = nullptr;
  bool has_last_stream = false;
  hipEvent_t order_event = nullptr;

  // autotuned kernel variants, keyed by (arch, kernel, size bucket)
  std::map<std::string, int> tuned;
  int forced[lpm_amd::KID_COUNT] = {-1, -1, -1, -1, -1, -1, -1, -1};
  // bumped whenever `tuned` or `forced` changes: captured graphs record the
  // kernels of the choice in force when they were captured
  uint64_t choice_serial = 0;

  // spatially compact slot orders of target sets (target_order)
  struct TargetOrder {
    const double* x = nullptr;
    int64_t es = 0, cs = 0, n = 0;
    uint64_t ranges = 0;  // hash of the range offsets
    uint64_t last_use = 0;
    lpm_amd::DevBuf perm;  // int32 per slot: target index
  };
  std::vector<std::unique_ptr<TargetOrder>> orders;
  uint64_t order_clock = 0;

  lpm_ctx() {
    for (lpm_amd::DevBuf* b :
         {&rank, &inv, &block_counts, &packed64, &packed64sy, &quad,
          &log_table, &split_part, &packed32, &centers, &mf_y, &mf_q, &mf_s,
          &mf_t, &mf_c, &mf_a, &mf_t32, &mf_is, &mf_g, &flag, &diag,
          &count_ident, &swe_packed, &swe_bounds, &swe_feat, &swe_far,
          &ens_queue, &rk_v, &rk_f, &swe_v, &swe_f, &ic2d_v, &ic2d_f})
      b->kept = &kept;
  }
};

namespace lpm_amd {

void set_error(lpm_ctx* ctx, const std::string& msg);

// Orders this call's work on stream s after everything the context issued
// on the stream of its previous call (the workspaces are shared by all of
// a context's calls).  No-op when the stream is unchanged or capturing; a
// capture is the caller's (the steps begin theirs later) and is counted in
// ctx->kept.
void order_stream(lpm_ctx* ctx, hipStream_t s);

// Kernel variants of a family (KID_*) and the autotuning table.
int variant_count(int family);
const char* variant_name(int family, int v);
int default_variant(int family);
std::string tune_key(const lpm_ctx* ctx, int family, int64_t n_targets);
// The forced or tuned variant, else dflt (default_variant).
int pick_variant(lpm_ctx* ctx, int family, int64_t n_targets, int dflt);
int pick_variant(lpm_ctx* ctx, int family, int64_t n_targets);
hipStream_t as_stream(void* s);

// grid_xy as a launch argument.
inline dim3 launch_grid(int64_t blocks, int threads) {
  const GridXY g = grid_xy(blocks, threads);
  return dim3(g.x, g.y);
}
#ifdef __HIP__
// Block index in such a launch.
__device__ __forceinline__ int flat_block() {
  return static_cast<int>(blockIdx.y * gridDim.x + blockIdx.x);
}
#endif

// Event bracket for a timed launch (no-op when timing is off).
struct TimedLaunch {
  lpm_ctx* ctx;
  int kid;
  hipStream_t stream;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  double pairs;
  TimedLaunch(lpm_ctx* c, int k, hipStream_t s, double p);
  ~TimedLaunch() noexcept(false);
};

// ---- prologue (bve_sums.hip) ----
RankMap build_rank(lpm_ctx* ctx, const uint8_t* mask, int64_t n,
                   hipStream_t s);
// Packs the source layouts in `layouts` (kLayout bits) into context buffers.
PackedSources pack_sources(lpm_ctx* ctx, unsigned layouts, CrdIn sx,
                           const double* zeta, const double* area,
                           const RankMap& map, int precision, hipStream_t s);

// The same prologue into caller-provided device buffers (no allocation).
// Sizes for n stored faces: counts ceil(n / kMaskScanChunk) + 1, rank and
// inv n each (unused without a mask), count_ident 1.
struct RankWs {
  int32_t* counts = nullptr;
  int32_t* rank = nullptr;
  int32_t* inv = nullptr;
  int32_t* count_ident = nullptr;
};
RankMap build_rank_into(const RankWs& ws, const uint8_t* mask, int64_t n,
                        hipStream_t s);
// The context's own buffers, sized (no launches: a step's prepare).
RankWs rank_workspace(lpm_ctx* ctx, const uint8_t* mask, int64_t n);

// Source layouts of the sums (bit set).  Every layout but kLayoutQuad,
// kLayoutRec and kLayoutMfma16 also needs the FP64 packing p64.  With tcap = 256 * ceil(n / 256)
// and ntile = tcap / 256 the arrays hold: quad 24 and rec 32 ceil(n / 4)
// double; p64 4 ceil(n / 4) and psy n double4; p32 n float4;
// centers, mf_c ntile double4; mf_y tcap float4; mf_q, mf_s tcap float;
// mf_t, mf_t32 4 tcap float; mf_a 2 tcap uint4; mf_is ntile double.
enum : unsigned {
  kLayoutSy = 1u,      // FP64 {s y} (psy)
  kLayoutVec32 = 2u,   // mixed vector-ALU kernels (p32, centers)
  kLayoutMfma = 4u,    // f32 matrix-core kernel (mf_y, mf_q, mf_s, mf_t, mf_c)
  kLayoutMfma16 = 8u,  // f16-split kernels (mf_y, mf_s, mf_c, mf_a, mf_t32,
                       // mf_is)
  kLayoutQuad = 16u,   // FP64 quad records (quad)
  kLayoutRec = 32u,    // FP64 records {y, s, s y, 0} (rec)
  kLayoutLog = 64u,    // with kLayoutMfma16: per-tile terms of the sums with a
                       // logarithm (mf_g, ntile double4)
};
struct PackWs {
  double* quad = nullptr;
  double* rec = nullptr;
  double4* p64 = nullptr;
  double4* psy = nullptr;
  float4* p32 = nullptr;
  double4* centers = nullptr;
  float4* mf_y = nullptr;
  float* mf_q = nullptr;
  float* mf_s = nullptr;
  float* mf_t = nullptr;
  double4* mf_c = nullptr;
  uint4* mf_a = nullptr;
  float* mf_t32 = nullptr;
  double* mf_is = nullptr;
  double4* mf_g = nullptr;
};
// The context's own buffers of every layout of a precision (no launches), so
// that a call of any kind or variant over n sources prepares the others: under a
// caller's capture none of them allocates.
PackWs pack_workspace(lpm_ctx* ctx, int64_t n, int precision);
PackedSources pack_sources_into(const PackWs& ws, unsigned layouts, CrdIn sx,
                                const double* zeta, const double* area,
                                const RankMap& map, int precision,
                                hipStream_t s);
// Targets that fill the device by themselves (12 blocks of 256 per CU) over so
// few sources that adding and storing chunk sums costs more than chunks gain:
// one chunk.  1e6 free targets against 320, 1,280 and 5,120 sources, in
// microseconds with chunks and without: FP64 velocity 134, 483, 1,708 and 117,
// 419, 1,612; Incompressible2D 309, 1,199, 4,734 and 310, 1,111, 4,303; shallow
// water 928, 3,598, 11,560 and 899, 2,961, 11,275; mixed velocity 154, 362,
// 1,528 and 144, 350, 1,395.  At 20,480 sources chunks are as fast in FP64 and
// 1.1 times as fast in mixed precision.
inline bool one_chunk(int64_t n_targets, int64_t n_src) {
  return n_targets >= (int64_t(3) << 18) && n_src <= 8192;
}
// Source chunks of the wave-split FP64 sums of a problem of n_targets
// targets (both segments) and n_src stored sources: at least 16 (the chunk is
// then fixed per XCD, block index mod 8, and its sources stay in that L2),
// doubled until the blocks of 128 targets times the chunks reach 2,048
// (eight per CU) while every wave keeps 40 stored sources or more.  Level 7:
// 44.3 ms for 8 and 16 chunks, 47.3 for 2; 7,682 x 5,120 pairs: 17.2 us for
// 16, 28 for 5; 12,345 x 11,904: 50 us for 32, 56 for 16.  It depends on the
// sizes alone, so a member of an ensemble has the chunks (and bits) of its
// one-problem call.
inline int wave_chunks(int64_t n_targets, int64_t n_src) {
  if (one_chunk(n_targets, n_src)) return 1;
  const int64_t blocks = (n_targets + 127) / 128;
  int64_t c = 16;
  while (c < 256 && blocks * c < 2048) c *= 2;
  while (c > 1 && n_src < 160 * c) c /= 2;
  return static_cast<int>(c);
}
// Source chunks of the sums with a logarithm (blocks of 64 targets, four waves
// per chunk): as wave_chunks with 80 stored sources or more per wave, whose
// pairs cost twice a velocity pair and whose blocks copy an 8 KiB table.
inline int log_chunks(int64_t n_targets, int64_t n_src) {
  int64_t c = wave_chunks(n_targets, n_src);
  while (c > 1 && n_src < 320 * c) c /= 2;
  return static_cast<int>(c);
}
// Source chunks of the chunked matrix-core velocity sums (blocks of 256
// targets, tiles of 256 sources): 8 (the chunk is then fixed per XCD),
// doubled until blocks times chunks reach 4,096 (three rounds of the resident
// blocks), at most three quarters of the stored sources' tiles (a uniform
// mesh's leaves) or both of two, so that a chunk holds a tile or more.
inline int mixed_chunks(int64_t n_targets, int64_t n_src) {
  if (one_chunk(n_targets, n_src)) return 1;
  const int64_t blocks = (n_targets + 255) / 256;
  const int64_t tiles = (n_src + 255) / 256;
  int64_t c = 8;
  while (c < 256 && blocks * c < 4096) c *= 2;
  c = std::min(c, tiles <= 2 ? tiles : tiles * 3 / 4);
  return static_cast<int>(std::max<int64_t>(1, c));
}
// Source chunks of the wave-split FP64 shallow-water sums (eight waves of a
// block share one): 8, doubled until the blocks of 64 targets times the
// chunks reach 1,024 (four per CU) while every wave keeps 20 stored sources.
inline int swe_chunks(int64_t n_targets, int64_t n_src) {
  if (one_chunk(n_targets, n_src)) return 1;
  const int64_t blocks = (n_targets + 63) / 64;
  int64_t c = 8;
  while (c < 128 && blocks * c < 1024) c *= 2;
  while (c > 1 && n_src < 160 * c) c /= 2;
  return static_cast<int>(c);
}
// Source chunks of the shallow-water sums' matrix-core far pass (blocks of 256
// targets, tiles of 256 sources): 8 (the chunk is then fixed per XCD), doubled
// until blocks times chunks reach 2,048 (four rounds of the two resident blocks
// per CU), at least two of three quarters of the stored sources' tiles a chunk
// above eight of them; 1 from 4,096 blocks on.  Sums of level 5 in
// microseconds for 2,048, 4,096: 546, 601; level 6 with 8, 4 chunks: 4,578,
// 4,648; 30 problems of level 4 with at least 1, 2 tiles a chunk: 2,052, 1,770;
// level 3 (five tiles) 117, 123.
inline int swe_mf_chunks(int64_t n_targets, int64_t n_src) {
  const int64_t blocks = (n_targets + 255) / 256;
  const int64_t tiles = (n_src + 255) / 256 * 3 / 4;
  if (blocks >= 4096) return 1;
  int64_t c = 8;
  while (c < 128 && blocks * c < 2048) c *= 2;
  c = std::min(c, tiles <= 8 ? tiles : tiles / 2);
  return static_cast<int>(std::max<int64_t>(1, c));
}
// Whether a velocity variant sums the sources in chunks by size.
bool bve_variant_chunked(int precision, int variant);
// Chunk sums of a velocity launch, not added up: component a of chunk k of slot
// c of segment g at part[g][(3 k + a) stride[g] + c].
struct ChunkSums {
  const double* part[2] = {nullptr, nullptr};
  int64_t stride[2] = {0, 0};
  int C = 0;
};
// Launches the chunk sums alone, in workspace `part` (bve_split_bytes).
ChunkSums launch_bve_chunks(lpm_ctx* ctx, const PackedSources& src,
                            const TargetSeg* segs, double eps2, int precision,
                            int variant, double* part, hipStream_t s);
// Variant of the BVE velocity kernel a launch over n_targets would use, and
// the source layouts it reads.
int bve_velocity_variant(lpm_ctx* ctx, int precision, int64_t n_targets);
unsigned bve_variant_layouts(int precision, int variant);
// Face targets of a collocated sum: every stored face (self skipped by
// rank) or, with skip_masked, only the undivided ones (compacted slots).
TargetSeg face_targets(CrdIn x, const RankMap& map, const uint8_t* mask,
                       bool skip_masked, CrdOut out, double* out_scalar);
// variant < 0: bve_velocity_variant's choice.  timed = false skips the
// timing events.  allow_split = false runs a source-split variant as its
// unsplit twin (same shape, one summation level less, no workspace).  The
// wave-split variant takes its partial sums' workspace from `part`
// (part_bytes), or with a null part from the context unless timed is false;
// without one each block takes every chunk itself (same bits).
void launch_bve_velocity(lpm_ctx* ctx, const PackedSources& src,
                         TargetSeg* segs, int nseg, double eps2, int precision,
                         hipStream_t s, int variant = -1, bool timed = true,
                         bool allow_split = false, double* part = nullptr,
                         size_t part_bytes = 0);
// Bytes of partial sums a source-split variant needs for n_targets over
// n_src stored sources (0 for every other variant).
size_t bve_split_bytes(int precision, int variant, int64_t n_targets,
                       int64_t n_src);
// The context's split workspace grown to `need` bytes, or nullptr when it
// cannot be: s is capturing and it is smaller, or the device is out of
// memory (the caller then runs an unsplit variant).
double* split_workspace(lpm_ctx* ctx, size_t need, hipStream_t s);
// The same for the sums in chunks by size, which also run without it, in whole
// blocks to the same bits: nullptr above kChunkBytes.  They keep up to 24 C
// (velocity), 8 C (stream function), 32 C (Incompressible2D) or 160 C
// (shallow water) bytes a target, C from 8 on, so a bound is needed: FP64
// shallow water of 1e7 targets would hold 12.8 GB.  At the bound, 2.8 million
// targets in FP64 velocity and 839,000 in shallow water, the target blocks
// alone fill the device many times.  Whole blocks against chunks: level 5
// 1.3 to 3.9 times as long, level 6 1.08 to 1.6, level 7 (600,742 slots, 231
// and 769 MB) 1.02 to 1.17; 1e6 and more targets 0.84 to 1.14.
constexpr size_t kChunkBytes = size_t(1) << 30;
double* chunk_workspace(lpm_ctx* ctx, size_t need, hipStream_t s);
// Uploads the table of the FP64 logarithm (context creation).
void make_log_table(lpm_ctx* ctx);
void launch_bve_stream_fn(lpm_ctx* ctx, const PackedSources& src,
                          TargetSeg* segs, int nseg, hipStream_t s);
void check_finite(lpm_ctx* ctx, const double* base, int64_t n, int64_t es,
                  int64_t cs, int ncomp, hipStream_t s);
// check_finite with a caller-provided device flag (one int32).
void check_finite_into(int32_t* flag, const double* base, int64_t n,
                       int64_t es, int64_t cs, int ncomp, hipStream_t s);

// ---- allocation-free velocity (noalloc.hip) ----
// Looks up the device's static scratch array (once per device; the device
// must be current).  Failures are recorded and reported by the entry point.
void noalloc_setup(int device);

// ---- RK4 (bve_rk4.hip) ----
void validate_bve_fields(const lpm_bve_fields* f);
// Runs issue() on stream s, or with use_graph replays the hipGraph captured
// from it under key_fn() (which must also allocate every workspace issue()
// uses, and launch nothing: it runs before every replay; the graph is
// re-captured when a workspace was reallocated).
void run_maybe_graph(lpm_ctx* ctx, bool use_graph, hipStream_t s,
                     const std::function<std::string()>& key_fn,
                     const std::function<void()>& issue);

// ---- ensembles (ensemble.hip, bve_ensemble.hip) ----
// Host view of an ensemble's member offsets (validated).
struct EnsembleDesc {
  int n_members = 0;
  const int64_t* voff = nullptr;  // host, n_members + 1
  const int64_t* foff = nullptr;  // host, n_members + 1
  int64_t n_verts = 0, n_faces = 0;
  int64_t max_member_faces = 0;
  int64_t total_padded_upper = 0;  // sum of member faces rounded up to 256
};
EnsembleDesc validate_members(int32_t n_members, const int64_t* voff,
                              const int64_t* foff, int64_t n_verts,
                              int64_t n_faces);

// Device member table entry.  v0/nv/f0/nf come from the host offsets; R
// (first compacted rank of the member's undivided faces), cnt (their
// number) and P (first packed slot, a multiple of kEnsTile) are computed on
// the device from the face mask at every evaluation.  The chunk counts and
// partial-sum offsets too come from the member offsets.
constexpr int kEnsTile = 256;
struct EnsMember {
  int64_t v0, nv, f0, nf;
  int32_t R, cnt, P;
  int32_t C;      // source chunks of the plan's chunked sums (1: whole)
  int64_t part0;  // partial sums of the members before: sum of C (nv + nf)
};

// Chunked sums a work plan is for: their chunk counts and partial sums.
enum EnsChunks : int {
  kEnsWhole = 0,   // none: the persistent kernels
  kEnsWave = 1,    // FP64 velocity (wave_chunks)
  kEnsSwe = 2,     // FP64 shallow water (swe_chunks)
  kEnsMixed = 3,   // matrix-core velocity (mixed_chunks)
  kEnsSweMixed = 4,  // matrix-core shallow water (swe_mf_chunks)
};

// Work plan of one offset layout for `per` targets per work item: items
// {member, segment (0 vertices, 1 faces), block, 0} ordered by decreasing
// member face count, and the member table.  A plan for chunked sums also
// lists every (item, chunk) as chunk_items {member, segment, block, chunk}:
// a grid of items times the largest chunk count, whose surplus blocks left
// at once, ran a third as fast with members of levels 5 and 6 together (the
// hardware deals blocks to the shader engines in turn, and the working ones
// then all land on the same).
struct EnsLayout {
  EnsMember* mem = nullptr;
  const int4* items = nullptr;
  int n_items = 0;
  const int4* chunk_items = nullptr;
  int n_chunk_items = 0;
  int64_t parts = 0;                // partial sums: chunks x targets
  int32_t* queue = nullptr;         // work-queue head
  int32_t* padded_total = nullptr;  // packed slots in use (device)
  double pairs = 0;                 // sum of (member targets) x (member faces)
  uint64_t serial = 0;              // changes whenever the plan is rebuilt
};
// Plan and workspaces only (no launches): safe before a stream capture.
EnsLayout ensemble_plan(lpm_ctx* ctx, const EnsembleDesc& d, int per,
                        EnsChunks chunks = kEnsWhole);
// ensemble_plan plus the device member table from the mask (launches on s).
EnsLayout ensemble_layout(lpm_ctx* ctx, const EnsembleDesc& d,
                          const RankMap& map, int per, hipStream_t s,
                          EnsChunks chunks = kEnsWhole);
// Persistent grid: resident blocks of `kernel` on the device, <= n_items.
int ensemble_grid(lpm_ctx* ctx, const void* kernel, int block, int n_items);

int ens_variant_count(int family);
const char* ens_variant_name(int family, int v);
int ens_default_variant(int family);
// BVE: allocates every workspace an evaluation uses (so that a stream
// capture that follows allocates nothing); returns the plan serial.
uint64_t ensemble_prepare(lpm_ctx* ctx, const EnsembleDesc& d,
                          const lpm_bve_fields& f, int precision,
                          hipStream_t s);
// BVE velocity of every member from positions (vx, fx) and face vorticity
// fzeta, written to f.vert_u / f.face_u.
void ensemble_velocity(lpm_ctx* ctx, const EnsembleDesc& d,
                       const lpm_bve_fields& f, CrdIn vx, CrdIn fx,
                       const double* fzeta, const RankMap& map, int precision,
                       unsigned flags, hipStream_t s);

// ---- sphere SWE sums (swe_sums.hip) ----
// Kernel variants of KID_SWE_F64 / KID_SWE_MIXED (the default is 0).
int swe_variant_count(int family);
const char* swe_variant_name(int family, int v);
int swe_default_variant(int family);
struct SwePacked {
  const void* data = nullptr;       // 64 B per source
  const double4* bounds = nullptr;  // per 256-source tile: centre, radius^2
  const int32_t* count = nullptr;
  int64_t capacity = 0;
};
struct SweTargets {
  TargetSeg base;                   // positions, slots, self, velocity out
  const double* surf = nullptr;     // target surface height (PSE)
  double* ddot = nullptr;
  double* laps = nullptr;
};
// Allocates the matrix-core workspaces a mixed launch over n_src stored
// faces and n_targets targets may use (so that a stream capture that follows
// allocates nothing).
void swe_feature_workspace(lpm_ctx* ctx, int64_t n_src, int64_t n_targets,
                           int precision);
// The same with the partial sums of the FP64 sums.
void swe_sums_workspace(lpm_ctx* ctx, int64_t n_src, int64_t n_targets,
                        int precision, hipStream_t s);
// Bounding spheres the sums read next to the packed sources.
enum SweBounds : int { kSweNoBounds, kSweTileBounds, kSweRunBounds };
// n_src: the sources of a call with arbitrary targets, else -1.
SweBounds swe_bounds(lpm_ctx* ctx, int precision, int64_t n_targets,
                     int64_t n_src);
// The packing's buffers, sized (no launches).
void swe_pack_workspace(lpm_ctx* ctx, int64_t n_src);
SwePacked swe_pack_sources(lpm_ctx* ctx, CrdIn sx, const double* zeta,
                           const double* sigma, const double* area,
                           const double* surf, const RankMap& map,
                           SweBounds bounds, hipStream_t s);
void launch_swe_sums(lpm_ctx* ctx, const SwePacked& src, SweTargets* segs,
                     int nseg, double eps, double pse_eps, int precision,
                     hipStream_t s);
// Slot order of n targets at positions x (target indices, int32 on the
// device) that keeps each wave's targets close together: Morton order of
// the positions within each range [off[m], off[m + 1]) (one range when off
// is null).  Computed on the host from the positions at the first call for
// these buffers (it synchronises the stream) and kept in the context (at
// most kOrderCacheMax orders); later calls reuse it as the positions move,
// which changes only how targets are grouped.  Returns nullptr (the given
// order) for n == 0 and for a first call made while s is being captured.
constexpr int kOrderCacheMax = 8;
const int32_t* target_order(lpm_ctx* ctx, CrdIn x, int64_t n,
                            const int64_t* off, int n_ranges, hipStream_t s);

// SWE ensembles: workspaces only (returns the plan serial), and the sums of
// every member at positions (vx, fx) from its own undivided faces.
uint64_t swe_ensemble_prepare(lpm_ctx* ctx, const EnsembleDesc& d,
                              const lpm_swe_fields& f, int precision,
                              hipStream_t s);
void swe_ensemble_sums(lpm_ctx* ctx, const EnsembleDesc& d,
                       const lpm_swe_fields& f, CrdIn vx, CrdIn fx,
                       const double* fzeta, const double* fsigma,
                       const double* farea, const RankMap& map, double eps,
                       double pse_eps, int precision, unsigned flags,
                       hipStream_t s);

}  // namespace lpm_amd
