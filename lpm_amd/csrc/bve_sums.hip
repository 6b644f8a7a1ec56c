// Tiled all-pairs Biot-Savart / Green's-function sums on the unit sphere for
// gfx950 (CDNA4), replacing LPM's one-team-per-target Kokkos reductions
// (src/lpm_bve_sphere_kernels.hpp:20-394).
//
// Prologue: undivided faces are compacted (mask scan) and packed as
//   FP64:  quads of {y, s y} (wave-split sums), {y, s, s y, 0} (sums with a
//          logarithm) or double4 {y0, y1, y2, s},  s = -zeta A / (4 pi)
//   mixed: matrix-core records (bve_device.hpp) or float4  {y0-c0, y1-c1, y2-c2, 2 s} relative to the FP64 centre c
//          of each 256-source packing tile, plus double4 centres.
// Main loop of the wave-split sums: see bve_device.hpp.  Of the others: each
// lane owns TPL targets held in registers; a block stages
// TILE packed sources in LDS and every lane reads them as wave-uniform
// broadcasts.  Per pair the FP64 kernel evaluates t = x.y, w = s/(1-t+eps^2)
// and accumulates S += w y; the velocity is x cross S, which equals
// sum_j w_j (x cross y_j) because x is fixed per target.  The mixed kernel
// evaluates d = y - x in tile-relative FP32, r2 = |d|^2 (= 2(1 - x.y) on the
// unit sphere), w = 2s / r2 and S += w d, carrying per-tile FP32 partials
// into FP64 sums; x cross sum w (y - x) = x cross sum w y.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "bve_device.hpp"
#include "internal.hpp"

namespace lpm_amd {

namespace {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 4;  // elements per thread in the mask scan
constexpr int kScanChunk = kScanBlock * kScanItems;
static_assert(kScanChunk == kMaskScanChunk, "scan chunk must match the header");
// Faces up to which one launch that re-reads the mask beats three (4.5 us
// each): the last of 128 blocks reads 128 KiB, 32 loads a thread.
constexpr int64_t kScanOneLaunch = int64_t(1) << 17;

// ------------------------------------------------------------ prologue ---
__global__ __launch_bounds__(kScanBlock) void mask_count_kernel(
    const uint8_t* __restrict__ mask, int64_t n, int32_t* __restrict__ counts) {
  __shared__ int32_t red[kScanBlock / 64];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanChunk;
  int c = 0;
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + threadIdx.x * kScanItems + k;
    if (i < n && !mask[i]) ++c;
  }
  // wave reduction then across waves
  for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int w = 0; w < kScanBlock / 64; ++w) t += red[w];
    counts[blockIdx.x] = t;
  }
}

// Exclusive scan of nb block counts in place; writes the total to counts[nb].
__global__ __launch_bounds__(1024) void scan_counts_kernel(
    int32_t* __restrict__ counts, int nb) {
  __shared__ int32_t buf[1024];
  __shared__ int32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int b0 = 0; b0 < nb; b0 += 1024) {
    const int i = b0 + threadIdx.x;
    const int v = i < nb ? counts[i] : 0;
    buf[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      const int add = threadIdx.x >= off ? buf[threadIdx.x - off] : 0;
      __syncthreads();
      buf[threadIdx.x] += add;
      __syncthreads();
    }
    if (i < nb) counts[i] = carry + buf[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry += buf[1023];
    __syncthreads();
  }
  if (threadIdx.x == 0) counts[nb] = carry;
}

__global__ __launch_bounds__(kScanBlock) void mask_rank_kernel(
    const uint8_t* __restrict__ mask, int64_t n,
    const int32_t* __restrict__ offsets, int32_t* __restrict__ rank,
    int32_t* __restrict__ inv) {
  __shared__ int32_t buf[kScanBlock];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanChunk +
                       static_cast<int64_t>(threadIdx.x) * kScanItems;
  int c = 0;
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    if (i < n && !mask[i]) ++c;
  }
  buf[threadIdx.x] = c;
  __syncthreads();
  for (int off = 1; off < kScanBlock; off <<= 1) {
    const int add = threadIdx.x >= off ? buf[threadIdx.x - off] : 0;
    __syncthreads();
    buf[threadIdx.x] += add;
    __syncthreads();
  }
  int r = offsets[blockIdx.x] + buf[threadIdx.x] - c;
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    if (i < n) {
      if (mask[i]) {
        rank[i] = -1 - r;
      } else {
        rank[i] = r;
        inv[r] = static_cast<int32_t>(i);
        ++r;
      }
    }
  }
}

// Undivided faces among four mask bytes (nonzero: divided).
__device__ __forceinline__ int undivided4(uint32_t v) {
  const uint32_t nz = ((v & 0x7f7f7f7fu) + 0x7f7f7f7fu) | v;
  return 4 - __popc(nz & 0x80808080u);
}

// The whole compaction in one launch: block b counts the faces before its own
// chunk itself (16 bytes per load; the mask is 16-byte aligned).
__global__ __launch_bounds__(kScanBlock) void mask_scan_kernel(
    const uint8_t* __restrict__ mask, int64_t n, int32_t* __restrict__ offsets,
    int32_t* __restrict__ rank, int32_t* __restrict__ inv) {
  constexpr int kWaves = kScanBlock / 64;
  __shared__ int32_t before[kWaves], own[kWaves];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t chunk0 = static_cast<int64_t>(blockIdx.x) * kScanChunk;
  int pre = 0;
  const uint4* m16 = reinterpret_cast<const uint4*>(mask);
#pragma unroll 4
  for (int64_t k = threadIdx.x; k < chunk0 / 16; k += kScanBlock) {
    const uint4 v = m16[k];
    pre += undivided4(v.x) + undivided4(v.y) + undivided4(v.z) + undivided4(v.w);
  }
  const int64_t base = chunk0 + threadIdx.x * kScanItems;
  bool live[kScanItems];
  int c = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    live[k] = base + k < n && !mask[base + k];
    c += live[k];
  }
  int incl = c;  // inclusive scan over the wave
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int add = __shfl_up(incl, off, 64);
    if (lane >= off) incl += add;
  }
  for (int off = 32; off > 0; off >>= 1) pre += __shfl_xor(pre, off, 64);
  if (lane == 0) before[w] = pre;
  if (lane == 63) own[w] = incl;
  __syncthreads();
  int first = 0, r = incl - c, total = 0;
#pragma unroll
  for (int k = 0; k < kWaves; ++k) {
    first += before[k];
    if (k < w) r += own[k];
    total += own[k];
  }
  r += first;
  if (threadIdx.x == 0) {
    offsets[blockIdx.x] = first;
    if (blockIdx.x + 1 == gridDim.x) offsets[gridDim.x] = first + total;
  }
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    if (i >= n) break;
    rank[i] = live[k] ? r : -1 - r;
    if (live[k]) inv[r++] = static_cast<int32_t>(i);
  }
}

__global__ void set_count_kernel(int32_t* __restrict__ count, int32_t value) {
  *count = value;
}

// Gathers the packed sources in packed order (coalesced writes), zero records
// up to a multiple of four; out_sy (optional) receives {s y, 0} for the kernels
// that take the weight from it.
__global__ __launch_bounds__(256) void pack_f64_kernel(
    const double* __restrict__ sx, int64_t es, int64_t cs,
    const double* __restrict__ zeta, const double* __restrict__ area,
    const int32_t* __restrict__ inv, const int32_t* __restrict__ count,
    double4* __restrict__ out, double4* __restrict__ out_sy) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t n = *count;
  if (r >= n) {
    if (r < (n + 3) / 4 * 4) out[r] = make_double4(0.0, 0.0, 0.0, 0.0);
    return;
  }
  const int64_t i = inv ? inv[r] : r;
  const double* p = sx + i * es;
  const double y0 = p[0], y1 = p[cs], y2 = p[2 * cs];
  const double sv = -zeta[i] * area[i] * kInv4Pi;
  out[r] = make_double4(y0, y1, y2, sv);
  if (out_sy) out_sy[r] = make_double4(sv * y0, sv * y1, sv * y2, 0.0);
}

// Quad records {y, s y} x 4 in packed order, zero records up to a multiple of
// four (a zero record adds nothing: distance 1, strength 0).
__global__ __launch_bounds__(256) void pack_quad_kernel(
    const double* __restrict__ sx, int64_t es, int64_t cs,
    const double* __restrict__ zeta, const double* __restrict__ area,
    const int32_t* __restrict__ inv, const int32_t* __restrict__ count,
    double* __restrict__ quad) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t n = *count;
  if (r >= (n + 3) / 4 * 4) return;
  double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (r < n) {
    const int64_t i = inv ? inv[r] : r;
    const double* p = sx + i * es;
    const double sv = -zeta[i] * area[i] * kInv4Pi;
    for (int a = 0; a < 3; ++a) {
      v[a] = p[a * cs];
      v[3 + a] = sv * v[a];
    }
  }
  double2* o = reinterpret_cast<double2*>(quad + r * 6);
  for (int a = 0; a < 3; ++a) o[a] = make_double2(v[2 * a], v[2 * a + 1]);
}

// Records {y, s, s y, 0} in packed order (64 B), zero records up to a multiple
// of four.
__global__ __launch_bounds__(256) void pack_rec_kernel(
    const double* __restrict__ sx, int64_t es, int64_t cs,
    const double* __restrict__ zeta, const double* __restrict__ area,
    const int32_t* __restrict__ inv, const int32_t* __restrict__ count,
    double* __restrict__ rec) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t n = *count;
  if (r >= (n + 3) / 4 * 4) return;
  double v[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (r < n) {
    const int64_t i = inv ? inv[r] : r;
    const double* p = sx + i * es;
    v[3] = -zeta[i] * area[i] * kInv4Pi;
    for (int a = 0; a < 3; ++a) {
      v[a] = p[a * cs];
      v[4 + a] = v[3] * v[a];
    }
  }
  double2* o = reinterpret_cast<double2*>(rec + r * 8);
  for (int a = 0; a < 4; ++a) o[a] = make_double2(v[2 * a], v[2 * a + 1]);
}

// ------------------------------------------------------- velocity sums ---
// One launch covers two target segments (vertices, then faces): blocks
// [0, s0.nblocks) take s0, the rest s1.
// SY: the weights come from the packed s y (src_sy), one multiply less per
// pair; otherwise src_sy is not read.
template <int BLOCK, int TPL, int TILE, bool EPS, int NR, bool PAIR,
          bool FUSE = false, bool QUAD = false, bool SY = false, int QU = 1>
__global__ __launch_bounds__(BLOCK) void bve_vel_f64_kernel(
    const double4* __restrict__ src, const double4* __restrict__ src_sy,
    const int32_t* __restrict__ count, SegArgs s0, SegArgs s1, double eps2) {
  __shared__ double4 tile[TILE];
  __shared__ double4 tile_sy[SY ? TILE : 1];
  const bool first = static_cast<int>(blockIdx.x) < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? blockIdx.x : blockIdx.x - s0.nblocks;
  f64_block<BLOCK, TPL, TILE, EPS, NR, PAIR, FUSE, QUAD, SY, QU>(
      src, src_sy, *count, sg, blk, eps2, tile, tile_sy);
}

// Source-split form: block b * KS + k sums source chunk k of target block
// b into sg.part; bve_split_reduce_kernel then adds the KS chunks in order
// and writes x cross S.  Equal-sized work items finer than a whole target
// block let every CU finish at nearly the same time.
template <int BLOCK, int TPL, int TILE, bool EPS, int NR, bool PAIR,
          bool FUSE, bool QUAD, bool SY, int QU, int KS>
__global__ __launch_bounds__(BLOCK) void bve_vel_f64_split_kernel(
    const double4* __restrict__ src, const double4* __restrict__ src_sy,
    const int32_t* __restrict__ count, SegArgs s0, SegArgs s1, double eps2) {
  __shared__ double4 tile[TILE];
  __shared__ double4 tile_sy[SY ? TILE : 1];
  const int b = static_cast<int>(blockIdx.x) / KS;
  const int chunk = static_cast<int>(blockIdx.x) % KS;
  const bool first = b < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? b : b - s0.nblocks;
  f64_block<BLOCK, TPL, TILE, EPS, NR, PAIR, FUSE, QUAD, SY, QU, KS>(
      src, src_sy, *count, sg, blk, eps2, tile, tile_sy, chunk);
}

// Wave-split sums (wave_f64_block): with partial sums (s0.part), block
// b * C + k sums chunk k of target block b; without, block b sums every chunk.
template <int TPL, bool EPS, bool MESH>
__global__ __launch_bounds__(256) void bve_wave_f64_kernel(
    const double* __restrict__ quads, const int32_t* __restrict__ count,
    SegArgs s0, SegArgs s1, double eps2, int C) {
  __shared__ double red[4][64 * TPL][3];
  const bool split = s0.part != nullptr;
  const int b = split ? flat_block() / C : flat_block();
  const int c0 = split ? flat_block() % C : 0;
  const bool first = b < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? b : b - s0.nblocks;
  wave_f64_block<TPL, EPS, MESH>(quads, *count, sg, blk, c0, split ? c0 + 1 : C,
                                 C, eps2, red);
}

__global__ __launch_bounds__(256) void bve_wave_reduce_kernel(SegArgs s0,
                                                              SegArgs s1,
                                                              int C) {
  const int64_t g = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const bool first = g < s0.n;
  const SegArgs& sg = pick(s0, s1, first);
  wave_reduce_one(sg, first ? g : g - s0.n, C);
}

// u = x cross (sum over the ks chunks of S, in chunk order) at every live
// slot of both segments.
__global__ __launch_bounds__(256) void bve_split_reduce_kernel(SegArgs s0,
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
  split_reduce_one(sg.part + c, sg.pstride, ks, sg.x + i * sg.es, sg.cs,
                   sg.out + i * sg.oes, sg.ocs);
}

template <int BLOCK, int TPL, int TILE, bool EPS, bool PAIR>
__global__ __launch_bounds__(BLOCK) void bve_vel_mixed_kernel(
    const float4* __restrict__ src, const double4* __restrict__ centers,
    const int32_t* __restrict__ count, SegArgs s0, SegArgs s1, float eps2x2) {
  __shared__ float4 tile[TILE];
  const bool first = static_cast<int>(blockIdx.x) < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? blockIdx.x : blockIdx.x - s0.nblocks;
  mixed_block<BLOCK, TPL, TILE, EPS, PAIR>(src, centers, *count, sg, blk,
                                           eps2x2, tile);
}

template <bool EPS>
__global__ __launch_bounds__(256) void bve_vel_mfma_kernel(
    MfmaSrc src, const int32_t* __restrict__ count, SegArgs s0, SegArgs s1,
    float eps2x2) {
  __shared__ float4 ly[kPackTile];
  __shared__ float lq[kPackTile];
  __shared__ float ls[kPackTile];
  __shared__ float4 lt[kPackTile];
  const bool first = static_cast<int>(blockIdx.x) < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? blockIdx.x : blockIdx.x - s0.nblocks;
  mfma_block<EPS>(src, *count, sg, blk, eps2x2, ly, lq, ls, lt);
}

// MINW: minimum waves per SIMD asked of the register allocator (1: none);
// RS: distances per reciprocal (1, 2 or 4).
template <bool EPS, int MINW = 1, int NACC = 1, int RS = 1>
__global__ __launch_bounds__(256, MINW) void bve_vel_mfma16_kernel(
    Mfma16Src src, const int32_t* __restrict__ count, SegArgs s0, SegArgs s1,
    float eps2x2) {
  __shared__ uint4 la[2 * kPackTile];
  __shared__ float4 lt[kPackTile];
  const bool first = static_cast<int>(blockIdx.x) < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? blockIdx.x : blockIdx.x - s0.nblocks;
  mfma16_block<EPS, NACC, 1, RS>(src, *count, sg, blk, eps2x2, la,
                                 lt);
}

// Source-split form of bve_vel_mfma16_kernel (block b * KS + k: chunk k of
// target block b, partial sums to sg.part; bve_split_reduce_kernel adds
// them): enough equal work items that the last round of waves is full.
template <bool EPS, int MINW, int NACC, int KS, int RS = 1>
__global__ __launch_bounds__(256, MINW) void bve_vel_mfma16_split_kernel(
    Mfma16Src src, const int32_t* __restrict__ count, SegArgs s0, SegArgs s1,
    float eps2x2) {
  __shared__ uint4 la[2 * kPackTile];
  __shared__ float4 lt[kPackTile];
  const int b = static_cast<int>(blockIdx.x) / KS;
  const int chunk = static_cast<int>(blockIdx.x) % KS;
  const bool first = b < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? b : b - s0.nblocks;
  mfma16_block<EPS, NACC, KS, RS>(src, *count, sg, blk, eps2x2, la,
                                  lt, chunk);
}

// Chunked form of the matrix-core sums (mfma16_chunks; the mixed default):
// with partial sums block b * C + k takes chunk k of target block b.
template <bool EPS>
__global__ __launch_bounds__(256, 5) void bve_vel_mfma16_chunk_kernel(
    Mfma16Src src, const int32_t* __restrict__ count, SegArgs s0, SegArgs s1,
    float eps2x2, int C) {
  __shared__ uint4 la[2 * kPackTile];
  __shared__ float4 lt[kPackTile];
  const bool split = s0.part != nullptr;
  const int b = split ? flat_block() / C : flat_block();
  const int c0 = split ? flat_block() % C : 0;
  const bool first = b < s0.nblocks;
  const SegArgs& sg = pick(s0, s1, first);
  const int blk = first ? b : b - s0.nblocks;
  mfma16_chunks<EPS>(src, *count, sg, blk, c0, C, eps2x2, la, lt);
}

// ------------------------------------------------------ stream function ---
// psi_i = sum_j s_j log(1 - x_i.y_j): a block of four waves owns 64 targets and
// one of C source chunks, as the wave-split velocity sums (bve_device.hpp:
// scalar-loaded sources {y, s}, quarters of a chunk per wave).
// What bounds it: FP64 issue, 17 FP64 and 8 32-bit operations per pair (27 and
// LDS-staged sources before).

// Quads [qa, qb): K += s k, R += s (rest of the log); CHECK drops source self.
template <bool CHECK>
__device__ __forceinline__ void psi_quads(const double4* __restrict__ src,
                                          int qa, int qb, const double* x,
                                          int self, const double2* ltab,
                                          double& K, double& R,
                                          uint32_t& top) {
#pragma unroll 1
  for (int q = qa; q < qb; ++q) {
    double4 y[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = src[4 * q + j];
    double d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      d[j] = __builtin_fma(
          -x[2], y[j].z,
          __builtin_fma(-x[1], y[j].y, __builtin_fma(-x[0], y[j].x, 1.0)));
      if (CHECK && 4 * q + j == self) d[j] = 1.0;  // log 1 = 0
      top = max(top, log_screen(d[j]));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      double k;
      const double v = log_part(d[j], ltab, k);
      K = __builtin_fma(y[j].w, k, K);
      R = __builtin_fma(y[j].w, v, R);
    }
  }
}

// The same, pair by pair with the library log (zero, negative, infinite and
// NaN arguments).
__device__ __forceinline__ double psi_redo(const double4* __restrict__ src,
                                           int qa, int qb, const double* x,
                                           int self) {
  double psi = 0.0;
#pragma unroll 1
  for (int j = 4 * qa; j < 4 * qb; ++j) {
    const double4 y = src[j];
    const double d = __builtin_fma(
        -x[2], y.z, __builtin_fma(-x[1], y.y, __builtin_fma(-x[0], y.x, 1.0)));
    const double v = y.w * log(d);
    psi += j == self ? 0.0 : v;
  }
  return psi;
}

// With partial sums, block b * C + k sums source chunk k of target block b into
// sg.part[k pstride + c]; without, block b adds every chunk in order.
__global__ __launch_bounds__(256) void bve_psi_kernel(
    const double4* __restrict__ src, const double2* __restrict__ table,
    const int32_t* __restrict__ count, SegArgs s0, SegArgs s1, int C) {
  __shared__ double2 ltab[kLogTable];
  __shared__ double red[4][64];
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
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t c = slot0 + lane;
  double x[3];
  int self;
  const int64_t i = lane_target(sg, c, c < n_live, x, &self);
  int lo, hi;
  wave_self_range<1>(&self, &lo, &hi);
  __syncthreads();
  double tot = 0.0;
#pragma unroll 1
  for (int k = c0; k < (split ? c0 + 1 : C); ++k) {
    int q0, q1;
    wave_range(nq, k, C, w, &q0, &q1);
    double S = 0.0;
#pragma unroll 1
    for (int q = q0; q < q1; q += kWaveTile) {
      const int e = min(q + kWaveTile, q1);
      double K = 0.0, R = 0.0;
      uint32_t top = 0;
      if (lo < 4 * e && hi >= 4 * q)
        psi_quads<true>(src, q, e, x, self, ltab, K, R, top);
      else
        psi_quads<false>(src, q, e, x, self, ltab, K, R, top);
      double T = __builtin_fma(K, kLn2, R);
      if (__ballot(top >= kLogScreen)) {
        const double redo = psi_redo(src, q, e, x, self);
        T = top >= kLogScreen ? redo : T;
      }
      S += T;
    }
    if (k > c0) __syncthreads();  // the previous chunk's sums are read
    red[w][lane] = S;
    __syncthreads();
    if (w == 0) tot += ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
  }
  if (w != 0 || c >= n_live) return;
  if (split)
    sg.part[c0 * sg.pstride + c] = tot;
  else if (!(sg.skip && sg.skip[i]))
    sg.out_scalar[i] = tot;
}

// psi = the ks chunk partials added in chunk order, at every live slot.
__global__ __launch_bounds__(256) void bve_psi_reduce_kernel(SegArgs s0,
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
  double psi = 0.0;
#pragma unroll 8
  for (int k = 0; k < ks; ++k) psi += sg.part[k * sg.pstride + c];
  sg.out_scalar[i] = psi;
}

__global__ __launch_bounds__(256) void finite_kernel(
    const double* __restrict__ base, int64_t n, int64_t es, int64_t cs,
    int ncomp, int32_t* __restrict__ flag) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  bool bad = false;
  for (int k = 0; k < ncomp; ++k) bad |= !isfinite(base[i * es + k * cs]);
  if (bad) atomicOr(flag, 1);
}

__global__ void zero_int_kernel(int32_t* p) { *p = 0; }

// ------------------------------------------------------ kernel registry ---
using F64Kernel = void (*)(const double4*, const double4*, const int32_t*,
                          SegArgs, SegArgs, double);
using MixedKernel = void (*)(const float4*, const double4*, const int32_t*,
                             SegArgs, SegArgs, float);
using MfmaKernel = void (*)(MfmaSrc, const int32_t*, SegArgs, SegArgs, float);
using Mfma16Kernel = void (*)(Mfma16Src, const int32_t*, SegArgs, SegArgs,
                              float);

struct F64Variant {
  F64Kernel fn, fn_eps;
  int block, tpl;
  const char* name;
  bool sy = false;  // reads the packed s y
  int ksplit = 1;   // > 1: source-split kernel (needs the partial sums
  int twin = -1;    // workspace); twin: the same shape unsplit
  bool wave = false;  // wave-split kernel on quad records
};
struct MixedVariant {
  MixedKernel fn, fn_eps;  // vector-ALU kernels (or null)
  MfmaKernel mfn, mfn_eps; // matrix-core kernels (or null)
  int block, tpl;
  const char* name;
  Mfma16Kernel m16, m16_eps;  // f16-split matrix-core kernels (or null)
  int ksplit = 1;  // > 1: source-split kernel (partial sums workspace);
  int twin = -1;   // twin: the same shape unsplit
  bool chunked = false;  // chunk count by mixed_chunks
};

#define LPM_F64_VARIANT(B, T, NR, PAIR)                                  \
  {bve_vel_f64_kernel<B, T, 256, false, NR, PAIR>,                      \
   bve_vel_f64_kernel<B, T, 256, true, NR, PAIR>, B, T,                 \
   "block" #B "_tpl" #T "_nr" #NR "_pair" #PAIR}
#define LPM_F64_FUSED(B, T, NR)                                          \
  {bve_vel_f64_kernel<B, T, 256, false, NR, true, true>,                \
   bve_vel_f64_kernel<B, T, 256, true, NR, true, true>, B, T,           \
   "block" #B "_tpl" #T "_nr" #NR "_pairtrue_fused"}
#define LPM_F64_QUAD(B, T, NR)                                           \
  {bve_vel_f64_kernel<B, T, 256, false, NR, true, true, true>,          \
   bve_vel_f64_kernel<B, T, 256, true, NR, true, true, true>, B, T,     \
   "block" #B "_tpl" #T "_nr" #NR "_quad_fused"}
#define LPM_F64_QUAD_SY(B, T, NR)                                        \
  {bve_vel_f64_kernel<B, T, 256, false, NR, true, true, true, true>,    \
   bve_vel_f64_kernel<B, T, 256, true, NR, true, true, true, true>, B, T, \
   "block" #B "_tpl" #T "_nr" #NR "_quad_fused_sy", true}
#define LPM_F64_QUAD_SY_U(B, T, NR, QU)                                   \
  {bve_vel_f64_kernel<B, T, 256, false, NR, true, true, true, true, QU>,  \
   bve_vel_f64_kernel<B, T, 256, true, NR, true, true, true, true, QU>,   \
   B, T, "block" #B "_tpl" #T "_nr" #NR "_quad_fused_sy_u" #QU, true}
#define LPM_F64_QUAD_SY_TILE(B, T, NR, TL, QU)                                 \
  {bve_vel_f64_kernel<B, T, TL, false, NR, true, true, true, true, QU>,        \
   bve_vel_f64_kernel<B, T, TL, true, NR, true, true, true, true, QU>, B, T,   \
   "block" #B "_tpl" #T "_nr" #NR "_quad_fused_sy_u" #QU "_tile" #TL, true}
// named as the twin (TAG: its tile suffix) + "_split" K
#define LPM_F64_QUAD_SY_SPLIT(B, T, NR, TL, TAG, QU, KS, TWIN)                  \
  {bve_vel_f64_split_kernel<B, T, TL, false, NR, true, true, true, true, QU, KS>, \
   bve_vel_f64_split_kernel<B, T, TL, true, NR, true, true, true, true, QU, KS>,  \
   B, T, "block" #B "_tpl" #T "_nr" #NR "_quad_fused_sy_u" #QU TAG "_split" #KS, \
   true, KS, TWIN}
#define LPM_MIXED_VARIANT(B, T, PAIR)                                     \
  {bve_vel_mixed_kernel<B, T, 256, false, PAIR>,                         \
   bve_vel_mixed_kernel<B, T, 256, true, PAIR>, nullptr, nullptr, B, T,  \
   "block" #B "_tpl" #T "_pair" #PAIR}

const F64Variant kF64Variants[] = {
    LPM_F64_VARIANT(256, 2, 2, false),  // 0: baseline loop
    LPM_F64_VARIANT(256, 2, 2, true),   // 1
    LPM_F64_VARIANT(256, 1, 2, true),   // 2
    LPM_F64_VARIANT(256, 4, 2, true),   // 3
    LPM_F64_VARIANT(128, 2, 2, true),   // 4
    LPM_F64_VARIANT(256, 2, 1, true),   // 5: one Newton step
    LPM_F64_VARIANT(256, 4, 1, true),   // 6
    LPM_F64_VARIANT(256, 1, 1, true),   // 7
    LPM_F64_FUSED(256, 2, 1),           // 8: 1 - x.y as one FMA chain
    LPM_F64_FUSED(256, 4, 1),           // 9
    LPM_F64_FUSED(256, 1, 1),           // 10
    LPM_F64_QUAD(256, 2, 1),            // 11: one reciprocal per 4 pairs
    LPM_F64_QUAD(256, 4, 1),            // 12
    LPM_F64_QUAD_SY(256, 2, 1),         // 13: weights from the packed s y
    LPM_F64_QUAD_SY(256, 4, 1),         // 14
    LPM_F64_QUAD_SY_U(256, 4, 1, 2),    // 15: two groups per iteration
    LPM_F64_QUAD_SY_U(256, 2, 1, 2),    // 16
    LPM_F64_QUAD_SY_U(256, 2, 1, 4),    // 17
    LPM_F64_QUAD_SY_TILE(256, 4, 1, 512, 2),   // 18: 512-source LDS tiles
    LPM_F64_QUAD_SY_TILE(256, 4, 1, 1024, 2),  // 19
    LPM_F64_QUAD_SY_TILE(256, 2, 1, 512, 2),   // 20
    // 21-25: the sources in 8 to 32 chunks per target block, partial
    // sums reduced in a second kernel (steps and init_velocity only; other
    // calls run the twin)
    LPM_F64_QUAD_SY_SPLIT(256, 4, 1, 1024, "_tile1024", 2, 8, 19),
    LPM_F64_QUAD_SY_SPLIT(256, 4, 1, 512, "_tile512", 2, 8, 18),
    LPM_F64_QUAD_SY_SPLIT(256, 4, 1, 512, "_tile512", 2, 16, 18),
    LPM_F64_QUAD_SY_SPLIT(256, 4, 1, 256, "", 2, 8, 15),
    LPM_F64_QUAD_SY_SPLIT(256, 4, 1, 512, "_tile512", 2, 32, 18),  // 25
    // 26: scalar-loaded sources divided among a block's waves (the default)
    {nullptr, nullptr, 256, 2, "wave4_scalar", false, 1, -1, true},
};
const MixedVariant kMixedVariants[] = {
    LPM_MIXED_VARIANT(256, 2, false),  // 0
    LPM_MIXED_VARIANT(256, 2, true),   // 1
    LPM_MIXED_VARIANT(256, 1, true),   // 2
    LPM_MIXED_VARIANT(256, 4, true),   // 3
    LPM_MIXED_VARIANT(128, 2, true),   // 4
    LPM_MIXED_VARIANT(256, 1, false),  // 5
    LPM_MIXED_VARIANT(256, 4, false),  // 6
    {nullptr, nullptr, bve_vel_mfma_kernel<false>, bve_vel_mfma_kernel<true>,
     256, 1, "mfma_block256_near3"},   // 7: matrix-core far field
    {nullptr, nullptr, nullptr, nullptr, 256, 1, "mfma16_block256_near3",
     bve_vel_mfma16_kernel<false>, bve_vel_mfma16_kernel<true>},  // 8: f16 split
    {nullptr, nullptr, nullptr, nullptr, 256, 1, "mfma16_occ5_block256_near3",
     bve_vel_mfma16_kernel<false, 5>, bve_vel_mfma16_kernel<true, 5>},  // 9
    {nullptr, nullptr, nullptr, nullptr, 256, 1,
     "mfma16_occ5_acc2_block256_near3", bve_vel_mfma16_kernel<false, 5, 2>,
     bve_vel_mfma16_kernel<true, 5, 2>},                                 // 10
    // 11-13: variant 10 with the sources in 2 to 8 chunks per target
    // block (steps and init_velocity only; other calls run variant 10)
    {nullptr, nullptr, nullptr, nullptr, 256, 1,
     "mfma16_occ5_acc2_block256_near3_split2",
     bve_vel_mfma16_split_kernel<false, 5, 2, 2>,
     bve_vel_mfma16_split_kernel<true, 5, 2, 2>, 2, 10},                // 11
    {nullptr, nullptr, nullptr, nullptr, 256, 1,
     "mfma16_occ5_acc2_block256_near3_split4",
     bve_vel_mfma16_split_kernel<false, 5, 2, 4>,
     bve_vel_mfma16_split_kernel<true, 5, 2, 4>, 4, 10},                // 12
    {nullptr, nullptr, nullptr, nullptr, 256, 1,
     "mfma16_occ5_acc2_block256_near3_split8",
     bve_vel_mfma16_split_kernel<false, 5, 2, 8>,
     bve_vel_mfma16_split_kernel<true, 5, 2, 8>, 8, 10},                // 13
    // 14-18: variants 10 (and its 8-chunk split) and 9 with one reciprocal
    // per two (prcp) or four (qrcp) distances
    {nullptr, nullptr, nullptr, nullptr, 256, 1,
     "mfma16_occ5_acc2_prcp_block256_near3",
     bve_vel_mfma16_kernel<false, 5, 2, 2>,
     bve_vel_mfma16_kernel<true, 5, 2, 2>},                              // 14
    {nullptr, nullptr, nullptr, nullptr, 256, 1,
     "mfma16_occ5_acc2_prcp_block256_near3_split8",
     bve_vel_mfma16_split_kernel<false, 5, 2, 8, 2>,
     bve_vel_mfma16_split_kernel<true, 5, 2, 8, 2>, 8, 14},             // 15
    {nullptr, nullptr, nullptr, nullptr, 256, 1,
     "mfma16_occ5_acc2_qrcp_block256_near3",
     bve_vel_mfma16_kernel<false, 5, 2, 4>,
     bve_vel_mfma16_kernel<true, 5, 2, 4>},                              // 16
    {nullptr, nullptr, nullptr, nullptr, 256, 1,
     "mfma16_occ5_acc2_qrcp_block256_near3_split8",
     bve_vel_mfma16_split_kernel<false, 5, 2, 8, 4>,
     bve_vel_mfma16_split_kernel<true, 5, 2, 8, 4>, 8, 16},             // 17
    {nullptr, nullptr, nullptr, nullptr, 256, 1,
     "mfma16_occ5_qrcp_block256_near3",
     bve_vel_mfma16_kernel<false, 5, 1, 4>,
     bve_vel_mfma16_kernel<true, 5, 1, 4>},                              // 18
    // 19: variant 16 with the sources in chunks by the problem's sizes (the
    // default)
    {nullptr, nullptr, nullptr, nullptr, 256, 1, "mfma16_chunked_near3",
     nullptr, nullptr, 1, -1, true},
};
constexpr int kNumF64 = sizeof(kF64Variants) / sizeof(kF64Variants[0]);
constexpr int kNumMixed = sizeof(kMixedVariants) / sizeof(kMixedVariants[0]);
// Variants used until the autotuner (or the caller) picks another one.  The
// wave-split kernel is the fastest FP64 shape from 2e6 pairs (L3: 8 us
// against 93 us for variant 1) to 1.6e11 (45 ms; variant 25 48.5, variant 1
// 70).  The others keep their numbers: saved tuning tables hold them.
constexpr int kDefaultF64 = 26;
// The mixed default is the matrix-core kernel: 1.71 ms per level-6 evaluation
// against 5.67 for the vector form of variant 0, with a smaller error (tile
// offsets from the centroid); 23 against 36 us at level 1.
constexpr int kDefaultMixed = 19;

}  // namespace

int variant_count(int family) {
  if (family == KID_BVE_VEL_F64) return kNumF64;
  if (family == KID_BVE_VEL_MIXED) return kNumMixed;
  if (family == KID_BVE_ENS_F64 || family == KID_BVE_ENS_MIXED)
    return ens_variant_count(family);
  if (family == KID_SWE_F64 || family == KID_SWE_MIXED)
    return swe_variant_count(family);
  return 0;
}

const char* variant_name(int family, int v) {
  if (v < 0 || v >= variant_count(family)) return nullptr;
  if (family == KID_BVE_ENS_F64 || family == KID_BVE_ENS_MIXED)
    return ens_variant_name(family, v);
  if (family == KID_SWE_F64 || family == KID_SWE_MIXED)
    return swe_variant_name(family, v);
  return family == KID_BVE_VEL_F64 ? kF64Variants[v].name
                                   : kMixedVariants[v].name;
}

int default_variant(int family) {
  if (family == KID_BVE_ENS_F64 || family == KID_BVE_ENS_MIXED)
    return ens_default_variant(family);
  if (family == KID_SWE_F64 || family == KID_SWE_MIXED)
    return swe_default_variant(family);
  return family == KID_BVE_VEL_F64 ? kDefaultF64 : kDefaultMixed;
}

namespace {

SegArgs to_args(const TargetSeg& t, int per_block) {
  SegArgs a{};
  a.x = t.x.base;
  a.es = t.x.es;
  a.cs = t.x.cs;
  a.n = t.n;
  a.index = t.index;
  a.d_n = t.d_n;
  a.self_rank = t.self_rank;
  a.self_identity = t.self_identity ? 1 : 0;
  a.nblocks = static_cast<int>((t.n + per_block - 1) / per_block);
  a.skip = t.skip;
  a.out = t.out.base;
  a.oes = t.out.es;
  a.ocs = t.out.cs;
  a.out_scalar = t.out_scalar;
  a.pstride = t.n;
  return a;
}

double count_pairs(const TargetSeg* segs, int nseg, int64_t nsrc_upper) {
  double p = 0;
  for (int s = 0; s < nseg; ++s) p += static_cast<double>(segs[s].n);
  return p * static_cast<double>(nsrc_upper);
}

}  // namespace

// --------------------------------------------------------------- hosts ---
RankMap build_rank_into(const RankWs& ws, const uint8_t* mask, int64_t n,
                        hipStream_t s) {
  LPM_ARG_CHECK(n >= 0 && n < (int64_t(1) << 31), "source count out of range");
  RankMap map;
  map.n = n;
  if (!mask) {
    set_count_kernel<<<1, 1, 0, s>>>(ws.count_ident, static_cast<int32_t>(n));
    LPM_HIP_CHECK(hipGetLastError());
    map.d_count = ws.count_ident;
    return map;
  }
  const int nb = static_cast<int>((n + kScanChunk - 1) / kScanChunk);
  if (nb > 0 && n <= kScanOneLaunch &&
      reinterpret_cast<uintptr_t>(mask) % 16 == 0) {
    mask_scan_kernel<<<nb, kScanBlock, 0, s>>>(mask, n, ws.counts, ws.rank,
                                               ws.inv);
    LPM_HIP_CHECK(hipGetLastError());
    map.rank = ws.rank;
    map.inv = ws.inv;
    map.d_count = ws.counts + nb;
    return map;
  }
  if (nb > 0) {
    mask_count_kernel<<<nb, kScanBlock, 0, s>>>(mask, n, ws.counts);
    LPM_HIP_CHECK(hipGetLastError());
  }
  scan_counts_kernel<<<1, 1024, 0, s>>>(ws.counts, nb);
  LPM_HIP_CHECK(hipGetLastError());
  if (nb > 0) {
    mask_rank_kernel<<<nb, kScanBlock, 0, s>>>(mask, n, ws.counts, ws.rank,
                                               ws.inv);
    LPM_HIP_CHECK(hipGetLastError());
  }
  map.rank = ws.rank;
  map.inv = ws.inv;
  map.d_count = ws.counts + nb;
  return map;
}

RankWs rank_workspace(lpm_ctx* ctx, const uint8_t* mask, int64_t n) {
  LPM_ARG_CHECK(n >= 0 && n < (int64_t(1) << 31), "source count out of range");
  RankWs ws;
  if (!mask) {
    ws.count_ident =
        static_cast<int32_t*>(ctx->count_ident.ensure(sizeof(int32_t)));
  } else {
    const int nb = static_cast<int>((n + kScanChunk - 1) / kScanChunk);
    ws.counts = static_cast<int32_t*>(
        ctx->block_counts.ensure(sizeof(int32_t) * (nb + 1)));
    const size_t nn = sizeof(int32_t) * std::max<int64_t>(n, 1);
    ws.rank = static_cast<int32_t*>(ctx->rank.ensure(nn));
    ws.inv = static_cast<int32_t*>(ctx->inv.ensure(nn));
  }
  return ws;
}

RankMap build_rank(lpm_ctx* ctx, const uint8_t* mask, int64_t n,
                   hipStream_t s) {
  return build_rank_into(rank_workspace(ctx, mask, n), mask, n, s);
}

TargetSeg face_targets(CrdIn x, const RankMap& map, const uint8_t* mask,
                       bool skip_masked, CrdOut out, double* out_scalar) {
  TargetSeg t;
  t.x = x;
  t.n = map.n;
  t.out = out;
  t.out_scalar = out_scalar;
  if (skip_masked && mask) {
    // live slots are the packed faces; slot c is its own source c
    t.index = map.inv;
    t.d_n = map.d_count;
    t.self_identity = true;
  } else if (map.rank) {
    t.self_rank = map.rank;
  } else {
    t.self_identity = true;
  }
  return t;
}

PackedSources pack_sources_into(const PackWs& ws, unsigned layouts, CrdIn sx,
                                const double* zeta, const double* area,
                                const RankMap& map, int precision,
                                hipStream_t s) {
  PackedSources ps;
  const int64_t n = map.n;
  ps.count = map.d_count;
  ps.capacity = n;
  const int64_t cap = std::max<int64_t>(n, 1);
  const bool sy = precision == LPM_FP64 && (layouts & kLayoutSy);
  if (layouts & kLayoutQuad) {
    LPM_ARG_CHECK(ws.quad, "packing buffers missing");
    if (n > 0) {
      pack_quad_kernel<<<static_cast<int>((n + 3 + 255) / 256), 256, 0, s>>>(
          sx.base, sx.es, sx.cs, zeta, area, map.inv, map.d_count, ws.quad);
      LPM_HIP_CHECK(hipGetLastError());
    }
    ps.quad = ws.quad;
    if (layouts == kLayoutQuad) return ps;
  }
  if (layouts & kLayoutRec) {
    LPM_ARG_CHECK(ws.rec, "packing buffers missing");
    if (n > 0) {
      pack_rec_kernel<<<static_cast<int>((n + 3 + 255) / 256), 256, 0, s>>>(
          sx.base, sx.es, sx.cs, zeta, area, map.inv, map.d_count, ws.rec);
      LPM_HIP_CHECK(hipGetLastError());
    }
    ps.rec = ws.rec;
    if (layouts == kLayoutRec) return ps;
  }
  if ((layouts & ~kLayoutLog) == kLayoutMfma16) {
    // the matrix-core records straight from the faces, one launch
    LPM_ARG_CHECK(ws.mf_y && ws.mf_s && ws.mf_c && ws.mf_a && ws.mf_t32 &&
                      ws.mf_is && (ws.mf_g || !(layouts & kLayoutLog)),
                  "packing buffers missing");
    Mfma16Out o{ws.mf_y,   ws.mf_s,  ws.mf_c, ws.mf_a,
                ws.mf_t32, ws.mf_is, ws.mf_g};
    const int tiles = static_cast<int>((cap + kPackTile - 1) / kPackTile);
    pack_mfma16_faces_kernel<<<tiles, kPackTile, 0, s>>>(
        sx.base, sx.es, sx.cs, zeta, area, map.inv, map.d_count, o);
    LPM_HIP_CHECK(hipGetLastError());
    ps.mf_y = ws.mf_y;
    ps.mf_s = ws.mf_s;
    ps.mf_c = ws.mf_c;
    ps.mf_a = ws.mf_a;
    ps.mf_t32 = ws.mf_t32;
    ps.mf_is = ws.mf_is;
    ps.mf_g = ws.mf_g;
    return ps;
  }
  LPM_ARG_CHECK(ws.p64 && (!sy || ws.psy), "packing buffers missing");
  if (n > 0) {
    pack_f64_kernel<<<static_cast<int>((n + 3 + 255) / 256), 256, 0, s>>>(
        sx.base, sx.es, sx.cs, zeta, area, map.inv, map.d_count, ws.p64,
        sy ? ws.psy : nullptr);
    LPM_HIP_CHECK(hipGetLastError());
  }
  ps.data = ws.p64;
  ps.sy = sy ? ws.psy : nullptr;
  if (precision != LPM_MIXED) return ps;
  const int ntile = static_cast<int>((cap + kPackTile - 1) / kPackTile);
  if (layouts & kLayoutVec32) {
    LPM_ARG_CHECK(ws.p32 && ws.centers, "packing buffers missing");
    pack_mixed_kernel<<<ntile, kPackTile, 0, s>>>(ws.p64, map.d_count, ws.p32,
                                                  ws.centers);
    LPM_HIP_CHECK(hipGetLastError());
    ps.data = ws.p32;
    ps.centers = ws.centers;
  }
  if (layouts & kLayoutMfma) {
    LPM_ARG_CHECK(ws.mf_y && ws.mf_s && ws.mf_c && ws.mf_q && ws.mf_t,
                  "packing buffers missing");
    pack_mfma_kernel<<<ntile, kPackTile, 0, s>>>(ws.p64, map.d_count, ws.mf_y,
                                                 ws.mf_q, ws.mf_s, ws.mf_t,
                                                 ws.mf_c);
    LPM_HIP_CHECK(hipGetLastError());
    ps.mf_y = ws.mf_y;
    ps.mf_s = ws.mf_s;
    ps.mf_c = ws.mf_c;
    ps.mf_q = ws.mf_q;
    ps.mf_t = ws.mf_t;
  }
  return ps;
}

PackWs pack_workspace(lpm_ctx* ctx, int64_t n, int precision) {
  const int64_t cap = std::max<int64_t>(n, 1);
  const int64_t ntile = (cap + kPackTile - 1) / kPackTile;
  const int64_t tcap = ntile * kPackTile;
  PackWs ws;
  auto buf = [](DevBuf& b, auto*& p, int64_t count) {
    p = static_cast<std::remove_reference_t<decltype(p)>>(
        b.ensure(sizeof(*p) * count));
  };
  buf(ctx->packed64, ws.p64, (cap + 3) / 4 * 4);
  if (precision == LPM_FP64) {
    buf(ctx->quad, ws.rec, (cap + 3) / 4 * 32);
    ws.quad = ws.rec;
    buf(ctx->packed64sy, ws.psy, cap);
    return ws;
  }
  buf(ctx->packed32, ws.p32, cap);
  buf(ctx->centers, ws.centers, ntile);
  buf(ctx->mf_y, ws.mf_y, tcap);
  buf(ctx->mf_s, ws.mf_s, tcap);
  buf(ctx->mf_c, ws.mf_c, ntile);
  buf(ctx->mf_q, ws.mf_q, tcap);
  buf(ctx->mf_t, ws.mf_t, 4 * tcap);
  buf(ctx->mf_a, ws.mf_a, 2 * tcap);
  buf(ctx->mf_t32, ws.mf_t32, 4 * tcap);
  buf(ctx->mf_is, ws.mf_is, ntile);
  buf(ctx->mf_g, ws.mf_g, ntile);
  return ws;
}

PackedSources pack_sources(lpm_ctx* ctx, unsigned layouts, CrdIn sx,
                           const double* zeta, const double* area,
                           const RankMap& map, int precision, hipStream_t s) {
  return pack_sources_into(pack_workspace(ctx, map.n, precision),
                           layouts, sx, zeta, area, map, precision, s);
}

int bve_velocity_variant(lpm_ctx* ctx, int precision, int64_t n_targets) {
  return pick_variant(
      ctx, precision == LPM_MIXED ? KID_BVE_VEL_MIXED : KID_BVE_VEL_F64,
      n_targets);
}

unsigned bve_variant_layouts(int precision, int variant) {
  if (precision == LPM_FP64) {
    LPM_ARG_CHECK(variant >= 0 && variant < kNumF64, "variant out of range");
    if (kF64Variants[variant].wave) return kLayoutQuad;
    return kF64Variants[variant].sy ? kLayoutSy : 0u;
  }
  LPM_ARG_CHECK(variant >= 0 && variant < kNumMixed, "variant out of range");
  const MixedVariant& v = kMixedVariants[variant];
  if (v.m16 || v.chunked) return kLayoutMfma16;
  if (v.mfn) return kLayoutMfma;
  return kLayoutVec32;
}

namespace {

// Chunks per target block of a variant (1: not source-split) and its
// unsplit twin.
int split_of(int precision, int variant, int* twin) {
  if (precision == LPM_FP64 && variant >= 0 && variant < kNumF64) {
    *twin = kF64Variants[variant].twin;
    return kF64Variants[variant].ksplit;
  }
  if (precision == LPM_MIXED && variant >= 0 && variant < kNumMixed) {
    *twin = kMixedVariants[variant].twin;
    return kMixedVariants[variant].ksplit;
  }
  *twin = -1;
  return 1;
}

}  // namespace

bool bve_variant_chunked(int precision, int variant) {
  if (precision == LPM_FP64)
    return variant >= 0 && variant < kNumF64 && kF64Variants[variant].wave;
  return variant >= 0 && variant < kNumMixed && kMixedVariants[variant].chunked;
}

size_t bve_split_bytes(int precision, int variant, int64_t n_targets,
                       int64_t n_src) {
  int twin;
  int ks = split_of(precision, variant, &twin);
  if (bve_variant_chunked(precision, variant))
    ks = precision == LPM_FP64 ? wave_chunks(n_targets, n_src)
                               : mixed_chunks(n_targets, n_src);
  if (ks <= 1) return 0;
  return sizeof(double) * 3 * static_cast<size_t>(ks) *
         static_cast<size_t>(std::max<int64_t>(n_targets, 1));
}

double* split_workspace(lpm_ctx* ctx, size_t need, hipStream_t s) {
  if (ctx->split_part.bytes >= need) return ctx->split_part.as<double>();
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  LPM_HIP_CHECK(hipStreamIsCapturing(s, &cs));
  if (cs != hipStreamCaptureStatusNone) return nullptr;
  try {
    return static_cast<double*>(ctx->split_part.ensure(need));
  } catch (const Error& e) {
    if (e.code != LPM_ERR_NOMEM) throw;
    (void)hipGetLastError();  // the failed hipMalloc's error is handled
    return nullptr;
  }
}

double* chunk_workspace(lpm_ctx* ctx, size_t need, hipStream_t s) {
  return need <= kChunkBytes ? split_workspace(ctx, need, s) : nullptr;
}

namespace {

void launch_split_reduce(const SegArgs& a0, const SegArgs& a1, int ks,
                         hipStream_t s) {
  const int64_t nt = a0.n + a1.n;
  hipLaunchKernelGGL(bve_split_reduce_kernel,
                     dim3(static_cast<unsigned>((nt + 255) / 256)), dim3(256),
                     0, s, a0, a1, ks);
  LPM_HIP_CHECK(hipGetLastError());
}

// The wave-split kernel: one target per lane while two would give fewer than
// four blocks per CU (1,922 x 1,280 pairs: 5.9 us against 6.5), else two
// (four measured the same and hold fewer waves).
void launch_wave_f64(lpm_ctx* ctx, const PackedSources& src,
                     const TargetSeg& t0, const TargetSeg& t1, double eps2,
                     double* part, size_t part_bytes, hipStream_t s,
                     bool reduce) {
  LPM_ARG_CHECK(src.quad, "quad records not packed");
  const int64_t nt = t0.n + t1.n;
  const int C = wave_chunks(nt, src.capacity);
  const size_t need = sizeof(double) * 3 * static_cast<size_t>(C) * nt;
  const bool split = C > 1 && part && need <= part_bytes;
  const int tpl = (nt + 127) / 128 * C >= 4 * ctx->num_cus ? 2 : 1;
  SegArgs a0 = to_args(t0, 64 * tpl), a1 = to_args(t1, 64 * tpl);
  if (split) {
    a0.part = part;
    a1.part = part + 3 * static_cast<int64_t>(C) * t0.n;
  }
  const dim3 grid = launch_grid(
      (static_cast<int64_t>(a0.nblocks) + a1.nblocks) * (split ? C : 1), 256);
  const bool mesh = t0.mesh && (t1.n == 0 || t1.mesh);
  const auto pick_kernel = [&](auto t) {
    constexpr int T = decltype(t)::value;
    return eps2 > 0 ? bve_wave_f64_kernel<T, true, false>
           : mesh   ? bve_wave_f64_kernel<T, false, true>
                    : bve_wave_f64_kernel<T, false, false>;
  };
  const auto kernel = tpl == 2 ? pick_kernel(std::integral_constant<int, 2>{})
                               : pick_kernel(std::integral_constant<int, 1>{});
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, src.quad, src.count, a0,
                     a1, eps2, C);
  LPM_HIP_CHECK(hipGetLastError());
  if (split && reduce) {
    hipLaunchKernelGGL(bve_wave_reduce_kernel,
                       dim3(static_cast<unsigned>((nt + 255) / 256)),
                       dim3(256), 0, s, a0, a1, C);
    LPM_HIP_CHECK(hipGetLastError());
  }
}

void launch_mixed_chunked(lpm_ctx*, const PackedSources& src,
                          const TargetSeg& t0, const TargetSeg& t1,
                          double eps2, double* part, size_t part_bytes,
                          hipStream_t s, bool reduce) {
  LPM_ARG_CHECK(src.mf_a, "matrix-core layout not packed");
  const int64_t nt = t0.n + t1.n;
  const int C = mixed_chunks(nt, src.capacity);
  const size_t need = sizeof(double) * 3 * static_cast<size_t>(C) * nt;
  const bool split = C > 1 && part && need <= part_bytes;
  SegArgs a0 = to_args(t0, 256), a1 = to_args(t1, 256);
  if (split) {
    a0.part = part;
    a1.part = part + 3 * static_cast<int64_t>(C) * t0.n;
  }
  Mfma16Src m{src.mf_y, src.mf_s, src.mf_a, src.mf_t32, src.mf_c, src.mf_is,
              nullptr};
  hipLaunchKernelGGL(eps2 > 0 ? bve_vel_mfma16_chunk_kernel<true>
                              : bve_vel_mfma16_chunk_kernel<false>,
                     launch_grid((static_cast<int64_t>(a0.nblocks) +
                                  a1.nblocks) * (split ? C : 1), 256),
                     dim3(256), 0, s, m, src.count, a0, a1,
                     static_cast<float>(2.0 * eps2), C);
  LPM_HIP_CHECK(hipGetLastError());
  if (split && reduce) {
    hipLaunchKernelGGL(bve_wave_reduce_kernel,
                       dim3(static_cast<unsigned>((nt + 255) / 256)),
                       dim3(256), 0, s, a0, a1, C);
    LPM_HIP_CHECK(hipGetLastError());
  }
}

}  // namespace

ChunkSums launch_bve_chunks(lpm_ctx* ctx, const PackedSources& src,
                            const TargetSeg* segs, double eps2, int precision,
                            int variant, double* part, hipStream_t s) {
  const TargetSeg &t0 = segs[0], &t1 = segs[1];
  const int64_t nt = t0.n + t1.n;
  const size_t bytes = bve_split_bytes(precision, variant, nt, src.capacity);
  LPM_ARG_CHECK(bve_variant_chunked(precision, variant) && bytes && part,
                "not a launch in chunks");
  const bool f64 = precision == LPM_FP64;
  TimedLaunch tl(ctx, f64 ? KID_BVE_VEL_F64 : KID_BVE_VEL_MIXED, s,
                 count_pairs(segs, 2, src.capacity));
  (f64 ? launch_wave_f64 : launch_mixed_chunked)(ctx, src, t0, t1, eps2, part,
                                                 bytes, s, false);
  ChunkSums r;
  r.C = f64 ? wave_chunks(nt, src.capacity) : mixed_chunks(nt, src.capacity);
  r.part[0] = part;
  r.part[1] = part + 3 * static_cast<int64_t>(r.C) * t0.n;
  r.stride[0] = t0.n;
  r.stride[1] = t1.n;
  return r;
}

void launch_bve_velocity(lpm_ctx* ctx, const PackedSources& src,
                         TargetSeg* segs, int nseg, double eps2, int precision,
                         hipStream_t s, int variant, bool timed,
                         bool allow_split, double* part, size_t part_bytes) {
  LPM_ARG_CHECK(nseg >= 1 && nseg <= 2, "one or two target segments");
  TargetSeg empty;
  const TargetSeg& t0 = segs[0];
  const TargetSeg& t1 = nseg > 1 ? segs[1] : empty;
  for (int k = 0; k < nseg; ++k)
    LPM_ARG_CHECK(segs[k].n >= 0 && segs[k].n < (int64_t(1) << 31),
                  "target count out of range");
  if (t0.n + t1.n == 0) return;
  const double pairs = count_pairs(segs, nseg, src.capacity);
  LPM_ARG_CHECK(precision == LPM_FP64 || precision == LPM_MIXED,
                "unknown precision");
  if (variant < 0) variant = bve_velocity_variant(ctx, precision, t0.n + t1.n);
  LPM_ARG_CHECK(variant >= 0 && variant < (precision == LPM_FP64 ? kNumF64
                                                                  : kNumMixed),
                "variant out of range");
  if (bve_variant_chunked(precision, variant)) {
    const size_t need =
        bve_split_bytes(precision, variant, t0.n + t1.n, src.capacity);
    if (!part && timed && need) {
      part = chunk_workspace(ctx, need, s);
      part_bytes = part ? need : 0;
    }
    const bool f64 = precision == LPM_FP64;
    TimedLaunch tl(ctx,
                   !timed ? -1 : f64 ? KID_BVE_VEL_F64 : KID_BVE_VEL_MIXED, s,
                   pairs);
    (f64 ? launch_wave_f64 : launch_mixed_chunked)(ctx, src, t0, t1, eps2,
                                                   part, part_bytes, s, true);
    return;
  }
  part = nullptr;
  int twin = -1;
  if (split_of(precision, variant, &twin) > 1) {
    // the partial sums live in a context workspace: a step's prepare sizes
    // it before capture; a call that may not allocate it (no permission,
    // capture with it too small, or no memory for it) runs the unsplit twin
    if (allow_split)
      part = split_workspace(
          ctx,
          bve_split_bytes(precision, variant, t0.n + t1.n, src.capacity), s);
    if (!part) variant = twin;
  }
  if (precision == LPM_FP64) {
    const F64Variant& v = kF64Variants[variant];
    const int per = v.block * v.tpl;
    SegArgs a0 = to_args(t0, per), a1 = to_args(t1, per);
    const int grid = a0.nblocks + a1.nblocks;
    LPM_ARG_CHECK(!v.sy || src.sy, "packed s y missing for the FP64 variant");
    LPM_ARG_CHECK(v.ksplit == 1 || part, "split workspace missing");
    TimedLaunch tl(ctx, timed ? KID_BVE_VEL_F64 : -1, s, pairs);
    if (part) {
      a0.part = part;
      a1.part = part + 3 * static_cast<int64_t>(v.ksplit) * t0.n;
    }
    hipLaunchKernelGGL(eps2 > 0 ? v.fn_eps : v.fn,
                       dim3(static_cast<unsigned>(grid) * v.ksplit),
                       dim3(v.block), 0, s,
                       static_cast<const double4*>(src.data), src.sy, src.count,
                       a0, a1, eps2);
    LPM_HIP_CHECK(hipGetLastError());
    if (part) launch_split_reduce(a0, a1, v.ksplit, s);
  } else if (precision == LPM_MIXED) {
    const MixedVariant& v = kMixedVariants[variant];
    const int per = v.block * v.tpl;
    SegArgs a0 = to_args(t0, per), a1 = to_args(t1, per);
    const int grid = a0.nblocks + a1.nblocks;
    TimedLaunch tl(ctx, timed ? KID_BVE_VEL_MIXED : -1, s, pairs);
    if (v.m16) {
      LPM_ARG_CHECK(src.mf_a, "matrix-core layout not packed");
      LPM_ARG_CHECK(v.ksplit == 1 || part, "split workspace missing");
      Mfma16Src m{src.mf_y, src.mf_s, src.mf_a, src.mf_t32, src.mf_c, src.mf_is,
              nullptr};
      if (part) {
        a0.part = part;
        a1.part = part + 3 * static_cast<int64_t>(v.ksplit) * t0.n;
      }
      hipLaunchKernelGGL(eps2 > 0 ? v.m16_eps : v.m16,
                         dim3(static_cast<unsigned>(grid) * v.ksplit),
                         dim3(v.block), 0, s, m, src.count, a0, a1,
                         static_cast<float>(2.0 * eps2));
      LPM_HIP_CHECK(hipGetLastError());
      if (part) launch_split_reduce(a0, a1, v.ksplit, s);
    } else if (v.mfn) {
      LPM_ARG_CHECK(src.mf_y, "matrix-core layout not packed");
      MfmaSrc m{src.mf_y, src.mf_q, src.mf_s, src.mf_t, src.mf_c};
      hipLaunchKernelGGL(eps2 > 0 ? v.mfn_eps : v.mfn, dim3(grid),
                         dim3(v.block), 0, s, m, src.count, a0, a1,
                         static_cast<float>(2.0 * eps2));
    } else {
      LPM_ARG_CHECK(src.centers, "mixed vector layout not packed");
      hipLaunchKernelGGL(eps2 > 0 ? v.fn_eps : v.fn, dim3(grid), dim3(v.block),
                         0, s, static_cast<const float4*>(src.data),
                         src.centers, src.count, a0, a1,
                         static_cast<float>(2.0 * eps2));
    }
    LPM_HIP_CHECK(hipGetLastError());
  } else {
    throw Error(LPM_ERR_ARG, "unknown precision");
  }
}

void launch_bve_stream_fn(lpm_ctx* ctx, const PackedSources& src,
                          TargetSeg* segs, int nseg, hipStream_t s) {
  TargetSeg empty;
  const TargetSeg& t0 = segs[0];
  const TargetSeg& t1 = nseg > 1 ? segs[1] : empty;
  const int64_t nt = t0.n + t1.n;
  if (nt == 0) return;
  SegArgs a0 = to_args(t0, 64), a1 = to_args(t1, 64);
  const int64_t blocks = static_cast<int64_t>(a0.nblocks) + a1.nblocks;
  const int C = log_chunks(nt, src.capacity);
  // one chunk, or no workspace (a caller's capture, no memory): whole blocks
  double* part =
      C > 1 ? chunk_workspace(ctx, sizeof(double) * static_cast<size_t>(C) * nt,
                              s)
            : nullptr;
  if (part) {
    a0.part = part;
    a1.part = part + static_cast<int64_t>(C) * t0.n;
  }
  TimedLaunch tl(ctx, KID_BVE_PSI, s, count_pairs(segs, nseg, src.capacity));
  hipLaunchKernelGGL(bve_psi_kernel,
                     launch_grid(blocks * (part ? C : 1), 256), dim3(256), 0, s,
                     static_cast<const double4*>(src.data),
                     ctx->log_table.as<double2>(), src.count, a0, a1, C);
  LPM_HIP_CHECK(hipGetLastError());
  if (part) {
    hipLaunchKernelGGL(bve_psi_reduce_kernel,
                       dim3(static_cast<unsigned>((nt + 255) / 256)),
                       dim3(256), 0, s, a0, a1, C);
    LPM_HIP_CHECK(hipGetLastError());
  }
}

void make_log_table(lpm_ctx* ctx) {
  std::vector<double> t(2 * kLogTable);
  for (int j = 0; j < kLogTable; ++j) {
    double c = 2.0 / (1.0 + (j + 0.5) / kLogTable);
    if (j == 0) c = 2.0;
    if (j == kLogTable - 1) c = 1.0;
    t[2 * j] = c;
    t[2 * j + 1] = -std::log(j < kLogTable / 2 ? 0.5 * c : c);
  }
  void* p = ctx->log_table.ensure(sizeof(double) * t.size());
  LPM_HIP_CHECK(hipMemcpy(p, t.data(), sizeof(double) * t.size(),
                          hipMemcpyHostToDevice));
}

void check_finite(lpm_ctx* ctx, const double* base, int64_t n, int64_t es,
                  int64_t cs, int ncomp, hipStream_t s) {
  if (n == 0) return;
  check_finite_into(static_cast<int32_t*>(ctx->flag.ensure(sizeof(int32_t))),
                    base, n, es, cs, ncomp, s);
}

void check_finite_into(int32_t* flag, const double* base, int64_t n,
                       int64_t es, int64_t cs, int ncomp, hipStream_t s) {
  if (n == 0) return;
  zero_int_kernel<<<1, 1, 0, s>>>(flag);
  finite_kernel<<<static_cast<int>((n + 255) / 256), 256, 0, s>>>(
      base, n, es, cs, ncomp, flag);
  LPM_HIP_CHECK(hipGetLastError());
  int32_t h = 0;
  LPM_HIP_CHECK(hipMemcpyAsync(&h, flag, sizeof(int32_t),
                               hipMemcpyDeviceToHost, s));
  LPM_HIP_CHECK(hipStreamSynchronize(s));
  if (h) throw Error(LPM_ERR_NONFINITE, "non-finite value in direct-sum output");
}

}  // namespace lpm_amd
