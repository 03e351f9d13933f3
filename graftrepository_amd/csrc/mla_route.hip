// mla_route.hip -- MLA latent-centroid route on gfx950.
//
// Law (cpp/grm_runtime.cpp:3518-3545 exact_mla_entry_score, :4299-4361
// route_mla_arena, row norms :3232-3241):
//   score(node) = float( dot / (qnorm * (double)norm_f + 1e-8) )
//   dot   = sum_d (double)q_d * (double)r_d, sequential in d
//   qnorm = sqrt(sum_d (double)q_d^2)        norm_f = float(sqrt(sum (double)r_d^2))
// Every node is scored with exactly these fp64 operations in this order, so
// scores are bit-identical to the reference's CPU router and the ranking
// needs no re-check.  fp64 costs nothing here: the kernel streams 4 bytes
// (fp32 bank) or 2 bytes (bf16 bank) per multiply-add and is bound by HBM.
//
// Bank layout in HBM ("chunk planes"): a row is cut into 16-byte chunks (4
// fp32 or 8 bf16 values); slots are grouped in tiles of 64 and chunk c of
// slot tile*64+l lives at [c][tile][l].  Lane l of a wavefront owns one slot
// and walks its row in d order (the law's order); every load instruction of
// a wave reads 1 KiB of contiguous memory, and waves working on neighbouring
// tiles read neighbouring KiB of the same plane, which keeps DRAM rows open
// the way a plain sequential stream does.
//
// Top-k is fused: each wave keeps a distributed top-k list (grm_common.hpp),
// blocks merge their waves' lists in LDS and write their k best entries to
// mapped host memory, where the host merges the per-block lists once every
// block has stored its completion flag -- the score vector never leaves
// registers.
//
// Batched queries take the matrix-core path (mla_batch.hpp, launched from
// mla_screen.hpp): an MFMA screen of every 32-slot tile against up to 256
// queries keeps a per-lane shortlist, a merge kernel certifies each query's
// top-k against a proven bound on the screen's rounding error and rescores
// the shortlist with the exact law; queries without a certificate are routed
// again here.
#include "grm_common.hpp"
#include "mla_screen.hpp"
#include "mla_values.hpp"
#include "slot_tables.hpp"
#include "grm_hip_router.h"

#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <mutex>
#include <vector>

namespace grm {
namespace mla {

constexpr uint32_t kMaxDim = 4096;
constexpr int kRouteWaves = 16;          // most waves per block of the single-query kernel
constexpr int kDeepWaves = 8;            // most waves per block of its deep form
constexpr uint32_t kStageRows = 1u << 16;  // rows per attach staging batch

// ------------------------------------------------------------------ kernels

template <int DT>
__device__ inline double chunk_dot(u32x4 v, const double* __restrict__ q,
                                   double acc) {
  // fma(r, q, acc) == acc + r*q exactly: r*q has <= 48 significant bits.
  if constexpr (DT == kF32) {
    acc = fma(static_cast<double>(__uint_as_float(v.x)), q[0], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.y)), q[1], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.z)), q[2], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.w)), q[3], acc);
  } else {
    acc = fma(static_cast<double>(__uint_as_float(v.x << 16)), q[0], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.x & 0xffff0000u)), q[1], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.y << 16)), q[2], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.y & 0xffff0000u)), q[3], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.z << 16)), q[4], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.z & 0xffff0000u)), q[5], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.w << 16)), q[6], acc);
    acc = fma(static_cast<double>(__uint_as_float(v.w & 0xffff0000u)), q[7], acc);
  }
  return acc;
}

// Stage the query as doubles in LDS (zero beyond dim).  Up to 8 loads per
// thread are in flight at once, unconditional ones: a block may be a single
// wave, which would otherwise wait for memory once per load.
template <typename T>
__device__ inline void stage_values(double* qd, const T* __restrict__ query, uint32_t dim,
                                    uint32_t dim_pad) {
  constexpr int kAhead = 8;
  for (uint32_t d0 = threadIdx.x; d0 < dim_pad; d0 += kAhead * blockDim.x) {
    T v[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) v[j] = query[min(d0 + j * blockDim.x, dim - 1)];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const uint32_t d = d0 + j * blockDim.x;
      float f;
      if constexpr (sizeof(T) == 2) {
        f = bf16_to_f32(v[j]);
      } else {
        f = v[j];
      }
      if (d < dim_pad) qd[d] = d < dim ? static_cast<double>(f) : 0.0;
    }
  }
}
__device__ inline void stage_query(double* qd, const void* __restrict__ query,
                                   int query_dtype, uint32_t dim,
                                   uint32_t dim_pad) {
  if (query_dtype == kBF16) {
    stage_values(qd, static_cast<const uint16_t*>(query), dim, dim_pad);
  } else {
    stage_values(qd, static_cast<const float*>(query), dim, dim_pad);
  }
}

// One query against every slot; each block writes its k best entries to
// block_out[blockIdx.x*k ..), then (with done) seq to done[blockIdx.x];
// with stamps a timed route's start and end ticks (RouteStamps).
//
// Waves walk 64-slot tiles, a lane per slot, d ascending (the law's order),
// as a software pipeline: while a batch of B chunks is folded into the fp64
// dot product the next batch (of the same tile or the wave's next tile) is
// in flight, and the row norm of the next tile is fetched ahead of its
// data.  A row whose chunks are no whole number of batches reads its last
// chunk again in place of the missing ones; the staged query is zero there,
// so they add exact zeros (a stored row is finite).  Wave w of block b
// starts at tile b * waves + w, or with `spread` at w * blocks + b
// (single_geom), and steps by blocks * waves.
//
// The query's norm (a serial sum over d) is formed by one wave while every
// wave's first batch is on its way from memory.
//
// Two forms, chosen by the bank's size (single_geom):
//  * kMaxNW = 16, B = 6..9: four waves per SIMD, 9 KiB in flight per wave --
//    bound by HBM (1M x 288 fp32: 170 us = 6.8 TB/s).
//  * kMaxNW = 8, B = 12..18 (deep): banks of at most 8 tiles per CU, a wave
//    per tile on every CU.  Bound by latency: one round trip to memory and
//    the fp64 chain of one row.  10k x 288 fp32 on the device's clock
//    (RouteStamps): 7.6 to 8.3 us, against 24.6 us for 16-wave blocks on 10
//    CUs; with two, four or eight waves per block at that size 9.9, 11.4
//    and 15.5 us.  100k x 288: 20.0 to 20.9 against 31.6 us.  (A kernel
//    trace, which holds the dispatch too, reads 12.3 and 25.6 us.)
template <int DT, int B, int kMaxNW>
__global__ __launch_bounds__(kMaxNW * kWave) void mla_route_kernel(
    const u32x4* __restrict__ tiles, const float* __restrict__ norms,
    const uint64_t* __restrict__ ids, uint32_t num_tiles, uint32_t chunks,
    size_t plane, uint32_t dim, const void* __restrict__ query, int query_dtype, int k,
    Cand* __restrict__ block_out, unsigned* __restrict__ done, unsigned seq, RouteStamps stamps,
    int spread) {
  route_start_stamp(stamps, seq);
  constexpr uint32_t EPC = DT == kF32 ? 4 : 8;
  extern __shared__ double qd[];  // nb * B * EPC values
  __shared__ double s_qnorm;
  __shared__ Cand s_lists[kMaxNW][kMaxTopK];
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t nw = blockDim.x / kWave;
  const uint32_t stride = gridDim.x * nw;
  const uint32_t nb = (chunks + B - 1) / B;
  // Beyond-the-end prefetches read tile 0 (never folded).
  auto load = [&](u32x4 (&v)[B], uint32_t t, uint32_t b) {
    const u32x4* base = tiles + (t < num_tiles ? static_cast<size_t>(t) * kWave : 0);
#pragma unroll
    for (uint32_t j = 0; j < B; ++j) {
      const uint32_t c = min(b * B + j, chunks - 1);
      v[j] = __builtin_nontemporal_load(base + static_cast<size_t>(c) * plane + lane);
    }
  };

  stage_query(qd, query, query_dtype, dim, nb * B * EPC);
  constexpr bool kDeep = kMaxNW <= kDeepWaves;
  uint32_t t = spread ? wave * gridDim.x + blockIdx.x : blockIdx.x * nw + wave;
  uint32_t b = 0;
  u32x4 bufA[B], bufB[B];
  float nrm_cur = norms[(t < num_tiles ? t : 0) * kWave + lane];
  load(bufA, t, 0);
  __syncthreads();
  if (threadIdx.x == 0) s_qnorm = staged_norm(qd, nb * B * EPC);
  __syncthreads();
  const double qnorm = s_qnorm;

  WaveList L;
  wl_init(L);
  double acc = 0.0;
  float nrm_next = 0.0f;
  // Fold `now` while the next batch loads into `later`; false at the end of
  // the wave's tiles.
  auto step = [&](u32x4 (&now)[B], u32x4 (&later)[B]) -> bool {
    uint32_t tn = t, bn = b + 1;
    if (bn == nb) {
      tn = t + stride;
      bn = 0;
      nrm_next = norms[(tn < num_tiles ? tn : 0) * kWave + lane];
    }
    load(later, tn, bn);
    const double* q = qd + b * B * EPC;
    if constexpr (kDeep) {
      // fma(r, q, acc) is exact as in chunk_dot
      stream_lds<B * EPC, (B * EPC) % 16 == 0 ? 16 : 12>(q, [&](double qv, int i) {
        acc = fma(chunk_value<DT>(now[i / EPC], i % EPC), qv, acc);
      });
    } else {
#pragma unroll
      for (uint32_t j = 0; j < B; ++j) acc = chunk_dot<DT>(now[j], q + j * EPC, acc);
    }
    if (bn == 0) {
      const uint32_t slot = t * kWave + lane;
      // NaN norm marks an empty or evicted slot
      const double den = qnorm * static_cast<double>(nrm_cur) + 1.0e-8;
      const float s = static_cast<float>(acc / den);
      const bool need = isfinite(s) && s >= L.th_s;
      uint64_t id = kNoId;
      if (need) id = ids[slot];
      wl_consume(L, k, s, id, slot, need);
      acc = 0.0;
      nrm_cur = nrm_next;
    }
    t = tn;
    b = bn;
    return t < num_tiles;
  };
  if (t < num_tiles) {
    while (step(bufA, bufB) && step(bufB, bufA)) {
    }
  }
  block_topk_write(L, k, static_cast<int>(nw), s_lists, block_out, done ? route_tag(seq) : kNoSlot);
  block_done_flag(done, seq, stamps.end);
}

// Place staged row-major rows into their tile slots and compute row norms
// (cpp/grm_runtime.cpp:3232-3241).  rows: [count][dim] of DT; slots/ids may be
// null (contiguous slots from slot0 / ids = slot).  norm_range[0] tracks the
// smallest positive norm ever placed, norm_range[1] the largest finite one
// (float bits, atomicMin / atomicMax).  A row holding a non-finite value
// has a NaN or infinite dot product with every query, so the law scores it
// NaN whatever its norm; such a row is stored as zeros with a NaN norm,
// which every route scores NaN as well (0 / NaN), and which the batched
// screen's products can then never overflow on.
//
// A row's norm is one fp64 chain in d order, so a row has one lane for it;
// what bounds a batch of few rows is latency.  A block takes kPlaceRows
// rows: its wavefronts load them along d into LDS, one wavefront runs the
// chains from there while the others write the tiles.  (A thread per row,
// loading value by value, took a trip to memory per value: 68 us for 1000
// rows of 288, where these blocks take 8 to 15 us per 450 rows straight
// from host memory.  A full batch of 65,536 rows from device memory takes
// them 102 us against 86, beside the 2 ms its upload takes.)  Rows longer than kPlaceCols go slice by slice, the chains'
// sums carried along; values past dim are zeros, which leave a sum as it is.
constexpr int kPlaceRows = 16;
constexpr int kPlaceCols = 320;  // values per slice
constexpr int kPlaceWaves = 4;
template <int DT>
__global__ __launch_bounds__(kPlaceWaves * kWave) void mla_place_rows_kernel(
    const void* __restrict__ rows, uint64_t count, uint32_t dim, uint32_t chunks, size_t plane,
    const uint64_t* __restrict__ slots, const uint64_t* __restrict__ ids, uint64_t slot0,
    u32x4* __restrict__ tiles, float* __restrict__ norms, uint64_t* __restrict__ slot_ids,
    unsigned* __restrict__ norm_range) {
  constexpr int EPC = DT == kF32 ? 4 : 8;
  constexpr int kLoads = kPlaceCols / kWave;                // values per lane and row
  constexpr int kRowsPerWave = kPlaceRows / kPlaceWaves;
  // row stride: 16 lanes reading 16 bytes at one offset of 16 rows fall in
  // distinct banks
  constexpr int kStride = kPlaceCols + 4;
  __shared__ __align__(16) float s_v[kPlaceRows][kStride];
  __shared__ uint64_t s_slot[kPlaceRows];
  __shared__ unsigned s_bad[kPlaceRows];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const uint32_t width = chunks * EPC;  // dim rounded up to whole pieces
  for (uint64_t r0 = blockIdx.x * static_cast<uint64_t>(kPlaceRows); r0 < count;
       r0 += static_cast<uint64_t>(gridDim.x) * kPlaceRows) {
    const int n = static_cast<int>(min(static_cast<uint64_t>(kPlaceRows), count - r0));
    if (static_cast<int>(threadIdx.x) < n) {
      s_slot[threadIdx.x] = slots ? slots[r0 + threadIdx.x] : slot0 + r0 + threadIdx.x;
    }
    double acc = 0.0;  // wavefront 0: lane's row
    for (uint32_t d0 = 0; d0 < width; d0 += kPlaceCols) {
      float v[kRowsPerWave][kLoads];
#pragma unroll
      for (int i = 0; i < kRowsPerWave; ++i) {
        const int r = wave + i * kPlaceWaves;
        const uint64_t row = (r0 + static_cast<uint64_t>(min(r, n - 1))) * dim;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
          const uint32_t d = d0 + static_cast<uint32_t>(j * kWave + lane);
          const uint64_t src = row + min(d, dim - 1u);
          const float f = DT == kF32 ? static_cast<const float*>(rows)[src]
                                     : bf16_to_f32(static_cast<const uint16_t*>(rows)[src]);
          v[i][j] = d < dim ? f : 0.0f;
        }
      }
#pragma unroll
      for (int i = 0; i < kRowsPerWave; ++i) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) s_v[wave + i * kPlaceWaves][j * kWave + lane] = v[i][j];
      }
      __syncthreads();
      const uint32_t w = min(width - d0, static_cast<uint32_t>(kPlaceCols));
      if (wave == 0) {
        if (lane < n) {
          const float4* row = reinterpret_cast<const float4*>(s_v[lane]);
#pragma unroll 4
          for (uint32_t q = 0; q < w / 4; ++q) {
            const float4 f = row[q];
            acc = fma(static_cast<double>(f.x), static_cast<double>(f.x), acc);
            acc = fma(static_cast<double>(f.y), static_cast<double>(f.y), acc);
            acc = fma(static_cast<double>(f.z), static_cast<double>(f.z), acc);
            acc = fma(static_cast<double>(f.w), static_cast<double>(f.w), acc);
          }
        }
      } else {
        for (uint32_t i = threadIdx.x - kWave; i < w / EPC * kPlaceRows;
             i += (kPlaceWaves - 1) * kWave) {
          const int r = static_cast<int>(i % kPlaceRows);
          const uint32_t c = i / kPlaceRows;
          if (r >= n) continue;
          const float* f = s_v[r] + c * EPC;
          u32x4 out;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (DT == kF32) {
              out[e] = __float_as_uint(f[e]);
            } else {
              out[e] = (__float_as_uint(f[2 * e]) >> 16) | (__float_as_uint(f[2 * e + 1]) & 0xffff0000u);
            }
          }
          const uint64_t slot = s_slot[r];
          tiles[slot / kWave * kWave + slot % kWave + static_cast<size_t>(d0 / EPC + c) * plane] = out;
        }
      }
      __syncthreads();  // the slice is read; the tiles' stores are ordered
    }
    if (wave == 0) {
      // squares of finite fp32 / bf16 values cannot overflow fp64
      const bool mine = lane < n;
      const bool finite_row = isfinite(acc);
      const float nf = finite_row ? static_cast<float>(sqrt(acc)) : __builtin_nanf("");
      if (mine) {
        s_bad[lane] = finite_row ? 0u : 1u;
        const uint64_t slot = s_slot[lane];
        norms[slot] = nf;
        slot_ids[slot] = ids ? ids[r0 + lane] : slot;
      }
      // norm range (non-negative floats order like their bits)
      const bool counts = mine && nf > 0.0f && isfinite(nf);
      unsigned lo = counts ? __float_as_uint(nf) : 0xffffffffu;
      unsigned hi = counts ? __float_as_uint(nf) : 0u;
#pragma unroll
      for (int off = 1; off < kPlaceRows; off <<= 1) {
        lo = min(lo, static_cast<unsigned>(__shfl_xor(static_cast<int>(lo), off)));
        hi = max(hi, static_cast<unsigned>(__shfl_xor(static_cast<int>(hi), off)));
      }
      if (lane == 0 && hi != 0u) {
        atomicMin(norm_range, lo);
        atomicMax(norm_range + 1, hi);
      }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < chunks * kPlaceRows; i += kPlaceWaves * kWave) {
      const int r = static_cast<int>(i % kPlaceRows);
      if (r >= n || s_bad[r] == 0u) continue;
      const uint64_t slot = s_slot[r];
      tiles[slot / kWave * kWave + slot % kWave + static_cast<size_t>(i / kPlaceRows) * plane] =
          u32x4{0u, 0u, 0u, 0u};
    }
    __syncthreads();
  }
}

__global__ void mla_evict_kernel(const uint64_t* __restrict__ slots,
                                 uint64_t count, float* __restrict__ norms,
                                 uint64_t* __restrict__ slot_ids) {
  for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x;
       i < count; i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const uint64_t s = slots[i];
    norms[s] = __uint_as_float(0xffffffffu);
    slot_ids[s] = kNoId;
  }
}

}  // namespace mla
}  // namespace grm

using grm::Cand;
using grm::kBF16;
using grm::kF16;
using grm::kF32;
using grm::kNoId;
using grm::mla::BatchPlan;
using grm::mla::PassMarks;
using grm::mla::PassQueries;
using grm::mla::PassShape;
using grm::mla::ScreenLaunch;
using grm::mla::u32x4;

// ------------------------------------------------------------------ host side

// Rows and ids of one bank update on their way to the device: pinned host
// memory, read by the update's kernels in place.  ev marks when they have.
struct MutStage {
  grm::MappedBuf buf;
  hipEvent_t ev = nullptr;
  bool pending = false;
};

struct MlaDeviceArena {
  int device = 0;
  int dtype = kF32;
  uint32_t dim = 0;
  uint32_t dim_pad = 0;
  uint32_t epc = 4;
  uint32_t chunks = 0;
  uint32_t planes = 0;      // chunk planes allocated: chunks, or (bf16) the ring screen's 2*KS
  uint64_t capacity = 0;    // slots, multiple of 64
  uint64_t high_water = 0;  // slots [0, high_water) may hold live rows
  uint64_t live = 0;
  uint64_t epoch = 0;
  u32x4* d_tiles = nullptr;
  float* d_norms = nullptr;
  uint64_t* d_ids = nullptr;
  std::vector<uint64_t> slot_id;  // kNoId when free
  grm::IdTable slot_of;
  grm::FreeSlots free_slots;  // freed slots below high_water
  void* d_queries = nullptr;
  size_t d_queries_bytes = 0;
  float* d_latent_q = nullptr;  // route key formed from a device latent (dim floats)
  uint64_t* d_fbits = nullptr;  // per-slot route filter bits (capacity), 0 until set
  float* d_fnorms = nullptr;    // per-route norms with filtered-out slots NaN (capacity)
  const float* route_norms = nullptr;  // set around a filtered route: norms it reads
  bool no_batch = false;               // set around a filtered route: single-query path only
  grm::MappedCands blocks_out;  // per-query, per-block top-k (host mapped)
  // What flag-waiting routes report (host mapped, one allocation, see
  // reserve_marks): a completion flag per (query, block), the number the
  // last such route stored there, device-clock stamps, and the clock at the
  // start of each batched pass's screen and merge.  ticks_per_ms: the
  // clock's rate (0: stream events).
  grm::MappedBuf marks;
  size_t marks_n = 0;           // flags it has room for
  grm::MappedBuf done_flags;    // these three lie in marks
  grm::MappedBuf stamps;
  grm::MappedBuf screen_ticks;
  unsigned route_seq = 0;
  double ticks_per_ms = 0.0;
  std::vector<Cand> merged;
  void* h_stage = nullptr;
  size_t h_stage_bytes = 0;
  void* d_stage = nullptr;
  size_t d_stage_bytes = 0;
  hipStream_t stream = nullptr;
  hipStream_t side = nullptr;
  hipEvent_t ev_start = nullptr;
  hipEvent_t ev_stop = nullptr;
  // updates take the two stages in turn, so one may be filled while the
  // kernels of the other still read; both run on `side`, so the newer
  // stage's event (mut[mut_last]) covers every update
  MutStage mut[2];
  int mut_last = 0;
  bool mut_pending = false;
  unsigned* d_min_norm = nullptr;  // [smallest positive, largest finite] row norm placed (float bits)
  // batched route: pass buffers and per-query results
  uint16_t* d_qpad = nullptr;
  size_t d_qpad_count = 0;
  float* d_inv_qn = nullptr;
  size_t d_inv_qn_count = 0;
  uint32_t* d_entries = nullptr;   // screen result planes
  size_t d_entries_count = 0;
  grm::MappedCands batch_out;
  // host queries staged for fetch_async (GRM_HIP_QUERY_COPY=dma: the copy
  // engine instead)
  grm::MappedBuf q_map;
  bool query_dma = false;
  int batch_min = 0;         // timed queries per call from which the batched path runs (0: by size)
  bool ring = true;          // full 256-query passes on the ring screen (GRM_HIP_BATCH_RING=0: off)
  float* d_winv = nullptr;   // slot weights of the ring screen (capacity), for bank epoch winv_epoch
  size_t d_winv_count = 0;
  uint64_t winv_epoch = ~0ull;
  size_t lds_max = 65536;    // dynamic LDS one block may use
  uint64_t batch_queries = 0;    // queries screened on the matrix cores
  uint64_t batch_fallbacks = 0;  // of those, routed again on the single-query path
  uint64_t batch_passes = 0;     // screen passes
  uint64_t single_queries = 0;   // queries through the single-query kernel
  std::vector<hipEvent_t> screen_ev;  // begin/end pairs around timed screens
  float screen_ms = 0.0f;        // screen-kernel time of the last batched route
  uint32_t cus = 256;       // compute units of the device
  uint32_t max_blocks = 0;  // single-query grid cap (GRM_HIP_MLA_BLOCKS; a block per CU)
};

// Per-block top-k lists of the allocation-free route (see route_noalloc).
constexpr size_t kScratchCands = 16384;  // 256 KiB
static __device__ __align__(256) Cand scratch[kScratchCands];

namespace {

size_t elem_size(int dtype) { return dtype == kF32 ? 4 : 2; }

void destroy_arena(MlaDeviceArena* a) {
  if (!a) return;
  (void)hipSetDevice(a->device);
  if (a->stream) (void)hipStreamSynchronize(a->stream);
  if (a->side) (void)hipStreamSynchronize(a->side);
  if (a->d_tiles) (void)hipFree(a->d_tiles);
  if (a->d_norms) (void)hipFree(a->d_norms);
  if (a->d_ids) (void)hipFree(a->d_ids);
  if (a->d_queries) (void)hipFree(a->d_queries);
  if (a->d_latent_q) (void)hipFree(a->d_latent_q);
  if (a->d_fbits) (void)hipFree(a->d_fbits);
  if (a->d_fnorms) (void)hipFree(a->d_fnorms);
  if (a->d_stage) (void)hipFree(a->d_stage);
  if (a->d_min_norm) (void)hipFree(a->d_min_norm);
  if (a->d_qpad) (void)hipFree(a->d_qpad);
  if (a->d_inv_qn) (void)hipFree(a->d_inv_qn);
  if (a->d_entries) (void)hipFree(a->d_entries);
  if (a->d_winv) (void)hipFree(a->d_winv);
  grm::release_mapped(&a->batch_out);
  grm::release_mapped_bytes(&a->marks);
  grm::release_mapped_bytes(&a->q_map);
  grm::release_mapped(&a->blocks_out);
  if (a->h_stage) (void)hipHostFree(a->h_stage);
  if (a->ev_start) (void)hipEventDestroy(a->ev_start);
  if (a->ev_stop) (void)hipEventDestroy(a->ev_stop);
  for (MutStage& m : a->mut) {
    grm::release_mapped_bytes(&m.buf);
    if (m.ev) (void)hipEventDestroy(m.ev);
  }
  for (hipEvent_t e : a->screen_ev) (void)hipEventDestroy(e);
  if (a->stream) (void)hipStreamDestroy(a->stream);
  if (a->side) (void)hipStreamDestroy(a->side);
  delete a;
}

template <typename T>
int reserve_device(T** ptr, size_t* have, size_t want) {
  if (want <= *have && *ptr) return 0;
  if (*ptr) {
    GRM_HIP_CHECK(hipFree(*ptr));
    *ptr = nullptr;
    *have = 0;
  }
  GRM_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(ptr), want * sizeof(T)));
  *have = want;
  return 0;
}

template <typename T>
int reserve_pinned(T** ptr, size_t* have, size_t want) {
  if (want <= *have && *ptr) return 0;
  if (*ptr) {
    GRM_HIP_CHECK(hipHostFree(*ptr));
    *ptr = nullptr;
    *have = 0;
  }
  GRM_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(ptr), want * sizeof(T),
                              hipHostMallocDefault));
  *have = want;
  return 0;
}

int wait_mutations(MlaDeviceArena* a) {
  if (a->mut_pending) {
    GRM_HIP_CHECK(hipEventSynchronize(a->mut[a->mut_last].ev));
    a->mut_pending = a->mut[0].pending = a->mut[1].pending = false;
  }
  return 0;
}

// Appends of up to this many bytes are placed straight from the pinned
// stage, in parts of kAppendPartBytes (one launch each); larger ones keep
// the copy engine, whose transfers do not hold compute units.
constexpr size_t kDirectAppendBytes = 8u << 20;
constexpr size_t kAppendPartBytes = 512u << 10;

// Launch the placement kernel over `count` staged rows on `stream`.
int launch_place(MlaDeviceArena* a, const void* d_rows, uint64_t count,
                 const uint64_t* d_slots, const uint64_t* d_ids, uint64_t slot0,
                 hipStream_t stream) {
  if (count == 0) return 0;
  const unsigned threads = grm::mla::kPlaceWaves * grm::kWave;
  const unsigned blocks = static_cast<unsigned>(
      std::min<uint64_t>((count + grm::mla::kPlaceRows - 1) / grm::mla::kPlaceRows, 4096));
  if (a->dtype == kF32) {
    grm::mla::mla_place_rows_kernel<kF32><<<blocks, threads, 0, stream>>>(
        d_rows, count, a->dim, a->chunks, a->capacity, d_slots, d_ids, slot0,
        a->d_tiles, a->d_norms, a->d_ids, a->d_min_norm);
  } else {
    grm::mla::mla_place_rows_kernel<kBF16><<<blocks, threads, 0, stream>>>(
        d_rows, count, a->dim, a->chunks, a->capacity, d_slots, d_ids, slot0,
        a->d_tiles, a->d_norms, a->d_ids, a->d_min_norm);
  }
  GRM_HIP_CHECK(hipGetLastError());
  return 0;
}

int create_arena(const void* rows, int dtype, uint64_t nodes, int dim,
                 const uint64_t* node_ids, uint64_t capacity,
                 MlaDeviceArena** out) {
  if (!out) return grm::fail(-1, "null output arena pointer");
  *out = nullptr;
  if (dim <= 0 || static_cast<uint32_t>(dim) > grm::mla::kMaxDim) {
    return grm::fail(-1, "dim must be in [1, 4096]");
  }
  if (dtype != kF32 && dtype != kBF16) {
    return grm::fail(-1, "MLA bank dtype must be F32 or BF16");
  }
  if (nodes > 0 && !rows) return grm::fail(-1, "null rows with nonzero nodes");
  if (capacity < nodes) capacity = nodes;
  if (capacity == 0) return grm::fail(-1, "bank needs nodes or capacity");
  if (capacity > (1ull << 31)) return grm::fail(-1, "capacity above 2^31 slots");
  auto* a = new MlaDeviceArena();
  int rc = 0;
  auto bail = [&](int code) {
    destroy_arena(a);
    return code;
  };
  if (hipGetDevice(&a->device) != hipSuccess) a->device = 0;
  a->dtype = dtype;
  a->dim = static_cast<uint32_t>(dim);
  a->epc = dtype == kF32 ? 4 : 8;
  a->dim_pad = (a->dim + a->epc - 1) / a->epc * a->epc;
  a->chunks = a->dim_pad / a->epc;
  // bf16 banks get zero planes up to the ring screen's 16-dimension
  // K-steps (16, 32 or 36 planes), which it then reads unconditionally
  a->planes = a->chunks;
  if (dtype == kBF16) {
    for (uint32_t p : {16u, 32u, 36u}) {
      if (a->chunks <= p) {
        a->planes = p;
        break;
      }
    }
  }
  a->capacity = (capacity + grm::kWave - 1) / grm::kWave * grm::kWave;
  {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, a->device) != hipSuccess ||
        cus <= 0) {
      cus = 256;
    }
    a->cus = static_cast<uint32_t>(cus);
    a->max_blocks = static_cast<uint32_t>(cus);
  }
  if (const char* env = getenv("GRM_HIP_MLA_BLOCKS")) {
    const long v = strtol(env, nullptr, 10);
    if (v >= 1 && v <= 65536) a->max_blocks = static_cast<uint32_t>(v);
  }
  if (const char* env = getenv("GRM_HIP_BATCH_RING")) a->ring = env[0] != '0';
  if (const char* env = getenv("GRM_HIP_QUERY_COPY")) a->query_dma = strcmp(env, "dma") == 0;
  a->ticks_per_ms = grm::wall_ticks_per_ms(a->device);
  if (const char* env = getenv("GRM_HIP_MLA_BATCH_MIN")) {
    const long v = strtol(env, nullptr, 10);
    if (v >= 1) a->batch_min = static_cast<int>(std::min<long>(v, 1l << 30));
  }
  {
    int lds = 0;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeSharedMemPerBlockOptin, a->device) == hipSuccess &&
        lds > 0) {
      a->lds_max = static_cast<size_t>(lds);
    } else if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, a->device) ==
                   hipSuccess &&
               lds > 0) {
      a->lds_max = static_cast<size_t>(lds);
    }
  }
  a->slot_id.assign(a->capacity, kNoId);
  a->free_slots.resize(a->capacity);
  a->slot_of.reserve(nodes);
  if (node_ids) {
    for (uint64_t i = 0; i < nodes; ++i) {
      if (!a->slot_of.emplace(node_ids[i], i)) {
        return bail(grm::fail(-1, "duplicate node id"));
      }
      a->slot_id[i] = node_ids[i];
    }
  } else {
    for (uint64_t i = 0; i < nodes; ++i) {
      a->slot_of.emplace(i, i);
      a->slot_id[i] = i;
    }
  }
  const size_t tile_bytes = static_cast<size_t>(a->planes) * grm::kWave * 16;
  const size_t tiles = a->capacity / grm::kWave;
#define BAIL_HIP(expr)                                  \
  do {                                                  \
    hipError_t e_ = (expr);                             \
    if (e_ != hipSuccess) return bail(grm::fail_hip(e_, #expr)); \
  } while (0)
  BAIL_HIP(hipStreamCreateWithFlags(&a->stream, hipStreamDefault));
  BAIL_HIP(hipStreamCreateWithFlags(&a->side, hipStreamNonBlocking));
  BAIL_HIP(hipEventCreate(&a->ev_start));
  BAIL_HIP(hipEventCreate(&a->ev_stop));
  for (MutStage& m : a->mut) BAIL_HIP(hipEventCreateWithFlags(&m.ev, hipEventDisableTiming));
  BAIL_HIP(hipMalloc(reinterpret_cast<void**>(&a->d_tiles), tiles * tile_bytes));
  BAIL_HIP(hipMalloc(reinterpret_cast<void**>(&a->d_norms), a->capacity * sizeof(float)));
  BAIL_HIP(hipMalloc(reinterpret_cast<void**>(&a->d_ids), a->capacity * sizeof(uint64_t)));
  BAIL_HIP(hipMemsetAsync(a->d_tiles, 0, tiles * tile_bytes, a->stream));
  BAIL_HIP(hipMemsetAsync(a->d_norms, 0xff, a->capacity * sizeof(float), a->stream));
  BAIL_HIP(hipMemsetAsync(a->d_ids, 0xff, a->capacity * sizeof(uint64_t), a->stream));
  BAIL_HIP(hipMalloc(reinterpret_cast<void**>(&a->d_min_norm), 2 * sizeof(unsigned)));
  {
    const unsigned range0[2] = {0x7f800000u, 0u};
    BAIL_HIP(hipMemcpyAsync(a->d_min_norm, range0, sizeof(range0), hipMemcpyHostToDevice,
                            a->stream));
    BAIL_HIP(hipStreamSynchronize(a->stream));
  }
  if (nodes > 0) {
    const size_t row_bytes = static_cast<size_t>(a->dim) * elem_size(dtype);
    const uint64_t batch = std::min<uint64_t>(nodes, grm::mla::kStageRows);
    rc = reserve_device(reinterpret_cast<unsigned char**>(&a->d_stage),
                        &a->d_stage_bytes,
                        batch * (row_bytes + sizeof(uint64_t)));
    if (rc) return bail(rc);
    for (uint64_t r0 = 0; r0 < nodes; r0 += batch) {
      const uint64_t n = std::min<uint64_t>(batch, nodes - r0);
      unsigned char* d_rows = static_cast<unsigned char*>(a->d_stage);
      uint64_t* d_idbuf = reinterpret_cast<uint64_t*>(d_rows + batch * row_bytes);
      BAIL_HIP(hipMemcpyAsync(d_rows,
                              static_cast<const unsigned char*>(rows) + r0 * row_bytes,
                              n * row_bytes, hipMemcpyHostToDevice, a->stream));
      if (node_ids) {
        BAIL_HIP(hipMemcpyAsync(d_idbuf, node_ids + r0, n * sizeof(uint64_t),
                                hipMemcpyHostToDevice, a->stream));
      }
      rc = launch_place(a, d_rows, n, nullptr, node_ids ? d_idbuf : nullptr,
                        r0, a->stream);
      if (rc) return bail(rc);
      // The staging buffer is reused by the next batch.
      BAIL_HIP(hipStreamSynchronize(a->stream));
    }
  }
  BAIL_HIP(hipStreamSynchronize(a->stream));
#undef BAIL_HIP
  a->high_water = nodes;
  a->live = nodes;
  *out = a;
  grm::clear_error();
  return 0;
}

// Launch geometry of the single-query route kernel.
struct SingleGeom {
  uint32_t num_tiles = 0, blocks = 0, nw = 0;
  int batch = 0;      // chunks per pipelined load batch
  bool deep = false;  // the deep form (mla_route_kernel)
  int spread = 0;     // tiles dealt out block by block rather than in runs per block
};

SingleGeom single_geom(const MlaDeviceArena* a) {
  SingleGeom g;
  g.num_tiles = static_cast<uint32_t>((a->high_water + grm::kWave - 1) / grm::kWave);
  const uint32_t cap = std::min(a->cus, a->max_blocks);
  // As many waves per block as spread the tiles over every CU, so banks of
  // few tiles run one wave on each of many CUs.
  const uint32_t per_cu = std::max<uint32_t>(1, (g.num_tiles + cap - 1) / cap);
  g.deep = per_cu <= static_cast<uint32_t>(grm::mla::kDeepWaves);
  g.nw = std::min<uint32_t>(per_cu, g.deep ? grm::mla::kDeepWaves : grm::mla::kRouteWaves);
  g.blocks = std::max<uint32_t>(1, std::min((g.num_tiles + g.nw - 1) / g.nw, cap));
  // Tiles per wave below 4 (or one): dealt out one per block in turn, since a
  // last round taken by whole blocks would leave CUs with nothing to do
  // (300k x 288 fp32: 55.7 us against 75.2).  From 4 rounds on a block's
  // waves take neighbouring tiles, which streams better (1M x 288: 170 us
  // against 173).
  g.spread = static_cast<uint64_t>(g.num_tiles) <= 3ull * g.blocks * g.nw ? 1 : 0;
  // the batch that pads the row's chunks least, the longest of those
  uint32_t best = ~0u;
  for (int b : {g.deep ? 18 : 9, g.deep ? 16 : 8, g.deep ? 12 : 6}) {
    const uint32_t padded = (a->chunks + b - 1) / b * b;
    if (padded < best) {
      best = padded;
      g.batch = b;
    }
  }
  return g;
}

// One query (device pointer q) through the single-query kernel; its
// per-block top-k lands at bout (g.blocks * topk entries), and with done
// its blocks' completion flags at done[0, g.blocks).
int launch_single(MlaDeviceArena* a, const SingleGeom& g, const void* q, int q_dtype, int topk,
                  Cand* bout, unsigned* done = nullptr,
                  const grm::RouteStamps& st = grm::RouteStamps{nullptr, nullptr}) {
  const size_t padded = (a->chunks + g.batch - 1) / g.batch * g.batch;
  const size_t lds = padded * a->epc * sizeof(double);
  const dim3 grid(g.blocks), block(g.nw * grm::kWave);
  const float* nrm = a->route_norms ? a->route_norms : a->d_norms;
#define GRM_MLA_ROUTE(DT, B, NW)                                                               \
  grm::mla::mla_route_kernel<DT, B, NW><<<grid, block, lds, a->stream>>>(                      \
      a->d_tiles, nrm, a->d_ids, g.num_tiles, a->chunks, a->capacity, a->dim, q, q_dtype, topk, \
      bout, done, a->route_seq, st, g.spread)
#define GRM_MLA_BATCH(DT)                                              \
  switch (g.batch) {                                                   \
    case 18: GRM_MLA_ROUTE(DT, 18, grm::mla::kDeepWaves); break;       \
    case 16: GRM_MLA_ROUTE(DT, 16, grm::mla::kDeepWaves); break;       \
    case 12: GRM_MLA_ROUTE(DT, 12, grm::mla::kDeepWaves); break;       \
    case 9: GRM_MLA_ROUTE(DT, 9, grm::mla::kRouteWaves); break;        \
    case 8: GRM_MLA_ROUTE(DT, 8, grm::mla::kRouteWaves); break;        \
    default: GRM_MLA_ROUTE(DT, 6, grm::mla::kRouteWaves); break;       \
  }
  if (a->dtype == kF32) {
    GRM_MLA_BATCH(kF32);
  } else {
    GRM_MLA_BATCH(kBF16);
  }
#undef GRM_MLA_BATCH
#undef GRM_MLA_ROUTE
  GRM_HIP_CHECK(hipGetLastError());
  return 0;
}

void write_cands(const Cand* c, int topk, uint64_t* out_ids, float* out_scores) {
  for (int j = 0; j < topk; ++j) {
    const bool ok = isfinite(c[j].score) && c[j].id != kNoId;
    out_ids[j] = ok ? c[j].id : kNoId;
    if (out_scores) out_scores[j] = ok ? c[j].score : __builtin_nanf("");
  }
}

// Slot code width of the batched screens.  The code costs the screen bound
// 2^(ibits-23) relative, so banks whose runs would need more than 16 bits
// route on the single-query path instead.
constexpr int kMaxSlotCodeBits = 16;

// Whether a segment of `queries` has a pass for the ring screen.
bool has_ring_pass(const BatchPlan& p, int queries) {
  return std::min(queries, p.qp_max) > grm::mla::kStreamMaxCols;
}

// Whether a batched call of q queries for the k best is worth it.
//
// A batched call costs 24 to 42 us on small banks (64 to 576 values)
// whatever its queries; a call of the single-query kernel costs about 10 us
// a query (8 to 13, by row length and k) and 10 us more.  So the batched
// call saves nothing up to two queries on small banks, and up to one and a
// half on banks of 8,192 slots and more: three queries took 31 against 41 us
// at 5,000 x 288 (k = 1) and two 31 against 31, but two took 33 against 38
// us at 20,000 x 288 and 74 against 97 at 100,000 x 576.
//
// Queries without a certificate are routed again on the single-query
// kernel, as many as they are and 12 us for the second round.  A list of the
// screen keeps two entries, so a query has no certificate when three of its
// k best fall into one list's slots; with them spread evenly over S lists,
// each holds three or more with probability p = P(Bin(k, 1/S) >= 3), and
// none does with (1 - p)^S.  Measured at 288 values, batched against single
// us: 300 slots, k = 8 (a third without certificate) 3 queries 47/41, 8
// queries 63/93; k = 16 (all) 64 queries 810/779; 600 slots, k = 16 (0.65)
// 8 queries 101/107, 3 queries 68/47; 1,000 slots, k = 16 (0.33) 3 queries
// 52/47, 8 queries 74/109; 2,000 slots, k = 16 (0.1) 3 queries 40/49.  Above
// 0.85 the most a call could save is less than its screen costs.
bool batch_pays(const MlaDeviceArena* a, const BatchPlan& p, int q, int k) {
  if (a->batch_min > 0) return q >= a->batch_min;
  // lists: a sub-stream's, or on the ring a lane half's of each run
  const bool ring = has_ring_pass(p, q);
  const double tiles = static_cast<double>(a->high_water) / 32.0;
  const double runs = ring ? static_cast<double>(a->cus) * grm::mla::kRingSegs : static_cast<double>(p.subs);
  const double lists = (ring ? 2.0 : 1.0) * std::min(tiles, runs);
  if (2.0 * std::ceil(lists) < k) return false;  // fewer entries than results: never a certificate
  const double x = std::min(1.0, 1.0 / lists);
  double two = 1.0;  // P(Bin(k, x) <= 2)
  if (k >= 3) {
    const double rest = std::pow(1.0 - x, k - 2);
    two = rest * ((1.0 - x) * (1.0 - x) + k * x * (1.0 - x) + 0.5 * k * (k - 1) * x * x);
  }
  const double certain = std::pow(two, lists);  // of a query
  if (certain < 0.15) return false;
  const double none = std::pow(certain, q);     // of all of them
  return q * certain > (a->high_water >= 8192 ? 1.5 : 2.0) + 1.2 * (1.0 - none);
}

// False where the screens do not take the bank.
bool batch_plan(const MlaDeviceArena* a, BatchPlan* p) {
  const uint32_t per_step = a->dtype == kF32 ? 4 : 2;  // chunks
  p->ks = static_cast<int>((a->chunks + per_step - 1) / per_step);
  // the steps in flight that pad the row least, the most of those
  int best = 0;
  for (int c : {18, 16, 12, 9, 8, 6, 4}) {
    if (a->dtype == kF32 ? c > 9 : (c == 9 || c == 6)) continue;
    const int padded = (p->ks + c - 1) / c * c;
    if (best == 0 || padded < best) {
      best = padded;
      p->p = c;
    }
  }
  p->nb = best / p->p;
  int qp = grm::mla::kStreamMaxCols;
  while (qp >= 32 && grm::mla::stream_screen_lds(a->dtype, *p, qp) > a->lds_max) qp /= 2;
  if (qp < 32) return false;
  p->qp_stream = qp;
  // the merge holds kMergePer sub-streams (screen wavefronts) per thread
  const uint32_t waves = a->cus * grm::mla::kBatchWaves;
  if (waves > static_cast<uint32_t>(grm::mla::kMergeLoaders) * grm::mla::kMergePer) return false;
  const uint32_t n_tiles32 = static_cast<uint32_t>((a->high_water + 31) / 32);
  if (n_tiles32 == 0) return false;
  // register, tile offset in the longest run, and (stream) the lane half
  auto code_bits = [&](uint32_t runs, int half_bits) {
    const uint32_t max_run = (n_tiles32 + runs - 1) / runs;
    int bits = 0;
    while ((1u << bits) < max_run) ++bits;
    return 4 + bits + half_bits;
  };
  p->subs = std::min(waves, n_tiles32);
  p->ibits = code_bits(p->subs, 1);
  if (p->ibits > kMaxSlotCodeBits) return false;
  p->ks_ring = p->ks <= 8 ? 8 : (p->ks <= 16 ? 16 : (p->ks <= 18 ? 18 : 0));
  p->ibits_ring = code_bits(a->cus * grm::mla::kRingSegs, 0);
  p->ring = a->ring && a->dtype == kBF16 && qp == grm::mla::kStreamMaxCols && p->ks_ring != 0 && a->planes >= 2u * p->ks_ring &&
            p->ibits_ring <= kMaxSlotCodeBits && grm::mla::RingShape<18>::kLds <= a->lds_max;
  p->qp_max = p->ring ? grm::mla::kRingQueries : qp;
  return true;
}

// One pass of qc queries: on the ring screen when the plan has it and the
// pass holds more than 128 queries (padded to 256).
PassShape pass_shape(const MlaDeviceArena* a, const BatchPlan& p, int qc) {
  if (qc > grm::mla::kStreamMaxCols) {
    return {true, grm::mla::kRingQueries, a->cus * 2 * grm::mla::kRingSegs, p.ibits_ring};
  }
  return {false, qc <= 32 ? 32 : (qc <= 64 ? 64 : 128), p.subs, p.ibits};
}

// The ring screen's slot weights (reserve_batch has their memory), formed
// again when the bank changed.
int ensure_weights(MlaDeviceArena* a) {
  if (a->winv_epoch != a->epoch) {
    const unsigned blocks = static_cast<unsigned>((a->capacity + 255) / 256);
    grm::mla::mla_batch_weights_kernel<<<blocks, 256, 0, a->stream>>>(a->d_norms, a->capacity,
                                                                     a->d_winv);
    GRM_HIP_CHECK(hipGetLastError());
    a->winv_epoch = a->epoch;
  }
  return 0;
}

// The launch of pass s's screen; its result planes at `planes`.
int screen_launch(MlaDeviceArena* a, const BatchPlan& p, const PassShape& s, const PassQueries& q,
                  uint32_t* planes, const PassMarks& m, ScreenLaunch* out) {
  if (s.ring) GRM_CHECK_RC(ensure_weights(a));
  *out = ScreenLaunch{a->dtype, a->cus, a->stream, a->d_tiles, a->d_norms, a->d_winv, a->capacity,
                      a->chunks, static_cast<uint32_t>((a->high_water + 31) / 32), a->dim, a->d_qpad,
                      a->d_inv_qn, p, s, q, planes, m, a->route_seq};
  return 0;
}

// What the screen's bound rests on: gamma bounds the fp32 accumulation of
// 16*ks products per product term in 32x32x16 steps (with the MFMA's
// internal order unknown), delta what the bf16 operands leave out.
grm::mla::ScreenBound screen_bound(const MlaDeviceArena* a, const BatchPlan& p, int ibits) {
  grm::mla::ScreenBound b;
  const bool split = a->dtype == kF32;
  b.gamma = 2.0 * 18.0 * p.ks * ldexp(1.0, -24);
  if (split) b.gamma *= 3.0 * (1.0 + ldexp(1.0, -6));
  b.delta = split ? ldexp(1.0, -16) : -1.0;
  b.absm = split ? 4.0 : 1.0;
  b.dim = a->dim;
  b.ibits = ibits;
  return b;
}

// One pass: the screen and the merge of queries q; results at
// out[0, count*topk), with done their completion flags (and end ticks).
int enqueue_batch_pass(MlaDeviceArena* a, const BatchPlan& p, const PassQueries& q, int topk,
                       Cand* out, unsigned* done, unsigned long long* end_tick, const PassMarks& m) {
  const PassShape s = pass_shape(a, p, q.count);
  ScreenLaunch l;
  GRM_CHECK_RC(screen_launch(a, p, s, q, a->d_entries, m, &l));
  GRM_CHECK_RC(grm::mla::launch_screen<false>(l));
  const uint32_t n_tiles32 = static_cast<uint32_t>((a->high_water + 31) / 32);
  auto kern = a->dtype == kF32 ? grm::mla::mla_batch_merge_kernel<kF32>
                               : grm::mla::mla_batch_merge_kernel<kBF16>;
  const size_t lds = grm::mla::merge_lds(a->dim);
  GRM_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>(lds)));
  kern<<<q.count, grm::mla::kMergeThreads, lds, a->stream>>>(
      a->d_entries, s.subs, s.ring, s.qp, n_tiles32, a->d_inv_qn, a->d_tiles, a->d_norms, a->d_ids,
      a->capacity, a->chunks, q.q, q.dtype, a->dim, screen_bound(a, p, s.ibits),
      a->d_min_norm, topk, out, done, a->route_seq, end_tick,
      m.screen_tick ? m.screen_tick + 1 : nullptr);
  GRM_HIP_CHECK(hipGetLastError());
  return 0;
}

// Buffers of the batched route, with those of the ring screen where it has
// a pass.  False when the device has no room for them: the queries then go
// one by one.
bool reserve_batch(MlaDeviceArena* a, const BatchPlan& p, bool ring) {
  const size_t cols = ring ? p.qp_max : p.qp_stream;
  size_t subs = p.subs * static_cast<size_t>(p.qp_stream);
  if (ring) subs = std::max<size_t>(subs, a->cus * size_t{2 * grm::mla::kRingSegs} * p.qp_max);
  const bool ok =
      (!ring || (reserve_device(&a->d_winv, &a->d_winv_count, static_cast<size_t>(a->capacity)) == 0 &&
                 reserve_device(&a->d_qpad, &a->d_qpad_count, cols * (16 * p.ks_ring + 8)) == 0)) &&
      reserve_device(&a->d_inv_qn, &a->d_inv_qn_count, cols) == 0 &&
      reserve_device(&a->d_entries, &a->d_entries_count, grm::mla::kEntryPlanes * subs) == 0;
  if (!ok) (void)hipGetLastError();
  return ok;
}

// Completion flags a route may wait on (one per query and route block).
constexpr size_t kMaxDoneFlags = 8192;

// Room for n flags, their stamps, and ticks of as many queries' batched
// passes (32 queries at least), in one pinned allocation: the first routes
// on a bank pay for each, and for each page.
int reserve_marks(MlaDeviceArena* a, size_t n) {
  if (n <= a->marks_n) return 0;
  size_t room = 512;
  while (room < n) room *= 2;
  const size_t flags = room * sizeof(unsigned);
  const size_t stamps = grm::stamps_bytes(room);
  const size_t ticks = (room / 32 + 1) * 2 * sizeof(unsigned long long);
  a->marks_n = 0;
  GRM_CHECK_RC(grm::reserve_mapped_bytes(&a->marks, flags + stamps + ticks));
  memset(a->marks.host, 0, a->marks.bytes);
  auto part = [&](size_t at, size_t bytes) {
    return grm::MappedBuf{static_cast<unsigned char*>(a->marks.host) + at,
                          static_cast<unsigned char*>(a->marks.dev) + at, bytes};
  };
  a->done_flags = part(0, flags);
  a->stamps = part(flags, stamps);
  a->screen_ticks = part(flags + stamps, ticks);
  a->marks_n = room;
  return 0;
}

int route_impl(MlaDeviceArena* a, const void* queries, int q_dtype,
               bool on_device, int q_count, int dim, int warmup, int topk,
               uint64_t* out_ids, float* out_scores, float* elapsed_ms) {
  if (!a || !queries || !out_ids) return grm::fail(-1, "null argument");
  if (dim != static_cast<int>(a->dim)) return grm::fail(-1, "query dim does not match bank");
  if (q_dtype != kF32 && q_dtype != kBF16) return grm::fail(-1, "query dtype must be F32 or BF16");
  if (q_count <= 0 || warmup < 0 || warmup >= q_count) {
    return grm::fail(-1, "need query_count > 0 and 0 <= warmup < query_count");
  }
  if (topk <= 0 || topk > grm::kMaxTopK || static_cast<uint64_t>(topk) > a->live) {
    return grm::fail(-1, "topk must be in [1, 16] and <= live nodes");
  }
  GRM_HIP_CHECK(hipSetDevice(a->device));
  const size_t qbytes = static_cast<size_t>(q_count) * a->dim * elem_size(q_dtype);
  const SingleGeom g = single_geom(a);
  const size_t per_q = static_cast<size_t>(g.blocks) * topk;
  const unsigned char* qbase = static_cast<const unsigned char*>(queries);
  if (!on_device) {
    // through a pinned, device-mapped buffer and a copy kernel on the
    // route's stream (fetch_async), as the GQA routes take theirs
    GRM_CHECK_RC(reserve_device(reinterpret_cast<unsigned char**>(&a->d_queries),
                                &a->d_queries_bytes, qbytes));
    GRM_CHECK_RC(grm::reserve_mapped_bytes(&a->q_map, qbytes));
    memcpy(a->q_map.host, queries, qbytes);
    if (a->query_dma) {
      GRM_HIP_CHECK(hipMemcpyAsync(a->d_queries, a->q_map.host, qbytes, hipMemcpyHostToDevice, a->stream));
    } else {
      GRM_CHECK_RC(grm::fetch_async(a->d_queries, a->q_map.dev, qbytes, a->stream));
    }
    qbase = static_cast<const unsigned char*>(a->d_queries);
  }
  if (a->mut_pending) GRM_HIP_CHECK(hipStreamWaitEvent(a->stream, a->mut[a->mut_last].ev, 0));
  const size_t qstride = static_cast<size_t>(a->dim) * elem_size(q_dtype);
  BatchPlan bp;
  const int timed = q_count - warmup;
  const bool batched = !a->no_batch && (timed > 1 || a->batch_min == 1) && batch_plan(a, &bp) &&
                       batch_pays(a, bp, timed, topk) &&
                       reserve_batch(a, bp, has_ring_pass(bp, std::max(warmup, timed)));
  a->screen_ms = 0.0f;
  std::vector<int> redo;  // queries for the single-query kernel
  if (batched) {
    GRM_CHECK_RC(grm::reserve_mapped(&a->batch_out, static_cast<size_t>(q_count) * topk));
    const int segments[2][2] = {{0, warmup}, {warmup, q_count}};
    // Completion as for single queries (below): a flag per query, the
    // times on the device clock; stream events where those cannot serve.
    const size_t n_q = static_cast<size_t>(q_count);
    const bool flags = n_q <= kMaxDoneFlags && !grm::blocking_sync() && a->ticks_per_ms > 0.0 &&
                       !(elapsed_ms && grm::event_timing());
    const int timed_passes = (timed + bp.qp_max - 1) / bp.qp_max;
    unsigned* d_done = nullptr;
    if (flags) {
      GRM_CHECK_RC(reserve_marks(a, n_q));
      GRM_CHECK_RC(grm::begin_flags(&a->done_flags, n_q, &a->route_seq));
      d_done = static_cast<unsigned*>(a->done_flags.dev);
    } else {
      while (a->screen_ev.size() < 2 * static_cast<size_t>(timed_passes)) {
        hipEvent_t e = nullptr;
        GRM_HIP_CHECK(hipEventCreate(&e));
        a->screen_ev.push_back(e);
      }
    }
    int tp = 0;
    for (int si = 0; si < 2; ++si) {
      if (si == 1 && !flags) GRM_HIP_CHECK(hipEventRecord(a->ev_start, a->stream));
      for (int q0 = segments[si][0]; q0 < segments[si][1]; q0 += bp.qp_max) {
        const PassQueries pq{qbase + q0 * qstride, q_dtype, std::min(bp.qp_max, segments[si][1] - q0)};
        PassMarks m;
        unsigned long long* end_tick = nullptr;
        if (flags) {
          const grm::RouteStamps st = grm::route_stamps(a->stamps, static_cast<size_t>(q0));
          if (si == 1 && q0 == warmup) m.start.start = st.start;
          end_tick = st.end;
        }
        if (si == 1) {
          if (flags) {
            m.screen_tick = static_cast<unsigned long long*>(a->screen_ticks.dev) + 2 * tp;
          } else {
            m.ev = &a->screen_ev[2 * tp];
          }
          ++tp;
        }
        GRM_CHECK_RC(enqueue_batch_pass(a, bp, pq, topk,
                                        a->batch_out.dev + static_cast<size_t>(q0) * topk,
                                        d_done ? d_done + q0 : nullptr, end_tick, m));
        a->batch_passes += 1;
      }
    }
    GRM_HIP_CHECK(hipEventRecord(a->ev_stop, a->stream));
    a->screen_ms = 0.0f;
    if (flags) {
      GRM_CHECK_RC(grm::wait_flags(a->done_flags, a->route_seq, n_q, a->ev_stop));
      GRM_CHECK_RC(grm::wait_tagged(a->batch_out.host, n_q * topk, a->route_seq, a->ev_stop));
      float ms = 0.0f;
      GRM_CHECK_RC(grm::stamps_elapsed(a->stamps, a->route_seq, static_cast<size_t>(warmup), n_q,
                                       a->ev_stop, a->ticks_per_ms, &ms));
      if (elapsed_ms) *elapsed_ms = ms;
      // a pass's screen ends where its merge starts; both ticks lie after
      // the route's start (grm::stamps_elapsed has seen that stamp)
      const volatile unsigned long long* tick =
          static_cast<const volatile unsigned long long*>(a->screen_ticks.host);
      const unsigned long long t0 = *static_cast<const volatile unsigned long long*>(a->stamps.host);
      for (int i = 0; i < 2 * tp; ++i) {
        if (tick[i] >= t0) continue;
        GRM_CHECK_RC(grm::wait_event(a->ev_stop));
        std::atomic_thread_fence(std::memory_order_acquire);
        break;
      }
      for (int i = 0; i < tp; ++i) {
        a->screen_ms += static_cast<float>(static_cast<double>(tick[2 * i + 1] - tick[2 * i]) / a->ticks_per_ms);
      }
    } else {
      GRM_CHECK_RC(grm::wait_event(a->ev_stop));
      if (elapsed_ms) GRM_HIP_CHECK(hipEventElapsedTime(elapsed_ms, a->ev_start, a->ev_stop));
      for (int i = 0; i < tp; ++i) {
        float ms = 0.0f;
        GRM_HIP_CHECK(hipEventElapsedTime(&ms, a->screen_ev[2 * i], a->screen_ev[2 * i + 1]));
        a->screen_ms += ms;
      }
    }
    for (int qi = 0; qi < q_count; ++qi) {
      const Cand* c = a->batch_out.host + static_cast<size_t>(qi) * topk;
      if (c->id != kNoId) {
        write_cands(c, topk, out_ids + static_cast<size_t>(qi) * topk,
                    out_scores ? out_scores + static_cast<size_t>(qi) * topk : nullptr);
      } else {
        redo.push_back(qi);
      }
    }
    a->batch_queries += static_cast<uint64_t>(q_count);
    a->batch_fallbacks += redo.size();
  } else {
    for (int qi = 0; qi < q_count; ++qi) redo.push_back(qi);
  }
  if (!redo.empty()) {
    a->single_queries += redo.size();
    GRM_CHECK_RC(grm::reserve_mapped(&a->blocks_out, per_q * redo.size()));
    // The host sees completion through per-block flags in host memory, as
    // soon as the last block stores its flag (no stream event on the
    // path).  A timed route without a batched pass does too when the
    // device reports its constant clock: its device time is then the
    // clock's ticks from the first timed launch's start to the last flag
    // (RouteStamps; GRM_HIP_ROUTE_TIMING=events keeps stream events).
    const size_t n_flags = static_cast<size_t>(g.blocks) * redo.size();
    const bool flaggable = n_flags <= kMaxDoneFlags && !grm::blocking_sync();
    const bool clocked =
        elapsed_ms && !batched && flaggable && a->ticks_per_ms > 0.0 && !grm::event_timing();
    const bool flags = flaggable && (!elapsed_ms || clocked);
    unsigned* d_done = nullptr;
    if (flags) {
      GRM_CHECK_RC(reserve_marks(a, n_flags));
      GRM_CHECK_RC(grm::begin_flags(&a->done_flags, n_flags, &a->route_seq));
      d_done = static_cast<unsigned*>(a->done_flags.dev);
    }
    // Uncertified batched queries add their time to the timed segment.
    bool started = false;
    for (size_t j = 0; j < redo.size(); ++j) {
      const int qi = redo[j];
      grm::RouteStamps st{nullptr, nullptr};
      if (clocked) st = grm::route_stamps(a->stamps, j * g.blocks);
      if (!started && elapsed_ms && (batched || qi == warmup)) {
        if (!clocked) GRM_HIP_CHECK(hipEventRecord(a->ev_start, a->stream));
        started = true;
      } else {
        st.start = nullptr;
      }
      GRM_CHECK_RC(launch_single(a, g, qbase + qi * qstride, q_dtype, topk,
                                 a->blocks_out.dev + j * per_q,
                                 d_done ? d_done + j * g.blocks : nullptr, st));
    }
    GRM_HIP_CHECK(hipEventRecord(a->ev_stop, a->stream));
    if (flags) {
      GRM_CHECK_RC(grm::wait_flags(a->done_flags, a->route_seq, n_flags, a->ev_stop));
      GRM_CHECK_RC(grm::wait_tagged(a->blocks_out.host, per_q * redo.size(), a->route_seq, a->ev_stop));
    } else {
      GRM_CHECK_RC(grm::wait_event(a->ev_stop));
    }
    if (clocked) {
      GRM_CHECK_RC(grm::stamps_elapsed(a->stamps, a->route_seq, static_cast<size_t>(warmup) * g.blocks, n_flags,
                                       a->ev_stop, a->ticks_per_ms, elapsed_ms));
    } else if (elapsed_ms) {
      float ms = 0.0f;
      GRM_HIP_CHECK(hipEventElapsedTime(&ms, a->ev_start, a->ev_stop));
      *elapsed_ms = batched ? *elapsed_ms + ms : ms;
    }
    a->merged.resize(topk);
    for (size_t j = 0; j < redo.size(); ++j) {
      const int qi = redo[j];
      grm::host_topk_merge(a->blocks_out.host + j * per_q, per_q, topk, a->merged.data());
      write_cands(a->merged.data(), topk, out_ids + static_cast<size_t>(qi) * topk,
                  out_scores ? out_scores + static_cast<size_t>(qi) * topk : nullptr);
    }
  }
  grm::clear_error();
  return 0;
}

// The next update's stage, of at least `bytes` (0: its event alone), once
// the kernels of the update before the last have read it.
int next_stage(MlaDeviceArena* a, size_t bytes, MutStage** out) {
  MutStage& m = a->mut[a->mut_last ^ 1];
  if (m.pending) {
    GRM_HIP_CHECK(hipEventSynchronize(m.ev));
    m.pending = false;
  }
  if (bytes > 0) GRM_CHECK_RC(grm::reserve_mapped_bytes(&m.buf, bytes));
  *out = &m;
  return 0;
}

// The update's kernels are all on the side stream.  Without an event to mark
// their end, they are waited for.
int end_update(MlaDeviceArena* a, MutStage* m) {
  if (hipEventRecord(m->ev, a->side) != hipSuccess) {
    (void)hipGetLastError();
    GRM_HIP_CHECK(hipStreamSynchronize(a->side));
    return 0;
  }
  m->pending = true;
  a->mut_last ^= 1;
  a->mut_pending = true;
  return 0;
}

int stage_upload(MlaDeviceArena* a, size_t bytes, void** host, void** dev) {
  GRM_CHECK_RC(wait_mutations(a));
  GRM_CHECK_RC(reserve_pinned(reinterpret_cast<unsigned char**>(&a->h_stage),
                              &a->h_stage_bytes, bytes));
  GRM_CHECK_RC(reserve_device(reinterpret_cast<unsigned char**>(&a->d_stage),
                              &a->d_stage_bytes, bytes));
  *host = a->h_stage;
  *dev = a->d_stage;
  return 0;
}

// Route key of one latent block, core/kv_graft.py:131-142
// (latent_centroid):
//   c = latent.astype(float32).mean(0);  key = c / (||c|| + 1e-8).
// The mean follows numpy's float32 reduce over axis 0 as mean() runs it
// (with a where mask, so from the identity): the accumulator starts at
// +0.0 (an all -0 column sums to +0), rows add in order, and one fp32
// division by the token count follows.  The norm is taken in
// fp64 and rounded to fp32.  The reference's comes from a BLAS dot in fp32
// whose summation order depends on the host CPU, so the key agrees with it
// to that dot's rounding (up to dim * 2^-24 of |c|^2), not bit for bit.
// normalize = 0 writes the mean alone.
//
// Columns are split over blocks, kLatentCols per block.  A block stages
// its strip of up to kLatentRows tokens in LDS at once (16-byte loads when
// rows allow them), then thread c adds column c over those tokens in order.
// The adds of a column stay one serial chain, as the law has them.  A
// one-block kernel then takes the norm and scales the key.
constexpr int kLatentThreads = 256;
constexpr uint32_t kLatentCols = 32;
constexpr uint32_t kLatentRows = 512;  // 64 KiB of fp32 strip per pass

__global__ __launch_bounds__(kLatentThreads) void latent_mean_kernel(
    const void* __restrict__ latent, int dtype, uint64_t tokens, uint32_t dim,
    uint64_t row_stride, float* __restrict__ out) {
  __shared__ float s_strip[kLatentRows * kLatentCols];  // [row][column]
  const uint32_t c0 = blockIdx.x * kLatentCols;
  const uint32_t width = min(kLatentCols, dim - c0);
  const uint32_t esize = dtype == kF32 ? 4u : 2u;
  const uint32_t epv = 16u / esize;  // values per 16-byte load
  const bool vec = width % epv == 0 && row_stride % epv == 0 && c0 % epv == 0 &&
                   reinterpret_cast<uintptr_t>(latent) % 16 == 0;
  auto cvt = [&](uint16_t b) -> float {
    return dtype == kBF16 ? grm::bf16_to_f32(b) : static_cast<float>(__builtin_bit_cast(_Float16, b));
  };
  float acc = 0.0f;  // column c0 + threadIdx.x (threads below width)
  for (uint64_t t0 = 0; t0 < tokens; t0 += kLatentRows) {
    const uint32_t rows = static_cast<uint32_t>(min<uint64_t>(kLatentRows, tokens - t0));
    if (vec) {
      const uint32_t per_row = width / epv;
      const uint32_t nv = rows * per_row;
      constexpr int kBatch = 8;
      for (uint32_t base = 0; base < nv; base += kBatch * kLatentThreads) {
        u32x4 v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          const uint32_t i = base + k * kLatentThreads + threadIdx.x;
          const uint64_t e = (t0 + i / per_row) * row_stride + c0 + (i % per_row) * epv;
          v[k] = i < nv ? *reinterpret_cast<const u32x4*>(
                              static_cast<const unsigned char*>(latent) + e * esize)
                        : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          const uint32_t i = base + k * kLatentThreads + threadIdx.x;
          if (i >= nv) continue;
          float* dst = s_strip + (i / per_row) * kLatentCols + (i % per_row) * epv;
          if (dtype == kF32) {
            dst[0] = __uint_as_float(v[k].x);
            dst[1] = __uint_as_float(v[k].y);
            dst[2] = __uint_as_float(v[k].z);
            dst[3] = __uint_as_float(v[k].w);
          } else {
            const uint32_t w[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
            for (int q = 0; q < 8; ++q) dst[q] = cvt(static_cast<uint16_t>(w[q / 2] >> (16 * (q % 2))));
          }
        }
      }
    } else {
      for (uint32_t i = threadIdx.x; i < rows * width; i += kLatentThreads) {
        const uint32_t r = i / width, c = i % width;
        const uint64_t e = (t0 + r) * row_stride + c0 + c;
        s_strip[r * kLatentCols + c] =
            dtype == kF32 ? static_cast<const float*>(latent)[e]
                          : cvt(static_cast<const uint16_t*>(latent)[e]);
      }
    }
    __syncthreads();
    if (threadIdx.x < width) {
      float a = acc;
#pragma unroll 8
      for (uint32_t r = 0; r < rows; ++r) a += s_strip[r * kLatentCols + threadIdx.x];
      acc = a;
    }
    __syncthreads();
  }
  if (threadIdx.x < width) out[c0 + threadIdx.x] = acc / static_cast<float>(tokens);
}

__global__ __launch_bounds__(kLatentThreads) void latent_normalize_kernel(uint32_t dim,
                                                                          float* __restrict__ out) {
  __shared__ double s_ss[kLatentThreads / grm::kWave];
  double ss = 0.0;
  for (uint32_t d = threadIdx.x; d < dim; d += kLatentThreads) {
    ss += static_cast<double>(out[d]) * static_cast<double>(out[d]);
  }
  for (int off = grm::kWave / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
  if ((threadIdx.x & (grm::kWave - 1)) == 0) s_ss[threadIdx.x / grm::kWave] = ss;
  __syncthreads();
  double total = 0.0;
  for (int w = 0; w < kLatentThreads / grm::kWave; ++w) total += s_ss[w];
  const float denom = static_cast<float>(sqrt(total)) + 1e-8f;
  for (uint32_t d = threadIdx.x; d < dim; d += kLatentThreads) out[d] = out[d] / denom;
}

// Route filters (cpp/grm_runtime.cpp:3074-3104, every filter value known,
// bits as route_filter_bits :2793-2838): a node passes when, for each
// category c with filters (bit c of cats), its bits meet that category's
// 16-bit mask, held at shift 16c in fmask.  Slots that do not pass get a
// NaN norm, the marker the route kernels already skip; the filtered route
// reads this copy in place of the bank's norms.
__global__ void mla_filter_norms_kernel(const float* __restrict__ norms,
                                        const uint64_t* __restrict__ fbits, uint64_t n,
                                        uint64_t fmask, uint32_t cats, float* __restrict__ out) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += stride) {
    const uint64_t hit = fbits[i] & fmask;
    bool ok = true;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if ((cats >> c) & 1u) ok = ok && ((hit >> (16 * c)) & 0xffffull) != 0;
    }
    out[i] = ok ? norms[i] : __builtin_nanf("");
  }
}

__global__ void mla_zero_bits_kernel(const uint64_t* __restrict__ slots, uint64_t n,
                                     uint64_t* __restrict__ fbits) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += stride) {
    fbits[slots[i]] = 0ull;
  }
}

__global__ void mla_scatter_bits_kernel(const uint64_t* __restrict__ slot_bits, uint64_t n,
                                        uint64_t* __restrict__ fbits) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) fbits[slot_bits[2 * i]] = slot_bits[2 * i + 1];
}

// Law scores (cpp/grm_runtime.cpp:3518-3545) of listed slots: the query
// staged in fp64, its norm summed in d order (as the route kernels), and
// per slot the fp64 dot in d order, then float(dot / (qnorm * norm_f +
// 1e-8)); NaN where that is not finite or the slot is empty.  One block;
// thread i scores slots i, i + blockDim.x, ...
template <int DT>
__global__ __launch_bounds__(256) void mla_score_slots_kernel(
    const u32x4* __restrict__ tiles, const float* __restrict__ norms, size_t plane,
    uint32_t chunks, uint32_t dim, uint32_t dim_pad, const void* __restrict__ query,
    int query_dtype, const uint64_t* __restrict__ slots, uint64_t n, float* __restrict__ out) {
  constexpr int EPC = DT == kF32 ? 4 : 8;
  extern __shared__ double qd[];
  __shared__ double s_qnorm;
  grm::mla::stage_query(qd, query, query_dtype, dim, dim_pad);
  __syncthreads();
  if (threadIdx.x == 0) {
    double acc = 0.0;
    for (uint32_t d = 0; d < dim; ++d) acc = fma(qd[d], qd[d], acc);
    s_qnorm = sqrt(acc);
  }
  __syncthreads();
  const double qnorm = s_qnorm;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const uint64_t slot = slots[i];
    // the route kernels' own chunk fold, chunks in order (zero past dim)
    double acc = 0.0;
    for (uint32_t c = 0; c < chunks; ++c) {
      acc = grm::mla::chunk_dot<DT>(tiles[static_cast<size_t>(c) * plane + slot], qd + c * EPC,
                                    acc);
    }
    const float nrm = norms[slot];
    const float sc = static_cast<float>(acc / (qnorm * static_cast<double>(nrm) + 1.0e-8));
    out[i] = isfinite(sc) ? sc : __builtin_nanf("");
  }
}

// Evict the `count` slots at d_slots on the side stream.
int launch_evict(MlaDeviceArena* a, const uint64_t* d_slots, uint64_t count) {
  const unsigned threads = 256;
  const unsigned blocks = static_cast<unsigned>(std::min<uint64_t>((count + threads - 1) / threads, 1024));
  grm::mla::mla_evict_kernel<<<blocks, threads, 0, a->side>>>(d_slots, count, a->d_norms, a->d_ids);
  GRM_HIP_CHECK(hipGetLastError());
  if (a->d_fbits) {
    // a slot reused by a later append starts with no filter bits
    mla_zero_bits_kernel<<<blocks, threads, 0, a->side>>>(d_slots, count, a->d_fbits);
    GRM_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

int enqueue_latent_query(MlaDeviceArena* a, const void* d_latent, int dtype, uint64_t tokens,
                         uint64_t row_stride, int normalize, float* d_out) {
  if (!d_latent || !d_out) return grm::fail(-1, "null pointer");
  if (dtype != kF32 && dtype != kBF16 && dtype != kF16) {
    return grm::fail(-1, "latent dtype must be F32, BF16 or F16");
  }
  if (tokens == 0) return grm::fail(-1, "latent has no tokens");
  if (tokens >= (1ull << 24)) return grm::fail(-1, "token count above 2^24");
  if (row_stride == 0) row_stride = a->dim;
  if (row_stride < a->dim) return grm::fail(-1, "row stride below the bank dim");
  GRM_HIP_CHECK(hipSetDevice(a->device));
  const uint32_t dim = static_cast<uint32_t>(a->dim);
  latent_mean_kernel<<<(dim + kLatentCols - 1) / kLatentCols, kLatentThreads, 0, a->stream>>>(
      d_latent, dtype, tokens, dim, row_stride, d_out);
  GRM_HIP_CHECK(hipGetLastError());
  if (normalize) latent_normalize_kernel<<<1, kLatentThreads, 0, a->stream>>>(dim, d_out);
  GRM_HIP_CHECK(hipGetLastError());
  return 0;
}

// ------------------------------------------------ allocation-free route
//
// grm_mla_hip_route_noalloc keeps the single-query kernel's per-block top-k
// lists in `scratch`, a file-scope device array, instead of memory the
// library allocates; a merge kernel then writes the k best of those lists
// straight to the caller's device outputs.  Each GPU holds its own copy of
// the array from load to process end, and host code reaches it only through
// the address hipGetSymbolAddress returns for the current device (the
// array's name in host code is a host-side stand-in, not a device address).
// Every call on one GPU shares that GPU's array, so calls on one GPU are
// serialised by a per-device mutex held from the first launch until the
// bank's stream has drained (on the error path too): two host threads
// routing different banks on one GPU take turns and each gets its own
// answer.  Queries run one after another on the bank's stream, so one
// query's lists fit the array: up to kScratchCands entries (grid blocks x
// topk; the grid has a block per compute unit at most, 256 x 16 here).
// Each block writes all k of its entries before the merge reads them, so
// nothing in the array has to start at zero.
constexpr int kScratchDevices = 64;

std::mutex g_scratch_mu;
Cand* g_scratch_ptr[kScratchDevices] = {};
// Held by a call from its first launch until its stream has drained.
std::mutex g_noalloc_mu[kScratchDevices];

// Device address of this device's scratch (the device must be current).
int scratch_for(int device, Cand** out) {
  if (device < 0 || device >= kScratchDevices) return grm::fail(-1, "device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    GRM_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return grm::fail(-1, "scratch symbol has no device address");
    g_scratch_ptr[device] = static_cast<Cand*>(p);
  }
  *out = g_scratch_ptr[device];
  return 0;
}

// k best of `count` per-block entries, written as ids and scores (unfilled:
// UINT64_MAX and NaN); one block.
__global__ __launch_bounds__(grm::kMergeWaves * grm::kWave) void mla_merge_out_kernel(
    const Cand* __restrict__ in, uint32_t count, int k, uint64_t* __restrict__ out_ids,
    float* __restrict__ out_scores) {
  __shared__ Cand s_lists[grm::kMergeWaves][grm::kMaxTopK];
  const int lane = threadIdx.x & (grm::kWave - 1);
  const int wave = threadIdx.x / grm::kWave;
  grm::WaveList G;
  grm::wl_init(G);
  grm::wl_consume_global(G, k, in, count, static_cast<uint32_t>(wave), grm::kMergeWaves);
  if (lane < grm::kMaxTopK) s_lists[wave][lane] = grm::wl_entry(G);
  __syncthreads();
  if (wave == 0) {
    grm::WaveList B;
    grm::block_merge(s_lists, grm::kMergeWaves, k, B);
    if (lane < k) {
      const bool ok = isfinite(B.s) && B.id != kNoId;
      out_ids[lane] = ok ? B.id : kNoId;
      if (out_scores) out_scores[lane] = ok ? B.s : __builtin_nanf("");
    }
  }
}

int route_noalloc(MlaDeviceArena* a, const void* d_queries, int q_dtype, int q_count, int dim,
                  int topk, uint64_t* d_out_ids, float* d_out_scores) {
  if (!a || !d_queries || !d_out_ids) return grm::fail(-1, "null argument");
  if (dim != static_cast<int>(a->dim)) return grm::fail(-1, "query dim does not match bank");
  if (q_dtype != kF32 && q_dtype != kBF16) return grm::fail(-1, "query dtype must be F32 or BF16");
  if (q_count <= 0) return grm::fail(-1, "need query_count > 0");
  if (topk <= 0 || topk > grm::kMaxTopK || static_cast<uint64_t>(topk) > a->live) {
    return grm::fail(-1, "topk must be in [1, 16] and <= live nodes");
  }
  const SingleGeom g = single_geom(a);
  const size_t per_q = static_cast<size_t>(g.blocks) * topk;
  if (per_q > kScratchCands) {
    return grm::fail(-1, "route grid blocks x topk exceed the 16384-entry scratch");
  }
  GRM_HIP_CHECK(hipSetDevice(a->device));
  Cand* lists = nullptr;
  GRM_CHECK_RC(scratch_for(a->device, &lists));
  std::lock_guard<std::mutex> hold(g_noalloc_mu[a->device]);
  const size_t qstride = static_cast<size_t>(a->dim) * elem_size(q_dtype);
  const unsigned char* qbase = static_cast<const unsigned char*>(d_queries);
  auto launch_all = [&]() -> int {
    if (a->mut_pending) GRM_HIP_CHECK(hipStreamWaitEvent(a->stream, a->mut[a->mut_last].ev, 0));
    for (int qi = 0; qi < q_count; ++qi) {
      GRM_CHECK_RC(launch_single(a, g, qbase + qi * qstride, q_dtype, topk, lists));
      mla_merge_out_kernel<<<1, grm::kMergeWaves * grm::kWave, 0, a->stream>>>(
          lists, static_cast<uint32_t>(per_q), topk,
          d_out_ids + static_cast<size_t>(qi) * topk,
          d_out_scores ? d_out_scores + static_cast<size_t>(qi) * topk : nullptr);
      GRM_HIP_CHECK(hipGetLastError());
    }
    return 0;
  };
  const int rc = launch_all();
  // Drain before the lock is released, also when a launch failed part way:
  // kernels already queued still write this GPU's scratch.
  const hipError_t sync = hipStreamSynchronize(a->stream);
  if (rc != 0) return rc;
  GRM_HIP_CHECK(sync);
  a->single_queries += static_cast<uint64_t>(q_count);
  grm::clear_error();
  return 0;
}

}  // namespace

// ============================================================ reference ABI

extern "C" int grm_mla_cuda_arena_create(const float* rows_host, int nodes,
                                         int dim, MlaDeviceArena** out_arena) {
  if (!rows_host || !out_arena || nodes <= 0 || dim <= 0) {
    return grm::fail(-1, "invalid MLA arena arguments");
  }
  return create_arena(rows_host, kF32, static_cast<uint64_t>(nodes), dim,
                      nullptr, static_cast<uint64_t>(nodes), out_arena);
}

extern "C" int grm_mla_cuda_arena_route(MlaDeviceArena* arena,
                                        const float* queries_host,
                                        int query_count, int dim, int warmup,
                                        int topk, uint64_t* out_topk_host,
                                        float* elapsed_ms_host) {
  if (!arena || !queries_host || query_count <= 0 || dim <= 0 ||
      !elapsed_ms_host) {
    return grm::fail(-1, "invalid MLA route arguments");
  }
  return route_impl(arena, queries_host, kF32, false, query_count, dim, warmup,
                    topk, out_topk_host, nullptr, elapsed_ms_host);
}

extern "C" int grm_mla_cuda_arena_route_device(MlaDeviceArena* arena,
                                               const float* d_queries,
                                               int query_count, int dim,
                                               int warmup, int topk,
                                               uint64_t* out_topk_host,
                                               float* elapsed_ms_host) {
  if (!arena || !elapsed_ms_host) return grm::fail(-1, "invalid MLA route arguments");
  return route_impl(arena, d_queries, kF32, true, query_count, dim, warmup,
                    topk, out_topk_host, nullptr, elapsed_ms_host);
}

extern "C" int grm_mla_cuda_upload_queries(const float* host_buf,
                                           size_t num_floats,
                                           float** out_device_ptr) {
  if (!host_buf || !out_device_ptr || num_floats == 0) {
    return grm::fail(-1, "invalid upload arguments");
  }
  *out_device_ptr = nullptr;
  float* d = nullptr;
  GRM_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&d), num_floats * sizeof(float)));
  hipError_t rc = hipMemcpy(d, host_buf, num_floats * sizeof(float), hipMemcpyHostToDevice);
  if (rc != hipSuccess) {
    (void)hipFree(d);
    return grm::fail_hip(rc, "hipMemcpy");
  }
  *out_device_ptr = d;
  return 0;
}

extern "C" int grm_mla_cuda_free_device_ptr(float* device_ptr) {
  if (!device_ptr) return 0;
  GRM_HIP_CHECK(hipFree(device_ptr));
  return 0;
}

extern "C" int grm_mla_cuda_arena_destroy(MlaDeviceArena* arena) {
  destroy_arena(arena);
  return 0;
}

extern "C" int grm_mla_cublas_route(const float* rows_host,
                                    const float* queries_host, int nodes,
                                    int dim, int query_count, int warmup,
                                    int topk, uint64_t* out_topk_host,
                                    float* elapsed_ms_host) {
  MlaDeviceArena* arena = nullptr;
  int rc = grm_mla_cuda_arena_create(rows_host, nodes, dim, &arena);
  if (rc != 0) return rc;
  rc = grm_mla_cuda_arena_route(arena, queries_host, query_count, dim, warmup,
                                topk, out_topk_host, elapsed_ms_host);
  const int drc = grm_mla_cuda_arena_destroy(arena);
  return rc != 0 ? rc : drc;
}

// =============================================================== extensions

extern "C" int grm_mla_hip_bank_create(const void* rows_host, int row_dtype,
                                       uint64_t nodes, int dim,
                                       const uint64_t* node_ids,
                                       uint64_t capacity,
                                       MlaDeviceArena** out_arena) {
  return create_arena(rows_host, row_dtype, nodes, dim, node_ids, capacity,
                      out_arena);
}

extern "C" int grm_mla_hip_route(MlaDeviceArena* arena, const void* queries,
                                 int query_dtype, int queries_on_device,
                                 int query_count, int dim, int warmup,
                                 int topk, uint64_t* out_ids_host,
                                 float* out_scores_host,
                                 float* elapsed_ms_host) {
  return route_impl(arena, queries, query_dtype, queries_on_device != 0,
                    query_count, dim, warmup, topk, out_ids_host,
                    out_scores_host, elapsed_ms_host);
}

extern "C" int grm_mla_hip_route_noalloc(MlaDeviceArena* arena, const void* d_queries,
                                         int query_dtype, int query_count, int dim, int topk,
                                         uint64_t* d_out_ids, float* d_out_scores) {
  return route_noalloc(arena, d_queries, query_dtype, query_count, dim, topk, d_out_ids,
                       d_out_scores);
}

extern "C" int grm_mla_hip_latent_query(MlaDeviceArena* arena, const void* d_latent,
                                        int latent_dtype, uint64_t tokens,
                                        uint64_t row_stride, int normalize, float* d_out) {
  if (!arena) return grm::fail(-1, "null arena");
  GRM_CHECK_RC(enqueue_latent_query(arena, d_latent, latent_dtype, tokens, row_stride,
                                    normalize, d_out));
  GRM_HIP_CHECK(hipStreamSynchronize(arena->stream));
  grm::clear_error();
  return 0;
}

extern "C" int grm_mla_hip_route_latent(MlaDeviceArena* arena, const void* d_latent,
                                        int latent_dtype, uint64_t tokens,
                                        uint64_t row_stride, int topk,
                                        uint64_t* out_ids_host, float* out_scores_host,
                                        float* elapsed_ms_host) {
  if (!arena) return grm::fail(-1, "null arena");
  if (!arena->d_latent_q) {
    GRM_HIP_CHECK(hipSetDevice(arena->device));
    GRM_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&arena->d_latent_q),
                            static_cast<size_t>(arena->dim) * sizeof(float)));
  }
  // The key is formed on the route stream; the route that follows on the
  // same stream reads it there, with no copy to the host in between.
  GRM_CHECK_RC(enqueue_latent_query(arena, d_latent, latent_dtype, tokens, row_stride, 1,
                                    arena->d_latent_q));
  return route_impl(arena, arena->d_latent_q, kF32, true, 1, static_cast<int>(arena->dim), 0,
                    topk, out_ids_host, out_scores_host, elapsed_ms_host);
}

extern "C" int grm_mla_hip_set_filter_bits(MlaDeviceArena* a, const uint64_t* node_ids,
                                           const uint64_t* bits, uint64_t count) {
  if (!a || (count > 0 && (!node_ids || !bits))) return grm::fail(-1, "invalid arguments");
  std::vector<uint64_t> pairs;
  pairs.reserve(2 * count);
  for (uint64_t i = 0; i < count; ++i) {
    const uint64_t* slot = a->slot_of.find(node_ids[i]);
    if (!slot) return grm::fail(-1, "filter bits for an id that is not live");
    pairs.push_back(*slot);
    pairs.push_back(bits[i]);
  }
  GRM_HIP_CHECK(hipSetDevice(a->device));
  GRM_CHECK_RC(wait_mutations(a));
  if (!a->d_fbits) {
    GRM_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&a->d_fbits),
                            a->capacity * sizeof(uint64_t)));
    GRM_HIP_CHECK(hipMemsetAsync(a->d_fbits, 0, a->capacity * sizeof(uint64_t), a->stream));
  }
  if (count > 0) {
    void* h = nullptr;
    void* d = nullptr;
    GRM_CHECK_RC(stage_upload(a, pairs.size() * sizeof(uint64_t), &h, &d));
    memcpy(h, pairs.data(), pairs.size() * sizeof(uint64_t));
    GRM_HIP_CHECK(hipMemcpyAsync(d, h, pairs.size() * sizeof(uint64_t), hipMemcpyHostToDevice,
                                 a->stream));
    mla_scatter_bits_kernel<<<static_cast<unsigned>((count + 255) / 256), 256, 0, a->stream>>>(
        static_cast<const uint64_t*>(d), count, a->d_fbits);
    GRM_HIP_CHECK(hipGetLastError());
  }
  GRM_HIP_CHECK(hipStreamSynchronize(a->stream));
  grm::clear_error();
  return 0;
}

extern "C" int grm_mla_hip_route_filtered(MlaDeviceArena* a, const void* query, int query_dtype,
                                          int query_on_device, int topk, uint64_t filter_mask,
                                          uint32_t filter_categories, uint64_t* out_ids_host,
                                          float* out_scores_host, float* elapsed_ms_host) {
  if (!a) return grm::fail(-1, "null arena");
  if (filter_categories & ~0xfu) return grm::fail(-1, "filter categories are bits 0..3");
  if (filter_categories == 0) {
    return route_impl(a, query, query_dtype, query_on_device != 0, 1, static_cast<int>(a->dim), 0,
                      topk, out_ids_host, out_scores_host, elapsed_ms_host);
  }
  GRM_HIP_CHECK(hipSetDevice(a->device));
  if (!a->d_fnorms) {
    GRM_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&a->d_fnorms), a->capacity * sizeof(float)));
  }
  if (!a->d_fbits) {
    // no bits set on any node: every node fails an active category
    GRM_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&a->d_fbits),
                            a->capacity * sizeof(uint64_t)));
    GRM_HIP_CHECK(hipMemsetAsync(a->d_fbits, 0, a->capacity * sizeof(uint64_t), a->stream));
  }
  if (a->mut_pending) GRM_HIP_CHECK(hipStreamWaitEvent(a->stream, a->mut[a->mut_last].ev, 0));
  // every slot the route scans: whole 64-slot tiles up to the high water
  // (capacity is a multiple of 64; the tail slots stay NaN)
  const uint64_t n = (a->high_water + grm::kWave - 1) / grm::kWave * grm::kWave;
  if (n > 0) {
    const unsigned blocks =
        static_cast<unsigned>(std::min<uint64_t>((n + 255) / 256, static_cast<uint64_t>(a->cus) * 16));
    mla_filter_norms_kernel<<<blocks, 256, 0, a->stream>>>(a->d_norms, a->d_fbits, n, filter_mask,
                                                          filter_categories, a->d_fnorms);
    GRM_HIP_CHECK(hipGetLastError());
  }
  a->route_norms = a->d_fnorms;
  a->no_batch = true;
  const int rc = route_impl(a, query, query_dtype, query_on_device != 0, 1,
                            static_cast<int>(a->dim), 0, topk, out_ids_host, out_scores_host,
                            elapsed_ms_host);
  a->route_norms = nullptr;
  a->no_batch = false;
  return rc;
}

namespace grm {
// Whether `count` appends fit once `n_drop` live rows are evicted (the
// device store checks this before it replaces an entry's keys).
bool mla_append_fits(const MlaDeviceArena* a, uint64_t n_drop, uint64_t count) {
  const uint64_t live = a->live >= n_drop ? a->live - n_drop : 0;
  return count <= a->capacity - live;
}
}  // namespace grm

extern "C" int grm_mla_hip_score_nodes(MlaDeviceArena* a, const void* query_host,
                                       int query_dtype, const uint64_t* node_ids, uint64_t count,
                                       float* out_scores_host) {
  if (!a || !query_host || (count > 0 && (!node_ids || !out_scores_host))) {
    return grm::fail(-1, "invalid arguments");
  }
  if (query_dtype != kF32 && query_dtype != kBF16) return grm::fail(-1, "query dtype must be F32 or BF16");
  if (count == 0) return 0;
  std::vector<uint64_t> slots(count);
  for (uint64_t i = 0; i < count; ++i) {
    const uint64_t* slot = a->slot_of.find(node_ids[i]);
    if (!slot) return grm::fail(-1, "score of an id that is not live");
    slots[i] = *slot;
  }
  GRM_HIP_CHECK(hipSetDevice(a->device));
  GRM_CHECK_RC(wait_mutations(a));
  const size_t qbytes = static_cast<size_t>(a->dim) * (query_dtype == kF32 ? 4 : 2);
  const size_t sbytes = count * sizeof(uint64_t);
  const size_t obytes = count * sizeof(float);
  const size_t q_off = 0, s_off = (qbytes + 255) / 256 * 256, o_off = s_off + (sbytes + 255) / 256 * 256;
  void* h = nullptr;
  void* d = nullptr;
  GRM_CHECK_RC(stage_upload(a, o_off + obytes, &h, &d));
  memcpy(static_cast<unsigned char*>(h) + q_off, query_host, qbytes);
  memcpy(static_cast<unsigned char*>(h) + s_off, slots.data(), sbytes);
  GRM_HIP_CHECK(hipMemcpyAsync(d, h, o_off, hipMemcpyHostToDevice, a->stream));
  auto* dq = static_cast<unsigned char*>(d) + q_off;
  auto* ds = reinterpret_cast<const uint64_t*>(static_cast<unsigned char*>(d) + s_off);
  auto* dout = reinterpret_cast<float*>(static_cast<unsigned char*>(d) + o_off);
  const size_t lds = static_cast<size_t>(a->dim_pad) * sizeof(double);
  // one thread per listed node, spread over the compute units; each block
  // stages the query itself
  const unsigned blocks = static_cast<unsigned>(
      std::min<uint64_t>((count + 255) / 256, static_cast<uint64_t>(a->cus) * 4));
  if (a->dtype == kF32) {
    mla_score_slots_kernel<kF32><<<blocks, 256, lds, a->stream>>>(a->d_tiles, a->d_norms, a->capacity,
                                                             a->chunks, a->dim, a->dim_pad, dq,
                                                             query_dtype, ds, count, dout);
  } else {
    mla_score_slots_kernel<kBF16><<<blocks, 256, lds, a->stream>>>(a->d_tiles, a->d_norms, a->capacity,
                                                              a->chunks, a->dim, a->dim_pad, dq,
                                                              query_dtype, ds, count, dout);
  }
  GRM_HIP_CHECK(hipGetLastError());
  GRM_HIP_CHECK(hipMemcpyAsync(static_cast<unsigned char*>(h) + o_off, dout, obytes,
                               hipMemcpyDeviceToHost, a->stream));
  GRM_HIP_CHECK(hipStreamSynchronize(a->stream));
  memcpy(out_scores_host, static_cast<unsigned char*>(h) + o_off, obytes);
  grm::clear_error();
  return 0;
}

extern "C" int grm_mla_hip_append(MlaDeviceArena* a, const void* rows_host,
                                  int row_dtype, uint64_t count,
                                  const uint64_t* node_ids,
                                  uint64_t* out_epoch) {
  if (!a || (count > 0 && (!rows_host || !node_ids))) {
    return grm::fail(-1, "invalid append arguments");
  }
  if (row_dtype != a->dtype) return grm::fail(-1, "append dtype differs from bank");
  if (count == 0) {
    if (out_epoch) *out_epoch = a->epoch;
    return 0;
  }
  // The ids enter the table at once, which finds live and repeated ones.
  // An append that does not come about leaves nothing behind: what it put
  // into the tables goes, and rows already placed are evicted.
  struct Entered {
    MlaDeviceArena* a;
    const uint64_t* ids;
    uint64_t n = 0;            // ids in the table
    const uint64_t* slots = nullptr;  // the slots taken, in order (in the stage)
    uint64_t taken = 0;
    const uint64_t* d_slots = nullptr;  // ... for the device, from when rows may be placed
    uint64_t high_water = 0;   // before the first was taken
    ~Entered() {
      if (d_slots) (void)launch_evict(a, d_slots, taken);
      if (taken > 0) (void)hipStreamSynchronize(a->side);  // the stage is read no more
      for (uint64_t i = 0; i < taken; ++i) {
        a->slot_id[slots[i]] = kNoId;
        if (slots[i] < high_water) a->free_slots.insert(slots[i]);
      }
      if (taken > 0) a->high_water = high_water;
      for (uint64_t i = 0; i < n; ++i) a->slot_of.erase(ids[i]);
    }
  } entered{a, node_ids};
  a->slot_of.reserve(a->slot_of.size() + count);
  for (uint64_t i = 0; i < count; ++i) {
    if (!a->slot_of.emplace(node_ids[i], 0)) {
      return grm::fail(-1, "append id already live or repeated");
    }
    entered.n = i + 1;
    if (node_ids[i] == kNoId) return grm::fail(-1, "node id UINT64_MAX is reserved");
  }
  const uint64_t room = a->free_slots.size() + (a->capacity - a->high_water);
  if (count > room) return grm::fail(-3, "MLA bank capacity exceeded");
  GRM_HIP_CHECK(hipSetDevice(a->device));
  const size_t row_bytes = static_cast<size_t>(a->dim) * elem_size(a->dtype);
  const size_t bytes = count * (2 * sizeof(uint64_t) + row_bytes);
  const bool direct = bytes <= kDirectAppendBytes;
  // small updates take the two stages in turn; large ones share the bank's
  // one (and its device copy), once the updates before have read theirs, so
  // that a bank holds one pinned copy of its largest append
  MutStage* stage = nullptr;
  void* h = nullptr;
  void* d = nullptr;
  GRM_CHECK_RC(next_stage(a, direct ? bytes : 0, &stage));
  if (direct) {
    h = stage->buf.host;
    d = stage->buf.dev;
  } else {
    GRM_CHECK_RC(stage_upload(a, bytes, &h, &d));
  }
  uint64_t* h_slots = static_cast<uint64_t*>(h);
  uint64_t* h_ids = h_slots + count;
  unsigned char* h_rows = reinterpret_cast<unsigned char*>(h_ids + count);
  const uint64_t* d_slots = static_cast<const uint64_t*>(d);
  const unsigned char* d_rows = reinterpret_cast<const unsigned char*>(d_slots + 2 * count);
  entered.slots = h_slots;
  entered.high_water = a->high_water;
  for (uint64_t i = 0; i < count; ++i) {
    uint64_t slot = a->free_slots.pop_lowest();
    if (slot == kNoId) slot = a->high_water++;
    h_slots[i] = slot;
    h_ids[i] = node_ids[i];
    a->slot_id[slot] = node_ids[i];
    *a->slot_of.find(node_ids[i]) = slot;
    entered.taken = i + 1;
  }
  if (direct) {
    // The placement reads the rows over the bus itself, in parts that
    // follow the host's copy: no copy on the device side, and the bus is
    // busy while the host still copies.  1000 rows of 288 fp32 values out
    // and in, then a route over 100k: 370 -> 123 us a call, with the
    // placement kernel, the flat tables and the second stage (an append no
    // longer waits for the evict's kernel).  The parts' launches take 8 to
    // 15 us each, the bus's time for 512 KiB.
    const uint64_t part = std::max<uint64_t>(grm::mla::kPlaceRows,
                                             kAppendPartBytes / row_bytes / grm::mla::kPlaceRows *
                                                 grm::mla::kPlaceRows);
    entered.d_slots = d_slots;
    for (uint64_t r0 = 0; r0 < count; r0 += part) {
      const uint64_t n = std::min<uint64_t>(part, count - r0);
      memcpy(h_rows + r0 * row_bytes, static_cast<const unsigned char*>(rows_host) + r0 * row_bytes,
             n * row_bytes);
      GRM_CHECK_RC(launch_place(a, d_rows + r0 * row_bytes, n, d_slots + r0, d_slots + count + r0, 0, a->side));
    }
  } else {
    memcpy(h_rows, rows_host, count * row_bytes);
    GRM_HIP_CHECK(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, a->side));
    entered.d_slots = d_slots;
    GRM_CHECK_RC(launch_place(a, d_rows, count, d_slots, d_slots + count, 0, a->side));
  }
  GRM_CHECK_RC(end_update(a, stage));
  entered.n = entered.taken = 0;
  entered.d_slots = nullptr;
  a->live += count;
  a->epoch += 1;
  if (out_epoch) *out_epoch = a->epoch;
  grm::clear_error();
  return 0;
}

extern "C" int grm_mla_hip_evict(MlaDeviceArena* a, const uint64_t* node_ids,
                                 uint64_t count, uint64_t* out_epoch) {
  if (!a || (count > 0 && !node_ids)) return grm::fail(-1, "invalid evict arguments");
  if (count == 0) {
    if (out_epoch) *out_epoch = a->epoch;
    return 0;
  }
  // the slots are marked free at once, which finds repeated ids, and
  // unmarked again if the evict does not come about
  struct Marked {
    MlaDeviceArena* a;
    std::vector<uint64_t> slots;
    bool staged = false;
    bool keep = false;
    ~Marked() {
      if (keep) return;
      if (staged) (void)hipStreamSynchronize(a->side);  // the stage is read no more
      for (uint64_t s : slots) a->free_slots.erase(s);
    }
  } marked{a, {}};
  marked.slots.reserve(count);
  for (uint64_t i = 0; i < count; ++i) {
    const uint64_t* slot = a->slot_of.find(node_ids[i]);
    if (!slot || !a->free_slots.insert(*slot)) {
      return grm::fail(-1, "evict id not live or repeated");
    }
    marked.slots.push_back(*slot);
  }
  const std::vector<uint64_t>& slots = marked.slots;
  GRM_HIP_CHECK(hipSetDevice(a->device));
  const size_t bytes = count * sizeof(uint64_t);
  MutStage* stage = nullptr;
  GRM_CHECK_RC(next_stage(a, bytes, &stage));
  memcpy(stage->buf.host, slots.data(), bytes);
  marked.staged = true;
  GRM_CHECK_RC(launch_evict(a, static_cast<const uint64_t*>(stage->buf.dev), count));  // read in place
  GRM_CHECK_RC(end_update(a, stage));
  marked.keep = true;
  for (uint64_t s : slots) {
    a->slot_of.erase(a->slot_id[s]);
    a->slot_id[s] = kNoId;
  }
  // Trailing free slots shrink the scanned range.
  while (a->high_water > 0 && a->slot_id[a->high_water - 1] == kNoId) {
    a->free_slots.erase(a->high_water - 1);
    a->high_water -= 1;
  }
  a->live -= count;
  a->epoch += 1;
  if (out_epoch) *out_epoch = a->epoch;
  grm::clear_error();
  return 0;
}

extern "C" int grm_mla_hip_sync(MlaDeviceArena* a) {
  if (!a) return grm::fail(-1, "null arena");
  GRM_HIP_CHECK(hipSetDevice(a->device));
  return wait_mutations(a);
}

extern "C" int grm_mla_hip_bank_info(MlaDeviceArena* a, uint64_t* out6) {
  if (!a || !out6) return grm::fail(-1, "null argument");
  out6[0] = a->live;
  out6[1] = a->capacity;
  out6[2] = a->high_water;
  out6[3] = a->epoch;
  out6[4] = a->dim;
  out6[5] = static_cast<uint64_t>(a->dtype);
  return 0;
}

extern "C" int grm_mla_hip_route_stats(MlaDeviceArena* a, uint64_t* out4) {
  if (!a || !out4) return grm::fail(-1, "null argument");
  out4[0] = a->batch_queries;
  out4[1] = a->batch_fallbacks;
  out4[2] = a->single_queries;
  out4[3] = a->batch_passes;
  return 0;
}

extern "C" int grm_mla_hip_screen_ms(MlaDeviceArena* a, float* ms) {
  if (!a || !ms) return grm::fail(-1, "null argument");
  *ms = a->screen_ms;
  return 0;
}

// ------------------------------------------------------- screen-bound probe
//
// Test entry: runs the batched route's screen (the same kernel, in its
// probe form) over every slot of a small bank and returns each
// screened score s~ with its query's bound B, so a test can hold
// |s~ - law score| <= B for every (query, node) pair.  Not on any route
// path; allocates its own buffers.
extern "C" int grm_mla_hip_probe_screen(MlaDeviceArena* a, const void* queries_host,
                                        int query_dtype, int query_count, float* out_values_host,
                                        double* out_bounds_host, uint64_t* out_slot_ids_host) {
  if (!a || !queries_host || !out_values_host || !out_bounds_host) {
    return grm::fail(-1, "null argument");
  }
  if (query_dtype != kF32 && query_dtype != kBF16) return grm::fail(-1, "query dtype must be F32 or BF16");
  BatchPlan p;
  if (!batch_plan(a, &p)) {
    return grm::fail(-1, "bank has no batched screen (rows too long or too many)");
  }
  if (query_count <= 0 || query_count > p.qp_max) return grm::fail(-1, "query_count out of range");
  const PassShape shape = pass_shape(a, p, query_count);
  const int qp = shape.qp;
  const uint64_t n = a->high_water;
  if (n == 0) return grm::fail(-1, "empty bank");
  if (a->capacity * static_cast<uint64_t>(qp) > (1ull << 26)) {
    return grm::fail(-1, "probe is for banks of at most 2^26 / 256 slots");
  }
  GRM_HIP_CHECK(hipSetDevice(a->device));
  struct Buf {
    void* p = nullptr;
    ~Buf() {
      if (p) (void)hipFree(p);
    }
  } d_q, d_planes, d_vals, d_bounds;
  const size_t qbytes = static_cast<size_t>(query_count) * a->dim * elem_size(query_dtype);
  GRM_HIP_CHECK(hipMalloc(&d_q.p, qbytes));
  GRM_HIP_CHECK(hipMalloc(&d_planes.p, static_cast<size_t>(qp) * a->capacity * sizeof(uint32_t)));
  GRM_HIP_CHECK(hipMalloc(&d_vals.p, static_cast<size_t>(query_count) * n * sizeof(float)));
  GRM_HIP_CHECK(hipMalloc(&d_bounds.p, static_cast<size_t>(query_count) * sizeof(double)));
  if (!reserve_batch(a, p, shape.ring)) return grm::fail(-1, "no memory for the probe's buffers");
  if (a->mut_pending) GRM_HIP_CHECK(hipStreamWaitEvent(a->stream, a->mut[a->mut_last].ev, 0));
  GRM_HIP_CHECK(hipMemcpyAsync(d_q.p, queries_host, qbytes, hipMemcpyHostToDevice, a->stream));
  const PassQueries pq{d_q.p, query_dtype, query_count};
  ScreenLaunch l;
  GRM_CHECK_RC(screen_launch(a, p, shape, pq, static_cast<uint32_t*>(d_planes.p), PassMarks{}, &l));
  GRM_CHECK_RC(grm::mla::launch_probe_screen(l));
  const uint32_t len = grm::mla::merge_len(a->dim);
  grm::mla::mla_batch_probe_finish_kernel<<<query_count, grm::kWave, len * sizeof(double), a->stream>>>(
      static_cast<const uint32_t*>(d_planes.p), a->capacity, static_cast<uint32_t>(n), a->d_inv_qn,
      d_q.p, query_dtype, a->dim, len, screen_bound(a, p, shape.ibits), a->d_min_norm,
      static_cast<float*>(d_vals.p), static_cast<double*>(d_bounds.p));
  GRM_HIP_CHECK(hipGetLastError());
  GRM_HIP_CHECK(hipMemcpyAsync(out_values_host, d_vals.p, static_cast<size_t>(query_count) * n * sizeof(float),
                               hipMemcpyDeviceToHost, a->stream));
  GRM_HIP_CHECK(hipMemcpyAsync(out_bounds_host, d_bounds.p, static_cast<size_t>(query_count) * sizeof(double),
                               hipMemcpyDeviceToHost, a->stream));
  if (out_slot_ids_host) {
    GRM_HIP_CHECK(hipMemcpyAsync(out_slot_ids_host, a->d_ids, n * sizeof(uint64_t),
                                 hipMemcpyDeviceToHost, a->stream));
  }
  GRM_HIP_CHECK(hipStreamSynchronize(a->stream));
  grm::clear_error();
  return 0;
}
