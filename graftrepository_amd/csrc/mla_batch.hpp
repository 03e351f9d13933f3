// mla_batch.hpp -- batched MLA route on the matrix cores: its kernels.
//
// Q queries against a bank, law as the single-query route
// (cpp/grm_runtime.cpp:3518-3545):
//   score = float( dot / (qnorm * (double)norm_f + 1e-8) ),  dot in fp64, d ascending.
// The scores of all Q x N pairs form a dense contraction.  It runs as bf16
// MFMA 32x32x16 with fp32 accumulation, reduced on the fly: the score
// matrix never leaves registers.  fp32 rows enter as the sum of two bf16
// values, as do their queries (three products).
//
//  * screen  -- every node tile (32 slots) against every query of a pass
//               (up to 128 staged in LDS, mla_batch_stream_kernel, or 256 in
//               registers, mla_batch_ring_kernel).  The screened score
//               s~ = u * (1/qnorm), u = acc * (1/norm_f) with the slot's
//               index written into the low `ibits` mantissa bits of u,
//               obeys |s~ - score| <= B, B a per-query constant (see
//               mla_batch_merge_kernel).  Each lane follows one query over
//               half of every tile its wavefront walks and keeps the three
//               largest u: the two best (each carrying its slot) and the
//               largest it did not keep; the two halves of a query are
//               merged at the end, one sub-stream per (wavefront, query).
//               "Largest" is the order of u's bits as a signed integer,
//               which is the float order on values >= +0 and puts every
//               negative value (and -0) below them; the merge certifies a
//               query only when its threshold t is positive, so only
//               positive values decide.
//  * merge   -- one block per query over the sub-streams' kept entries:
//               v_k = the k-th best kept s~, t = v_k - 2B.  A node whose
//               s~ lies below t scores below v_k - B, so if every
//               sub-stream's largest dropped s~ lies below t, the law's
//               top-k is among the kept entries at or above t.  Those are
//               scored with the law in fp64 and ranked (score desc, node id
//               asc); the k-th exact score must reach v_k - B (which fails
//               only where a law score is not finite).  A query without
//               this certificate is routed again on the exact single-query
//               path.
#pragma once

#include "grm_common.hpp"
#include "mla_values.hpp"

namespace grm {
namespace mla {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// v_med3_i32 and v_and_or_b32: the compiler forms neither from the
// equivalent min/max and and/or expressions, and the screen's per-score
// work is these two instructions and a maximum.
// b = med3(a, b, c), in place
__device__ __forceinline__ void med3_i32_into(int a, int& b, int c) {
  asm("v_med3_i32 %0, %1, %0, %2" : "+v"(b) : "v"(a), "v"(c));
}
__device__ __forceinline__ uint32_t and_or_b32(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

constexpr int kBatchWaves = 8;       // wavefronts per stream-screen block (one block per CU)
constexpr int kStreamMaxCols = 128;  // queries per stream-screen pass
constexpr int kEntryPlanes = 3;      // u1, u2, nk

// Screen results, one row of n_sub values per (plane, query): plane p of
// query q at planes + (p*QP + q)*n_sub, sub-stream i = the wavefront:
//   u1, u2  the two best u a sub-stream kept (float bits, slot code in
//   the low ibits bits), nk the largest u it did not keep.
//
// Slot code of a value: ((t - t_begin) << 4) | r for result register r in
// tile t of a sub-stream whose tiles start at t_begin, in the stream screen
// with the lane half at bit ibits - 1 (the ring screen's halves are
// sub-streams of their own).  The host picks ibits from the longest run of
// tiles a sub-stream walks.
// Writing the code moves u by less than 2^(ibits-23) |u| (2^(ibits-149)
// near zero), which the merge adds to B.

// bf16 pattern of f, to nearest even.
__device__ __forceinline__ uint32_t bf16_bits_rne(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// ---------------------------------------------------------- stream screen
//
// Passes of up to 32*CT queries against a bank of either type and any row
// length whose query rows fit LDS.  Grid = one block of kBatchWaves
// wavefronts per CU.  Sub-stream i walks 32-slot tiles
// [i*T/n_sub, (i+1)*T/n_sub); with fewer tiles than wavefronts each tile
// is a sub-stream of its own and they are dealt out block by block, so
// every CU takes part.
//
// LDS holds the pass's queries: s_qb[QP][stride] bf16 (stride =
// 16*steps + 8, an odd number of 16-byte pieces, so the reads of 32 rows
// hit distinct banks; zero past dim), for an fp32 bank followed by the
// same array of the remainders q - bf16(q), rounded to bf16.  For K-step
// ks the A fragment of lane l is dims 16*ks + 8*(l/32) .. +8 of slot
// tile*32 + l%32 (one 16-byte chunk of a bf16 bank, two of an fp32 bank)
// and the B fragment the same dims of query ct*32 + l%32; result register
// r of lane l is slot tile*32 + 8*(r/4) + 4*(l/32) + r%4 against that
// query.  An fp32 fragment x is split in registers, xh = bf16(x),
// xl = bf16(x - xh), and takes three products: xh qh + xl qh + xh ql.
//
// The wavefront's fragments form a ring of P K-steps: a step's registers
// are loaded again, for the step P further on (in this tile or the next),
// as soon as it is consumed, so P KiB (bf16) or 2 P KiB (fp32) per
// wavefront are always in flight.  A row of ks_need K-steps runs
// nb * P >= ks_need steps; the steps past its end, and the chunks past its
// end in its last step, read the row's last chunk again, against zeros
// (stored rows are finite).
//
// What bounds it: HBM.  Per tile of 288 fp32 values a wavefront issues 18
// steps of 24 conversions and 3 CT MFMAs -- 54 MFMAs of 32 cycles at CT = 1
// against 36 KiB to stream, 15 % of the matrix cores' rate.  On small banks
// (1.5 tiles a wavefront at 100k x 280 fp32, 27.6 us; 2.3 at 150k x 200
// bf16, 22.2 us) the trips before the first tile and the last reload of the
// ring, which is never folded, weigh as much: 1.26 and 1.36 x the bank's
// bytes come from HBM.
//
// kProbe (tests of the screen bound only): every coded u goes to
// planes[q*cap + slot] instead of the lists, and nothing else is written.
template <int DT, int P, int CT, bool kProbe = false>
__global__ __launch_bounds__(kBatchWaves * kWave) void mla_batch_stream_kernel(
    const u32x4* __restrict__ tiles, const float* __restrict__ norms, uint64_t cap,
    uint32_t chunks, uint32_t n_tiles32, uint32_t n_sub, uint32_t nb, uint32_t ks_need,
    const void* __restrict__ query, int q_dtype, int qc, uint32_t dim, float* __restrict__ inv_qn,
    int ibits, uint32_t* __restrict__ planes, RouteStamps stamps, unsigned seq,
    unsigned long long* __restrict__ screen_tick) {
  route_start_stamp(stamps, seq);
  if (screen_tick && blockIdx.x == 0 && threadIdx.x == 0) *screen_tick = wall_clock64();
  constexpr bool kSplit = DT == kF32;
  constexpr int V = kSplit ? 2 : 1;  // 16-byte pieces of a fragment
  constexpr int QP = 32 * CT;
  const uint32_t steps = nb * P;
  const uint32_t stride = 16 * steps + 8;
  extern __shared__ uint16_t s_qb[];
  uint16_t* s_ql = s_qb + QP * stride;  // remainders (fp32 banks)
  const int lane = threadIdx.x & (kWave - 1);
  const int half = lane >> 5;
  const int col = lane & 31;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t sub = n_sub == gridDim.x * kBatchWaves ? blockIdx.x * kBatchWaves + wv
                                                        : wv * gridDim.x + blockIdx.x;
  uint32_t t_begin = 0, t_end = 0;
  if (sub < n_sub) {
    t_begin = static_cast<uint32_t>(static_cast<uint64_t>(sub) * n_tiles32 / n_sub);
    t_end = static_cast<uint32_t>(static_cast<uint64_t>(sub + 1) * n_tiles32 / n_sub);
  }
  auto load_frag = [&](u32x4 (&a)[V], uint32_t t, uint32_t ks) {
    const uint32_t c0 = V * (2 * min(ks, ks_need - 1) + half);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const uint32_t c = min(c0 + v, chunks - 1);
      a[v] = __builtin_nontemporal_load(tiles + static_cast<uint64_t>(c) * cap +
                                        static_cast<uint64_t>(t) * 32 + col);
    }
  };
  // Row norms of a tile are wave-uniform loads, fetched one tile ahead.
  float ns[32];
  auto load_norms = [&](uint32_t t) {
#pragma unroll
    for (int j = 0; j < 32; ++j) ns[j] = norms[static_cast<size_t>(t) * 32 + j];
  };
  u32x4 a[P][V];
  if (t_begin < t_end) {
    load_norms(t_begin);
#pragma unroll
    for (int j = 0; j < P; ++j) load_frag(a[j], t_begin, j);
  }
  // Stage the queries while the first fragments are on their way: a
  // wavefront per query row, a pair of values per lane and iteration.
  // Block j also forms 1/||q_j|| (fp32; NaN for columns past qc).
  auto value = [&](uint32_t q, uint32_t d) -> float {
    const size_t i = static_cast<size_t>(q) * dim + min(d, dim - 1);
    const float f = q_dtype == kBF16 ? bf16_to_f32(static_cast<const uint16_t*>(query)[i])
                                     : static_cast<const float*>(query)[i];
    return d < dim ? f : 0.0f;
  };
  constexpr int kStage = 4;
  for (uint32_t q = wv; q < QP; q += kBatchWaves) {
    uint32_t* hi = reinterpret_cast<uint32_t*>(s_qb + q * stride);
    uint32_t* lo = reinterpret_cast<uint32_t*>(s_ql + q * stride);
    const uint32_t qs = min(q, static_cast<uint32_t>(qc - 1));
    for (uint32_t p0 = lane; p0 < 8 * steps; p0 += kStage * kWave) {
      float f[kStage][2];
#pragma unroll
      for (int j = 0; j < kStage; ++j) {
        f[j][0] = value(qs, 2 * (p0 + j * kWave));
        f[j][1] = value(qs, 2 * (p0 + j * kWave) + 1);
      }
#pragma unroll
      for (int j = 0; j < kStage; ++j) {
        const uint32_t p = p0 + j * kWave;
        if (p >= 8 * steps) continue;
        const bool on = q < static_cast<uint32_t>(qc);
        const uint32_t h0 = on ? bf16_bits_rne(f[j][0]) : 0u, h1 = on ? bf16_bits_rne(f[j][1]) : 0u;
        hi[p] = h0 | (h1 << 16);
        if constexpr (kSplit) {
          const uint32_t l0 = on ? bf16_bits_rne(f[j][0] - bf16_to_f32(h0)) : 0u;
          const uint32_t l1 = on ? bf16_bits_rne(f[j][1] - bf16_to_f32(h1)) : 0u;
          lo[p] = l0 | (l1 << 16);
        }
      }
    }
  }
  if (wv == kBatchWaves - 1) {
    for (uint32_t q = blockIdx.x; q < QP; q += gridDim.x) {
      double ss = 0.0;
      if (q < static_cast<uint32_t>(qc)) {
        for (uint32_t d = lane; d < dim; d += kWave) {
          const double f = value(q, d);
          ss = fma(f, f, ss);
        }
      }
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) ss += __shfl_xor(ss, off);
      if (lane == 0) {
        inv_qn[q] = q < static_cast<uint32_t>(qc) ? static_cast<float>(1.0 / sqrt(ss)) : __builtin_nanf("");
      }
    }
  }
  __syncthreads();

  // per column tile: the three largest coded u as signed-integer bits
  // (b1 >= b2 >= b3)
  int b1[CT], b2[CT], b3[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) b1[ct] = b2[ct] = b3[ct] = INT32_MIN;
  const uint32_t keep_mask = ~((1u << ibits) - 1u);
  const uint16_t* qrow = s_qb + col * stride + 8 * half;
  // Lanes track u = acc * (1/norm_f); s~ = u * (1/qnorm) is formed by the
  // merge (rounding is monotone, so the largest u give the largest s~).
  // A slot that never ranks (tombstone, unused slot, non-finite row: the
  // bank stores its row as zeros) has 1/norm_f = -0, so u is a zero and
  // never outranks a positive value.  An accumulation may overflow only
  // where the merge does not certify (it checks the norms), or on a row
  // whose own norm overflowed (a law score of zero; the norms' range leaves
  // it out): its u is then a NaN.  One with a set sign bit, as gfx950 forms
  // it, lies below +0 in the integer order and decides nothing; one with a
  // clear sign bit would lie above every number, and so be its sub-stream's
  // largest, which voids the query's certificate.  u's low bits take the
  // slot code, and the three largest move by two medians and a maximum of
  // the integer bits: b3 = med3(b2, b3, v), b2 = med3(b1, b2, v),
  // b1 = max(b1, v) keep b1 >= b2 >= b3 the three
  // largest values seen.
  auto offer = [&](int v, int ct) {
    med3_i32_into(b2[ct], b3[ct], v);
    med3_i32_into(b1[ct], b2[ct], v);
    b1[ct] = max(b1[ct], v);
  };
  for (uint32_t t = t_begin; t < t_end; ++t) {
    // 1/norm_f: -0 for a slot that never ranks (norm NaN) and for a norm
    // that overflowed (its law score is a zero), 0 for an all-zero row
    // (score 0, exact).
    float wr[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int j = 8 * (r / 4) + (r % 4);
      const float nf = __uint_as_float(half ? __float_as_uint(ns[j + 4]) : __float_as_uint(ns[j]));
      wr[r] = nf == 0.0f ? 0.0f : (nf < INFINITY ? __builtin_amdgcn_rcpf(nf) : -0.0f);
    }
    const uint32_t t_next = t + 1 < t_end ? t + 1 : t;  // the last reload is never folded
    load_norms(t_next);
    f32x16 acc[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[ct] = f32x16{};
    for (uint32_t kb = 0; kb < nb; ++kb) {
      const bool last = kb + 1 == nb;
      const uint32_t t_load = last ? t_next : t;
      const uint32_t k_load = last ? 0 : (kb + 1) * P;
#pragma unroll
      for (int j = 0; j < P; ++j) {
        const uint16_t* qk = qrow + 16 * (kb * P + j);
        u32x4 bh[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          bh[ct] = *reinterpret_cast<const u32x4*>(qk + ct * 32 * stride);
        }
        if constexpr (kSplit) {
          u32x4 bl[CT];
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            bl[ct] = *reinterpret_cast<const u32x4*>(qk + (QP + ct * 32) * stride);
          }
          const u32x4 w0 = a[j][0], w1 = a[j][V - 1];
          const uint32_t w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
          bf16x8 xh, xl;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float x = __uint_as_float(w[e]);
            xh[e] = static_cast<__bf16>(x);
            xl[e] = static_cast<__bf16>(x - static_cast<float>(xh[e]));
          }
          load_frag(a[j], t_load, k_load + j);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, __builtin_bit_cast(bf16x8, bh[ct]),
                                                              acc[ct], 0, 0, 0);
          }
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xl, __builtin_bit_cast(bf16x8, bh[ct]),
                                                              acc[ct], 0, 0, 0);
          }
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, __builtin_bit_cast(bf16x8, bl[ct]),
                                                              acc[ct], 0, 0, 0);
          }
        } else {
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[j][0]),
                                                              __builtin_bit_cast(bf16x8, bh[ct]),
                                                              acc[ct], 0, 0, 0);
          }
          load_frag(a[j], t_load, k_load + j);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    const uint32_t tcode = (static_cast<uint32_t>(half) << (ibits - 1)) | ((t - t_begin) << 4);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t u = and_or_b32(__float_as_uint(acc[ct][r] * wr[r]), keep_mask,
                                      tcode | static_cast<uint32_t>(r));
        if constexpr (kProbe) {
          const uint32_t slot = t * 32u + 8u * (r / 4) + 4u * half + (r % 4);
          planes[static_cast<size_t>(ct * 32u + col) * cap + slot] = u;
        } else {
          offer(static_cast<int>(u), ct);
        }
      }
    }
  }
  if constexpr (kProbe) return;
  if (sub >= n_sub) return;
  // The two lane halves of a column hold disjoint slots: merge their lists
  // (each half's three values go through the same update as a score).
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int o1 = __shfl_xor(b1[ct], 32);
    const int o2 = __shfl_xor(b2[ct], 32);
    const int o3 = __shfl_xor(b3[ct], 32);
    offer(o1, ct);
    offer(o2, ct);
    offer(o3, ct);
    if (half == 0) {
      const size_t q = static_cast<size_t>(ct * 32 + col);
      planes[(0 * QP + q) * n_sub + sub] = static_cast<uint32_t>(b1[ct]);
      planes[(1 * QP + q) * n_sub + sub] = static_cast<uint32_t>(b2[ct]);
      planes[(2 * QP + q) * n_sub + sub] = static_cast<uint32_t>(b3[ct]);
    }
  }
}

// ------------------------------------------------------------ ring screen
//
// The same screen for a full pass of 256 queries on a bf16 bank, with the
// roles of LDS and registers swapped: each wavefront holds 64 queries' B
// fragments in registers for the whole bank, and the bank's 32-slot tiles
// stream into LDS, so every A fragment read from LDS feeds two MFMAs (the
// query fragments of mla_batch_stream_kernel cost one 1 KiB LDS read per
// MFMA).
//
//  * One block of four wavefronts per CU; wavefront w holds queries
//    [64 w, 64 w + 64) and has SIMD w to itself, so its 512 registers hold
//    the queries, two sets of accumulators and A fragments four K-steps
//    ahead.  The MFMAs of tile s and the reductions of tile s - 1 form one
//    straight-line region, each MFMA followed by its share of the
//    reductions and a scheduling barrier: the matrix core and the VALU work
//    side by side within the wavefront.
//  * Block b of W walks tiles [b * n_tiles32 / W, (b + 1) * n_tiles32 / W),
//    one per step, as kRingSegs runs: run j = kRingSegs b + g starts at
//    j * n_tiles32 / (kRingSegs W).  Each lane starts its lists afresh at a
//    run's first tile and keeps the finished ones in registers, so
//    sub-stream (2 b + half) kRingSegs + g is run j as seen by one lane
//    half, and its slot code has no half bit.  With one sub-stream per
//    block, three of a query's best rows in one of 256 sub-streams sent 0.3
//    (k = 8) to 2.7 (k = 16) of 256 queries to the exact kernel, 100 us
//    each at 1M x 288; with 2,048 about one call in a hundred has one, and
//    the shorter code tightens the bound (2^-14 instead of 2^-11).
//  * A ring of kRing tiles in LDS (2 KS chunk planes of 512 bytes each,
//    chunk c of the tile at c * 512) with their 32 slot weights.  Direct
//    loads (global_load_lds_dwordx4) fill it without registers.  A step is
//    KS tile loads of 1 KiB (two chunk planes each) and one weight load,
//    spread so that every wavefront issues the same number
//    (kLoadsPerWave); wavefronts without a tile load left for their last
//    issue all bring the weights (8 lanes carry the 128 bytes, the rest
//    repeat them into the pad of a 1 KiB weight area).  kRing - 1 tiles are
//    in flight while one is screened.
//  * Step s: each wavefront waits for its own loads of tile s (vmcnt) and
//    its LDS reads of tile s - 1 (lgkmcnt); the block barrier then makes
//    the whole tile visible and says every wavefront is done with tile
//    s - 1, whose slot the loads of tile s + kRing - 1 then refill.  Loads
//    past the block's last tile re-read that tile (never screened), so
//    every step has the same load count.
//  * The slot weights 1/norm_f come from mla_batch_weights_kernel, the
//    values mla_batch_stream_kernel forms per tile (same reciprocal).
template <int KS>
struct RingShape {
  static constexpr int kRing = 8;                         // tiles in LDS
  static constexpr int kTileU4 = 2 * KS * 32;             // u32x4 per tile
  static constexpr int kTileLoads = KS;                   // 1 KiB loads per tile
  static constexpr int kLoadsPerWave = kTileLoads / 4 + 1;  // every wavefront, every step
  static constexpr size_t kWeightOffset = static_cast<size_t>(kRing) * kTileU4 * 16;
  static constexpr size_t kWeightArea = 1024;             // bytes per tile (128 used)
  static constexpr size_t kLds = kWeightOffset + static_cast<size_t>(kRing) * kWeightArea;
};

constexpr int kRingWaves = 4;      // wavefronts per block, one block per CU
constexpr int kRingSegs = 4;       // runs of tiles with lists of their own, per block
constexpr int kRingQueries = 256;  // queries per ring pass

// s_waitcnt vmcnt(n) lgkmcnt(0) (gfx9 encoding; expcnt left alone): the
// wavefront's loads but the last n are done, and so are its LDS reads.
template <int N>
__device__ __forceinline__ void wait_vmcnt_lds() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0070);
}

// The slot weights the screens multiply by: 1/norm_f (v_rcp_f32), 0 for
// an all-zero row, -0 for a slot that never ranks (NaN norm: tombstone,
// unused slot, non-finite row) and for a norm that overflowed.
static __global__ void mla_batch_weights_kernel(const float* __restrict__ norms, uint64_t n,
                                         float* __restrict__ winv) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float nf = norms[i];
  winv[i] = nf == 0.0f ? 0.0f : (nf < INFINITY ? __builtin_amdgcn_rcpf(nf) : -0.0f);
}

template <int KS, bool kProbe = false>
__global__ __launch_bounds__(kRingWaves * kWave, 1) void mla_batch_ring_kernel(
    const u32x4* __restrict__ tiles, const float* __restrict__ winv, uint64_t cap,
    uint32_t n_tiles32, const uint16_t* __restrict__ qpad, int ibits, uint32_t* __restrict__ planes,
    unsigned long long* __restrict__ screen_tick) {
  if (screen_tick && blockIdx.x == 0 && threadIdx.x == 0) *screen_tick = wall_clock64();
  using RS = RingShape<KS>;
  constexpr int stride = 16 * KS + 8;  // qpad row stride (bf16 elements)
  constexpr int QP = kRingQueries;
  constexpr int kPre = 4;              // A fragments in flight ahead of their MFMAs
  extern __shared__ u32x4 s_ring[];   // [kRing][2 KS][32 slots], then the weights
  unsigned char* s_w = reinterpret_cast<unsigned char*>(s_ring) + RS::kWeightOffset;
  const int lane = threadIdx.x & (kWave - 1);
  const int half = lane >> 5;
  const int col = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // query group
  const uint32_t W = gridDim.x;
  const uint32_t t_begin = static_cast<uint32_t>(static_cast<uint64_t>(blockIdx.x) * n_tiles32 / W);
  const uint32_t t_end = static_cast<uint32_t>(static_cast<uint64_t>(blockIdx.x + 1) * n_tiles32 / W);
  const uint32_t steps = t_end - t_begin;

  // B fragments of the wavefront's 64 queries: column tile c, K-step ks:
  // query 64 wv + 32 c + col at dims 16 ks + 8 half .. +8
  u32x4 bq[2][KS];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const uint16_t* row = qpad + static_cast<size_t>(64 * wv + 32 * c + col) * stride + 8 * half;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) bq[c][ks] = *reinterpret_cast<const u32x4*>(row + 16 * ks);
  }
  // The fragments are in registers before the ring's loads start, so the
  // only loads a step waits for are the ring's own (the empty asm uses
  // each value, which keeps its load ahead of the ring's).  They live in
  // AGPRs (the MFMAs read their B operand there), which leaves the VGPRs
  // to the accumulators, so the reductions read them without copies
  // (mla_route.hip is built with the MFMA VGPR-accumulator form).
#pragma unroll
  for (int c = 0; c < 2; ++c) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+a"(bq[c][ks]));
  }
  asm volatile("" ::: "memory");

  // The wavefront's loads of a step: tile loads m = wv + 4 j while
  // m < KS (load m: chunk planes 2 m and 2 m + 1), and for its last
  // issue, when no tile load is left, the step's weights.  Branch-free:
  // every issue is one 16-byte direct load whose addresses are selected.
  constexpr int kPer = RS::kLoadsPerWave;
  const u32x4* w16 = reinterpret_cast<const u32x4*>(winv);
  auto issue_step = [&](uint32_t s) {
    const int slot = static_cast<int>(s % RS::kRing);
    const uint32_t t = min(t_begin + s, t_end - 1);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int m = wv + kRingWaves * j;
      const bool tile_load = m < RS::kTileLoads;
      const u32x4* src_t = tiles + static_cast<uint64_t>(2 * m + half) * cap +
                           static_cast<uint64_t>(t) * 32 + col;
      const u32x4* src_w = w16 + static_cast<uint64_t>(t) * 8 + (lane & 7);
      u32x4* dst_t = s_ring + slot * RS::kTileU4 + m * 64;
      u32x4* dst_w = reinterpret_cast<u32x4*>(s_w + slot * RS::kWeightArea);
      __builtin_amdgcn_global_load_lds(tile_load ? src_t : src_w,
                                       (__attribute__((address_space(3))) void*)(tile_load ? dst_t : dst_w),
                                       16, 0, 0);
    }
  };
  // Wait for tile s, pass the barrier, refill the slot of tile s - 1.
  auto enter_step = [&](uint32_t s) {
    asm volatile("" ::: "memory");
    wait_vmcnt_lds<(RS::kRing - 2) * kPer>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue_step(s + RS::kRing - 1);
  };

  // per column tile: the three largest coded u as signed-integer bits
  int b1[2], b2[2], b3[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) b1[c] = b2[c] = b3[c] = INT32_MIN;
  const uint32_t keep_mask = ~((1u << ibits) - 1u);

  // One tile's screen results: accumulators, the weights of the lane's
  // result rows 8 (r / 4) + 4 half + r % 4, and the tile.
  struct Res {
    f32x16 acc[2];
    float w[16];
    uint32_t t;
    uint32_t tcode;
  };
  uint32_t base = 0;  // first step of the run in progress
  // Reduction of value v = 16 c + r of a finished tile.
  auto reduce_one = [&](const Res& R, int v) {
    const int c = v >> 4;
    const int r = v & 15;
    const uint32_t code = R.tcode | static_cast<uint32_t>(r);
    if constexpr (kProbe) {
      const uint32_t slot_id = R.t * 32u + 8u * (r / 4) + 4u * half + (r % 4);
      const uint32_t q = 64u * wv + 32u * c + col;
      planes[static_cast<size_t>(q) * cap + slot_id] =
          and_or_b32(__float_as_uint(R.acc[c][r] * R.w[r]), keep_mask, code);
    } else {
      const int u = static_cast<int>(and_or_b32(__float_as_uint(R.acc[c][r] * R.w[r]),
                                                keep_mask, code));
      med3_i32_into(b2[c], b3[c], u);
      med3_i32_into(b1[c], b2[c], u);
      b1[c] = max(b1[c], u);
    }
  };
  // Tile s into R: its reads and MFMAs, with the 32 reductions of the
  // previous tile P (when there is one) spread over its MFMAs, each MFMA
  // and its share fenced (sched_barrier) so that the share runs on the
  // VALU while its MFMA executes.  The weights are read as integers: the compiler then
  // does not order them after the ring's pending loads.
  auto step_tile = [&](uint32_t s, Res& R, const Res& P, auto has_prev) {
    const int slot = static_cast<int>(s % RS::kRing);
    const u32x4* tile = s_ring + slot * RS::kTileU4;
    const uint32_t* wt = reinterpret_cast<const uint32_t*>(s_w + slot * RS::kWeightArea);
    u32x4 af[kPre];
#pragma unroll
    for (int j = 0; j < kPre; ++j) af[j] = tile[(2 * j + half) * 32 + col];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x4 w4 = *reinterpret_cast<const u32x4*>(wt + 8 * i + 4 * half);
      R.w[4 * i] = __uint_as_float(w4.x);
      R.w[4 * i + 1] = __uint_as_float(w4.y);
      R.w[4 * i + 2] = __uint_as_float(w4.z);
      R.w[4 * i + 3] = __uint_as_float(w4.w);
    }
    R.t = t_begin + s;
    R.tcode = (s - base) << 4;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 a = af[ks % kPre];
      if (ks + kPre < KS) af[ks % kPre] = tile[(2 * (ks + kPre) + half) * 32 + col];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        R.acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, bq[c][ks]),
            ks == 0 ? f32x16{} : R.acc[c], 0, 0, 0);
        // the 32 reductions spread over the tile's 2 KS MFMAs (one each,
        // about 6 VALU issues, at KS = 16 or 18; two at KS = 8): they
        // issue while the MFMA runs, before the next MFMA (issue is in order)
        if constexpr (decltype(has_prev)::value) {
          constexpr int kM = 2 * KS;
          const int m = 2 * ks + c;
#pragma unroll
          for (int v = m * 32 / kM; v < (m + 1) * 32 / kM; ++v) reduce_one(P, v);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  auto reduce_tile = [&](const Res& R) {
#pragma unroll
    for (int v = 0; v < 32; ++v) reduce_one(R, v);
  };

  // Lists of the finished runs, the latest last.
  int done[kRingSegs - 1][2][3];
#pragma unroll
  for (int g = 0; g < kRingSegs - 1; ++g) {
#pragma unroll
    for (int c = 0; c < 2; ++c) done[g][c][0] = done[g][c][1] = done[g][c][2] = INT32_MIN;
  }
  auto next_run = [&]() {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int g = 0; g + 1 < kRingSegs - 1; ++g) {
#pragma unroll
        for (int x = 0; x < 3; ++x) done[g][c][x] = done[g + 1][c][x];
      }
      done[kRingSegs - 2][c][0] = b1[c];
      done[kRingSegs - 2][c][1] = b2[c];
      done[kRingSegs - 2][c][2] = b3[c];
      b1[c] = b2[c] = b3[c] = INT32_MIN;
    }
  };
  // first step of run g
  auto run_start = [&](uint32_t g) -> uint32_t {
    return static_cast<uint32_t>(static_cast<uint64_t>(blockIdx.x * kRingSegs + g) * n_tiles32 /
                                 (static_cast<uint64_t>(W) * kRingSegs)) - t_begin;
  };
  uint32_t run = 0, next = run_start(1);  // next: first step of run + 1
  // Step s, whose reductions are those of tile s - 1: a run that starts at
  // step s (or empty runs before it) takes over once they are in.
  auto step = [&](uint32_t s, Res& R, const Res& P, auto has_prev) {
    const bool turn = run + 1 < kRingSegs && s == next;
    if (turn) base = s;
    enter_step(s);
    step_tile(s, R, P, has_prev);
    if (turn) {
      do {
        next_run();
        ++run;
        next = run_start(run + 1);
      } while (run + 1 < kRingSegs && s == next);
    }
  };
  Res RA, RB;
  if (steps > 0) {
#pragma unroll
    for (int s = 0; s < RS::kRing - 1; ++s) issue_step(static_cast<uint32_t>(s));
    step(0, RA, RB, std::false_type{});
  }
  uint32_t s = 1;
  for (; s + 1 < steps; s += 2) {
    step(s, RB, RA, std::true_type{});
    step(s + 1, RA, RB, std::true_type{});
  }
  if (s < steps) {
    step(s, RB, RA, std::true_type{});
    reduce_tile(RB);
  } else if (steps > 0) {
    reduce_tile(RA);
  }
  // runs past the block's last tile are empty
  for (; run + 1 < kRingSegs; ++run) next_run();
  // no load may still be writing LDS when the block ends
  asm volatile("" ::: "memory");
  wait_vmcnt_lds<0>();
  if constexpr (kProbe) return;
  // a lane's lists: one 16-byte store per (plane, query)
  const size_t n_sub = static_cast<size_t>(W) * 2 * kRingSegs;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const size_t q = static_cast<size_t>(64 * wv + 32 * c + col);
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      u32x4 v;
#pragma unroll
      for (int g = 0; g < kRingSegs - 1; ++g) v[g] = static_cast<uint32_t>(done[g][c][x]);
      v[kRingSegs - 1] = static_cast<uint32_t>(x == 0 ? b1[c] : (x == 1 ? b2[c] : b3[c]));
      *reinterpret_cast<u32x4*>(planes + (x * QP + q) * n_sub + (2 * blockIdx.x + half) * kRingSegs) = v;
    }
  }
}
static_assert(kRingSegs == 4, "a lane's lists of one kind are one 16-byte store");

// Query rows of one ring pass: qpad[j][0, stride) = query j's
// values rounded to bf16 (nearest even; bf16 queries are copied), zero past
// dim; inv_qn[j] = 1 / ||q_j|| rounded to fp32.  Rows j >= qc are zero with
// inv_qn NaN (nothing is kept for them).  grid = QP blocks.
static __global__ __launch_bounds__(kWave) void mla_batch_qprep_kernel(
    const void* __restrict__ query, int q_dtype, int qc, uint32_t dim, int stride,
    uint16_t* __restrict__ qpad, float* __restrict__ inv_qn, RouteStamps stamps, unsigned seq) {
  route_start_stamp(stamps, seq);
  const int j = blockIdx.x;
  const int lane = threadIdx.x;
  double ss = 0.0;
  for (int d = lane; d < stride; d += kWave) {
    uint16_t bits = 0;
    if (j < qc && static_cast<uint32_t>(d) < dim) {
      const size_t idx = static_cast<size_t>(j) * dim + d;
      float f;
      if (q_dtype == kBF16) {
        bits = static_cast<const uint16_t*>(query)[idx];
        f = bf16_to_f32(bits);
      } else {
        f = static_cast<const float*>(query)[idx];
        bits = static_cast<uint16_t>(bf16_bits_rne(f));
      }
      ss = fma(static_cast<double>(f), static_cast<double>(f), ss);
    }
    qpad[static_cast<size_t>(j) * stride + d] = bits;
  }
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) ss += __shfl_xor(ss, off);
  if (lane == 0) inv_qn[j] = j < qc ? static_cast<float>(1.0 / sqrt(ss)) : __builtin_nanf("");
}

// Descending bitonic sort of one value per lane across the wavefront
// (values must not be NaN).
__device__ inline float wave_sort_desc(float v) {
  const int lane = __lane_id();
#pragma unroll
  for (int size = 2; size <= kWave; size <<= 1) {
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      const float o = __shfl_xor(v, stride);
      const bool desc = (lane & size) == 0;  // run direction; the last run (size 64) descends
      const bool low = (lane & stride) == 0;
      v = (low == desc) ? fmaxf(v, o) : fminf(v, o);
    }
  }
  return v;
}

// Merge, certificate and exact rescore; grid = one block of kMergeThreads
// per query of the pass.  planes: the screen's rows (n_sub sub-streams
// of the stream or ring screen, QP queries); query qi (pass column) has its `dim` values at
// query + qi*qstride elements (F32 or BF16) and 1/||q|| at inv_qn[qi].
// The screened score of a kept value u is s~ = u * inv_qn[qi], its slot
// the code in u's low ibits bits.  The screen bound for the query
// (|s~ - score|):
//   B0 = (gamma + delta) * (1 + 2^-20) + 8 * 2^-24
//        + 1.01e-8 / (qn * nmin) + m * sqrt(dim) * 2^-125 * (1/qn + 1/nmin)
//        + m * dim * 2^-125 / (qn * nmin),
//   B  = B0 + 2^(ibits-23) * (1 + B0) * (1 + 2^-20) + 2^(ibits-148) / qn,
// gamma bounding the fp32 accumulation, delta what the bf16 operands leave
// out (of a bf16 bank ||q - bf16(q)|| / ||q||, Cauchy-Schwarz, about a
// third of 2^-8 for an fp32 query and 0 for a bf16 one; of an fp32 bank, with
// x = xh + xl + ex and q = qh + ql + eq, |xl| <= 2^-9 |x| and
// |ex| <= 2^-18 |x| per value: ex q, x eq and xl ql, below 4 * 2^-18
// together), 8 * 2^-24 the reciprocals and products of the screened
// score and the score's own rounding, the 1e-8 term the law's
// denominator, the next terms bf16 values or products flushed near zero
// (m = 1, or 4 for the fp32 bank's two parts a value and three products);
// the last two the slot code written into u (relative to |u|, with
// |score| <= 1, and absolute near zero).  qn is the law's query norm and
// nmin the smallest positive row norm.
//
// Steps: the last wavefront stages the query while the others load the
// sub-streams' entries and each sort their lanes' largest kept s~; the
// largest k-th of those, L, is a lower bound on v_k, so every kept entry at
// or above t lies at or above L - 2B.  The positive ones of those (at most
// kSurvMax, else no certificate; fewer than k, and t is not positive) are
// collected in LDS, one thread each: it ranks its
// entry by (s~ desc, sub-stream asc) and counts the entries above s~ + 2B.
// Fewer than k such entries holds for every entry at or above t (those
// above it then lie above v_k), so the entries passing that count -- a
// prefix of the ranking -- form the law's dot products of their rows and
// are ranked by law score (score desc, node id asc).  Rescoring entries
// below t as well changes nothing: they are real nodes with law scores.
//
// The kernel is a chain of latencies (one block per query), so what can run
// side by side does: the prefix's rows come in by all threads at once, a
// chunk each, as doubles (a conversion costs more than its multiply-add),
// while the last wavefront sums the law's norm; then a lane per row runs
// the fp64 chain from LDS.  With the norm formed first and a lane loading
// its row itself, 36 chunks at a time, the kernel took 17.2 us for 32 queries
// x 100k x 280 fp32 and 25.6 for 256 x 1M x 288 bf16; it takes 14.1 and 20.5
// to 22.9.
// Writes out[qi*k ..) (host mapped): the law's top-k where certified, else
// k entries without a node (kNoId: route qi again on the exact path).  With
// `done` the entries carry the route's tag and done[qi] takes its number
// (store_entry, block_done_flag).
//
// Dynamic LDS: the query as doubles, zero past dim up to whole stages of
// kMergeStage values (merge_len), then merge_rows rows of as many, merge_pitch
// apart (an odd number of 16-byte pieces: lanes read distinct banks).
constexpr uint32_t kMergeStage = 16;

__host__ __device__ inline uint32_t merge_len(uint32_t dim) {
  return (dim + kMergeStage - 1) / kMergeStage * kMergeStage;
}
__host__ __device__ inline uint32_t merge_pitch(uint32_t dim) { return merge_len(dim) + 2; }
// Rows staged at once: what fits 64 KiB, at most a wavefront's lanes.
__host__ __device__ inline uint32_t merge_rows(uint32_t dim) {
  const uint32_t fit = 65536u / (8u * merge_pitch(dim));
  return fit < 1u ? 1u : (fit > 64u ? 64u : fit);
}
inline size_t merge_lds(uint32_t dim) {
  return (merge_len(dim) + static_cast<size_t>(merge_rows(dim)) * merge_pitch(dim)) * sizeof(double);
}

// sum over d of a[d] * b[d], d ascending from 0, one fma each: the serial
// chain, its values read from LDS a stage ahead.
__device__ inline double serial_dot(const double* __restrict__ a, const double* __restrict__ b,
                                    uint32_t len) {
  constexpr int N = kMergeStage / 2;
  double x[N], y[N], xn[N], yn[N];
#pragma unroll
  for (int e = 0; e < N; ++e) {
    x[e] = a[e];
    y[e] = b[e];
  }
  double dot = 0.0;
  for (uint32_t d = 0; d < len; d += 2 * N) {
    auto half = [&](double (&p)[N], double (&q)[N], double (&pn)[N], double (&qn)[N], uint32_t ahead) {
#pragma unroll
      for (int e = 0; e < N; ++e) {
        pn[e] = a[ahead + e];
        qn[e] = b[ahead + e];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < N; ++e) dot = fma(p[e], q[e], dot);
    };
    half(x, y, xn, yn, d + N);
    half(xn, yn, x, y, d + 2 * N < len ? d + 2 * N : 0);
  }
  return dot;
}

// One wavefront stages query qi (`dim` values, F32 or BF16, qstride elements
// apart) as doubles in s_q[0, len), zero past dim, and returns
// ||q - bf16(q)|| in every lane.
__device__ inline double stage_row_query(double* __restrict__ s_q, const void* __restrict__ query,
                                         int q_dtype, size_t qstride, int qi, uint32_t dim,
                                         uint32_t len, int lane) {
  const unsigned char* qbase = static_cast<const unsigned char*>(query) +
                               static_cast<size_t>(qi) * qstride * (q_dtype == kBF16 ? 2 : 4);
  constexpr int kAhead = 8;
  double rr = 0.0;
  for (uint32_t d0 = lane; d0 < len; d0 += kAhead * kWave) {
    float f[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const uint32_t d = min(d0 + j * kWave, dim - 1);
      f[j] = q_dtype == kBF16 ? bf16_to_f32(reinterpret_cast<const uint16_t*>(qbase)[d])
                              : reinterpret_cast<const float*>(qbase)[d];
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const uint32_t d = d0 + j * kWave;
      if (d < len) s_q[d] = d < dim ? static_cast<double>(f[j]) : 0.0;
      const double r = f[j] - bf16_to_f32(bf16_bits_rne(f[j]));  // exact
      if (d < dim) rr = fma(r, r, rr);
    }
  }
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) rr += __shfl_xor(rr, off);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  return sqrt(rr);
}

// What the screen bound of a pass rests on besides the norms.
struct ScreenBound {
  double gamma;  // fp32 accumulation
  double delta;  // operands' rounding to bf16; negative: that of the query alone
  double absm;   // m: the terms near zero
  uint32_t dim;
  int ibits;     // slot code width
};

// The screen bound B of a query (|s~ - score|, see mla_batch_merge_kernel)
// from the query's norm qn (or less), rest = ||q - bf16(q)|| and the
// smallest positive row norm nmin;
// it holds where screen_in_range(qn, nmax).
__device__ inline double batch_screen_bound(const ScreenBound& b, double qn, double rest, double nmin) {
  const double dim = static_cast<double>(b.dim);
  const double delta = b.delta < 0.0 ? rest / qn : b.delta;
  const double bound0 = (b.gamma + delta) * (1.0 + 0x1p-20) + 8.0 * 0x1p-24 + 1.01e-8 / (qn * nmin) +
                        b.absm * sqrt(dim) * 0x1p-125 * (1.0 / qn + 1.0 / nmin) +
                        b.absm * dim * 0x1p-125 / (qn * nmin);
  return bound0 + ldexp(1.0 + bound0, b.ibits - 23) * (1.0 + 0x1p-20) + ldexp(1.0, b.ibits - 148) / qn;
}
// No product or partial sum of the screen can reach the fp32 overflow
// threshold (Cauchy-Schwarz, with the operands' and the accumulation's
// rounding), and no value its rounding to bf16; nmax the largest row norm.
__device__ inline bool screen_in_range(double qn, double nmax) {
  return qn * nmax < 0x1p125 && qn < 0x1p126 && nmax < 0x1p126;
}

constexpr int kMergeThreads = 512;
constexpr int kMergeWavesB = kMergeThreads / kWave;
constexpr int kMergeLoaders = kMergeThreads - kWave;  // threads of the entry-loading wavefronts
constexpr int kMergePer = 8;       // sub-streams per loading thread: n_sub <= 3584
constexpr int kSurvMax = kMergeThreads;

template <int DT>
__global__ __launch_bounds__(kMergeThreads) void mla_batch_merge_kernel(
    const uint32_t* __restrict__ planes, uint32_t n_sub, bool ring, int QP, uint32_t n_tiles32,
    const float* __restrict__ inv_qn, const u32x4* __restrict__ tiles,
    const float* __restrict__ norms, const uint64_t* __restrict__ ids, uint64_t cap,
    uint32_t chunks, const void* __restrict__ query, int q_dtype, size_t qstride, ScreenBound sb,
    const unsigned* __restrict__ norm_range, int k, Cand* __restrict__ out,
    unsigned* __restrict__ done, unsigned seq, unsigned long long* __restrict__ end_tick,
    unsigned long long* __restrict__ screen_tick) {
  if (screen_tick && blockIdx.x == 0 && threadIdx.x == 0) *screen_tick = wall_clock64();
  constexpr uint32_t EPC = DT == kF32 ? 4 : 8;
  extern __shared__ double s_q[];           // the query, zero past dim; the staged rows
  double* s_rows = s_q + merge_len(sb.dim);
  __shared__ float s_lw[kMergeWavesB];      // per wavefront: k-th largest lane maximum
  __shared__ float s_nk[kMergeWavesB];      // per wavefront: largest dropped s~
  __shared__ __align__(16) float s_sv[kSurvMax];       // survivors: s~
  __shared__ float s_su[kSurvMax];                     //   u
  __shared__ __align__(16) uint32_t s_key[kSurvMax];   //   2 * sub-stream + (second kept entry)
  __shared__ float s_vrank[kMaxTopK];       // s~ of the k best survivors
  __shared__ uint32_t s_rslot[kSurvMax];    // slots of the prefix, by rank
  __shared__ float s_es[kSurvMax];          // law scores of the ranked prefix (NaN: not finite)
  __shared__ uint64_t s_eid[kSurvMax];
  __shared__ Cand s_top[kMaxTopK];
  __shared__ double s_qn, s_bound, s_qhi;
  __shared__ float s_ek;
  __shared__ unsigned s_count;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int qi = blockIdx.x;
  const size_t plane = static_cast<size_t>(QP) * n_sub;
  const size_t row = static_cast<size_t>(qi) * n_sub;
  const float* p_u1 = reinterpret_cast<const float*>(planes) + row;
  const float* p_u2 = p_u1 + plane;
  const float* p_nk = p_u2 + plane;
  const float iq = inv_qn[qi];
  const int ibits = sb.ibits;
  // slot of coded value u kept by sub-stream i (see the screens' slot codes)
  const uint32_t tbits = ring ? ibits - 4 : ibits - 5;
  const uint32_t runs = ring ? n_sub / 2 : n_sub;
  auto slot_of = [&](float u, uint32_t i) -> uint32_t {
    const uint32_t c = __float_as_uint(u);
    const uint32_t run = ring ? i / (2 * kRingSegs) * kRingSegs + i % kRingSegs : i;
    const uint32_t half = ring ? i / kRingSegs % 2 : (c >> (ibits - 1)) & 1u;
    const uint32_t t_begin = static_cast<uint32_t>(static_cast<uint64_t>(run) * n_tiles32 / runs);
    const uint32_t r = c & 15u;
    const uint32_t t = t_begin + ((c >> 4) & ((1u << tbits) - 1u));
    const uint32_t slot = t * 32u + 8u * (r >> 2) + 4u * half + (r & 3u);
    // every code the screen writes names a slot of a tile it walked; the
    // clamp only keeps a corrupted value from reading past the bank
    return slot < cap ? slot : static_cast<uint32_t>(cap - 1);
  };

  float u1[kMergePer], u2[kMergePer];
  float nk = -INFINITY;
#pragma unroll
  for (int j = 0; j < kMergePer; ++j) {
    const uint32_t i = static_cast<uint32_t>(j * kMergeLoaders + tid);
    u1[j] = u2[j] = -INFINITY;
    if (tid < kMergeLoaders && i < n_sub) {
      u1[j] = p_u1[i];
      u2[j] = p_u2[i];
      nk = fmaxf(nk, p_nk[i] * iq);
    }
  }
  if (wave == kMergeWavesB - 1) {
    const double rest = stage_row_query(s_q, query, q_dtype, qstride, qi, sb.dim, merge_len(sb.dim), lane);
    if (lane == 0) {
      // 1/iq is the query's norm to within 2^-23
      const double qa = 1.0 / static_cast<double>(iq);
      s_qhi = qa * (1.0 + 0x1p-20);
      s_bound = batch_screen_bound(sb, qa * (1.0 - 0x1p-20), rest,
                                   static_cast<double>(__uint_as_float(norm_range[0])));
    }
  }
  if (tid == 0) s_count = 0u;
  bool over = false;
  if (wave != kMergeWavesB - 1) {
    // largest finite kept s~ of the thread; a +inf s~ voids the certificate,
    // and so does a NaN u that lies above every number (see the screen): it
    // may have pushed real entries out of its sub-stream
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < kMergePer; ++j) {
      const float v1 = u1[j] * iq, v2 = u2[j] * iq;
      if (isfinite(v1)) m = fmaxf(m, v1);
      if (isfinite(v2)) m = fmaxf(m, v2);
      over = over || v1 == INFINITY || v2 == INFINITY || __float_as_int(u1[j]) >= 0x7f800000;
    }
    const float ms = wave_sort_desc(m);
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) nk = fmaxf(nk, __shfl_xor(nk, off));
    if (lane == k - 1) s_lw[wave] = ms;
    if (lane == 0) s_nk[wave] = nk;
  }
  const int any_over = __syncthreads_or(over ? 1 : 0);

  const double nmax = static_cast<double>(__uint_as_float(norm_range[1]));
  const double bound = s_bound;
  float L = -INFINITY, nk_all = -INFINITY;
#pragma unroll
  for (int w = 0; w < kMergeWavesB - 1; ++w) {
    L = fmaxf(L, s_lw[w]);
    nk_all = fmaxf(nk_all, s_nk[w]);
  }
  const double floor_s = static_cast<double>(L) - 2.0 * bound - 0x1p-40;
  auto offer = [&](float u, uint32_t key) {
    // an entry at or above t is positive; zeros (a list without a tile holds
    // -0) would only fill the survivors' places
    const float v = u * iq;
    if (v > 0.0f && isfinite(v) && static_cast<double>(v) >= floor_s) {
      const unsigned at = atomicAdd(&s_count, 1u);
      if (at < static_cast<unsigned>(kSurvMax)) {
        s_sv[at] = v;
        s_su[at] = u;
        s_key[at] = key;
      }
    }
  };
#pragma unroll
  for (int j = 0; j < kMergePer; ++j) {
    const uint32_t i = static_cast<uint32_t>(j * kMergeLoaders + tid);
    offer(u1[j], 2u * i);
    offer(u2[j], 2u * i + 1u);
  }
  __syncthreads();
  const unsigned count = s_count;
  const int n = static_cast<int>(count < static_cast<unsigned>(kSurvMax) ? count : kSurvMax);
  int my_rank = 0;
  bool sup = false;
  if (tid < n) {
    const float sv = s_sv[tid];
    const uint32_t key = s_key[tid];
    // s~ + 2B rounded up: entries that round into it count as below
    const double h = static_cast<double>(sv) + 2.0 * bound + 0x1p-40;
    const float hi = static_cast<float>(h + fabs(h) * 0x1p-22 + 0x1p-140);
    int above = 0;
    int i = 0;
    for (; i + 4 <= n; i += 4) {
      const float4 o = *reinterpret_cast<const float4*>(&s_sv[i]);
      const uint4 kk = *reinterpret_cast<const uint4*>(&s_key[i]);
      my_rank += (o.x > sv || (o.x == sv && kk.x < key)) ? 1 : 0;
      my_rank += (o.y > sv || (o.y == sv && kk.y < key)) ? 1 : 0;
      my_rank += (o.z > sv || (o.z == sv && kk.z < key)) ? 1 : 0;
      my_rank += (o.w > sv || (o.w == sv && kk.w < key)) ? 1 : 0;
      above += (o.x > hi) + (o.y > hi) + (o.z > hi) + (o.w > hi);
    }
    for (; i < n; ++i) {
      const float o = s_sv[i];
      my_rank += (o > sv || (o == sv && s_key[i] < key)) ? 1 : 0;
      above += o > hi ? 1 : 0;
    }
    if (my_rank < k) s_vrank[my_rank] = sv;
    sup = above < k;
    if (sup) s_rslot[my_rank] = slot_of(s_su[tid], key >> 1);
  }
  const int n_el = __syncthreads_count(sup ? 1 : 0);
  // the prefix's rows, merge_rows at a time; the row's thread (thread = rank
  // within the round) keeps its dot product.  Rows are staged by chunk, zero
  // past dim as they are stored, and on to whole stages.
  const uint32_t rows = merge_rows(sb.dim);
  const uint32_t len = merge_len(sb.dim), pitch = merge_pitch(sb.dim);
  double dot = 0.0;
  float nf = 0.0f;
  uint64_t eid = kNoId;
  for (uint32_t r0 = 0; r0 == 0 || r0 < static_cast<uint32_t>(n_el); r0 += rows) {
    const uint32_t r1 = min(r0 + rows, static_cast<uint32_t>(n_el));
    if (r0 > 0) __syncthreads();  // the rows before are done with
    if (wave == kMergeWavesB - 1) {
      if (r0 == 0 && lane == 0) s_qn = sqrt(serial_dot(s_q, s_q, len));
    } else {
      for (uint32_t r = r0 + wave; r < r1; r += kMergeWavesB - 1) {
        const uint32_t slot = s_rslot[r];
        for (uint32_t c = lane; c * EPC < len; c += kWave) {
          u32x4 v = {0u, 0u, 0u, 0u};
          if (c < chunks) v = tiles[static_cast<size_t>(c) * cap + slot];
#pragma unroll
          for (int e = 0; e < static_cast<int>(EPC); ++e) {
            s_rows[(r - r0) * pitch + c * EPC + e] = chunk_value<DT>(v, e);
          }
        }
      }
    }
    const uint32_t r = tid;
    const bool mine = r >= r0 && r < r1;
    if (mine) {
      nf = norms[s_rslot[r]];
      eid = ids[s_rslot[r]];
    }
    __syncthreads();
    if (mine) dot = serial_dot(s_rows + (r - r0) * pitch, s_q, len);
  }
  const double qn = s_qn;
  const float vk = n >= k ? s_vrank[k - 1] : -INFINITY;
  const double t = static_cast<double>(vk) - 2.0 * bound - 0x1p-40;
  // t > 0: the screen kept its values by their integer bits, the float
  // order only from +0 up.
  const bool pre = any_over == 0 && count <= static_cast<unsigned>(kSurvMax) && n >= k &&
                   static_cast<double>(nk_all) < t && t > 0.0 && screen_in_range(s_qhi, nmax);
  // the rescored prefix: ranks [0, n_el)
  if (tid < n_el) {
    const float sc = static_cast<float>(dot / (qn * static_cast<double>(nf) + 1e-8));
    const bool fin = isfinite(sc);
    s_es[tid] = fin ? sc : __builtin_nanf("");
    s_eid[tid] = fin ? eid : kNoId;
  }
  __syncthreads();
  // rank the prefix by (law score desc, node id asc)
  const bool fin = pre && tid < n_el && isfinite(s_es[tid]);
  if (fin) {
    const float es = s_es[tid];
    const uint64_t id = s_eid[tid];
    int rank = 0;
    for (int i = 0; i < n_el; ++i) rank += better(s_es[i], s_eid[i], es, id) ? 1 : 0;
    if (rank < k) {
      Cand c;
      c.score = es;
      c.slot = kNoSlot;
      c.id = id;
      s_top[rank] = c;
    }
    if (rank == k - 1) s_ek = es;
  }
  const int n_fin = __syncthreads_count(fin ? 1 : 0);
  if (tid < k) {
    // every node outside the prefix scores below v_k - B
    const bool ok = pre && n_fin >= k &&
                    static_cast<double>(s_ek) >= static_cast<double>(vk) - bound;
    Cand c;
    c.score = __builtin_nanf("");
    c.slot = kNoSlot;
    c.id = kNoId;
    if (ok) c = s_top[tid];
    store_entry(out + static_cast<size_t>(qi) * k + tid, c, done ? route_tag(seq) : kNoSlot);
  }
  block_done_flag(done, seq, end_tick);
}

// Tests of the screen bound: the screened scores s~ = u * (1/||q||) of a
// probe screen (planes[q*cap + slot], coded u bits) for slots [0, n),
// out_values[qi*n + slot], and the query's bound B, out_bounds[qi] (+inf
// where it is not established, screen_in_range).  grid = queries
// of the pass, one wavefront each.
static __global__ __launch_bounds__(kWave) void mla_batch_probe_finish_kernel(
    const uint32_t* __restrict__ planes, uint64_t cap, uint32_t n, const float* __restrict__ inv_qn,
    const void* __restrict__ query, int q_dtype, size_t qstride, uint32_t len, ScreenBound sb,
    const unsigned* __restrict__ norm_range, float* __restrict__ out_values,
    double* __restrict__ out_bounds) {
  extern __shared__ double s_q[];  // len values
  const int qi = blockIdx.x;
  const int lane = threadIdx.x;
  const double rest = stage_row_query(s_q, query, q_dtype, qstride, qi, sb.dim, len, lane);
  if (lane == 0) {
    const double qn = staged_norm(s_q, len);
    const double nmin = static_cast<double>(__uint_as_float(norm_range[0]));
    const double nmax = static_cast<double>(__uint_as_float(norm_range[1]));
    out_bounds[qi] = screen_in_range(qn, nmax) ? batch_screen_bound(sb, qn, rest, nmin)
                                               : static_cast<double>(INFINITY);
  }
  const float iq = inv_qn[qi];
  for (uint32_t s = lane; s < n; s += kWave) {
    out_values[static_cast<size_t>(qi) * n + s] =
        __uint_as_float(planes[static_cast<size_t>(qi) * cap + s]) * iq;
  }
}

}  // namespace mla
}  // namespace grm
