// mla_screen.hpp -- launches of the batched route's screens.
//
// launch_screen<true> (the screens' probe forms, which only tests of the
// screen bound reach) is instantiated in mla_screen_probe.hip alone: its
// kernels are a third of the MLA code, and a code object of their own is
// not loaded with the first bank of a process (first bank 20.5 -> 19.4 ms).
#pragma once

#include "mla_batch.hpp"

#include <algorithm>

namespace grm {
namespace mla {

// Batched-route plan.
struct BatchPlan {
  int ks = 0;          // K-steps of 16 dims that cover a row
  int p = 0;           // K-steps in flight per wavefront of the stream screen
  int nb = 0;          // batches of p steps: nb * p >= ks
  int qp_max = 0;      // queries per pass (32, 64, 128, or 256 on the ring)
  int qp_stream = 0;   // queries per stream-screen pass
  uint32_t subs = 0;   // sub-streams of a stream-screen pass
  int ibits = 0;       // width of the slot code the stream screen writes into its values
  bool ring = false;   // full passes of a bf16 bank run mla_batch_ring_kernel
  int ks_ring = 0;     // its K-steps (8, 16 or 18)
  int ibits_ring = 0;  // its slot code width
};

// LDS of a stream-screen pass of qp queries (of an fp32 bank their bf16
// parts and remainders).
inline size_t stream_screen_lds(int dtype, const BatchPlan& p, int qp) {
  return static_cast<size_t>(qp) * (16 * p.nb * p.p + 8) * (dtype == kF32 ? 4 : 2);
}

// Columns, sub-streams and slot code width of one pass.
struct PassShape {
  bool ring;
  int qp;          // columns
  uint32_t subs;   // sub-streams
  int ibits;
};

// A pass's queries (device) and what its kernels report on the way.
struct PassQueries {
  const void* q;
  int dtype;
  int count;
};
struct PassMarks {
  RouteStamps start{nullptr, nullptr};         // the route's first timed kernel
  unsigned long long* screen_tick = nullptr;   // [screen start, merge start]
  hipEvent_t* ev = nullptr;                    // events around the screen kernel
};

// One pass's screen: the bank, the pass's buffers and what it reports.
struct ScreenLaunch {
  int dtype;
  uint32_t cus;
  hipStream_t stream;
  const u32x4* tiles;
  const float* norms;
  const float* winv;  // slot weights (ring)
  uint64_t cap;
  uint32_t chunks;
  uint32_t n_tiles32;
  uint32_t dim;
  uint16_t* qpad;     // padded queries (ring)
  float* inv_qn;
  BatchPlan p;
  PassShape s;
  PassQueries q;
  uint32_t* planes;
  PassMarks m;
  unsigned seq;
};

template <int KS, bool kProbe>
int launch_ring(const ScreenLaunch& l) {
  using RS = RingShape<KS>;
  auto kern = mla_batch_ring_kernel<KS, kProbe>;
  GRM_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>(RS::kLds)));
  kern<<<l.cus, kRingWaves * kWave, RS::kLds, l.stream>>>(l.tiles, l.winv, l.cap, l.n_tiles32, l.qpad,
                                                          l.s.ibits, l.planes, l.m.screen_tick);
  GRM_HIP_CHECK(hipGetLastError());
  return 0;
}

template <int DT, int P, int CT, bool kProbe>
int launch_stream_form(const ScreenLaunch& l) {
  auto kern = mla_batch_stream_kernel<DT, P, CT, kProbe>;
  const size_t lds = stream_screen_lds(l.dtype, l.p, 32 * CT);
  if (lds > 65536) {
    GRM_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(lds)));
  }
  kern<<<l.cus, kBatchWaves * kWave, lds, l.stream>>>(
      l.tiles, l.norms, l.cap, l.chunks, l.n_tiles32, l.p.subs, static_cast<uint32_t>(l.p.nb),
      static_cast<uint32_t>(l.p.ks), l.q.q, l.q.dtype, l.q.count, l.dim, l.inv_qn, l.s.ibits, l.planes,
      l.m.start, l.seq, l.m.screen_tick);
  GRM_HIP_CHECK(hipGetLastError());
  return 0;
}

template <int DT, int P, bool kProbe>
int launch_stream(const ScreenLaunch& l) {
  if (l.s.qp == 32) return launch_stream_form<DT, P, 1, kProbe>(l);
  if (l.s.qp == 64) return launch_stream_form<DT, P, 2, kProbe>(l);
  return launch_stream_form<DT, P, 4, kProbe>(l);
}

// The screen of one pass, its queries prepared first where the screen does
// not do so itself.
template <bool kProbe>
int launch_screen(const ScreenLaunch& l) {
  if (l.s.ring) {
    mla_batch_qprep_kernel<<<l.s.qp, kWave, 0, l.stream>>>(
        l.q.q, l.q.dtype, l.q.count, l.dim, 16 * l.p.ks_ring + 8, l.qpad, l.inv_qn, l.m.start, l.seq);
    GRM_HIP_CHECK(hipGetLastError());
  }
  if (l.m.ev) GRM_HIP_CHECK(hipEventRecord(l.m.ev[0], l.stream));
  int rc = 0;
  if (l.s.ring) {
    switch (l.p.ks_ring) {
      case 8: rc = launch_ring<8, kProbe>(l); break;
      case 16: rc = launch_ring<16, kProbe>(l); break;
      default: rc = launch_ring<18, kProbe>(l); break;
    }
  } else if (l.dtype == kF32) {
    switch (l.p.p) {
      case 9: rc = launch_stream<kF32, 9, kProbe>(l); break;
      case 8: rc = launch_stream<kF32, 8, kProbe>(l); break;
      case 6: rc = launch_stream<kF32, 6, kProbe>(l); break;
      default: rc = launch_stream<kF32, 4, kProbe>(l); break;
    }
  } else {
    switch (l.p.p) {
      case 18: rc = launch_stream<kBF16, 18, kProbe>(l); break;
      case 16: rc = launch_stream<kBF16, 16, kProbe>(l); break;
      case 12: rc = launch_stream<kBF16, 12, kProbe>(l); break;
      case 8: rc = launch_stream<kBF16, 8, kProbe>(l); break;
      default: rc = launch_stream<kBF16, 4, kProbe>(l); break;
    }
  }
  GRM_CHECK_RC(rc);
  if (l.m.ev) GRM_HIP_CHECK(hipEventRecord(l.m.ev[1], l.stream));
  return 0;
}

// launch_screen<true>, in mla_screen_probe.hip.
int launch_probe_screen(const ScreenLaunch& l);

}  // namespace mla
}  // namespace grm
