// Kernel instantiations for one element type and one kernel family.
// Compiled once per (SA_DTYPE_ID, SA_KIND) pair so that the families build in parallel.
//   SA_DTYPE_ID: 0 fp32, 1 fp16, 2 bf16        SA_KIND: 0 forward, 1 delta + dQ, 2 dK/dV, 3 one-launch backward
//   SA_DGROUP: 0 head dims 16..128, 1 head dim 256
#include <algorithm>
#include <mutex>
#include "sa_launch.h"
#include "sa_f32.h"
#if SA_KIND == 0
#include "sa_fwd.h"
#ifndef SA_NO_ASM_KERNELS
#include "sa_fwd3.h"
#endif
#else
#include "sa_bwd.h"
#ifndef SA_NO_ASM_KERNELS
#include "sa_bwd3.h"
#include "sa_bwd4.h"
#endif
#include "sa_bwd_split.h"
#include "sa_bwd_fused.h"
#endif

namespace sa {

#if SA_DTYPE_ID == 0
using ElemT = float;
#elif SA_DTYPE_ID == 1
using ElemT = _Float16;
#elif SA_DTYPE_ID == 2
using ElemT = __bf16;
#else
#error "SA_DTYPE_ID must be 0, 1 or 2"
#endif

// Kernels whose dynamic LDS exceeds the 64 KiB default need the limit raised once per kernel
// and per device (the attribute belongs to the device that is current when it is set).  The
// outcome of that one call is kept and handed to every caller on that device.
struct PrepareState {
  static constexpr int kMaxDevices = 64;
  std::mutex mu;
  bool done[kMaxDevices] = {};
  int rc[kMaxDevices] = {};
};
template <typename K> static int prepare(K kernel, size_t lds_bytes, PrepareState& state) {
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= PrepareState::kMaxDevices) {
    return (int)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
  }
  std::lock_guard<std::mutex> lock(state.mu);
  if (!state.done[dev]) {
    state.rc[dev] = (int)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    state.done[dev] = true;
  }
  return state.rc[dev];
}

static int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// LDS of a float32 kernel on the 16-bit matrix pipe: its split tiles, or the float32 tiles of the rows it goes through again.
// (or the own rows of its waves, `own` sets of them, or their row patches: whichever is most)
template <int D, int NW> constexpr size_t split_lds(size_t split_bytes, size_t rows_bytes, int own) {
  return std::max({split_bytes, rows_bytes, direct_rows(D, NW) ? 0 : (size_t)own * NW * OwnRows32<D>::ELEMS * sizeof(float),
                   64 + (size_t)NW * RowPatch32<D>::ELEMS * sizeof(float)});
}
template <int D> constexpr size_t float_tiles = (size_t)2 * 2 * 32 * TileGeom<float, D>::PITCH * sizeof(float);   // two stages

// float32, head dimensions 16 to 64: workgroups of 64 rows (two waves) instead of 128 where twice as many still find a CU
// each and their windows are at least a tenth shorter -- such a launch takes as long as one workgroup, and that as long as
// its tiles.  Forward and backward in us, 128 rows -> 64, at D=16; 32; 64.  Chunks of 64, 2 back, B*H=8, T=512 11.2, 27.7 ->
// 9.3, 22.2; 12.6, 33.0 -> 10.3, 25.9; 17.4, 47.5 -> 15.1, 39.3, and with 128 workgroups (B*H=32) 11.3, 28.0 -> 9.5, 22.8; 12.8,
// 33.7 -> 10.5, 26.7; 17.7, 48.8 -> 15.5, 41.0; chunks of 10, 9 back, 128 workgroups 12.6, 29.0 -> 10.7, 25.6; 15.1, 35.9 -> 12.5,
// 30.1; 20.4, 51.3 -> 18.1, 45.7.  On the other side of the rule: the same window (chunks of 128, 1 back, B*H=8, T=1024) 11.6, 28.7 ->
// 11.4, 27.9; 12.9, 34.1 -> 12.6, 32.1; 17.4, 48.1 -> 18.9, 49.2 (half the threads stage a tile); 192 workgroups (B*H=48, T=512)
// 11.5, 28.3 -> 11.9, 30.5; 13.0, 34.0 -> 13.7, 37.8; 17.9, 49.3 -> 20.6, 50.3.
template <typename P> static bool half_workgroups(const P& p) {
  if ((int64_t)p.B * p.H * ceil_div(p.T, 128) > 128) return false;
  const int64_t back = std::min((int64_t)p.C * p.R, (int64_t)1 << 32);   // ten times it stays within 64 bits
  return 10 * (back + ceil_div(64, p.C) * p.C) <= 9 * (back + ceil_div(128, p.C) * p.C);
}

// TileOrder of the float32 kernels, with the period of the largest workgroup that a kernel has at this head dimension, whatever
// the grid picks: no window holds two multiples of it, so the windows of a smaller workgroup start at the same tile or have none of
// them, and every row goes through its tiles in the same order.  At head dimension 16 the order gained nothing.
template <int D, typename P> static void tile_order_f32(P& p, int largest) {
  if (D > 16) set_tile_order(p, largest, 32);
}

// SA_DGROUP 0 holds head dimensions 16..128, SA_DGROUP 1 holds 256 (built with different
// compiler options, see the Makefile).
#if SA_DGROUP == 0
#define SA_FOR_EACH_D(X) \
  switch (D) {           \
    case 16: X(16);      \
    case 32: X(32);      \
    case 64: X(64);      \
    case 128: X(128);    \
    default: return SA_ERR_HEAD_DIM; \
  }
#else
#define SA_FOR_EACH_D(X) \
  switch (D) {           \
    case 256: X(256);    \
    default: return SA_ERR_HEAD_DIM; \
  }
#endif

#if SA_KIND == 0
template <int D, int NW, int TK, bool SHORT> static int fwd2_launch(FwdParams p, hipStream_t st) {
  using C = Cfg<ElemT>;
  constexpr int TQ = NW * C::FWD2_QB * 32;
  // tile stages; the epilogue's row patches (one per wave) reuse the same memory
  constexpr size_t stages = (D == 256 ? (size_t)Fwd2Slots::ROWS : (size_t)RING * 2 * TK) * D * sizeof(ElemT);
  constexpr size_t patches = (size_t)NW * RowPatch<ElemT, D>::ELEMS * sizeof(ElemT);
  constexpr size_t lds = stages > patches ? stages : patches;
  auto kern = fwd2_kernel<ElemT, D, C::FWD2_QB, NW, TK, SHORT>;
  static PrepareState once;
  if (int rc = prepare(kern, lds, once)) return rc;
  const int64_t blocks = set_tiles(p, TQ, SHORT ? SHORT_LAST : PLAIN);
  if (TK != 32) set_length_order(p, 768);
  set_tile_order(p, TQ, TK);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), lds, st, p);
  return (int)hipGetLastError();
}
// hand-scheduled loop, one wave per SIMD, 64 queries per wave (head dimension 128)
template <int D> static int fwd3_launch(FwdParams p, hipStream_t st) {
#ifdef SA_NO_ASM_KERNELS
  (void)p; (void)st;
  return SA_ERR_HEAD_DIM;
#else
  using C = Cfg<ElemT>;
  if constexpr (C::fwd2(D) && D == 128) {
    constexpr int NW = 4, TQ = NW * 64, NST = 4;
    constexpr size_t stages = (size_t)NST * 2 * 64 * D * sizeof(ElemT);
    constexpr size_t patches = (size_t)NW * RowPatch<ElemT, D>::ELEMS * sizeof(ElemT);
    constexpr size_t lds = stages > patches ? stages : patches;
    auto kern = fwd3_kernel<ElemT, D, NST>;
    static PrepareState once;
    if (int rc = prepare(kern, lds, once)) return rc;
    const int64_t blocks = set_tiles(p, TQ, PLAIN);
    if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), lds, st, p);
    return (int)hipGetLastError();
  } else {
    return SA_ERR_HEAD_DIM;
  }
#endif
}
template <int D, int NW, int NST, bool BY_LENGTH> static int fwd_split_run(const FwdParams& p, int64_t blocks, hipStream_t st) {
  constexpr size_t lds = split_lds<D, NW>((size_t)NST * 2 * SplitTile<D, 32>::ELEMS * sizeof(__bf16), float_tiles<D>, 1);
  auto kern = fwd_split_kernel<D, NW, NST, BY_LENGTH>;
  static PrepareState once;
  if (int rc = prepare(kern, lds, once)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), lds, st, p);
  return (int)hipGetLastError();
}
template <int D, int NW, int NST> static int fwd_split_launch(FwdParams p, hipStream_t st) {
  const int64_t blocks = set_tiles(p, NW * 32, SHORT_LAST);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  tile_order_f32<D>(p, D == 128 ? 256 : 128);
  if constexpr (D != 128 || NW == 8) {
    // a kernel of its own: with the branch in one, launches without the order were 0.5 to 2 % slower (D=128, 16 x 16 x 400 98.9 -> 99.8 us)
    set_length_order(p, D == 128 ? 768 : 384);
    if (p.by_length) return fwd_split_run<D, NW, NST, true>(p, blocks, st);
  }
  return fwd_split_run<D, NW, NST, false>(p, blocks, st);
}
template <int D> static int fwd_first_launch(FwdParams p, hipStream_t st) {
  using C = Cfg<ElemT>;
  constexpr int TQ = C::NW * 32;
  constexpr size_t lds = (size_t)2 * 2 * C::FWD_TK * TileGeom<ElemT, D>::PITCH * sizeof(ElemT);
  auto kern = fwd_kernel<ElemT, D, C::NW, C::FWD_TK>;
  static PrepareState once;
  if (int rc = prepare(kern, lds, once)) return rc;
  const int64_t blocks = set_tiles(p, TQ, PLAIN);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(C::NW * 64), lds, st, p);
  return (int)hipGetLastError();
}
template <int D> static int fwd_d(FwdParams p, hipStream_t st) {
  using C = Cfg<ElemT>;
  if constexpr (C::fwd2(D)) {
    if constexpr (D == 16) {
      if (!slices_fit(p)) return fwd_first_launch<D>(p, st);
    }
    if constexpr (D == 128) {
      if (launch_choice(D, p.C, p.R).fwd == FWD_PIPELINED) return fwd3_launch<D>(p, st);
    }
    // windows of less than 1024 keys (the table's first two window classes) run the short-window form
    if (window_class(p.C, p.R) <= 1) {
      if constexpr (D <= 64) {
        if (forward_in_two_waves(D, p.C, p.R)) return fwd2_launch<D, 2, 32, true>(p, st);
      }
      return fwd2_launch<D, C::NARROW_NW, C::FWD_TK, true>(p, st);
    }
    return fwd2_launch<D, C::NARROW_NW, C::FWD_TK, false>(p, st);
  } else if constexpr (C::split(D)) {
    // Head dimension 128: eight waves share one workgroup's two 48 KiB stages, two waves per SIMD, once that makes a
    // workgroup per CU; smaller grids run twice as many four-wave workgroups with one stage (B*H=24, T=1024: 34
    // against 44 us; B*H=64, T=2048, 512 of the large ones: 91 against 82 us).
    if constexpr (D == 128) {
      if ((int64_t)p.B * p.H * ceil_div(p.T, 256) < 256) return fwd_split_launch<D, 4, 1>(p, st);
      return fwd_split_launch<D, 8, 2>(p, st);
    } else {
      if (half_workgroups(p)) return fwd_split_launch<D, 2, 2>(p, st);
      return fwd_split_launch<D, 4, 2>(p, st);
    }
  } else {
    return fwd_first_launch<D>(p, st);
  }
}
template <> int launch_fwd<ElemT, SA_DGROUP>(const FwdParams& p, int D, hipStream_t st) {
#define X(d) return fwd_d<d>(p, st)
  SA_FOR_EACH_D(X)
#undef X
}
#elif SA_KIND == 1
template <int D> static int delta_d(const DeltaParams& p, hipStream_t st) {
  constexpr int RPB = 256 / (D / Elem<ElemT>::VEC);
  const int64_t rows = (int64_t)p.B * p.H * p.T;
  const int64_t blocks = ceil_div(rows, RPB);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  hipLaunchKernelGGL((delta_kernel<ElemT, D>), dim3((unsigned)blocks), dim3(256), 0, st, p);
  return (int)hipGetLastError();
}
template <> int launch_delta<ElemT, SA_DGROUP>(const DeltaParams& p, int D, hipStream_t st) {
#define X(d) return delta_d<d>(p, st)
  SA_FOR_EACH_D(X)
#undef X
}
template <int D, int NW> static int dq2_launch(BwdParams p, hipStream_t st) {
  using C = Cfg<ElemT>;
  constexpr int TQ = NW * 32;
  // beside the stages up to head dimension 64: a workgroup's dO rows
  constexpr size_t stages = (size_t)(RING + (D <= 64 ? 1 : 0)) * 2 * C::DQ2_TK * D * sizeof(ElemT);
  constexpr size_t patches = (size_t)NW * RowPatch<ElemT, D>::ELEMS * sizeof(ElemT);
  constexpr size_t lds = stages > patches ? stages : patches;
  auto kern = dq2_kernel<ElemT, D, NW, C::DQ2_TK>;
  static PrepareState once;
  if (int rc = prepare(kern, lds, once)) return rc;
  const int64_t blocks = set_tiles(p, TQ, D == 256 ? backward_tail_256(p.lens) : SHORT_LAST);
  set_tile_order(p, TQ, C::DQ2_TK);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), lds, st, p);
  return (int)hipGetLastError();
}
// hand-scheduled loop, one wave per SIMD, 64 queries per wave (head dimension 128)
template <int D> static int dq3_launch(BwdParams p, hipStream_t st) {
#ifdef SA_NO_ASM_KERNELS
  (void)p; (void)st;
  return SA_ERR_HEAD_DIM;
#else
  using C = Cfg<ElemT>;
  if constexpr (C::fwd2(D) && D == 128) {
    constexpr int NW = 4, TQ = NW * 64, NST = 4;
    constexpr size_t stages = (size_t)(NST + 1) * 2 * 64 * D * sizeof(ElemT);   // one for half of the dO rows
    constexpr size_t patches = (size_t)NW * RowPatch<ElemT, D>::ELEMS * sizeof(ElemT);
    constexpr size_t lds = stages > patches ? stages : patches;
    auto kern = dq3_kernel<ElemT, D, NST>;
    static PrepareState once;
    if (int rc = prepare(kern, lds, once)) return rc;
    const int64_t blocks = set_tiles(p, TQ, SHORT_LAST);
    if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), lds, st, p);
    return (int)hipGetLastError();
  } else {
    return SA_ERR_HEAD_DIM;
  }
#endif
}
template <int D, int NW> static int dq_split_launch(BwdParams p, hipStream_t st) {
  constexpr int TQ = NW * 32;
  constexpr size_t lds = split_lds<D, NW>((size_t)2 * 2 * SplitTile<D, 32>::ELEMS * sizeof(__bf16), float_tiles<D>, 2);
  auto kern = dq_split_kernel<D, NW>;
  static PrepareState once;
  if (int rc = prepare(kern, lds, once)) return rc;
  const int64_t blocks = set_tiles(p, TQ, SHORT_LAST);
  tile_order_f32<D>(p, 128);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), lds, st, p);
  return (int)hipGetLastError();
}
template <int D> static int dq_first_launch(BwdParams p, hipStream_t st) {
  using C = Cfg<ElemT>;
  if (p.delta_out) return SA_ERR_ARG;
  constexpr int TQ = C::NW * 32;
  constexpr size_t lds = (size_t)2 * 2 * C::DQ_TK * TileGeom<ElemT, D>::PITCH * sizeof(ElemT);
  auto kern = dq_kernel<ElemT, D, C::NW, C::DQ_TK>;
  static PrepareState once;
  if (int rc = prepare(kern, lds, once)) return rc;
  const int64_t blocks = set_tiles(p, TQ, PLAIN);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(C::NW * 64), lds, st, p);
  return (int)hipGetLastError();
}
template <int D> static int dq_d(BwdParams p, hipStream_t st) {
  using C = Cfg<ElemT>;
  if constexpr (C::fwd2(D)) {
    if constexpr (D == 16) {
      if (!slices_fit(p)) return dq_first_launch<D>(p, st);
    }
    if constexpr (D == 128) {
      if (launch_choice(D, p.C, p.R).dq == DQ_PIPELINED) return dq3_launch<D>(p, st);
    }
    return dq2_launch<D, C::NARROW_NW>(p, st);
  } else if constexpr (C::split(D)) {
    if constexpr (D <= 64) {
      if (half_workgroups(p)) return dq_split_launch<D, 2>(p, st);
    }
    return dq_split_launch<D, 4>(p, st);
  } else {
    return dq_first_launch<D>(p, st);
  }
}
template <> int launch_dq<ElemT, SA_DGROUP>(const BwdParams& p, int D, hipStream_t st) {
#define X(d) return dq_d<d>(p, st)
  SA_FOR_EACH_D(X)
#undef X
}
#elif SA_KIND == 2
template <int D> static int dkdv3_launch(BwdParams p, hipStream_t st) {
#ifdef SA_NO_ASM_KERNELS
  (void)p; (void)st;
  return SA_ERR_HEAD_DIM;
#else
  using C = Cfg<ElemT>;
  if constexpr (C::fwd2(D) && D == 128) {
    constexpr int TKB = 128, TQ = 64;
    // tile stages; the epilogue's row patches (one per wave) reuse the same memory
    constexpr size_t stages = (size_t)C::DKDV3_NST * (2 * TQ * D * sizeof(ElemT) + 2 * TQ * sizeof(float)) +
                              (size_t)4 * OwnRows<ElemT, D>::ELEMS * sizeof(ElemT);   // a workgroup's V rows
    constexpr size_t patches = (size_t)4 * RowPatch<ElemT, D>::ELEMS * sizeof(ElemT);
    constexpr size_t lds = stages > patches ? stages : patches;
    auto kern = dkdv3_kernel<ElemT, D, C::DKDV3_NST>;
    static PrepareState once;
    if (int rc = prepare(kern, lds, once)) return rc;
    const int64_t blocks = set_tiles(p, TKB, SHORT_LAST);
    if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), lds, st, p);
    return (int)hipGetLastError();
  } else {
    return SA_ERR_HEAD_DIM;
  }
#endif
}
// wave pairs: 8 waves (two per SIMD) own 128 keys
template <int D> static int dkdv_split_launch(BwdParams p, hipStream_t st) {
  using C = Cfg<ElemT>;
  if constexpr (C::fwd2(D) && D >= 64 && D <= 128) {
    constexpr int TKB = 128, TQ = 64, NST = 3, NW = 8;
    // tile stages followed by the pairs' exchange slots; the epilogue's row patches reuse the stages
    constexpr size_t stages = (size_t)NST * (2 * TQ * D * sizeof(ElemT) + 2 * TQ * sizeof(float));
    constexpr size_t patches = (size_t)NW * RowPatch<ElemT, D>::ELEMS * sizeof(ElemT);
    static_assert(patches <= stages, "row patches must not reach the exchange slots");
    constexpr size_t rows = stages / NST * (NST - 1) + (size_t)NW * OwnRows<ElemT, D>::ELEMS * sizeof(ElemT);
    constexpr size_t lds = std::max(stages + (size_t)4 * 2 * 2048, rows);
    auto kern = dkdv_split_kernel<ElemT, D, NST>;
    static PrepareState once;
    if (int rc = prepare(kern, lds, once)) return rc;
    const int64_t blocks = set_tiles(p, TKB, SHORT_FIRST);
    if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), lds, st, p);
    return (int)hipGetLastError();
  } else {
    return SA_ERR_HEAD_DIM;
  }
}
// wave pairs at head dimension 256: 8 waves (two per SIMD) own 128 keys
template <int D> static int dkdv_split_wide_launch(BwdParams p, hipStream_t st) {
  using S = DkdvSplitWide<ElemT, D>;
  auto kern = dkdv_split_wide_kernel<ElemT, D>;
  static PrepareState once;
  if (int rc = prepare(kern, S::lds, once)) return rc;
  const int64_t blocks = set_tiles(p, S::TKB, backward_tail_256(p.lens));
  set_tile_order(p, S::TKB, S::TQ);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(2 * S::NP * 64), S::lds, st, p);
  return (int)hipGetLastError();
}
template <int D, int NW> static int dkdv_split_f32_launch(BwdParams p, hipStream_t st) {
  constexpr int TKB = NW * 32;
  constexpr size_t rows = (size_t)2 * 2 * 32 * sizeof(float);   // lse and delta
  constexpr size_t lds = split_lds<D, NW>((size_t)2 * 2 * SplitTile<D, 32>::ELEMS * sizeof(__bf16) + rows, float_tiles<D> + rows, 2);
  auto kern = dkdv_split_f32_kernel<D, NW>;
  static PrepareState once;
  if (int rc = prepare(kern, lds, once)) return rc;
  const int64_t blocks = set_tiles(p, TKB, SHORT_LAST);
  tile_order_f32<D>(p, 128);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), lds, st, p);
  return (int)hipGetLastError();
}
template <int D> static int dkdv_first_launch(BwdParams p, hipStream_t st) {
  using C = Cfg<ElemT>;
  constexpr int TKB = C::NW * 32;
  constexpr size_t lds =
      (size_t)2 * (2 * C::DKDV_TQ * TileGeom<ElemT, D>::PITCH * sizeof(ElemT) + 2 * C::DKDV_TQ * sizeof(float));
  const int64_t blocks = set_tiles(p, TKB, PLAIN);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  if constexpr (sizeof(ElemT) == 4 && D == 256) {
    // both accumulators and both resident rows do not fit a lane's registers: one launch per gradient
    auto kern_dv = dkdv_kernel<ElemT, D, C::NW, C::DKDV_TQ, 1>;
    auto kern_dk = dkdv_kernel<ElemT, D, C::NW, C::DKDV_TQ, 2>;
    static PrepareState once_dv, once_dk;
    if (int rc = prepare(kern_dv, lds, once_dv)) return rc;
    if (int rc = prepare(kern_dk, lds, once_dk)) return rc;
    hipLaunchKernelGGL(kern_dv, dim3((unsigned)blocks), dim3(C::NW * 64), lds, st, p);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(kern_dk, dim3((unsigned)blocks), dim3(C::NW * 64), lds, st, p);
    return (int)hipGetLastError();
  } else {
    auto kern = dkdv_kernel<ElemT, D, C::NW, C::DKDV_TQ>;
    static PrepareState once;
    if (int rc = prepare(kern, lds, once)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(C::NW * 64), lds, st, p);
    return (int)hipGetLastError();
  }
}
template <int D> static int dkdv_d(BwdParams p, hipStream_t st) {
  using C = Cfg<ElemT>;
  if constexpr (C::fwd2(D) && D == 256) {
    return dkdv_split_wide_launch<D>(p, st);
  } else if constexpr (C::fwd2(D)) {
    if constexpr (D == 16) {
      if (!slices_fit(p)) return dkdv_first_launch<D>(p, st);
    }
    if constexpr (D >= 64) {   // a 64-byte row splits over four waves' copies, not over eight
      if (launch_choice(D, p.C, p.R).dkdv == DKDV_SPLIT) return dkdv_split_launch<D>(p, st);
    }
    // The pipelined kernel (head dimension 128) makes every wave walk the whole window of its
    // workgroup's 128 keys; that wastes nothing once a chunk holds at least those 128 keys.  Smaller
    // chunks go to the kernel whose waves skip the query tiles outside their own 32 keys' windows.
    if constexpr (D == 128) {
      if (launch_choice(D, p.C, p.R).dkdv == DKDV_PIPELINED) return dkdv3_launch<D>(p, st);
    }
    constexpr int TKB = C::DKDV2_NW * 32;
    constexpr size_t stages =
        (size_t)RING * (2 * C::DKDV2_TQ * D * sizeof(ElemT) + 2 * C::DKDV2_TQ * sizeof(float)) +
        (size_t)C::DKDV2_NW * OwnRows<ElemT, D>::ELEMS * sizeof(ElemT);   // a workgroup's V rows
    constexpr size_t patches = (size_t)C::DKDV2_NW * RowPatch<ElemT, D>::ELEMS * sizeof(ElemT);
    constexpr size_t lds = stages > patches ? stages : patches;
    auto kern = dkdv2_kernel<ElemT, D, C::DKDV2_NW, C::DKDV2_TQ>;
    static PrepareState once;
    if (int rc = prepare(kern, lds, once)) return rc;
    const int64_t blocks = set_tiles(p, TKB, SHORT_LAST);
    set_tile_order(p, TKB, C::DKDV2_TQ);
    if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(C::DKDV2_NW * 64), lds, st, p);
    return (int)hipGetLastError();
  } else if constexpr (C::split(D)) {
    if constexpr (D <= 64) {
      if (half_workgroups(p)) return dkdv_split_f32_launch<D, 2>(p, st);
    }
    return dkdv_split_f32_launch<D, 4>(p, st);
  } else {
    return dkdv_first_launch<D>(p, st);
  }
}
template <> int launch_dkdv<ElemT, SA_DGROUP>(const BwdParams& p, int D, hipStream_t st) {
#define X(d) return dkdv_d<d>(p, st)
  SA_FOR_EACH_D(X)
#undef X
}
#else
template <int D, int NW, int TT> static int bwd_fused_launch(BwdParams p, hipStream_t st) {
  using S = BwdFused<NW, TT>;
  p.fused_rows = rows_in_reach(p.C, p.R, S::ROWS, TT);
  const size_t lds = S::template lds_bytes<ElemT, D>(p.fused_rows);
  auto kern = bwd_fused_kernel<ElemT, D, NW, TT>;
  static PrepareState once;
  if (int rc = prepare(kern, S::template lds_bytes<ElemT, D>(BWD_FUSED_MAX_ROWS), once)) return rc;
  const int64_t blocks = set_tiles(p, S::ROWS, PLAIN);
  if (blocks > 0x7fffffffLL) return SA_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NW * 64), lds, st, p);
  return (int)hipGetLastError();
}
template <int D> static int bwd_fused_d(BwdParams p, hipStream_t st) {
  if constexpr (fused_backward_exists<ElemT>(D)) {
    if (fused_backward_in_two_waves(D, p.C, p.R)) return bwd_fused_launch<D, 2, 32>(p, st);
    return bwd_fused_launch<D, 4, 64>(p, st);
  } else {
    return SA_ERR_HEAD_DIM;
  }
}
template <> int launch_bwd_fused<ElemT>(const BwdParams& p, int D, hipStream_t st) {
#define X(d) return bwd_fused_d<d>(p, st)
  SA_FOR_EACH_D(X)
#undef X
}
#endif

}  // namespace sa
