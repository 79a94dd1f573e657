// Host-side launch entry points, one explicit instantiation per element type.
// Each returns 0, a positive hipError_t, or a negative SA_ERR_* code.
#pragma once
#include <atomic>
#include "../../include/streaming_attention.h"
#include "sa_common.h"

#define SA_OK 0

namespace sa {


template <typename T, int DGROUP> int launch_fwd(const FwdParams& p, int D, hipStream_t st);
template <typename T, int DGROUP> int launch_delta(const DeltaParams& p, int D, hipStream_t st);
template <typename T, int DGROUP> int launch_dq(const BwdParams& p, int D, hipStream_t st);
template <typename T, int DGROUP> int launch_dkdv(const BwdParams& p, int D, hipStream_t st);
template <typename T> int launch_bwd_fused(const BwdParams& p, int D, hipStream_t st);

// tile sizes, shared between the launchers and sa_query()
#ifndef SA_FWD2_QB
#define SA_FWD2_QB 1
#endif
#ifndef SA_DQ2_TK
#define SA_DQ2_TK 64
#endif
#ifndef SA_DKDV2_NW
#define SA_DKDV2_NW 4
#endif
#ifndef SA_DKDV2_TQ
#define SA_DKDV2_TQ 64
#endif
#ifndef SA_DKDV3_NST
#define SA_DKDV3_NST 3
#endif
// ---- launch-configuration table -------------------------------------------------------------------
// The 16-bit kernels for head dimensions 64 and 128 exist in several shapes (256 in one); which one runs is read
// from a table indexed by head dimension, chunk-size class and window-size class.  The entries are
// the fastest variant measured on an MI355X at B=4, H=16, T=16384 (`bench.py --tune-sweep`, turned into
// sa_tune_table.inc by gen_tune_table.py); float16 and bfloat16 measured alike and share the entries.
enum FwdVariant : int { FWD_NARROW = 0,     // 4 waves (128 queries) per workgroup, two workgroups per CU
                        FWD_PIPELINED = 1,  // hand-scheduled loop, 4 waves of 64 queries (head dimension 128 only)
                        FWD_VARIANTS = 2 };
enum DqVariant : int { DQ_NARROW = 0,      // 4 waves (128 queries) per workgroup
                       DQ_PIPELINED = 1,   // hand-scheduled loop, 4 waves of 64 queries (head dimension 128 only)
                       DQ_VARIANTS = 2 };
enum DkdvVariant : int { DKDV_BLOCKSKIP = 0,   // every wave skips the query tiles outside its own 32 keys' windows
                         DKDV_PIPELINED = 1,   // hand-scheduled loop, head dimension 128 only
                         DKDV_SPLIT = 2,       // wave pairs share 32 keys: one wave forms S and dV, the other dP and dK
                         DKDV_VARIANTS = 3 };
struct LaunchChoice { int fwd, dq, dkdv; };
constexpr int TUNE_CHUNK_CLASSES = 7;    // context_size < 32, < 64, < 128, < 256, < 512, < 1024, >= 1024
constexpr int TUNE_WINDOW_CLASSES = 4;   // context_size * (back_contexts + 1) < 256, < 1024, < 4096, >= 4096
constexpr int chunk_class(int chunk) {
  return chunk < 32 ? 0 : chunk < 64 ? 1 : chunk < 128 ? 2 : chunk < 256 ? 3 : chunk < 512 ? 4 : chunk < 1024 ? 5 : 6;
}
constexpr int window_class(int chunk, int back) {
  const long long w = (long long)chunk * ((long long)back + 1);
  return w < 256 ? 0 : w < 1024 ? 1 : w < 4096 ? 2 : 3;
}
#include "sa_tune_table.inc"
// Variants pinned through sa_tune_override() for measurements and tests; -1 = use the table.  Atomics, so
// that a launch on one thread reads a whole value while another thread pins or releases a variant.
extern std::atomic<int> g_tune_override[3];
// The hand-scheduled kernels are single assembly statements over fixed registers.  A build with
// -DSA_NO_ASM_KERNELS leaves them out (for a compiler that cannot satisfy their register constraints)
// and serves their table cells with the compiler-scheduled kernels.
#ifdef SA_NO_ASM_KERNELS
constexpr bool kAsmKernels = false;
#else
constexpr bool kAsmKernels = true;
#endif
inline LaunchChoice launch_choice(int D, int chunk, int back) {
  // head dimension 256 has one shape per kernel, variant 0 whatever it is called elsewhere (dK/dV: dkdv_split_wide_kernel)
  if (D == 256) return LaunchChoice{FWD_NARROW, DQ_NARROW, DKDV_BLOCKSKIP};
  LaunchChoice c = (D == 128 ? TUNE_D128 : TUNE_D64)[chunk_class(chunk)][window_class(chunk, back)];
  const int o0 = g_tune_override[0].load(std::memory_order_relaxed);
  const int o1 = g_tune_override[1].load(std::memory_order_relaxed);
  const int o2 = g_tune_override[2].load(std::memory_order_relaxed);
  if (o0 >= 0 && o0 < FWD_VARIANTS) c.fwd = o0;
  if (o1 >= 0 && o1 < DQ_VARIANTS) c.dq = o1;
  if (o2 >= 0 && o2 < DKDV_VARIANTS) c.dkdv = o2;
  const bool pipelined = kAsmKernels && D == 128;
  if (!pipelined && c.dkdv == DKDV_PIPELINED) c.dkdv = DKDV_BLOCKSKIP;
  if (!pipelined && c.dq == DQ_PIPELINED) c.dq = DQ_NARROW;
  if (!pipelined && c.fwd == FWD_PIPELINED) c.fwd = FWD_NARROW;
  return c;
}

// Rows that a workgroup of `rows` rows goes through for its windows, in whole tiles: the most over all positions.
inline int rows_in_reach(int chunk, int back, int rows, int tile) {
  int period = chunk;   // the pattern repeats after chunk / gcd(chunk, rows) workgroups
  while (period % 2 == 0 && period > chunk / rows) period /= 2;
  int most = 0;
  for (int i = 0; i < period; ++i) {
    const int first = rows * i / chunk * chunk / tile, last = ((rows * i + rows - 1) / chunk + back + 1) * chunk;
    most = (last + tile - 1) / tile - first > most ? (last + tile - 1) / tile - first : most;
  }
  return most * tile;
}
// The tiles of a full window of a workgroup of `rows` rows, for TileOrder; 0 where the order has nothing to gain: a window
// that covers the sequence (every workgroup begins at the first tile anyway).
inline int tiles_of_window(int T, int chunk, int back, int rows, int tile) {
  const long long chunks = chunk % rows == 0 ? 1 : rows % chunk == 0 ? rows / chunk : (rows + chunk - 2) / chunk + 1;
  const long long span = (chunks + back) * chunk;
  if (span >= T) return 0;
  const bool aligned = chunk % tile == 0 || (rows % chunk == 0 && (long long)chunk * back % tile == 0);
  return (int)((span + tile - 1 + (aligned ? 0 : tile - 1)) / tile);
}
// The workgroups of a launch, `rows` rows each, and how they are dispatched (tile_coords).  Those whose windows are still growing
// (query tiles: the first R chunks of a sequence) or already shrinking (key tiles: the last) come last with SHORT_LAST, where
// the pairs divide over the XCDs and they are no more than half.  SHORT_FIRST, for kernels with one workgroup per CU: equal
// workgroups that start together stay in step, all CUs fetch their rows at the same time and the memory idles while all
// multiply (a fifth of dQ at head dimension 256 went by at full memory rate); short workgroups at the beginning leave the CUs at
// different points.  Only from 512 workgroups on: with few rounds the long ones that come last show (256 at D=256: 73.4 -> 73.8).
// Forward and backward in us, short last -> first, dkdv_split_kernel, D=128: 64, 1 back, T=2048, 1280 workgroups 140 -> 137, ragged 94 ->
// 89; 50, 3 back, T=3000, 1536 workgroups 218 -> 208, ragged 178 -> 174; on large grids within 1 % (8192, ragged 710 -> 724 at the
// worst).  Two or three workgroups per CU keep each other busy and lose: D=64, 128, 4 back 422 -> 431; the forward at D=256, whole
// lengths -2 to +10 %, ragged up to +21 % (200, 2 back, 640 workgroups 52.4 -> 63.6).  The other kernels of head dimension 128 gain on
// some windows and lose as much on others.
enum Tail { PLAIN, SHORT_LAST, SHORT_FIRST };
// The backward at D=256: first where every sequence has its whole length (64, 3 back, T=2048, 640 workgroups 202 -> 196, T=4096, 2048
// workgroups 567 -> 550; 128, 4 back 886 -> 869; 200, 2 back, T=1000 223 -> 218).  Of ragged lengths a part of the workgroups is
// empty, fewer rounds are left and the long ones that come last show: any lengths in [1, T], 200, 2 back, T=1000 162 -> 186, T=2048
// 600 -> 659; 128, 4 back 133 -> 151, 531 -> 583; short chunks would gain (64, 3 back 200 -> 195, 714 -> 699) less than those lose.
inline Tail backward_tail_256(const void* lens) { return lens ? SHORT_LAST : SHORT_FIRST; }
template <typename P> int64_t set_tiles(P& p, int rows, Tail tail) {
  TileMap& m = p.tiles;
  m.n_tiles = (int)(((int64_t)p.T + rows - 1) / rows);
  const int64_t nbh = (int64_t)p.B * p.H, growing = ((int64_t)p.C * p.R + rows - 1) / rows;
  m.nbh = (int)nbh;
  m.n_tail = tail != PLAIN && nbh % 8 == 0 && (int64_t)p.C * p.R < p.T && 2 * growing <= m.n_tiles ? (int)growing : 0;
  m.tail_first = tail == SHORT_FIRST && nbh * m.n_tiles >= 512 ? (int)(nbh / 8) * m.n_tail : 0;
  m.by_tiles = chunk_div(m.n_tiles);
  m.by_lead = chunk_div(m.n_tiles - m.n_tail);
  m.by_pairs = chunk_div(nbh >= 16 && nbh <= 0x7fffffff ? (int)(nbh >> 3) : 1);
  m.by_heads = chunk_div(p.H);
  return nbh * m.n_tiles;
}
// tile_coords_by_length where it can (one length and one pair of an XCD to a lane, pairs that divide over the XCDs), on more workgroups
// than CUs, and from the length on at which they live long enough to pay for it (about a microsecond each).  Forward in us, lengths in
// [T/2, T] unless said otherwise, without -> with.  Float16, D=64: 8 x 12 x 1500 54.6 -> 48.3, any lengths 28.1 -> 25.2; 4 x 8 x 2048 36.8 ->
// 34.8; 8 x 12 x 900, any lengths 24.3 -> 20.5; 32 x 8 x 1024, any lengths 45.7 -> 41.2; D=128, 3 x 8 x 2000 48.0 -> 41.5; D=32, 16 x 12 x
// 1500 64.4 -> 58.5; D=16, 16 x 12 x 900 30.1 -> 28.1; D=256, 8 x 8 x 1500 119.6 -> 115.2.  On the other side, D=64: 16 x 12 x 700 28.8 ->
// 29.3, 500 17.7 -> 17.0, 300 10.1 -> 10.9; 32 x 12 x 300, any lengths 11.9 -> 14.2; 192 workgroups, D=128, 2 x 12 x 1000 20.3 -> 20.7.
// Float32: D=64, 8 x 8 x 1500 157 -> 152, 16 x 8 x 600 at D=16 36 -> 32; D=32, 16 x 12 x 900 100 -> 84, 400 27.6 -> 25.2; D=16, 16 x 12 x 900 82 -> 69; below the
// line either way, 16 x 8 x 300 at D=64 25.9 -> 24.2, 32 x 16 x 260 at 64, 32, 16 46.8 -> 48.2, 31.3 -> 32.9, 26.1 -> 28.0.  D=128 in eight waves, 8 x 8 x 1500 322
// -> 306, 16 x 8 x 800 186 -> 160; below the line either way, 16 x 16 x 600 215 -> 217, 8 x 16 x 700 131 -> 134, 16 x 16 x 400 99.6 -> 94.5; in four waves 6 x 4 x
// 1800 208 -> 214.  Longest sequences first with the empty tiles left among the others: float16, D=64, 8 x 12 x 1500 51.1, any lengths 31.0.
inline void set_length_order(FwdParams& p, int shortest) {
  const bool whole = (int64_t)p.C * ((int64_t)p.R + 1) >= p.T && p.T >= shortest;
  const bool fits = p.B <= 32 && p.tiles.nbh % 8 == 0 && p.tiles.nbh <= 512;
  p.by_length = p.lens && whole && fits && p.B > 1 && (int64_t)p.tiles.nbh * p.tiles.n_tiles > 256 ? p.B : 0;
}
template <typename P> void set_tile_order(P& p, int rows, int tile) {
  p.period = tiles_of_window(p.T, p.C, p.R, rows, tile);
  p.pdiv = chunk_div(p.period > 0 ? p.period : 1);
}
// Short windows, head dimensions 16 to 64: workgroups of two waves (64 rows, tiles of 32) instead of four (128 rows,
// tiles of 64).  In the large workgroup every wave waits at the barriers of about twice as many tiles as it sees itself,
// and half as many waves are resident; the small one goes through more rows per row of its own unless the windows begin and
// end where its rows do.  So it is taken where that costs nothing (chunks divide 32 or are divided by it, and the
// rows in reach are no more per row), and where the windows lie across the 32-row blocks, so that the kernel is bound by
// what it computes, not by what it reads.
inline bool aligned_chunks(int chunk) { return 32 % chunk == 0 || chunk % 32 == 0; }
inline bool two_waves_read_no_more(int chunk, int back) {
  return aligned_chunks(chunk) && 2 * rows_in_reach(chunk, back, 64, 32) <= rows_in_reach(chunk, back, 128, 64);
}
// The windows alone decide, not the size of the grid: the two forms look for the maximum of a row in tiles of different
// size, and a sequence has the same bits alone and in any batch.
// The forward in us, four waves -> two.  D=32, B=225, H=4, T<=993: chunks of 16, 2 back 37.5 -> 29.5; 10, 9 back 48.7 -> 38.1; 64, 1 back
// 36.8 -> 32.1; 64, 7 back 54.7 -> 52.9; 10, 40 back (410 keys) 61 -> 55; on the other side 128, none back 34.4 -> 32.6 (64 x 8 x
// 1024: 26.6 -> 26.5), 128, 3 back 53.0 -> 55.5.  D=64, B=128, H=12, T=1354: 10, 9 back 248 -> 229; 50, 1 back 254 -> 228; 10, 20 back
// 313 -> 307; 16, 2 back 189 -> 182; 32, 1 back 188 -> 181; on the other side 32, 2 back 193 -> 197 (64 x 8 x 1024: 55.5 -> 58.0),
// 64, 2 back 65.9 -> 74.6, 128, none back 53.8 -> 62.2, 10, 40 back 406 -> 424.  On grids of up to 1024 workgroups of 128 rows the
// other side differs less, either way (16 x 8 x 1024 ragged): 32, 2 back 14.1 -> 13.0; 128, none back 14.1 -> 12.2; 64, 2 back 16.1
// -> 15.6; 64, 1 back 14.6 -> 15.4.
// D=16, B=225, H=4, T<=993; 64 x 8 x 1024: 16, 2 back 29.4 -> 21.4; 24.4 -> 18.7; 10, 9 back 40.7 -> 30.0; 35.5 -> 28.5; 64, 1 back 27.3 ->
// 23.1; 23.2 -> 20.2; 64, 7 back 45.7 -> 44.0; 44.9 -> 44.3; on the other side 128, none back 26.8 -> 24.0; 19.5 -> 20.3; 128, 3 back
// 43.1 -> 45.0; 42.7 -> 45.6.
inline bool forward_in_two_waves(int D, int chunk, int back) {
  const long long window = (long long)chunk * ((long long)back + 1);
  if (D <= 32) return chunk < 128 && window <= 512;
  return D == 64 && window <= 256 && (!aligned_chunks(chunk) || two_waves_read_no_more(chunk, back));
}

// The kernels with copies into LDS address the rows of a (batch, head) slice with 32-bit byte offsets.  At head dimension 16
// slices that are longer go to the first kernels (sa_fwd.h, sa_bwd.h), which have no such limit.
inline bool offsets_fit(int T, int64_t row_stride) { return ((int64_t)T + 1024) * row_stride * 2 < (int64_t(1) << 32); }
inline bool slices_fit(const FwdParams& p) { return offsets_fit(p.T, p.q_st) && offsets_fit(p.T, p.k_st) && offsets_fit(p.T, p.v_st); }
inline bool slices_fit(const BwdParams& p) {
  return offsets_fit(p.T, p.q_st) && offsets_fit(p.T, p.k_st) && offsets_fit(p.T, p.v_st) && offsets_fit(p.T, p.do_st);
}

// The one-launch backward (sa_bwd_fused.h), 16-bit elements.
template <typename T> constexpr bool fused_backward_exists(int D) { return sizeof(T) == 2 && (D == 16 || D == 32 || D == 64); }
// Used while the query rows that a workgroup of 128 rows goes through for dK and dV are few: beyond its own 128 it reads and
// multiplies rows that belong to its neighbours.  Forward and backward against the two launches, rows: gain -- D=64, B=8, H=16,
// T=4096 128: 1.12 to 1.24; 192: 1.06 to 1.17; 256: 1.01 to 1.05; 320: 0.95 to 0.99; B=64, H=12, T=1354 1.17 to 1.31; 1.11 to 1.27; 1.04
// to 1.06; 1.00 to 1.02; the backward alone, when it came, 384: 0.94; 448: 0.91.  D=32, B=225, H=4, T=993 and B=16, H=16, T=4096 128:
// 1.06 to 1.22; 192: 1.06 to 1.19; 256: 1.02 to 1.04; the backward alone, when it came, 320: 0.98; 384: 0.91.  D=16, the same problems,
// forward and backward: 192 80.0 against 88.3 us, 256 95.9 against 99.5 and 88 against 90.
constexpr int BWD_FUSED_MAX_ROWS = 320;
inline bool fused_backward(int D, int chunk, int back) {
  if (!fused_backward_exists<__bf16>(D)) return false;
  // a pinned dQ or dK/dV variant asks for the launches of their own
  if (g_tune_override[1].load(std::memory_order_relaxed) >= 0 || g_tune_override[2].load(std::memory_order_relaxed) >= 0)
    return false;
  if ((long long)chunk * ((long long)back + 1) > BWD_FUSED_MAX_ROWS) return false;
  return rows_in_reach(chunk, back, 128, 64) <= (D == 64 ? BWD_FUSED_MAX_ROWS : 256);
}
// Forward and backward in us, four waves -> two.  D=32, B=225, H=4, T<=993: chunks of 16, 2 back 125.4 -> 119.2; 40, 2 back 158.0 -> 148.9;
// 10, 9 back 157.5 -> 151.7; on the other side 32, 3 back 130.1 -> 128.1 (64 x 8 x 1024: 104.9 -> 111.0), 64, 1 back 124.7 -> 122.2 (98.8 ->
// 102.4), 128, none back 116.5 -> 122.4.  D=64, B=64, H=12, T=1354: 8, 3 back 339 -> 324; 16, 2 back 335 -> 323; 64, none back 306 -> 293; on the
// other side 10, 9 back 463 -> 465, 32, 2 back 348 -> 347 (64 x 8 x 1024: 182 -> 189), 32, 3 back 390 -> 396, 128, none back 344 -> 365.
// D=16 reads little and takes the small workgroups for all chunks below 128: B=225, H=4, T<=993; 64 x 8 x 1024, backward alone: 16, 2 back
// 64.4 -> 53.5; 52.4 -> 46.3; 32, 3 back 66.8 -> 59.0; 56.2 -> 53.0; 64, 1 back 64.0 -> 55.4; 52.5 -> 49.0; 64, 2 back 71.2 -> 63.2; 61.0 ->
// 61.1; on the other side 128, none back 60.4 -> 59.0; 44.3 -> 48.2.
inline bool fused_backward_in_two_waves(int D, int chunk, int back) {
  if (D == 16) return chunk < 128;
  return (D == 32 && !aligned_chunks(chunk)) || two_waves_read_no_more(chunk, back);
}

template <typename T> struct Cfg {
  static constexpr int NW = 4;                                   // waves per workgroup
  // 16-bit, D in {64, 128, 256}: forward kernel with QB query blocks per wave.
  // The compiler-scheduled forward and dQ kernels run 4 waves (128 queries) per workgroup, two workgroups
  // per CU (an 8-wave shape measured slower or equal in every cell of the tuning sweep and was removed).
  static constexpr int NARROW_NW = 4;
  static constexpr int DQ2_TK = SA_DQ2_TK;
  static constexpr int DKDV2_NW = SA_DKDV2_NW, DKDV2_TQ = SA_DKDV2_TQ;
  // The software-pipelined dK/dV kernel exists at head dimension 128 only: at 64 a block step has
  // half the MFMAs for the same softmax arithmetic, the loop is bound by its vector work and dkdv2
  // is faster (0.23 against 0.30 ms at B=8, H=16, T=4096, chunk 128).
  static constexpr int DKDV3_NST = SA_DKDV3_NST;
  static constexpr int FWD2_QB = SA_FWD2_QB;
#ifdef SA_FWD2_DISABLE
  static constexpr bool fwd2(int) { return false; }
#else
  static constexpr bool fwd2(int D) { return sizeof(T) == 2 && (D == 16 || D == 32 || D == 64 || D == 128 || D == 256); }
#endif
  // float32 on the 16-bit matrix pipe (sa_f32.h); at 256 the parts of the resident rows exceed the registers
  static constexpr bool split(int D) { return sizeof(T) == 4 && D <= 128; }
#ifdef SA_FWD_TK16
  static constexpr int FWD_TK = sizeof(T) == 4 ? 32 : SA_FWD_TK16;
#else
  static constexpr int FWD_TK = sizeof(T) == 4 ? 32 : 64;        // keys per forward step
#endif
  static constexpr int DQ_TK = 32;                               // keys per dQ step
  static constexpr int DKDV_TQ = 32;                             // queries per dK/dV step
};

}  // namespace sa
