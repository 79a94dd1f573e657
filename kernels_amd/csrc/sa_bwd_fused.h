// The whole backward pass in one launch, for windows of about a hundred keys (16-bit elements, head dimensions 16 to 64).
//
// On such windows the two backward kernels are bound by memory: dQ reads q, k, v, O, dO and writes dQ, dK/dV
// reads q, k, v, dO again and writes two tensors -- twelve passes, of which eight are needed.  Here one
// workgroup owns the same 128 rows as queries and as keys: it forms delta for every query row that it
// is going to see (its own and the neighbours' in reach, whose O and dO rows the neighbouring
// workgroups of the same XCD read at about the same time), walks the key tiles of its queries (dq2_kernel's
// loop, three stages), picks up its own K and V rows from the tiles that are still in LDS, and walks the query tiles of
// its keys (dkdv2_kernel's loop).  A row that is read again ten microseconds later has mostly left the 4 MiB L2 of its XCD
// at this rate, which is why the pick-up counts: with two stages and the rows read again the kernel gained half as
// much.  Counters on the first problem below: 7.5 tensors fetched where five are needed and three written (192 rows in reach
// make the loads of a workgroup 11 tensors' worth; 5.4 TB/s, a copy reaches 6.25); the two launches fetched 10.9 and wrote 3.1.
//
// B=128, H=12, T=3000, D=64, chunks of 32, 2 back (float16): 1370 us in two launches, 1083 here; the same without the products
// 946; with results past the caches and the Q and dO rows of a wave through LDS 1031, 4.6 TB/s of the eight tensors.  When it came also B=8, H=16, T=4096, D=64, one
// chunk of 128: 160 -> 127 us.
// B=16, H=8, T=2048 ragged, D=64, chunks of 64, 1 back: 46 -> 39.  B=225, H=4, T=993 ragged, D=32, chunks of 16, 2 back: 94 -> 92.
// Two waves and 32-row tiles instead of four and 64 where that reads no more rows per row of its own (and at D = 32 on
// windows that lie across the 32-row blocks, at D = 16 on all chunks below 128): fused_backward_in_two_waves in sa_launch.h has the rule and both sides' times.
// A form that slides along a sequence and reads every row once (scores formed once, dS handed over in LDS) took 967 us
// on the first problem and up to twice as long on windows of more than four 32-row blocks: one workgroup per CU, steps
// in lockstep.
#pragma once
#include "sa_bwd.h"

namespace sa {

template <int NW_, int TT_> struct BwdFused {
  static constexpr int NW = NW_, ROWS = NW * 32, TT = TT_, NST = 3;
  // two stages, then the third or the row patches of the dQ store, then lse and delta of `rows` query rows
  template <typename T, int D> static constexpr int rows_offset() {
    constexpr int stage = 2 * TT * D * (int)sizeof(T), patches = NW * RowPatch<T, D>::ELEMS * (int)sizeof(T);
    return 2 * stage + (stage > patches ? stage : patches);
  }
  template <typename T, int D> static constexpr size_t lds_bytes(int rows) { return rows_offset<T, D>() + 2 * rows * sizeof(float); }
};

template <typename T, int D, int NW, int TT>
__global__ __launch_bounds__(NW * 64, (D == 64 ? 3 : 1)) void bwd_fused_kernel(const BwdParams p) {
  using E = Elem<T>;
  using G = TileGeom<T, D>;
  using Frag = typename E::Frag;
  static_assert(G::SWZ, "swizzled 16-bit tiles");
  using Shape = BwdFused<NW, TT>;
  constexpr int ROWS = Shape::ROWS, NT = NW * 64;
  constexpr int NF = G::NF, DB = G::DB, TILE = TT * D, STAGE = 2 * TILE;
  constexpr int PG = D == 64 ? 2 : 4;   // see dkdv2_kernel
  using Loader = TilePair<T, D, TT, NW, true>;
  constexpr int NST = Shape::NST, LPT = Loader::PER_WAVE;

  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  T* smem = reinterpret_cast<T*>(smem_raw);
  float* lse_s = reinterpret_cast<float*>(smem_raw + Shape::template rows_offset<T, D>());
  float* delta_s = lse_s + p.fused_rows;

  const int tid = threadIdx.x;
  const int lane = tid & 63, c = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int bh, rt;
  tile_coords(blockIdx.x, gridDim.x, p.tiles, bh, rt);
  const int b = div_by(bh, p.tiles.by_heads), hd = bh - b * p.H;
  const int T_ = p.T, C = p.C, R = p.R;
  auto cdiv = [&](int x) { return div_by(x, p.cdiv); };   // x / C
  int L = T_;
  if (p.lens) {
    L = p.lens[(int64_t)b * p.lens_stride];
    L = L < 0 ? 0 : (L > T_ ? T_ : L);
  }
  const int r0 = rt * ROWS, r1 = r0 + ROWS < T_ ? r0 + ROWS : T_;
  const int64_t out_row = (int64_t)bh * T_;
  T* dq_base = reinterpret_cast<T*>(p.dq) + out_row * D;
  T* dk_base = reinterpret_cast<T*>(p.dk) + out_row * D;
  T* dv_base = reinterpret_cast<T*>(p.dv) + out_row * D;
  if (r0 >= L) {
    zero_rows<T, D, NT>(dq_base, r0, r1, tid);
    zero_rows<T, D, NT>(dk_base, r0, r1, tid);
    zero_rows<T, D, NT>(dv_base, r0, r1, tid);
    for (int r = r0 + tid; r < r1; r += NT) p.delta_out[out_row + r] = 0.0f;
    return;
  }

  // ---- windows: keys of a query, queries of a key ---------------------------------------------------------
  auto valid = [&](int r) { return r < L ? r : L - 1; };   // rows past L mimic the last valid row
  auto k_lo = [&](int q) { const int x = cdiv(q); return (x > R ? x - R : 0) * C; };
  auto k_hi = [&](int q) { const int e = (cdiv(q) + 1) * C; return e < L ? e : L; };
  auto q_lo = [&](int k) { return cdiv(k) * C; };
  auto q_hi = [&](int k) { const int e = (cdiv(k) + R + 1) * C; return e < L ? e : L; };   // C * (R + 2) is small here
  const int row = r0 + wave * 32 + c;
  const int w_first = valid(r0 + wave * 32), w_last = valid(r0 + wave * 32 + 31), g_last = valid(r0 + ROWS - 1);
  const bool wave_live = r0 + wave * 32 < L;
  const WaveWindow wq{k_lo(valid(row)), k_hi(valid(row)), k_lo(w_last), k_hi(w_first), k_lo(w_first), wave_live ? k_hi(w_last) : 0};
  const WaveWindow wk{q_lo(valid(row)), q_hi(valid(row)), q_lo(w_last), q_hi(w_first), q_lo(w_first), wave_live ? q_hi(w_last) : 0};
  const int kt0 = k_lo(r0) / TT, kt1 = (k_hi(g_last) + TT - 1) / TT;
  const int qt0 = q_lo(r0) / TT, qt1 = (q_hi(g_last) + TT - 1) / TT;

  const T* qbase = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.q_sb + (int64_t)hd * p.q_sh;
  const T* kbase = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.k_sb + (int64_t)hd * p.k_sh;
  const T* vbase = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.v_sb + (int64_t)hd * p.v_sh;
  const T* obase = reinterpret_cast<const T*>(p.o) + (int64_t)b * p.o_sb + (int64_t)hd * p.o_sh;
  const T* gbase = reinterpret_cast<const T*>(p.d_o) + (int64_t)b * p.do_sb + (int64_t)hd * p.do_sh;

  Loader tiles;
  auto issue_tile = [&](int stage) {
    tiles.issue(smem + stage * STAGE, wave);
    tiles.advance();
  };
  tiles.init(kbase, p.k_st, vbase, p.v_st, kt0 * TT, L - 1, wave, lane);
  // this wave's Q and dO rows go where the third and the second tile will be
  using Rows = OwnRows<T, D>;
  static_assert(NW * Rows::ELEMS == STAGE, "the rows of a workgroup fill a stage");
  T* const q_area = smem + 2 * STAGE + wave * Rows::ELEMS;
  T* const g_area = smem + STAGE + wave * Rows::ELEMS;
  Rows::send(qbase, p.q_st, r0 + wave * 32, L - 1, q_area, lane);
  Rows::send(gbase, p.do_st, r0 + wave * 32, L - 1, g_area, lane);
  issue_tile(0);

  // ---- lse and delta of the query rows in reach, at their places in the tiles from qt0 on (rows beside them are masked) --
  const int d0 = qt0 * TT;
  {
    constexpr int LPR = D / 8, RPP = NT / LPR, U = 256 / RPP < 8 ? 256 / RPP : 8;   // lanes per row, rows per pass, passes in flight
    const int sub = tid % LPR, nd = q_hi(g_last) - d0;
    for (int base = 0; base < nd; base += RPP * U) {
      Frag of[U], gf[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = base + u * RPP + tid / LPR;
        const int64_t gr = d0 + (r < nd ? r : nd - 1);
        of[u] = *reinterpret_cast<const Frag*>(obase + gr * p.o_st + sub * 8);
        gf[u] = *reinterpret_cast<const Frag*>(gbase + gr * p.do_st + sub * 8);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = base + u * RPP + tid / LPR;
        float sum = dot_frag(of[u], gf[u], 0.0f);
#pragma unroll
        for (int off = LPR / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
        if (sub == 0 && r < nd) delta_s[r] = sum;
      }
    }
    for (int r = tid; r < nd; r += NT) lse_s[r] = p.lse[out_row + d0 + r];
  }

  Frag kf[NF], vf[NF];   // this wave's key rows, for the second half
  // ---- dQ -------------------------------------------------------------------------------------------------
  {
    const float sl2e = fabsf(p.scale_log2e);
    Frag qf[NF], gf[NF];
    landed();
#pragma unroll
    for (int g = 0; g < NF; ++g) {
      qf[g] = Rows::read(q_area, g, lane);
      if (p.scale_log2e < 0.0f) qf[g] = negate<T>(qf[g]);
      gf[g] = negate<T>(Rows::read(g_area, g, lane));
    }
    __syncthreads();   // lse_s, delta_s; the rows have been read
    if (kt0 + 1 < kt1) issue_tile(1);
    if (tid < ROWS && r0 + tid < T_) p.delta_out[out_row + r0 + tid] = r0 + tid < L ? delta_s[r0 + tid - d0] : 0.0f;
    const float lse_q = row < L ? lse_s[row - d0] : INFINITY;   // rows past L: P = exp2(-inf) = 0
    f32x16 dinit, acc[DB];
#pragma unroll
    for (int i = 0; i < 16; ++i) dinit[i] = delta_s[valid(row) - d0];
#pragma unroll
    for (int m = 0; m < DB; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;

    int st = 0;
    for (int t = kt0; t < kt1; ++t, st = st == NST - 1 ? 0 : st + 1) {
      if (t + 1 < kt1) wait_loads<LPT>();
      else wait_loads<0>();
      __syncthreads();   // tile t is in LDS and tile t - 1 has no reader left
      if (t + 2 < kt1) issue_tile(st == 0 ? 2 : st - 1);
      const T* Kt = smem + st * STAGE;
      if (!wq.seen(t * TT, TT)) continue;
      dq2_tile<T, D, TT>(acc, Kt, Kt + TILE, t * TT, wq, qf, gf, sl2e, lse_q, dinit, lane);
    }
    // the last three key tiles are still in LDS: as a rule the workgroup's own rows are among them
    if (kt1 * TT <= r0 + NST * TT) {
      const int own = (r0 + wave * 32) / TT;                       // this wave's tile, from one to three back
      const int back = kt1 - own;
      int s2 = st - back;                                           // st is one past the last tile's stage
      s2 = s2 < 0 ? s2 + NST : s2;
      if (wave_live) {
        const T* Kt = smem + s2 * STAGE + wave * 32 % TT * D;
#pragma unroll
        for (int g = 0; g < NF; ++g) {
          kf[g] = *reinterpret_cast<const Frag*>(Kt + G::off(c, (g * 2 + h) * E::VEC));
          vf[g] = *reinterpret_cast<const Frag*>(Kt + TILE + G::off(c, (g * 2 + h) * E::VEC));
        }
      }
    } else {
      const T* kp = kbase + (int64_t)valid(row) * p.k_st;
      const T* vp = vbase + (int64_t)valid(row) * p.v_st;
#pragma unroll
      for (int g = 0; g < NF; ++g) {
        kf[g] = *reinterpret_cast<const Frag*>(kp + (g * 2 + h) * E::VEC);
        vf[g] = *reinterpret_cast<const Frag*>(vp + (g * 2 + h) * E::VEC);
      }
    }
    __syncthreads();   // no wave reads a stage any more: the first query tiles go to stages 0 and 1, the row patches over stage 2
    tiles.init(qbase, p.q_st, gbase, p.do_st, qt0 * TT, L - 1, wave, lane);
    issue_tile(0);
    if (qt0 + 1 < qt1) issue_tile(1);
    if (row >= L) {
#pragma unroll
      for (int m = 0; m < DB; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
    }
    const int row0 = r0 + wave * 32;
    store_rows_coalesced<T, D, DB>(smem + 2 * STAGE + wave * RowPatch<T, D>::ELEMS, dq_base + (int64_t)row0 * D, T_ - row0,
                                   acc, -p.scale, lane);
  }

  // ---- dK, dV ---------------------------------------------------------------------------------------------
#pragma unroll
  for (int g = 0; g < NF; ++g) {
    kf[g] = dkdv2_keys<T, D>(kf[g], p.scale_log2e);
    vf[g] = negate<T>(vf[g]);
  }
  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int m = 0; m < DB; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[m][i] = 0.0f, dv[m][i] = 0.0f;

  int st = 0;
  for (int t = qt0; t < qt1; ++t, st = st == NST - 1 ? 0 : st + 1) {
    if (t + 1 < qt1) wait_loads<LPT>();
    else wait_loads<0>();
    __syncthreads();
    if (t + 2 < qt1) issue_tile(st == 0 ? 2 : st - 1);
    const T* Qt = smem + st * STAGE;
    if (!wk.seen(t * TT, TT)) continue;
    const float* l = lse_s + (t - qt0) * TT;
    const float* d = delta_s + (t - qt0) * TT;
    dkdv2_tile<T, D, TT, PG>(dk, dv, Qt, Qt + TILE, t * TT, wk, kf, vf, p.scale_log2e, [&](int r, f32x4& l4, f32x4& d4) {
      l4 = *reinterpret_cast<const f32x4*>(l + r);
      d4 = *reinterpret_cast<const f32x4*>(d + r);
    }, lane);
  }

  if (row >= L) {
#pragma unroll
    for (int m = 0; m < DB; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i) dk[m][i] = 0.0f, dv[m][i] = 0.0f;
  }
  __syncthreads();   // the row patches lie over the stages
  {
    T* patch = smem + wave * RowPatch<T, D>::ELEMS;
    const int row0 = r0 + wave * 32;
    store_rows_coalesced<T, D, DB>(patch, dk_base + (int64_t)row0 * D, T_ - row0, dk, -p.scale, lane);
    store_rows_coalesced<T, D, DB>(patch, dv_base + (int64_t)row0 * D, T_ - row0, dv, 1.0f, lane);
  }
}

}  // namespace sa
