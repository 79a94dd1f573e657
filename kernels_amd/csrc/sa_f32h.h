// float32 kernels on the 16-bit matrix pipe with two float16 parts per number: head dimension 128, and the wide windows of 32 and
// 64 (in_halves in sa_inst.hip; the others have three bfloat16 parts, sa_f32.h).
//
// A row is multiplied by a power of two that brings its largest element to the top of float16's range, [2^14, 2^15).  An element is then
// the sum of a float16 number and the rounded remainder: 11 + 11 significand bits and the remainder's sign, 2^-24 of the element, or 2^-39
// of the row's largest where the remainder reaches the bottom of the range.  A product is
//   x*y = x1*y1 + (x1*y2 + x2*y1) + [x2*y2],
// of which the bracket, at most 2^-24 of |x*y|, is left out: three products instead of six, every one formed exactly and added up in
// float32.  Errors of O, dQ, dK, dV and the LSE against float64 are below those of three bfloat16 parts, as the sums have half the
// roundings (B=2, H=2, T=1000, D=128, chunks of 128, 4 back 3.97, 5.03, 6.04, 5.93e-7, 4.4e-8 -> 3.12, 3.96, 4.66, 4.43e-7, 3.0e-8;
// D=64, B=2, H=4, T=512, chunks of 64, 2 back 2.65, 3.74, 3.97, 3.81e-7 -> 2.33, 3.16, 3.28, 3.05e-7); with rows of V and dO spread over 2^24 in
// size too, row by row.
//
// The powers of two come off again where a result is scaled anyway.  In a product over D they are factors of the result's row and
// column (the streamed row's is kept in LDS beside the tile).  In a product over keys or queries the streamed row's factor goes into
// the probability or dS that it meets, and that column of the resident operand is brought into range by a unit of its own (OwnUnit),
// set from the values themselves: a row that a query does not see, or that has no weight for it, costs the others no bits.
//
// What float32 arithmetic represents and this does not (infinities, units beyond 2^+-100, rows of dO and V from 2^59 on, whose dP may
// leave the range of float32 where float32 arithmetic keeps it) goes through its rows again with the float32 instruction, by the
// workgroup, as in sa_f32.h.
#pragma once
#include "sa_f32.h"

namespace sa {

// Magnitudes of several lanes are compared as whole numbers, the bits of a float without a sign.
SA_DEV uint32_t larger(uint32_t a, uint32_t b) { return a > b ? a : b; }
// The largest over groups of N neighbouring lanes (4, 8 or 16), left in all of them.
template <int N> SA_DEV uint32_t lanes_max(uint32_t x) {
  auto step = [](uint32_t a, auto ctrl) {
    return larger(a, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)a, decltype(ctrl)::value, 0xf, 0xf, true));
  };
  x = step(x, std::integral_constant<int, 0xB1>());                          // lane ^ 1
  x = step(x, std::integral_constant<int, 0x4E>());                          // lane ^ 2
  if constexpr (N >= 8) x = step(x, std::integral_constant<int, 0x141>());   // the other four of eight
  if constexpr (N >= 16) x = step(x, std::integral_constant<int, 0x140>());  // the other eight of sixteen
  return x;
}
SA_DEV uint32_t halves_max(uint32_t x) {
  auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return larger(r[0], r[1]);
}
SA_DEV float abs_max3(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}
// m and the magnitudes of four elements, the largest that is a number: NaN keeps its place in the parts, whatever the factor
SA_DEV float abs_max4(float m, const f32x4& x) { return abs_max3(abs_max3(m, x[0], x[1]), x[2], x[3]); }
// Powers of two for a row whose largest magnitude is m: times `to` it is in [2^14, 2^15) (less below 2^-112), from = 1 / to.
struct RowScale {
  float to = 0.0f, from = 0.0f;
  SA_DEV RowScale() {}
  SA_DEV explicit RowScale(uint32_t m) {
    const uint32_t e = m == 0 ? 127u << 23 : larger(m & 0x7F800000u, 15u << 23);
    to = __uint_as_float((268u << 23) - e);
    from = __uint_as_float(e - (14u << 23));
  }
};

// Two float16 fragments that add up to eight scaled values.
struct Half8 {
  f16x8 p[2];
};
// Elements 2*e and 2*e+1 of a fragment, x0 and x1 times powers of two.
SA_DEV void halve_pair(Half8& s, int e, float x0, float f0, float x1, float f1) {
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  f16x2 hi = {(_Float16)(x0 * f0), (_Float16)(x1 * f1)};
  uint32_t h = __builtin_bit_cast(uint32_t, hi);
  asm("" : "+v"(h));   // the packed conversion's result is what is subtracted: one instruction per remainder
  hi = __builtin_bit_cast(f16x2, h);
  const f16x2 lo = {(_Float16)__builtin_fmaf(x0, f0, -(float)hi[0]), (_Float16)__builtin_fmaf(x1, f1, -(float)hi[1])};
  u32x4 w = __builtin_bit_cast(u32x4, s.p[0]);
  w[e] = h;
  s.p[0] = __builtin_bit_cast(f16x8, w);
  w = __builtin_bit_cast(u32x4, s.p[1]);
  w[e] = __builtin_bit_cast(uint32_t, lo);
  s.p[1] = __builtin_bit_cast(f16x8, w);
}
SA_DEV void mma3(f32x16& acc, const Half8& a, const Half8& b) {
  mma(acc, a.p[1], b.p[0]);
  mma(acc, a.p[0], b.p[1]);
  mma(acc, a.p[0], b.p[0]);
}

template <int D> struct HalfTile {
  using G = TileGeom<_Float16, D>;
  static constexpr int PLANE = 32 * G::PITCH;   // elements
  static constexpr int ELEMS = 2 * PLANE;
};

// Copy of a [32][D] float32 tile through registers into a HalfTile and its rows' factors, eight elements per thread and step.
// Rows are clamped to last_row (the values are masked by the caller).
template <int D, int NT> struct HalfStager {
  using G = TileGeom<_Float16, D>;
  static constexpr int CPR = D / 8, TOTAL = 32 * CPR, N = (TOTAL + NT - 1) / NT;
  static_assert(TOTAL % NT == 0 || N == 1, "whole steps, or one for some of the threads");
  f32x4 regs[N][2];

  SA_DEV void load(const float* base, int64_t row_stride, int row0, int last_row, int tid) {
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const int ch = tid + it * NT;
      int gr = row0 + ch / CPR;   // (threads beyond the tile load rows of the next one)
      gr = gr < last_row ? gr : last_row;
      const float* src = base + (int64_t)gr * row_stride + (ch % CPR) * 8;
      regs[it][0] = *reinterpret_cast<const f32x4*>(src);
      regs[it][1] = *reinterpret_cast<const f32x4*>(src + 4);
    }
  }
  // the work of store() in STEPS pieces
  static constexpr int STEPS = 6 * N;
  RowScale scale;
  Half8 parts;
  float most = 0.0f;   // largest factor that this thread has stored
  SA_DEV void step(int x, _Float16* tile, float* factors, int tid, float mul = 1.0f) {   // mul: of the factors
    const int it = x / 6, e = x % 6 - 1;
    if (e < 0) {
      scale = RowScale(lanes_max<CPR>(__float_as_uint(abs_max4(abs_max4(0.0f, regs[it][0]), regs[it][1]))));
      most = fast_max(most, scale.from);
    } else if (e < 4) {
      halve_pair(parts, e, regs[it][e / 2][2 * (e % 2)], scale.to, regs[it][e / 2][2 * (e % 2) + 1], scale.to);
    } else {
      const int ch = tid + it * NT;
      if (TOTAL % NT != 0 && ch >= TOTAL) return;
      _Float16* dst = tile + G::off(ch / CPR, (ch % CPR) * 8);
      *reinterpret_cast<f16x8*>(dst) = parts.p[0];
      *reinterpret_cast<f16x8*>(dst + HalfTile<D>::PLANE) = parts.p[1];
      if (ch % CPR == 0) factors[ch / CPR] = scale.from * mul;
    }
  }
  SA_DEV void store(_Float16* tile, float* factors, int tid, float mul = 1.0f) {
#pragma unroll
    for (int x = 0; x < STEPS; ++x) step(x, tile, factors, tid, mul);
  }
};

// The parts of this lane's half of a row.
template <int D> SA_DEV RowScale halve_row(Half8 (&f)[D / 16], const HalfRow<D>& row) {
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < D / 8; ++i) m = abs_max4(m, row.r[i]);
  const RowScale sc(halves_max(__float_as_uint(m)));
#pragma unroll
  for (int g = 0; g < D / 16; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      halve_pair(f[g], e, row.r[2 * g + e / 2][2 * (e % 2)], sc.to, row.r[2 * g + e / 2][2 * (e % 2) + 1], sc.to);
  return sc;
}

// The factors of the rows that a lane's registers of a C fragment stand for.
SA_DEV void row_factors(float (&f)[16], const float* factors, int h) {
#pragma unroll
  for (int g4 = 0; g4 < 4; ++g4) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(factors + 8 * g4 + 4 * h);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * g4 + e] = v[e];
  }
}

// Keeps fragments that every step multiplies in accumulation registers, where the matrix instruction reads them.  Left alone the
// compiler copies those that it has put there back for every use: 127 copies among the 960 instructions of a dQ step at D=128, 430 of
// 1500 in dK/dV.  Counted over the 4k case below, with the masks by bits alone and the factors by v_max3: vector instructions of dQ
// 108 -> 86 million, of dK/dV 182 -> 133, cycles 269 -> 257 and 393 -> 339; the clock follows the power, so the times less (two kernels
// 1220 -> 1125 us).  Not where two waves share the registers of a SIMD (forward in eight waves: 80 registers spilled instead of 29).
template <int N> SA_DEV void keep_in_agprs(Half8 (&f)[N]) {
#pragma unroll
  for (int g = 0; g < N; ++g) asm("" : "+a"(f[g].p[0]), "+a"(f[g].p[1]));
}

// acc[row r][col c] += sum_k tile[r][k] * B[k][c] for the 32 rows of a tile; side(g) is vector work placed behind step g.
template <int D, typename Side = NoSide>
SA_DEV void mma_rows_half(f32x16& acc, const _Float16* tile, const Half8 (&b)[D / 16], int lane, Side&& side = Side()) {
  using G = TileGeom<_Float16, D>;
  const int c = lane & 31, h = lane >> 5;
  const _Float16* base = tile + c * G::PITCH;
  const int sw = G::swz(c);
  pipeline<D / 16, 2>(
      [&](int g) {
        Half8 a;
#pragma unroll
        for (int k = 0; k < 2; ++k)
          a.p[k] = *reinterpret_cast<const f16x8*>(base + k * HalfTile<D>::PLANE + (((g * 2 + h) ^ sw) * 8));
        return a;
      },
      [&](int g, const Half8& a) { mma3(acc, a, b[g]); side(g); });
}

// acc[m] += X^T * P for the 32 rows of a tile, P given by its parts (rows 0 to 15 in b[0], the others in b[1]).
template <int D, int NM, typename Side = NoSide>
SA_DEV void mma_tr_half(f32x16 (&acc)[NM], const _Float16* X, const Half8 (&b)[2], int lane, Side&& side = Side()) {
  using G = TileGeom<_Float16, D>;
  static_assert(NM == G::DB, "one accumulator per 32-wide block of the head dimension");
  const int g16 = lane >> 4, j = lane & 15;
  const int r_lo = 4 * (g16 >> 1) + (j >> 2);
  const int col = (g16 & 1) * 16 + 4 * (j & 3);
  pipeline<2 * NM, 2>(
      [&](int it) {
        const int half = it / NM, m = it % NM;
        Half8 a;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const _Float16* p0 = X + k * HalfTile<D>::PLANE + G::off(half * 16 + r_lo, m * 32 + col);
          const _Float16* p1 = X + k * HalfTile<D>::PLANE + G::off(half * 16 + 8 + r_lo, m * 32 + col);
          s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((SA_LDS s16x4*)(p0));
          s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((SA_LDS s16x4*)(p1));
          a.p[k] = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
        return a;
      },
      [&](int it, const Half8& a) { mma3(acc[it % NM], a, b[it / NM]); side(it); });
}

// 1 / x for a power of two that has a normal reciprocal
SA_DEV float power_inverse(float x) { return __uint_as_float((254u << 23) - __float_as_uint(x)); }

// The power of two that a lane's column of P or dS, times the factors of its rows, is brought into float16's range with; the
// accumulators are in units of it.  It is set from the first values that are not zero, with 2^8 to spare (set to the top of the range
// it moved in every few tiles, which cost the kernels 10 to 20 %), and moves when larger ones leave the range.  Parts reach down to 2^-25:
// 2^-31 of the largest value or less.
struct OwnUnit {
  float up = 0.0f;             // 0: none yet
  bool out_of_range = false;   // it would have to be no normal number
  // the parts of x0 * f0 * up and x1 * f1 * up, elements i and i + 1 of the column; most: largest magnitude so far
  SA_DEV void pair(Half8 (&b)[2], int i, float x0, float f0, float x1, float f1, float& most) const {
    const float y0 = x0 * f0 * up, y1 = x1 * f1 * up;
    most = abs_max3(most, y0, y1);
    halve_pair(b[i / 8], (i % 8) / 2, y0, 1.0f, y1, 1.0f);
  }
  // whether some lane has to move for the values x, of which the largest came to most
  SA_DEV bool leaves(const f32x16& x, float most) const {
    uint64_t leave = __builtin_amdgcn_ballot_w64(most > 0x1p15f);
    if (__builtin_amdgcn_ballot_w64(up == 0.0f) != 0) {
      most = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; i += 2) most = abs_max3(most, x[i], x[i + 1]);
      leave |= __builtin_amdgcn_ballot_w64(up == 0.0f && most > 0.0f);
    }
    return leave != 0;
  }
  SA_DEV bool halve(Half8 (&b)[2], const f32x16& x, const float (&f)[16]) const {
    float most = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i += 2) pair(b, i, x[i], f[i], x[i + 1], f[i + 1], most);
    return leaves(x, most);
  }
  SA_DEV float move(const f32x16& x, const float (&f)[16]) {
    float most = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i += 2) most = abs_max3(most, x[i] * f[i], x[i + 1] * f[i + 1]);
    most = half_max(most);
    if (most == 0.0f) return 1.0f;
    out_of_range = out_of_range || !(most >= 0x1p-100f && most <= 0x1p100f);
    const float to = __builtin_amdgcn_ldexpf(1.0f, 7 - __builtin_amdgcn_frexp_expf(most));   // the largest is then below 2^7
    if (up != 0.0f && !(to < up)) return 1.0f;   // the lane is in range
    const float by = up == 0.0f ? 1.0f : to * power_inverse(up);
    up = to;
    return by;
  }
  SA_DEV float value() const { return up == 0.0f ? 0.0f : power_inverse(up); }
  // The accumulators in units of their own; whether they, times mul, are finite and no value was out of range.
  template <int D, int NM> SA_DEV bool settle(f32x16 (&acc)[NM], float mul) const {
    const float to = value();
    float z = 0.0f;   // becomes NaN
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        acc[m][i] *= to;
        z = __builtin_fmaf(acc[m][i] * mul, 0.0f, z);
      }
    return z == 0.0f && !out_of_range;
  }
};
// Forward.  One wave per 32 queries, tiles of 32 keys in two stages.  Bound by the vector work that forms parts (P's, and the streamed
// tiles': eleven instructions per two elements) beside a matrix pipe that is 40 % busy: of the two waves on a SIMD one stages before its
// products and the other one after them, so that one's products meet the other's vector work (in step they cost 10 % more at D=128).
// B=4, H=16, T=4096, chunks of 128, 4 back, us from three bfloat16 parts -> here: D=128 428 -> 312, D=64 218 -> 186, D=32 131 -> 121; one chunk of 1500,
// B=4, H=8, D=128 197 -> 116.  Products of one tile among the vector work of the next in one wave: D=128 500 and more, D=64 204.
template <int D, int NW>
__global__ __launch_bounds__(NW * 64, (D == 128 && NW == 4 ? 1 : 2)) void fwd_halves_kernel(const FwdParams p) {
  constexpr int TQ = NW * 32, NT = NW * 64, TK = 32, DB = TileGeom<_Float16, D>::DB;
  constexpr int TILE = HalfTile<D>::ELEMS;
  constexpr float kRescaleGap = 8.0f;
  constexpr float kSumLimit = 256.0f;

  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  _Float16* smem = reinterpret_cast<_Float16*>(smem_raw);   // [stage][K|V][part][TK][PITCH], then [stage][K|V][TK] factors
  float* const factors = reinterpret_cast<float*>(smem + 4 * TILE);

  const int tid = threadIdx.x;
  const int lane = tid & 63, c = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int bh, qt, L = p.T;
  if (p.by_length) tile_coords_by_length<TQ>(blockIdx.x, p.tiles, p.by_length, p.lens, p.lens_stride, p.T, p.H, lane, bh, qt, L);
  else tile_coords(blockIdx.x, gridDim.x, p.tiles, bh, qt);
  const int T_ = p.T;
  const int b = div_by(bh, p.tiles.by_heads), hd = bh - b * p.H;
  if (p.lens && !p.by_length) {
    L = p.lens[(int64_t)b * p.lens_stride];
    L = L < 0 ? 0 : (L > T_ ? T_ : L);
  }
  const int q0 = qt * TQ;
  float* o_base = reinterpret_cast<float*>(p.o) + (int64_t)bh * T_ * D;
  float* lse_base = p.lse ? p.lse + (int64_t)bh * T_ : nullptr;
  const int q_end = q0 + TQ < T_ ? q0 + TQ : T_;
  if (q0 >= L) {
    zero_rows<float, D, NT>(o_base, q0, q_end, tid);
    if (lse_base)
      for (int r = q0 + tid; r < q_end; r += NT) lse_base[r] = 0.0f;
    return;
  }

  const int qrow = q0 + wave * 32 + c;
  const QueryWindow w(q0, wave, TQ, qrow, L, p.C, p.R, p.cdiv);
  const int kt0 = w.lo_wg / TK, kt1 = (w.hi_wg + TK - 1) / TK;

  const float* kbase = reinterpret_cast<const float*>(p.k) + (int64_t)b * p.k_sb + (int64_t)hd * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.v) + (int64_t)b * p.v_sb + (int64_t)hd * p.v_sh;
  float* const q_area = reinterpret_cast<float*>(smem_raw) + wave * OwnRows32<D>::ELEMS;
  const float* qbase = reinterpret_cast<const float*>(p.q) + (int64_t)b * p.q_sb + (int64_t)hd * p.q_sh;
  constexpr bool DIRECT = direct_rows(D, NW);
  if (!DIRECT) OwnRows32<D>::send(qbase, p.q_st, q0 + wave * 32, L - 1, q_area, lane);
  const TileOrder order(kt0, kt1, p.period, p.pdiv);
  HalfStager<D, NT> sk, sv;
  auto load_tile = [&](int t) {
    sk.load(kbase, p.k_st, t * TK, L - 1, tid);
    sv.load(vbase, p.v_st, t * TK, L - 1, tid);
  };
  auto store_tile = [&](int st) {
    sk.store(smem + st * 2 * TILE, factors + st * 2 * TK, tid);
    sv.store(smem + st * 2 * TILE + TILE, factors + st * 2 * TK + TK, tid);
  };
  load_tile(order.first);

  Half8 qf[D / 16];
  float cq;   // times a key's factor: score to base-2 exponent
  {
    HalfRow<D> qr;
    if (DIRECT) {
      qr.load(qbase + (int64_t)(qrow < L ? qrow : L - 1) * p.q_st, h);
    } else {
      landed();
      qr.read(q_area, lane);
    }
    cq = halve_row<D>(qf, qr).from * p.scale_log2e;
  }
  if (!DIRECT) __syncthreads();   // the tiles go where the rows were

  f32x16 oacc[DB];
#pragma unroll
  for (int m = 0; m < DB; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[m][i] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;
  OwnUnit unit;   // of the accumulators

  store_tile(0);
  // Of two waves on a SIMD one brings the next tile's parts into LDS before its products, the other one after them.
  const bool early = wave >= 4;
  if (early && order.next(order.first) != order.first) load_tile(order.next(order.first));
  __syncthreads();

  for (int t = order.first, it = 0; it < kt1 - kt0; ++it, t = order.next(t)) {
    if constexpr (D == 128 && NW == 4) keep_in_agprs(qf);
    const _Float16* Kt = smem + (it & 1) * 2 * TILE;
    const _Float16* Vt = Kt + TILE;
    const float* kv = factors + (it & 1) * 2 * TK;
    const bool more = order.next(t) != order.first;
    if (more && early) {
      store_tile(~it & 1);
      const int then = order.next(order.next(t));
      if (then != order.first) load_tile(then);
    } else if (more) {
      load_tile(order.next(t));
    }
    const int k0 = t * TK;
    if (k0 + TK > w.lo_min && k0 < w.hi_max) {   // some query of this wave sees the tile
      f32x16 s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.0f;
      mma_rows_half<D>(s, Kt, qf, lane);
      float f[16];
      row_factors(f, kv, h);
#pragma unroll
      for (int i = 0; i < 16; ++i) f[i] *= cq;
      const bool interior = k0 >= w.lo_max && k0 + TK <= w.hi_min;
      const uint32_t rm = interior ? ~0u : row_mask(w.lo - k0, w.hi - k0, h);
      // as in fwd_split_kernel, but masked probabilities are cleared, whatever the score was: no score is kept beside its factor
      f32x16 pr;
      float rs0, rs1;
      auto probabilities = [&](float m_use) {
        rs0 = rs1 = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) pr[i] = fast_exp2(__builtin_fmaf(s[i], f[i], -m_use));
        if (!interior) {
#pragma unroll
          for (int i = 0; i < 16; ++i) pr[i] = keep_or_zero(pr[i], keep_bits(rm, i));
        }
#pragma unroll
        for (int i = 0; i < 16; i += 2) rs0 += pr[i], rs1 += pr[i + 1];
      };
      probabilities(m_run == -INFINITY ? 0.0f : m_run);
      const bool behind = !(rs0 + rs1 <= kSumLimit) || m_run == -INFINITY;   // true for NaN too
      if (__builtin_amdgcn_ballot_w64(behind) != 0) {
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fast_max(mx, keep_or_neg_inf(s[i] * f[i], keep_bits(rm, i)));
        mx = half_max(mx);
        const bool move = mx > m_run + kRescaleGap;   // false for mx = -inf or NaN
        if (__builtin_amdgcn_ballot_w64(move) != 0) {
          const float alpha = move ? fast_exp2(m_run - mx) : 1.0f;
          m_run = move ? mx : m_run;
          l_run *= alpha;
#pragma unroll
          for (int m = 0; m < DB; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) oacc[m][i] *= alpha;
          probabilities(m_run == -INFINITY ? 0.0f : m_run);
        }
      }
      l_run += rs0 + rs1;
      row_factors(f, kv + TK, h);
      Half8 pb[2];
      if (unit.halve(pb, pr, f)) {
        const float by = unit.move(pr, f);
#pragma unroll
        for (int m = 0; m < DB; ++m)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[m][i] *= by;
        unit.halve(pb, pr, f);
      }
      mma_tr_half<D>(oacc, Vt, pb, lane);   // O^T[d][q] += V^T P^T
    }
    if (more && !early) store_tile(~it & 1);
    __syncthreads();
  }

  const float l_tot = half_sum(l_run);
  const bool odd = q0 + wave * 32 < L && (!(l_tot > 0.0f) || !all_finite<D>(oacc) || unit.out_of_range || scale_too_small(p.scale_log2e));
  if (any_in_workgroup<NW>(odd, smem_raw, wave, lane)) {
    fwd_rows<float, D, NW, TK>(p, again_s(bh), again_s(qt), again_v(tid));
    return;
  }
  const bool valid = qrow < L;
  const float inv = 1.0f / l_tot;
#pragma unroll
  for (int m = 0; m < DB; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[m][i] = valid ? oacc[m][i] * inv : 0.0f;   // the unit last: both together may leave the range
  const int row0 = q0 + wave * 32;
  store_rows_f32<D, DIRECT>(row_patch<D>(smem_raw, wave), o_base + (int64_t)row0 * D, T_ - row0, oacc, unit.value(), lane);
  if (lse_base && h == 0 && qrow < T_) {
    // the logarithm of the significand: that of the whole number has the error of a larger one
    const float lg = __builtin_amdgcn_logf(__builtin_amdgcn_frexp_mantf(l_tot));
    const float e = (float)__builtin_amdgcn_frexp_expf(l_tot), whole = m_run + e, moved = whole - m_run;
    const float rest = (m_run - (whole - moved)) + (e - moved);   // what the sum was rounded by: the LSE is rounded once
    lse_base[qrow] = valid ? whole + (lg + rest) : 0.0f;
  }
}

// Rows of dO and of V that reach 2^59: their dP may leave the range of float32 where float32 arithmetic leaves it, but not here.
SA_DEV bool too_large(float factor) { return factor >= 0x1p45f; }

// dQ, one wave per 32 queries, tiles of 32 keys, two stages, delta as in dq_split_kernel.  The next tile's parts are formed behind the
// products of S and the exponentials behind those of dP.  Same problem as above, dQ and dK/dV together, us: D=128 1562 -> 1125 (traced
// alone 713 -> 563; one wave per SIMD, whose vector work is what is left between products), D=64 812 -> 590, D=32 430 -> 350.
// Tried at D=128: dS formed behind the products of the next tile and dQ added a step later, from three stages: 257 -> 277 million cycles;
// the loads of the next tile right behind its predecessor's parts instead of at the end of a step: 257 -> 269.
template <int D, int NW>
__global__ __launch_bounds__(NW * 64, (D <= 64 ? 2 : 1)) void dq_halves_kernel(const BwdParams p) {
  constexpr int TQ = NW * 32, NT = NW * 64, TK = 32, NF = D / 16, DB = TileGeom<_Float16, D>::DB;
  constexpr int TILE = HalfTile<D>::ELEMS;

  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  _Float16* smem = reinterpret_cast<_Float16*>(smem_raw);   // [stage][K|V][part][TK][PITCH], then [stage][K|V][TK] factors
  float* const factors = reinterpret_cast<float*>(smem + 4 * TILE);

  const int tid = threadIdx.x;
  const int lane = tid & 63, c = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int bh, qt;
  tile_coords(blockIdx.x, gridDim.x, p.tiles, bh, qt);
  const int b = div_by(bh, p.tiles.by_heads), hd = bh - b * p.H;
  const int T_ = p.T;
  int L = T_;
  if (p.lens) {
    L = p.lens[(int64_t)b * p.lens_stride];
    L = L < 0 ? 0 : (L > T_ ? T_ : L);
  }
  const int q0 = qt * TQ;
  float* dq_base = reinterpret_cast<float*>(p.dq) + (int64_t)bh * T_ * D;
  const int q_end = q0 + TQ < T_ ? q0 + TQ : T_;
  if (q0 >= L) {
    zero_rows<float, D, NT>(dq_base, q0, q_end, tid);
    if (p.delta_out)
      for (int r = q0 + tid; r < q_end; r += NT) p.delta_out[(int64_t)bh * T_ + r] = 0.0f;
    return;
  }

  const int qrow = q0 + wave * 32 + c;
  const QueryWindow w(q0, wave, TQ, qrow, L, p.C, p.R, p.cdiv);
  const int kt0 = w.lo_wg / TK, kt1 = (w.hi_wg + TK - 1) / TK;

  const float* kbase = reinterpret_cast<const float*>(p.k) + (int64_t)b * p.k_sb + (int64_t)hd * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.v) + (int64_t)b * p.v_sb + (int64_t)hd * p.v_sh;
  using Rows = OwnRows32<D>;
  const int row0 = q0 + wave * 32;
  float* const q_area = reinterpret_cast<float*>(smem_raw) + wave * Rows::ELEMS;
  float* const g_area = q_area + NW * Rows::ELEMS;
  const float* gbase = reinterpret_cast<const float*>(p.d_o) + (int64_t)b * p.do_sb + (int64_t)hd * p.do_sh;
  const float* qbase = reinterpret_cast<const float*>(p.q) + (int64_t)b * p.q_sb + (int64_t)hd * p.q_sh;
  // (no branch around the loads: without a row of O to read, the dO row is read; see dq2_kernel)
  const float* obase = p.delta_out ? reinterpret_cast<const float*>(p.o) + (int64_t)b * p.o_sb + (int64_t)hd * p.o_sh : gbase;
  const int64_t o_st = p.delta_out ? p.o_st : p.do_st;
  constexpr bool DIRECT = direct_rows(D, NW);
  RowDots32<D> dots;
  if (!DIRECT) {
    Rows::send(qbase, p.q_st, row0, L - 1, q_area, lane);
    Rows::send(gbase, p.do_st, row0, L - 1, g_area, lane);
    dots.load(obase, o_st, row0, L - 1, lane);
  }
  const TileOrder order(kt0, kt1, p.period, p.pdiv);
  HalfStager<D, NT> sk, sv;
  auto load_tile = [&](int t) {
    sk.load(kbase, p.k_st, t * TK, L - 1, tid);
    sv.load(vbase, p.v_st, t * TK, L - 1, tid);
  };
  load_tile(order.first);

  Half8 qf[NF], gf[NF];
  float cq;       // times a key's factor: score to base-2 exponent
  RowScale g_scale;
  const int qr = qrow < L ? qrow : L - 1;
  const float lse_q = qrow < L ? p.lse[(int64_t)bh * T_ + qr] : INFINITY;   // rows past L: P = exp2(-inf) = 0
  float delta_q;
  {
    float sum;
    HalfRow<D> q_row, g_row;
    if (DIRECT) {
      HalfRow<D> o_row;
      q_row.load(qbase + (int64_t)qr * p.q_st, h);
      g_row.load(gbase + (int64_t)qr * p.do_st, h);
      o_row.load(obase + (int64_t)qr * o_st, h);
      sum = o_row.dot_half_row(g_row);
    } else {
      landed();
      g_row.read(g_area, lane);
      q_row.read(q_area, lane);
      dots.partial(g_area, q_area, lane);
      sum = RowDots32<D>::total(q_area, lane);
    }
    g_scale = halve_row<D>(gf, g_row);
    cq = halve_row<D>(qf, q_row).from * p.scale_log2e;
    if (p.delta_out) {
      delta_q = sum;
      if (h == 0 && qrow < T_) p.delta_out[(int64_t)bh * T_ + qrow] = qrow < L ? delta_q : 0.0f;
    } else {
      delta_q = p.delta[(int64_t)bh * T_ + qr];
    }
  }
  if (!DIRECT) __syncthreads();   // the tiles go where the rows were

  // dP and delta in units of 2^14 times the dO row's factor, whose parts reach up to 2^15
  constexpr float kUnit = 0x1p14f, kToUnit = 0x1p-14f;
  const float delta_u = delta_q * g_scale.to * kToUnit;

  f32x16 acc[DB];
#pragma unroll
  for (int m = 0; m < DB; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
  OwnUnit unit;   // of the accumulators
  sk.store(smem, factors, tid);
  sv.store(smem + TILE, factors + TK, tid, kToUnit);
  if (order.next(order.first) != order.first) load_tile(order.next(order.first));
  __syncthreads();

  for (int t = order.first, it = 0; it < kt1 - kt0; ++it, t = order.next(t)) {
    if constexpr (D == 128) {
      keep_in_agprs(qf);
      keep_in_agprs(gf);
    }
    const _Float16* Kt = smem + (it & 1) * 2 * TILE;
    const _Float16* Vt = Kt + TILE;
    const float* kv = factors + (it & 1) * 2 * TK;
    const bool more = order.next(t) != order.first;
    _Float16* const next_tile = smem + (~it & 1) * 2 * TILE;
    float* const next_factors = factors + (~it & 1) * 2 * TK;
    auto stage = [&](int x) {
      constexpr int S = HalfStager<D, NT>::STEPS;
      if (x < S) sk.step(x, next_tile, next_factors, tid);
      else sv.step(x - S, next_tile + TILE, next_factors + TK, tid, kToUnit);
    };
    constexpr int WORK = 2 * HalfStager<D, NT>::STEPS;
    const int k0 = t * TK;
    if (k0 + TK > w.lo_min && k0 < w.hi_max) {
      f32x16 s, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.0f, dp[i] = 0.0f;
      // (the next tile's parts are formed whether there is one or not: no branch between the products)
      mma_rows_half<D>(s, Kt, qf, lane, [&](int g) {
#pragma unroll
        for (int x = g * WORK / NF; x < (g + 1) * WORK / NF; ++x) stage(x);
      });
      float fk[16], fv[16];
      row_factors(fk, kv, h);
      row_factors(fv, kv + TK, h);
      mma_rows_half<D>(dp, Vt, gf, lane, [&](int g) {
#pragma unroll
        for (int i = g * 16 / NF; i < (g + 1) * 16 / NF; ++i) s[i] = fast_exp2(__builtin_fmaf(s[i], fk[i] * cq, -lse_q));
      });
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] *= __builtin_fmaf(dp[i], fv[i], -delta_u);   // dS
      if (!(k0 >= w.lo_max && k0 + TK <= w.hi_min)) {
        const uint32_t rm = row_mask(w.lo - k0, w.hi - k0, h);
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = keep_or_zero(s[i], keep_bits(rm, i));
      }
      Half8 sb[2];
      if (unit.halve(sb, s, fk)) {
        const float by = unit.move(s, fk);
#pragma unroll
        for (int m = 0; m < DB; ++m)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[m][i] *= by;
        unit.halve(sb, s, fk);
      }
      mma_tr_half<D>(acc, Kt, sb, lane);   // dQ^T[d][q] += K^T dS^T
    } else {
#pragma unroll
      for (int x = 0; x < WORK; ++x) stage(x);
    }
    if (more) {
      const int then = order.next(order.next(t));
      if (then != order.first) load_tile(then);
    }
    __syncthreads();
  }

  const float mul = g_scale.from * kUnit * p.scale;
  const bool odd = !unit.settle<D>(acc, mul) || too_large(g_scale.from) || too_large(sv.most) || scale_too_small(p.scale_log2e);
  if (any_in_workgroup<NW>(odd, smem_raw, wave, lane)) {
    dq_rows<float, D, NW, TK>(p, again_s(bh), again_s(qt), again_v(tid), [&](int) { return delta_q; });   // this lane's query
    return;
  }
  if (qrow >= L) {
#pragma unroll
    for (int m = 0; m < DB; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
  }
  store_rows_f32<D, DIRECT>(row_patch<D>(smem_raw, wave), dq_base + (int64_t)row0 * D, T_ - row0, acc, mul, lane);
}

// dK and dV, one wave per 32 keys, tiles of 32 queries, two stages, the vector work behind the products as in dkdv_split_f32_kernel
// (times above; D=128 traced alone 881 -> 775).  Every tile is masked: a mask that is all ones costs two instructions per element, one that is
// left out of inner tiles by a branch three, as the compiler makes a select of it (a tenth of the vector instructions at D=128, no spills at 32);
// two bodies, with and without, cost 240 copies of registers each.  The next tile's elements held in LDS on their way, to free 32
// registers: no difference.  Held to 256 registers for a second wave per SIMD D=64 spills and
// is slower.
template <int D, int NW>
__global__ __launch_bounds__(NW * 64, (D <= 32 ? 2 : 1)) void dkdv_halves_kernel(const BwdParams p) {
  constexpr int TKB = NW * 32, NT = NW * 64, TQ = 32, NF = D / 16, DB = TileGeom<_Float16, D>::DB;
  constexpr int TILE = HalfTile<D>::ELEMS;
  constexpr int STAGE_BYTES = 2 * TILE * 2 + 4 * TQ * 4;   // [Q][dO][lse, delta, factors of Q, of dO]

  extern __shared__ __attribute__((aligned(16))) char smem_raw[];

  const int tid = threadIdx.x;
  const int lane = tid & 63, c = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int bh, kt, L;
  key_tile_coords(blockIdx.x, gridDim.x, p.tiles, TKB, p.T, p.lens, p.lens_stride, bh, kt, L);
  const int b = div_by(bh, p.tiles.by_heads), hd = bh - b * p.H;
  const int T_ = p.T, C = p.C, R = p.R;
  const int k0 = kt * TKB;
  float* dk_base = reinterpret_cast<float*>(p.dk) + (int64_t)bh * T_ * D;
  float* dv_base = reinterpret_cast<float*>(p.dv) + (int64_t)bh * T_ * D;
  const int k_end = k0 + TKB < T_ ? k0 + TKB : T_;
  if (k0 >= L) {
    zero_rows<float, D, NT>(dk_base, k0, k_end, tid);
    zero_rows<float, D, NT>(dv_base, k0, k_end, tid);
    return;
  }

  // query window [qlo, qhi) of a key: its own chunk and the R chunks after it, below L
  auto win_lo = [&](int key) { return div_by(key, p.cdiv) * C; };
  auto win_hi = [&](int key) {
    const int64_t e = ((int64_t)div_by(key, p.cdiv) + R + 1) * (int64_t)C;
    return e < (int64_t)L ? (int)e : L;
  };
  auto valid = [&](int key) { return key < L ? key : L - 1; };   // keys past L mimic the last valid key
  const int krow = k0 + wave * 32 + c;
  const int qlo = win_lo(valid(krow)), qhi = win_hi(valid(krow));
  const int wk_first = valid(k0 + wave * 32), wk_last = valid(k0 + wave * 32 + 31);
  const int qhi_min = win_hi(wk_first), qlo_max = win_lo(wk_last);
  const int qlo_min = win_lo(wk_first), qhi_max = k0 + wave * 32 < L ? win_hi(wk_last) : 0;
  const int qt0 = win_lo(k0) / TQ, qt1 = (win_hi(valid(k0 + TKB - 1)) + TQ - 1) / TQ;

  const float* qbase = reinterpret_cast<const float*>(p.q) + (int64_t)b * p.q_sb + (int64_t)hd * p.q_sh;
  const float* gbase = reinterpret_cast<const float*>(p.d_o) + (int64_t)b * p.do_sb + (int64_t)hd * p.do_sh;
  const float* row_base = (tid < TQ ? p.lse : p.delta) + (int64_t)bh * T_;
  HalfStager<D, NT> sq, sg;
  float r_row = 0.0f;   // threads [0, TQ) stage lse, [TQ, 2*TQ) delta
  auto load_tile = [&](int t) {
    sq.load(qbase, p.q_st, t * TQ, L - 1, tid);
    sg.load(gbase, p.do_st, t * TQ, L - 1, tid);
    if (tid < 2 * TQ) r_row = row_base[valid(t * TQ + tid % TQ)];
  };
  const TileOrder order(qt0, qt1, p.period, p.pdiv);
  auto stage_step = [&](int it, int x) {   // tile of the it-th step
    constexpr int S = HalfStager<D, NT>::STEPS;
    _Float16* st = reinterpret_cast<_Float16*>(smem_raw + (it & 1) * STAGE_BYTES);
    float* const rows = reinterpret_cast<float*>(st + 2 * TILE);
    if (x < S) sq.step(x, st, rows + 2 * TQ, tid);
    else sg.step(x - S, st + TILE, rows + 3 * TQ, tid);
    if (x == 0 && tid < 2 * TQ) rows[tid] = r_row;
  };
  constexpr int WORK = 2 * HalfStager<D, NT>::STEPS;
  static_assert(2 * TQ <= NT, "one thread per staged row value");
  using Rows = OwnRows32<D>;
  const int row0 = k0 + wave * 32;
  float* const k_area = reinterpret_cast<float*>(smem_raw) + wave * Rows::ELEMS;
  float* const v_area = k_area + NW * Rows::ELEMS;
  const float* kbase = reinterpret_cast<const float*>(p.k) + (int64_t)b * p.k_sb + (int64_t)hd * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.v) + (int64_t)b * p.v_sb + (int64_t)hd * p.v_sh;
  constexpr bool DIRECT = direct_rows(D, NW);
  if (!DIRECT) {
    Rows::send(kbase, p.k_st, row0, L - 1, k_area, lane);
    Rows::send(vbase, p.v_st, row0, L - 1, v_area, lane);
  }
  load_tile(order.first);

  Half8 kf[NF], vf[NF];
  float ck;   // times a query's factor: score to base-2 exponent
  RowScale v_scale;
  {
    HalfRow<D> k_row, v_row;
    if (DIRECT) {
      k_row.load(kbase + (int64_t)valid(krow) * p.k_st, h);
      v_row.load(vbase + (int64_t)valid(krow) * p.v_st, h);
    } else {
      landed();
      k_row.read(k_area, lane);
      v_row.read(v_area, lane);
    }
    ck = halve_row<D>(kf, k_row).from * p.scale_log2e;
    v_scale = halve_row<D>(vf, v_row);
  }
  if (!DIRECT) __syncthreads();   // the tiles go where the rows were

  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int m = 0; m < DB; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[m][i] = 0.0f, dv[m][i] = 0.0f;
  constexpr bool HOLD = D < 128;          // the rows' values are held in registers, which there is no room for at 128
  OwnUnit k_unit, v_unit;                 // of the accumulators
#pragma unroll
  for (int x = 0; x < WORK; ++x) stage_step(0, x);
  if (order.next(order.first) != order.first) load_tile(order.next(order.first));
  __syncthreads();

  for (int t = order.first, it = 0; it < qt1 - qt0; ++it, t = order.next(t)) {
    if constexpr (D >= 64) {
      keep_in_agprs(kf);
      keep_in_agprs(vf);
    }
    const _Float16* Qt = reinterpret_cast<const _Float16*>(smem_raw + (it & 1) * STAGE_BYTES);
    const _Float16* Gt = Qt + TILE;
    const float* rows = reinterpret_cast<const float*>(Qt + 2 * TILE);
    const bool more = order.next(t) != order.first;
    const int qs = t * TQ;
    if (qs + TQ > qlo_min && qs < qhi_max) {
      const bool interior = qs >= qlo_max && qs + TQ <= qhi_min;
      const uint32_t rm = interior ? ~0u : row_mask(qlo - qs, qhi - qs, h);
      enum { LSE, DELTA, Q_FACTOR, G_FACTOR };   // of the query that register i stands for
      float held[4][16];
      if constexpr (HOLD) {
#pragma unroll
        for (int what = LSE; what <= G_FACTOR; ++what) row_factors(held[what], rows + what * TQ, h);
      }
      auto of_row = [&](int what, int i) {
        return HOLD ? held[what][i] : (*reinterpret_cast<const f32x4*>(rows + what * TQ + 8 * (i / 4) + 4 * h))[i % 4];
      };
      f32x16 s, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.0f, dp[i] = 0.0f;
      Half8 pb[2], sb[2];
      float most = 0.0f;
      // (the next tile's parts are formed whether there is one or not: no branch between the products)
      mma_rows_half<D>(s, Qt, kf, lane, [&](int g) {         // S[q][key]
#pragma unroll
        for (int x = g * WORK / NF; x < (g + 1) * WORK / NF; ++x) stage_step(it + 1, x);
      });
      mma_rows_half<D>(dp, Gt, vf, lane, [&](int g) {        // dP[q][key], in units of the V row's factor
#pragma unroll
        for (int i = g * 16 / NF; i < (g + 1) * 16 / NF; i += 2) {
#pragma unroll
          for (int e = i; e < i + 2; ++e) {
            s[e] = fast_exp2(__builtin_fmaf(s[e], of_row(Q_FACTOR, e) * ck, -of_row(LSE, e)));
            s[e] = keep_or_zero(s[e], keep_bits(rm, e));
          }
          v_unit.pair(pb, i, s[i], of_row(G_FACTOR, i), s[i + 1], of_row(G_FACTOR, i + 1), most);
        }
      });
      if (v_unit.leaves(s, most)) {
        float fg[16];
        row_factors(fg, rows + G_FACTOR * TQ, h);
        const float by = v_unit.move(s, fg);
#pragma unroll
        for (int m = 0; m < DB; ++m)
#pragma unroll
          for (int i = 0; i < 16; ++i) dv[m][i] *= by;
        v_unit.halve(pb, s, fg);
      }
      mma_tr_half<D>(dv, Gt, pb, lane, [&](int it) {         // dV^T[d][key] += dO^T P
#pragma unroll
        for (int i = it * 8 / DB; i < (it + 1) * 8 / DB; ++i) {
          s[i] *= __builtin_fmaf(dp[i], of_row(G_FACTOR, i), -of_row(DELTA, i) * v_scale.to);
          // a masked dP may hold anything (NaN included): P = 0 does not clear it
          s[i] = keep_or_zero(s[i], keep_bits(rm, i));
        }
      });
      float fq[16];
      row_factors(fq, rows + Q_FACTOR * TQ, h);
      if (k_unit.halve(sb, s, fq)) {
        const float by = k_unit.move(s, fq);
#pragma unroll
        for (int m = 0; m < DB; ++m)
#pragma unroll
          for (int i = 0; i < 16; ++i) dk[m][i] *= by;
        k_unit.halve(sb, s, fq);
      }
      mma_tr_half<D>(dk, Qt, sb, lane);                      // dK^T[d][key] += Q^T dS
    } else {
#pragma unroll
      for (int x = 0; x < WORK; ++x) stage_step(it + 1, x);
    }
    if (more) {
      const int then = order.next(order.next(t));
      if (then != order.first) load_tile(then);
    }
    __syncthreads();
  }

  const float mul = v_scale.from * p.scale;
  const bool odd = !k_unit.settle<D>(dk, mul) || !v_unit.settle<D>(dv, 1.0f) || too_large(v_scale.from) || too_large(sg.most) || scale_too_small(p.scale_log2e);
  if (any_in_workgroup<NW>(odd, smem_raw, wave, lane)) {
    dkdv_rows<float, D, NW, TQ>(p, again_s(bh), again_s(kt), again_v(tid));
    return;
  }
  if (krow >= L) {
#pragma unroll
    for (int m = 0; m < DB; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i) dk[m][i] = 0.0f, dv[m][i] = 0.0f;
  }
  float* const patch = row_patch<D>(smem_raw, wave);
  store_rows_f32<D, DIRECT>(patch, dk_base + (int64_t)row0 * D, T_ - row0, dk, mul, lane);
  store_rows_f32<D, DIRECT>(patch, dv_base + (int64_t)row0 * D, T_ - row0, dv, 1.0f, lane);
}

}  // namespace sa
