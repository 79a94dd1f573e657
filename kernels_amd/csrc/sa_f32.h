// float32 kernels on the 16-bit matrix pipe, head dimensions 16 to 128.
//
// v_mfma_f32_32x32x2_f32 does 64 flop per cycle and SIMD, v_mfma_f32_32x32x16_bf16 1024.  A float32
// number is the sum of three bfloat16 numbers (24 = 8 + 8 + 8 significand bits; each part is the rounded
// remainder of the ones before), so a float32 product is
//   x*y = x1*y1 + (x1*y2 + x2*y1) + (x1*y3 + x2*y2 + x3*y1) + [x2*y3 + x3*y2 + x3*y3],
// every term of which the bfloat16 instruction forms exactly and adds up in float32 (the decomposition of Henry, Tang
// and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision computations", 2019).
// The bracket is left out: it is at most 2^-24 of |x*y|, to which float32 rounds a product (or a running sum) too, and
// 2^-27 in the root mean square.  Six products at 16 times the rate take 6/16 of the matrix time, and the
// sums have fewer roundings (16 contraction slots per instruction instead of 2).  Measured on problems of 200 to 4096
// positions against float64: errors of O, dQ, dK, dV at or below those of the float32 instruction
// kernels (see the comment at each kernel for times).
//
// The parts reach down to 2^-133, bfloat16's smallest number, and float32 to 2^-149: every operand is multiplied by
// kUp = 2^16 before it is split, exactly, and the products' powers of two are taken out where the result is scaled anyway.
// What then exceeds the exponent range (elements from 2^111 on, infinities, sums and dS beyond about 2^80 to 2^96)
// or was not a number to begin with leaves a result that is not finite, since a part of it is NaN; a workgroup
// that sees one goes through its rows again with the float32 instruction (fwd_rows, dq_rows, dkdv_rows).
//
// The parts of the resident operand are formed once per wave and stay in registers; those of the streamed
// tiles are formed once per workgroup on the way into LDS, where each part is a bfloat16 tile of its own
// (the swizzled layout and transposing reads of the 16-bit kernels apply unchanged).  Probabilities and dS
// are split in registers.
#pragma once
#include "sa_bwd.h"
#include "sa_common.h"
#include "sa_fwd.h"

namespace sa {

constexpr float kUp = 0x1p16f;                                 // of one operand
constexpr float kUp2 = 0x1p32f, kDown2 = 0x1p-32f;             // of a product of two
constexpr float kDown3 = 0x1p-48f;                             // of dS (a product of two) times an operand
// A scale that times these powers of two is no normal number.
SA_DEV bool scale_too_small(float scale_log2e) { return scale_log2e != 0.0f && fabsf(scale_log2e) < 0x1p-60f; }

// Three bfloat16 fragments that add up to eight float32 values.
struct Split8 {
  bf16x8 p[3];
};
// The parts of two values, packed: one conversion for both, widened again with one shift and one mask.
SA_DEV void split2(float x0, float x1, uint32_t (&u)[3]) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  f32x2 r = {x0, x1};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    u[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
    r[0] -= __uint_as_float(u[k] << 16);
    r[1] -= __uint_as_float(u[k] & 0xFFFF0000u);
  }
}
// Elements 2*e and 2*e+1 of a fragment.
SA_DEV void split_pair(Split8& s, int e, float x0, float x1) {
  uint32_t u[3];
  split2(x0, x1, u);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    u32x4 w = __builtin_bit_cast(u32x4, s.p[k]);
    w[e] = u[k];
    s.p[k] = __builtin_bit_cast(bf16x8, w);
  }
}
SA_DEV Split8 split8(const float (&x)[8]) {
  Split8 s;
#pragma unroll
  for (int e = 0; e < 4; ++e) split_pair(s, e, x[2 * e], x[2 * e + 1]);
  return s;
}
// The six products, smallest first.
SA_DEV void mma6(f32x16& acc, const Split8& a, const Split8& b) {
  mma(acc, a.p[2], b.p[0]);
  mma(acc, a.p[0], b.p[2]);
  mma(acc, a.p[1], b.p[1]);
  mma(acc, a.p[1], b.p[0]);
  mma(acc, a.p[0], b.p[1]);
  mma(acc, a.p[0], b.p[0]);
}

// One LDS tile of ROWS rows: three bfloat16 tiles, one per part.
template <int D, int ROWS> struct SplitTile {
  using G = TileGeom<__bf16, D, D == 16>;
  static constexpr int PLANE = ROWS * G::PITCH;   // elements
  static constexpr int ELEMS = 3 * PLANE;
};

// Copy of a [ROWS][D] float32 tile through registers into a SplitTile, eight elements per thread and step.
// Rows are clamped to last_row (the values are masked by the caller).
template <int D, int ROWS, int NT> struct SplitStager {
  using G = TileGeom<__bf16, D, D == 16>;
  static constexpr int CPR = D / 8, TOTAL = ROWS * CPR, N = (TOTAL + NT - 1) / NT;
  f32x4 regs[N][2];

  SA_DEV void load(const float* base, int64_t row_stride, int row0, int last_row, int tid) {
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const int ch = tid + it * NT;
      if (TOTAL % NT == 0 || ch < TOTAL) {
        int gr = row0 + ch / CPR;
        gr = gr < last_row ? gr : last_row;
        const float* src = base + (int64_t)gr * row_stride + (ch % CPR) * 8;
        regs[it][0] = *reinterpret_cast<const f32x4*>(src);
        regs[it][1] = *reinterpret_cast<const f32x4*>(src + 4);
      }
    }
  }
  SA_DEV void store(__bf16* tile, int tid) const {
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const int ch = tid + it * NT;
      if (TOTAL % NT == 0 || ch < TOTAL) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = regs[it][e / 4][e % 4] * kUp;
        __bf16* dst = tile + G::off(ch / CPR, (ch % CPR) * 8);
        const Split8 s = split8(x);
#pragma unroll
        for (int k = 0; k < 3; ++k) *reinterpret_cast<bf16x8*>(dst + k * SplitTile<D, ROWS>::PLANE) = s.p[k];
      }
    }
  }
};

// The 32 rows that a wave keeps, as copies of whole rows through 32 * D floats of LDS of its own (see OwnRows in sa_common.h,
// whose swizzle of rows of as many bytes this is).  The addresses are formed per lane, in 64 bits: float32 tensors have no
// limit on their row stride.  Rows past the last valid one have its values.
template <int D> struct OwnRows32 {
  using G = TileGeom<__bf16, 2 * D>;
  static constexpr int ELEMS = 32 * D, CPR = D / 4, RPI = 64 / CPR, N = 32 / RPI;
  SA_DEV static int off(int row, int chunk) { return G::off(row, chunk * 8) / 2; }   // of sixteen bytes, in floats
  SA_DEV static void send(const float* base, int64_t row_stride, int row0, int last_row, float* area, int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = i * RPI + lane / CPR, gr = row0 + r < last_row ? row0 + r : last_row;
      const float* src = base + (int64_t)gr * row_stride + ((lane % CPR) ^ G::swz(r)) * 4;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (SA_LDS void*)(area + i * 256), 16, 0, 0);
    }
  }
};
// What own rows through LDS, whole-row stores past the caches and the tile order give each, us with the other two in place, without ->
// with: forward and backward B=4, H=8, T<=2000, chunks of 50, 3 back, D=128 285, 281, 277 -> 275, D=64 151, 150, 148 -> 147, D=32 91, 90, 91 ->
// 88; B=4, H=16, T=4096, chunks of 128, 4 back, D=128 1965, 1966, 1969 -> 1954 (spread 16); the stores lose on D=128, lengths in [1, 4096],
// chunks of 32, 2 back 782 -> 795.  The copies' addresses cost registers: see the spills at the kernels.
// Not where a row is a sixteenth of a kilobyte (D = 16: B=8, H=16, T=1000, chunks of 20, 4 back, forward and backward 88.1 us, 91.5
// this way) nor in the workgroups of two waves, whose grids take as long as one workgroup's chain of latencies (see
// half_workgroups; B=2, H=4, T=512, D=64 forward 15.0, 15.4 this way): there a lane loads its half row itself and stores its
// row itself.  The size of the grid picks the workgroups of a head dimension, so all of them add up in the same order and a
// sequence has the same bits in any batch: row sums as dot_half_row, tiles in the order of the largest workgroup's
// windows (tile_order_f32 in sa_inst.hip).
constexpr bool direct_rows(int D, int NW) { return D == 16 || NW == 2; }
// Row sums of the products of a wave's rows of O, read whole from memory, with those of dO in LDS (see RowDots).
SA_DEV float dot4(const f32x4& a, const f32x4& b) { return __builtin_fmaf(a[0], b[0], a[1] * b[1]) + __builtin_fmaf(a[2], b[2], a[3] * b[3]); }
template <int D> struct RowDots32 {
  using Rows = OwnRows32<D>;
  static constexpr int CPR = Rows::CPR, RPI = Rows::RPI, N = Rows::N, PITCH = CPR + 4;
  f32x4 of[N];
  SA_DEV void load(const float* base, int64_t row_stride, int row0, int last_row, int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = row0 + i * RPI + lane / CPR;
      of[i] = *reinterpret_cast<const f32x4*>(base + (int64_t)(r < last_row ? r : last_row) * row_stride + lane % CPR * 4);
    }
  }
  SA_DEV void partial(const float* g_area, float* scratch, int lane) const {
    wave_exchange();
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = i * RPI + lane / CPR, ch = lane % CPR;
      const f32x4 gf = *reinterpret_cast<const f32x4*>(g_area + Rows::off(r, ch));
      scratch[r * PITCH + ch] = dot4(of[i], gf);
    }
  }
  SA_DEV static float total(const float* scratch, int lane) {
    wave_exchange();
    const float* row = scratch + (lane & 31) * PITCH + (lane >> 5) * 2;
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < CPR / 2; ++i) sum += row[(i / 2) * 4 + i % 2];   // the chunks of HalfRow
    return half_sum(sum);
  }
};

// Whole rows from the accumulators (X^T: a lane owns a row), 64 columns at a time through a patch of LDS of the wave's own, so
// that a store instruction writes whole cache lines and may pass the caches (store_streaming).
template <int D> struct RowPatch32 {
  static constexpr int W = D < 64 ? D : 64, PITCH = W + 4, ELEMS = 32 * PITCH, CPR = W / 4, RPI = 64 / CPR;
};
template <int D, bool DIRECT, int DB>
SA_DEV void store_rows_f32(float* patch, float* out_rows, int rows_valid, const f32x16 (&acc)[DB], float mul, int lane) {
  using P = RowPatch32<D>;
  const int c = lane & 31, h = lane >> 5;
  if constexpr (DIRECT) {
    if (c < rows_valid) store_acc_T<float, D, DB>(out_rows + (int64_t)c * D, acc, mul, h);
    return;
  }
#pragma unroll
  for (int col = 0; col < D; col += P::W) {
    wave_exchange();
#pragma unroll
    for (int m = col / 32; m < DB && m * 32 < col + P::W; ++m)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = m * 32 - col + 8 * g + 4 * h;
        store4<float>(patch + c * P::PITCH + d, acc[m][4 * g] * mul, acc[m][4 * g + 1] * mul, acc[m][4 * g + 2] * mul,
                      acc[m][4 * g + 3] * mul);
      }
    wave_exchange();
#pragma unroll
    for (int j = 0; j < 32 / P::RPI; ++j) {
      const int row = j * P::RPI + lane / P::CPR, ch = lane % P::CPR;
      const u32x4 v16 = *reinterpret_cast<const u32x4*>(patch + row * P::PITCH + ch * 4);
      if (row < rows_valid) store_streaming(out_rows + (int64_t)row * D + col + ch * 4, v16);
    }
  }
}

// This lane's half of a float32 row, and its split fragments (as a B operand).
template <int D> struct HalfRow {
  f32x4 r[D / 8];
  SA_DEV void load(const float* row, int h) {
#pragma unroll
    for (int i = 0; i < D / 8; ++i) r[i] = *reinterpret_cast<const f32x4*>(row + (i / 2) * 16 + h * 8 + (i % 2) * 4);
  }
  SA_DEV void read(const float* area, int lane) {
    const int c = lane & 31, h = lane >> 5;
#pragma unroll
    for (int i = 0; i < D / 8; ++i) r[i] = *reinterpret_cast<const f32x4*>(area + OwnRows32<D>::off(c, (i / 2) * 4 + h * 2 + i % 2));
  }
  SA_DEV float dot_half_row(const HalfRow& other) const {   // RowDots32 adds up the same numbers in the same order
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < D / 8; ++i) {
      if constexpr (D == 16) {   // every workgroup reads its rows directly: one chain, as near as any order
#pragma unroll
        for (int e = 0; e < 4; ++e) sum = __builtin_fmaf(r[i][e], other.r[i][e], sum);
      } else {
        sum += dot4(r[i], other.r[i]);
      }
    }
    return half_sum(sum);
  }
  SA_DEV void split(Split8 (&f)[D / 16], bool negative) const {
    const float mul = negative ? -kUp : kUp;
#pragma unroll
    for (int g = 0; g < D / 16; ++g) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = r[2 * g + e / 4][e % 4] * mul;
      f[g] = split8(x);
    }
  }
};

// acc[row r][col c] += sum_k tile[r][k] * B[k][c] for the 32 rows of a split tile.  side(g) is vector work placed
// behind the matrix instructions of step g: a wave that has a SIMD to itself has nothing else to fill them with.
template <int D, int ROWS, typename Side = NoSide>
SA_DEV void mma_rows_split(f32x16& acc, const __bf16* tile, const Split8 (&b)[D / 16], int lane, Side&& side = Side()) {
  using G = TileGeom<__bf16, D, D == 16>;
  const int c = lane & 31, h = lane >> 5;
  const __bf16* base = tile + c * G::PITCH;
  const int sw = G::swz(c);
  pipeline<D / 16, 1>(
      [&](int g) {
        Split8 a;
#pragma unroll
        for (int k = 0; k < 3; ++k)
          a.p[k] = *reinterpret_cast<const bf16x8*>(base + k * SplitTile<D, ROWS>::PLANE + (((g * 2 + h) ^ sw) * 8));
        return a;
      },
      [&](int g, const Split8& a) { mma6(acc, a, b[g]); side(g); });
}

// acc[m] += X^T * P for 16*NH rows of a split tile X, from row 16*half0; P is a C fragment, split by the caller (rows
// 16*(half0 + j) and up in b[j]).  Step it = j * NM + m.
template <int D, int ROWS, int NM, int NH, typename Side = NoSide>
SA_DEV void mma_tr_split(f32x16 (&acc)[NM], const __bf16* X, const Split8 (&b)[NH], int lane, Side&& side = Side(),
                         int half0 = 0) {
  using G = TileGeom<__bf16, D, D == 16>;
  static_assert(NM == G::DB, "one accumulator per 32-wide block of the head dimension");
  const int g16 = lane >> 4, j = lane & 15;
  const int r_lo = 4 * (g16 >> 1) + (j >> 2);
  const int col = (g16 & 1) * 16 + 4 * (j & 3);
  pipeline<NH * NM, 1>(
      [&](int it) {
        const int half = half0 + it / NM, m = it % NM;
        Split8 a;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const __bf16* p0 = X + k * SplitTile<D, ROWS>::PLANE + G::off(half * 16 + r_lo, m * 32 + col);
          const __bf16* p1 = X + k * SplitTile<D, ROWS>::PLANE + G::off(half * 16 + 8 + r_lo, m * 32 + col);
          s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((SA_LDS s16x4*)(p0));
          s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((SA_LDS s16x4*)(p1));
          a.p[k] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
        return a;
      },
      [&](int it, const Split8& a) { mma6(acc[it % NM], a, b[it / NM]); side(it); });
}
// The split B operand of mma_tr_split from a whole C fragment, times mul (a power of two).
SA_DEV void split_c(Split8 (&b)[2], const f32x16& P, float mul = 1.0f) {
#pragma unroll
  for (int i = 0; i < 16; i += 2) split_pair(b[i / 8], (i % 8) / 2, P[i] * mul, P[i + 1] * mul);
}

// Whether the rows of an accumulator that stand for elements of the head dimension are finite (at 16 half of them do).
template <int D, int NM> SA_DEV bool all_finite(const f32x16 (&acc)[NM]) {
  float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};   // becomes NaN
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (m * 32 + 8 * (i >> 2) < D) z[i & 3] = __builtin_fmaf(acc[m][i], 0.0f, z[i & 3]);
  return (z[0] + z[1]) + (z[2] + z[3]) == 0.0f;
}
// The same value as one that the compiler knows nothing of: what the second way through the rows derives from it is computed
// there, not kept in registers through the loop of the first.
SA_DEV int again_s(int x) {
  asm volatile("" : "+s"(x));
  return x;
}
SA_DEV int again_v(int x) {
  asm volatile("" : "+v"(x));
  return x;
}
// Whether some lane of the workgroup says so; smem is not read by anyone any more and free again after the call.
template <int NW> SA_DEV bool any_in_workgroup(bool x, void* smem, int wave, int lane) {
  volatile SA_LDS uint32_t* flags = (volatile SA_LDS uint32_t*)smem;
  const bool mine = __builtin_amdgcn_ballot_w64(x) != 0;
  if (lane == 0) flags[wave] = mine;
  __syncthreads();
  uint32_t any = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) any |= flags[w];
  if (__builtin_expect(__builtin_amdgcn_readfirstlane(any) == 0, 1)) return false;
  __syncthreads();
  return true;
}

// A wave's row patch after any_in_workgroup, whose flags other waves may still read.
template <int D> SA_DEV float* row_patch(char* smem, int wave) {
  return reinterpret_cast<float*>(smem + 64) + wave * RowPatch32<D>::ELEMS;
}

// The windows of a wave's 32 queries, of one lane's query, and of the workgroup.
struct QueryWindow {
  int lo, hi;            // this lane's keys
  int lo_max, hi_min;    // keys every query of the wave sees
  int lo_min, hi_max;    // keys any query of the wave sees (empty for a wave of padding)
  int lo_wg, hi_wg;      // keys any query of the workgroup sees
  SA_DEV QueryWindow(int q0, int wave, int TQ, int qrow, int L, int C, int R, ChunkDiv cd) {
    auto low = [&](int q) { const int x = div_by(q, cd); return (x > R ? x - R : 0) * C; };
    auto high = [&](int q) { const int e = (div_by(q, cd) + 1) * C; return e < L ? e : L; };
    auto valid = [&](int q) { return q < L ? q : L - 1; };   // rows past L mimic the last valid row
    lo = low(valid(qrow)), hi = high(valid(qrow));
    const int first = valid(q0 + wave * 32), last = valid(q0 + wave * 32 + 31);
    lo_max = low(last), hi_min = high(first);
    lo_min = low(first), hi_max = q0 + wave * 32 < L ? high(last) : 0;
    lo_wg = low(q0), hi_wg = high(valid(q0 + TQ - 1));
  }
};

// Forward.  One wave per 32 queries, tiles of 32 keys in NST stages.  Bound by the matrix pipe: 1.1 PFLOP/s of
// bfloat16 products.  B=4, H=16, T=4096, chunks of 128, 4 back, us with the float32 instruction -> here: D=128 720 -> 455,
// D=64 392 -> 220, D=32 200 -> 125, D=16 167 -> 107 (with OwnRows32, whole-row stores and TileOrder 456 -> 432, 223 -> 218, 129 -> 128).
// The register limits (four waves per SIMD up to 32, three at 64, two at 128) make D=64 and 128 spill 19 and 31
// registers per lane, 82 in the four-wave form of 128, around the products.
template <int D, int NW, int NST, bool BY_LENGTH>
__global__ __launch_bounds__(NW * 64, (D <= 32 ? 4 : D == 64 && NW == 4 ? 3 : 2)) void fwd_split_kernel(const FwdParams p) {
  constexpr int TQ = NW * 32, NT = NW * 64, TK = 32, DB = TileGeom<__bf16, D, D == 16>::DB;
  constexpr int TILE = SplitTile<D, TK>::ELEMS;
  constexpr float kRescaleGap = 8.0f;
  constexpr float kSumLimit = 256.0f;

  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  __bf16* smem = reinterpret_cast<__bf16*>(smem_raw);   // [stage][K|V][part][TK][PITCH]

  const int tid = threadIdx.x;
  const int lane = tid & 63, c = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int bh, qt, L = p.T;
  if (BY_LENGTH) tile_coords_by_length<TQ>(blockIdx.x, p.tiles, p.by_length, p.lens, p.lens_stride, p.T, p.H, lane, bh, qt, L);
  else tile_coords(blockIdx.x, gridDim.x, p.tiles, bh, qt);
  const int T_ = p.T;
  const int b = div_by(bh, p.tiles.by_heads), hd = bh - b * p.H;
  if (p.lens && !BY_LENGTH) {
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
  // never exactly 0, so that a masked score of -inf stays -inf after scaling
  const float sl2e = fmaxf(fabsf(p.scale_log2e) * kDown2, 0x1p-126f);

  const float* kbase = reinterpret_cast<const float*>(p.k) + (int64_t)b * p.k_sb + (int64_t)hd * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.v) + (int64_t)b * p.v_sb + (int64_t)hd * p.v_sh;
  float* const q_area = reinterpret_cast<float*>(smem_raw) + wave * OwnRows32<D>::ELEMS;
  const float* qbase = reinterpret_cast<const float*>(p.q) + (int64_t)b * p.q_sb + (int64_t)hd * p.q_sh;
  constexpr bool DIRECT = direct_rows(D, NW);
  if (!DIRECT) OwnRows32<D>::send(qbase, p.q_st, q0 + wave * 32, L - 1, q_area, lane);
  const TileOrder order(kt0, kt1, p.period, p.pdiv);
  SplitStager<D, TK, NT> sk, sv;
  sk.load(kbase, p.k_st, order.first * TK, L - 1, tid);
  sv.load(vbase, p.v_st, order.first * TK, L - 1, tid);

  Split8 qf[D / 16];
  {
    HalfRow<D> qr;
    if (DIRECT) {
      qr.load(qbase + (int64_t)(qrow < L ? qrow : L - 1) * p.q_st, h);
    } else {
      landed();
      qr.read(q_area, lane);
    }
    qr.split(qf, p.scale_log2e < 0.0f);
  }
  if (!DIRECT) __syncthreads();   // the tiles go where the rows were

  f32x16 oacc[DB];
#pragma unroll
  for (int m = 0; m < DB; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[m][i] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;

  sk.store(smem, tid);
  sv.store(smem + TILE, tid);
  __syncthreads();

  for (int t = order.first, it = 0; it < kt1 - kt0; ++it, t = order.next(t)) {
    const __bf16* Kt = smem + (it % NST) * 2 * TILE;
    const __bf16* Vt = Kt + TILE;
    const bool more = order.next(t) != order.first;
    if (more) {
      sk.load(kbase, p.k_st, order.next(t) * TK, L - 1, tid);
      sv.load(vbase, p.v_st, order.next(t) * TK, L - 1, tid);
    }
    const int k0 = t * TK;
    if (k0 + TK > w.lo_min && k0 < w.hi_max) {   // some query of this wave sees the tile
      f32x16 s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.0f;
      mma_rows_split<D, TK>(s, Kt, qf, lane);
      if (!(k0 >= w.lo_max && k0 + TK <= w.hi_min)) {
        const uint32_t rm = row_mask(w.lo - k0, w.hi - k0, h);
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = keep_or_neg_inf(s[i], keep_bits(rm, i));
      }
      // probabilities against the running maximum as it stands; it is searched for when their sum shows that
      // it has been left behind, or when a lane has none yet (see fwd2_kernel)
      f32x16 pr;
      float rs0, rs1;
      auto probabilities = [&](float m_use) {
        rs0 = rs1 = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) pr[i] = fast_exp2(__builtin_fmaf(s[i], sl2e, -m_use));
#pragma unroll
        for (int i = 0; i < 16; i += 2) rs0 += pr[i], rs1 += pr[i + 1];
      };
      probabilities(m_run == -INFINITY ? 0.0f : m_run);
      const bool behind = !(rs0 + rs1 <= kSumLimit) || m_run == -INFINITY;   // true for NaN too
      if (__builtin_amdgcn_ballot_w64(behind) != 0) {
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; i += 2) mx = fast_max3(mx, s[i], s[i + 1]);
        mx = half_max(mx) * sl2e;
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
      Split8 pb[2];
      split_c(pb, pr, kUp);
      mma_tr_split<D, TK>(oacc, Vt, pb, lane);   // O^T[d][q] += V^T P^T
    }
    if (more) {
      if (NST == 1) __syncthreads();   // the only stage has no reader left
      __bf16* nxt = smem + ((it + 1) % NST) * 2 * TILE;
      sk.store(nxt, tid);
      sv.store(nxt + TILE, tid);
    }
    __syncthreads();
  }

  const float l_tot = half_sum(l_run);
  const bool odd = q0 + wave * 32 < L && (!(l_tot > 0.0f) || !all_finite<D>(oacc) || scale_too_small(p.scale_log2e));
  if (any_in_workgroup<NW>(odd, smem_raw, wave, lane)) {
    fwd_rows<float, D, NW, TK>(p, again_s(bh), again_s(qt), again_v(tid));
    return;
  }
  const bool valid = qrow < L;
  const float inv = valid ? 1.0f / l_tot * kDown2 : 0.0f;
  if (!valid) {
#pragma unroll
    for (int m = 0; m < DB; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[m][i] = 0.0f;
  }
  const int row0 = q0 + wave * 32;
  store_rows_f32<D, DIRECT>(row_patch<D>(smem_raw, wave), o_base + (int64_t)row0 * D, T_ - row0, oacc, inv, lane);
  if (lse_base && h == 0 && qrow < T_) lse_base[qrow] = valid ? m_run + __builtin_amdgcn_logf(l_tot) : 0.0f;
}

// dQ, one wave per 32 queries, tiles of 32 keys, two stages.  delta = rowsum(O * dO) is formed in the prologue (the
// O row is read beside the dO row) and written for the dK/dV kernel that runs after this one, or read when the caller
// has computed it (p.delta_out == null).  Same problem as above: D=128 1027 -> 679 us (one wave per SIMD: the parts of Q
// and dO are 192 registers), D=64 557 -> 309, D=32 274 -> 181, D=16 197 -> 117; forming delta here saves a pass of 40 us over
// O and dO at D=128.
template <int D, int NW>
__global__ __launch_bounds__(NW * 64, (D <= 64 ? 2 : 1)) void dq_split_kernel(const BwdParams p) {
  constexpr int TQ = NW * 32, NT = NW * 64, TK = 32, NF = D / 16, DB = TileGeom<__bf16, D, D == 16>::DB;
  constexpr int TILE = SplitTile<D, TK>::ELEMS;

  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  __bf16* smem = reinterpret_cast<__bf16*>(smem_raw);

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
  const float sl2e = fabsf(p.scale_log2e) * kDown2;

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
  SplitStager<D, TK, NT> sk, sv;
  sk.load(kbase, p.k_st, order.first * TK, L - 1, tid);
  sv.load(vbase, p.v_st, order.first * TK, L - 1, tid);

  Split8 qf[NF], gf[NF];
  const int qr = qrow < L ? qrow : L - 1;
  const float lse_q = qrow < L ? p.lse[(int64_t)bh * T_ + qr] : INFINITY;   // rows past L: P = exp2(-inf) = 0
  float delta_q;
  {
    float sum = 0.0f;
    if (DIRECT) {
      HalfRow<D> q_row, g_row, o_row;
      q_row.load(qbase + (int64_t)qr * p.q_st, h);
      g_row.load(gbase + (int64_t)qr * p.do_st, h);
      o_row.load(obase + (int64_t)qr * o_st, h);
      q_row.split(qf, p.scale_log2e < 0.0f);
      g_row.split(gf, false);
      sum = o_row.dot_half_row(g_row);
    } else {
      HalfRow<D> row;
      landed();
      row.read(g_area, lane);
      row.split(gf, false);
      row.read(q_area, lane);
      row.split(qf, p.scale_log2e < 0.0f);
      dots.partial(g_area, q_area, lane);
      sum = RowDots32<D>::total(q_area, lane);
    }
    if (p.delta_out) {
      delta_q = sum;
      if (h == 0 && qrow < T_) p.delta_out[(int64_t)bh * T_ + qrow] = qrow < L ? delta_q : 0.0f;
    } else {
      delta_q = p.delta[(int64_t)bh * T_ + qr];
    }
  }
  if (!DIRECT) __syncthreads();   // the tiles go where the rows were

  const float dinit = -delta_q * kUp2;

  f32x16 acc[DB];
#pragma unroll
  for (int m = 0; m < DB; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
  sk.store(smem, tid);
  sv.store(smem + TILE, tid);
  __syncthreads();

  for (int t = order.first, it = 0; it < kt1 - kt0; ++it, t = order.next(t)) {
    const __bf16* Kt = smem + (it & 1) * 2 * TILE;
    const __bf16* Vt = Kt + TILE;
    const bool more = order.next(t) != order.first;
    if (more) {
      sk.load(kbase, p.k_st, order.next(t) * TK, L - 1, tid);
      sv.load(vbase, p.v_st, order.next(t) * TK, L - 1, tid);
    }
    const int k0 = t * TK;
    if (k0 + TK > w.lo_min && k0 < w.hi_max) {
      f32x16 s, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.0f, dp[i] = dinit;
      mma_rows_split<D, TK>(s, Kt, qf, lane);
      mma_rows_split<D, TK>(dp, Vt, gf, lane, [&](int g) {
#pragma unroll
        for (int i = g * 16 / NF; i < (g + 1) * 16 / NF; ++i) s[i] = fast_exp2(__builtin_fmaf(s[i], sl2e, -lse_q));
      });
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] *= dp[i];   // dS
      if (!(k0 >= w.lo_max && k0 + TK <= w.hi_min)) {
        const uint32_t rm = row_mask(w.lo - k0, w.hi - k0, h);
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = keep_or_zero(s[i], keep_bits(rm, i));
      }
      Split8 sb[2];
      split_c(sb, s);
      mma_tr_split<D, TK>(acc, Kt, sb, lane);   // dQ^T[d][q] += K^T dS^T
    }
    if (more) {
      __bf16* nxt = smem + (~it & 1) * 2 * TILE;
      sk.store(nxt, tid);
      sv.store(nxt + TILE, tid);
    }
    __syncthreads();
  }

  if (any_in_workgroup<NW>(!all_finite<D>(acc) || scale_too_small(p.scale_log2e), smem_raw, wave, lane)) {
    dq_rows<float, D, NW, TK>(p, again_s(bh), again_s(qt), again_v(tid), [&](int) { return delta_q; });   // this lane's query
    return;
  }
  if (qrow >= L) {
#pragma unroll
    for (int m = 0; m < DB; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
  }
  store_rows_f32<D, DIRECT>(row_patch<D>(smem_raw, wave), dq_base + (int64_t)row0 * D, T_ - row0, acc, p.scale * kDown3, lane);
}

// dK and dV, one wave per 32 keys, tiles of 32 queries, two stages.  Four products per tile; the vector work sits behind
// their matrix instructions (the exponentials and the parts of P behind dP, dS and its parts behind dV): from head
// dimension 64 on a wave has its SIMD to itself.  Held to 256 registers for a second wave, D=64 spilled and measured
// the same or slower.  Same problem as above: D=128 1470 -> 883 us (42 registers spilled), D=64 665 -> 476, D=32 351 -> 245,
// D=16 261 -> 194.
template <int D, int NW>
__global__ __launch_bounds__(NW * 64, (D <= 32 ? 2 : 1)) void dkdv_split_f32_kernel(const BwdParams p) {
  constexpr int TKB = NW * 32, NT = NW * 64, TQ = 32, NF = D / 16, DB = TileGeom<__bf16, D, D == 16>::DB;
  constexpr int TILE = SplitTile<D, TQ>::ELEMS;
  constexpr int STAGE_BYTES = 2 * TILE * 2 + 2 * TQ * 4;   // [Q][dO][lse, delta]

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
  const float sl2e = fabsf(p.scale_log2e) * kDown2;

  const float* qbase = reinterpret_cast<const float*>(p.q) + (int64_t)b * p.q_sb + (int64_t)hd * p.q_sh;
  const float* gbase = reinterpret_cast<const float*>(p.d_o) + (int64_t)b * p.do_sb + (int64_t)hd * p.do_sh;
  const float* row_base = (tid < TQ ? p.lse : p.delta) + (int64_t)bh * T_;
  SplitStager<D, TQ, NT> sq, sg;
  float r_row = 0.0f;   // threads [0, TQ) stage lse, [TQ, 2*TQ) delta
  auto load_tile = [&](int t) {
    sq.load(qbase, p.q_st, t * TQ, L - 1, tid);
    sg.load(gbase, p.do_st, t * TQ, L - 1, tid);
    if (tid < 2 * TQ) r_row = row_base[valid(t * TQ + tid % TQ)];
  };
  constexpr bool DIRECT = direct_rows(D, NW);
  const TileOrder order(qt0, qt1, p.period, p.pdiv);
  auto store_tile = [&](int it) {
    __bf16* st = reinterpret_cast<__bf16*>(smem_raw + (it & 1) * STAGE_BYTES);
    sq.store(st, tid);
    sg.store(st + TILE, tid);
    if (tid < 2 * TQ) reinterpret_cast<float*>(st + 2 * TILE)[tid] = tid < TQ ? r_row : r_row * kUp2;
  };
  static_assert(2 * TQ <= NT, "one thread per staged row value");
  using Rows = OwnRows32<D>;
  const int row0 = k0 + wave * 32;
  float* const k_area = reinterpret_cast<float*>(smem_raw) + wave * Rows::ELEMS;
  float* const v_area = k_area + NW * Rows::ELEMS;
  const float* kbase = reinterpret_cast<const float*>(p.k) + (int64_t)b * p.k_sb + (int64_t)hd * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.v) + (int64_t)b * p.v_sb + (int64_t)hd * p.v_sh;
  if (!DIRECT) {
    Rows::send(kbase, p.k_st, row0, L - 1, k_area, lane);
    Rows::send(vbase, p.v_st, row0, L - 1, v_area, lane);
  }
  load_tile(order.first);

  Split8 kf[NF], vf[NF];
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
    k_row.split(kf, p.scale_log2e < 0.0f);
    v_row.split(vf, false);
  }
  if (!DIRECT) __syncthreads();   // the tiles go where the rows were

  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int m = 0; m < DB; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[m][i] = 0.0f, dv[m][i] = 0.0f;
  store_tile(0);
  __syncthreads();

  for (int t = order.first, it = 0; it < qt1 - qt0; ++it, t = order.next(t)) {
    const __bf16* Qt = reinterpret_cast<const __bf16*>(smem_raw + (it & 1) * STAGE_BYTES);
    const __bf16* Gt = Qt + TILE;
    const float* rows = reinterpret_cast<const float*>(Qt + 2 * TILE);
    const bool more = order.next(t) != order.first;
    if (more) load_tile(order.next(t));
    const int qs = t * TQ;
    if (qs + TQ > qlo_min && qs < qhi_max) {
      const bool interior = qs >= qlo_max && qs + TQ <= qhi_min;
      const uint32_t rm = interior ? ~0u : row_mask(qlo - qs, qhi - qs, h);
      f32x16 s, dp, lse_r;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(rows + 8 * g4 + 4 * h);
        const f32x4 d4 = *reinterpret_cast<const f32x4*>(rows + TQ + 8 * g4 + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[4 * g4 + e] = 0.0f, dp[4 * g4 + e] = -d4[e], lse_r[4 * g4 + e] = l4[e];
      }
      Split8 pb[2], sb[2];
      mma_rows_split<D, TQ>(s, Qt, kf, lane);                // S[q][key]
      mma_rows_split<D, TQ>(dp, Gt, vf, lane, [&](int g) {   // dP[q][key] - delta[q]
#pragma unroll
        for (int i = g * 16 / NF; i < (g + 1) * 16 / NF; i += 2) {
          s[i] = fast_exp2(__builtin_fmaf(s[i], sl2e, -lse_r[i]));
          s[i + 1] = fast_exp2(__builtin_fmaf(s[i + 1], sl2e, -lse_r[i + 1]));
          if (!interior) s[i] = keep_or_zero(s[i], keep_bits(rm, i)), s[i + 1] = keep_or_zero(s[i + 1], keep_bits(rm, i + 1));
          split_pair(pb[i / 8], (i % 8) / 2, s[i] * kUp, s[i + 1] * kUp);
        }
      });
      mma_tr_split<D, TQ>(dv, Gt, pb, lane, [&](int it) {    // dV^T[d][key] += dO^T P
#pragma unroll
        for (int i = it * 8 / DB; i < (it + 1) * 8 / DB; i += 2) {
          float a = s[i] * dp[i], e = s[i + 1] * dp[i + 1];
          // a masked dP may hold anything (NaN included): P = 0 does not clear it
          if (!interior) a = keep_or_zero(a, keep_bits(rm, i)), e = keep_or_zero(e, keep_bits(rm, i + 1));
          split_pair(sb[i / 8], (i % 8) / 2, a, e);
        }
      });
      mma_tr_split<D, TQ>(dk, Qt, sb, lane);                 // dK^T[d][key] += Q^T dS
    }
    if (more) store_tile(it + 1);
    __syncthreads();
  }

  const bool odd = !all_finite<D>(dk) || !all_finite<D>(dv) || scale_too_small(p.scale_log2e);
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
  store_rows_f32<D, DIRECT>(patch, dk_base + (int64_t)row0 * D, T_ - row0, dk, p.scale * kDown3, lane);
  store_rows_f32<D, DIRECT>(patch, dv_base + (int64_t)row0 * D, T_ - row0, dv, kDown2, lane);
}

}  // namespace sa
