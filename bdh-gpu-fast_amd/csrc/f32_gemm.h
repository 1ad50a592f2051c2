// fp32 tile products on the bf16 matrix cores of gfx950.
//
// An fp32 value times 2^16 is the exact sum of three bf16 values (8 significant
// bits each, every step rounded to nearest even):
//   a' = 2^16 a, p1 = bf16(a'), p2 = bf16(a' - p1), p3 = bf16(a' - p1 - p2).
// The factor lifts fp32's last bit (2^-149) to bf16's (2^-133): without it the
// lower planes of values below 2^-110 fall short (2.5e-6 of the result at
// 2^-116, 6e-4 at 2^-124).  The sums are 2^32 times theirs.
// A product keeps six of the nine plane products,
//   a' b' = p1 q1 + (p1 q2 + p2 q1) + (p1 q3 + p2 q2 + p3 q1) + d,
// all exact in fp32, accumulated in fp32 by v_mfma_f32_32x32x16_bf16.  What is
// dropped, d = p2 q3 + p3 q2 + p3 q3, is at most about 2^-24 of the product
// (|p2| <= 2^-8 |a'|, |p3| <= 2^-17 |a'|); the sum has six accumulator updates
// per 16 k against eight of v_mfma_f32_32x32x2_f32.  Error against 64 bits, the
// fp32 instruction before and this: 4.66e-7 -> 4.06e-7 at B = 8, nh = 4, T = 512,
// N = 8192 (forward), no larger in any shape measured.
//
// Why: the fp32 matrix rate of this chip is 1/16 of its bf16 rate (157
// TFLOP/s against 2.5 PFLOP/s); six bf16 products for one fp32 product still
// leave 2.7 times the fp32 rate.
//
// Infinities, NaN and values from about 2^112 on make the lower planes NaN, so
// every affected sum is NaN; a sum from 2^96 on is an infinity.  A workgroup that finds a sum that is not finite computes its tile
// once more with the fp32 matrix instruction (EXACT), which gives what plain
// fp32 arithmetic gives.
//
// LDS: per stage of 16 k and operand, three planes of [row][16] bf16 (32-byte
// rows, so a 32-row MFMA fragment is one contiguous 1 KB read without bank
// conflicts), two buffers.  The operands go through registers: the raw values
// of the next stage are loaded while the current stage multiplies, and split
// and written to the other buffer among its MFMAs.
#pragma once

#include <type_traits>

#include "common.h"

namespace bdh {

constexpr int kFK = 16;     // k per stage
constexpr float kF32Scale = 65536.f, kF32Unscale = 1.f / (65536.f * 65536.f);  // of an operand; of a sum
constexpr int kF32Valu = 3;  // VALU instructions per MFMA of a stage (f32_interleave)

// Waves WM x WN, each owning MI x NJ blocks of 32 x 32.
template <int WM_, int WN_, int MI_, int NJ_> struct F32Cfg {
  static constexpr int WM = WM_, WN = WN_, MI = MI_, NJ = NJ_;
  static constexpr int NT = 64 * WM * WN;
  static constexpr int TM = WM * MI * 32, TN = WN * NJ * 32;
  // one stage buffer: planes, or (EXACT) fp32 rows of kFK + 1 floats
  static constexpr int kBufA = TM * 32 * 3, kBuf = (TM + TN) * 32 * 3;
  static constexpr int kLds = 2 * kBuf;
  static_assert((kFK + 1) * 4 <= 32 * 3, "fp32 rows fit the planes' space");
};
typedef F32Cfg<2, 4, 4, 2> F32Big;   // 256 x 256, 8 waves, 96 KB
typedef F32Cfg<2, 2, 2, 2> F32Mid;   // 128 x 128, 4 waves, 48 KB
typedef F32Cfg<2, 2, 1, 2> F32Flat;  // 64 x 128, 4 waves, 36 KB

// The three planes of four consecutive k (8 bytes each), times kF32Scale.
__device__ __forceinline__ void f32_split4(const float (&f)[4], u32x2 (&p)[3]) {
  float r[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = f[e] * kF32Scale;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const uint32_t lo = pack_bf2(r[0], r[1]), hi = pack_bf2(r[2], r[3]);
    p[q] = u32x2{lo, hi};
    if (q < 2) {
      r[0] -= __uint_as_float(lo << 16);
      r[1] -= __uint_as_float(lo & 0xffff0000u);
      r[2] -= __uint_as_float(hi << 16);
      r[3] -= __uint_as_float(hi & 0xffff0000u);
    }
  }
}

// Four k values of operand row `row` at k offset kc of the stage into the
// operand's buffer (ROWS rows).
template <bool EXACT, int ROWS>
__device__ __forceinline__ void f32_put4(char* buf, int row, int kc, const float (&f)[4]) {
  if constexpr (EXACT) {
    float* d = reinterpret_cast<float*>(buf) + row * (kFK + 1) + kc;
#pragma unroll
    for (int e = 0; e < 4; ++e) d[e] = f[e];
  } else {
    u32x2 p[3];
    f32_split4(f, p);
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x2*>(buf + q * (ROWS * 32) + row * 32 + kc * 2) = p[q];
  }
}

__device__ __forceinline__ void f32_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ------------------------------------------------------------------------
// Fragments and products of one stage.  a / b: the operands' buffers; the
// block lists say which 32-row blocks of A and B the wave reads.
// ------------------------------------------------------------------------
template <int ROWS> __device__ __forceinline__ bf16x8 f32_frag(const char* buf, int plane, int blk, int lane) {
  return *reinterpret_cast<const bf16x8*>(buf + plane * (ROWS * 32) + blk * 1024 + (lane & 31) * 32 + (lane >> 5) * 16);
}

// Plane pairs from the smallest products to the largest.
constexpr int kF32Pa[6] = {2, 0, 1, 1, 0, 0};
constexpr int kF32Pb[6] = {0, 2, 1, 0, 1, 0};

template <bool EXACT, class C>
__device__ __forceinline__ void f32_mma(const char* a, const char* b, int wm, int wn, int lane,
                                        f32x16 (&acc)[C::MI][C::NJ]) {
  if constexpr (EXACT) {
    const float* fa = reinterpret_cast<const float*>(a) + (wm * C::MI * 32 + (lane & 31)) * (kFK + 1) + (lane >> 5);
    const float* fb = reinterpret_cast<const float*>(b) + (wn * C::NJ * 32 + (lane & 31)) * (kFK + 1) + (lane >> 5);
#pragma unroll 2
    for (int kk = 0; kk < kFK; kk += 2) {
#pragma unroll
      for (int i = 0; i < C::MI; ++i)
#pragma unroll
        for (int j = 0; j < C::NJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i * 32 * (kFK + 1) + kk], fb[j * 32 * (kFK + 1) + kk],
                                                           acc[i][j], 0, 0, 0);
    }
  } else {
    bf16x8 fb[C::NJ][3];
#pragma unroll
    for (int j = 0; j < C::NJ; ++j)
#pragma unroll
      for (int q = 0; q < 3; ++q) fb[j][q] = f32_frag<C::TN>(b, q, wn * C::NJ + j, lane);
    // rows in pairs: four (two for a single row) independent accumulators in turn
    constexpr int G = C::MI >= 2 ? 2 : 1;
#pragma unroll
    for (int i0 = 0; i0 < C::MI; i0 += G) {
      bf16x8 fa[G][3];
#pragma unroll
      for (int i = 0; i < G; ++i)
#pragma unroll
        for (int q = 0; q < 3; ++q) fa[i][q] = f32_frag<C::TM>(a, q, wm * C::MI + i0 + i, lane);
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int i = 0; i < G; ++i)
#pragma unroll
          for (int j = 0; j < C::NJ; ++j)
            acc[i0 + i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][kF32Pa[q]], fb[j][kF32Pb[q]],
                                                                     acc[i0 + i][j], 0, 0, 0);
    }
  }
}

template <class C> __device__ __forceinline__ void f32_zero(f32x16 (&acc)[C::MI][C::NJ]) {
#pragma unroll
  for (int i = 0; i < C::MI; ++i)
#pragma unroll
    for (int j = 0; j < C::NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
}

// Sums that the bf16 planes may have spoiled: NaN, or an infinity that fp32
// products need not reach.
template <int N> __device__ __forceinline__ float f32_largest(const f32x16 (&acc)[N]) {
  float m = 0.f;  // the largest magnitude; NaN if there is one (v_maximum3_f32, two sums each)
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int r = 0; r < 16; r += 2)
      m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(acc[n][r])),
                                        __builtin_fabsf(acc[n][r + 1]));
  return m;
}
template <int N> __device__ __forceinline__ bool f32_spoiled(const f32x16 (&acc)[N]) {
  return !(f32_largest(acc) <= 3.40282347e+38f);
}
template <int M, int N> __device__ __forceinline__ bool f32_spoiled(const f32x16 (&acc)[M][N]) {
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < M; ++i) m = __builtin_elementwise_maximum(m, f32_largest(acc[i]));
  return !(m <= 3.40282347e+38f);
}

// Among the MFMAs of a stage, the VALU work of staging the next one: without
// these the compiler puts it all behind the last MFMA.  N MFMAs, V VALU
// instructions after each.
template <int N, int V> __device__ __forceinline__ void f32_interleave() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
  }
}

// Main loop over k in [kb, ke), stages of kFK from kb.  Loads past the last
// stage wrap round (into a buffer that nobody reads), so every stage runs the
// same code.  off: the stage to begin with (the k order of the sum).  Safe to call again after itself (its first barrier waits for
// the readers of the buffers).  BISA: the A rows are the B operand too.  ACT:
// whether this wave multiplies (it stages either way).  V: VALU instructions
// per MFMA, by kernel (2, 3, 4, 5 at B = 2, nh = 4, T = 387, N = 8192, in us:
// scores 108, 106, 107, 103; score x V 26.0, 25.7, 28.1, 28.4; G 28.0, 28.3,
// 26.4, 27.7; dQ 185, 187, 173, 187).
template <bool EXACT, class C, bool BISA = false, bool ACT = true, int V = kF32Valu, class LA, class LB>
__device__ __forceinline__ void f32_loop(char* lds, LA& la, LB& lb, int kb, int ke, int wm, int wn, int lane,
                                         f32x16 (&acc)[C::MI][C::NJ], int off = 0) {
  if (kb >= ke) return;
  const int n = (ke - kb + kFK - 1) / kFK;
  auto step = [&](int s) { return s + 1 == n ? 0 : s + 1; };
  int s1 = off, s2 = step(off);
  la.load(kb + s1 * kFK);
  if constexpr (!BISA) lb.load(kb + s1 * kFK);
  f32_barrier();
  la.template store<EXACT>(lds, kb + s1 * kFK);
  if constexpr (!BISA) lb.template store<EXACT>(lds + C::kBufA, kb + s1 * kFK);
  la.load(kb + s2 * kFK);
  if constexpr (!BISA) lb.load(kb + s2 * kFK);
  f32_barrier();
  int cur = 0;
  for (int i = 0; i < n; ++i) {
    const char* a = lds + cur * C::kBuf;
    char* nx = lds + (cur ^ 1) * C::kBuf;
    s1 = s2;
    s2 = step(s2);
    if constexpr (ACT) f32_mma<EXACT, C>(a, BISA ? a : a + C::kBufA, wm, wn, lane, acc);
    la.template store<EXACT>(nx, kb + s1 * kFK);
    if constexpr (!BISA) lb.template store<EXACT>(nx + C::kBufA, kb + s1 * kFK);
    if constexpr (ACT && !EXACT) f32_interleave<6 * C::MI * C::NJ, V>();
    la.load(kb + s2 * kFK);
    if constexpr (!BISA) lb.load(kb + s2 * kFK);
    f32_barrier();
    cur ^= 1;
  }
}

// Whether any thread of the workgroup passed true (every wave calls it).
__device__ __forceinline__ bool f32_any(bool mine, int* flag) {
  f32_barrier();  // the previous readers of *flag are done
  if (threadIdx.x == 0) *flag = 0;
  f32_barrier();
  if (__any(mine)) *flag = 1;
  f32_barrier();
  return *flag != 0;
}

// ------------------------------------------------------------------------
// K-form loader: operand row r is a row of a matrix, k contiguous (rows of
// x, q, k; G; score tiles).  Rows outside [rlo, nrows) read the nearest row
// inside: their sums belong to no output.  k >= K reads zero.  ROPE rotates
// adjacent k pairs at position pos0 + row.  MASK 1 keeps k < row, 2 k > row.
// ------------------------------------------------------------------------
template <typename TIn, bool ROPE, int MASK, int ROWS, int NT, bool QR = false> struct F32Rows {
  static constexpr int CPT = ROWS * 4 / NT;  // 4-value chunks per thread: rows NT / 4 apart, one k offset
  const TIn* base = nullptr;
  int64_t rs = 0;
  int r0 = 0, nrows = 0, rlo = 0;
  int K = 0;
  bool vec = false;  // 4-value aligned rows
  const float* freqs = nullptr;
  float pos0 = 0.f;
  void* qr = nullptr;  // QR: copy of the rotated rows
  int64_t qr_rs = 0;
  bool qr_bf = false, qr_vec = false;  // qr_vec: 4-value aligned rows

  TIn v[CPT][4];
  float fq[2];

  F32Rows() = default;
  // The operand of o (QR may differ).
  template <bool Q> __device__ __forceinline__ explicit F32Rows(const F32Rows<TIn, ROPE, MASK, ROWS, NT, Q>& o)
      : base(o.base), rs(o.rs), r0(o.r0), nrows(o.nrows), rlo(o.rlo), K(o.K), vec(o.vec), freqs(o.freqs), pos0(o.pos0) {}

  __device__ __forceinline__ int row(int c) const { return int(threadIdx.x >> 2) + c * (NT / 4); }
  __device__ __forceinline__ int kc() const { return int(threadIdx.x & 3) * 4; }

  __device__ __forceinline__ void load(int k0) {
    const int gk = k0 + kc();
    if (vec && k0 + kFK <= K) {
#pragma unroll
      for (int c = 0; c < CPT; ++c) {
        const int gr = min(max(r0 + row(c), rlo), nrows - 1);
        const TIn* p = base + int64_t(gr - rlo) * rs + gk;
        if constexpr (sizeof(TIn) == 4)
          *reinterpret_cast<uint4*>(v[c]) = *reinterpret_cast<const uint4*>(p);
        else
          *reinterpret_cast<uint2*>(v[c]) = *reinterpret_cast<const uint2*>(p);
      }
      if constexpr (ROPE) {
        fq[0] = freqs[gk];
        fq[1] = freqs[gk + 2];
      }
    } else {
#pragma unroll
      for (int c = 0; c < CPT; ++c) {
        const int gr = min(max(r0 + row(c), rlo), nrows - 1);
        const TIn* p = base + int64_t(gr - rlo) * rs + gk;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[c][e] = gk + e < K ? p[e] : TIn(0);
      }
      if constexpr (ROPE) {
        fq[0] = gk < K ? freqs[gk] : 0.f;
        fq[1] = gk + 2 < K ? freqs[gk + 2] : 0.f;
      }
    }
  }

  template <bool EXACT> __device__ __forceinline__ void store(char* dst, int k0) {
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      const int gr = r0 + row(c), gk = k0 + kc();
      float f[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] = to_f(v[c][e]);
      if constexpr (ROPE) {
        const float pos = pos0 + float(gr);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float cs, sn;
          rope_cs(pos, fq[q], cs, sn);
          const float x0 = f[2 * q], x1 = f[2 * q + 1];
          f[2 * q] = x0 * cs - x1 * sn;
          f[2 * q + 1] = x1 * cs + x0 * sn;
        }
        if constexpr (QR)
          if (gr < nrows) put_qr(gr, gk, f);
      }
      if constexpr (MASK == 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (!(gk + e < gr)) f[e] = 0.f;
      } else if constexpr (MASK == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (!(gk + e > gr)) f[e] = 0.f;
      }
      f32_put4<EXACT, ROWS>(dst, row(c), kc(), f);
    }
  }

  __device__ __forceinline__ void put_qr(int gr, int gk, const float (&f)[4]) const {
    if (qr_bf) {
      bf16_t* o = reinterpret_cast<bf16_t*>(qr) + int64_t(gr) * qr_rs + gk;
      if (qr_vec && gk + 4 <= K) {
        *reinterpret_cast<u32x2*>(o) = u32x2{pack_bf2(f[0], f[1]), pack_bf2(f[2], f[3])};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (gk + e < K) o[e] = f2bf(f[e]);
      }
    } else {
      float* o = reinterpret_cast<float*>(qr) + int64_t(gr) * qr_rs + gk;
      if (qr_vec && gk + 4 <= K) {
        *reinterpret_cast<f32x4*>(o) = f32x4{f[0], f[1], f[2], f[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (gk + e < K) o[e] = f[e];
      }
    }
  }
};

// ------------------------------------------------------------------------
// N-form loader: operand row n is a column of a [k][n] matrix (n contiguous;
// V, dO, X).  A thread takes two adjacent columns at four consecutive k;
// sixteen lanes read 128 consecutive bytes of fp32, and the lanes of a wave
// write their 8-byte pieces to LDS without bank conflicts.  k >= krows reads
// zero; columns >= ncols read the last ones (their sums belong to no output).  ROPE rotates the column pair at position pos0 + k.
// ------------------------------------------------------------------------
template <typename TIn, bool ROPE, int ROWS, int NT> struct F32Cols {
  static_assert(ROWS * kFK == 8 * NT || ROWS * kFK == 4 * NT, "one or half a unit per thread");
  static constexpr bool HALF = ROWS * kFK == 4 * NT;  // only the first half of the threads has a unit
  const TIn* base = nullptr;
  int64_t rs = 0;
  int n0 = 0, ncols = 0, krows = 0;
  bool vec = false;  // 2-value aligned rows
  const float* freqs = nullptr;
  float pos0 = 0.f;

  TIn v[4][2];
  float fq;

  __device__ __forceinline__ int col() const { return 2 * (int(threadIdx.x & 15) + 16 * int(threadIdx.x >> 6)); }
  __device__ __forceinline__ int kc() const { return int((threadIdx.x >> 4) & 3) * 4; }
  __device__ __forceinline__ bool mine() const { return !HALF || threadIdx.x < NT / 2; }

  __device__ __forceinline__ void load(int k0) {
    if (!mine()) return;
    const int gn = n0 + col();
    if (vec && k0 + kFK <= krows) {
      const int gc = min(gn, ncols - 2);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const TIn* p = base + int64_t(k0 + kc() + e) * rs + gc;
        if constexpr (sizeof(TIn) == 4)
          *reinterpret_cast<uint2*>(v[e]) = *reinterpret_cast<const uint2*>(p);
        else
          *reinterpret_cast<uint32_t*>(v[e]) = *reinterpret_cast<const uint32_t*>(p);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int gk = k0 + kc() + e;
        const TIn* p = base + int64_t(gk) * rs + gn;
#pragma unroll
        for (int x = 0; x < 2; ++x) v[e][x] = (gk < krows && gn + x < ncols) ? p[x] : TIn(0);
      }
    }
    if constexpr (ROPE) fq = gn < ncols ? freqs[gn] : 0.f;
  }

  template <bool EXACT> __device__ __forceinline__ void store(char* dst, int k0) {
    if (!mine()) return;
    float f[2][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x0 = to_f(v[e][0]), x1 = to_f(v[e][1]);
      if constexpr (ROPE) {
        float cs, sn;
        rope_cs(pos0 + float(k0 + kc() + e), fq, cs, sn);
        const float y0 = x0 * cs - x1 * sn;
        x1 = x1 * cs + x0 * sn;
        x0 = y0;
      }
      f[0][e] = x0;
      f[1][e] = x1;
    }
#pragma unroll
    for (int x = 0; x < 2; ++x) f32_put4<EXACT, ROWS>(dst, col() + x, kc(), f[x]);
  }
};

// ------------------------------------------------------------------------
// The masked score matrix M = tril(S, -1) of one slab in packed lower tiles
// of TE x TE floats, row-major inside a tile (tiles from packed index t0 on).
// ------------------------------------------------------------------------
__device__ __forceinline__ int f32_tile_index(int ti, int tj) { return ti * (ti + 1) / 2 + tj; }

// Rows of M as the A operand (k = column): rows r0 .. r0 + ROWS of one row of tiles.
template <int ROWS, int NT> struct F32MRows : F32Rows<float, false, 0, ROWS, NT> {
  typedef F32Rows<float, false, 0, ROWS, NT> Base;
  const float* slab = nullptr;
  int te_log = 0, t0 = 0;  // tile edge 1 << te_log
  __device__ __forceinline__ void load(int k0) {
    const int te = 1 << te_log, ti = this->r0 >> te_log, tj = k0 >> te_log;
    const float* t = slab + (int64_t(f32_tile_index(ti, tj) - t0) << (2 * te_log));
    const int rin = this->r0 & (te - 1), kin = (k0 & (te - 1)) + this->kc();
#pragma unroll
    for (int c = 0; c < Base::CPT; ++c)
      *reinterpret_cast<uint4*>(this->v[c]) =
          *reinterpret_cast<const uint4*>(t + ((rin + this->row(c)) << te_log) + kin);
  }
};

// Columns of M as the A operand (k = row): columns n0 .. n0 + ROWS of one column of tiles.
template <int ROWS, int NT> struct F32MCols : F32Cols<float, false, ROWS, NT> {
  const float* slab = nullptr;
  int te_log = 0, t0 = 0;
  __device__ __forceinline__ void load(int k0) {
    if (!this->mine()) return;
    const int te = 1 << te_log, ti = k0 >> te_log, tj = this->n0 >> te_log;
    const float* t = slab + (int64_t(f32_tile_index(ti, tj) - t0) << (2 * te_log));
    const int kin = (k0 & (te - 1)) + this->kc(), nin = (this->n0 & (te - 1)) + this->col();
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *reinterpret_cast<uint2*>(this->v[e]) = *reinterpret_cast<const uint2*>(t + ((kin + e) << te_log) + nin);
  }
};

// Tile-relative coordinates of register r of block (i, j).
__device__ __forceinline__ int f32_row(int blk, int lane, int r) { return blk * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }
__device__ __forceinline__ int f32_col(int blk, int lane) { return blk * 32 + (lane & 31); }

}  // namespace bdh
