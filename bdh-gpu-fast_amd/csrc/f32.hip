// fp32 strict-tril attention for gfx950, forward and backward, on the bf16
// matrix cores (f32_gemm.h: three bf16 planes per operand, six products).
//
//   out[b,h,i,:] = sum_{j<i} <Q_i, K_j> V_j,   optionally Q = K = RoPE(x)
//
// Forward:
//  1. k_f32_scores (T > 128) / k_f32_scores_mid: M = tril(Q K^T, -1) in
//     packed lower tiles, split over N; RoPE applied as rows are staged.
//  2. k_f32_msum: the splits' partial tiles added up (more than one split).
//  3. k_f32_sv: out = M V.
// Backward:
//  1. M as above; k_f32_dv: dV = sum_h M^T dO.
//  2. k_f32_g: G = dS + dS^T, dS = tril(dO V^T, -1).
//  3. k_f32_dq: dQ = G X (self attention; with RoPE X is rotated as it is
//     staged and the transpose rotation is applied to the sums), or
//     lower(G) K and upper(G) Q.
#include <algorithm>

#include "f32_gemm.h"
#include "fwd.h"

namespace bdh {
namespace {

// ------------------------------------------------------------------ scores
constexpr int kF32ScoresValu = 5;  // (f32_loop's V)
enum : int { kF32Full = 0, kF32Diag2 = 1, kF32Diag1 = 2 };

struct F32ScoresArgs {
  View q, k;
  int64_t H;
  int T, K, past;
  int q_is_k;
  bool vec_q, vec_k;
  const float* freqs;
  int64_t rope_start;
  float* m;        // [split][slab][tile - t0][TE * TE]
  int64_t split_stride;
  int kc;          // k extent of one split
  int nsplit, nslab, ntl, t0, s0, nt;
  int nfull, per;  // full tiles and work items of one split of a slab
  View qr;
  bool qr_bf, qr_vec;
};

// A wave's 9 of the 36 lower blocks of a diagonal 256 x 256 tile: the row
// blocks it reads (f) and its blocks as pairs of indices into them.
template <int P> struct DiagProg;
template <> struct DiagProg<0> {  // rows 5-7 x columns 0-2
  static constexpr int NF = 6, f[6] = {0, 1, 2, 5, 6, 7};
  static constexpr int r[9] = {3, 3, 3, 4, 4, 4, 5, 5, 5}, c[9] = {0, 1, 2, 0, 1, 2, 0, 1, 2};
};
template <> struct DiagProg<1> {  // rows 3-4 x columns 0-2 and their own triangle
  static constexpr int NF = 5, f[5] = {0, 1, 2, 3, 4};
  static constexpr int r[9] = {3, 3, 3, 4, 4, 4, 3, 4, 4}, c[9] = {0, 1, 2, 0, 1, 2, 3, 3, 4};
};
template <> struct DiagProg<2> {  // rows 5-7 x columns 3-4, triangle 5-6
  static constexpr int NF = 5, f[5] = {3, 4, 5, 6, 7};
  static constexpr int r[9] = {2, 2, 3, 3, 4, 4, 2, 3, 3}, c[9] = {0, 1, 0, 1, 0, 1, 2, 2, 3};
};
template <> struct DiagProg<3> {  // triangle 0-2, row 7 x columns 5-7
  static constexpr int NF = 6, f[6] = {0, 1, 2, 5, 6, 7};
  static constexpr int r[9] = {0, 1, 1, 2, 2, 2, 5, 5, 5}, c[9] = {0, 0, 1, 0, 1, 2, 3, 4, 5};
};

template <bool EXACT, class P>
__device__ __forceinline__ void diag_mma(const char* a, int lane, f32x16 (&acc)[9]) {
  if constexpr (EXACT) {
    const float* fa = reinterpret_cast<const float*>(a) + (lane & 31) * (kFK + 1) + (lane >> 5);
#pragma unroll 2
    for (int kk = 0; kk < kFK; kk += 2) {
      float x[P::NF];
#pragma unroll
      for (int n = 0; n < P::NF; ++n) x[n] = fa[P::f[n] * 32 * (kFK + 1) + kk];
#pragma unroll
      for (int n = 0; n < 9; ++n)
        acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[P::r[n]], x[P::c[n]], acc[n], 0, 0, 0);
    }
  } else {
    bf16x8 fr[3][P::NF];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int n = 0; n < P::NF; ++n) fr[q][n] = f32_frag<256>(a, q, P::f[n], lane);
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int n = 0; n < 9; ++n)
        acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[kF32Pa[q]][P::r[n]], fr[kF32Pb[q]][P::c[n]], acc[n], 0,
                                                         0, 0);
  }
}

// The loop of f32_loop with the diagonal programs: la / lb stage the rows of
// the two diagonal tiles, this wave multiplies those at `mine`.  ONE: the
// same tile's rows 16 k apart, each half of the waves summing every other
// stage.
template <bool EXACT, bool ONE, class P, class L>
__device__ __forceinline__ void diag_loop(char* lds, L& la, L& lb, int kb, int ke, int off, int mine, int lane,
                                          f32x16 (&acc)[9]) {
  if (kb >= ke) return;
  constexpr int STEP = ONE ? 2 * kFK : kFK, OFF = ONE ? kFK : 0;
  const int n = (ke - kb + STEP - 1) / STEP;
  auto step = [&](int s) { return s + 1 == n ? 0 : s + 1; };
  int s1 = ONE ? off / 2 : off, s2 = step(s1);
  la.load(kb + s1 * STEP);
  lb.load(kb + s1 * STEP + OFF);
  f32_barrier();
  la.template store<EXACT>(lds, kb + s1 * STEP);
  lb.template store<EXACT>(lds + F32Big::kBufA, kb + s1 * STEP + OFF);
  la.load(kb + s2 * STEP);
  lb.load(kb + s2 * STEP + OFF);
  f32_barrier();
  int cur = 0;
  for (int i = 0; i < n; ++i) {
    char* nx = lds + (cur ^ 1) * F32Big::kBuf;
    s1 = s2;
    s2 = step(s2);
    diag_mma<EXACT, P>(lds + cur * F32Big::kBuf + mine, lane, acc);
    la.template store<EXACT>(nx, kb + s1 * STEP);
    lb.template store<EXACT>(nx + F32Big::kBufA, kb + s1 * STEP + OFF);
    if constexpr (!EXACT) f32_interleave<54, kF32ScoresValu>();
    la.load(kb + s2 * STEP);
    lb.load(kb + s2 * STEP + OFF);
    f32_barrier();
    cur ^= 1;
  }
}

template <bool ONE, class P, class L>
__device__ __forceinline__ void diag_item(char* lds, int* flag, L& la, L& lb, int kb, int ke, int off, int wave, int lane,
                                          float* tile, int r0, int T) {
  const int half = wave >> 2;
  f32x16 acc[9];
  auto run = [&](auto exact) {
#pragma unroll
    for (int n = 0; n < 9; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
    diag_loop<decltype(exact)::value, ONE, P>(lds, la, lb, kb, ke, off, half * F32Big::kBufA, lane, acc);
  };
  run(std::false_type{});
  float us = kF32Unscale;
  if (f32_any(f32_spoiled(acc), flag)) {
    run(std::true_type{});
    us = 1.f;
  }
  if constexpr (ONE) {  // the second half's sums through LDS, three blocks at a time
    f32x4* x = reinterpret_cast<f32x4*>(lds) + ((wave & 3) * 3 * 4 * 64 + lane);
#pragma unroll
    for (int n0 = 0; n0 < 9; n0 += 3) {
      f32_barrier();
      if (half) {
#pragma unroll
        for (int n = 0; n < 3; ++n)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            x[(n * 4 + r) * 64] = f32x4{acc[n0 + n][4 * r], acc[n0 + n][4 * r + 1], acc[n0 + n][4 * r + 2], acc[n0 + n][4 * r + 3]};
      }
      f32_barrier();
      if (!half) {
#pragma unroll
        for (int n = 0; n < 3; ++n)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const f32x4 w = x[(n * 4 + r) * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[n0 + n][4 * r + e] += w[e];
          }
      }
    }
    if (half) return;
  }
#pragma unroll
  for (int n = 0; n < 9; ++n) {
    const int rb = P::f[P::r[n]], cb = P::f[P::c[n]];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = f32_row(rb, lane, r), col = f32_col(cb, lane);
      tile[row * 256 + col] = (row > col && r0 + row < T) ? acc[n][r] * us : 0.f;
    }
  }
}

template <bool ONE, class L>
__device__ __forceinline__ void diag_waves(char* lds, int* flag, L& la, L& lb, int kb, int ke, int off, int wave, int lane,
                                           float* tile, int r0, int T) {
  switch (wave & 3) {
    case 0: diag_item<ONE, DiagProg<0>>(lds, flag, la, lb, kb, ke, off, wave, lane, tile, r0, T); break;
    case 1: diag_item<ONE, DiagProg<1>>(lds, flag, la, lb, kb, ke, off, wave, lane, tile, r0, T); break;
    case 2: diag_item<ONE, DiagProg<2>>(lds, flag, la, lb, kb, ke, off, wave, lane, tile, r0, T); break;
    default: diag_item<ONE, DiagProg<3>>(lds, flag, la, lb, kb, ke, off, wave, lane, tile, r0, T); break;
  }
}

// 256 x 256 tiles.  Bound by the matrix cores beside the staging's VALU work
// (split, and RoPE's sine and cosine): per 16 k a wave issues 48 MFMAs of 32
// clocks (54 on a diagonal pair) and about 180 VALU instructions, so the tile
// is as large as two waves per SIMD allow, and the two diagonal tiles of a
// pair share a workgroup (with Q = K each needs its rows once).  B = 8, nh =
// 4, T = 512, N = 8192 with RoPE: 350-390 us by box (the fp32 matrix
// instruction on 128 x 128 tiles: 1160 us); without the loop's loads 289,
// without RoPE's sine and cosine 360, with one of the six products 205.
template <bool ROPE, bool QR>
__global__ __launch_bounds__(512, 2) void k_f32_scores(F32ScoresArgs a) {
  __shared__ __attribute__((aligned(1024))) char f32_lds[F32Big::kLds];
  __shared__ int flag;
  // (slab, split) groups on one XCD each (workgroup id % 8): the items of a
  // group read the same rows
  const int x = int(blockIdx.x) & 7, rest = int(blockIdx.x) >> 3;
  const int grp = rest / a.per * 8 + x;
  int it = rest % a.per;
  if (grp >= a.nslab * a.nsplit) return;
  const int slab = grp / a.nsplit, split = grp % a.nsplit;
  const int b = slab / int(a.H), h = slab % int(a.H);
  const int kb = split * a.kc, ke = min(a.K, kb + a.kc);
  const int ns = (ke - kb + kFK - 1) / kFK;
  // rows lie a power of two apart, so one k offset falls on few memory
  // channels: the groups start at evenly spread stages (B = 8, nh = 4, T =
  // 512, N = 8192: 414 -> 349 us against all starting at the first)
  const int off = int(int64_t(grp) * ns / (a.nslab * a.nsplit));
  int ta, tb, kind;
  if (it < a.nfull) {
    int t = a.s0, n = a.q_is_k ? t : t + 1;
    while (it >= n) {
      it -= n;
      ++t;
      n = a.q_is_k ? t : t + 1;
    }
    ta = t;
    tb = it;
    kind = kF32Full;
  } else {
    ta = a.s0 + 2 * (it - a.nfull);
    tb = min(ta + 1, a.nt - 1);
    kind = tb == ta ? kF32Diag1 : kF32Diag2;
  }
  F32Rows<float, ROPE, 0, 256, 512> la, lb;
  la.base = static_cast<const float*>(a.q.p) + b * a.q.s0 + h * a.q.s1;
  la.rs = a.q.s2;
  la.r0 = ta * 256;
  la.nrows = a.T;
  la.rlo = a.past;
  la.K = a.K;
  la.vec = a.vec_q;
  lb.base = static_cast<const float*>(a.k.p) + b * a.k.s0 + h * a.k.s1;
  lb.rs = a.k.s2;
  lb.r0 = tb * 256;
  lb.nrows = a.T;
  lb.K = a.K;
  lb.vec = a.vec_k;
  if constexpr (ROPE) {
    la.freqs = lb.freqs = a.freqs;
    la.pos0 = lb.pos0 = float(a.rope_start);
  }
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  float* out = a.m + split * a.split_stride + int64_t(slab) * a.ntl * 65536;
  if (kind == kF32Full) {
    const int wm = wave >> 2, wn = wave & 3;
    f32x16 acc[4][2];
    f32_zero<F32Big>(acc);
    f32_loop<false, F32Big, false, true, kF32ScoresValu>(f32_lds, la, lb, kb, ke, wm, wn, lane, acc, off);
    float us = kF32Unscale;
    if (f32_any(f32_spoiled(acc), &flag)) {
      f32_zero<F32Big>(acc);
      f32_loop<true, F32Big>(f32_lds, la, lb, kb, ke, wm, wn, lane, acc, off);
      us = 1.f;
    }
    float* tile = out + int64_t(f32_tile_index(ta, tb) - a.t0) * 65536;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = f32_row(wm * 4 + i, lane, r), col = f32_col(wn * 2 + j, lane);
          const int gi = ta * 256 + row;
          tile[row * 256 + col] = (tb * 256 + col < gi && gi < a.T) ? acc[i][j][r] * us : 0.f;
        }
    return;
  }
  const int half = wave >> 2, t = half ? tb : ta;
  float* tile = out + int64_t(f32_tile_index(t, t) - a.t0) * 65536;
  // the blocks above the diagonal: read by the products that follow
  if (half == 0 || kind == kF32Diag2)
    for (int e = (wave & 3) * 64 + lane; e < 256 * 64; e += 256) {
      const int row = e >> 6, c4 = (e & 63) * 4;
      if ((c4 >> 5) > (row >> 5)) *reinterpret_cast<f32x4*>(tile + row * 256 + c4) = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  // every row is in one diagonal tile, which writes its RoPE(x) copy
  F32Rows<float, ROPE, 0, 256, 512, QR> da(la), db(lb);
  if constexpr (QR) {
    da.qr = db.qr = const_cast<char*>(static_cast<const char*>(a.qr.p)) + (b * a.qr.s0 + h * a.qr.s1) * (a.qr_bf ? 2 : 4);
    da.qr_rs = db.qr_rs = a.qr.s2;
    da.qr_bf = db.qr_bf = a.qr_bf;
    da.qr_vec = db.qr_vec = a.qr_vec;
  }
  if (kind == kF32Diag2)
    diag_waves<false>(f32_lds, &flag, da, db, kb, ke, off, wave, lane, tile, t * 256, a.T);
  else {
    da.K = db.K = ke;  // an odd count of stages ends with one of zeros
    diag_waves<true>(f32_lds, &flag, da, db, kb, ke, off, wave, lane, tile, t * 256, a.T);
  }
}

// T <= 128: one 128 x 128 tile per slab and split.  Short: bound by the latency
// of a split's few stages (B = 2, nh = 4, T = 100, N = 1024: 10.9 us on the
// fp32 instruction, 9.2 here).
template <bool ROPE, bool QR>
__global__ __launch_bounds__(256, 2) void k_f32_scores_mid(F32ScoresArgs a) {
  __shared__ __attribute__((aligned(1024))) char f32_lds[F32Mid::kLds];
  __shared__ int flag;
  const int slab = int(blockIdx.x), split = int(blockIdx.y);
  const int b = slab / int(a.H), h = slab % int(a.H);
  const int kb = split * a.kc, ke = min(a.K, kb + a.kc);
  F32Rows<float, ROPE, 0, 128, 256, QR> la;
  F32Rows<float, ROPE, 0, 128, 256> lb;
  la.base = static_cast<const float*>(a.q.p) + b * a.q.s0 + h * a.q.s1;
  la.rs = a.q.s2;
  la.nrows = a.T;
  la.rlo = a.past;
  la.K = a.K;
  la.vec = a.vec_q;
  lb.base = static_cast<const float*>(a.k.p) + b * a.k.s0 + h * a.k.s1;
  lb.rs = a.k.s2;
  lb.nrows = a.T;
  lb.K = a.K;
  lb.vec = a.vec_k;
  if constexpr (ROPE) {
    la.freqs = lb.freqs = a.freqs;
    la.pos0 = lb.pos0 = float(a.rope_start);
    if constexpr (QR) {
      la.qr = const_cast<char*>(static_cast<const char*>(a.qr.p)) + (b * a.qr.s0 + h * a.qr.s1) * (a.qr_bf ? 2 : 4);
      la.qr_rs = a.qr.s2;
      la.qr_bf = a.qr_bf;
      la.qr_vec = a.qr_vec;
    }
  }
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1;
  f32x16 acc[2][2];
  auto run = [&](auto exact) {
    constexpr bool E = decltype(exact)::value;
    f32_zero<F32Mid>(acc);
    if (wm == 0 && wn == 1) {  // rows 0-63 x columns 64-127: above the diagonal
      if (a.q_is_k)
        f32_loop<E, F32Mid, true, false>(f32_lds, la, lb, kb, ke, wm, wn, lane, acc);
      else
        f32_loop<E, F32Mid, false, false>(f32_lds, la, lb, kb, ke, wm, wn, lane, acc);
    } else {
      if (a.q_is_k)
        f32_loop<E, F32Mid, true>(f32_lds, la, lb, kb, ke, wm, wn, lane, acc);
      else
        f32_loop<E, F32Mid>(f32_lds, la, lb, kb, ke, wm, wn, lane, acc);
    }
  };
  run(std::false_type{});
  float us = kF32Unscale;
  if (f32_any(f32_spoiled(acc), &flag)) {
    run(std::true_type{});
    us = 1.f;
  }
  float* tile = a.m + split * a.split_stride + int64_t(slab) * kTileElems;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = f32_row(wm * 2 + i, lane, r), col = f32_col(wn * 2 + j, lane);
        tile[row * 128 + col] = (row > col && row < a.T) ? acc[i][j][r] * us : 0.f;
      }
}

// The splits' partial tiles added into the first: a stream, four values a
// thread and four splits in flight (bound by memory: 17-19 us at B = 8, nh = 4,
// T = 512, which saves the splits' cost in every reader of M).
__global__ __launch_bounds__(256) void k_f32_msum(float* m, int64_t n4, int64_t stride4, int nsplit) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n4) return;
  f32x4* p = reinterpret_cast<f32x4*>(m) + i;
  f32x4 s = p[0];
  int n = 1;
  for (; n + 4 <= nsplit; n += 4) {
    const f32x4 w0 = p[n * stride4], w1 = p[(n + 1) * stride4], w2 = p[(n + 2) * stride4], w3 = p[(n + 3) * stride4];
    s += w0;
    s += w1;
    s += w2;
    s += w3;
  }
  for (; n < nsplit; ++n) s += p[n * stride4];
  p[0] = s;
}

// --------------------------------------------------------------- score x V
struct F32SvArgs {
  const float* m;
  int te_log, ntl, t0;
  View v, o;
  int64_t H, Hv;
  int T, Dv, past, R0, nR;  // row tiles of 64: R0 .. R0 + nR
  bool vec_v;
};

// 64 rows x 128 columns: the grid has few tiles (a row of tiles per 64
// tokens), so a small one spreads over more CUs; longest rows first.  Bound by
// the longest row's serial chain of stages: B = 8, T = 512, D = 256: 134 -> 48
// us; B = 2, T = 387: 196 -> 24 us (128 x 128 tiles of the fp32 instruction
// before).
template <typename TV, typename TO>
__global__ __launch_bounds__(256, 2) void k_f32_sv(F32SvArgs a) {
  __shared__ __attribute__((aligned(1024))) char f32_lds[F32Flat::kLds];
  __shared__ int flag;
  const int R = a.R0 + a.nR - 1 - int(blockIdx.x), Dt = blockIdx.y, slab = blockIdx.z;
  const int b = slab / int(a.H), h = slab % int(a.H);
  const int hv = a.Hv == 1 ? 0 : h;
  F32MRows<64, 256> la;
  la.slab = a.m + (int64_t(slab) * a.ntl << (2 * a.te_log));
  la.te_log = a.te_log;
  la.t0 = a.t0;
  la.r0 = R * 64;
  F32Cols<TV, false, 128, 256> lb;
  lb.base = static_cast<const TV*>(a.v.p) + b * a.v.s0 + hv * a.v.s1;
  lb.rs = a.v.s2;
  lb.n0 = Dt * 128;
  lb.ncols = a.Dv;
  lb.krows = a.T;
  lb.vec = a.vec_v;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1;
  const int ke = min(a.T, R * 64 + 64);
  f32x16 acc[1][2];
  f32_zero<F32Flat>(acc);
  f32_loop<false, F32Flat>(f32_lds, la, lb, 0, ke, wm, wn, lane, acc);
  float us = kF32Unscale;
  if (f32_any(f32_spoiled(acc), &flag)) {
    f32_zero<F32Flat>(acc);
    f32_loop<true, F32Flat>(f32_lds, la, lb, 0, ke, wm, wn, lane, acc);
    us = 1.f;
  }
  TO* o = static_cast<TO*>(const_cast<void*>(a.o.p)) + b * a.o.s0 + h * a.o.s1;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int gi = R * 64 + f32_row(wm, lane, r), gd = Dt * 128 + f32_col(wn * 2 + j, lane);
      if (gi >= a.past && gi < a.T && gd < a.Dv) o[int64_t(gi - a.past) * a.o.s2 + gd] = from_f<TO>(acc[0][j][r] * us);
    }
}

// ------------------------------------------------------------------ dV
struct F32DvArgs {
  const float* m;
  int te_log, ntl;
  View dO, o;
  int64_t H, Hv;
  int T, Dv;
  int parts;    // pieces the (head, 64-row chunk) list of a tile is dealt into
  float* part;  // [part][b * Hv + hv][T][Dv] (parts > 1)
  bool vec_do;
};

// dV of 64 rows x 128 columns: sum over the heads of M^T dO, contracted over
// the rows i >= j0 in 64-row chunks.  The (head, chunk) list of a tile is
// cut into `parts` pieces so that a small batch still fills the chip (their
// sums go to `part`, added up by k_f32_dvsum in piece order).  B = 2, nh = 4, T
// = 387, D = 256: 897 us on 16 workgroups of the fp32 instruction, 20 us here.
template <typename TDO, typename TO>
__global__ __launch_bounds__(256, 2) void k_f32_dv(F32DvArgs a) {
  __shared__ __attribute__((aligned(1024))) char f32_lds[F32Flat::kLds];
  __shared__ int flag;
  const int R = blockIdx.x / a.parts, piece = blockIdx.x % a.parts, Dt = blockIdx.y, bv = blockIdx.z;
  const int b = bv / int(a.Hv), hv = bv % int(a.Hv);
  const int h_lo = a.Hv == 1 ? 0 : hv, nh = a.Hv == 1 ? int(a.H) : 1;
  const int nc = (a.T + 63) / 64 - R;  // chunks per head
  const int i0 = int(int64_t(nh) * nc * piece / a.parts), i1 = int(int64_t(nh) * nc * (piece + 1) / a.parts);
  F32MCols<64, 256> la;
  la.te_log = a.te_log;
  la.n0 = R * 64;
  F32Cols<TDO, false, 128, 256> lb;
  lb.rs = a.dO.s2;
  lb.n0 = Dt * 128;
  lb.ncols = a.Dv;
  lb.krows = a.T;
  lb.vec = a.vec_do;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1;
  f32x16 acc[1][2];
  auto run = [&](auto exact) {
    f32_zero<F32Flat>(acc);
    for (int i = i0; i < i1;) {  // the chunks of one head at a time
      const int hh = i / nc, c0 = i % nc, c1 = min(nc, c0 + i1 - i);
      const int slab = b * int(a.H) + h_lo + hh;
      la.slab = a.m + (int64_t(slab) * a.ntl << (2 * a.te_log));
      lb.base = static_cast<const TDO*>(a.dO.p) + b * a.dO.s0 + (h_lo + hh) * a.dO.s1;
      f32_loop<decltype(exact)::value, F32Flat>(f32_lds, la, lb, (R + c0) * 64, min(a.T, (R + c1) * 64), wm, wn, lane,
                                                acc);
      i += c1 - c0;
    }
  };
  run(std::false_type{});
  float us = kF32Unscale;
  if (f32_any(f32_spoiled(acc), &flag)) {
    run(std::true_type{});
    us = 1.f;
  }
  TO* o = static_cast<TO*>(const_cast<void*>(a.o.p)) + b * a.o.s0 + hv * a.o.s1;
  float* pp = a.part + (int64_t(piece) * gridDim.z + bv) * a.T * a.Dv;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int gj = R * 64 + f32_row(wm, lane, r), gd = Dt * 128 + f32_col(wn * 2 + j, lane);
      if (gj < a.T && gd < a.Dv) {
        if (a.parts > 1)
          pp[int64_t(gj) * a.Dv + gd] = acc[0][j][r] * us;
        else
          o[int64_t(gj) * a.o.s2 + gd] = from_f<TO>(acc[0][j][r] * us);
      }
    }
}

template <typename TO>
__global__ __launch_bounds__(256) void k_f32_dvsum(F32DvArgs a, int64_t n) {
  const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (e >= n) return;
  float s = 0.f;
  int p = 0;
  for (; p + 4 <= a.parts; p += 4) {
    const float w0 = a.part[p * n + e], w1 = a.part[(p + 1) * n + e], w2 = a.part[(p + 2) * n + e],
                w3 = a.part[(p + 3) * n + e];
    s = s + w0 + w1 + w2 + w3;
  }
  for (; p < a.parts; ++p) s += a.part[p * n + e];
  const int64_t row = e / a.Dv;
  const int gd = int(e - row * a.Dv), gj = int(row % a.T), bv = int(row / a.T);
  TO* o = static_cast<TO*>(const_cast<void*>(a.o.p)) + (bv / int(a.Hv)) * a.o.s0 + (bv % int(a.Hv)) * a.o.s1;
  o[int64_t(gj) * a.o.s2 + gd] = from_f<TO>(s);
}

// ------------------------------------------------------------------ G
struct F32GArgs {
  View dO, v;
  int64_t H, Hv;
  int T, Dv;
  bool vec_do, vec_v;
  float* g;  // [slab][tpad][tpad]
  int tpad;
};

// Lower 128 x 128 tile of dO V^T, written to G at (i, j) and (j, i); zero on
// the diagonal.  Every element has one writer.  Bound by the matrix cores over
// a short contraction (B = 2, nh = 4, T = 387, D = 256: 62 -> 26 us).
template <typename TDO, typename TV>
__global__ __launch_bounds__(256, 2) void k_f32_g(F32GArgs a) {
  __shared__ __attribute__((aligned(1024))) char f32_lds[F32Mid::kLds];
  __shared__ int flag;
  int ti, tj;
  lower_tile_coords(int(blockIdx.x), ti, tj);
  const int slab = blockIdx.y;
  const int b = slab / int(a.H), h = slab % int(a.H);
  const int hv = a.Hv == 1 ? 0 : h;
  F32Rows<TDO, false, 0, 128, 256> la;
  la.base = static_cast<const TDO*>(a.dO.p) + b * a.dO.s0 + h * a.dO.s1;
  la.rs = a.dO.s2;
  la.r0 = ti * 128;
  la.nrows = a.T;
  la.K = a.Dv;
  la.vec = a.vec_do;
  F32Rows<TV, false, 0, 128, 256> lb;
  lb.base = static_cast<const TV*>(a.v.p) + b * a.v.s0 + hv * a.v.s1;
  lb.rs = a.v.s2;
  lb.r0 = tj * 128;
  lb.nrows = a.T;
  lb.K = a.Dv;
  lb.vec = a.vec_v;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1;
  f32x16 acc[2][2];
  f32_zero<F32Mid>(acc);
  f32_loop<false, F32Mid, false, true, 4>(f32_lds, la, lb, 0, a.Dv, wm, wn, lane, acc);
  float us = kF32Unscale;
  if (f32_any(f32_spoiled(acc), &flag)) {
    f32_zero<F32Mid>(acc);
    f32_loop<true, F32Mid>(f32_lds, la, lb, 0, a.Dv, wm, wn, lane, acc);
    us = 1.f;
  }
  float* g = a.g + int64_t(slab) * a.tpad * a.tpad;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gi = ti * 128 + f32_row(wm * 2 + i, lane, r), gj = tj * 128 + f32_col(wn * 2 + j, lane);
        if (gj > gi) continue;
        const float val = gj == gi ? 0.f : acc[i][j][r] * us;
        g[int64_t(gi) * a.tpad + gj] = val;
        g[int64_t(gj) * a.tpad + gi] = val;
      }
}

// ------------------------------------------------------------------ dQ
struct F32DqArgs {
  const float* g;
  int tpad;
  View x, o;
  int64_t H;
  int T, N;
  bool vec_x;
  const float* freqs;
  int64_t rope_start;
};

// Bound by the matrix cores and the split of X as it is staged (with RoPE its
// sine and cosine too): B = 2, nh = 4, T = 387, N = 8192: 346 us on the fp32
// instruction, 162 here.
// MASK: 0 full G (self attention), 1 keep j < i (dQ = dS K), 2 keep j > i (dK = dS^T Q).
template <class C, typename TO, int MASK, bool ROPE>
__global__ __launch_bounds__(C::NT, 2) void k_f32_dq(F32DqArgs a) {
  __shared__ __attribute__((aligned(1024))) char f32_lds[C::kLds];
  __shared__ int flag;
  const int ti = blockIdx.x, tn = blockIdx.y, slab = blockIdx.z;
  const int b = slab / int(a.H), h = slab % int(a.H);
  F32Rows<float, false, MASK, C::TM, C::NT> la;
  la.base = a.g + int64_t(slab) * a.tpad * a.tpad;
  la.rs = a.tpad;
  la.r0 = ti * C::TM;
  la.nrows = a.T;
  la.K = a.T;
  la.vec = true;
  F32Cols<float, ROPE, C::TN, C::NT> lb;
  lb.base = static_cast<const float*>(a.x.p) + b * a.x.s0 + h * a.x.s1;
  lb.rs = a.x.s2;
  lb.n0 = tn * C::TN;
  lb.ncols = a.N;
  lb.krows = a.T;
  lb.vec = a.vec_x;
  lb.freqs = a.freqs;
  lb.pos0 = float(a.rope_start);
  int kb = 0, ke = a.T;
  if (MASK == 1) ke = min(a.T, (ti + 1) * C::TM);
  if (MASK == 2) kb = ti * C::TM;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int wm = wave / C::WN, wn = wave % C::WN;
  f32x16 acc[C::MI][C::NJ];
  f32_zero<C>(acc);
  f32_loop<false, C, false, true, 4>(f32_lds, la, lb, kb, ke, wm, wn, lane, acc);
  float us = kF32Unscale;
  if (f32_any(f32_spoiled(acc), &flag)) {
    f32_zero<C>(acc);
    f32_loop<true, C>(f32_lds, la, lb, kb, ke, wm, wn, lane, acc);
    us = 1.f;
  }
  TO* o = static_cast<TO*>(const_cast<void*>(a.o.p)) + b * a.o.s0 + h * a.o.s1;
  const bool even = (lane & 1) == 0;
#pragma unroll
  for (int j = 0; j < C::NJ; ++j) {
    const int gn = tn * C::TN + f32_col(wn * C::NJ + j, lane);
    float fr = 0.f;
    if constexpr (ROPE) fr = gn < a.N ? a.freqs[gn & ~1] : 0.f;
#pragma unroll
    for (int i = 0; i < C::MI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gi = ti * C::TM + f32_row(wm * C::MI + i, lane, r);
        float val = acc[i][j][r] * us;
        if constexpr (ROPE) {
          // column pairs (2m, 2m+1) sit in lanes (2l, 2l+1): swap partners, rotate back
          const float other = __shfl_xor(val, 1, 64);
          float cs, sn;
          rope_cs(float(a.rope_start) + float(gi), fr, cs, sn);
          const float g0 = even ? val : other, g1 = even ? other : val;
          val = even ? (g0 * cs + g1 * sn) : (-g0 * sn + g1 * cs);
        }
        if (gi < a.T && gn < a.N) o[int64_t(gi) * a.o.s2 + gn] = from_f<TO>(val);
      }
  }
}

// ---------------------------------------------------------------- host side
bool rows_aligned(const bdh_tensor4* t, int n) {  // rows start at multiples of n values, length too
  if ((reinterpret_cast<uintptr_t>(t->data) % (n * esize(t->dtype))) != 0) return false;
  for (int i = 0; i < 3; ++i)
    if (t->size[i] > 1 && t->stride[i] % n != 0) return false;
  return t->size[3] % n == 0;
}

}  // namespace

// Tiles, work items and splits of the fp32 score pass.  T <= 128: one
// 128-row tile (a 256-row tile would be mostly padding).  The number of
// splits minimises an estimate of the kernel's end in stages of 16 k: items
// over 256 workgroups (one per CU), six stages of start and end an item, and
// the splits' partial tiles, written and read, at a stage's worth (about 2 us)
// per 10 MB.
F32Plan plan_f32(int64_t B, int64_t H, int64_t T, int64_t K, bool self, int64_t past) {
  F32Plan p;
  p.te_log = T <= 128 ? 7 : 8;
  const int64_t te = int64_t(1) << p.te_log;
  p.nt = (T + te - 1) / te;
  p.s0 = past >> p.te_log;
  p.t0 = p.s0 * (p.s0 + 1) / 2;
  p.ntl = p.nt * (p.nt + 1) / 2 - p.t0;
  const int64_t rows = p.nt - p.s0;
  p.nfull = self ? p.ntl - rows : p.ntl;
  p.per = self ? p.nfull + (rows + 1) / 2 : p.ntl;
  const int64_t stages = (K + kFK - 1) / kFK;
  const double tile_mb = double(B * H) * double(p.ntl) * double(te * te) * 8e-6;
  const int64_t items = B * H * p.per;
  const double slots = p.te_log == 7 ? 768. : 256.;
  int64_t best = 1;
  double best_t = 0;
  for (int64_t s = 1; s <= 32 && (s == 1 || stages / s >= 8); ++s) {
    const int64_t waves = int64_t((double(items * s) + slots - 1) / slots);
    const double t = double(waves) * (double((stages + s - 1) / s) + 6.) + (s > 1 ? double(s) * tile_mb / 10. : 0.);
    if (s == 1 || t < best_t * 0.97) {
      best = s;
      best_t = t;
    }
  }
  const int64_t kc = std::max<int64_t>(1, (stages + best - 1) / best);
  p.kc = kc * kFK;
  p.splits = std::max<int64_t>(1, (stages + kc - 1) / kc);
  p.tile_bytes = size_t(B * H) * size_t(p.ntl) * size_t(te * te) * sizeof(float);
  p.m_bytes = size_t(p.splits) * p.tile_bytes;
  return p;
}

int f32_scores(const ScoresArgs& s, const F32Plan& p, int64_t BH, hipStream_t st) {
  F32ScoresArgs a;
  a.q = s.q;
  a.k = s.k;
  a.H = s.H;
  a.T = int(s.T);
  a.K = int(s.K);
  a.past = int(s.past);
  a.q_is_k = s.q_is_k && s.past == 0;
  a.vec_q = s.vec_q;
  a.vec_k = s.vec_k;
  a.freqs = s.freqs;
  a.rope_start = s.rope_start;
  a.m = s.sp;
  a.split_stride = int64_t(p.tile_bytes / sizeof(float));
  a.kc = int(p.kc);
  a.nsplit = int(p.splits);
  a.nslab = int(BH);
  a.ntl = int(p.ntl);
  a.t0 = int(p.t0);
  a.s0 = int(p.s0);
  a.nt = int(p.nt);
  a.nfull = int(p.nfull);
  a.per = int(p.per);
  a.qr = s.qr;
  a.qr_bf = s.qr_bf;
  a.qr_vec = s.qr_vec;
  if (p.te_log == 7) {
    const dim3 grid((unsigned)(BH), unsigned(p.splits));
    if (s.freqs && s.qr.p)
      BDH_LAUNCH("k_f32_scores_mid", (k_f32_scores_mid<true, true>), grid, dim3(256), 0, st, a);
    else if (s.freqs)
      BDH_LAUNCH("k_f32_scores_mid", (k_f32_scores_mid<true, false>), grid, dim3(256), 0, st, a);
    else
      BDH_LAUNCH("k_f32_scores_mid", (k_f32_scores_mid<false, false>), grid, dim3(256), 0, st, a);
  } else {
    const int64_t groups = (BH * p.splits + 7) / 8 * 8;
    const dim3 grid((unsigned)(groups * p.per));
    if (s.freqs && s.qr.p)
      BDH_LAUNCH("k_f32_scores", (k_f32_scores<true, true>), grid, dim3(512), 0, st, a);
    else if (s.freqs)
      BDH_LAUNCH("k_f32_scores", (k_f32_scores<true, false>), grid, dim3(512), 0, st, a);
    else
      BDH_LAUNCH("k_f32_scores", (k_f32_scores<false, false>), grid, dim3(512), 0, st, a);
  }
  if (p.splits > 1) {
    const int64_t n4 = a.split_stride / 4;
    BDH_LAUNCH("k_f32_msum", k_f32_msum, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, a.m, n4, n4, a.nsplit);
  }
  return BDH_OK;
}

namespace {
template <typename TV, typename TO> int launch_sv(const F32SvArgs& a, int64_t BH, hipStream_t st) {
  const dim3 grid((unsigned)(a.nR), unsigned((a.Dv + 127) / 128), unsigned(BH));
  BDH_LAUNCH("k_f32_sv", (k_f32_sv<TV, TO>), grid, dim3(256), 0, st, a);
  return BDH_OK;
}
template <typename TDO, typename TO> int launch_dv(const F32DvArgs& a, int64_t nr, int64_t BHv, hipStream_t st) {
  const dim3 grid((unsigned)(nr * a.parts), unsigned((a.Dv + 127) / 128), unsigned(BHv));
  BDH_LAUNCH("k_f32_dv", (k_f32_dv<TDO, TO>), grid, dim3(256), 0, st, a);
  if (a.parts > 1) {
    const int64_t n = BHv * a.T * a.Dv;
    BDH_LAUNCH("k_f32_dvsum", k_f32_dvsum<TO>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, n);
  }
  return BDH_OK;
}
template <typename TDO, typename TV> int launch_g(const F32GArgs& a, int64_t ntl, int64_t BH, hipStream_t st) {
  BDH_LAUNCH("k_f32_g", (k_f32_g<TDO, TV>), dim3((unsigned)(ntl), unsigned(BH)), dim3(256), 0, st, a);
  return BDH_OK;
}
template <class C, typename TO, int MASK, bool ROPE> int launch_dq_c(const F32DqArgs& a, int64_t BH, hipStream_t st) {
  const dim3 grid((unsigned)((a.T + C::TM - 1) / C::TM), unsigned((a.N + C::TN - 1) / C::TN), unsigned(BH));
  BDH_LAUNCH("k_f32_dq", (k_f32_dq<C, TO, MASK, ROPE>), grid, dim3(C::NT), 0, st, a);
  return BDH_OK;
}
// 256 x 256 tiles unless T or N fits one 128-wide tile (the rest of a large
// tile would be padding).
template <typename TO, int MASK, bool ROPE> int launch_dq(const F32DqArgs& a, int64_t BH, hipStream_t st) {
  return a.T > 128 && a.N > 128 ? launch_dq_c<F32Big, TO, MASK, ROPE>(a, BH, st)
                                : launch_dq_c<F32Mid, TO, MASK, ROPE>(a, BH, st);
}
template <int MASK, bool ROPE> int pick_dq(const F32DqArgs& a, int64_t BH, int32_t odt, hipStream_t st) {
  return odt == BDH_BF16 ? launch_dq<bf16_t, MASK, ROPE>(a, BH, st) : launch_dq<float, MASK, ROPE>(a, BH, st);
}
}  // namespace

int f32_score_v(const float* m, const F32Plan& p, const bdh_tensor4* v, const bdh_tensor4* out, int64_t T, int64_t past,
                hipStream_t st) {
  F32SvArgs a;
  a.m = m;
  a.te_log = p.te_log;
  a.ntl = int(p.ntl);
  a.t0 = int(p.t0);
  a.v = view_of(v);
  a.o = view_of(out);
  a.o.s1 = out->stride[1];
  a.H = out->size[1];
  a.Hv = v->size[1];
  a.T = int(T);
  a.Dv = int(v->size[3]);
  a.past = int(past);
  a.R0 = int(past / 64);
  a.nR = int((T + 63) / 64) - a.R0;
  a.vec_v = rows_aligned(v, 2);
  const int64_t BH = out->size[0] * out->size[1];
  const bool ob = out->dtype == BDH_BF16;
  if (v->dtype == BDH_BF16) return ob ? launch_sv<bf16_t, bf16_t>(a, BH, st) : launch_sv<bf16_t, float>(a, BH, st);
  return ob ? launch_sv<float, bf16_t>(a, BH, st) : launch_sv<float, float>(a, BH, st);
}

// Pieces per dV tile: enough workgroups for two per CU, at least two chunks
// of 64 rows each.
int64_t f32_dv_parts(int64_t B, int64_t H, int64_t Hv, int64_t T, int64_t Dv) {
  const int64_t nr = (T + 63) / 64, tiles = nr * ((Dv + 127) / 128) * B * Hv;
  if (tiles <= 0) return 1;
  const int64_t chunks = (Hv == 1 ? H : 1) * nr;  // of the longest tile
  return std::max<int64_t>(1, std::min({(512 + tiles - 1) / tiles, chunks / 2, int64_t(32)}));
}
size_t f32_dv_bytes(int64_t B, int64_t H, int64_t Hv, int64_t T, int64_t Dv) {
  const int64_t parts = f32_dv_parts(B, H, Hv, T, Dv);
  return parts > 1 ? size_t(parts) * size_t(B * Hv) * size_t(T) * size_t(Dv) * sizeof(float) : 0;
}

int f32_dv(const float* m, const F32Plan& p, const bdh_tensor4* dout, const bdh_tensor4* dv, float* part,
           hipStream_t st) {
  F32DvArgs a;
  const int64_t B = dout->size[0], H = dout->size[1], T = dout->size[2], Hv = dv->size[1], Dv = dv->size[3];
  a.m = m;
  a.te_log = p.te_log;
  a.ntl = int(p.ntl);
  a.dO = view_of(dout);
  a.dO.s1 = dout->stride[1];
  a.o = view_of(dv);
  a.o.s1 = dv->stride[1];
  a.H = H;
  a.Hv = Hv;
  a.T = int(T);
  a.Dv = int(Dv);
  a.parts = int(f32_dv_parts(B, H, Hv, T, Dv));
  a.part = part;
  a.vec_do = rows_aligned(dout, 2);
  const int64_t nr = (T + 63) / 64;
  const bool ob = dv->dtype == BDH_BF16;
  if (dout->dtype == BDH_BF16)
    return ob ? launch_dv<bf16_t, bf16_t>(a, nr, B * Hv, st) : launch_dv<bf16_t, float>(a, nr, B * Hv, st);
  return ob ? launch_dv<float, bf16_t>(a, nr, B * Hv, st) : launch_dv<float, float>(a, nr, B * Hv, st);
}

int f32_g(const bdh_tensor4* dout, const bdh_tensor4* v, float* g, int64_t tpad, hipStream_t st) {
  F32GArgs a;
  a.dO = view_of(dout);
  a.dO.s1 = dout->stride[1];
  a.v = view_of(v);
  a.H = dout->size[1];
  a.Hv = v->size[1];
  a.T = int(dout->size[2]);
  a.Dv = int(v->size[3]);
  a.vec_do = rows_aligned(dout, 4);
  a.vec_v = rows_aligned(v, 4);
  a.g = g;
  a.tpad = int(tpad);
  const int64_t nt = tpad / 128, BH = dout->size[0] * dout->size[1];
  const bool vb = v->dtype == BDH_BF16;
  if (dout->dtype == BDH_BF16)
    return vb ? launch_g<bf16_t, bf16_t>(a, nt * (nt + 1) / 2, BH, st) : launch_g<bf16_t, float>(a, nt * (nt + 1) / 2, BH, st);
  return vb ? launch_g<float, bf16_t>(a, nt * (nt + 1) / 2, BH, st) : launch_g<float, float>(a, nt * (nt + 1) / 2, BH, st);
}

int f32_dq(const float* g, int64_t tpad, const bdh_tensor4* x, const bdh_tensor4* out, int mask, const float* freqs,
           int64_t rope_start, hipStream_t st) {
  F32DqArgs a;
  a.g = g;
  a.tpad = int(tpad);
  a.x = view_of(x);
  a.x.s1 = x->stride[1];
  a.o = view_of(out);
  a.o.s1 = out->stride[1];
  a.H = x->size[1];
  a.T = int(x->size[2]);
  a.N = int(x->size[3]);
  a.vec_x = rows_aligned(x, 2);
  a.freqs = freqs;
  a.rope_start = rope_start;
  const int64_t BH = x->size[0] * x->size[1];
  if (mask == 1) return pick_dq<1, false>(a, BH, out->dtype, st);
  if (mask == 2) return pick_dq<2, false>(a, BH, out->dtype, st);
  return freqs ? pick_dq<0, true>(a, BH, out->dtype, st) : pick_dq<0, false>(a, BH, out->dtype, st);
}

}  // namespace bdh
