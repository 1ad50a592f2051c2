// KV-cache decode step for gfx950: out = (q K_past^T) V_past.
//
// HBM-bound: every past key row (N = 8192 elements) is read exactly once per
// query row.  Work is split over the past (chunks of keys per workgroup, from
// 64 down to 4 so that a small batch or a short past still fills the chip:
// dec_chunk); partial outputs over chunks are summed by a second small kernel
// (the op is linear in the scores, so no renormalisation is needed).  One
// sequence of 4 heads at S = 301, fp32 keys: 53.5 us in 64-key chunks (20
// workgroups), 14 in 4-key ones; 64 sequences at S = 511 read at 6.3 TB/s.
//
// Three score kernels share that shape: k_decode_bf16 (bf16 q and keys,
// v_dot2 products), k_decode_f32q (fp32 arithmetic, fp32 or bf16 keys, q of
// either dtype) and k_decode_partial (any strides and widths).  Each wave64
// streams key rows with 16-byte loads, reduces the dot product across the wave
// with shuffles and records the score in LDS; then all 256 threads form the
// partial out[d] = sum_s score_s V[s,d] with coalesced V row reads.
#include <algorithm>
#include <mutex>

#include "common.h"
#include "few.h"

namespace bdh {

constexpr int kDecNT = 256;
constexpr int kChunk = 32;  // most keys per workgroup

struct DecodeArgs {
  View q, k, v;
  int64_t H, Tq, S, Dk, Dv, Hv;
  int vec_k;
  float* part;    // [nchunk][rows][Dv]
  int64_t rows;   // B*H*Tq
  int chunk;      // keys per workgroup
};

template <typename TK>
__device__ __forceinline__ float dot_row(const float* qs, const TK* kp, int64_t Dk, int lane, bool vec) {
  float acc = 0.f;
  if (vec) {
    constexpr int EK = 16 / sizeof(TK);
    int64_t e0 = int64_t(lane) * EK;
    constexpr int STEP = 64 * EK;
    // four 16-byte loads in flight per lane per iteration
    for (; e0 + 3 * STEP < Dk; e0 += 4 * STEP) {
      u32x4 w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kp + e0 + u * STEP));
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const TK* x = reinterpret_cast<const TK*>(&w[u]);
        const float* qq = qs + e0 + u * STEP;
#pragma unroll
        for (int e = 0; e < EK; ++e) acc += qq[e] * to_f(x[e]);
      }
    }
    for (; e0 < Dk; e0 += STEP) {
      u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kp + e0));
      const TK* x = reinterpret_cast<const TK*>(&w);
#pragma unroll
      for (int e = 0; e < EK; ++e) acc += qs[e0 + e] * to_f(x[e]);
    }
  } else {
    for (int64_t e = lane; e < Dk; e += 64) acc += qs[e] * to_f(kp[e]);
  }
  return wave_sum(acc);
}

template <typename TQ, typename TK, typename TV>
__global__ __launch_bounds__(kDecNT) void k_decode_partial(DecodeArgs a) {
  extern __shared__ float smem[];
  float* qs = smem;              // Dk
  float* sc = smem + a.Dk;       // kChunk scores
  const int64_t row = blockIdx.y;
  const int64_t t = row % a.Tq, bh = row / a.Tq;
  const int64_t h = bh % a.H, b = bh / a.H;
  const int64_t hv = a.Hv == 1 ? 0 : h;

  const TQ* qp = static_cast<const TQ*>(a.q.p) + b * a.q.s0 + h * a.q.s1 + t * a.q.s2;
  for (int64_t e = threadIdx.x; e < a.Dk; e += kDecNT) qs[e] = to_f(qp[e]);
  __syncthreads();

  const int64_t s0 = int64_t(blockIdx.x) * a.chunk;
  const int64_t s1 = min(a.S, s0 + a.chunk);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const TK* kb = static_cast<const TK*>(a.k.p) + b * a.k.s0 + h * a.k.s1;
  for (int64_t s = s0 + wave; s < s1; s += kDecNT / 64) {
    const float d = dot_row<TK>(qs, kb + s * a.k.s2, a.Dk, lane, a.vec_k != 0);
    if (lane == 0) sc[s - s0] = d;
  }
  __syncthreads();

  const TV* vb = static_cast<const TV*>(a.v.p) + b * a.v.s0 + hv * a.v.s1;
  float* out = a.part + (int64_t(blockIdx.x) * a.rows + row) * a.Dv;
  for (int64_t d = threadIdx.x; d < a.Dv; d += kDecNT) {
    float o = 0.f;
    for (int64_t s = s0; s < s1; ++s) o += sc[s - s0] * to_f(vb[s * a.v.s2 + d]);
    out[d] = o;
  }
}

// bf16 q and K_past (the cache path): q is staged once as bf16 (16 KB at
// N = 8192); each wave scores two key rows at a time with eight 16-byte loads
// in flight per lane, accumulating v_dot2_f32_bf16 (exact bf16 products, fp32
// sums) against the staged q; then the 256 threads form the chunk's partial
// out[d] = sum_s score_s V[s,d].  Needs Dk a multiple of 2048.
// HALF (chunks of 4, a key per wave): the eight loads in flight go to the two
// halves of one key row; Dk a multiple of 4096.
constexpr int kDecChunkB = 64;  // most keys per workgroup
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// (The dwords are copied to scalars before the bit cast: this clang lowers
// __builtin_bit_cast of a vector element such as k.y as element 0.)
__device__ __forceinline__ float dot2w(uint32_t k, uint32_t q, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, k), __builtin_bit_cast(bf16x2, q), acc, false);
}
__device__ __forceinline__ float dot8(u32x4 k, u32x4 q, float acc) {
  const uint32_t k0 = k.x, k1 = k.y, k2 = k.z, k3 = k.w;
  const uint32_t q0 = q.x, q1 = q.y, q2 = q.z, q3 = q.w;
  acc = dot2w(k0, q0, acc);
  acc = dot2w(k1, q1, acc);
  acc = dot2w(k2, q2, acc);
  return dot2w(k3, q3, acc);
}

template <typename TV, bool HALF>
__global__ __launch_bounds__(kDecNT) void k_decode_bf16(DecodeArgs a) {
  extern __shared__ float smem[];
  float* sc = smem;                                         // kDecChunkB scores
  u32x4* qs = reinterpret_cast<u32x4*>(smem + kDecChunkB);  // q as Dk / 8 chunks of 8 bf16
  const int64_t row = blockIdx.y;
  const int64_t t = row % a.Tq, bh = row / a.Tq;
  const int64_t h = bh % a.H, b = bh / a.H;
  const int64_t hv = a.Hv == 1 ? 0 : h;
  const bf16_t* qp = static_cast<const bf16_t*>(a.q.p) + b * a.q.s0 + h * a.q.s1 + t * a.q.s2;
  for (int64_t i = threadIdx.x; i < a.Dk / 8; i += kDecNT) qs[i] = *reinterpret_cast<const u32x4*>(qp + 8 * i);
  __syncthreads();

  const int64_t s0 = int64_t(blockIdx.x) * a.chunk;
  const int64_t s1 = min(a.S, s0 + a.chunk);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const bf16_t* kb = static_cast<const bf16_t*>(a.k.p) + b * a.k.s0 + h * a.k.s1;
  const int nc = int(a.Dk / (HALF ? 1024 : 512));  // 16-byte chunks per lane per key row (or half)
  // keys s0 + wave + 4 j of this wave, in pairs (s, s + 4)
  for (int64_t s = s0 + wave; s < s1; s += 8) {
    const bool two = !HALF && s + 4 < s1;
    const bf16_t* k0 = kb + s * a.k.s2 + lane * 8;
    const bf16_t* k1 = HALF ? k0 + nc * 512 : kb + (two ? s + 4 : s) * a.k.s2 + lane * 8;
    float acc0 = 0.f, acc1 = 0.f;
    for (int c = 0; c < nc; c += 4) {
      u32x4 x0[4], x1[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x0[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(k0 + (c + u) * 512));
        x1[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(k1 + (c + u) * 512));
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const u32x4 q = qs[(c + u) * 64 + lane];
        acc0 = dot8(x0[u], q, acc0);
        acc1 = dot8(x1[u], HALF ? qs[(nc + c + u) * 64 + lane] : q, acc1);
      }
    }
    if constexpr (HALF) {
      acc0 = wave_sum(acc0 + acc1);
    } else {
      acc0 = wave_sum(acc0);
      acc1 = wave_sum(acc1);
    }
    if (lane == 0) {
      sc[s - s0] = acc0;
      if (two) sc[s + 4 - s0] = acc1;
    }
  }
  __syncthreads();

  const TV* vb = static_cast<const TV*>(a.v.p) + b * a.v.s0 + hv * a.v.s1;
  float* out = a.part + (int64_t(blockIdx.x) * a.rows + row) * a.Dv;
  for (int64_t d = threadIdx.x; d < a.Dv; d += kDecNT) {
    float o = 0.f;
    for (int64_t s = s0; s < s1; ++s) o += sc[s - s0] * to_f(vb[s * a.v.s2 + d]);
    out[d] = o;
  }
}

// fp32 arithmetic against fp32 or bf16 keys, q of either dtype: the
// reference's decode computes in fp32 (its cache casts a 16-bit past up
// before the products), and widening bf16 to fp32 is exact, so reading a bf16
// cache in place gives the products of its fp32 cast copy without the copy.
// q is staged once per workgroup as fp32 in LDS, arranged so that the 16-byte
// key piece a lane loads (EK elements) meets its q values in EK / 4
// contiguous 16-byte LDS reads: float4 plane p of piece c sits at
// qs[(NP c + p) 64 + lane].  Each wave scores two key rows at a time with
// eight 16-byte loads in flight per lane; then the 256 threads form the
// chunk's partial out[d] = sum_s score_s V[s,d].  Needs Dk a multiple of
// 64 EK and 16-byte aligned q and key rows.  HALF as in k_decode_bf16; Dk a
// multiple of 512 EK.
template <typename TK>
__device__ __forceinline__ float dot_piece(const u32x4& w, const float4* qs4, int np_stride, float acc) {
  if constexpr (sizeof(TK) == 4) {
    const float4 q = qs4[0];
    acc = fmaf(__uint_as_float(w.x), q.x, acc);
    acc = fmaf(__uint_as_float(w.y), q.y, acc);
    acc = fmaf(__uint_as_float(w.z), q.z, acc);
    return fmaf(__uint_as_float(w.w), q.w, acc);
  } else {
    const float4 qa = qs4[0], qb = qs4[np_stride];
    const uint32_t w0 = w.x, w1 = w.y, w2 = w.z, w3 = w.w;
    acc = fmaf(__uint_as_float(w0 << 16), qa.x, acc);
    acc = fmaf(__uint_as_float(w0 & 0xffff0000u), qa.y, acc);
    acc = fmaf(__uint_as_float(w1 << 16), qa.z, acc);
    acc = fmaf(__uint_as_float(w1 & 0xffff0000u), qa.w, acc);
    acc = fmaf(__uint_as_float(w2 << 16), qb.x, acc);
    acc = fmaf(__uint_as_float(w2 & 0xffff0000u), qb.y, acc);
    acc = fmaf(__uint_as_float(w3 << 16), qb.z, acc);
    return fmaf(__uint_as_float(w3 & 0xffff0000u), qb.w, acc);
  }
}

template <typename TQ, typename TK, typename TV, bool HALF>
__global__ __launch_bounds__(kDecNT) void k_decode_f32q(DecodeArgs a) {
  constexpr int EK = 16 / int(sizeof(TK));  // key elements per 16-byte piece
  constexpr int NP = EK / 4;                // float4 planes of q per piece
  extern __shared__ float smem[];
  float* sc = smem;                                         // kDecChunkB scores
  float4* qs = reinterpret_cast<float4*>(smem + kDecChunkB);  // Dk / 4 float4
  const int64_t row = blockIdx.y;
  const int64_t t = row % a.Tq, bh = row / a.Tq;
  const int64_t h = bh % a.H, b = bh / a.H;
  const int64_t hv = a.Hv == 1 ? 0 : h;
  const TQ* qp = static_cast<const TQ*>(a.q.p) + b * a.q.s0 + h * a.q.s1 + t * a.q.s2;
  for (int64_t i = threadIdx.x; i < a.Dk / 4; i += kDecNT) {
    const int64_t l = i & 63, cp = i >> 6;
    const int64_t e = ((cp / NP) * 64 + l) * EK + (cp % NP) * 4;
    float4 v;
    if constexpr (sizeof(TQ) == 4) {
      v = *reinterpret_cast<const float4*>(qp + e);
    } else {
      const u32x2 w = *reinterpret_cast<const u32x2*>(qp + e);
      const uint32_t w0 = w.x, w1 = w.y;
      v = make_float4(__uint_as_float(w0 << 16), __uint_as_float(w0 & 0xffff0000u), __uint_as_float(w1 << 16),
                      __uint_as_float(w1 & 0xffff0000u));
    }
    qs[i] = v;
  }
  __syncthreads();

  const int64_t s0 = int64_t(blockIdx.x) * a.chunk;
  const int64_t s1 = min(a.S, s0 + a.chunk);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const TK* kb = static_cast<const TK*>(a.k.p) + b * a.k.s0 + h * a.k.s1;
  const int nc = int(a.Dk / ((HALF ? 128 : 64) * EK));  // 16-byte pieces per lane per key row (or half)
  const float4* ql = qs + lane;
  // keys s0 + wave + 4 j of this wave, in pairs (s, s + 4)
  for (int64_t s = s0 + wave; s < s1; s += 8) {
    const bool two = !HALF && s + 4 < s1;
    const TK* k0 = kb + s * a.k.s2 + lane * EK;
    const TK* k1 = HALF ? k0 + nc * 64 * EK : kb + (two ? s + 4 : s) * a.k.s2 + lane * EK;
    float acc0 = 0.f, acc1 = 0.f;
    int c = 0;
    for (; c + 4 <= nc; c += 4) {
      u32x4 x0[4], x1[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x0[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(k0 + (c + u) * 64 * EK));
        x1[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(k1 + (c + u) * 64 * EK));
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4* q = ql + (NP * (c + u)) * 64;
        acc0 = dot_piece<TK>(x0[u], q, 64, acc0);
        acc1 = dot_piece<TK>(x1[u], HALF ? q + NP * nc * 64 : q, 64, acc1);
      }
    }
    for (; !HALF && c < nc; ++c) {
      const u32x4 x0 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(k0 + c * 64 * EK));
      const u32x4 x1 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(k1 + c * 64 * EK));
      const float4* q = ql + (NP * c) * 64;
      acc0 = dot_piece<TK>(x0, q, 64, acc0);
      acc1 = dot_piece<TK>(x1, q, 64, acc1);
    }
    if constexpr (HALF) {
      acc0 = wave_sum(acc0 + acc1);
    } else {
      acc0 = wave_sum(acc0);
      acc1 = wave_sum(acc1);
    }
    if (lane == 0) {
      sc[s - s0] = acc0;
      if (two) sc[s + 4 - s0] = acc1;
    }
  }
  __syncthreads();

  const TV* vb = static_cast<const TV*>(a.v.p) + b * a.v.s0 + hv * a.v.s1;
  float* out = a.part + (int64_t(blockIdx.x) * a.rows + row) * a.Dv;
  for (int64_t d = threadIdx.x; d < a.Dv; d += kDecNT) {
    float o = 0.f;
    for (int64_t s = s0; s < s1; ++s) o += sc[s - s0] * to_f(vb[s * a.v.s2 + d]);
    out[d] = o;
  }
}

// out = sum over the chunks of their partials: 32 outputs a workgroup, eight
// groups of lanes each take every eighth chunk with four loads in flight, the
// groups' sums added through LDS (a few dozen chunks of a small batch are a
// chain of loads otherwise).
constexpr int kRedCols = 32, kRedGroups = kDecNT / kRedCols;
template <typename TO>
__global__ __launch_bounds__(kDecNT) void k_decode_reduce(const float* part, int64_t nchunk, int64_t rows,
                                                          int64_t Dv, View o, int64_t H, int64_t Tq) {
  __shared__ float sums[kRedGroups][kRedCols];
  const int g = threadIdx.x / kRedCols, l = threadIdx.x % kRedCols;
  const int64_t idx = int64_t(blockIdx.x) * kRedCols + l, n = rows * Dv;
  float s = 0.f;
  if (idx < n) {
    for (int64_t c = g; c < nchunk; c += 4 * kRedGroups) {
      float w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = part[min(c + u * kRedGroups, nchunk - 1) * n + idx];
#pragma unroll
      for (int u = 0; u < 4; ++u) s += c + u * kRedGroups < nchunk ? w[u] : 0.f;
    }
  }
  sums[g][l] = s;
  __syncthreads();
  if (g != 0 || idx >= n) return;
#pragma unroll
  for (int u = 1; u < kRedGroups; ++u) s += sums[u][l];
  const int64_t row = idx / Dv, d = idx % Dv;
  const int64_t t = row % Tq, bh = row / Tq, h = bh % H, b = bh / H;
  TO* op = static_cast<TO*>(const_cast<void*>(o.p)) + b * o.s0 + h * o.s1 + t * o.s2;
  op[d] = from_f<TO>(s);
}

// The same with LN(row) behind it (one query a head, Dv = 64 E): a workgroup of
// eight waves a row, a wave takes every eighth chunk, four in flight.  What it
// saves is a launch: 32 rows of 256, 75 chunks: 4.8 us and 4.6 for the row
// LayerNorm before, 4.8 now.
template <int E>
__global__ __launch_bounds__(512) void k_decode_ln(const float* part, int64_t nchunk, int64_t rows, View o, int64_t H) {
  __shared__ float sums[8][64 * E];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int64_t row = blockIdx.x, n = rows * 64 * E;
  const float* pr = part + row * 64 * E + lane;
  float s[E];
#pragma unroll
  for (int e = 0; e < E; ++e) s[e] = 0.f;
  for (int64_t c = g; c < nchunk; c += 32) {
    float w[4][E];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < E; ++e) w[u][e] = pr[min(c + 8 * u, nchunk - 1) * n + 64 * e];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < E; ++e) s[e] += c + 8 * u < nchunk ? w[u][e] : 0.f;
  }
#pragma unroll
  for (int e = 0; e < E; ++e) sums[g][64 * e + lane] = s[e];
  __syncthreads();
  if (g != 0) return;
#pragma unroll
  for (int e = 0; e < E; ++e) {
#pragma unroll
    for (int u = 1; u < 8; ++u) s[e] += sums[u][64 * e + lane];
    s[e] = bf_round(s[e]);
  }
  ln_row<E>(s, 64 * E);
  bf16_t* op = static_cast<bf16_t*>(const_cast<void*>(o.p)) + (row / H) * o.s0 + (row % H) * o.s1 + lane;
#pragma unroll
  for (int e = 0; e < E; ++e) op[64 * e] = f2bf(s[e]);
}

// Keys per workgroup: 64 where that already makes three workgroups per CU
// (8 sequences, 32 rows, S = 1500: 127 us, 145 in 32-key chunks), else the
// largest of 32 ... 4 that makes eight, as long as the partial sums fit the
// no-allocation scratch (a call that fits it with 64-key chunks keeps doing
// so).  N = 8192, nh = 4, 64-key chunks -> this rule: one sequence of fp32
// keys at S = 301 53.5 -> 14 us, at S = 1500 58 -> 39; 8 sequences of bf16
// keys at S = 301 40 -> 32, at S = 100 37 -> 15.
static int dec_chunk(int64_t rows, int64_t S, int64_t Dv) {
  int chunk = kDecChunkB;
  if (rows * ((S + chunk - 1) / chunk) >= 768) return chunk;
  while (chunk > 4 && rows * ((S + chunk - 1) / chunk) < 2048 &&
         (S + chunk / 2 - 1) / (chunk / 2) * rows * Dv * int64_t(sizeof(float)) <= BDH_NOALLOC_SCRATCH_BYTES)
    chunk /= 2;
  return chunk;
}
static int64_t n_chunks(int64_t S, int64_t chunk) { return S > 0 ? (S + chunk - 1) / chunk : 1; }

template <typename TQ, typename TK, typename TV>
static int launch_partial(const DecodeArgs& a, int64_t nchunk, hipStream_t s) {
  dim3 grid((unsigned)(nchunk), unsigned(a.rows));
  const size_t shm = size_t(a.Dk + kChunk) * sizeof(float);
  BDH_LAUNCH("k_decode_partial", (k_decode_partial<TQ, TK, TV>), grid, dim3(kDecNT), shm, s, a);
  return BDH_OK;
}

template <typename TQ, typename TK>
static int pick_v(const DecodeArgs& a, int64_t nchunk, int32_t vdt, hipStream_t s) {
  return vdt == BDH_BF16 ? launch_partial<TQ, TK, bf16_t>(a, nchunk, s)
                         : launch_partial<TQ, TK, float>(a, nchunk, s);
}

template <typename TQ>
static int pick_k(const DecodeArgs& a, int64_t nchunk, int32_t kdt, int32_t vdt, hipStream_t s) {
  return kdt == BDH_BF16 ? pick_v<TQ, bf16_t>(a, nchunk, vdt, s) : pick_v<TQ, float>(a, nchunk, vdt, s);
}

template <typename TQ, typename TK, typename TV>
static int launch_f32q_t(const DecodeArgs& a, int64_t nred, hipStream_t s) {
  const dim3 grid((unsigned)nred, unsigned(a.rows));
  const size_t shm = size_t(kDecChunkB) * sizeof(float) + size_t(a.Dk) * sizeof(float);
  if (a.chunk == 4 && a.Dk % (8192 / int(sizeof(TK))) == 0)
    BDH_LAUNCH("k_decode_f32q", (k_decode_f32q<TQ, TK, TV, true>), grid, dim3(kDecNT), shm, s, a);
  else
    BDH_LAUNCH("k_decode_f32q", (k_decode_f32q<TQ, TK, TV, false>), grid, dim3(kDecNT), shm, s, a);
  return BDH_OK;
}

template <typename TQ, typename TK>
static int launch_f32q_v(const DecodeArgs& a, int64_t nred, int32_t vdt, hipStream_t s) {
  return vdt == BDH_BF16 ? launch_f32q_t<TQ, TK, bf16_t>(a, nred, s) : launch_f32q_t<TQ, TK, float>(a, nred, s);
}

static int launch_f32q(const DecodeArgs& a, int64_t nred, int32_t qdt, int32_t kdt, int32_t vdt, hipStream_t s) {
  if (qdt == BDH_BF16)
    return kdt == BDH_BF16 ? launch_f32q_v<bf16_t, bf16_t>(a, nred, vdt, s) : launch_f32q_v<bf16_t, float>(a, nred, vdt, s);
  return kdt == BDH_BF16 ? launch_f32q_v<float, bf16_t>(a, nred, vdt, s) : launch_f32q_v<float, float>(a, nred, vdt, s);
}

}  // namespace bdh

using namespace bdh;

extern "C" size_t bdh_tril_decode_workspace(int64_t B, int64_t H, int64_t Tq, int64_t S, int64_t Dk,
                                            int64_t Dv) {
  (void)Dk;
  const int64_t chunk = std::min(kChunk, dec_chunk(B * H * Tq, S, Dv));
  return size_t(n_chunks(S, chunk)) * size_t(B * H * Tq) * size_t(Dv) * sizeof(float);
}

namespace bdh {
namespace {

// Shape/dtype contract of decode (kernels/cuda_attn.py:114-131,
// csrc/tril_attn_cpu.cpp:214-223) and the launch plan: part_bytes is the
// partial-sum storage the chosen kernels need.
enum DecodeKind { kDecGeneric = 0, kDecBf16 = 1, kDecF32q = 2 };
struct DecodePlan {
  DecodeArgs a;
  DecodeKind kind = kDecGeneric;
  int64_t nred = 0;
  size_t part_bytes = 0;
};

int decode_plan(const bdh_tensor4* q, const bdh_tensor4* k, const bdh_tensor4* v, const bdh_tensor4* out,
                DecodePlan& p) {
  BDH_TRY(check_view(q));
  BDH_TRY(check_view(k));
  BDH_TRY(check_view(v));
  BDH_TRY(check_view(out));
  const int64_t B = q->size[0], H = q->size[1], Tq = q->size[2], Dk = q->size[3];
  const int64_t S = k->size[2], Dv = v->size[3];
  if (k->size[0] != B || k->size[1] != H || k->size[3] != Dk) return BDH_ERR_SHAPE;
  if (v->size[0] != B || v->size[2] != S) return BDH_ERR_SHAPE;
  if (v->size[1] != 1 && v->size[1] != H) return BDH_ERR_SHAPE;
  if (out->size[0] != B || out->size[1] != H || out->size[2] != Tq || out->size[3] != Dv)
    return BDH_ERR_SHAPE;
  if (views_overlap(out, q) || views_overlap(out, k) || views_overlap(out, v)) return BDH_ERR_ALIAS;
  if (B * H * Tq > 65535 || n_chunks(S, kChunk) > int64_t(1) << 30) return BDH_ERR_SHAPE;
  if ((Dk + kChunk) * int64_t(sizeof(float)) > 64 * 1024) return BDH_ERR_SHAPE;
  DecodeArgs& a = p.a;
  a.q = view_of(q);
  a.q.s1 = q->stride[1];
  a.k = view_of(k);
  a.k.s1 = k->stride[1];
  a.v = view_of(v);
  a.H = H;
  a.Tq = Tq;
  a.S = S;
  a.Dk = Dk;
  a.Dv = Dv;
  a.Hv = v->size[1];
  a.vec_k = vec16_ok(k) ? 1 : 0;
  a.part = nullptr;
  a.rows = B * H * Tq;
  // streaming kernels (64-key chunks) where q and the key rows allow
  // 16-byte pieces; the generic kernel otherwise
  const bool vec = vec16_ok(q) && vec16_ok(k) && S > 0;
  if (vec && q->dtype == BDH_BF16 && k->dtype == BDH_BF16 && Dk % 2048 == 0 && Dk * 2 + kDecChunkB * 4 <= 64 * 1024)
    p.kind = kDecBf16;
  else if (vec && Dk % (64 * (k->dtype == BDH_BF16 ? 8 : 4)) == 0 && Dk * 4 + kDecChunkB * 4 <= 64 * 1024)
    p.kind = kDecF32q;
  else
    p.kind = kDecGeneric;
  a.chunk = dec_chunk(a.rows, S, Dv);
  if (p.kind == kDecGeneric) a.chunk = std::min(kChunk, a.chunk);
  p.nred = n_chunks(S, a.chunk);
  p.part_bytes = size_t(p.nred) * size_t(a.rows) * size_t(Dv) * sizeof(float);
  return BDH_OK;
}

// The partial kernels write every (chunk, row, column) of part, so part needs
// no clearing between calls.
int decode_parts(const DecodePlan& p, const bdh_tensor4* q, const bdh_tensor4* k, const bdh_tensor4* v, float* part,
                 hipStream_t st) {
  DecodeArgs a = p.a;
  a.part = part;
  if (p.kind == kDecBf16) {
    const dim3 grid((unsigned)p.nred, unsigned(a.rows));
    const size_t shm = size_t(kDecChunkB) * sizeof(float) + size_t(a.Dk) * 2;
    const bool half = a.chunk == 4 && a.Dk % 4096 == 0;
    if (v->dtype == BDH_BF16) {
      if (half)
        BDH_LAUNCH("k_decode_bf16", (k_decode_bf16<bf16_t, true>), grid, dim3(kDecNT), shm, st, a);
      else
        BDH_LAUNCH("k_decode_bf16", (k_decode_bf16<bf16_t, false>), grid, dim3(kDecNT), shm, st, a);
    } else {
      if (half)
        BDH_LAUNCH("k_decode_bf16", (k_decode_bf16<float, true>), grid, dim3(kDecNT), shm, st, a);
      else
        BDH_LAUNCH("k_decode_bf16", (k_decode_bf16<float, false>), grid, dim3(kDecNT), shm, st, a);
    }
  } else if (p.kind == kDecF32q) {
    const int rc = launch_f32q(a, p.nred, q->dtype, k->dtype, v->dtype, st);
    if (rc != BDH_OK) return rc;
  } else {
    const int rc = q->dtype == BDH_BF16 ? pick_k<bf16_t>(a, p.nred, k->dtype, v->dtype, st)
                                        : pick_k<float>(a, p.nred, k->dtype, v->dtype, st);
    if (rc != BDH_OK) return rc;
  }
  return BDH_OK;
}

int decode_run(const DecodePlan& p, const bdh_tensor4* q, const bdh_tensor4* k, const bdh_tensor4* v,
               const bdh_tensor4* out, float* part, hipStream_t st) {
  BDH_TRY(decode_parts(p, q, k, v, part, st));
  const DecodeArgs& a = p.a;
  View o = view_of(out);
  o.s1 = out->stride[1];
  const int64_t total = a.rows * a.Dv;
  dim3 grid((unsigned)((total + kRedCols - 1) / kRedCols));
  if (out->dtype == BDH_BF16)
    BDH_LAUNCH("k_decode_reduce", k_decode_reduce<bf16_t>, grid, dim3(kDecNT), 0, st, part, p.nred, a.rows,
               a.Dv, o, a.H, a.Tq);
  else
    BDH_LAUNCH("k_decode_reduce", k_decode_reduce<float>, grid, dim3(kDecNT), 0, st, part, p.nred, a.rows,
               a.Dv, o, a.H, a.Tq);
  return BDH_OK;
}

// A workspace of 32-key partials is enough (one sized for a longer past may be
// smaller than what this one's smaller chunks take): the chunks grow until
// their partials fit.
int decode_fit(DecodePlan& p, const void* workspace, size_t workspace_bytes) {
  auto bytes = [&](int64_t chunk) {
    return size_t(n_chunks(p.a.S, chunk)) * size_t(p.a.rows) * size_t(p.a.Dv) * sizeof(float);
  };
  if (workspace == nullptr || workspace_bytes < bytes(kChunk)) return BDH_ERR_WORKSPACE;
  while (bytes(p.a.chunk) > workspace_bytes) p.a.chunk *= 2;
  p.nred = n_chunks(p.a.S, p.a.chunk);
  p.part_bytes = bytes(p.a.chunk);
  return BDH_OK;
}

}  // namespace

int decode_ln(const bdh_tensor4* q, const bdh_tensor4* k, const bdh_tensor4* v, const bdh_tensor4* out, void* workspace,
              size_t workspace_bytes, hipStream_t s) {
  DecodePlan p;
  BDH_TRY(decode_plan(q, k, v, out, p));
  if (out->dtype != BDH_BF16 || p.a.Tq != 1) return BDH_ERR_ARG;
  if (numel4(out) == 0) return BDH_OK;
  BDH_TRY(decode_fit(p, workspace, workspace_bytes));
  float* part = static_cast<float*>(workspace);
  BDH_TRY(decode_parts(p, q, k, v, part, s));
  const View o = view_of(out);
  const dim3 grid{unsigned(p.a.rows)};
  switch (p.a.Dv) {
    case 64: BDH_LAUNCH("k_decode_ln", k_decode_ln<1>, grid, dim3(512), 0, s, part, p.nred, p.a.rows, o, p.a.H); break;
    case 128: BDH_LAUNCH("k_decode_ln", k_decode_ln<2>, grid, dim3(512), 0, s, part, p.nred, p.a.rows, o, p.a.H); break;
    case 256: BDH_LAUNCH("k_decode_ln", k_decode_ln<4>, grid, dim3(512), 0, s, part, p.nred, p.a.rows, o, p.a.H); break;
    case 512: BDH_LAUNCH("k_decode_ln", k_decode_ln<8>, grid, dim3(512), 0, s, part, p.nred, p.a.rows, o, p.a.H); break;
    case 1024: BDH_LAUNCH("k_decode_ln", k_decode_ln<16>, grid, dim3(512), 0, s, part, p.nred, p.a.rows, o, p.a.H); break;
    default: return BDH_ERR_SHAPE;
  }
  return BDH_OK;
}
}  // namespace bdh

extern "C" int bdh_tril_decode(const bdh_tensor4* q, const bdh_tensor4* k, const bdh_tensor4* v,
                               const bdh_tensor4* out, void* workspace, size_t workspace_bytes,
                               bdh_stream stream) {
  DecodePlan p;
  BDH_TRY(decode_plan(q, k, v, out, p));
  if (numel4(out) == 0) return BDH_OK;
  BDH_TRY(decode_fit(p, workspace, workspace_bytes));
  return decode_run(p, q, k, v, out, static_cast<float*>(workspace), static_cast<hipStream_t>(stream));
}

// ------------------------------------------------------- no allocation
// The partial sums of bdh_tril_decode_noalloc live in this library-owned
// array: every GPU the library runs on holds its own copy (allocated when the
// code object loads on that device, kept until the process ends).  In host
// code `scratch` only names the symbol; its device address comes from
// hipGetSymbolAddress with the device current, once per device.
static __device__ __align__(256) uint8_t scratch[BDH_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of the current device's scratch array (looked up on the
// first call on that device), or nullptr when the lookup fails.
void* scratch_of_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr) return nullptr;
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}
}  // namespace

extern "C" int bdh_tril_decode_noalloc(const bdh_tensor4* q, const bdh_tensor4* k, const bdh_tensor4* v,
                                       const bdh_tensor4* out, bdh_stream stream) {
  DecodePlan p;
  BDH_TRY(decode_plan(q, k, v, out, p));
  if (numel4(out) == 0) return BDH_OK;
  if (p.part_bytes > size_t(BDH_NOALLOC_SCRATCH_BYTES)) return BDH_ERR_SCRATCH;
  void* part = scratch_of_current_device();
  if (part == nullptr) return BDH_ERR_LAUNCH;
  return decode_run(p, q, k, v, out, static_cast<float*>(part), static_cast<hipStream_t>(stream));
}
