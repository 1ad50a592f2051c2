// The layer's dense products for the few tokens of a generate step (one MFMA
// block of 32, two in the decoder), gfx950, bf16 operands, fp32 sums.
//
// A step reads each weight once (16.8 MB a product at nh N = 32768, 256
// features) and multiplies little, so what counts is how soon every CU has
// its loads out: one shot per workgroup, no loop of stages, all of its weight
// rows in flight at once.
#include <algorithm>

#include "common.h"
#include "few.h"
#include "lds_dma.h"

namespace bdh {
namespace {

// out[m, h, n] = [x[m, h, n] *] relu(sum_k y[m, h, k] wt[h, n, k]): a wave
// takes 32 rows of wt for all tokens.  Its rows go from memory straight into
// the MFMA's A registers (lane l: row l % 32, the 16-byte chunks 2 s + l / 32
// of k: four consecutive steps share each 128-byte line), the tokens' y rows
// into the B registers; the result leaves a lane four
// consecutive columns of one token, 8-byte pieces.
struct FewArgs {
  const bf16_t* y;
  int64_t y0, y1, y2;  // (B, nh, T, K)
  const bf16_t* w;
  int64_t w1, w2;      // (1, nh, N, K)
  const bf16_t* x;
  int64_t x0, x1, x2;  // (B, T, nh, N)
  bf16_t* o;
  int64_t o0, o1, o2;
  int T, M, N, nnb;
  const float *c, *sn;  // (N) tables of k_few_gemm's RoPE
  bf16_t* r;
  int64_t r0, r1;  // (B, nh, 1, N)
};

enum : int { kFewRelu = 0, kFewMul = 1, kFewRope = 2 };

// kFewRope (one token a sequence): RoPE of the rounded result goes to a second
// output, as k_rope8 rounds it; a lane holds whole pairs.
template <int K, int MODE>
__global__ __launch_bounds__(256) void k_few_gemm(const FewArgs a) {
  constexpr int S = K / 16;
  const int h = int(blockIdx.x) / a.nnb, nb = int(blockIdx.x) - h * a.nnb;
  const int lane = threadIdx.x & 63, l32 = lane & 31, hl = lane >> 5;
  const int n0 = nb * 128 + int(threadIdx.x >> 6) * 32;
  if (n0 >= a.N) return;  // (no barrier below)
  const bf16_t* wr = a.w + h * a.w1 + int64_t(min(n0 + l32, a.N - 1)) * a.w2 + hl * 8;
  bf16x8 wf[S];
#pragma unroll
  for (int s = 0; s < S; ++s) wf[s] = *reinterpret_cast<const bf16x8*>(wr + s * 16);
  const int m = min(l32, a.M - 1), b = m / a.T, t = m - b * a.T;
  const bf16_t* yr = a.y + b * a.y0 + h * a.y1 + t * a.y2 + hl * 8;
  bf16x8 yf[S];
#pragma unroll
  for (int s = 0; s < S; ++s) yf[s] = *reinterpret_cast<const bf16x8*>(yr + s * 16);
  u32x2 xv[4];
  f32x4 cv[4], sv[4];
  if constexpr (MODE == kFewRope) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = min(n0 + 8 * q + 4 * hl, a.N - 4);
      cv[q] = *reinterpret_cast<const f32x4*>(a.c + n);
      sv[q] = *reinterpret_cast<const f32x4*>(a.sn + n);
    }
  }
  if constexpr (MODE == kFewMul) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      xv[q] = *reinterpret_cast<const u32x2*>(a.x + b * a.x0 + t * a.x1 + h * a.x2 + min(n0 + 8 * q + 4 * hl, a.N - 4));
  }
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
  for (int s = 0; s < S; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[s], yf[s], acc, 0, 0, 0);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float u = acc[4 * q + e];
      v[e] = u != u ? u : fmaxf(u, 0.f);
    }
    uint32_t lo = pack_bf2(v[0], v[1]), hi = pack_bf2(v[2], v[3]);  // relu(s) as bf16, as the tile kernel rounds it
    if constexpr (MODE == kFewMul) {
      const uint32_t x0 = xv[q].x, x1 = xv[q].y;
      lo = pack_bf2(__uint_as_float(x0 << 16) * __uint_as_float(lo << 16),
                    __uint_as_float(x0 & 0xffff0000u) * __uint_as_float(lo & 0xffff0000u));
      hi = pack_bf2(__uint_as_float(x1 << 16) * __uint_as_float(hi << 16),
                    __uint_as_float(x1 & 0xffff0000u) * __uint_as_float(hi & 0xffff0000u));
    }
    const int n = n0 + 8 * q + 4 * hl;
    if (l32 < a.M && n < a.N) {
      *reinterpret_cast<u32x2*>(a.o + b * a.o0 + t * a.o1 + h * a.o2 + n) = u32x2{lo, hi};
      if constexpr (MODE == kFewRope) {
        uint32_t w[2] = {lo, hi};
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const float x0 = __uint_as_float(w[p] << 16), x1 = __uint_as_float(w[p] & 0xffff0000u);
          w[p] = pack_bf2(bf_round(x0 * cv[q][2 * p]) + bf_round((-x1) * sv[q][2 * p]),
                          bf_round(x1 * cv[q][2 * p + 1]) + bf_round(x0 * sv[q][2 * p + 1]));
        }
        *reinterpret_cast<u32x2*>(a.r + b * a.r0 + h * a.r1 + n) = u32x2{w[0], w[1]};
      }
    }
  }
}

template <int K> int launch_few(const FewArgs& a, int64_t H, hipStream_t s) {
  const dim3 grid(unsigned(a.nnb * H));
  if (a.x != nullptr)
    BDH_LAUNCH("k_few_gemm", (k_few_gemm<K, kFewMul>), grid, dim3(256), 0, s, a);
  else if (a.r != nullptr)
    BDH_LAUNCH("k_few_gemm", (k_few_gemm<K, kFewRope>), grid, dim3(256), 0, s, a);
  else
    BDH_LAUNCH("k_few_gemm", (k_few_gemm<K, kFewRelu>), grid, dim3(256), 0, s, a);
  return BDH_OK;
}

// Partial sums of out = a (M, K) b (K, 256) over 128 rows of b a workgroup:
// its rows (64 KB) land in LDS by DMA at once, chunk c of row r at
// c ^ 4 (r & 3); wave w owns columns 64 w .. + 64 and reads them as B
// fragments with transposing loads; a's rows are A fragments as they stand.
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
constexpr int kFdRows = 128, kFdD = 256;

struct FewDecArgs {
  const bf16_t* a;
  int64_t as;
  const bf16_t* b;
  int64_t bs;
  float* part;  // [split][M][256]
  int M, K;
};

__global__ __launch_bounds__(256) void k_few_dec(const FewDecArgs a) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kFdRows * 512];
  const int lane = threadIdx.x & 63, l32 = lane & 31, hl = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int k0 = blockIdx.x * kFdRows;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_u8*)lds);
  const void* base = sgpr_ptr(a.b + int64_t(k0) * a.bs);
  // instruction u of wave w: rows 2 (4 u + w) + lane / 32 (the host keeps 128
  // rows of b below 4 GiB)
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int r = 2 * (4 * u + w) + hl, c = l32 ^ (4 * (r & 3));
    dma16<0>(lds0 + uint32_t((4 * u + w) * 1024), base, uint32_t((int64_t(r) * a.bs + 8 * c) * 2));
  }
  bf16x8 af[2][8];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bf16_t* ar = a.a + int64_t(min(32 * i + l32, a.M - 1)) * a.as + k0 + hl * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (i == 0 || a.M > 32) af[i][s] = *reinterpret_cast<const bf16x8*>(ar + s * 16);
  }
  sy_wait<0>();
  __syncthreads();
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  // group lane q = 4 k + c of a 16-lane group addresses row k0 + k, columns
  // nb + 4 c ..; lane i receives four rows of column nb + i
  const int g4 = lane >> 4, q = lane & 15;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    bf16x8 bf[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = 64 * w + 32 * j + 16 * (g4 & 1) + 4 * (q & 3);
      const int row = 16 * s + 8 * (g4 >> 1) + (q >> 2);
      const uint8_t* p = lds + row * 512 + (((col >> 3) ^ (4 * (row & 3))) * 16) + ((col >> 2) & 1) * 8;
      const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
      const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(p + 4 * 512));
      bf[j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[0][s], bf[j], acc[0][j], 0, 0, 0);
      if (a.M > 32) acc[1][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[1][s], bf[j], acc[1][j], 0, 0, 0);
    }
  }
  float* out = a.part + int64_t(blockIdx.x) * a.M * kFdD;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = 32 * i + 8 * (r >> 2) + 4 * hl + (r & 3);
        if (m < a.M) out[int64_t(m) * kFdD + 64 * w + 32 * j + l32] = acc[i][j][r];
      }
}

// Their sum: 16 groups of 16 threads take every 16th split, four consecutive
// columns a thread and four splits in flight, and add up through LDS in group
// order (few rows make few workgroups, so each must be short).
template <typename TO>
__global__ __launch_bounds__(256) void k_few_reduce(const float* __restrict__ part, int nsplit, int M, TO* out,
                                                    int64_t os) {
  __shared__ f32x4 sums[16][16];
  const int g = threadIdx.x >> 4, l = threadIdx.x & 15;
  const int64_t e = (int64_t(blockIdx.x) * 16 + l) * 4, n = int64_t(M) * kFdD;  // (n is a multiple of 64)
  f32x4 s{0.f, 0.f, 0.f, 0.f};
  for (int p = g; p < nsplit; p += 64) {
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const f32x4*>(part + int64_t(min(p + 16 * u, nsplit - 1)) * n + e);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (p + 16 * u < nsplit) s += v[u];
  }
  sums[g][l] = s;
  __syncthreads();
  if (g != 0) return;
#pragma unroll
  for (int u = 1; u < 16; ++u) s += sums[u][l];
  TO* o = out + (e / kFdD) * os + e % kFdD;
#pragma unroll
  for (int c = 0; c < 4; ++c) o[c] = from_f<TO>(s[c]);
}

// The same with the layer's end behind it: o = LN(x + LN(sum rounded to bf16))
// and o2 the same rounded, a workgroup of 16 waves a row (a wave takes every
// 16th split, eight in flight).  Short, so what it saves is a launch: 8 rows,
// 256 splits 4.0 us and 3.4 for the row LayerNorm before, 6.0 now.
struct FewLnArgs {
  const float* part;
  int nsplit, M;
  const float* x;
  int64_t xs;
  float* o;
  int64_t os;
  bf16_t* o2;  // may be null
  int64_t o2s;
};
__global__ __launch_bounds__(1024) void k_few_ln(const FewLnArgs a) {
  __shared__ f32x4 sums[16][64];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int64_t n = int64_t(a.M) * kFdD, e = int64_t(blockIdx.x) * kFdD + 4 * lane;
  f32x4 s{0.f, 0.f, 0.f, 0.f};
  for (int p = g; p < a.nsplit; p += 128) {
    f32x4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const f32x4*>(a.part + int64_t(min(p + 16 * u, a.nsplit - 1)) * n + e);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (p + 16 * u < a.nsplit) s += v[u];
  }
  sums[g][lane] = s;
  __syncthreads();
  if (g != 0) return;
#pragma unroll
  for (int u = 1; u < 16; ++u) s += sums[u][lane];
  const float* x = a.x + blockIdx.x * a.xs + 4 * lane;
  float v[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = bf_round(s[c]);
  ln_row<4>(v, kFdD);
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] += x[c];
  ln_row<4>(v, kFdD);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    a.o[blockIdx.x * a.os + 4 * lane + c] = v[c];
    if (a.o2 != nullptr) a.o2[blockIdx.x * a.o2s + 4 * lane + c] = f2bf(v[c]);
  }
}

}  // namespace

// Whether the few-row kernel takes a [gated] ReLU product: up to 32 tokens, one
// MFMA block (N a multiple of 8, rows of 16 bytes as its caller checks).  11 ->
// 6.2 us for 8 tokens at nh N = 32768, K = 256 against the 256 x 128 tile kernel.
bool few_gemm_takes(int64_t M, int64_t K) { return M <= 32 && (K == 64 || K == 128 || K == 256 || K == 512); }

int few_gemm_launch(const bdh_tensor4* y, const bdh_tensor4* wt, const bdh_tensor4* x, const bdh_tensor4* out,
                    const FewRope* rope, hipStream_t s) {
  FewArgs a;
  a.y = static_cast<const bf16_t*>(y->data);
  a.y0 = y->stride[0];
  a.y1 = y->stride[1];
  a.y2 = y->stride[2];
  a.w = static_cast<const bf16_t*>(wt->data);
  a.w1 = wt->stride[1];
  a.w2 = wt->stride[2];
  a.x = x != nullptr ? static_cast<const bf16_t*>(x->data) : nullptr;
  a.x0 = x != nullptr ? x->stride[0] : 0;
  a.x1 = x != nullptr ? x->stride[1] : 0;
  a.x2 = x != nullptr ? x->stride[2] : 0;
  a.o = static_cast<bf16_t*>(out->data);
  a.o0 = out->stride[0];
  a.o1 = out->stride[1];
  a.o2 = out->stride[2];
  a.T = int(out->size[1]);
  a.M = int(out->size[0] * out->size[1]);
  a.N = int(out->size[3]);
  a.nnb = (a.N + 127) / 128;
  a.c = rope != nullptr ? rope->cos : nullptr;
  a.sn = rope != nullptr ? rope->sin : nullptr;
  a.r = rope != nullptr ? rope->out : nullptr;
  a.r0 = rope != nullptr ? rope->s0 : 0;
  a.r1 = rope != nullptr ? rope->s1 : 0;
  const int64_t H = out->size[2];
  if (int64_t(a.nnb) * H >= (int64_t(1) << 31)) return BDH_ERR_SHAPE;
  switch (y->size[3]) {
    case 64: return launch_few<64>(a, H, s);
    case 128: return launch_few<128>(a, H, s);
    case 256: return launch_few<256>(a, H, s);
    default: return launch_few<512>(a, H, s);
  }
}

// Whether k_few_dec takes a decode step's decoder product (its splits of 128
// rows then number K / 128): M = 8, K = 32768, D = 256: 6.5 us and 4.0 for the
// sum, against 13.7 and 4.2 on the 128-tile engine (128 splits of 256 rows).
bool few_dec_takes(const bdh_tensor4* a, const bdh_tensor4* b) {
  const int64_t M = a->size[2], K = a->size[3];
  auto al = [](const bdh_tensor4* t) {
    return (reinterpret_cast<uintptr_t>(t->data) & 15) == 0 && t->stride[2] % 8 == 0;
  };
  return M <= 64 && b->size[3] == kFdD && K % kFdRows == 0 && K / kFdRows <= 65535 && al(a) && al(b) &&
         b->stride[2] < (int64_t(1) << 23);
}

// part: 16-byte aligned, K / 128 x M x 256 floats.
static int few_dec_parts(const bdh_tensor4* a, const bdh_tensor4* b, float* part, FewDecArgs& g, hipStream_t s) {
  g.a = static_cast<const bf16_t*>(a->data);
  g.as = a->stride[2];
  g.b = static_cast<const bf16_t*>(b->data);
  g.bs = b->stride[2];
  g.part = part;
  g.M = int(a->size[2]);
  g.K = int(a->size[3]);
  BDH_LAUNCH("k_few_dec", k_few_dec, dim3(unsigned(g.K / kFdRows)), dim3(256), 0, s, g);
  return BDH_OK;
}

int few_dec_launch(const bdh_tensor4* a, const bdh_tensor4* b, const bdh_tensor4* out, float* part, hipStream_t s) {
  FewDecArgs g;
  BDH_TRY(few_dec_parts(a, b, part, g, s));
  const dim3 grid(unsigned(g.M * (kFdD / 64)));
  if (out->dtype == BDH_BF16)
    BDH_LAUNCH("k_few_reduce", k_few_reduce<bf16_t>, grid, dim3(256), 0, s, part, g.K / kFdRows, g.M,
               static_cast<bf16_t*>(out->data), out->stride[2]);
  else
    BDH_LAUNCH("k_few_reduce", k_few_reduce<float>, grid, dim3(256), 0, s, part, g.K / kFdRows, g.M,
               static_cast<float*>(out->data), out->stride[2]);
  return BDH_OK;
}

// out = LN(x + LN(a b)), x and out fp32 rows, out2 (may be null) bf16 rows.
int few_dec_ln_launch(const bdh_tensor4* a, const bdh_tensor4* b, const bdh_tensor4* x, const bdh_tensor4* out,
                      const bdh_tensor4* out2, float* part, hipStream_t s) {
  FewDecArgs g;
  BDH_TRY(few_dec_parts(a, b, part, g, s));
  FewLnArgs l;
  l.part = part;
  l.nsplit = g.K / kFdRows;
  l.M = g.M;
  l.x = static_cast<const float*>(x->data);
  l.xs = x->stride[2];
  l.o = static_cast<float*>(out->data);
  l.os = out->stride[2];
  l.o2 = out2 != nullptr ? static_cast<bf16_t*>(out2->data) : nullptr;
  l.o2s = out2 != nullptr ? out2->stride[2] : 0;
  BDH_LAUNCH("k_few_ln", k_few_ln, dim3(unsigned(g.M)), dim3(1024), 0, s, l);
  return BDH_OK;
}

}  // namespace bdh
