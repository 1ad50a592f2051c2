// Backward of the BDH layer's gated product for gfx950 (bf16 operands, fp32
// sums).  With s = y wt^T and g = dout dec^T per head (dout the gradient of
// the decoder's output, K = n_embd wide like y):
//   dx = g relu(s)
//   dz = g x where s > 0     (d y = dz wt, d wt = dz^T y)
// and the ReLU gradient that joins the two uses of x:
//   out = (a + b) where x > 0.
#include "fwd.h"
#include "lds_dma.h"

namespace bdh {
namespace {

// One workgroup makes a 128-token x 128-column tile of one head: first s,
// then g, both 64 x 64 per wave (2 x 2 blocks of 32 x 32) with K in stages of
// 32 through one ring of three LDS buffers filled by LDS DMA two stages ahead
// (16-byte chunk c of row r at c ^ ((r >> 2) & 3): conflict-free fragment
// reads).  relu(s) is kept in registers as bf16 (the value the forward's GEMM
// would store), g in fp32.  The products are MFMA(w rows, token rows), so a
// lane holds four consecutive columns of one token: 8-byte pieces.
//
// Bound by HBM: x is read once and two tensors of its size are written
// (3.2 GB at 16384 tokens, 4 heads, N = 8192), against 5.5e11 flops.  So each
// wave moves its own 64 x 64 block through 9 KB of LDS of its own (no
// barrier after the products) in whole 128-byte lines stored past the caches,
// and three workgroups share a CU so that one's stores run under another's
// products.  At that size 1105 us (2.9 TB/s; two workgroups a CU 1262, plain
// stores 1120, without its stores 923).
constexpr int kBM = 128, kBN = 128, kBK32 = 32, kBRing = 3, kBGroup = 2;
constexpr int kBStageA = kBM * 64, kBStageB = kBN * 64, kBStage = kBStageA + kBStageB;
constexpr int kBRow = 64 * 2 + 16;       // bytes of a row of a wave's block in LDS
constexpr int kBWave = 64 * kBRow;       // 9216
constexpr int kBLds = kBRing * kBStage;  // 48 KB
static_assert(4 * kBWave <= kBLds, "the waves' blocks fit the ring");

struct GatedBwdArgs {
  const bf16_t *y, *g;         // (B, nh, T, K), (B, T, K)
  int64_t y0, y1, y2, g0, g2;
  const bf16_t *w, *d;         // (nh, N, K) rows of encoder_v and of the decoder
  int64_t w1, w2, d1, d2;
  const bf16_t* x;             // (B, T, nh, N)
  int64_t x0, x1, x2;
  bf16_t* o[2];                // dx, dz
  int64_t o0[2], o1[2], o2[2];
  int T, M, N, K, nmb, nnb;
  int64_t total, per_xcd;
};

// A wave's accesses to its own LDS block stay in program order (LDS serves a
// wave in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() { asm volatile("" ::: "memory"); }

__device__ __forceinline__ int b_sw(int row, int c) { return row * 64 + ((c ^ ((row >> 2) & 3)) * 16); }

__global__ __launch_bounds__(256, 3) void k_gated_bwd(const GatedBwdArgs a) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kBLds];
  // tiles in groups of kBGroup row blocks, rows fastest, a contiguous range per
  // XCD: neighbouring columns of the same rows are written at about the same
  // time, and two row blocks share each pass over the weights (groups of 1 / 2
  // / 4 / 8 / 16 row blocks: 1148 / 1105 / 1127 / 1257 / 1465 us)
  const int bid = blockIdx.x, xcd = bid & 7, kk = bid >> 3;
  if (kk >= a.per_xcd) return;
  const int64_t t = int64_t(xcd) * a.per_xcd + kk;
  if (t >= a.total) return;
  const int64_t per_head = int64_t(a.nmb) * a.nnb;
  const int h = int(t / per_head);
  const int gi = int(t - int64_t(h) * per_head);
  const int rg = gi / (kBGroup * a.nnb), in = gi - rg * kBGroup * a.nnb;
  const int gsz = min(kBGroup, a.nmb - rg * kBGroup);
  const int nbi = in / gsz, mbi = rg * kBGroup + in - nbi * gsz;
  const int m0 = mbi * kBM, n0 = nbi * kBN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  // LDS DMA: instruction u of wave w fills rows 16 (4u + w) + lane / 4 of the
  // token and of the column part (u = 0, 1); slot lane & 3 of a row holds
  // chunk (lane & 3) ^ ((row >> 2) & 3)
  const int dc = (lane & 3) ^ ((lane >> 4) & 3);
  uint32_t yoff[2], goff[2], woff[2], doff[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int m = min(m0 + 16 * (4 * u + w) + (lane >> 2), a.M - 1);
    const int b = m / a.T, tt = m - b * a.T;
    yoff[u] = uint32_t((b * a.y0 + tt * a.y2 + dc * 8) * 2);
    goff[u] = uint32_t((b * a.g0 + tt * a.g2 + dc * 8) * 2);
    const int n = min(n0 + 16 * (4 * u + w) + (lane >> 2), a.N - 1);
    woff[u] = uint32_t((int64_t(n) * a.w2 + dc * 8) * 2);
    doff[u] = uint32_t((int64_t(n) * a.d2 + dc * 8) * 2);
  }
  const void* ybase = sgpr_ptr(a.y + h * a.y1);
  const void* wbase = sgpr_ptr(a.w + h * a.w1);
  const void* gbase = sgpr_ptr(a.g);
  const void* dbase = sgpr_ptr(a.d + h * a.d1);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_u8*)lds);
  const int nst = a.K / kBK32;
  auto issue = [&](int s) __attribute__((always_inline)) {
    const uint32_t m0b = lds0 + uint32_t((s % kBRing) * kBStage) + uint32_t(w) * 1024u;
    if (s < nst) {
      const uint32_t kb = uint32_t(s * kBK32 * 2);
      dma16<0>(m0b, ybase, yoff[0] + kb);
      dma16<4096>(m0b, ybase, yoff[1] + kb);
      dma16<kBStageA>(m0b, wbase, woff[0] + kb);
      dma16<kBStageA + 4096>(m0b, wbase, woff[1] + kb);
    } else {
      const uint32_t kb = uint32_t((s - nst) * kBK32 * 2);
      dma16<0>(m0b, gbase, goff[0] + kb);
      dma16<4096>(m0b, gbase, goff[1] + kb);
      dma16<kBStageA>(m0b, dbase, doff[0] + kb);
      dma16<kBStageA + 4096>(m0b, dbase, doff[1] + kb);
    }
  };

  // wave (wm, wn): tokens 64 wm .., columns 64 wn ..
  const int wm = w >> 1, wn = w & 1, fr = lane & 31, fh = lane >> 5;
  f32x16 acc[2][2];  // [column block][token block]
  auto zero = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[c][i][r] = 0.f;
  };
  auto stages = [&](int s0, int s1) __attribute__((always_inline)) {
    for (int s = s0; s < s1; ++s) {
      // stage s + 2 goes to the slot of stage s - 1, which every wave finished
      // before the barrier that ended stage s - 1
      if (s + 2 < 2 * nst) issue(s + 2);
      const uint8_t* base = lds + (s % kBRing) * kBStage;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        bf16x8 va[2], vb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          va[i] = *reinterpret_cast<const bf16x8*>(base + b_sw(64 * wm + 32 * i + fr, 2 * j + fh));
          vb[i] = *reinterpret_cast<const bf16x8*>(base + kBStageA + b_sw(64 * wn + 32 * i + fr, 2 * j + fh));
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int i = 0; i < 2; ++i)
            acc[c][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vb[c], va[i], acc[c][i], 0, 0, 0);
      }
      if (s + 1 < 2 * nst) {
        if (s + 2 < 2 * nst)
          sy_wait<4>();  // stage s + 1 landed (only s + 2 outstanding)
        else
          sy_wait<0>();
      }
      __syncthreads();  // (after the last stage: the ring becomes the waves' blocks)
    }
  };
  issue(0);
  issue(1);
  sy_wait<4>();
  __syncthreads();
  zero();
  stages(0, nst);
  uint32_t rp[2][2][8];  // relu(s), bf16 pairs
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float u = acc[c][i][2 * q], v = acc[c][i][2 * q + 1];
        rp[c][i][q] = pack_bf2(u != u ? u : fmaxf(u, 0.f), v != v ? v : fmaxf(v, 0.f));
      }
  zero();
  stages(nst, 2 * nst - 1);

  // this wave's 64 x 64 block: tokens mw .., columns nw ..; its x goes out
  // with the last stage, so its latency runs under those products
  uint8_t* blk = lds + w * kBWave;
  const int mw = m0 + 64 * wm, nw = n0 + 64 * wn;
  const int prow = lane >> 3, pcol = (lane & 7) * 8;  // 16-byte pieces: 8 rows of 128 bytes an instruction
  const int gn = nw + pcol;
  auto piece = [&](int e) __attribute__((always_inline)) {
    return reinterpret_cast<u32x4*>(blk + (8 * e + prow) * kBRow + pcol * 2);
  };
  u32x4 xr[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int m = min(mw + 8 * e + prow, a.M - 1);
    const int b = m / a.T, tt = m - b * a.T;
    xr[e] = *reinterpret_cast<const u32x4*>(a.x + b * a.x0 + tt * a.x1 + h * a.x2 + min(gn, a.N - 8));
  }
  stages(2 * nst - 1, 2 * nst);
#pragma unroll
  for (int e = 0; e < 8; ++e) *piece(e) = xr[e];
  wave_lds_fence();
  uint32_t dxp[2][2][8];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        u32x2* p = reinterpret_cast<u32x2*>(blk + (32 * i + fr) * kBRow + (32 * c + 8 * q + 4 * fh) * 2);
        const u32x2 xv = *p;
        const uint32_t xw[2] = {xv.x, xv.y};
        uint32_t dzw[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint32_t rw = rp[c][i][2 * q + u];
          const float r0 = __uint_as_float(rw << 16), r1 = __uint_as_float(rw & 0xffff0000u);
          const float x0 = __uint_as_float(xw[u] << 16), x1 = __uint_as_float(xw[u] & 0xffff0000u);
          const float g0 = acc[c][i][4 * q + 2 * u], g1 = acc[c][i][4 * q + 2 * u + 1];
          dxp[c][i][2 * q + u] = pack_bf2(g0 * r0, g1 * r1);
          dzw[u] = pack_bf2(r0 != 0.f ? g0 * x0 : 0.f, r1 != 0.f ? g1 * x1 : 0.f);
        }
        *p = u32x2{dzw[0], dzw[1]};
      }
  auto put = [&](const uint32_t (&v)[2][2][8]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<u32x2*>(blk + (32 * i + fr) * kBRow + (32 * c + 8 * q + 4 * fh) * 2) =
              u32x2{v[c][i][2 * q], v[c][i][2 * q + 1]};
    wave_lds_fence();
  };
  auto out = [&](int k) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int m = mw + 8 * e + prow;
      const u32x4 v = *piece(e);
      if (m < a.M && gn < a.N) {
        const int b = m / a.T, tt = m - b * a.T;
        __builtin_nontemporal_store(
            v, reinterpret_cast<u32x4*>(a.o[k] + b * a.o0[k] + tt * a.o1[k] + h * a.o2[k] + gn));
      }
    }
    wave_lds_fence();
  };
  wave_lds_fence();
  out(1);
  put(dxp);
  out(0);
}

// out = (a + b) where x > 0, else 0 (NaN x passes, as torch's ReLU gradient):
// a stream of three reads and one write.  A thread takes 16 bytes of four
// rows, so twelve loads are in flight; the result is not read soon and is
// stored past the caches.  1.14-1.24 ms at B = 32, nh = 4, T = 512, N = 8192 (4.3
// GB); where the forward kept its score tiles the dQ kernel's epilogue does the
// same for 0.3 ms, and this pass is left for the rest.
constexpr int kReluRows = 4;
struct ReluAddArgs {
  View a, b, x, o;
  int64_t d1, d2, n, rows;
};
__global__ __launch_bounds__(256) void k_relu_bwd_add(ReluAddArgs p) {
  const int64_t c = (int64_t(blockIdx.y) * 256 + threadIdx.x) * 8;
  if (c >= p.n) return;
  u32x4 va[kReluRows], vb[kReluRows], vx[kReluRows];
  bf16_t* o[kReluRows];
#pragma unroll
  for (int r = 0; r < kReluRows; ++r) {
    const int64_t row = min(int64_t(blockIdx.x) * kReluRows + r, p.rows - 1);  // (past the end: the last row again)
    const int64_t i2 = row % p.d2, r1 = row / p.d2;
    const int64_t i1 = r1 % p.d1, i0 = r1 / p.d1;
    auto at = [&](const View& v) {
      return static_cast<const bf16_t*>(v.p) + i0 * v.s0 + i1 * v.s1 + i2 * v.s2 + c;
    };
    va[r] = *reinterpret_cast<const u32x4*>(at(p.a));
    vb[r] = *reinterpret_cast<const u32x4*>(at(p.b));
    vx[r] = *reinterpret_cast<const u32x4*>(at(p.x));
    o[r] = const_cast<bf16_t*>(at(p.o));
  }
#pragma unroll
  for (int r = 0; r < kReluRows; ++r) {
    if (int64_t(blockIdx.x) * kReluRows + r >= p.rows) break;
    const uint32_t wa[4] = {va[r].x, va[r].y, va[r].z, va[r].w}, wb[4] = {vb[r].x, vb[r].y, vb[r].z, vb[r].w};
    const uint32_t wx[4] = {vx[r].x, vx[r].y, vx[r].z, vx[r].w};
    uint32_t wo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float s0 = __uint_as_float(wa[i] << 16) + __uint_as_float(wb[i] << 16);
      const float s1 = __uint_as_float(wa[i] & 0xffff0000u) + __uint_as_float(wb[i] & 0xffff0000u);
      const float x0 = __uint_as_float(wx[i] << 16), x1 = __uint_as_float(wx[i] & 0xffff0000u);
      wo[i] = pack_bf2(x0 <= 0.f ? 0.f : s0, x1 <= 0.f ? 0.f : s1);
    }
    __builtin_nontemporal_store(u32x4{wo[0], wo[1], wo[2], wo[3]}, reinterpret_cast<u32x4*>(o[r]));
  }
}

bool rows_16(const bdh_tensor4* t) {
  if ((reinterpret_cast<uintptr_t>(t->data) & 15) != 0) return false;
  for (int i = 0; i < 3; ++i)
    if (t->size[i] > 1 && t->stride[i] % 8 != 0) return false;
  return true;
}

View full_view(const bdh_tensor4* t) {
  View v;
  v.p = t->data;
  v.s0 = t->stride[0];
  v.s1 = t->stride[1];
  v.s2 = t->stride[2];
  return v;
}

}  // namespace
}  // namespace bdh

using namespace bdh;

extern "C" int bdh_gated_bwd(const bdh_tensor4* y, const bdh_tensor4* wt, const bdh_tensor4* x,
                             const bdh_tensor4* dec, const bdh_tensor4* dout, const bdh_tensor4* dx,
                             const bdh_tensor4* dz, bdh_stream stream) {
  const bdh_tensor4* all[7] = {y, wt, x, dec, dout, dx, dz};
  for (const bdh_tensor4* t : all) {
    BDH_TRY(check_view(t));
    if (t->dtype != BDH_BF16) return BDH_ERR_DTYPE;
  }
  const int64_t B = x->size[0], T = x->size[1], H = x->size[2], N = x->size[3], K = y->size[3];
  if (y->size[0] != B || y->size[1] != H || y->size[2] != T) return BDH_ERR_SHAPE;
  if (wt->size[0] != 1 || wt->size[1] != H || wt->size[2] != N || wt->size[3] != K) return BDH_ERR_SHAPE;
  if (dec->size[0] != 1 || dec->size[1] != H || dec->size[2] != N || dec->size[3] != K) return BDH_ERR_SHAPE;
  if (dout->size[0] != B || dout->size[1] != 1 || dout->size[2] != T || dout->size[3] != K) return BDH_ERR_SHAPE;
  const bdh_tensor4* outs[2] = {dx, dz};
  for (int o = 0; o < 2; ++o) {
    for (int i = 0; i < 4; ++i)
      if (outs[o]->size[i] != x->size[i]) return BDH_ERR_SHAPE;
    for (int i = 0; i < 5; ++i)
      if (views_overlap(outs[o], all[i])) return BDH_ERR_ALIAS;
    for (int p = 0; p < o; ++p)
      if (views_overlap(outs[o], outs[p])) return BDH_ERR_ALIAS;
  }
  if (numel4(x) == 0) return BDH_OK;
  if (K < kBK32 || K % kBK32 != 0 || N % 8 != 0) return BDH_ERR_SHAPE;
  for (const bdh_tensor4* t : all)
    if (!rows_16(t)) return BDH_ERR_STRIDE;
  const int64_t M = B * T;
  if (M >= (int64_t(1) << 31) || T >= (int64_t(1) << 31)) return BDH_ERR_SHAPE;
  // the DMA takes 32-bit byte offsets from the per-head bases
  auto span = [&](int64_t n0, int64_t s0, int64_t n2, int64_t s2) { return ((n0 - 1) * s0 + (n2 - 1) * s2 + K) * 2; };
  const int64_t lim = int64_t(1) << 32;
  if (span(B, y->stride[0], T, y->stride[2]) > lim || span(B, dout->stride[0], T, dout->stride[2]) > lim ||
      span(1, 0, N, wt->stride[2]) > lim || span(1, 0, N, dec->stride[2]) > lim)
    return BDH_ERR_SHAPE;
  GatedBwdArgs a;
  a.y = static_cast<const bf16_t*>(y->data);
  a.y0 = y->stride[0];
  a.y1 = y->stride[1];
  a.y2 = y->stride[2];
  a.g = static_cast<const bf16_t*>(dout->data);
  a.g0 = dout->stride[0];
  a.g2 = dout->stride[2];
  a.w = static_cast<const bf16_t*>(wt->data);
  a.w1 = wt->stride[1];
  a.w2 = wt->stride[2];
  a.d = static_cast<const bf16_t*>(dec->data);
  a.d1 = dec->stride[1];
  a.d2 = dec->stride[2];
  a.x = static_cast<const bf16_t*>(x->data);
  a.x0 = x->stride[0];
  a.x1 = x->stride[1];
  a.x2 = x->stride[2];
  for (int o = 0; o < 2; ++o) {
    a.o[o] = static_cast<bf16_t*>(outs[o]->data);
    a.o0[o] = outs[o]->stride[0];
    a.o1[o] = outs[o]->stride[1];
    a.o2[o] = outs[o]->stride[2];
  }
  a.T = int(T);
  a.M = int(M);
  a.N = int(N);
  a.K = int(K);
  a.nmb = int((M + kBM - 1) / kBM);
  a.nnb = int((N + kBN - 1) / kBN);
  a.total = int64_t(a.nmb) * a.nnb * H;
  a.per_xcd = (a.total + 7) / 8;
  const int64_t grid = 8 * a.per_xcd;
  if (grid >= (int64_t(1) << 31)) return BDH_ERR_SHAPE;
  BDH_LAUNCH("k_gated_bwd", k_gated_bwd, dim3(unsigned(grid)), dim3(256), 0, static_cast<hipStream_t>(stream), a);
  return BDH_OK;
}

extern "C" int bdh_relu_bwd_add(const bdh_tensor4* a, const bdh_tensor4* b, const bdh_tensor4* x,
                                const bdh_tensor4* out, bdh_stream stream) {
  for (const bdh_tensor4* t : {a, b, x, out}) {
    BDH_TRY(check_view(t));
    if (t->dtype != BDH_BF16) return BDH_ERR_DTYPE;
    for (int i = 0; i < 4; ++i)
      if (t->size[i] != x->size[i]) return BDH_ERR_SHAPE;
  }
  if (numel4(x) == 0) return BDH_OK;
  if (x->size[3] % 8 != 0) return BDH_ERR_SHAPE;
  for (const bdh_tensor4* t : {a, b, x, out})
    if (!rows_16(t)) return BDH_ERR_STRIDE;
  // out may be one of the inputs itself (each element is read before it is written)
  auto same = [&](const bdh_tensor4* t) {
    if (t->data != out->data) return false;
    for (int i = 0; i < 3; ++i)
      if (t->stride[i] != out->stride[i]) return false;
    return true;
  };
  for (const bdh_tensor4* t : {a, b, x})
    if (!same(t) && views_overlap(out, t)) return BDH_ERR_ALIAS;
  const int64_t rows = x->size[0] * x->size[1] * x->size[2];
  const int64_t ncol = (x->size[3] + 2047) / 2048;
  if (rows >= (int64_t(1) << 31) || ncol > 65535) return BDH_ERR_SHAPE;
  ReluAddArgs p;
  p.a = full_view(a);
  p.b = full_view(b);
  p.x = full_view(x);
  p.o = full_view(out);
  p.d1 = x->size[1];
  p.d2 = x->size[2];
  p.n = x->size[3];
  p.rows = rows;
  BDH_LAUNCH("k_relu_bwd_add", k_relu_bwd_add, dim3(unsigned((rows + kReluRows - 1) / kReluRows), unsigned(ncol)),
             dim3(256), 0, static_cast<hipStream_t>(stream), p);
  return BDH_OK;
}

// 32-bit DMA offsets inside one split of one head.
extern "C" int bdh_tn_gemm_takes(int64_t H, int64_t K, int64_t M, int64_t N, int64_t a_row, int64_t b_row,
                                 int64_t splits) {
  const int64_t S = splits, lim = int64_t(1) << 31, sizes[7] = {H, K, M, N, a_row, b_row, S};
  for (int64_t n : sizes)
    if (n < 1 || n >= lim) return 0;
  if (K % (32 * S) != 0 || M % 8 != 0 || N % 256 != 0 || a_row % 8 != 0 || b_row % 8 != 0) return 0;
  const int64_t ks = K / S;
  if ((ks * a_row + M) * 2 >= lim || (ks * b_row + N) * 2 >= lim || S * H > (int64_t(1) << 24)) return 0;
  return S * H * ((M + 255) / 256) <= (lim * 256 - 1) / N ? 1 : 0;  // workgroups of 256 x 256 outputs
}

extern "C" int bdh_tn_gemm(const bdh_tensor4* a, const bdh_tensor4* b, const bdh_tensor4* out, bdh_stream stream) {
  for (const bdh_tensor4* t : {a, b, out}) BDH_TRY(check_view(t));
  if (a->dtype != BDH_BF16 || b->dtype != BDH_BF16 || out->dtype != BDH_F32) return BDH_ERR_DTYPE;
  const int64_t S = out->size[0], H = a->size[1], K = a->size[2], M = a->size[3], N = b->size[3];
  if (a->size[0] != 1 || b->size[0] != 1 || b->size[1] != H || b->size[2] != K) return BDH_ERR_SHAPE;
  if (out->size[1] != H || out->size[2] != M || out->size[3] != N) return BDH_ERR_SHAPE;
  if (views_overlap(out, a) || views_overlap(out, b)) return BDH_ERR_ALIAS;
  if (numel4(out) == 0) return BDH_OK;
  if (!rows_16(a) || !rows_16(b)) return BDH_ERR_STRIDE;
  if (!bdh_tn_gemm_takes(H, K, M, N, a->stride[2], b->stride[2], S) || out->stride[2] >= (int64_t(1) << 26))
    return BDH_ERR_SHAPE;
  return sy_tn(a, b, out, static_cast<hipStream_t>(stream));
}
