// One generate step of the whole model as one call: the layers' kernels are
// launched back to back from here, so a step costs the host its launches and
// one call instead of six calls a layer through the binding.  Every layer runs the
// library's entry points in the order of the model's cached forward,
//   lat  = relu(x encoder)            (x: the bf16 row in this layer's V slot)
//   KR slot = RoPE(lat), y = decode(KR slot, past)
//   xy   = lat * relu(LN(y) encoder_v), y_mlp = xy decoder
//   x    = LN(x + LN(y_mlp)), rounded to bf16 into the next layer's V slot,
// with what is a launch of a few microseconds behind a product fused into it:
// RoPE in the few-row encoder product, the LayerNorms in the sums of the
// decode's chunks and of the decoder's splits (8 sequences, 6 layers, D = 256, S
// = 300: 417 -> 380 us a step).
#include <algorithm>

#include "common.h"
#include "few.h"

namespace bdh {
namespace {

struct StepWs {
  size_t lat, xy, yln, ymlp, xa, dec, gemm, end;
};

StepWs step_ws(int64_t B, int64_t nh, int64_t N, int64_t D, int64_t S) {
  StepWs w;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t p = at;
    at = align_up(at + bytes, 256);
    return p;
  };
  w.lat = take(size_t(B * nh * N) * 2);
  w.xy = take(size_t(B * nh * N) * 2);
  w.yln = take(size_t(B * nh * D) * 2);
  w.ymlp = take(size_t(B * D) * 2);
  w.xa = take(size_t(B * D) * 4 * 2);  // the residual stream, two buffers in turn
  w.dec = take(bdh_tril_decode_workspace(B, nh, 1, S, N, D));
  w.gemm = take(bdh_small_gemm_workspace(B, nh * N, D));
  w.end = at;
  return w;
}

bdh_tensor4 view4(const void* p, int32_t dt, int64_t n0, int64_t n1, int64_t n2, int64_t n3, int64_t s0, int64_t s1,
                  int64_t s2) {
  bdh_tensor4 t{};
  t.data = const_cast<void*>(p);
  const int64_t n[4] = {n0, n1, n2, n3}, s[4] = {s0, s1, s2, 1};
  for (int i = 0; i < 4; ++i) {
    t.size[i] = n[i];
    t.stride[i] = s[i];
  }
  t.dtype = dt;
  return t;
}

}  // namespace
}  // namespace bdh

using namespace bdh;

extern "C" size_t bdh_decode_step_workspace(int64_t B, int64_t nh, int64_t N, int64_t D, int64_t S) {
  if (B <= 0 || nh <= 0 || N <= 0 || D <= 0 || S <= 0) return 0;
  return step_ws(B, nh, N, D, S).end;
}

extern "C" int bdh_decode_step(const bdh_tensor4* x, const bdh_tensor4* out, const bdh_tensor4* enc_t,
                               const bdh_tensor4* encv_t, const bdh_tensor4* dec, const bdh_tensor4* cos,
                               const bdh_tensor4* sin, const bdh_tensor4* kr, int64_t kr_layer, const bdh_tensor4* v,
                               int64_t v_layer, int32_t n_layer, int64_t seq_len, void* workspace,
                               size_t workspace_bytes, bdh_stream stream) {
  for (const bdh_tensor4* t : {x, out, enc_t, encv_t, dec, cos, sin, kr, v}) BDH_TRY(check_view(t));
  const int64_t B = x->size[2], D = x->size[3], nh = enc_t->size[1], N = enc_t->size[2], cap = kr->size[2];
  if (x->dtype != BDH_F32 || out->dtype != BDH_F32 || kr->dtype != BDH_BF16 || v->dtype != BDH_BF16)
    return BDH_ERR_DTYPE;
  if (x->size[0] != 1 || x->size[1] != 1 || enc_t->size[3] != D || dec->size[2] != nh * N || dec->size[3] != D)
    return BDH_ERR_SHAPE;
  for (int i = 0; i < 4; ++i)
    if (out->size[i] != x->size[i] || encv_t->size[i] != enc_t->size[i] || cos->size[i] != sin->size[i])
      return BDH_ERR_SHAPE;
  if (cos->size[0] != 1 || cos->size[1] != 1 || cos->size[2] != 1 || cos->size[3] != N) return BDH_ERR_SHAPE;
  if (kr->size[0] != B || kr->size[1] != nh || kr->size[3] != N) return BDH_ERR_SHAPE;
  if (v->size[0] != B || v->size[1] != 1 || v->size[2] != cap || v->size[3] != D) return BDH_ERR_SHAPE;
  if (n_layer < 1 || seq_len < 1 || seq_len >= cap) return BDH_ERR_ARG;
  if (numel4(x) == 0) return BDH_OK;
  const StepWs o = step_ws(B, nh, N, D, seq_len);
  if (workspace == nullptr || workspace_bytes < o.end) return BDH_ERR_WORKSPACE;
  if ((reinterpret_cast<uintptr_t>(workspace) & 15) != 0) return BDH_ERR_WORKSPACE;
  char* w = static_cast<char*>(workspace);
  const bdh_tensor4 lat = view4(w + o.lat, BDH_BF16, B, 1, nh, N, nh * N, nh * N, N);
  const bdh_tensor4 lat_h = view4(w + o.lat, BDH_BF16, B, nh, 1, N, nh * N, N, N);
  const bdh_tensor4 xy = view4(w + o.xy, BDH_BF16, B, 1, nh, N, nh * N, nh * N, N);
  const bdh_tensor4 xy_rows = view4(w + o.xy, BDH_BF16, 1, 1, B, nh * N, B * nh * N, B * nh * N, nh * N);
  const bdh_tensor4 yln = view4(w + o.yln, BDH_BF16, B, nh, 1, D, nh * D, D, D);
  const bdh_tensor4 ymlp = view4(w + o.ymlp, BDH_BF16, 1, 1, B, D, B * D, B * D, D);
  const bdh_tensor4 cos_h = view4(cos->data, cos->dtype, B, nh, 1, N, 0, 0, 0);
  const bdh_tensor4 sin_h = view4(sin->data, sin->dtype, B, nh, 1, N, 0, 0, 0);
  const bool few_dec = dec->dtype == BDH_BF16 && dec->size[0] == 1 && dec->size[1] == 1 && few_dec_takes(&xy_rows, dec) &&
                       size_t(nh * N / 128) * size_t(B * D) * 4 <= o.end - o.gemm;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  bdh_tensor4 cur = *x;
  for (int32_t l = 0; l < n_layer; ++l) {
    const char* krl = static_cast<const char*>(kr->data) + int64_t(l) * kr_layer * 2;
    const char* vl = static_cast<const char*>(v->data) + int64_t(l) * v_layer * 2;
    const bdh_tensor4 past_k = view4(krl, BDH_BF16, B, nh, seq_len, N, kr->stride[0], kr->stride[1], kr->stride[2]);
    const bdh_tensor4 past_v = view4(vl, BDH_BF16, B, 1, seq_len, D, v->stride[0], v->stride[1], v->stride[2]);
    const bdh_tensor4 slot_k = view4(krl + seq_len * kr->stride[2] * 2, BDH_BF16, B, nh, 1, N, kr->stride[0],
                                     kr->stride[1], kr->stride[2]);
    // this token's bf16 row for the heads to share
    const bdh_tensor4 row = view4(vl + seq_len * v->stride[2] * 2, BDH_BF16, B, nh, 1, D, v->stride[0], 0, v->stride[2]);
    const FewRope rope{static_cast<const float*>(cos->data), static_cast<const float*>(sin->data),
                       static_cast<bf16_t*>(slot_k.data), slot_k.stride[0], slot_k.stride[1]};
    const bool can_rope = cos->dtype == BDH_F32 && sin->dtype == BDH_F32 && vec16_ok(cos) && vec16_ok(sin) &&
                          vec16_ok(&slot_k) && !views_overlap(&slot_k, &lat) && !views_overlap(&slot_k, &row) &&
                          !views_overlap(&slot_k, enc_t) && !views_overlap(&slot_k, cos) && !views_overlap(&slot_k, sin);
    bool roped = false;
    BDH_TRY(relu_gemm_rope(&row, enc_t, &lat, can_rope ? &rope : nullptr, &roped, stream));
    if (!roped) BDH_TRY(bdh_rope_rotate(&lat_h, &cos_h, &sin_h, &slot_k, 0, stream));
    BDH_TRY(decode_ln(&slot_k, &past_k, &past_v, &yln, w + o.dec, o.gemm - o.dec, s));
    BDH_TRY(bdh_gated_gemm(&yln, encv_t, &lat, &xy, stream));
    const bool last = l + 1 == n_layer;
    const bdh_tensor4 nxt = last ? *out
                                 : view4(w + o.xa + size_t(l & 1) * size_t(B * D) * 4, BDH_F32, 1, 1, B, D, B * D,
                                         B * D, D);
    const bdh_tensor4 slot_v = view4(vl + (v_layer + seq_len * v->stride[2]) * 2, BDH_BF16, 1, 1, B, D, 0, 0,
                                     v->stride[0]);
    const bdh_tensor4* out2 = last ? nullptr : &slot_v;
    if (views_overlap(&nxt, &cur) || (out2 != nullptr && (views_overlap(out2, &nxt) || views_overlap(out2, &cur))))
      return BDH_ERR_ALIAS;
    if (few_dec) {
      BDH_TRY(few_dec_ln_launch(&xy_rows, dec, &cur, &nxt, out2, reinterpret_cast<float*>(w + o.gemm), s));
    } else {
      BDH_TRY(bdh_small_gemm(&xy_rows, dec, &ymlp, w + o.gemm, o.end - o.gemm, stream));
      BDH_TRY(last ? bdh_layer_norm_rows(&cur, &ymlp, &nxt, stream)
                   : bdh_layer_norm_rows2(&cur, &ymlp, &nxt, &slot_v, stream));
    }
    cur = nxt;
  }
  return BDH_OK;
}
