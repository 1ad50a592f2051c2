// Products of a few token rows (few.hip) and what the generate step fuses
// behind them.
#pragma once

#include "common.h"

namespace bdh {

// RoPE of the ReLU product into a second output (B, nh, 1, N): fp32 tables of N
// entries, 16-byte aligned; out 8-byte aligned, strides multiples of 4.
struct FewRope {
  const float *cos, *sin;
  bf16_t* out;
  int64_t s0, s1;
};

bool few_gemm_takes(int64_t M, int64_t K);
int few_gemm_launch(const bdh_tensor4* y, const bdh_tensor4* wt, const bdh_tensor4* x, const bdh_tensor4* out,
                    const FewRope* rope, hipStream_t s);
bool few_dec_takes(const bdh_tensor4* a, const bdh_tensor4* b);
int few_dec_launch(const bdh_tensor4* a, const bdh_tensor4* b, const bdh_tensor4* out, float* part, hipStream_t s);
int few_dec_ln_launch(const bdh_tensor4* a, const bdh_tensor4* b, const bdh_tensor4* x, const bdh_tensor4* out,
                      const bdh_tensor4* out2, float* part, hipStream_t s);

// bdh_relu_gemm with that second output where the few-row kernel takes the
// product (*roped true), without it elsewhere.
int relu_gemm_rope(const bdh_tensor4* y, const bdh_tensor4* wt, const bdh_tensor4* out, const FewRope* rope,
                   bool* roped, bdh_stream stream);

// The decode of one query a head with LN behind it: out = LN(decode rounded to
// bf16), bf16 (decode.hip).
int decode_ln(const bdh_tensor4* q, const bdh_tensor4* k, const bdh_tensor4* v, const bdh_tensor4* out, void* workspace,
              size_t workspace_bytes, hipStream_t s);

}  // namespace bdh
