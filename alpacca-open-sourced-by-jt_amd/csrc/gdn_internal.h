// GDN step launcher shared by the step entry point and the fused
// recurrent-layer step (no timing bracket of its own).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "alpx_common.h"

namespace alpx {

// Input type tag of ALPX_F32_PLANES.
struct planes_t {};

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// The N bf16 planes of two fp32 values, each the rounding of what the
// planes before it left.  Two at a time: one v_cvt_pk_bf16_f32 per plane
// (one value at a time the compiler spends a conversion on each).
template <int N>
__device__ __forceinline__ void split_planes2(float x0, float x1, bf16x2 (&p)[N]) {
  f32x2 r = {x0, x1};
#pragma unroll
  for (int n = 0; n < N; ++n) {
    p[n] = __builtin_convertvector(r, bf16x2);
    if (n + 1 < N) r = r - __builtin_convertvector(p[n], f32x2);
  }
}

// Output scale 1 / sqrt(Dk) of the GDN read-out o = S q / sqrt(Dk).
inline float gdn_output_scale(int key_dim) { return 1.0f / sqrtf((float)key_dim); }

int gdn_step_launch(float* state, const void* q, const void* k, const void* v, const float* beta,
                    const float* log_decay, void* out, int batch, int key_heads,
                    int value_heads, int key_dim, int value_dim, int dtype, int out_dtype,
                    hipStream_t s);

}  // namespace alpx
