// glu.hip — out = act(gate) * up elementwise, over rows of n values: the
// GLU between an MLP's gate and up products where they did not run as one
// fused launch (the reference's silu_mul / swiglu_oai_mul / gelu product,
// src/inference/fast_math.rs:48-130). The arithmetic is glu_act.h's, the
// fused decode kernel's.
#include "glu_act.h"
#include "qmm_launch.h"

namespace qmm {

namespace {

template <int ACT>
__global__ __launch_bounds__(256) void glu_kernel(const float* __restrict__ gate, int64_t ldg,
                                                  const float* __restrict__ up, int64_t ldu, float* __restrict__ out,
                                                  int64_t ldo, int64_t n, int64_t rows) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n * rows) return;
  const int64_t r = i / n, c = i - r * n;
  out[r * ldo + c] = glu_act<ACT>(gate[r * ldg + c], up[r * ldu + c]);
}

// The gate and up products as `splits` slots of `total` values (rows x n)
// each, added in slot order: 4 values a thread where n, ldo and the output
// allow 16-byte accesses (V = 4), else 1.
typedef float f4v __attribute__((ext_vector_type(4)));
template <int ACT, int V>
__global__ __launch_bounds__(256) void glu_slots_kernel(const float* __restrict__ gate, const float* __restrict__ up,
                                                        int splits, float* __restrict__ out, int64_t ldo, uint32_t n,
                                                        int64_t total) {
  const int64_t i = V * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (i >= total) return;
  float g[V], u[V];
  auto load = [&](const float* p, float (&v)[V]) {
    if constexpr (V == 4) {
      const f4v x = *(const f4v*)p;
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = x[e];
    } else {
      v[0] = *p;
    }
  };
  load(gate + i, g);
  load(up + i, u);
#pragma unroll 4
  for (int s = 1; s < splits; s++) {
    float a[V], b[V];
    load(gate + s * total + i, a);
    load(up + s * total + i, b);
#pragma unroll
    for (int e = 0; e < V; e++) {
      g[e] += a[e];
      u[e] += b[e];
    }
  }
  const uint32_t r = (uint32_t)i / n;  // total < 2^31
  float* o = out + r * ldo + ((uint32_t)i - r * n);
#pragma unroll
  for (int e = 0; e < V; e++) g[e] = glu_act<ACT>(g[e], u[e]);
  if constexpr (V == 4)
    *(f4v*)o = f4v{g[0], g[1], g[2], g[3]};
  else
    *o = g[0];
}

template <int ACT>
hipError_t launch_slots(const float* gate, const float* up, int splits, float* out, int64_t ldo, int64_t n,
                        int64_t rows, hipStream_t st) {
  const int64_t total = n * rows;
  if (total >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  const bool vec = n % 4 == 0 && ldo % 4 == 0 && (((uintptr_t)gate | (uintptr_t)up | (uintptr_t)out) & 15) == 0;
  if (vec)
    glu_slots_kernel<ACT, 4><<<dim3((unsigned)((total / 4 + 255) / 256)), 256, 0, st>>>(gate, up, splits, out, ldo,
                                                                                     (uint32_t)n, total);
  else
    glu_slots_kernel<ACT, 1><<<dim3((unsigned)((total + 255) / 256)), 256, 0, st>>>(gate, up, splits, out, ldo,
                                                                                 (uint32_t)n, total);
  return hipGetLastError();
}

template <int ACT>
hipError_t launch(const float* gate, int64_t ldg, const float* up, int64_t ldu, float* out, int64_t ldo, int64_t n,
                  int64_t rows, hipStream_t st) {
  const int64_t total = n * rows;
  if ((total + 255) / 256 >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  glu_kernel<ACT><<<dim3((unsigned)((total + 255) / 256)), 256, 0, st>>>(gate, ldg, up, ldu, out, ldo, n, rows);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_glu(int act, const float* gate, int64_t ldg, const float* up, int64_t ldu, float* out, int64_t ldo,
                      int64_t n, int64_t rows, hipStream_t st) {
  QMM_NOTE_LAUNCH();
  if (n <= 0 || rows <= 0) return hipSuccess;
  if (act == GLU_SILU) return launch<GLU_SILU>(gate, ldg, up, ldu, out, ldo, n, rows, st);
  if (act == GLU_SWIGLU_OAI) return launch<GLU_SWIGLU_OAI>(gate, ldg, up, ldu, out, ldo, n, rows, st);
  if (act == GLU_GELU) return launch<GLU_GELU>(gate, ldg, up, ldu, out, ldo, n, rows, st);
  return hipErrorInvalidValue;
}

hipError_t launch_glu(int act, const float* gate, const float* up, int splits, float* out, int64_t ldo, int64_t n,
                      int64_t rows, hipStream_t st) {
  QMM_NOTE_LAUNCH();
  if (act == GLU_SILU) return launch_slots<GLU_SILU>(gate, up, splits, out, ldo, n, rows, st);
  if (act == GLU_SWIGLU_OAI) return launch_slots<GLU_SWIGLU_OAI>(gate, up, splits, out, ldo, n, rows, st);
  if (act == GLU_GELU) return launch_slots<GLU_GELU>(gate, up, splits, out, ldo, n, rows, st);
  return hipErrorInvalidValue;
}

}  // namespace qmm
