// wire.hip — the Q8_0 hidden-state wire codec: the bytes a layer split sends
// between the peers that hold consecutive layers
// (src/inference/quant.rs:1-107, quantize_q8_0 / dequantize_q8_0).
//
// Per 32 values: [f16 scale][32 x i8] = 34 bytes, a partial trailing group
// zero-padded. The block maximum skips non-finite values; scale = amax / 127
// (f32), the codes clamp(round(v * (1 / scale)), -127, 127) with the
// reciprocal of the unrounded f32 scale; the scale travels as f16 (round to
// nearest even) and decoding multiplies by that f16 value. Built without FP
// contraction: the codes are the reference's bit for bit.
#include "qmm_device.h"
#include "qmm_launch.h"

namespace qmm {

namespace {

// A workgroup's 64 blocks are 2048 values and 2176 bytes: 4 lanes a block, 8
// values a lane, moved as 16-byte pieces; the 34-byte blocks are put together
// and taken apart in LDS. What bounds both directions is memory: 2048 x 8192
// values (67 MB f32, 18 MB of blocks) encode in 16.6 us and decode in 17.5 us
// (a lane a value, 4-byte loads and 1-byte stores: 50 and 23).
constexpr int kBlocks = 64, kValues = 32 * kBlocks, kBytes = 34 * kBlocks;

// Largest of the 4 lanes of a block.
__device__ __forceinline__ float quad_max(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true)));  // quad 1,0,3,2
  return fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true)));  // quad 2,3,0,1
}

// Rust's `f32 as i8` after f32::clamp(-127, 127): NaN -> 0.
__device__ __forceinline__ int8_t wire_code(float v, float inv) {
  const float qf = roundf(v * inv);  // f32::round: half away from zero
  if (qf != qf) return 0;
  return (int8_t)(qf < -127.0f ? -127.0f : (qf > 127.0f ? 127.0f : qf));
}

// xa / oa: x / out 16-byte aligned (else 4-byte loads, byte stores).
__global__ __launch_bounds__(256) void wire_encode_kernel(const float* __restrict__ x, int64_t n,
                                                          uint8_t* __restrict__ out, int64_t out_bytes, int xa, int oa) {
  __shared__ __attribute__((aligned(16))) uint16_t s_out[kBytes / 2];
  const int tid = (int)threadIdx.x, q = tid & 3;
  const int64_t i = (int64_t)blockIdx.x * kValues + 8 * tid;
  float v[8];
  if (xa && i + 8 <= n) {
    const float4 a = *(const float4*)(x + i), b = *(const float4*)(x + i + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = i + e < n ? x[i + e] : 0.0f;  // a partial group is zero-padded
  }
  float amax = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; e++) amax = fmaxf(amax, __builtin_isfinite(v[e]) ? fabsf(v[e]) : 0.0f);
  amax = quad_max(amax);
  const float scale = amax == 0.0f ? 0.0f : amax / 127.0f;
  const float inv = scale == 0.0f ? 0.0f : 1.0f / scale;
  uint16_t* b = s_out + 17 * (tid >> 2);
  if (q == 0) b[0] = f2h(scale);
#pragma unroll
  for (int e = 0; e < 4; e++)
    b[1 + 4 * q + e] = (uint16_t)((uint8_t)wire_code(v[2 * e], inv) | ((uint8_t)wire_code(v[2 * e + 1], inv) << 8));
  __syncthreads();
  const int64_t o = (int64_t)blockIdx.x * kBytes;
  const int64_t left = out_bytes - o;
  const int len = left < kBytes ? (int)left : kBytes;
  const int whole = oa ? len / 16 : 0;
  for (int p = tid; p < whole; p += 256) *(uint4*)(out + o + 16 * p) = *(const uint4*)((const uint8_t*)s_out + 16 * p);
  for (int p = 16 * whole + tid; p < len; p += 256) out[o + p] = ((const uint8_t*)s_out)[p];
}

// ia / oa: in / out 16-byte aligned.
__global__ __launch_bounds__(256) void wire_decode_kernel(const uint8_t* __restrict__ in, int64_t in_bytes, int64_t n,
                                                          float* __restrict__ out, int ia, int oa) {
  __shared__ __attribute__((aligned(16))) uint16_t s_in[kBytes / 2];
  const int tid = (int)threadIdx.x, q = tid & 3;
  const int64_t o = (int64_t)blockIdx.x * kBytes;
  const int64_t left = in_bytes - o;
  const int len = left < kBytes ? (int)left : kBytes;
  const int whole = ia ? len / 16 : 0;
  for (int p = tid; p < whole; p += 256) *(uint4*)((uint8_t*)s_in + 16 * p) = *(const uint4*)(in + o + 16 * p);
  for (int p = 16 * whole + tid; p < len; p += 256) ((uint8_t*)s_in)[p] = in[o + p];
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * kValues + 8 * tid;
  if (i >= n) return;
  const uint16_t* b = s_in + 17 * (tid >> 2);
  const float scale = h2f(b[0]);
  float v[8];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const uint16_t c = b[1 + 4 * q + e];
    v[2 * e] = (float)(int8_t)(c & 0xFF) * scale;
    v[2 * e + 1] = (float)(int8_t)(c >> 8) * scale;
  }
  if (oa && i + 8 <= n) {
    *(float4*)(out + i) = make_float4(v[0], v[1], v[2], v[3]);
    *(float4*)(out + i + 4) = make_float4(v[4], v[5], v[6], v[7]);
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++)
      if (i + e < n) out[i + e] = v[e];
  }
}

int aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

int64_t wire_bytes(int64_t n) {
  if (n < 0) return -1;
  const int64_t blocks = n / 32 + (n % 32 != 0);
  if (blocks > INT64_MAX / 34) return -1;
  return blocks * 34;
}

hipError_t launch_wire_encode(const float* x, int64_t n, void* out, hipStream_t st) {
  QMM_NOTE_LAUNCH();
  const int64_t groups = (n + kValues - 1) / kValues;
  if (groups >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  wire_encode_kernel<<<dim3((unsigned)groups), 256, 0, st>>>(x, n, (uint8_t*)out, wire_bytes(n), aligned16(x),
                                                             aligned16(out));
  return hipGetLastError();
}

hipError_t launch_wire_decode(const void* in, int64_t n, float* out, hipStream_t st) {
  QMM_NOTE_LAUNCH();
  const int64_t groups = (n + kValues - 1) / kValues;
  if (groups >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  wire_decode_kernel<<<dim3((unsigned)groups), 256, 0, st>>>((const uint8_t*)in, wire_bytes(n), n, out, aligned16(in),
                                                             aligned16(out));
  return hipGetLastError();
}

}  // namespace qmm
