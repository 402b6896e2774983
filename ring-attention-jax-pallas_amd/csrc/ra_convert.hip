// Between a caller's arrays (bf16, fp16 or fp32, any head dim up to 128) and the operands of the
// attention kernels (bf16, head dim 32, 64, 96 or 128): conversion and padding in one pass, several arrays in
// one launch.
#include "ra_launch.h"

namespace ra {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;

RA_DEV float row_element(const void* base, int dtype, long long at) {
  if (dtype == RA_DTYPE_F32) return ((const float*)base)[at];
  if (dtype == RA_DTYPE_F16) return (float)((const _Float16*)base)[at];
  return (float)((const bf16_t*)base)[at];
}

// Eight elements of a row per thread, neighbouring threads on neighbouring chunks; grid dimension y is
// the batch row, z the array.  HBM bound: every element is read and written once, where a cast and a
// pad of each array by themselves move it three times in three launches.
// k and v of 2 x 4791 x 8 x 96 fp16 with q of 1047 rows to head dim 128: 14.5 us (74 MB, 5.1 TB/s), against
// 88 us as nine launches of fills, copies and casts.
__global__ __launch_bounds__(256) void convert_kernel(const ConvertArgs a) {
  const ConvertItem& it = a.item[blockIdx.z];
  const unsigned cpr = (unsigned)(it.dst_d + 7) / 8, line = cpr * (unsigned)it.H;
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  const int b = blockIdx.y;
  const unsigned l = i / line;
  if (b >= it.B || l >= (unsigned)it.L) return;
  const unsigned in_line = i - l * line, h = in_line / cpr;
  const int d0 = 8 * (int)(in_line - h * cpr);
  const long long src = b * it.src_sb + (long long)l * it.src_sl + h * it.src_sh + d0;
  const long long dst = b * it.dst_sb + (long long)l * it.dst_sl + h * it.dst_sh + d0;
  const int n = min(8, it.src_d - d0), m = min(8, it.dst_d - d0);  // elements there are to read, to write
  float x[8];
  if (it.src_vec && n == 8) {
    if (it.src_dtype == RA_DTYPE_F32) {
      const f32x4 t0 = *(const f32x4*)((const float*)it.src + src), t1 = *(const f32x4*)((const float*)it.src + src + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = t0[e];
        x[4 + e] = t1[e];
      }
    } else if (it.src_dtype == RA_DTYPE_F16) {
      const f16x8 t = *(const f16x8*)((const _Float16*)it.src + src);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = (float)t[e];
    } else {
      const bf16x8 t = *(const bf16x8*)((const bf16_t*)it.src + src);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = (float)t[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (e < n) ? row_element(it.src, it.src_dtype, src + e) : 0.f;
  }
  if (it.dst_vec && m == 8) {
    if (it.dst_dtype == RA_DTYPE_F32) {
      *(f32x4*)((float*)it.dst + dst) = (f32x4){x[0], x[1], x[2], x[3]};
      *(f32x4*)((float*)it.dst + dst + 4) = (f32x4){x[4], x[5], x[6], x[7]};
    } else if (it.dst_dtype == RA_DTYPE_F16) {
      f16x8 t;
#pragma unroll
      for (int e = 0; e < 8; ++e) t[e] = (_Float16)x[e];
      *(f16x8*)((_Float16*)it.dst + dst) = t;
    } else {
      bf16x8 t;
#pragma unroll
      for (int e = 0; e < 8; ++e) t[e] = (bf16_t)x[e];
      *(bf16x8*)((bf16_t*)it.dst + dst) = t;
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (e >= m) continue;
    if (it.dst_dtype == RA_DTYPE_F32) ((float*)it.dst)[dst + e] = x[e];
    else if (it.dst_dtype == RA_DTYPE_F16) ((_Float16*)it.dst)[dst + e] = (_Float16)x[e];
    else ((bf16_t*)it.dst)[dst + e] = (bf16_t)x[e];
  }
}

hipError_t launch_convert(const ConvertArgs& a, int n, hipStream_t stream) {
  long long most = 0;
  int batch = 0;
  for (int i = 0; i < n; ++i) {
    const ConvertItem& it = a.item[i];
    const long long chunks = (long long)it.L * it.H * ((it.dst_d + 7) / 8);
    most = chunks > most ? chunks : most;
    batch = it.B > batch ? it.B : batch;
  }
  hipLaunchKernelGGL(convert_kernel, dim3((unsigned)((most + 255) / 256), (unsigned)batch, (unsigned)n), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace ra
