// The row-wise work of a hooked layer around its read (xenc/injector.py:54-58, 185-197), for steps
// without a gradient.  One workgroup per row, the row in registers, every sum in a fixed order:
//
//   hook_norm_kernel   hn = h * rsqrt(mean(h^2) + eps)
//   hook_unit_kernel   q = q / (|q| + eps), in place
//   hook_add_kernel    out = h + delta, ratio = |delta| / (|h| + 1e-6)
//
// Bound by launches: as torch operators the three were 5 + 3 + 6 launches of 1.3-6 us a layer, each
// with its share of the host's time (a step of 4 layers, 4 rows x 5120: 839 us, 842 of it the host's
// 100-odd calls); 3 us each here.
#include "xenc_common.h"

namespace xenc {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kHookThreads = 256, kHookVec = 8;   // a pass covers 8192 columns in registers

// Sum of v over the workgroup, every thread getting it (waves added in order).
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < kHookThreads / kWave; ++w) s += red[w];
  __syncthreads();
  return s;
}

// The sum of squares of row x (d % 4 == 0, 16-byte aligned); its first kHookVec float4 of a thread
// stay in v, longer rows are read again by the caller.
__device__ __forceinline__ float row_squares(const float* __restrict__ x, int d, f32x4 (&v)[kHookVec], float* red) {
  float s = 0.f;
#pragma unroll
  for (int u = 0; u < kHookVec; ++u) {
    const int i = (u * kHookThreads + (int)threadIdx.x) * 4;
    v[u] = i < d ? *reinterpret_cast<const f32x4*>(x + i) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int u = 0; u < kHookVec; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) s = fmaf(v[u][e], v[u][e], s);
  for (int i = (kHookVec * kHookThreads + (int)threadIdx.x) * 4; i < d; i += kHookThreads * 4) {
    const f32x4 y = *reinterpret_cast<const f32x4*>(x + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) s = fmaf(y[e], y[e], s);
  }
  return block_sum(s, red);
}

// y = x * f over the row (y may be x).
__device__ __forceinline__ void row_scaled(const float* x, float* y, int d, float f, const f32x4 (&v)[kHookVec]) {
#pragma unroll
  for (int u = 0; u < kHookVec; ++u) {
    const int i = (u * kHookThreads + (int)threadIdx.x) * 4;
    if (i < d) *reinterpret_cast<f32x4*>(y + i) = f32x4{v[u][0] * f, v[u][1] * f, v[u][2] * f, v[u][3] * f};
  }
  for (int i = (kHookVec * kHookThreads + (int)threadIdx.x) * 4; i < d; i += kHookThreads * 4) {
    const f32x4 z = *reinterpret_cast<const f32x4*>(x + i);
    *reinterpret_cast<f32x4*>(y + i) = f32x4{z[0] * f, z[1] * f, z[2] * f, z[3] * f};
  }
}

__global__ __launch_bounds__(kHookThreads) void hook_norm_kernel(const float* __restrict__ h, long long ldh, int d,
                                                                 float eps, float* __restrict__ hn) {
  __shared__ float red[kHookThreads / kWave];
  const float* x = h + (long long)blockIdx.x * ldh;
  f32x4 v[kHookVec];
  const float s = row_squares(x, d, v, red);
  row_scaled(x, hn + (long long)blockIdx.x * d, d, rsqrtf(s / (float)d + eps), v);
}

__global__ __launch_bounds__(kHookThreads) void hook_unit_kernel(float* q, long long ldq, int d, float eps) {
  __shared__ float red[kHookThreads / kWave];
  float* x = q + (long long)blockIdx.x * ldq;
  f32x4 v[kHookVec];
  const float n = sqrtf(row_squares(x, d, v, red)) + eps;
#pragma unroll
  for (int u = 0; u < kHookVec; ++u) {
    const int i = (u * kHookThreads + (int)threadIdx.x) * 4;
    if (i < d) *reinterpret_cast<f32x4*>(x + i) = f32x4{v[u][0] / n, v[u][1] / n, v[u][2] / n, v[u][3] / n};
  }
  for (int i = (kHookVec * kHookThreads + (int)threadIdx.x) * 4; i < d; i += kHookThreads * 4) {
    const f32x4 z = *reinterpret_cast<const f32x4*>(x + i);
    *reinterpret_cast<f32x4*>(x + i) = f32x4{z[0] / n, z[1] / n, z[2] / n, z[3] / n};
  }
}

__global__ __launch_bounds__(kHookThreads) void hook_add_kernel(const float* __restrict__ h, long long ldh,
                                                                const float* __restrict__ delta, long long ldd, int d,
                                                                float* __restrict__ out, float* __restrict__ ratio) {
  __shared__ float red[kHookThreads / kWave];
  const float* x = h + (long long)blockIdx.x * ldh;
  const float* y = delta + (long long)blockIdx.x * ldd;
  float* o = out + (long long)blockIdx.x * d;
  float sx = 0.f, sy = 0.f;
  for (int i = threadIdx.x * 4; i < d; i += kHookThreads * 4) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(x + i), b = *reinterpret_cast<const f32x4*>(y + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sx = fmaf(a[e], a[e], sx);
      sy = fmaf(b[e], b[e], sy);
    }
    *reinterpret_cast<f32x4*>(o + i) = a + b;
  }
  sx = block_sum(sx, red);
  sy = block_sum(sy, red);
  if (threadIdx.x == 0) ratio[blockIdx.x] = sqrtf(sy) / (sqrtf(sx) + 1e-6f);
}

int check_rows(int M, int d, long long ld) {
  return M < 0 || d <= 0 || d % 4 != 0 || ld < d || ld % 4 != 0 ? XENC_EINVAL : XENC_OK;
}

}  // namespace
}  // namespace xenc

using namespace xenc;

extern "C" int xenc_hook_norm(const float* h, long long ldh, int M, int d, float eps, float* hn, void* stream) {
  if (int rc = check_rows(M, d, ldh)) return rc;
  if (M == 0) return XENC_OK;
  if (!h || !hn) return XENC_ENULL;
  if (!aligned16(h) || !aligned16(hn)) return XENC_EALIGN;
  hipLaunchKernelGGL(hook_norm_kernel, dim3(M), dim3(kHookThreads), 0, reinterpret_cast<hipStream_t>(stream), h, ldh, d,
                     eps, hn);
  return check_launch();
}

extern "C" int xenc_hook_unit(float* q, long long ldq, int M, int d, float eps, void* stream) {
  if (int rc = check_rows(M, d, ldq)) return rc;
  if (M == 0) return XENC_OK;
  if (!q) return XENC_ENULL;
  if (!aligned16(q)) return XENC_EALIGN;
  hipLaunchKernelGGL(hook_unit_kernel, dim3(M), dim3(kHookThreads), 0, reinterpret_cast<hipStream_t>(stream), q, ldq, d,
                     eps);
  return check_launch();
}

extern "C" int xenc_hook_add(const float* h, long long ldh, const float* delta, long long ldd, int M, int d, float* out,
                             float* ratio, void* stream) {
  if (int rc = check_rows(M, d, ldh)) return rc;
  if (ldd < d || ldd % 4 != 0) return XENC_EINVAL;
  if (M == 0) return XENC_OK;
  if (!h || !delta || !out || !ratio) return XENC_ENULL;
  if (!aligned16(h) || !aligned16(delta) || !aligned16(out)) return XENC_EALIGN;
  hipLaunchKernelGGL(hook_add_kernel, dim3(M), dim3(kHookThreads), 0, reinterpret_cast<hipStream_t>(stream), h, ldh,
                     delta, ldd, d, out, ratio);
  return check_launch();
}
