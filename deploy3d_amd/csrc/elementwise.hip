// Elementwise steps between the operators of a pass: the sum of two feature tensors (residual branches, skip connections)
// and the conversion of the voxeliser's float means to the backbone's storage type.
//
// Bound by HBM: 16 bytes per lane and tensor, one pass.  Both round once, to nearest even, as torch's kernels for the
// same step do, so a scheduled pass equals the step-by-step one bit for bit.
#include <hip/hip_fp16.h>

#include "common.h"

namespace d3d {
namespace {

template <class T, int N> struct __attribute__((aligned(sizeof(T) * N))) Pack {
  T v[N];
};

template <class T>
__global__ void __launch_bounds__(256) ewSum(const T* __restrict__ a, const T* __restrict__ b, T* __restrict__ out, int64_t n,
                                             int aligned) {
  constexpr int N = 16 / sizeof(T);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  const int64_t tid = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t packs = aligned ? n / N : 0;
  for (int64_t i = tid; i < packs; i += stride) {
    const Pack<T, N> x = reinterpret_cast<const Pack<T, N>*>(a)[i], y = reinterpret_cast<const Pack<T, N>*>(b)[i];
    Pack<T, N> z;
#pragma unroll
    for (int j = 0; j < N; ++j) z.v[j] = static_cast<T>(static_cast<float>(x.v[j]) + static_cast<float>(y.v[j]));
    reinterpret_cast<Pack<T, N>*>(out)[i] = z;
  }
  for (int64_t i = packs * N + tid; i < n; i += stride)
    out[i] = static_cast<T>(static_cast<float>(a[i]) + static_cast<float>(b[i]));
}

template <class T>
__global__ void __launch_bounds__(256) ewCast(const float* __restrict__ a, T* __restrict__ out, int64_t n, int aligned) {
  constexpr int N = 4;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  const int64_t tid = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t packs = aligned ? n / N : 0;
  for (int64_t i = tid; i < packs; i += stride) {
    const Pack<float, N> x = reinterpret_cast<const Pack<float, N>*>(a)[i];
    Pack<T, N> z;
#pragma unroll
    for (int j = 0; j < N; ++j) z.v[j] = static_cast<T>(x.v[j]);
    reinterpret_cast<Pack<T, N>*>(out)[i] = z;
  }
  for (int64_t i = packs * N + tid; i < n; i += stride) out[i] = static_cast<T>(a[i]);
}

unsigned ewBlocks(int64_t items) {
  const int64_t blocks = (items + 255) / 256;
  return static_cast<unsigned>(blocks < 1 ? 1 : (blocks > 4096 ? 4096 : blocks));
}

bool aligned16(const void* a, const void* b, const void* c) {
  return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(c)) & 15) == 0;
}

}  // namespace

int32_t launchSum(int32_t dtype, const void* a, const void* b, void* out, int64_t n, hipStream_t stream) {
  if (n <= 0) return D3D_OK;
  const int al = aligned16(a, b, out) ? 1 : 0;
#define D3D_EW_SUM(T, PER)                                                                                             \
  hipLaunchKernelGGL(ewSum<T>, dim3(ewBlocks(n / (al ? PER : 1) + 1)), dim3(256), 0, stream, static_cast<const T*>(a), \
                     static_cast<const T*>(b), static_cast<T*>(out), n, al)
  switch (dtype) {
    case D3D_FLOAT: D3D_EW_SUM(float, 4); break;
    case D3D_HALF: D3D_EW_SUM(_Float16, 8); break;
    case D3D_BF16: D3D_EW_SUM(__bf16, 8); break;
    default: setError("sum: dtype %d not implemented", dtype); return D3D_ERR_UNSUPPORTED;
  }
#undef D3D_EW_SUM
  D3D_HIP_CHECK(hipGetLastError());
  return D3D_OK;
}

int32_t launchCastFromFloat(int32_t dtype, const float* a, void* out, int64_t n, hipStream_t stream) {
  if (n <= 0) return D3D_OK;
  const int al = aligned16(a, out, out) ? 1 : 0;
  const unsigned blocks = ewBlocks(n / (al ? 4 : 1) + 1);
  switch (dtype) {
    case D3D_HALF:
      hipLaunchKernelGGL(ewCast<_Float16>, dim3(blocks), dim3(256), 0, stream, a, static_cast<_Float16*>(out), n, al);
      break;
    case D3D_BF16:
      hipLaunchKernelGGL(ewCast<__bf16>, dim3(blocks), dim3(256), 0, stream, a, static_cast<__bf16*>(out), n, al);
      break;
    default: setError("cast: dtype %d not implemented", dtype); return D3D_ERR_UNSUPPORTED;
  }
  D3D_HIP_CHECK(hipGetLastError());
  return D3D_OK;
}

}  // namespace d3d
