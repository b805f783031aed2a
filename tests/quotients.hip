// Device values of the shared-denominator quotients and the square root
// (csu_amd/csrc/device_math.h), element by element, for
// tests/test_gpu_quotients.py.  Built by __graft_entry__.build().
#include <hip/hip_runtime.h>
#include "device_math.h"

using namespace csu;

// op 0: a / b by Den(b); 1: by Den(b, rb); 2: fsqrt(a)
template <typename T>
__global__ void k_eval(int n, int op, const T* a, const T* b, const T* rb, T* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (op == 2) out[i] = fsqrt(a[i]);
  else if constexpr (sizeof(T) == 8) out[i] = op == 1 ? Den<T>(b[i], rb[i])(a[i]) : Den<T>(b[i])(a[i]);
  else out[i] = Den<T>(b[i])(a[i]);
}

template <typename T>
static int eval(int n, int op, const T* a, const T* b, const T* rb, T* out) {
  if (n <= 0) return 1;
  const size_t sz = (size_t)n * sizeof(T);
  T* d = nullptr;
  if (hipMalloc((void**)&d, 4 * sz) != hipSuccess) return 2;
  int rc = 0;
  if (hipMemcpy(d, a, sz, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(d + n, b, sz, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(d + 2 * (size_t)n, rb, sz, hipMemcpyHostToDevice) != hipSuccess)
    rc = 3;
  if (!rc) {
    hipLaunchKernelGGL(k_eval<T>, dim3((n + 255) / 256), dim3(256), 0, nullptr, n, op, d, d + n, d + 2 * (size_t)n,
                       d + 3 * (size_t)n);
    if (hipGetLastError() != hipSuccess || hipMemcpy(out, d + 3 * (size_t)n, sz, hipMemcpyDeviceToHost) != hipSuccess)
      rc = 4;
  }
  (void)hipFree(d);
  return rc;
}

extern "C" int quotients_f64(int n, int op, const double* a, const double* b, const double* rb, double* out) {
  return eval<double>(n, op, a, b, rb, out);
}
extern "C" int quotients_f32(int n, int op, const float* a, const float* b, const float* rb, float* out) {
  return eval<float>(n, op, a, b, rb, out);
}
