// Device functions of the column kernels, for tests/test_fp64_math_gpu.py and tests/test_group_order.py.
#include <hip/hip_runtime.h>

#include "../../openifs_amd/csrc/cloudsc_device.h"
#include "../../openifs_amd/csrc/fp64_math.h"

// which: 0 exp(x), 1 x^y, 2 (x^y)^z with x^y as a base only
__global__ void evaluate(int which, const double* x, const double* y, const double* z, double* out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (which == 0)
    out[i] = fp64::exp(x[i]);
  else if (which == 1)
    out[i] = fp64::pow(fp64::log(x[i]), y[i]);
  else
    out[i] = fp64::pow(fp64::log_of_pow(fp64::log(x[i]), y[i]), z[i]);
}

extern "C" int fp64_check(int which, const double* x, const double* y, const double* z, double* out, int n,
                          void* stream) {
  if (which < 0 || which > 2 || !x || !y || !z || !out || n < 1) return -1;
  hipLaunchKernelGGL(evaluate, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, which, x, y, z, out, n);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

// The order of work-groups on the XCDs, on the host.
extern "C" unsigned group_order(unsigned id, unsigned n) { return cloudsc_gpu::xcd_group(id, n); }
