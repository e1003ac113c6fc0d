// arith.hip -- the kernels' own reciprocal and division over arrays, so that a
// test can compare them with IEEE division (built into libvkdt_calib.so).
#include "../common.h"

__global__ void __launch_bounds__(256) k_arith_div(const float *a, const float *b, float *r, float *q, long n)
{
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if(i >= n) return;
  r[i] = rcp_rn(b[i]);
  q[i] = div_rn(a[i], b[i], r[i]);
}

// device arrays of n: r = rcp_rn(b), q = div_rn(a, b, r).  Returns the HIP error code
extern "C" int vkdt_calib_div(const float *a, const float *b, float *r, float *q, long n, void *stream)
{
  if(n <= 0 || n > (1l << 31)) return -1;
  hipLaunchKernelGGL(k_arith_div, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, a, b, r, q, n);
  return (int)hipGetLastError();
}
