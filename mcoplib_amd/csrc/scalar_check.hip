// scalar_check.hip -- the short per-row scalar sequences of rowkern.h against the correctly rounded
// forms of numerics.h, bit for bit over a range of binary32 values.  The sequences start from the
// hardware's approximate reciprocal and reciprocal root, whose errors only a comparison over all
// values bounds.
#include <hip/hip_runtime.h>

#include <cfloat>

#include "../../include/mcop_norm.h"
#include "mcop_testing.h"
#include "rowkern.h"

namespace mcop {

__device__ __forceinline__ void count_if(bool differs, uint64_t* n) {
  const uint64_t b = __builtin_amdgcn_ballot_w64(differs);
  if (b != 0 && (threadIdx.x & 63) == 0) {
    atomicAdd(reinterpret_cast<unsigned long long*>(n), (unsigned long long)__popcll(b));
  }
}

// NaN is NaN whatever its payload.
__device__ __forceinline__ bool differ(float a, float b) {
  return __builtin_bit_cast(uint32_t, a) != __builtin_bit_cast(uint32_t, b) && (a == a || b == b);
}

// Whole workgroups of values: the host passes n as a multiple of the workgroup size.
__global__ void __launch_bounds__(256)
k_check_row_scalars(uint64_t* __restrict__ bad, uint32_t first, int64_t n, int hidden, float eps) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float a = __builtin_bit_cast(float, first + (uint32_t)i);
    count_if(differ(row_rcp(a), mcop_div_rn(1.0f, a)), bad + MCOP_SCALAR_RCP);
    count_if(differ(row_div<127>(a), mcop_div_rn(a, 127.0f)), bad + MCOP_SCALAR_DIV_127);
    count_if(differ(row_div<448>(a), mcop_div_rn(a, 448.0f)), bad + MCOP_SCALAR_DIV_448);
    count_if(differ(row_ratio(127.0f, a), mcop_div_rn(127.0f, a)), bad + MCOP_SCALAR_RATIO_127);
    // the smallest scale floors that the operators apply
    count_if(differ(__builtin_fmaxf(div_floored<127>(a), FLT_EPSILON),
                    __builtin_fmaxf(mcop_div_rn(a, 127.0f), FLT_EPSILON)),
             bad + MCOP_SCALAR_FLOORED_127);
    count_if(differ(__builtin_fmaxf(div_floored<448>(a), 1.0f / 229376.0f),
                    __builtin_fmaxf(mcop_div_rn(a, 448.0f), 1.0f / 229376.0f)),
             bad + MCOP_SCALAR_FLOORED_448);
    count_if(differ(row_inv_rms((double)a, hidden, eps), mcop_inv_rms((double)a, hidden, eps)),
             bad + MCOP_SCALAR_INV_RMS);
  }
}

}  // namespace mcop

extern "C" int mcop_check_row_scalars(uint64_t* mismatches, uint32_t first, int64_t n, int hidden,
                                      float epsilon, void* stream) {
  using namespace mcop;
  if (!mismatches || n <= 0 || n % 256 != 0 || hidden <= 0 ||
      (int64_t)first + n > ((int64_t)1 << 32)) {
    return set_error(MCOP_E_INVALID, "check_row_scalars: first=%u n=%lld hidden=%d", first,
                     (long long)n, hidden);
  }
  const int64_t blocks = n / 256 < 8192 ? n / 256 : 8192;
  hipLaunchKernelGGL(k_check_row_scalars, dim3((unsigned)blocks), dim3(256), 0,
                     static_cast<hipStream_t>(stream), mismatches, first, n, hidden, epsilon);
  return check_launch("check_row_scalars");
}
