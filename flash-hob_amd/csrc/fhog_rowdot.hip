// d_i = sum_c O_ic dO_ic as a kernel of its own: pass 0 where it is asked for alone, and the first step of the 16-bit
// first-order backward (the sweeps of the double-backward take d in their first one).
#include "fhog_split_util.h"

namespace fhog {
using namespace splitk;
namespace {

// Pass 0: d_i = sum_c O_ic dO_ic  (fhog/triton_bwdbwd.py:580), fp32 result. 16 lanes per row.
template <typename T, int D>
__global__ void __launch_bounds__(256) rowdot_kernel(Params p) {
  const int64_t rows = (int64_t)p.batch * p.n_q;
  const int64_t r = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int sub = threadIdx.x & 15;
  float acc = 0.f;
  if (r < rows) {
    const int64_t bh = r / p.n_q, i = r % p.n_q;
    const T* o = (const T*)p.o + bh * p.stride_qb + i * p.stride_qn;
    const T* g = (const T*)p.dO + bh * p.stride_qb + i * p.stride_qn;
#pragma unroll
    for (int c = sub * 8; c < D; c += 128) {
      const Chunk<T> a = load_chunk<T>(o + c), b = load_chunk<T>(g + c);
#pragma unroll
      for (int e = 0; e < 8; e++) acc = __builtin_fmaf(chunk_elem(a, e), chunk_elem(b, e), acc);
    }
  }
  acc += __shfl_xor(acc, 8);
  acc += __shfl_xor(acc, 4);
  acc += __shfl_xor(acc, 2);
  acc += __shfl_xor(acc, 1);
  if (r < rows && sub == 0) p.ws_d[r] = acc;
}

template <typename T>
hipError_t launch_rowdot_t(const Params& p, hipStream_t s) {
  const int64_t rows = (int64_t)p.batch * p.n_q;
  const dim3 grid((unsigned)((rows + 15) / 16)), block(256);
  switch (p.d) {
    case 32: hipLaunchKernelGGL((rowdot_kernel<T, 32>), grid, block, 0, s, p); break;
    case 64: hipLaunchKernelGGL((rowdot_kernel<T, 64>), grid, block, 0, s, p); break;
    case 128: hipLaunchKernelGGL((rowdot_kernel<T, 128>), grid, block, 0, s, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_rowdot(const Params& p, int dtype, hipStream_t s) {
  if (dtype == FHOG_DTYPE_FP32) return launch_rowdot_t<float>(p, s);
  return dtype == FHOG_DTYPE_FP16 ? launch_rowdot_t<_Float16>(p, s) : launch_rowdot_t<__bf16>(p, s);
}

}  // namespace fhog
