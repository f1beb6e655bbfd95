// Per-row parameter arrays of a call whose parameters are the same for every
// row (one launch in place of one fill per parameter).
#include "fl_kernels.h"

namespace fl {

namespace {

__global__ void k_fill_rows(const fl_row_values v, const int64_t batch, uint32_t* out) {
  const int64_t b = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  out[b] = __float_as_uint(v.temperature);
  out[batch + b] = static_cast<uint32_t>(v.top_k);
  out[2 * batch + b] = __float_as_uint(v.top_p);
  out[3 * batch + b] = __float_as_uint(v.min_p);
  out[4 * batch + b] = __float_as_uint(v.rep_penalty);
  out[5 * batch + b] = static_cast<uint32_t>(v.hist_len);
}

}  // namespace

hipError_t launch_fill_rows(const fl_row_values& v, int64_t batch, void* out, hipStream_t s) {
  constexpr int NT_FILL = 256;
  const dim3 grid(static_cast<unsigned>((batch + NT_FILL - 1) / NT_FILL));
  hipLaunchKernelGGL(k_fill_rows, grid, dim3(NT_FILL), 0, s, v, batch, static_cast<uint32_t*>(out));
  return hipGetLastError();
}

}  // namespace fl
