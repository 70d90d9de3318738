// The default bias of ragged batches, -log(key length of each sequence) in
// fp32 (sigmoid_triton_padded.py:995-996), from the lengths on the device.
// Launch-bound: one launch in place of the conversion, logarithm and negation
// (and the difference of packed offsets) as element-wise operators, each of
// which costs the stream about 4.5 us at these sizes, more than a tenth of a
// decoding step.  Built with -ffp-contract=off: the logarithm's bits are then
// the element-wise operator's (with contraction 38 % of the first million
// lengths differ in the last bit).
#include <hip/hip_runtime.h>

#include "../../include/sigattn.h"

namespace {
__global__ __launch_bounds__(256) void default_bias_kernel(const int32_t *lens, const int32_t *cu, int64_t B,
                                                           float *bias) {
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (b >= B) return;
  // Offsets differ as the int32 tensors would (modulo 2^32).
  const int32_t n = lens != nullptr ? lens[b] : (int32_t)((uint32_t)cu[b + 1] - (uint32_t)cu[b]);
  bias[b] = -logf((float)n);
}
}  // namespace

extern "C" int sigattn_default_bias(const int32_t *seq_lens, const int32_t *cu_seqlens, int64_t B, float *bias,
                                    void *stream) {
  if (B < 0 || (B + 255) / 256 > INT32_MAX) return SIGATTN_ERR_SHAPE;
  if (B == 0) return SIGATTN_OK;
  if (bias == nullptr || (seq_lens == nullptr && cu_seqlens == nullptr)) return SIGATTN_ERR_NULL_ARG;
  if (seq_lens != nullptr && cu_seqlens != nullptr) return SIGATTN_ERR_LAYOUT;
  (void)hipGetLastError();
  default_bias_kernel<<<dim3((unsigned)((B + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>(seq_lens, cu_seqlens,
                                                                                               B, bias);
  return hipGetLastError() == hipSuccess ? SIGATTN_OK : SIGATTN_ERR_LAUNCH;
}
