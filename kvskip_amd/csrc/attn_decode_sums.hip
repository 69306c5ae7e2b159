// The dense split pass over a ragged batch with per-block statistics and key sums
// (kvskip_attn_args.key_sums): a planner's first step reads the prefix's K once for both. Before, the sums
// were a pass over K of their own (kvskip_block_sums; figures at block_key_sums). Kept apart from attn_decode.hip so the two compile in parallel.
#include "attn_decode.hpp"

namespace kvs {
namespace {

template <int D, int G>
__global__ void __launch_bounds__(NT, 2) decode_sums_kernel(const AttnP p, float* sums, int cap) {
  decode_body<D, G, false, true, true, true, true, false, false, true>(p, blockIdx.x, nullptr, sums, cap);
}

}  // namespace

hipError_t launch_decode_sums(const AttnP& p, int D, int G, float* sums, int cap, int phase, hipStream_t s) {
#define KVS_CASE(DD, GG)                                                                              \
  if (D == DD && G == GG) {                                                                           \
    hipLaunchKernelGGL((decode_sums_kernel<DD, GG>), attn_grid(p), dim3(NT), 0, s, p, sums, cap);     \
    const hipError_t e = hipGetLastError();                                                           \
    return e != hipSuccess || !(phase & 2) ? e : launch_combine(p, D, false, s);                      \
  }
  KVS_FOR_G(KVS_CASE, 64)
  KVS_FOR_G(KVS_CASE, 128)
#undef KVS_CASE
  return hipErrorInvalidValue;
}

}  // namespace kvs
