// The bf16 instances of fq_tile_kernel.
#include "flatquant_tile.h"

namespace qo {

template <>
bool launch_tile<BF16T>(const void* x, int64_t tokens, int64_t x_ld, const void* left, const void* right, int M, int N,
                       float clip, int pack, void* out_codes, float* out_scales, hipStream_t stream) {
  return launch_tile_any<BF16T>(x, tokens, x_ld, left, right, M, N, clip, pack, out_codes, out_scales, stream);
}

}  // namespace qo
