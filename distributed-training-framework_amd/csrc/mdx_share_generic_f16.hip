// Instantiates the reduce-scatter share of fp16 contributions for the
// remaining (reduction, shard) dtype pairs, at every width class
// (runtime W).
#include "mdx_reduce_impl.h"

namespace mdx {

hipError_t launch_share_generic_f16(int acc_dtype, int out_dtype, int wmax, const PieceBatch& b, const ReduceParams& p,
                                    hipStream_t stream) {
  return reduce_impl::launch_share_generic_for<f16>(acc_dtype, out_dtype, wmax, b, p, stream);
}

}  // namespace mdx
