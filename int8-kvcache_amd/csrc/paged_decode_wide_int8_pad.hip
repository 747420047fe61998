// The range kernel for GQA groups above 16 over one cache type (int8, head_dims below the kernels' 64, 128 and 256), instantiated here so that
// the cache types compile in parallel (see paged_decode_wide.h).

#include "paged_decode_wide.h"

namespace int8kv {

int launch_wide_int8_pad(const DecodeArgs& a, const HostPlan& hp, int query_dtype, hipStream_t s) {
  return launch_wide_q<kI8, true>(a, hp, query_dtype, s);
}

}  // namespace int8kv
