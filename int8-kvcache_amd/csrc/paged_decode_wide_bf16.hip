// The range kernel for GQA groups above 16 over one cache type (bf16), instantiated here so that
// the cache types compile in parallel (see paged_decode_wide.h).

#include "paged_decode_wide.h"

namespace int8kv {

int launch_wide_bf16(const DecodeArgs& a, const HostPlan& hp, int query_dtype, hipStream_t s) {
  return hp.pad ? launch_wide_q<kBF16, true>(a, hp, query_dtype, s)
                : launch_wide_q<kBF16, false>(a, hp, query_dtype, s);
}

}  // namespace int8kv
