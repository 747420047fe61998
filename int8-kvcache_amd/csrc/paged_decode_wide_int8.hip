// The range kernel for GQA groups above 16 over one cache type (int8), instantiated here so that
// the cache types compile in parallel (see paged_decode_wide.h).

#include "paged_decode_wide.h"

namespace int8kv {

int launch_wide_int8(const DecodeArgs& a, const HostPlan& hp, int query_dtype, hipStream_t s) {
  return launch_wide_q<kI8, false>(a, hp, query_dtype, s);
}

}  // namespace int8kv
