// Shared by the two files that serve dh_attn_spec (attention_spec.hip, attention_prefill.hip).
#pragma once
#include "attention_keys.h"
#include "dh_common.h"

namespace dh {
// Host-side validation of a spec: 0, or fail().
int attn_spec_check(const char* op, const dh_attn_spec* s);
// The key ranges of a step whose key count is read on the device.
DynKeys attn_spec_keys(const dh_attn_spec* s, const uint32_t* kv_len, int max_kv_len, bool wide);
// Splits of a wide launch for a step that can see `keys` keys at most.
int attn_spec_wide_splits(const dh_attn_spec* s, int keys);
// What a product that merges a step's key splits (dense_gemv.hip) takes of them: a lane each makes a head's factors, which stand in LDS beside the row.
constexpr int kMergedSplits = 64;
constexpr int kMergedFactors = 16384;      // bytes
inline bool product_merges(int heads, int splits) { return splits <= kMergedSplits && (int64_t)4 * heads * (splits + 1) <= kMergedFactors; }
// Key elements that all heads of a token share (a rotated part beside every head's own): head keys are [D own | dim shared],
// row r of the shared part lies ld elements behind row r - 1.  dim 0: none.
struct SharedKey {
  const void* rows;
  int dim;
  int64_t ld;
};
// T queries with the any-shape kernel (the cache rows up to each query's own are written).
int attn_spec_prefill_general(const char* op, const dh_attn_spec* s, const float* d_qkv, const void* K, const void* V,
                              void* d_out, int out_dtype, int ld_out, int T, int start_pos, const SharedKey& shared);
}  // namespace dh
