// few_merge.h -- the split-KV partials of one sequence's bf16 decode attention, as
// decode.hip leaves them for few_rows.hip's o_proj.
#pragma once

#include "common.h"

namespace crane {

constexpr int kFewMergeSplits = 8;      // partials per head the merging product takes
constexpr int kFewMergeOutputs = 1024;  // outputs: one workgroup per CU
constexpr int kFewMergeHeads = 16;      // heads: one 16-byte piece of the row per thread

struct FewMerge {
    const float* rows;  // bf16 rows [Hq, nsplit, 128], each normalised by its chunk's sum
    const float* ml;    // (max, sum) [Hq, nsplit]
    const int32_t* kv_len;
    int max_kv, chunk, nsplit;
};

// y[N] = attn w[N, K]^T, K = Hq 128 a multiple of 512, Hq <= kFewMergeHeads, N <= kFewMergeOutputs, 1 <
// nsplit <= kFewMergeSplits.  attn: the row of a sequence of one chunk.
int few_merge_linear(const FewMerge& m, const void* attn, const void* w, void* y, int N, int K, hipStream_t st);

}  // namespace crane
