// amf_prefill.h - launch of the many-row attention kernel (amf_prefill.hip).
#pragma once

#include "amf_attn.h"

namespace amf {

struct PrefillPlan {
  int waves;             // waves of 32 query rows per workgroup
  int64_t tiles;         // workgroups over the rows of one (batch, KV head)
  int64_t n_splits;      // splits of the KV tokens
  int64_t split_tokens;  // tokens per split, a multiple of 64
};

// Fewest query rows of a (batch, KV head) for the tiles: one of 32 columns
// costs the same for 2 rows as for 32, the one-row kernel's cost grows with the
// rows (8 heads, bf16, one-row / tiles, us: 4 batches x 8192 tokens 2 rows 27 /
// 31, 4 rows 42 / 32; 8 x 16384 4 rows 178 / 103, 7 rows 520 / 104).
constexpr int64_t kPrefillMinRows = 4;
// head_dim 256: the (query row, token) pairs that a call has to exceed; below,
// the one-row kernel's shorter chain is the faster (8 / 8 heads, bf16, one-row /
// tiles, GPU us: 4 rows x 1024 tokens 11.9 / 12.8, 16 x 1024 15.7 / 13.9, 4 x 4096
// 17.3 / 16.1).  Twice as many for fp16, whose V takes two terms (16 x 1024 15.4 /
// 16.9, 8 x 4096 25.3 / 20.4), and for split four-wave workgroups (64 x 256 15.1 /
// 18.9, 33 x 1024 28 / 19).  None where several heads of a group share a wave of
// the one-row kernel, which then starts slower: groups that are a multiple of 4
// (32 / 8 heads, 2 x 64 26.6 / 16.0) or, for bf16, of 2 (16 / 8 heads, 4 x 1024
// 16.1 / 12.8).
constexpr int64_t kPrefillMinPairs = 1 << 16;
// Workgroups a launch aims for (all resident at once: 4 waves at 2 waves per
// SIMD, or one wave) and the fewest 64-token chunks of a split.  4 heads a
// group x 16 rows, 4096 tokens: 37 / 23 / 20 us with 8 / 4 / 2 chunks.
constexpr int64_t kPrefillGroups1 = 2048;
constexpr int64_t kPrefillGroups4 = 512;
constexpr int64_t kPrefillMinChunks1 = 1;
constexpr int64_t kPrefillMinChunks4 = 2;
// Most splits: kPrefillSplits, or as many as give kMaxPrefillSplits workgroups
// (16 rows x 16384 tokens, 64 / 256 splits: one KV head of 64 dims 14.6 / 10.0 us;
// 8 of 128 26 / 34 us, spent on the partials).
constexpr int64_t kPrefillSplits = 64;
constexpr int64_t kMaxPrefillSplits = 256;

// Whether a shape takes the many-row kernel, and with at most max_splits
// splits how it is cut.
bool prefill_plan(int64_t batch, int32_t num_q_heads, int32_t num_kv_heads, int64_t q_len,
                  int64_t kv_len, int32_t head_dim, int64_t max_splits, PrefillPlan* p);

// Whether the tiles are the faster for a call that prefill_plan takes.
bool prefill_pays(const PrefillPlan& p, int64_t batch, int32_t num_q_heads, int32_t num_kv_heads,
                  int64_t q_len, int64_t kv_len, int32_t head_dim, bool fp16);

// Workspace bytes of one split (none are needed when there is only one).
int64_t prefill_split_bytes(int64_t batch, int32_t num_q_heads, int64_t q_len, int32_t head_dim);

// Launches the kernel and, for more than one split, the merge.  dtype bf16 or
// fp16; q, k, v 16-byte aligned (int4: codes 4-byte aligned, a.k_scales and
// a.v_scales set).
void launch_prefill(const AttnArgs& a, int32_t dtype, int32_t out_dtype, bool int4, float* part,
                    const PrefillPlan& p, hipStream_t st);

// The one-row split kernel's merge (amf_attn.hip): a workgroup per query row.
void launch_merge(const AttnArgs& a, int32_t out_dtype, int64_t rows, const float* part,
                  int64_t n_splits, hipStream_t st);

}  // namespace amf
