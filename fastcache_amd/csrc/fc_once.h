// SnapKV per-key sums with every logit formed once (fc_once.hip).
#pragma once
#include "fc_common.h"

#define SO_KEYS 256          // keys of a chunk
#define SO_LISTS 8           // lists the columns are shared out over, at most
#define SO_CHUNKS_MAX 48     // chunks of the longest column

// Whether the kernel takes the shape, and whether it is the faster one for sequences of that mean length of which at most
// `kept` tokens stay; whole: instead of one launch per pass.
bool fc_once_takes(const fc_kv_view* keys, int32_t num_q_heads, int32_t window);
bool fc_once_pays(const fc_kv_view* keys, int32_t num_q_heads, int32_t window, int32_t mean_len, int32_t kept, bool whole);
int64_t fc_once_workspace_bytes(int32_t num_layers, int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t window,
                                int32_t max_seq_len);
int fc_once_groups(const fc_kv_view* keys, int32_t num_q_heads, int32_t window);   // of four blocks of 32 window queries
// Per-key sums of the window queries' probabilities into raw[group][column][raw_stride] (keys before the window; rows no longer
// than the window are left as they are): the groups' sums are to be added.  Arguments are checked by the caller.  workgroups:
// at most so many, 0 for two per compute unit.
int fc_once_sums(const char* who, const fc_kv_view* keys, const void* queries, int32_t num_q_heads, int32_t window,
                 int32_t causal_window, float scale, float* raw, int32_t raw_stride, void* workspace, int32_t workgroups,
                 void* stream);
