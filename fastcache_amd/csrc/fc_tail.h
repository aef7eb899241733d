// Selection of every column's kept positions from scores, per-key sums or key norms, with or without the gather of the
// kept rows into other tensors (fc_tail.hip).
#pragma once
#include "fc_common.h"

struct ColumnSelect {
  const float* in;      // [layer][batch][kv head][stride]: scores (SRC 0) or per-key sums (SRC 1)
  int stride;
  int addends;          // arrays of sums (SRC 1) that are added, addend_stride floats apart (0: one)
  long long addend_stride;
  int k;                // kept positions per row when n_kept is null
  const int* n_kept;    // [batch] in device memory, or null
  int window;           // the last `window` positions of a sequence are kept and not entered (0: all are entered)
  int ksz;              // width of the moving average (SRC 1)
  float out_mul;
  int* indices;         // [layer][batch][kv head][index_stride], written when parts == 0
  int index_stride;
  int parts;            // workgroups per column that gather; 0 = write the indices instead
  int part_rows;        // rows a workgroup gathers at most (its LDS)
};

enum { CS_SCORES = 0, CS_SUMS = 1, CS_NORMS = 2 };
#define CS_WIDE 4096               // longer columns get one gathering workgroup per compute unit (fc_gather_parts)
#define CS_NORMS_MAX 4096         // columns that the gathering workgroups score themselves: their scores lie in LDS

// Launches the selection for columns of at most keys->max_seq_len keys; the out views are read only when a.parts > 0.
int fc_column_select(const char* who, int src, const fc_kv_view* keys, const fc_kv_view* values, const fc_kv_view* out_k,
                     const fc_kv_view* out_v, ColumnSelect a, hipStream_t st);

// Workgroups per column for a gather, no share below 64 rows: about two per compute unit in all, one for columns above
// CS_WIDE.  Every one of them selects its whole column.  Up to 16 384 keys 1024 threads do, of which a compute unit holds one
// workgroup: what does not fit the first round would select behind it.  Of longer columns it holds two (512 threads), but
// they share its time and gather half as many rows each for one selection more.  us per hook, half kept, one -> two per
// compute unit: Knorm, 32 columns of 20 000 keys 113 -> 112, 64 228 -> 235, of 30 000 330 -> 344; SnapKV, 32 of 20 000
// 195 -> 194, of 30 000 279 -> 318, 64 of 20 000 359 -> 384; up to 16 columns get the 16 parts they may have either way.
static inline int fc_gather_parts(long long cols, int n, int k) {
  const long long ncu = fc_compute_units();
  long long p = n > CS_WIDE ? ncu / cols : (2 * ncu + cols - 1) / cols;
  if (p > (k + 63) / 64) p = (k + 63) / 64;
  p = p < 1 ? 1 : p > 16 ? 16 : p;
  const int lds = (k + 8191) / 8192;      // a share's positions are in LDS, at most 32 KB of them
  return (int)(p < lds ? lds : p);
}
