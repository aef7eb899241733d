// Selection of every column's kept positions from scores, per-key sums or key norms, with or without the gather of the
// kept rows into other tensors (fc_tail.hip).
#pragma once
#include "fc_common.h"

struct ColumnSelect {
  const float* in;      // [layer][batch][kv head][stride]: scores (SRC 0) or per-key sums (SRC 1)
  int stride;
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
#define CS_WIDE 4096               // longer columns are selected by 1024 threads
#define CS_NORMS_MAX 4096         // columns that the gathering workgroups score themselves: their scores lie in LDS

// Launches the selection for columns of at most keys->max_seq_len keys; the out views are read only when a.parts > 0.
int fc_column_select(const char* who, int src, const fc_kv_view* keys, const fc_kv_view* values, const fc_kv_view* out_k,
                     const fc_kv_view* out_v, ColumnSelect a, hipStream_t st);

// Workgroups per column for a gather, no share below 64 rows: about two per compute unit in all; one where columns are long
// enough to be selected by 1024 threads each (CS_WIDE), of which a compute unit holds one workgroup: what does not fit the
// first round would select its column behind it.
static inline int fc_gather_parts(long long cols, int n, int k) {
  const long long ncu = fc_compute_units();
  long long p = n > CS_WIDE ? ncu / cols : (2 * ncu + cols - 1) / cols;
  if (p > (k + 63) / 64) p = (k + 63) / 64;
  p = p < 1 ? 1 : p > 16 ? 16 : p;
  const int lds = (k + 8191) / 8192;      // a share's positions are in LDS, at most 32 KB of them
  return (int)(p < lds ? lds : p);
}
