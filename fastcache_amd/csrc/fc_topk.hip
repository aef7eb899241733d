// Row-wise top-k selection with lowest-index tie-break and ascending-index output.
//
// One workgroup per score row, the row's order-preserving 32-bit keys in registers (tk_select_row_regs): 256 threads for
// rows of up to 512 scores, 512 up to 4096, 1024 up to 16 384, where few such rows make a launch and each has to be
// walked by more lanes, 512 again up to 36 864 with part of the keys in LDS, so that two rows share a compute unit (288
// rows of 30 000: 47 us; 71 us with 1024 threads and one row at a time).  Longer
// rows are selected with the keys re-read from global memory (L2-resident), four passes of 8 bits over an LDS histogram
// and an ordered pass.  Bound by the chain of short steps of a row, not by its bytes.
#include "fc_select.h"

#define TK_MAX_REG_KEYS (512 * 72)

// KPT = keys per thread in registers; 0 = re-read from memory
template <int TK_THREADS, int KPT>
__global__ __launch_bounds__(TK_THREADS, KPT > 16 ? 4 : 1) void topk_kernel(const float* __restrict__ scores,
                                                          int score_stride, int len,
                                                          const int* __restrict__ row_lens,
                                                          int rows_per_len, int row_lens_mod, int k,
                                                          const int* __restrict__ n_kept,
                                                          int* __restrict__ indices, int index_stride) {
  __shared__ TkArea<TK_THREADS> sh;
  __shared__ unsigned rest[TK_LDS_KEYS(TK_THREADS, KPT) + 1];

  const int r = blockIdx.x;
  const int tid = threadIdx.x;
  const int li = (row_lens || n_kept) ? (r / rows_per_len) % row_lens_mod : 0;
  int n = row_lens ? row_lens[li] : len;
  if (n > len) n = len;
  int kk = n_kept ? n_kept[li] : k;
  if (kk > n) kk = n;
  if (kk > index_stride) kk = index_stride;
  if (n <= 0 || kk <= 0) return;
  const float* row = scores + (long long)r * score_stride;
  int* out = indices + (long long)r * index_stride;

  if (kk == n) {
    for (int i = tid; i < n; i += TK_THREADS) out[i] = i;
    return;
  }
  auto key_at = [&](int i) -> unsigned { return tk_key(row[i]); };
  auto emit = [&](int pos, int i) { out[pos] = i; };
  if constexpr (KPT > 0)
    tk_select_row_regs<TK_THREADS, KPT>(sh.reg_keys, rest, key_at, n, kk, emit);
  else
    tk_select_row<TK_THREADS>(sh.lds_keys, key_at, n, kk, emit);
}

extern "C" int fc_topk_select(const float* scores, int32_t score_stride, int32_t rows, int32_t len,
                              const int32_t* row_lens, int32_t rows_per_len, int32_t row_lens_mod,
                              int32_t k,
                              const int32_t* n_kept, int32_t* indices, int32_t index_stride,
                              void* stream) {
  FC_REQUIRE(scores && indices, FC_EINVAL, "fc_topk_select: null pointer");
  FC_REQUIRE(rows >= 0 && len >= 0 && score_stride >= len && index_stride >= 0, FC_EINVAL,
             "fc_topk_select: bad sizes rows=%d len=%d score_stride=%d index_stride=%d", rows, len,
             score_stride, index_stride);
  FC_REQUIRE(n_kept != nullptr || (k >= 0 && k <= index_stride), FC_EINVAL,
             "fc_topk_select: k=%d does not fit index_stride=%d", k, index_stride);
  FC_REQUIRE((row_lens == nullptr && n_kept == nullptr) || (row_lens_mod > 0 && rows_per_len > 0),
             FC_EINVAL, "fc_topk_select: rows_per_len and row_lens_mod must be positive when per-row sizes are given");
  if (rows == 0 || len == 0) return FC_OK;
  hipStream_t st = (hipStream_t)stream;
#define TK_LAUNCH(TH, KPT)                                                                                         \
  hipLaunchKernelGGL((topk_kernel<TH, KPT>), dim3(rows), dim3(TH), 0, st, scores, score_stride, len, row_lens,     \
                     rows_per_len, row_lens_mod, k, n_kept, indices, index_stride)
  if (len <= 512) TK_LAUNCH(256, 2);
  else if (len <= 4096) TK_LAUNCH(512, 8);
  else if (len <= 16384) TK_LAUNCH(1024, 16);
  else if (len <= TK_MAX_REG_KEYS) TK_LAUNCH(512, 72);
  else TK_LAUNCH(1024, 0);
#undef TK_LAUNCH
  FC_CHECK_LAUNCH("fc_topk_select");
  return FC_OK;
}
