// Library-wide pieces of libfastcache_hip: ABI version, per-thread error text, view validation.
#include <string.h>
#include "fc_common.h"
#include <atomic>

static thread_local char g_err[512] = "";

void fc_set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

extern "C" int fc_abi_version(void) { return FC_ABI_VERSION; }
extern "C" const char* fc_last_error(void) { return g_err; }

int fc_compute_units() {
  static std::atomic<int> cus[64];
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if ((n = cus[dev].load(std::memory_order_relaxed)) > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
  cus[dev].store(n, std::memory_order_relaxed);
  return n;
}

int fc_check_view(const fc_kv_view* v, const char* who) {
  FC_REQUIRE(v != nullptr, FC_EINVAL, "%s: null view", who);
  FC_REQUIRE(v->base != nullptr, FC_EINVAL, "%s: null base pointer", who);
  FC_REQUIRE(v->dtype == FC_F32 || v->dtype == FC_F16 || v->dtype == FC_BF16, FC_EINVAL,
             "%s: unknown dtype %d", who, v->dtype);
  FC_REQUIRE(v->head_dim == FC_HEAD_DIM, FC_EUNSUPPORTED, "%s: head_dim %d (only %d is built)", who,
             v->head_dim, FC_HEAD_DIM);
  FC_REQUIRE(v->num_layers > 0 && v->batch > 0 && v->num_kv_heads > 0, FC_EINVAL,
             "%s: layers/batch/heads must be positive (%d, %d, %d)", who, v->num_layers, v->batch,
             v->num_kv_heads);
  FC_REQUIRE(v->max_seq_len >= 0, FC_EINVAL, "%s: negative max_seq_len", who);
  FC_REQUIRE(v->batch <= 65535 && v->num_layers <= 65535, FC_EUNSUPPORTED,
             "%s: batch/layers beyond grid limits", who);
  if (v->block_tables) {
    FC_REQUIRE(v->block_size > 0, FC_EINVAL, "%s: block_size must be positive", who);
    FC_REQUIRE((int64_t)v->table_stride * v->block_size >= v->max_seq_len, FC_EINVAL,
               "%s: block table (%d entries of %d tokens) shorter than max_seq_len %d", who,
               v->table_stride, v->block_size, v->max_seq_len);
  }
  // 16-byte vector accesses: every stride must keep rows 16-byte aligned.
  const int64_t q = 16 / fc_elem_bytes(v->dtype);
  FC_REQUIRE(((uintptr_t)v->base & 15) == 0, FC_EINVAL, "%s: base not 16-byte aligned", who);
  FC_REQUIRE(v->stride_layer % q == 0 && v->stride_block % q == 0 && v->stride_batch % q == 0 &&
                 v->stride_token % q == 0 && v->stride_head % q == 0,
             FC_EINVAL, "%s: strides must be multiples of %lld elements", who, (long long)q);
  return FC_OK;
}

// ---- a few numbers from the host to the device ------------------------------------------------------------------
// They travel as the kernel's arguments: no staging memory, no event that guards it, and a launch where the runtime's copy
// of pinned memory is a call, an event and a kernel of its own.  us per pass, copy -> arguments: Knorm on one sequence of 1024
// tokens 315 -> 312, of 571 51.1 -> 48.9; a decode step of one short sequence by its graph 91.9 -> 87.1, of three eagerly 286 -> 281; MLP on
// two sequences of 590 and 628 320 -> 300.  The arguments are as long as the smallest of three sizes that holds the numbers,
// since the runtime copies all of them.
template <int WORDS>
struct UploadWords {
  uint32_t w[WORDS];
};
template <int WORDS>
__global__ __launch_bounds__(256) void upload_kernel(const UploadWords<WORDS> a, uint32_t* __restrict__ dst, int words) {
  for (int i = threadIdx.x; i < words; i += 256) dst[i] = a.w[i];
}

template <int WORDS>
static void upload(void* dst, const void* host, int words, hipStream_t st) {
  UploadWords<WORDS> a;
  memcpy(a.w, host, (size_t)words * 4);
  hipLaunchKernelGGL((upload_kernel<WORDS>), dim3(1), dim3(256), 0, st, a, (uint32_t*)dst, words);
}

extern "C" int fc_upload(void* dst, const void* host, int32_t bytes, void* stream) {
  const char* who = "fc_upload";
  FC_REQUIRE(dst && host && bytes >= 0, FC_EINVAL, "%s: bad arguments", who);
  FC_REQUIRE(bytes % 4 == 0 && ((uintptr_t)dst & 3) == 0, FC_EINVAL, "%s: whole 4-byte words only", who);
  FC_REQUIRE(bytes <= FC_UPLOAD_MAX, FC_EUNSUPPORTED, "%s: %d bytes (at most %d)", who, bytes, FC_UPLOAD_MAX);
  if (bytes == 0) return FC_OK;
  const int words = bytes / 4;
  hipStream_t st = (hipStream_t)stream;
  if (words <= 64) upload<64>(dst, host, words, st);
  else if (words <= 256) upload<256>(dst, host, words, st);
  else upload<FC_UPLOAD_MAX / 4>(dst, host, words, st);
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}
