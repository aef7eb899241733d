// What follows the scoring of a press when the kept rows do not move inside their own column by the workgroup that
// scored it: selection of every column's kept positions, and the gather of its K and V rows into other tensors.
//
// column_select_kernel: one workgroup per column and part.  The column's keys are held in registers (of the longest rows, 72
// keys per thread of 512, 40 in registers and the rest in LDS), scored on the way in: given scores, per-key sums of the
// SnapKV sweep still to be pooled, or the norms of the key rows themselves.  It either writes the kept positions (a
// compaction launch follows) or, with `parts` workgroups per column that all make the same selection, copies its share of
// the kept rows: a HuggingFace hook has a handful of columns, and eight workgroups that each select are faster than one that
// selects for a second launch.
// Bound by latency: a column's selection is about 8 us of short steps (4096 keys; 24 us with the keys in LDS and digits
// at fixed places), the rows of one layer are then in flight over the whole chip.  288 rows of 30 000 pooled sums: 63 us
// (147 us with 1024 threads and one workgroup to a compute unit, the terms of the pooling read one by one).
#include "fc_norm.h"
#include "fc_rows.h"
#include "fc_select.h"
#include "fc_tail.h"

// Pooling: 64-key groups a wavefront stages at a time, and its floats for them (a kernel of at most 63 reaches 62 keys past
// the groups).  The longest rows stage fewer, so that with their keys in LDS two workgroups fit a compute unit's 160 KB.
// A lane's keys are a whole number of them: a key past the lane's last would be put where the wavefronts stage.
#define CS_GROUPS(KPT) ((KPT) > 16 ? 4 : (KPT) < 8 ? (KPT) : (KPT) % 8 == 0 ? 8 : 6)
#define CS_STAGE(KPT) (CS_GROUPS(KPT) * 64 + 64)

template <int SRC, int DTYPE, int THREADS, int KPT>
__global__ __launch_bounds__(THREADS, KPT > 16 ? 4 : 1) void column_select_kernel(KvView kv, KvView vv, KvView dk, KvView dv, ColumnSelect a) {
  static_assert(KPT % CS_GROUPS(KPT) == 0, "the pooling fills every key of a lane and no other");
  constexpr int EB = DTYPE == FC_F32 ? 4 : 2;
  constexpr int LPR = FC_HEAD_DIM * EB / 16, RPP = THREADS / LPR;
  extern __shared__ __align__(16) int cs_lds[];   // [part_rows] kept positions, the keys that registers do not hold, then what SRC stages
  __shared__ TkSharedRegs<THREADS> sh;
  unsigned* rest = reinterpret_cast<unsigned*>(cs_lds + a.part_rows);
  const int tid = threadIdx.x;
  const int parts = a.parts > 0 ? a.parts : 1;
  // Workgroups go to the XCDs in turn: with the heads as the fastest index all parts of a column read its scores, and rows
  // near each other, through one or two L2 caches, in which the scoring launch, laid out alike, left them.  us per SnapKV hook,
  // parts fastest -> heads: 32 columns of 1000 keys 25.1 -> 24.2, 16 of 2000 25.8 -> 25.2, of 6000 42.3 -> 41.4, 8 of 4000
  // 33.1 -> 32.4; 4 heads the same.  Parts that score their column themselves rather read it through all caches at once (8
  // columns of 333 keys 8.8, heads fastest 8.9).
  const int across = SRC == CS_NORMS ? parts : kv.num_kv_heads;
  const int slow = (int)blockIdx.x / across, fast = (int)blockIdx.x - slow * across;
  const int h = SRC == CS_NORMS ? slow : fast, part = SRC == CS_NORMS ? fast : slow;
  const int b = blockIdx.y, l = blockIdx.z;
  const int S = fc_seq_len(kv, b);
  int kk = a.n_kept ? a.n_kept[b] : a.k;
  kk = min(min(kk, S), a.index_stride);
  if (kk <= 0) return;
  const long long row = ((long long)l * kv.batch + b) * kv.num_kv_heads + h;
  const int tail = min(a.window, S);
  const int n = S - tail, want = kk - tail;
  const int per = a.parts > 0 ? (kk + parts - 1) / parts : 0;
  const int p0 = part * per, p1 = min(kk, p0 + per);
  int* idx_row = a.indices + row * a.index_stride;
  auto emit = [&](int pos, int i) {
    if (a.parts == 0) idx_row[pos] = i;
    else if (pos >= p0 && pos < p1) cs_lds[pos - p0] = i;
  };
  if (n <= 0) {              // every position is a window position: the first kept-count of them
    for (int i = tid; i < kk; i += THREADS) emit(i, i);
  } else if (want < 0) {     // not a selection that keeps the window; the host does not ask for it
    return;
  } else if (want >= n) {    // everything (want == n) stays
    for (int i = tid; i < kk; i += THREADS) emit(i, i);
  } else if (want == 0) {    // the window alone
    for (int i = tid; i < tail; i += THREADS) emit(i, n + i);
  } else {
    const float* in = a.in + row * a.stride;
    if constexpr (SRC == CS_NORMS) {
      // the arithmetic of knorm_kernel; of a short column twice as many rows per lane in flight
      constexpr int NR = KPT == 1 ? 8 : 4;
      float* sc = reinterpret_cast<float*>(cs_lds + a.part_rows + TK_LDS_KEYS(THREADS, KPT));
      const int sub = tid % LPR, rg = tid / LPR;
      const char* kbase = kv.base + ((long long)l * kv.stride_layer + (long long)h * kv.stride_head) * EB + sub * 16;
      for (int r0 = 0; r0 < n; r0 += RPP * NR) {
        uint4 x[NR];
        unsigned live = 0;
#pragma unroll
        for (int u = 0; u < NR; ++u) {
          if (r0 + u * RPP >= n) continue;         // wave-uniform: no loads of rows that are not there
          long long off = fc_token_offset(kv, b, min(r0 + u * RPP + rg, n - 1));
          live |= off >= 0 ? (1u << u) : 0u;
          off = off < 0 ? 0 : off;
          x[u] = *reinterpret_cast<const uint4*>(kbase + off * EB);
        }
#pragma unroll
        for (int u = 0; u < NR; ++u) {
          if (r0 + u * RPP >= n) continue;
          float part_sum = fc_group_sum<16>(row_sumsq_part<DTYPE>(x[u]));
          if (LPR == 32) part_sum += __shfl_xor(part_sum, 16, 64);
          const int r = r0 + u * RPP + rg;
          if (r < n && sub == 0) sc[r] = (live >> u) & 1u ? -sqrtf(part_sum) : -INFINITY;
        }
      }
      __syncthreads();
      tk_select_row_regs<THREADS, KPT>(sh, rest, [&](int i) { return tk_key(sc[i]); }, n, want, emit);
    } else if constexpr (SRC == CS_SUMS) {
      // Zero-padded moving average of the per-key sums, each key's terms in ascending order like the pooling kernel's.
      // A wavefront stages its own segment, CS_GROUPS keys a lane and the neighbours at both ends at a time, in LDS of its own
      // (terms read from memory one by one made the launch above 40 us longer).
      const TkSegment<THREADS> sg(n);
      const int hw = a.ksz >> 1, lane = tid & 63;
      float* st = reinterpret_cast<float*>(rest + TK_LDS_KEYS(THREADS, KPT)) + (tid >> 6) * CS_STAGE(KPT);
      TkKeys<THREADS, KPT> key(rest);
      constexpr int G = CS_GROUPS(KPT);
      float v[G + 1];                       // what the wavefront stages next, on its way while the keys before it are pooled
      auto fetch = [&](int e0) {
#pragma unroll
        for (int g = 0; g <= G; ++g) v[g] = in[min(max(sg.beg + (e0 + g) * 64 - hw + lane, 0), n - 1)];
        for (int q = 1; q < a.addends; ++q) {
#pragma unroll
          for (int g = 0; g <= G; ++g) v[g] += in[q * a.addend_stride + min(max(sg.beg + (e0 + g) * 64 - hw + lane, 0), n - 1)];
        }
      };
      fetch(0);
#pragma unroll
      for (int e0 = 0; e0 < KPT; e0 += G) {
#pragma unroll
        for (int g = 0; g <= G; ++g) {
          const int x = sg.beg + (e0 + g) * 64 - hw + lane;
          st[g * 64 + lane] = x >= 0 && x < n ? v[g] : 0.f;
        }
        if (e0 + G < KPT) fetch(e0 + G);
        tk_wave_sync();
        float s[G];
#pragma unroll
        for (int g = 0; g < G; ++g) s[g] = 0.f;
        for (int j = 0; j < a.ksz; ++j) {
#pragma unroll
          for (int g = 0; g < G; ++g) s[g] += st[g * 64 + lane + j];
        }
        tk_wave_sync();
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int e = e0 + g;
          key.set(e, e < sg.live && sg.pos(e) < sg.end ? tk_key(s[g] * a.out_mul) : 0u);
        }
        if constexpr (KPT > G) __builtin_amdgcn_sched_barrier(0);
      }
      tk_select_loaded<THREADS, KPT>(sh, sg, key, want, emit);
    } else {
      tk_select_row_regs<THREADS, KPT>(sh, rest, [&](int i) { return tk_key(in[i]); }, n, want, emit);
    }
    for (int i = tid; i < tail; i += THREADS) emit(want + i, n + i);
  }
  if (a.parts == 0) return;
  __syncthreads();
  // This workgroup's rows of both planes: source and destination are different tensors, any order will do.  Non-temporal
  // stores: the kept rows take no room from rows still to be gathered, nor from what the layer goes on with; a prefill reads them
  // after its last layer.  us, plain -> non-temporal, hook alone / with a product and a sum on 2048 channels of the layer's tokens
  // behind it, bf16: Knorm, 4 x 4096 keys, 8 heads, 25.9 -> 25.6 / 181 -> 178, 32 heads, 4 x 2000 41.2 -> 41.3 / 121 -> 118, 8 x 2000,
  // 70 % kept, 102 -> 91 / 255 -> 249, 2 x 12 000 162 -> 144 / 385 -> 383, 12 x 4000 251 -> 234 / 718 -> 728; SnapKV, 4 x 4096, 8 heads,
  // 49.8 -> 48.4 / 209 -> 206, 32 heads, 5 x 5000 184 -> 171 / 455 -> 456; of 36 shapes each 0.96 to 1.12 times as fast, 0.98 to 1.03.  Only a
  // pass that reads the rows right behind the hook pays (4 x 4096 doubled 40.6 -> 43.5, a token appended 76.7 -> 80.7).  The
  // loads stay plain: the scoring pass has left part of the rows there.
  const int sub = tid % LPR, rg = tid / LPR;
  const long long kcol = ((long long)l * kv.stride_layer + (long long)h * kv.stride_head) * EB + sub * 16;
  const long long vcol = ((long long)l * vv.stride_layer + (long long)h * vv.stride_head) * EB + sub * 16;
  const long long dkcol = ((long long)l * dk.stride_layer + (long long)h * dk.stride_head) * EB + sub * 16;
  const long long dvcol = ((long long)l * dv.stride_layer + (long long)h * dv.stride_head) * EB + sub * 16;
  constexpr int U = 4;
  for (int j0 = p0; j0 < p1; j0 += RPP * U) {
    cp_u32x4 kb[U], vb[U];
    unsigned kok = 0, vok = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {      // every lane always loads; rows past the end re-read the last one
      const int s = cs_lds[min(j0 + u * RPP + rg, p1 - 1) - p0];
      const long long ko = fc_token_offset(kv, b, s), vo = fc_token_offset(vv, b, s);
      kok |= ko >= 0 ? (1u << u) : 0u;
      vok |= vo >= 0 ? (1u << u) : 0u;
      kb[u] = *reinterpret_cast<const cp_u32x4*>(kv.base + kcol + max(ko, 0ll) * EB);
      vb[u] = *reinterpret_cast<const cp_u32x4*>(vv.base + vcol + max(vo, 0ll) * EB);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = j0 + u * RPP + rg;
      if (j >= p1) continue;
      const long long ko = fc_token_offset(dk, b, j), vo = fc_token_offset(dv, b, j);
      if (ko >= 0 && ((kok >> u) & 1u)) fc_store16<true>(dk.base + dkcol + ko * EB, kb[u]);
      if (vo >= 0 && ((vok >> u) & 1u)) fc_store16<true>(dv.base + dvcol + vo * EB, vb[u]);
    }
  }
}

int fc_column_select(const char* who, int src, const fc_kv_view* keys, const fc_kv_view* values, const fc_kv_view* out_k,
                     const fc_kv_view* out_v, ColumnSelect a, hipStream_t st) {
  const int n = keys->max_seq_len;
  static_assert(512 * 72 >= FC_SELECT_MAX_KEYS, "the longest rows are held by 512 threads of 72 keys");
  FC_REQUIRE(n <= FC_SELECT_MAX_KEYS, FC_EUNSUPPORTED, "%s: %d keys in a column (at most %d)", who, n, FC_SELECT_MAX_KEYS);
  const int parts = a.parts > 0 ? a.parts : 1;
  a.part_rows = a.parts > 0 ? (a.index_stride + parts - 1) / parts : 0;
  const KvView kv = fc_make_view(keys), vv = fc_make_view(values);
  const KvView dk = fc_make_view(out_k ? out_k : keys), dv = fc_make_view(out_v ? out_v : values);
  FC_REQUIRE((long long)keys->num_kv_heads * parts <= 0x7fffffffLL, FC_EUNSUPPORTED, "%s: grid too large", who);
  dim3 grid(keys->num_kv_heads * parts, keys->batch, keys->num_layers);
  FC_REQUIRE(src != CS_SUMS || (a.ksz >= 1 && a.ksz <= 63), FC_EINVAL, "%s: kernel_size %d", who, a.ksz);
#define CS_LAUNCH(SRC, DT, TH, KPT)                                                                               \
  do {                                                                                                            \
    const size_t lds = 4 * ((size_t)a.part_rows + TK_LDS_KEYS(TH, KPT) +                                          \
                            (SRC == CS_NORMS ? n : SRC == CS_SUMS ? TH / 64 * CS_STAGE(KPT) : 0));                \
    FC_REQUIRE(lds <= 120 * 1024, FC_EUNSUPPORTED, "%s: %zu bytes of LDS per workgroup", who, lds);                \
    FC_ALLOW_LDS((column_select_kernel<SRC, DT, TH, KPT>), 120 * 1024);                                            \
    hipLaunchKernelGGL((column_select_kernel<SRC, DT, TH, KPT>), grid, dim3(TH), lds, st, kv, vv, dk, dv, a);       \
  } while (0)
  // Keys per thread as few as hold the row: the passes over them are unrolled, and keys that are not there still cost their
  // share.  512 threads up to 4096 keys, 1024 for longer rows, where lanes shorten the chain, and 512 again for the longest,
  // two workgroups to a compute unit (288 rows are then one round, not two).  us per hook, half kept, 256 threads of 2 keys
  // up to 512, 512 of 8 up to 4096, 1024 of 16 up to 16384 -> this: Knorm, 8 columns of 333 keys 10.7 -> 9.2, of 500
  // 12.5 -> 10.4, of 1000 (norms first) 11.9 -> 11.0, of 5000 22.3 -> 19.7, of 9000 28.1 -> 27.0; SnapKV, 8 of 1000
  // 25.0 -> 23.6, 32 of 2000 35.2 -> 33.9, of 7000 81.8 -> 79.3.
#define CS_SIZE(SRC, DT)                               \
  if (n <= 512) CS_LAUNCH(SRC, DT, 512, 1);            \
  else if (n <= 1024) CS_LAUNCH(SRC, DT, 512, 2);      \
  else if (n <= 2048) CS_LAUNCH(SRC, DT, 512, 4);      \
  else if (n <= 4096) CS_LAUNCH(SRC, DT, 512, 8);      \
  else if (n <= 8192) CS_LAUNCH(SRC, DT, 1024, 8);     \
  else if (n <= 12288) CS_LAUNCH(SRC, DT, 1024, 12);   \
  else if (n <= 16384) CS_LAUNCH(SRC, DT, 1024, 16);   \
  else CS_LAUNCH(SRC, DT, 512, 72)
#define CS_SIZE_SHORT(SRC, DT)                         \
  if (n <= 512) CS_LAUNCH(SRC, DT, 512, 1);            \
  else CS_LAUNCH(SRC, DT, 512, 8)
#define CS_DTYPE(SRC)                                                                                 \
  if (keys->dtype == FC_F32) { CS_SIZE(SRC, FC_F32); }                                                \
  else { CS_SIZE(SRC, FC_F16); }          /* rows of two-byte elements are moved, not computed with */
  if (src == CS_SCORES) {
    CS_DTYPE(CS_SCORES);
  } else if (src == CS_SUMS) {
    CS_SIZE(CS_SUMS, FC_F16);
  } else if (keys->dtype == FC_F32) {
    CS_SIZE_SHORT(CS_NORMS, FC_F32);
  } else if (keys->dtype == FC_BF16) {
    CS_SIZE_SHORT(CS_NORMS, FC_BF16);
  } else {
    CS_SIZE_SHORT(CS_NORMS, FC_F16);
  }
#undef CS_DTYPE
#undef CS_SIZE_SHORT
#undef CS_SIZE
#undef CS_LAUNCH
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}

static int cs_check(const char* who, const fc_kv_view* keys, const fc_kv_view* values, const fc_kv_view* out_k,
                    const fc_kv_view* out_v, int k) {
  int rc;
  for (const fc_kv_view* v : {keys, values, out_k, out_v})
    if ((rc = fc_check_view(v, who))) return rc;
  for (const fc_kv_view* v : {values, out_k, out_v})
    FC_REQUIRE(keys->dtype == v->dtype && keys->num_layers == v->num_layers && keys->batch == v->batch &&
                   keys->num_kv_heads == v->num_kv_heads,
               FC_EINVAL, "%s: views disagree on dtype/layers/batch/heads", who);
  FC_REQUIRE(keys->max_seq_len == values->max_seq_len, FC_EINVAL, "%s: key and value views disagree on length", who);
  FC_REQUIRE(k >= 0 && k <= keys->max_seq_len && k <= out_k->max_seq_len && k <= out_v->max_seq_len, FC_EINVAL,
             "%s: k=%d exceeds a view's max_seq_len", who, k);
  return FC_OK;
}

// Whether a press into other tensors should select and gather in launches of their own.  The workgroups that gather a
// column each select it as well; of columns of more than 4096 keys there is one round of them (fc_gather_parts), and what
// they lose against a gather over the whole chip is the time the selection takes, with fewer rows in flight after it: apart
// where a workgroup's share is large.  us per hook, gather inside -> apart: Knorm, 24 columns of 5000 keys, 350 rows a share
// 30.7, 37.4; 64 of 8000, 1400 a share 91.8, 101.6; 128 of 8000, 2800 a share 210, 210; of 12000, 4200 a share 317, 309, 1200 a
// share 160, 169; 192 of 5000, 3500 a share 200, 199; 256 of 8000, 1600 a share 205, 214, 5600 a share 417, 396; SnapKV, 24 of 7000
// 60.5, 66.5, 128 of 7000 177, 187.  Above 16 384 keys likewise: Knorm, 32 of 20 000, 1250 a share 113, 119, 64 of 20 000,
// 2500 a share 227, 230, of 30 000, 3750 a share 336, 331, 128 of 20 000, 2000 a share 269, 268, 5000 a share 424, 407; SnapKV,
// 64 of 30 000, 1500 a share 403, 406, 3750 a share 512, 506.  Shorter columns, two and more workgroups to a compute unit: 96 of
// 4000 76, 77, 64 of 2000 29, 34.
extern "C" int fc_press_gather_apart(int32_t columns, int32_t max_seq_len, int32_t k) {
  if (columns <= 0 || k <= 0 || max_seq_len <= CS_WIDE) return 0;
  const int parts = fc_gather_parts(columns, max_seq_len, k);
  return (long long)columns * parts > fc_compute_units() || (k + parts - 1) / parts > 2600;
}

extern "C" int fc_knorm_press_into(const fc_kv_view* keys, const fc_kv_view* values, const fc_kv_view* out_k,
                                   const fc_kv_view* out_v, int32_t k, float* scores, int32_t score_stride, int32_t* indices,
                                   void* stream) {
  const char* who = "fc_knorm_press_into";
  int rc = cs_check(who, keys, values, out_k, out_v, k);
  if (rc) return rc;
  if (k == 0 || keys->max_seq_len == 0) return FC_OK;
  ColumnSelect a{};
  a.k = a.index_stride = k;
  a.parts = indices ? 0 : fc_gather_parts((long long)keys->num_layers * keys->batch * keys->num_kv_heads, keys->max_seq_len, k);
  a.indices = indices;
  if (!scores) {   // the workgroups that select a column score it as well
    FC_REQUIRE(keys->max_seq_len <= CS_NORMS_MAX, FC_EUNSUPPORTED, "%s: columns of more than %d keys need a score buffer", who,
               CS_NORMS_MAX);
  } else if ((rc = fc_knorm_score(keys, scores, score_stride, stream))) {
    return rc;
  }
  a.in = scores;
  a.stride = score_stride;
  rc = fc_column_select(who, scores ? CS_SCORES : CS_NORMS, keys, values, out_k, out_v, a, (hipStream_t)stream);
  return rc || !indices ? rc : fc_compact(keys, values, out_k, out_v, indices, k, keys->num_kv_heads, k, nullptr, stream);
}
