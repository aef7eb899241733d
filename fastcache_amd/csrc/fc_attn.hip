// Decode-side kernels over the paged cache: append one K/V row per sequence, advance the lengths,
// and single-query paged attention (split over chunks of 256 to 1024 tokens, then merged).
//
// Attention is HBM-bound (one pass over K and V, ~1 FLOP per byte per query head), so the kernel is
// organised around keeping loads in flight.  A workgroup owns one (sequence, kv head, chunk of
// 256..1024 tokens, a multiple of 32 the host picks per launch) and serves all query heads of the group from the same K/V bytes;
// each of its four wavefronts streams its 32-token K tiles and then the matching V tiles from global memory straight
// into a private two-stage LDS ring (global_load_lds, rows XOR-swizzled), 16 KB per wavefront in
// flight, no workgroup barrier between a load and its use.
//   phase 1  logits: one v_mfma_f32_32x32x16 block per tile, query heads as (zero-padded) rows;
//   phase 2  chunk softmax statistics (max, sum of exp2), one wavefront per query head;
//   phase 3  sum of p * V rows from LDS: on the VALU, 8 output dims per lane, 16 partial sums folded through
//            LDS; for 8 heads per workgroup on the matrix pipe with V read transposed from LDS (there an infinity in V
//            gives NaN: the second half of its probability is zero or negative);
// Each chunk writes (max, sum, unnormalised output) to the workspace and a second kernel merges the chunks of a sequence; where a
// chunk holds every sequence whole, it writes the output itself.  Grid sizes depend only on the view's max_seq_len, never on the
// lengths on the device, so the launches can be replayed from a graph while the lengths grow.
#include <type_traits>
#include "fc_common.h"
#include <atomic>
#include <stdlib.h>

#define DA_THREADS 256
#define DA_CHUNK 256               // smallest chunk (tokens per workgroup); it sizes the workspace
#define DA_CHUNK_MAX 1024          // largest: the host picks a multiple of 32 in between from the launch's shape
#define DA_LOG2E 1.4426950408889634f

template <int DTYPE>
__device__ __forceinline__ void da_unpack8(const uint4& x, float (&f)[8]) {
  const unsigned w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (DTYPE == FC_BF16) {
      f[2 * i] = __uint_as_float(w[i] << 16);
      f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    } else {
      f[2 * i] = fc_half_to_float((unsigned short)(w[i] & 0xffff));
      f[2 * i + 1] = fc_half_to_float((unsigned short)(w[i] >> 16));
    }
  }
}

template <int DTYPE>
__device__ __forceinline__ float da_unpack(unsigned short x) {
  return DTYPE == FC_BF16 ? fc_bf16_to_float(x) : fc_half_to_float(x);
}

template <int DTYPE>
__device__ __forceinline__ unsigned short da_pack(float f) {
  return DTYPE == FC_BF16 ? fc_float_to_bf16(f) : fc_float_to_half(f);
}


#define DA_PV_MFMA_MIN 8               // heads per workgroup from which p * V runs on the matrix pipe (measured: no gain below)
// What probabilities are multiplied with before they become 16-bit operands, and outputs divided by: fp16's exponent ends at
// 2^-14 (subnormal step 2^-24), so of a probability p <= 1 as hi + lo the second half would lose bits from 2^-3 down, and
// all of p below 2^-25, which still counts in the sum.  A power of two: exact, and 1 stays below fp16's largest value.
#define DA_P_SCALE(DT) ((DT) == FC_F16 ? 16384.f : 1.f)
#define DA_TILE 32                     // keys per tile: one MFMA block, 8 KB of K or V rows
// The chunk's block-table entries are prefetched one per lane of a wavefront: the largest chunk in the smallest
// page the fast path takes (32 tokens, block_shift >= 5), starting anywhere in a page, must span at most 64 entries.
static_assert(DA_CHUNK_MAX / DA_TILE + 1 <= 64, "a chunk's block-table entries must fit one per lane");
static_assert(DA_CHUNK % DA_TILE == 0 && DA_CHUNK_MAX % 64 == 0, "chunk bounds: whole tiles, whole statistics registers");
#define DA_TILEB (DA_TILE * 256)
#define DA_RING (4 * 2 * DA_TILEB)     // four wavefronts, two stages each

template <int GT>
struct DaCfg {
  // ring | logits, then probabilities [GT][chunk]: fp32, or with eight heads (p * V on the matrix pipe) each
  // probability as two 16-bit halves hi + lo in the cache dtype
  static constexpr bool PV_MFMA = GT >= DA_PV_MFMA_MIN;
  static constexpr int lds(int chunk) { return DA_RING + GT * chunk * 4 + GT * 4; }
};

struct DaAppend {                 // the step's new rows, one per sequence (k_new null: nothing to append)
  const char *k_new, *v_new;
  long long k_stride, v_stride;   // bytes between sequences; heads are adjacent
  const int* slots;               // flat cache slot per sequence, negative = skip
};


// A new row inside a workgroup's range [t0, end) is written by this workgroup, which then has to see it land before it reads
// it back (true is returned), whichever sequence of the batch it belongs to (a table may be listed twice with lengths one
// apart, or a page be shared): nobody depends on another workgroup's write.  The sequence's own row is also written by its last
// workgroup, since it usually lies right behind the range.  Workgroups that write one row write the same bytes.
// slot: of sequence `lane` (negative: none), TWO: slot2 of sequence 64 + `lane`, asked for with it, ktbl: table entry tbl0 + `lane`
// of sequence b; both planes use one table.
template <bool TWO>
__device__ __forceinline__ bool da_append_rows(const KvView& kc, const KvView& vc, const DaAppend& ap, const char* kbase,
                                               const char* vbase, int slot, int slot2, int ktbl, int tbl0, int b, int h, int nb, int t0, int end,
                                               int len, int tid) {
  const int lane = tid & 63, l15 = tid & 15;
  const int e0 = t0 >> kc.block_shift, e1 = (end - 1) >> kc.block_shift;      // pages of the range (none: e1 < e0)
  bool inside = false;
  for (int j0 = 0; j0 < nb; j0 += FC_WAVE) {
    if (TWO && j0 == FC_WAVE) slot = slot2;
    else if (j0 > 0) slot = j0 + lane < nb ? ap.slots[j0 + lane] : -1;
    const int page = slot >> kc.block_shift, at = slot & (kc.block_size - 1);
    bool hit = false;
    for (int e = e0; e <= e1; ++e) {
      const int pos = (e << kc.block_shift) + at;
      hit |= slot >= 0 && page == __builtin_amdgcn_readlane(ktbl, e - tbl0) && pos >= t0 && pos < end;
    }
    unsigned long long todo = __ballot(hit);
    inside |= todo != 0ull;
    if (end == len) todo |= __ballot(slot >= 0 && j0 + lane == b);
    while (todo) {                                                            // wave-uniform
      const int j = __builtin_ctzll(todo);
      todo &= todo - 1;
      const int row = __builtin_amdgcn_readlane(slot, j);
      const long long rpage = row >> kc.block_shift, rat = row & (kc.block_size - 1);
      if (tid < 32) {
        const bool is_v = tid >= 16;
        const long long koff = rpage * kc.stride_block + rat * kc.stride_token, voff = rpage * vc.stride_block + rat * vc.stride_token;
        char* dst = is_v ? const_cast<char*>(vbase) + voff * 2 : const_cast<char*>(kbase) + koff * 2;
        const char* src = is_v ? ap.v_new + (j0 + j) * ap.v_stride : ap.k_new + (j0 + j) * ap.k_stride;
        *reinterpret_cast<uint4*>(dst + l15 * 16) = *reinterpret_cast<const uint4*>(src + (long long)h * FC_HEAD_DIM * 2 + l15 * 16);
      }
    }
  }
  return inside;
}

// Table entry `e` of the k-th sequence after b, round the batch (k from 0; no such sequence: -1).  A page that another sequence's
// table names at the same place belongs to a prefix that they share, and their workgroups read the same bytes.
__device__ __forceinline__ int da_peer_page(const KvView& v, int b, int nb, int k, int e) {
  const int p = b + 1 + k;
  return k < nb - 1 ? v.block_tables[(long long)(p < nb ? p : p - nb) * v.table_stride + min(e, v.table_stride - 1)] : -1;
}

// GT = query heads served per workgroup (a tile of the group, at most 8).
// FAST = a 32-token tile never straddles two pages (dense view, or pages of 32*2^n tokens), so a tile
// load is a wave-uniform base plus a per-lane offset.
//
// Wavefront w owns the key tiles w and w+4 of the chunk (32 tokens each) and streams them through
// its private two-stage ring in LDS with global_load_lds: K tile a, K tile b, then V tile a and
// V tile b into the same stages as soon as the logits of the K tile in them are done, so 16 KB per
// wavefront are in flight for most of the kernel and no load waits behind a workgroup barrier.
// Logits are one v_mfma_f32_32x32x16 block per tile with the query heads as rows (padded with zero
// rows to 32): whatever the group size, K is read from LDS once.
// WHOLE: the chunk holds every sequence: the workgroup writes the output (as the merge of one chunk would) and, asked to
// (one kv head a workgroup, one table for both planes), appends the step's rows.  APPEND: several chunks do as well, FAST.
template <int DTYPE, int GT, bool FAST, bool WHOLE, bool APPEND>
__global__ __launch_bounds__(DA_THREADS, 2) void decode_attn_kernel(KvView kc, KvView vc, int layer,
                                                                    const char* __restrict__ q, int Hq,
                                                                    const int* __restrict__ lens, float c,
                                                                    float* __restrict__ part_o,
                                                                    float* __restrict__ part_ml, int max_splits,
                                                                    int chunk, char* __restrict__ out, DaAppend ap) {
  extern __shared__ __align__(16) char smem[];
  float* sc = reinterpret_cast<float*>(smem + DA_RING);          // [GT][chunk]
  unsigned* p2 = reinterpret_cast<unsigned*>(smem + DA_RING);    // the same seen as (hi, lo) pairs
  float* sums = reinterpret_cast<float*>(smem + DA_RING + GT * chunk * 4);   // WHOLE: [GT]
  constexpr bool PV_MFMA = DaCfg<GT>::PV_MFMA;
  float(*red)[GT][FC_HEAD_DIM] = reinterpret_cast<float(*)[GT][FC_HEAD_DIM]>(smem);  // [16] partial outputs, reuses the ring
  static_assert(16 * GT * FC_HEAD_DIM * 4 <= DA_RING, "partial outputs must fit in the ring");

  // Workgroups go to the eight XCDs round-robin in launch order (blockIdx.x fastest).  With the chunk
  // index taken straight from blockIdx.x and a multiple of eight chunks per sequence, each XCD would
  // serve one chunk position of every sequence, and the late positions are mostly empty; rotating the
  // chunk index by the head and sequence spreads the live chunks over all XCDs.
  const int b = blockIdx.z;
  const int split = (int)((blockIdx.x + blockIdx.y + blockIdx.z) % gridDim.x);
  const int Hkv = kc.num_kv_heads;
  const int G = Hq / Hkv;
  const int gtiles = (G + GT - 1) / GT;
  const int h = blockIdx.y / gtiles, g0 = (blockIdx.y - h * gtiles) * GT;
  const int tid = threadIdx.x, lane = tid & 63;
  const int t0 = split * chunk;
  // The chunk's block-table entries, one per lane (a chunk of at most 1024 tokens in pages of at least 32 spans at
  // most 33), fetched before anything waits for the sequence length: a tile's address then costs a lane read instead
  // of a table load that the tile's own loads would have to wait for.
  int ktbl = 0, vtbl = 0;
  int peer = -1, peer2 = -1;     // the range's first page in the tables of the 128 sequences after this one
  if constexpr (FAST) {
    if (kc.block_tables) {
      const int e = min((t0 >> kc.block_shift) + lane, kc.table_stride - 1);
      ktbl = kc.block_tables[(long long)b * kc.table_stride + e];
      if (gtiles == 1) {
        peer = da_peer_page(kc, b, gridDim.z, lane, t0 >> kc.block_shift);
        if ((int)gridDim.z > FC_WAVE + 1) peer2 = da_peer_page(kc, b, gridDim.z, FC_WAVE + lane, t0 >> kc.block_shift);
      }
    }
    if (vc.block_tables) {
      const int e = min((t0 >> vc.block_shift) + lane, vc.table_stride - 1);
      vtbl = vc.block_tables[(long long)b * vc.table_stride + e];
    }
  }
  int len = __builtin_amdgcn_readfirstlane(lens[b]);
  len = min(len, kc.max_seq_len);
  const int nb = (int)gridDim.z;
  int slot = -1;
  if constexpr (WHOLE) {
    if (ap.k_new && lane < nb) slot = ap.slots[lane];
  }
  int slot2 = -1;
  if constexpr (APPEND) {
    slot = lane < nb ? ap.slots[lane] : -1;
    if (FC_WAVE + lane < nb) slot2 = ap.slots[FC_WAVE + lane];
  }
  if (!WHOLE && t0 >= len && (!APPEND || split != 0)) return;
  const int ntok = min(chunk, len - t0);

  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int sub = lane & 15, rg = lane >> 4;   // V rows: 16 lanes per row, 4 rows per pass

  // query heads as MFMA A-operand rows; rows past the group tile are zero
  uint4 qf[8];
  {
    const bool ok = lrow < GT && g0 + lrow < G;
    const char* qp = q + (((long long)b * Hq + (h * G + g0 + (ok ? lrow : 0))) * FC_HEAD_DIM + lhalf * 8) * 2;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = ok ? *reinterpret_cast<const uint4*>(qp + ks * 32) : make_uint4(0, 0, 0, 0);
  }

  const char* kbase = kc.base + ((long long)layer * kc.stride_layer + (long long)h * kc.stride_head) * 2;
  const char* vbase = vc.base + ((long long)layer * vc.stride_layer + (long long)h * vc.stride_head) * 2;
  if constexpr (WHOLE) {
    len = max(len, 0);
    if (ap.k_new && da_append_rows<false>(kc, vc, ap, kbase, vbase, slot, -1, ktbl, 0, b, h, nb, 0, len, len, tid)) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    if (len == 0) {
      unsigned short* orow = reinterpret_cast<unsigned short*>(out) + ((long long)b * Hq + h * G + g0) * FC_HEAD_DIM;
      for (int i = tid; i < min(GT, G - g0) * FC_HEAD_DIM; i += DA_THREADS) orow[i] = 0;
      return;
    }
  }
  if constexpr (APPEND) {
    len = max(len, 0);
    if (da_append_rows<true>(kc, vc, ap, kbase, vbase, slot, slot2, ktbl, t0 >> kc.block_shift, b, h, nb, t0, min(len, t0 + chunk), len, tid)) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    if (len == 0) return;                  // the merge writes the zeros
  }
  const unsigned ring_lds = __builtin_amdgcn_readfirstlane(fc_lds_addr(smem)) + wave * (2 * DA_TILEB);
  char* ring = smem + wave * (2 * DA_TILEB);
  // Where this workgroup alone reads its columns' bytes, the loads leave no line in the L2.  Workgroups that share a group of
  // heads find the bytes there (4 layers of 16 x 4096..8192, 128/4 heads, 591 -> 715 with such loads), and so do those of
  // sequences that share a prefix: a range whose first page another table names loads plainly.  us a pass, 16 captured bf16
  // layers on the same caches step after step, plain loads / such loads whatever is shared / as here: 90 x 128..2048 tokens, 32/32 heads, 4611 / 4218 / 4171, 56 x
  // 156..1565, 32/8, 965 / 923 / 877, 90 x 200..1400, 28/4, 912 / 853 / 782; 48 x 1300..1500 in groups of eight with the first
  // 1280 in common, 32/32, 1647 / 2429 / 1613, 16 x 4096 with 3840, 32/8, 829 / 943 / 824, 90 x 1500 with 512, 32/32, 4643 / 5012 /
  // 3755; where one head a group reads little else, 16 x 2048 with 1792, 1088 / 1269 / 1200.  (Asked for behind the first two
  // loads instead: 0.94 to 1.1 times this one's time with a prefix, 1.0 to 1.15 without.)
  const int page0 = __builtin_amdgcn_readfirstlane(ktbl);
  const bool alone = gtiles == 1 && (!FAST || !kc.block_tables || !__any(page0 >= 0 && (peer == page0 || peer2 == page0)));

  // Tile `tile` of the chunk into this wavefront's stage: eight wave-loads of four rows.  Lane i
  // writes LDS chunk i of the 64 chunks of those rows and fetches the global chunk (i & 15) ^ (row & 15)
  // of row i / 16 (XOR swizzle, so that the operand reads of 32 rows at the same chunk fall on
  // distinct banks).  Rows past the sequence end re-read its last row; their logits are masked.
  auto issue = [&](const KvView& v, const char* base, int tile, int stage, int tbl_reg) {
    const int s0 = t0 + tile * DA_TILE;
    const unsigned dst = ring_lds + stage * DA_TILEB;
    const int rmax = len - 1 - s0;
    if constexpr (FAST) {
      long long tb;
      if (v.block_tables) {
        const int blk = max(__builtin_amdgcn_readlane(tbl_reg, (s0 >> v.block_shift) - (t0 >> v.block_shift)), 0);
        tb = (long long)blk * v.stride_block + (long long)(s0 & (v.block_size - 1)) * v.stride_token;
      } else {
        tb = (long long)b * v.stride_batch + (long long)s0 * v.stride_token;
      }
      const char* g = base + tb * 2;
      const unsigned tok_bytes = (unsigned)v.stride_token * 2;
      const auto lane_off = [&](int r) { return (unsigned)min(r, rmax) * tok_bytes + ((sub ^ (r & 15)) << 4); };
      if (alone) {
#pragma unroll
        for (int u = 0; u < 8; ++u) fc_load_lds_once(g, lane_off(4 * u + rg), dst + u * 1024);
      } else {
#pragma unroll
        for (int u = 0; u < 8; ++u) fc_load_lds(g, lane_off(4 * u + rg), dst + u * 1024);
      }
    } else {
      long long off[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int r = 4 * u + rg;
        off[u] = fc_token_offset(v, b, s0 + min(r, rmax));
        if (off[u] < 0) off[u] = 0;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int r = 4 * u + rg;
        fc_load_lds(base + off[u] * 2 + ((sub ^ (r & 15)) << 4), dst + u * 1024);
      }
    }
  };

  // This wavefront's tiles are wave, wave + 4, wave + 8, ...: nj of them hold tokens.  Their K tiles and then
  // their V tiles form one stream of 2 * nj items; item i goes to stage i & 1 and is issued as soon as item
  // i - 2 has been consumed, so two items (16 KB) are in flight for most of the kernel.
  const int live_tiles = (ntok + DA_TILE - 1) / DA_TILE;
  const int nj = wave < live_tiles ? (live_tiles - wave + 3) / 4 : 0;   // wave-uniform
  auto issue_item = [&](int i) {
    if (i < nj) issue(kc, kbase, wave + 4 * i, i & 1, ktbl);
    else if (i < 2 * nj) issue(vc, vbase, wave + 4 * (i - nj), i & 1, vtbl);
  };
  // item i has landed when at most the loads of item i + 1 (eight per lane) are outstanding
  auto wait_item = [&](int i) {
    if (i + 1 < 2 * nj) fc_wait_vm<8>(); else fc_wait_vm<0>();
  };
  issue_item(0);
  issue_item(1);

  // ---- phase 1: logits of this wavefront's tiles --------------------------------------------------
  // C[head][key]: the lane owns key lrow of the tile and the heads (i/4)*8 + lhalf*4 + i%4, of which
  // only heads < 8 exist, that is registers 0..3.  Tokens past the sequence end get -inf; tiles past
  // it are never read (the statistics below stop at ntok).
  const unsigned xs = (unsigned)((lhalf ^ (lrow & 15)) << 4) + lrow * 256;
  auto logits = [&](int tile, int stage) {
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const uint4 kf = *reinterpret_cast<const uint4*>(ring + stage * DA_TILEB + (xs ^ (unsigned)(ks * 32)));
      acc = fc_mfma<DTYPE>(qf[ks], kf, acc);
    }
    const int t = tile * DA_TILE + lrow;
    const bool live = t < ntok;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int g = lhalf * 4 + i;
      if (g < GT) sc[g * chunk + t] = live ? acc[i] * c : -INFINITY;
    }
  };
  for (int i = 0; i < nj; ++i) {
    wait_item(i);
    logits(wave + 4 * i, i & 1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the stage's reads are done before the next item lands in it
    issue_item(i + 2);
  }
  fc_lds_barrier();

  // ---- phase 2: chunk statistics, one wavefront per query head -------------------------------------
  for (int g = wave; g < GT; g += 4) {
    float x[DA_CHUNK_MAX / 64];
#pragma unroll
    for (int j = 0; j < DA_CHUNK_MAX / 64; ++j) x[j] = lane + 64 * j < ntok ? sc[g * chunk + lane + 64 * j] : -INFINITY;
    float mx = x[0];
#pragma unroll
    for (int j = 1; j < DA_CHUNK_MAX / 64; ++j) mx = fmaxf(mx, x[j]);
    const float m = fc_wave_max_uniform(mx);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < DA_CHUNK_MAX / 64; ++j) {
      const float p = __builtin_amdgcn_exp2f(x[j] - m);   // exp2(-inf) = 0 for the padded slots
      if (lane + 64 * j < live_tiles * DA_TILE) {         // every slot of a live tile is read by phase 3
        if constexpr (PV_MFMA) {
          const float ps = p * DA_P_SCALE(DTYPE);
          const unsigned short hi = da_pack<DTYPE>(ps);
          const float hf = DTYPE == FC_BF16 ? fc_bf16_to_float(hi) : fc_half_to_float(hi);
          p2[g * chunk + lane + 64 * j] = (unsigned)hi | ((unsigned)da_pack<DTYPE>(ps - hf) << 16);
        } else {
          sc[g * chunk + lane + 64 * j] = p;
        }
      }
      sum += p;
    }
    sum = fc_wave_sum_uniform(sum);
    if (WHOLE) {
      if (lane == 0) sums[g] = sum;
    } else if (lane == 0 && g0 + g < G) {
      float* ml = part_ml + (((long long)b * Hq + (h * G + g0 + g)) * max_splits + split) * 2;
      ml[0] = m;
      ml[1] = sum;
    }
  }
  fc_lds_barrier();

  const auto put = [&](int g, int d, float o) {
    const long long row = (long long)b * Hq + (h * G + g0 + g);
    if constexpr (WHOLE) reinterpret_cast<unsigned short*>(out)[row * FC_HEAD_DIM + d] = da_pack<DTYPE>(o / sums[g]);
    else part_o[(row * max_splits + split) * FC_HEAD_DIM + d] = o;
  };

  // ---- phase 3: sum of p * V over this wavefront's tiles -------------------------------------------
  if constexpr (PV_MFMA) {
    // O[head][d] = P[head][key] * V[key][d] on the matrix pipe.  A = P rows from LDS (8 consecutive keys per
    // lane), as two operands hi and lo so that the probabilities keep ~16-22 mantissa bits; the B operand
    // wants 8 consecutive KEYS of one output dimension per lane, i.e. V transposed, which is read as
    // 2-byte pieces from the swizzled rows (lanes of a half-wave read neighbouring dimensions of one row,
    // the two half-waves rows 8 apart whose chunks are swizzled onto other banks).
    f32x16 oacc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[nb][i] = 0.f;
    auto pv = [&](int tile, int stage) {
      const char* vt = ring + stage * DA_TILEB + (lrow & 7) * 2;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int k0 = s * 16 + lhalf * 8;   // first of this lane's 8 keys of the k-step
        uint4 a = make_uint4(0, 0, 0, 0), a2 = make_uint4(0, 0, 0, 0);
        if (lrow < GT) {
          const uint4 d0 = *reinterpret_cast<const uint4*>(&p2[lrow * chunk + tile * DA_TILE + k0]);
          const uint4 d1 = *reinterpret_cast<const uint4*>(&p2[lrow * chunk + tile * DA_TILE + k0 + 4]);
          // v_perm_b32 bytes: 0-3 second operand, 4-7 first operand
          a = make_uint4(__builtin_amdgcn_perm(d0.y, d0.x, 0x05040100u), __builtin_amdgcn_perm(d0.w, d0.z, 0x05040100u),
                         __builtin_amdgcn_perm(d1.y, d1.x, 0x05040100u), __builtin_amdgcn_perm(d1.w, d1.z, 0x05040100u));
          a2 = make_uint4(__builtin_amdgcn_perm(d0.y, d0.x, 0x07060302u), __builtin_amdgcn_perm(d0.w, d0.z, 0x07060302u),
                          __builtin_amdgcn_perm(d1.y, d1.x, 0x07060302u), __builtin_amdgcn_perm(d1.w, d1.z, 0x07060302u));
        }
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
          const int chunk = nb * 4 + (lrow >> 3);
          unsigned w[4];
#pragma unroll
          for (int e2 = 0; e2 < 4; ++e2) {
            const int ka = k0 + 2 * e2, kb = ka + 1;
            const unsigned lo = *reinterpret_cast<const unsigned short*>(vt + ka * 256 + ((chunk ^ (ka & 15)) << 4));
            const unsigned hi = *reinterpret_cast<const unsigned short*>(vt + kb * 256 + ((chunk ^ (kb & 15)) << 4));
            w[e2] = lo | (hi << 16);
          }
          const uint4 bfrag = make_uint4(w[0], w[1], w[2], w[3]);
          oacc[nb] = fc_mfma<DTYPE>(a, bfrag, oacc[nb]);
          oacc[nb] = fc_mfma<DTYPE>(a2, bfrag, oacc[nb]);
        }
      }
    };
    for (int i = nj; i < 2 * nj; ++i) {
      wait_item(i);
      pv(wave + 4 * (i - nj), i & 1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue_item(i + 2);
    }
    fc_lds_barrier();   // every wavefront is done with its ring before the ring becomes `red`
    // C layout: the lane holds output dimension nb*32 + lrow of the heads lhalf*4 + i (registers 0..3)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int g = lhalf * 4 + i;
      if (g < GT) {
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) red[wave][g][nb * 32 + lrow] = oacc[nb][i];
      }
    }
    fc_lds_barrier();
    for (int i = tid; i < GT * FC_HEAD_DIM; i += DA_THREADS) {
      const int g = i / FC_HEAD_DIM, d = i - g * FC_HEAD_DIM;
      if (g0 + g < G) {
        const float o = ((red[0][g][d] + red[1][g][d]) + (red[2][g][d] + red[3][g][d])) * (1.f / DA_P_SCALE(DTYPE));
        put(g, d, o);
      }
    }
  } else {
    float acc[GT][8];
#pragma unroll
    for (int g = 0; g < GT; ++g)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[g][e] = 0.f;
    auto pv = [&](int tile, int stage, float (&to)[GT][8]) {
#pragma unroll
      for (int p = 0; p < 8; ++p) {
        const int r = 4 * p + rg;
        const uint4 vx = *reinterpret_cast<const uint4*>(ring + stage * DA_TILEB + r * 256 + ((sub ^ (r & 15)) << 4));
        float vf[8];
        da_unpack8<DTYPE>(vx, vf);
#pragma unroll
        for (int g = 0; g < GT; ++g) {
          const float pr = sc[g * chunk + tile * DA_TILE + r];
#pragma unroll
          for (int e = 0; e < 8; ++e) to[g][e] = fmaf(pr, vf[e], to[g][e]);
        }
      }
    };
    for (int i = nj; i < 2 * nj; ++i) {
      wait_item(i);
      // Of whole columns a tile's products are summed by themselves: one chain of 64 of them was further from 64 bits than chunks of
      // 256 tokens merged (1024 tokens of 1 head a group, logits of deviation 1 / 3: 1.09 to 1.10 / 1.03 to 1.04 of their error,
      // now 0.98 / 1.00).
      if constexpr (WHOLE) {
        float own[GT][8] = {};
        pv(wave + 4 * (i - nj), i & 1, own);
#pragma unroll
        for (int g = 0; g < GT; ++g)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[g][e] += own[g][e];
      } else {
        pv(wave + 4 * (i - nj), i & 1, acc);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue_item(i + 2);
    }
    fc_lds_barrier();   // every wavefront is done with its ring before the ring becomes `red`
    // 16 partial outputs (4 wavefronts x 4 row slots) through LDS, summed in a fixed order
    {
      const int slot = wave * 4 + rg;
#pragma unroll
      for (int g = 0; g < GT; ++g) {
        float4* dst = reinterpret_cast<float4*>(&red[slot][g][sub * 8]);
        dst[0] = make_float4(acc[g][0], acc[g][1], acc[g][2], acc[g][3]);
        dst[1] = make_float4(acc[g][4], acc[g][5], acc[g][6], acc[g][7]);
      }
    }
    fc_lds_barrier();
    for (int i = tid; i < GT * FC_HEAD_DIM; i += DA_THREADS) {
      const int g = i / FC_HEAD_DIM, d = i - g * FC_HEAD_DIM;
      if (g0 + g < G) {
        float o = 0.f;
#pragma unroll
        for (int sl = 0; sl < 16; ++sl) o += red[sl][g][d];
        put(g, d, o);
      }
    }
  }
}

template <int DTYPE>
__global__ __launch_bounds__(FC_HEAD_DIM) void decode_merge_kernel(const float* __restrict__ part_o,
                                                                   const float* __restrict__ part_ml,
                                                                   const int* __restrict__ lens, int max_seq_len,
                                                                   int Hq, int max_splits, int chunk, int alone,
                                                                   char* __restrict__ out) {
  const int hq = blockIdx.x, b = blockIdx.y, d = threadIdx.x;
  int len = min(lens[b], max_seq_len);
  unsigned short* o = reinterpret_cast<unsigned short*>(out) + ((long long)b * Hq + hq) * FC_HEAD_DIM + d;
  if (len <= 0) {
    *o = 0;
    return;
  }
  const int ns = len <= chunk + alone ? 1 : (len + chunk - 1) / chunk;
  const float* ml = part_ml + ((long long)b * Hq + hq) * max_splits * 2;
  const float* po = part_o + ((long long)b * Hq + hq) * max_splits * FC_HEAD_DIM + d;
  // eight splits per step so that their loads are in flight together
  float M = -INFINITY;
  for (int s0 = 0; s0 < ns; s0 += 8) {
    float m[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) m[j] = s0 + j < ns ? ml[2 * (s0 + j)] : -INFINITY;
#pragma unroll
    for (int j = 0; j < 8; ++j) M = fmaxf(M, m[j]);
  }
  float L = 0.f, acc = 0.f;
  for (int s0 = 0; s0 < ns; s0 += 8) {
    float m[8], l[8], x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool ok = s0 + j < ns;
      m[j] = ok ? ml[2 * (s0 + j)] : -INFINITY;
      l[j] = ok ? ml[2 * (s0 + j) + 1] : 0.f;
      x[j] = ok ? po[(long long)(s0 + j) * FC_HEAD_DIM] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float w = __builtin_amdgcn_exp2f(m[j] - M);
      L = fmaf(w, l[j], L);
      acc = fmaf(w, x[j], acc);
    }
  }
  *o = da_pack<DTYPE>(acc / L);
}

// ---- few columns: one short chain per workgroup ----------------------------------------------------------------------
// A step of a few sequences is latency, not bandwidth: three users of 300 to 900 tokens move 3.4 MB a layer, and the
// split kernel spent 11.3 us on it, the merge 3.3 and the append 1.9, each behind the one before (bf16, 28 query heads on
// 4).  Here a workgroup of eight wavefronts owns a range of a (sequence, kv head) column, the whole context where that is
// short: the wavefronts take the 32-token tiles in turn, K and V of a wavefront's first two tiles are requested
// at once instead of K before V, every wavefront carries its own running softmax and no phase waits for the workgroup,
// and the eight are merged through LDS.  The step's new K and V rows may be appended by the same workgroups (k_new).
// The ranges of a column are merged by a launch of their own or (TURN) by the workgroup of the column that arrives last.
//   S^T[key][head] = K Q^T  on v_mfma_f32_16x16x32: the A operand (16 keys x 64 contiguous bytes per instruction)
//                           comes straight from memory; the lane then owns ONE head and 8 keys of the tile, so maxima
//                           and sums run over its registers and two lane exchanges;
//   O^T[dim][head] = V^T P^T: the probabilities are already the B operand (keys in the order the accumulator gives
//                           them); V goes straight to the wavefront's 16 KB of LDS, two tiles, and is read transposed by
//                           the hardware (ds_read_b64_tr_b16).
// Probabilities enter as a sum of 16-bit operands in the cache dtype: two for groups of 5 and more heads (as in the split
// kernel), three for up to 4 heads, where the split kernel multiplies in fp32: three bf16 operands hold all 24 bits, three
// fp16 operands all bits of a probability down to 2^-15, and what they drop is below 2^-39 of the tile's largest
// (DA_P_SCALE).  A tile's products are summed by themselves, least operands first, and rounded into the output once.
// Error of the unrounded output against 64 bits, geometric mean over 7 settings (1 / 2 / 4 heads a group, 2 to 64 contexts of
// 500 to 3500 keys, 12 seeds), this kernel / the split kernel: logits of deviation 1, fp16 2.03 / 2.10e-7, bf16
// 1.85 / 1.97e-7; of deviation 3, 1.003 and 1.002 of it; of deviation 6, 1.000 and 0.999 (two fp16 operands, and operands
// added to the output one by one: 1.010 and 1.014, 1.012 and 1.016, 1.002 and 1.004 of the split kernel's).
// An infinite value in V meets operands that are zero or negative and gives NaN, in both kernels, for groups of 5 and more
// heads.  For up to 4, what is no number after the last tile is formed again with the probabilities in fp32.
#define DC_WAVES 8
#define DC_THREADS (DC_WAVES * 64)
#define DC_HEADS 16
#define DC_PSTRIDE 132                                             // floats per partial output row (padded against bank conflicts)
// A sequence that reaches at most this far into its column's second range is its first workgroup's alone: a second tile for half
// of the wavefronts is shorter than a merge.  us a layer, 16 captured layers of columns of 270 to 375 tokens, merged -> alone:
// 4 columns 9.5 -> 8.1 to 8.7, 48 10.9 -> 8.9 to 9.6; of 400 9.5 -> 9.4, of 500 10.0 -> 10.6.
#define DC_ALONE 128
#define DC_ONCE_BYTES (16ll << 20)                                 // K and V; 16 layers of it are what the memory-side cache holds
#define DC_STAGES 2                                                // V tiles of a wavefront in LDS or on their way
#define DC_MERGE 8                                                // partial rows in flight per thread of the merge
#define DC_PART (DC_WAVES * DC_STAGES * DA_TILEB)                   // V stages, then the partial outputs
#define DC_LDS (DC_PART + DC_WAVES * DC_HEADS * 8)
static_assert(DC_PART >= DC_WAVES * DC_HEADS * DC_PSTRIDE * 4, "the partial outputs share the V stages' memory");

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned da_u32x4 __attribute__((ext_vector_type(4)));   // native vector: arrays of it stay in registers

// C[16][16] += A[16][32] * B[32][16]: lane (row or column l % 16, quarter l / 16) holds k = quarter * 8 .. + 7; result:
// column l % 16, rows quarter * 4 + i
template <int DTYPE>
__device__ __forceinline__ f32x4 da_mfma16(const uint4& a, const uint4& b, f32x4 c) {
  if constexpr (DTYPE == FC_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// two floats -> packed storage dtype, round to nearest even, in one conversion instruction
template <int DTYPE>
__device__ __forceinline__ unsigned da_pack2(float x, float y) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {x, y};
  if constexpr (DTYPE == FC_BF16) return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
  else return __builtin_bit_cast(unsigned, __builtin_convertvector(v, f16x2));
}

// 8 floats -> 8 values of the storage dtype; the floats keep what the rounding left
template <int DTYPE>
__device__ __forceinline__ uint4 da_split8(float (&p)[8]) {
  unsigned w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    w[e] = da_pack2<DTYPE>(p[2 * e], p[2 * e + 1]);
    p[2 * e] -= DTYPE == FC_BF16 ? __uint_as_float(w[e] << 16) : fc_half_to_float((unsigned short)(w[e] & 0xffff));
    p[2 * e + 1] -= DTYPE == FC_BF16 ? __uint_as_float(w[e] & 0xffff0000u) : fc_half_to_float((unsigned short)(w[e] >> 16));
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// 8 bytes a lane from an absolute LDS address, transposed among 16 lanes: lane i of them gets the i-th 2-byte value of what
// lanes 0 .. 3, 4 .. 7, 8 .. 11 and 12 .. 15 read (ds_read_b64_tr_b16)
__device__ __forceinline__ uint2 da_lds_transposed(unsigned addr) {
  typedef short da_s16x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                       reinterpret_cast<__attribute__((address_space(3))) da_s16x4*>((size_t)addr)));
}

// Arrivals per column of a launch whose last workgroup merges, a row of counters per turn (fc_decode_layer_turn) or the
// caller's (fc_decode_layer_arrivals).  Zero between launches: whoever merges puts the zero back.
#define DC_COLUMNS FC_DECODE_ARRIVALS
static __device__ unsigned dc_arrived[FC_DECODE_TURNS][DC_COLUMNS];

// Partial results that another workgroup of the same launch reads go past the caches of this XCD.
template <bool TURN>
__device__ __forceinline__ void dc_put(float* p, float x) {
  if constexpr (TURN) __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = x;
}
__device__ __forceinline__ float2 dc_get2(const float* p) {      // 8-byte aligned
  return __builtin_bit_cast(float2, __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT));
}

template <int DTYPE, int TERMS, bool PAGED, bool TURN>
__global__ __launch_bounds__(DC_THREADS, 2) void decode_column_kernel(KvView kc, KvView vc, int layer,
                                                                      const char* __restrict__ q, int Hq,
                                                                      const int* __restrict__ lens, float c,
                                                                      char* __restrict__ out, DaAppend ap, int chunk,
                                                                      float* part_o, float* part_ml, int max_splits,
                                                                      int turn, unsigned* arrivals) {
  extern __shared__ __align__(16) char smem[];
  const int b = blockIdx.y;
  const int G = Hq / kc.num_kv_heads, gtiles = (G + DC_HEADS - 1) / DC_HEADS;
  const int h = blockIdx.x / gtiles, g0 = (blockIdx.x - h * gtiles) * DC_HEADS;
  const int ng = min(G - g0, DC_HEADS);
  const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, qd = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // PAGED: both views are, and a sequence's table fits one entry per lane; otherwise both are dense
  int ktbl = 0, vtbl = 0;
  if constexpr (PAGED) {
    ktbl = kc.block_tables[(long long)b * kc.table_stride + min(lane, kc.table_stride - 1)];
    vtbl = vc.block_tables[(long long)b * vc.table_stride + min(lane, vc.table_stride - 1)];
  }
  int len = __builtin_amdgcn_readfirstlane(lens[b]);
  len = max(min(len, kc.max_seq_len), 0);
  const int nb = (int)gridDim.y;
  int slot = PAGED && ap.k_new && lane < nb ? ap.slots[lane] : -1;   // the new rows' slots, 64 sequences at a time
  const int span = max_splits > 1 && len <= chunk + DC_ALONE ? chunk + DC_ALONE : chunk;
  const int t0 = (int)blockIdx.z * span;
  if (t0 >= len && blockIdx.z != 0) return;
  const int end = min(len, t0 + span);
  // the query heads as B operand; columns past the group are zero
  uint4 qf[4];
  {
    const bool ok = l15 < ng;
    const char* qp = q + (((long long)b * Hq + (h * G + g0 + (ok ? l15 : 0))) * FC_HEAD_DIM + qd * 8) * 2;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qf[ks] = ok ? *reinterpret_cast<const uint4*>(qp + ks * 64) : make_uint4(0, 0, 0, 0);
  }
  const char* kbase = kc.base + ((long long)layer * kc.stride_layer + (long long)h * kc.stride_head) * 2;
  const char* vbase = vc.base + ((long long)layer * vc.stride_layer + (long long)h * vc.stride_head) * 2;
  if (PAGED && ap.k_new) {
    if (da_append_rows<false>(kc, vc, ap, kbase, vbase, slot, -1, ktbl, 0, b, h, nb, t0, end, len, tid)) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
  }
  unsigned short* orow = reinterpret_cast<unsigned short*>(out) + ((long long)b * Hq + h * G + g0) * FC_HEAD_DIM;
  const bool whole = max_splits == 1 || (TURN && len <= span);
  if (len <= 0) {       // with several workgroups per column the merge writes the zeros
    if (whole)
      for (int i = tid; i < ng * FC_HEAD_DIM; i += DC_THREADS) orow[i] = 0;
    return;
  }

  const unsigned ktok = (unsigned)kc.stride_token * 2, vtok = (unsigned)vc.stride_token * 2;
  auto tile_base = [&](const KvView& v, const char* base, int s0, int tbl) {
    if constexpr (!PAGED) return base + ((long long)b * v.stride_batch + (long long)s0 * v.stride_token) * 2;
    const int blk = max(__builtin_amdgcn_readlane(tbl, s0 >> v.block_shift), 0);
    return base + ((long long)blk * v.stride_block + (long long)(s0 & (v.block_size - 1)) * v.stride_token) * 2;
  };
  // Rows past the end of the sequence re-read its last row, except K rows of a paged tile, which lies inside its page: they
  // are read as they are, their logits are masked.  The scheduling barriers keep the loads from moving up before the tile
  // their registers held has been used up.
  const unsigned klane = (unsigned)l15 * ktok + qd * 16;
  auto load_k = [&](da_u32x4 (&kf)[8], int tile) {
    const int s0 = t0 + tile * DA_TILE, rmax = end - 1 - s0;
    const char* kg = tile_base(kc, kbase, s0, ktbl);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const char* g = PAGED ? kg + kb * 16 * (unsigned long long)ktok : kg;
      const unsigned o = PAGED ? klane : (unsigned)min(kb * 16 + l15, rmax) * ktok + qd * 16;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) kf[kb * 4 + ks] = *reinterpret_cast<const da_u32x4*>(g + o + ks * 64);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // V rows go to LDS without registers between, 4 rows of 256 bytes an instruction; the 16-byte pieces of a row are XOR-ed
  // with the row number, so that the transposed reads of 16 rows at one place meet all banks.
  // Of groups of up to 4 heads whole tiles leave no line in the L2 (us a pass, 16 captured bf16 layers, plain -> so: 32/8 heads, 4 x
  // 4000 tokens 339 -> 322, the first 3840 in common 256 -> 250, 24 x 700..768, 512 in common, 267 -> 250, 1 x 8000 282 -> 275, 32/32,
  // 1 x 8000 486 -> 462, 8/8, 4 x 1000 198.5 -> 197.5), where the batch may hold DC_ONCE_BYTES a layer.  Less stays in the
  // memory-side cache from step to step: 32/8, 1 x 300 147 -> 157, 1 x 1000 175 -> 183, 32/32, 1 x 300 155 -> 159.  Larger groups
  // gain less and read a shared prefix from there: 28/4, 16 x 3900..4096 545 -> 513, but with 3840 in common 340 -> 367, 12 x
  // 1800..2000 with 1792 231 -> 238, so they load plainly; asking the tables first costs the launch its start (28 eager layers of 3
  // x 300..900 305 plain, 297 so, 313 asked).  K stays: an instruction takes 64 bytes of a row, the rest of the line would be
  // fetched again (16 x 3280, 28/4, 464 -> 480, 32 x 1000..4000 700 -> 778).
  const bool once = TERMS == 3 && (long long)gridDim.y * kc.max_seq_len * kc.num_kv_heads * (4 * FC_HEAD_DIM) >= DC_ONCE_BYTES;
  const unsigned v_lds = __builtin_amdgcn_readfirstlane(fc_lds_addr(smem) + wave * DC_STAGES * DA_TILEB);
  unsigned vlane[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) vlane[j] = (unsigned)qd * vtok + ((l15 ^ (4 * j + qd)) << 4);
  auto load_v = [&](int stage, int tile) {
    const int s0 = t0 + tile * DA_TILE, rmax = end - 1 - s0;
    const char* vg = tile_base(vc, vbase, s0, vtbl);
    if (once && rmax >= DA_TILE - 1) {
#pragma unroll
      for (int u = 0; u < 8; ++u) fc_load_lds_once(vg + u * 4 * (unsigned long long)vtok, vlane[u & 3], v_lds + stage * DA_TILEB + u * 1024);
    } else if (rmax >= DA_TILE - 1) {
#pragma unroll
      for (int u = 0; u < 8; ++u) fc_load_lds(vg + u * 4 * (unsigned long long)vtok, vlane[u & 3], v_lds + stage * DA_TILEB + u * 1024);
    } else {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        fc_load_lds(vg, (unsigned)min(4 * u + qd, rmax) * vtok + ((l15 ^ ((4 * u + qd) & 15)) << 4), v_lds + stage * DA_TILEB + u * 1024);
    }
  };

  float m = -INFINITY, l = 0.f;      // of head l15: the maximum is the tile group's, the sum this lane's keys'
  f32x4 o[8];
  // Transposed reads: 16 lanes take four rows, 32 bytes of each, 8 bytes a lane, and lane i gets column i of the four: here
  // dimension db * 16 + l15 of keys 4 qd .. 4 qd + 3 (and of the 16 keys further).
  unsigned v_get[8];
  {
    const int row = 4 * qd + (l15 >> 2);
    const unsigned at = (((l15 & 3) >> 1) ^ row) << 4;
#pragma unroll
    for (int db = 0; db < 8; ++db) v_get[db] = v_lds + row * 256 + (at ^ (db * 32)) + (l15 & 1) * 8;
  }
  const int tiles = (end - t0 + DA_TILE - 1) / DA_TILE, last = tiles - 1;
  auto dot = [&](const da_u32x4 (&kf)[8], f32x4 (&s)[2]) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      s[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) s[kb] = da_mfma16<DTYPE>(__builtin_bit_cast(uint4, kf[kb * 4 + ks]), qf[ks], s[kb]);
    }
  };
  // One tile: its logits, its probabilities, its V rows; then the tile after the next starts loading into the registers and
  // the stage that became free.  V is asked for before K: whoever waits for a tile's K has its V as well.
  // NEWER: whether the next tile has been asked for already, LOAD: whether there is one after the next; compile-time, since a
  // branch around loads has the compiler wait for all that might be under way.
  auto use_tile = [&](da_u32x4 (&kf)[8], auto stage, auto first, auto newer, auto load, int tile) {
    constexpr int ST = decltype(stage)::value;
    constexpr bool FIRST = decltype(first)::value, NEWER = decltype(newer)::value, LOAD = decltype(load)::value;
    const int live = end - t0 - tile * DA_TILE;
    f32x4 s[2];
    dot(kf, s);
    float p[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) p[e] = s[e >> 2][e & 3] * c;
    if (live < DA_TILE) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if ((e >> 2) * 16 + qd * 4 + (e & 3) >= live) p[e] = -INFINITY;
    }
    float mx = p[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) mx = fmaxf(mx, p[e]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mo = m;
    m = FIRST ? mx : fmaxf(m, mx);
    const float ref = m == -INFINITY ? 0.f : m;   // so far only logits of -inf: they weigh nothing, and -inf - -inf is NaN
    const float alpha = FIRST ? 0.f : __builtin_amdgcn_exp2f(mo - ref);
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = __builtin_amdgcn_exp2f(p[e] - ref);
      sum += p[e];
      p[e] *= DA_P_SCALE(DTYPE);
    }
    l = FIRST ? sum : fmaf(l, alpha, sum);
    uint4 pt[TERMS];
#pragma unroll
    for (int t = 0; t < TERMS; ++t) pt[t] = da_split8<DTYPE>(p);
    fc_wait_vm<NEWER ? 16 : 0>();      // this tile's V rows are in LDS
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      const uint2 lo = da_lds_transposed(v_get[db] + ST * DA_TILEB), hi = da_lds_transposed(v_get[db] + ST * DA_TILEB + 4096);
      const uint4 vt = make_uint4(lo.x, lo.y, hi.x, hi.y);
      f32x4 pv = f32x4{0.f, 0.f, 0.f, 0.f};        // the tile's own sum, least operands first: o is rounded once a tile
#pragma unroll
      for (int t = TERMS; t > 0; --t) pv = da_mfma16<DTYPE>(vt, pt[t - 1], pv);
      o[db] = FIRST ? pv : o[db] * alpha + pv;
      // not more transposed reads in flight than registers beside the tiles hold
      if ((db & 3) == 3) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (LOAD) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the reads of the stage before what overwrites it
      load_v(ST, tile + 2 * DC_WAVES);
      load_k(kf, tile + 2 * DC_WAVES);
    }
  };

  const int own = (tiles - wave + DC_WAVES - 1) / DC_WAVES;    // this wavefront's tiles (none: 0 or less)
#pragma unroll
  for (int db = 0; db < 8; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  {
    constexpr std::integral_constant<int, 0> s0{};
    constexpr std::integral_constant<int, 1> s1{};
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    da_u32x4 ka[8], kb[8];
    if (own == 1) {
      load_v(0, wave);
      load_k(ka, wave);
      use_tile(ka, s0, yes, no, no, wave);
    } else if (own > 1) {
      load_v(0, wave);
      load_k(ka, wave);
      load_v(1, wave + DC_WAVES);
      load_k(kb, wave + DC_WAVES);
      int t = wave, left = own;
      for (; left > 3; left -= 2, t += 2 * DC_WAVES) {
        use_tile(ka, s0, no, yes, yes, t);
        use_tile(kb, s1, no, yes, yes, t + DC_WAVES);
      }
      if (left == 3) {
        use_tile(ka, s0, no, yes, yes, t);
        use_tile(kb, s1, no, yes, no, t + DC_WAVES);
        use_tile(ka, s0, no, no, no, t + 2 * DC_WAVES);
      } else {
        use_tile(ka, s0, no, yes, no, t);
        use_tile(kb, s1, no, no, no, t + DC_WAVES);
      }
    }
  }

  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  // Results that are no number, formed again with the probabilities in fp32: an infinity in V gives an infinity then, unless
  // its key weighs nothing.  Never taken with finite keys and values.  Groups of up to 4 heads alone, as in the split kernel:
  // the question is 16 comparisons a lane, and 28 layers of 3 sequences of 900 tokens in groups of 7 take 313 us with it, 311
  // without.
  bool redo = false;
  if constexpr (TERMS == 3) {
#pragma unroll
    for (int db = 0; db < 8; ++db)
#pragma unroll
      for (int i = 0; i < 4; i += 2) redo |= __builtin_isunordered(o[db][i], o[db][i + 1]);
  }
  if (TERMS == 3 && __builtin_expect(__any(redo), 0)) {
#pragma unroll
    for (int db = 0; db < 8; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float ref = m == -INFINITY ? 0.f : m;
    for (int t = wave; t < tiles; t += DC_WAVES) {
      da_u32x4 kf[8];
      f32x4 s[2];
      load_v(0, t);
      load_k(kf, t);
      dot(kf, s);
      float p[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] = __builtin_amdgcn_exp2f(s[e >> 2][e & 3] * c - ref) * DA_P_SCALE(DTYPE);
      fc_wait_vm<0>();
      const int live = end - t0 - t * DA_TILE;
#pragma unroll 1
      for (int e = 0; e < 8; ++e) {
        const float own = p[0];
#pragma unroll
        for (int j = 0; j < 7; ++j) p[j] = p[j + 1];
#pragma unroll 1
        for (int k4 = 0; k4 < 4; ++k4) {
          const int key = (e >> 2) * 16 + k4 * 4 + (e & 3);
          const float pk = __shfl(own, k4 * 16 + l15, 64);
          if (key >= live) continue;                           // wave-uniform
          const char* r = smem + wave * DC_STAGES * DA_TILEB + key * 256 + (qd & 1) * 8;
#pragma unroll
          for (int db = 0; db < 8; ++db) {
            const uint2 x = *reinterpret_cast<const uint2*>(r + (((2 * db + (qd >> 1)) ^ (key & 15)) << 4));
            const unsigned w[2] = {x.x, x.y};
#pragma unroll
            for (int i = 0; i < 4; ++i) o[db][i] = fmaf(pk, da_unpack<DTYPE>((unsigned short)(w[i >> 1] >> (i & 1) * 16)), o[db][i]);
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  }

  // ---- the eight wavefronts' results into one ---------------------------------------------------------------------
  float2* ml = reinterpret_cast<float2*>(smem + DC_PART);   // [wavefront][head]: maximum, sum
  if (qd == 0) ml[wave * DC_HEADS + l15] = make_float2(m, l);
  __syncthreads();                                         // also: every wavefront is done with its V rows
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < DC_WAVES; ++w) M = fmaxf(M, ml[w * DC_HEADS + l15].x);
  float* part = reinterpret_cast<float*>(smem);
  {
    const float wgt = __builtin_amdgcn_exp2f(m - (M == -INFINITY ? 0.f : M)) * (1.f / DA_P_SCALE(DTYPE));   // 0 for a wavefront without tiles
    if (l15 < ng) {
#pragma unroll
      for (int db = 0; db < 8; ++db)
        *reinterpret_cast<f32x4*>(part + (wave * DC_HEADS + l15) * DC_PSTRIDE + db * 16 + qd * 4) = o[db] * wgt;
    }
  }
  __syncthreads();
  for (int i = tid; i < ng * FC_HEAD_DIM; i += DC_THREADS) {
    const int g = i / FC_HEAD_DIM, d = i - g * FC_HEAD_DIM;
    float mg = -INFINITY, lg = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < DC_WAVES; ++w) mg = fmaxf(mg, ml[w * DC_HEADS + g].x);
#pragma unroll
    for (int w = 0; w < DC_WAVES; ++w) {
      const float2 x = ml[w * DC_HEADS + g];
      lg = fmaf(__builtin_amdgcn_exp2f(x.x - (mg == -INFINITY ? 0.f : mg)), x.y, lg);
      acc += part[(w * DC_HEADS + g) * DC_PSTRIDE + d];
    }
    if (whole) {
      orow[i] = da_pack<DTYPE>(acc / lg);
    } else {
      const long long at = ((long long)b * Hq + h * G + g0 + g) * max_splits + blockIdx.z;
      dc_put<TURN>(part_o + at * FC_HEAD_DIM + d, acc);
      if (d == 0) {
        dc_put<TURN>(part_ml + at * 2, mg);
        dc_put<TURN>(part_ml + at * 2 + 1, lg);
      }
    }
  }
  if (!TURN || whole) return;

  // ---- the column's workgroups into one: whoever arrives last ------------------------------------------------------
  // Every workgroup whose range holds a token gets here, ns of them; nobody waits.  The partial results have reached the
  // device's point of coherence before the workgroup counts itself, so the last one reads all of them there.  (Ordinary
  // stores with a release and an acquire, which write back and drop caches, instead: 341 us for the 28 layers that take
  // 296 this way and 374 with the merge's own launch, host bound.)
  const int ns = (len + span - 1) / span;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  unsigned* arrived = (arrivals ? arrivals : dc_arrived[turn]) + (blockIdx.y * gridDim.x + blockIdx.x);
  unsigned* before = reinterpret_cast<unsigned*>(smem);
  if (tid == 0) *before = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (*before != (unsigned)(ns - 1)) return;
  if (tid == 0) __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const long long col = ((long long)b * Hq + h * G + g0) * max_splits;
  float2* all = reinterpret_cast<float2*>(smem + 16);       // [head][range]: maximum, sum
  constexpr int PAIRS = FC_HEAD_DIM / 2;
  float2 x[DC_MERGE];
  const auto load_o = [&](int i, int s0) {                  // two dimensions of a head, ranges s0 ..
    const float* po = part_o + (col + (long long)(i / PAIRS) * max_splits) * FC_HEAD_DIM + i % PAIRS * 2;
#pragma unroll
    for (int j = 0; j < DC_MERGE; ++j)
      x[j] = s0 + j < ns ? dc_get2(po + (long long)(s0 + j) * FC_HEAD_DIM) : make_float2(0.f, 0.f);
  };
  if (tid < ng * PAIRS) load_o(tid, 0);
  for (int i = tid; i < ng * ns; i += DC_THREADS) all[i] = dc_get2(part_ml + (col + (long long)(i / ns) * max_splits + i % ns) * 2);
  __syncthreads();
  // the arithmetic and the order of decode_merge_kernel
  for (int i = tid; i < ng * PAIRS; i += DC_THREADS) {
    const float2* ml = all + i / PAIRS * ns;
    float M = -INFINITY, L = 0.f;
    float2 acc = make_float2(0.f, 0.f);
    for (int s = 0; s < ns; ++s) M = fmaxf(M, ml[s].x);
    for (int s0 = 0; s0 < ns; s0 += DC_MERGE) {
      if (i != tid || s0) load_o(i, s0);
#pragma unroll
      for (int j = 0; j < DC_MERGE; ++j) {
        const float2 e = s0 + j < ns ? ml[s0 + j] : make_float2(-INFINITY, 0.f);
        const float w = __builtin_amdgcn_exp2f(e.x - M);
        L = fmaf(w, e.y, L);
        acc.x = fmaf(w, x[j].x, acc.x);
        acc.y = fmaf(w, x[j].y, acc.y);
      }
    }
    reinterpret_cast<unsigned*>(orow)[i] = (unsigned)da_pack<DTYPE>(acc.x / L) | ((unsigned)da_pack<DTYPE>(acc.y / L) << 16);
  }
}

// ---- append / advance ----------------------------------------------------------------------------------
template <int EB>
__global__ __launch_bounds__(256) void store_kv_kernel(KvView kc, KvView vc, const char* __restrict__ k_new,
                                                       const char* __restrict__ v_new,
                                                       const int* __restrict__ lens) {
  const int b = blockIdx.x, l = blockIdx.y;
  const int pos = lens[b];
  if (pos < 0 || pos >= kc.max_seq_len) return;
  const int H = kc.num_kv_heads;
  constexpr int CPR = FC_HEAD_DIM * EB / 16;  // 16-byte chunks per head row
  const long long koff = fc_token_offset(kc, b, pos), voff = fc_token_offset(vc, b, pos);
  if (koff < 0 || voff < 0) return;
  const long long row = ((long long)l * kc.batch + b) * H;
  for (int i = threadIdx.x; i < H * CPR; i += 256) {
    const int h = i / CPR, part = i - h * CPR;
    const long long srcb = ((row + h) * FC_HEAD_DIM) * EB + part * 16;
    *reinterpret_cast<uint4*>(kc.base + ((long long)l * kc.stride_layer + koff + (long long)h * kc.stride_head) * EB +
                              part * 16) = *reinterpret_cast<const uint4*>(k_new + srcb);
    *reinterpret_cast<uint4*>(vc.base + ((long long)l * vc.stride_layer + voff + (long long)h * vc.stride_head) * EB +
                              part * 16) = *reinterpret_cast<const uint4*>(v_new + srcb);
  }
}

// one new row per token i: cache[slot_mapping[i]] <- key[i], value[i]; a row is row_bytes long
__global__ __launch_bounds__(256) void store_slots_kernel(const char* __restrict__ key, long long key_stride_b,
                                                          const char* __restrict__ value, long long value_stride_b,
                                                          char* __restrict__ k_cache, char* __restrict__ v_cache,
                                                          const int* __restrict__ slot_mapping, int row_bytes) {
  const int i = blockIdx.x;
  const long long slot = slot_mapping[i];
  if (slot < 0) return;
  for (int o = threadIdx.x * 16; o < row_bytes; o += 256 * 16) {
    *reinterpret_cast<uint4*>(k_cache + slot * row_bytes + o) = *reinterpret_cast<const uint4*>(key + i * key_stride_b + o);
    *reinterpret_cast<uint4*>(v_cache + slot * row_bytes + o) = *reinterpret_cast<const uint4*>(value + i * value_stride_b + o);
  }
}

__global__ void advance_lens_kernel(int* lens, int n, int delta) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && lens[i] >= 0) lens[i] += delta;
}

// A step's inputs into the static buffers of a captured graph, whole: rows [layer][sequence] of q, k and v into buffers
// of max_batch sequences per layer, and slots, lengths and tables with the padding rows reset (slot -1, length 0, table
// 0).  One launch instead of the nine fills and copies of a few microseconds each that stood before every replay.
struct StageRows {
  const uint4* src;
  uint4* dst;
  long long src_layer, src_row, dst_layer;   // in 16-byte pieces; destination rows are adjacent
  int pieces;                                // per row
};
__global__ __launch_bounds__(256) void stage_decode_kernel(StageRows q, StageRows k, StageRows v, int layers, int bs,
                                                           const int* __restrict__ slots, const int* __restrict__ lens,
                                                           const int* __restrict__ tables, int width,
                                                           int* __restrict__ g_slots, int* __restrict__ g_lens,
                                                           int* __restrict__ g_tables, int max_bs, int g_width) {
  const long long step = (long long)gridDim.x * 256;
  const int per_row = q.pieces + k.pieces + v.pieces;
  const long long n = (long long)layers * bs * per_row;
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += step) {
    const long long row = i / per_row;
    int p = (int)(i - row * per_row);
    const int l = (int)(row / bs), b = (int)(row - (long long)l * bs);
    if (p < q.pieces) {
      q.dst[l * q.dst_layer + (long long)b * q.pieces + p] = q.src[l * q.src_layer + b * q.src_row + p];
    } else if ((p -= q.pieces) < k.pieces) {
      k.dst[l * k.dst_layer + (long long)b * k.pieces + p] = k.src[l * k.src_layer + b * k.src_row + p];
    } else {
      p -= k.pieces;
      v.dst[l * v.dst_layer + (long long)b * v.pieces + p] = v.src[l * v.src_layer + b * v.src_row + p];
    }
  }
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < (long long)max_bs * g_width; i += step) {
    const int b = (int)(i / g_width), j = (int)(i - (long long)b * g_width);
    g_tables[i] = b < bs && j < width ? tables[(long long)b * width + j] : 0;
    if (j == 0) {
      g_slots[b] = b < bs ? slots[b] : -1;
      g_lens[b] = b < bs ? lens[b] : 0;
    }
  }
}

extern "C" int fc_stage_decode(const void* q, int64_t q_layer, int64_t q_row, const void* k, int64_t k_layer, int64_t k_row,
                               const void* v, int64_t v_layer, int64_t v_row, int32_t num_layers, int32_t batch,
                               int32_t q_elems, int32_t kv_elems, int32_t dtype, const int32_t* slots,
                               const int32_t* context_lens, const int32_t* tables, int32_t table_width, void* q_static,
                               void* k_static, void* v_static, int32_t* slots_static, int32_t* lens_static,
                               int32_t* tables_static, int32_t max_batch, int32_t max_width, void* stream) {
  const char* who = "fc_stage_decode";
  FC_REQUIRE(q && k && v && slots && context_lens && tables && q_static && k_static && v_static && slots_static &&
                 lens_static && tables_static,
             FC_EINVAL, "%s: null pointer", who);
  FC_REQUIRE(dtype == FC_F32 || dtype == FC_F16 || dtype == FC_BF16, FC_EINVAL, "%s: unknown dtype %d", who, dtype);
  FC_REQUIRE(num_layers > 0 && batch > 0 && batch <= max_batch && table_width > 0 && table_width <= max_width && q_elems > 0 &&
                 kv_elems > 0,
             FC_EINVAL, "%s: bad sizes", who);
  const int eb = fc_elem_bytes(dtype);
  const int64_t all = (q_layer | q_row | k_layer | k_row | v_layer | v_row | q_elems | kv_elems) * eb;
  FC_REQUIRE((all & 15) == 0 && (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)q_static | (uintptr_t)k_static |
                                  (uintptr_t)v_static) & 15) == 0,
             FC_EINVAL, "%s: rows, strides and pointers must be multiples of 16 bytes", who);
  const auto rows = [&](const void* src, int64_t layer, int64_t row, void* dst, int elems) {
    return StageRows{(const uint4*)src, (uint4*)dst, layer * eb / 16, row * eb / 16, (long long)max_batch * elems * eb / 16,
                     elems * eb / 16};
  };
  const long long n = (long long)num_layers * batch * (q_elems + 2 * kv_elems) * eb / 16;
  const unsigned grid = (unsigned)(n / 256 + 1 < 1024 ? n / 256 + 1 : 1024);
  hipLaunchKernelGGL(stage_decode_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream,
                     rows(q, q_layer, q_row, q_static, q_elems), rows(k, k_layer, k_row, k_static, kv_elems),
                     rows(v, v_layer, v_row, v_static, kv_elems), num_layers, batch, slots, context_lens, tables, table_width,
                     slots_static, lens_static, tables_static, max_batch, max_width);
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}

extern "C" int fc_store_kv(const fc_kv_view* k_cache, const fc_kv_view* v_cache, const void* k_new,
                           const void* v_new, const int32_t* context_lens, void* stream) {
  const char* who = "fc_store_kv";
  int rc;
  if ((rc = fc_check_view(k_cache, who)) || (rc = fc_check_view(v_cache, who))) return rc;
  FC_REQUIRE(k_cache->dtype == v_cache->dtype && k_cache->num_layers == v_cache->num_layers &&
                 k_cache->batch == v_cache->batch && k_cache->num_kv_heads == v_cache->num_kv_heads,
             FC_EINVAL, "%s: K and V views disagree", who);
  FC_REQUIRE(k_new && v_new && context_lens, FC_EINVAL, "%s: null pointer", who);
  FC_REQUIRE((((uintptr_t)k_new | (uintptr_t)v_new) & 15) == 0, FC_EINVAL, "%s: new rows not 16-byte aligned", who);
  KvView k = fc_make_view(k_cache), v = fc_make_view(v_cache);
  dim3 grid(k_cache->batch, k_cache->num_layers);
  hipStream_t st = (hipStream_t)stream;
  if (k_cache->dtype == FC_F32)
    hipLaunchKernelGGL((store_kv_kernel<4>), grid, dim3(256), 0, st, k, v, (const char*)k_new, (const char*)v_new,
                       context_lens);
  else
    hipLaunchKernelGGL((store_kv_kernel<2>), grid, dim3(256), 0, st, k, v, (const char*)k_new, (const char*)v_new,
                       context_lens);
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}

extern "C" int fc_store_kv_slots(const void* key, int64_t key_stride, const void* value, int64_t value_stride,
                                 void* k_cache, void* v_cache, const int32_t* slot_mapping, int32_t num_tokens,
                                 int32_t row_elems, int32_t dtype, void* stream) {
  const char* who = "fc_store_kv_slots";
  FC_REQUIRE(key && value && k_cache && v_cache && slot_mapping, FC_EINVAL, "%s: null pointer", who);
  FC_REQUIRE(dtype == FC_F32 || dtype == FC_F16 || dtype == FC_BF16, FC_EINVAL, "%s: unknown dtype %d", who, dtype);
  FC_REQUIRE(num_tokens >= 0 && row_elems > 0, FC_EINVAL, "%s: bad sizes", who);
  const int eb = fc_elem_bytes(dtype);
  FC_REQUIRE(((int64_t)row_elems * eb) % 16 == 0 && (key_stride * eb) % 16 == 0 && (value_stride * eb) % 16 == 0,
             FC_EINVAL, "%s: rows and strides must be multiples of 16 bytes", who);
  FC_REQUIRE((((uintptr_t)key | (uintptr_t)value | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0, FC_EINVAL,
             "%s: pointers must be 16-byte aligned", who);
  if (num_tokens == 0) return FC_OK;
  hipLaunchKernelGGL(store_slots_kernel, dim3(num_tokens), dim3(256), 0, (hipStream_t)stream, (const char*)key,
                     (long long)key_stride * eb, (const char*)value, (long long)value_stride * eb, (char*)k_cache,
                     (char*)v_cache, slot_mapping, row_elems * eb);
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}

extern "C" int fc_advance_lens(int32_t* context_lens, int32_t batch, int32_t delta, void* stream) {
  FC_REQUIRE(context_lens && batch > 0, FC_EINVAL, "fc_advance_lens: bad arguments");
  hipLaunchKernelGGL(advance_lens_kernel, dim3((batch + 255) / 256), dim3(256), 0, (hipStream_t)stream, context_lens,
                     batch, delta);
  FC_CHECK_LAUNCH("fc_advance_lens");
  return FC_OK;
}

extern "C" int64_t fc_decode_attn_workspace_bytes(int32_t batch, int32_t num_q_heads, int32_t max_seq_len) {
  if (batch <= 0 || num_q_heads <= 0 || max_seq_len < 0) return -1;
  const int64_t splits = (max_seq_len + DA_CHUNK - 1) / DA_CHUNK;
  return (int64_t)batch * num_q_heads * (splits > 0 ? splits : 1) * (FC_HEAD_DIM + 2) * (int64_t)sizeof(float);
}

// A 32-token tile never straddles two pages and its byte offsets fit 32 bits.
static bool da_tile_in_page(const fc_kv_view* v) {
  return v->stride_token >= 0 && v->stride_token < (1 << 24) &&
         (v->block_tables == nullptr || (v->block_size >= DA_TILE && (v->block_size & (v->block_size - 1)) == 0));
}

// Tokens per workgroup of the column kernel, 0 = the launch does not take it.  It takes launches whose workgroups are all
// resident at once (one per compute unit: registers) and, of groups of 5 and more heads, twice as many short columns: beyond
// that bandwidth counts and the split kernel streams better (128 columns of 1024 tokens: 19.4 us a layer against 19.6 to 23).  One 32-token tile per wavefront, 256 tokens, is
// the shortest chain (a second tile costs about 3 us, a merge 3.5): 12 columns of 1024 tokens 13.2 -> 10.1 us, of 256
// tokens without a merge 7.1, 48 columns of 1024 tokens 16.9 -> 13.0.  Where 256 would be too many workgroups, columns
// short enough for one workgroup each still gain by not being merged: 192 columns of 512 tokens 16.7 -> 15.4 us, 256 of
// 768 tokens 23.6 -> 22.5.
// Longer ranges, several tiles a wavefront, as long as one round of workgroups holds them, against the split kernel (us a
// pass: eager layers, 28 or 16 of them, append and merge launches included; captured layers gain the same shares).  Groups of
// 5 and more heads, where a K and V read once feeds the matrix pipe for all of them: 2 tiles, 48 columns of 1500 tokens
// 569 -> 464, 24 of 5000 639 -> 489; 4, 64 of 4000 in groups of 8 1012 -> 752; 8, 200 of 1700 1073 -> 929; 8, 64 of 8000
// 784 -> 697; and two rounds of whole columns, 360 of 600 621 -> 451, 400 of 300 529 -> 330, but not of longer ones (360 of
// 2000 1030 -> 1054).  Smaller groups leave those to the split kernel, which holds them whole as well (12 captured layers, this /
// that: 32 heads, 10 of 100 to 250 186 / 165, 14 of 250 247 / 220, 16 of 500 342 / 333; 32 heads on 8, 48 of 100 to 500
// 287 / 289, of 500 373 / 337, 40 of 700 445 / 394, 36 of 100 to 700 301 / 315).
// Up to 4 heads a group, where the split kernel holds columns of up to 1024 tokens whole and appends inside: us a captured layer,
// split kernel / this (eager layers of these sizes: the same shares), lengths equal | a tenth to all of the longest.
// Two tiles always: 32 heads, 2 of 2048 21.0 / 19.8 | 20.1 / 19.0, on 8 kv heads 8 of 2048 25.4 / 22.6 | 21.5 / 20.1.
// Groups of 3 and 4, 3 and 4 tiles: on 8 kv heads 8 of 2560 27.9 / 25.8 | 22.9 / 21.5, of 4096 34.0 / 32.0 | 31.0 / 28.8, 24 of
// 1024 30.4 / 26.1 | 26.9 / 23.1, 16 of 2048 34.0 / 32.4 | 30.1 / 28.5, 4 of 6144 30.4 / 27.3 | 26.6 / 23.2, 12 of 1280
// 24.2 / 23.4 | 19.4 / 20.0; but 4 tiles of few ranges that are not full and leave a quarter of the compute units idle do not
// pay: 12 of 1792 26.8 / 27.1 | 24.0 / 25.3.  5 and 6 tiles: 12 of 2304 31.9 / 32.4 | 25.8 / 28.3, 20 of 1536 31.9 / 32.4 |
// 27.3 / 30.2.
// Groups of 1 and 2, 3 to 6 tiles: whole columns that fill three quarters of the compute units, 32 heads, 6 of 1024 26.6 / 25.2 |
// 24.7 / 24.0, of 1280 33.9 / 30.2 | 28.5 / 26.5, of 1536 37.8 / 35.0 | 33.9 / 33.1, 8 of 1280 36.1 / 35.0 | 28.9 / 28.4, but of
// 1536 with one head a group 41.1 / 40.6 | 34.4 / 36.0; ranges 85 % full, seven eighths of the compute units busy, where two of
// three hold: 3 tiles, 7 ranges or more, two heads a group or all units busy: 32 heads, 1 of 5120 26.1 / 24.3, of 8192
// 37.2 / 32.3, of 10240 39.7 / 37.8, 2 of 3072 26.0 / 25.6 | 26.8 / 26.4, on 16 kv heads 3 of 3584 25.8 / 25.0 | 22.4 / 22.4, 2 of
// 7168 31.7 / 30.2 | 29.4 / 28.6; else 4 of 1792 28.4 / 29.4 | 26.4 / 27.8, of 2304 33.5 / 35.1 | 27.8 / 30.6, 2 of 4608
// 36.1 / 36.8 | 29.6 / 30.9, on 16 3 of 5632 33.6 / 35.3 | 28.9 / 30.9; 8 heads, 5 of 4096 23.7 / 24.7 | 20.7 / 21.4, of 5632
// 29.0 / 30.5 | 23.6 / 25.9.
#define DC_ONE 768
#define DC_TILES_FEW 6
#define DC_TILES_SOME 4
#define DC_TILES_MANY 16
// Eager layers, launched one by one, gain where the last workgroup of a column merges it: a launch less for the host
// (12 to 13 us a layer before) and 0 to 1 us of waiting for the device.  28 layers, merge launch -> last workgroup: 2 ranges
// 379 -> 284 us, 4 of 12 to 48 columns 372 -> 296 to 346, 10 of 8 columns 380 -> 318, 14 of 4 columns 379 -> 327, 15 of 16
// columns 375 -> 381, 16 of 8 columns 379 -> 364, 24 to 31 of 8 columns 1 to 2 % slower (28 of 4 columns 6 % faster): the
// ranges of a column are read eight at a time by one workgroup, past the caches.
#define DC_SPLITS 14
static int da_column_chunk(const fc_kv_view* k, const fc_kv_view* v, int num_q_heads) {
  const int G = num_q_heads / k->num_kv_heads;
  const long long cols = (long long)k->num_kv_heads * ((G + DC_HEADS - 1) / DC_HEADS) * k->batch;
  const long long slots = fc_compute_units();
  const auto pages_ok = [](const fc_kv_view* x) {       // one block-table entry per lane
    return x->block_tables == nullptr || (x->max_seq_len - 1) / x->block_size < FC_WAVE;
  };
  if ((k->block_tables == nullptr) != (v->block_tables == nullptr) || k->max_seq_len <= 0 || !da_tile_in_page(k) ||
      !da_tile_in_page(v) || !pages_ok(k) || !pages_ok(v))
    return 0;
  const int chunk = DC_WAVES * DA_TILE;
  if (cols * ((k->max_seq_len + chunk - 1) / chunk) <= slots) return chunk;
  if (cols <= (G > 4 ? 2 : 1) * slots && k->max_seq_len <= DC_ONE) return DC_ONE;
  const int most = G > 4 ? DC_TILES_MANY : G > 2 ? DC_TILES_SOME : DC_TILES_FEW;
  for (int m = 2; m <= most; ++m) {
    const long long ranges = (k->max_seq_len + m * chunk - 1) / (m * chunk), wgs = cols * ranges;
    if (wgs > slots) continue;
    const bool busy = 8 * wgs >= 7 * slots, all = wgs == slots;
    const auto full = [&](int percent) { return 100ll * k->max_seq_len >= percent * ranges * m * chunk; };
    if (m == 2 || G > 4) return m * chunk;
    if (G > 2) return m == 3 || busy || ranges == 1 || ranges > 3 || full(90) ? m * chunk : 0;
    if (ranges == 1) return 4 * wgs >= 3 * slots && (m < DC_TILES_FEW || G == 2 || !busy) ? m * chunk : 0;
    return busy && full(85) && (m == 3) + (ranges >= 7) + (all || G == 2) >= 2 ? m * chunk : 0;
  }
  return 0;
}

// the smallest tile that holds the whole group (padded head rows cost nothing; splitting a group would
// read its K and V once per tile); groups of more than 8 heads are served 8 at a time
static int da_group_tile(int G) { return G > 4 ? 8 : G > 2 ? 4 : G > 1 ? 2 : 1; }

// Tokens per workgroup: the multiple of 32 between 256 and 1024 that minimises rounds * (chunk + fixed part),
// rounds = workgroups / (two per compute unit), rounded up.  Longer chunks spend less of a workgroup's life on
// its ramp (first tiles in flight, nothing to compute yet) and its tail (statistics, partial results, no loads
// in flight); a launch of few workgroups wants the chunk that fills whole rounds.  Measured: cfg4 (2880
// columns, up to 2304 tokens) 0.327 ms per layer with 256, 0.297 with 512, 0.294 with 768; cfg5's decode (64
// columns, 3584 tokens) 33.3 us with 256, 30.4 with 448.  Two workgroups must still fit a compute unit's LDS, which
// caps the chunk for groups of 8 query heads.  Only the view's max_seq_len enters, never the lengths on the
// device, so the choice is the same at capture and at every replay.
static int da_split_chunk(const fc_kv_view* k, const fc_kv_view* v, int num_q_heads) {
  const int G = num_q_heads / k->num_kv_heads, gt = da_group_tile(G);
  const int slots = 2 * fc_compute_units();
  const long long cols = (long long)k->num_kv_heads * ((G + gt - 1) / gt) * k->batch;
  const auto fits = [&](int cand) { return (DA_RING + gt * cand * 4) * 2 <= 158 * 1024; };
  int chunk = DA_CHUNK;
  double best = -1.0;
  for (int cand = DA_CHUNK; cand <= DA_CHUNK_MAX && fits(cand); cand += DA_TILE) {
    const long long wgs = cols * ((k->max_seq_len + cand - 1) / cand);
    const double cost = (double)((wgs + slots - 1) / slots) * (cand + 96.0);
    if (best < 0 || cost < best - 1e-9) {
      best = cost;
      chunk = cand;
    }
  }
  // Whole columns need no merge and append by themselves, two launches and 4 us a layer less, and long workgroups of different
  // lengths even out where chunks come in rounds: 300 tokens of a round; workgroups past the first round cost their share of one.
  // us per step, 12 captured layers, chunks -> whole: 32 heads, 20 sequences of 100 to 300 tokens 319 -> 272, of 500 546 -> 494,
  // of 100 to 700 480 -> 413, of 100 to 1000 555 -> 417, of 1000 870 -> 829, 10 of 750 422 -> 371, 9 of 1000 472 -> 451, 60 of 100 to
  // 500 800 -> 742, 90 of 500 1729 -> 1686; 32 on 16, 20 of 100 to 700 341 -> 272, 40 499 -> 448; 32 on 8, 90 of 128 to 500
  // 579 -> 471, of 700 807 -> 723.  Fewer columns: 7 of 1000 328 -> 329, 5 of 100 to 900 247 -> 256.
  const int whole = (k->max_seq_len + DA_TILE - 1) / DA_TILE * DA_TILE;
  if (whole >= DA_CHUNK && whole <= DA_CHUNK_MAX && fits(whole) && da_tile_in_page(k) && da_tile_in_page(v) &&
      fmax(1.0, (double)cols / slots) * (whole + 96.0) - 300.0 < best)
    return whole;
  return chunk;
}

// What a launch of this shape is, decided once a call: the column kernel, or the split kernel in chunks or with whole columns (no
// merge).
struct DaPlan {
  int column;      // tokens a workgroup of the column kernel, 0: the split kernel
  int chunk;       // ... of the split kernel
  bool whole;      // the split kernel holds every sequence in one chunk
};
static DaPlan da_plan(const fc_kv_view* k, const fc_kv_view* v, int num_q_heads) {
  DaPlan p{da_column_chunk(k, v, num_q_heads), 0, false};
  if (p.column) return p;
  p.chunk = da_split_chunk(k, v, num_q_heads);
  p.whole = k->max_seq_len > 0 && k->max_seq_len <= p.chunk && da_tile_in_page(k) && da_tile_in_page(v);
  return p;
}

static int da_merge(const char* who, const fc_kv_view* k_cache, const float* part_o, const float* part_ml,
                    const int32_t* context_lens, int num_q_heads, int splits, int chunk, int alone, void* out, void* stream) {
  dim3 grid(num_q_heads, k_cache->batch);
  if (k_cache->dtype == FC_BF16)
    hipLaunchKernelGGL((decode_merge_kernel<FC_BF16>), grid, dim3(FC_HEAD_DIM), 0, (hipStream_t)stream, part_o, part_ml,
                       context_lens, k_cache->max_seq_len, num_q_heads, splits, chunk, alone, (char*)out);
  else
    hipLaunchKernelGGL((decode_merge_kernel<FC_F16>), grid, dim3(FC_HEAD_DIM), 0, (hipStream_t)stream, part_o, part_ml,
                       context_lens, k_cache->max_seq_len, num_q_heads, splits, chunk, alone, (char*)out);
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}

// Checks and launches shared by the entry points; `workspace` is a device address, `plan` the caller's where it has one.
static int da_enqueue(const char* who, const fc_kv_view* k_cache, const fc_kv_view* v_cache, int32_t layer,
                      const void* q, void* out, int32_t num_q_heads, const int32_t* context_lens, float scale,
                      void* workspace, int64_t workspace_bytes, void* stream, const DaAppend* append = nullptr,
                      int turn = -1, uint32_t* arrivals = nullptr, const DaPlan* plan = nullptr) {
  int rc;
  if ((rc = fc_check_view(k_cache, who)) || (rc = fc_check_view(v_cache, who))) return rc;
  FC_REQUIRE(k_cache->dtype == v_cache->dtype && k_cache->num_layers == v_cache->num_layers &&
                 k_cache->batch == v_cache->batch && k_cache->num_kv_heads == v_cache->num_kv_heads &&
                 k_cache->max_seq_len == v_cache->max_seq_len,
             FC_EINVAL, "%s: K and V views disagree", who);
  FC_REQUIRE(k_cache->dtype == FC_F16 || k_cache->dtype == FC_BF16, FC_EUNSUPPORTED, "%s: fp16/bf16 caches only", who);
  FC_REQUIRE(layer >= 0 && layer < k_cache->num_layers, FC_EINVAL, "%s: layer %d out of range", who, layer);
  FC_REQUIRE(num_q_heads > 0 && num_q_heads % k_cache->num_kv_heads == 0, FC_EINVAL,
             "%s: num_q_heads %d not a multiple of num_kv_heads %d", who, num_q_heads, k_cache->num_kv_heads);
  FC_REQUIRE(q && out && context_lens, FC_EINVAL, "%s: null pointer", who);
  const DaPlan shape = plan ? *plan : da_plan(k_cache, v_cache, num_q_heads);
  const int column = shape.column;
  const int csplits = column ? (k_cache->max_seq_len + column - 1) / column : 0;
  // one workgroup per column needs no workspace; a caller that appends in the same call has asked whether one is needed
  FC_REQUIRE(workspace || (csplits == 1 && append), FC_EINVAL, "%s: null workspace", who);
  FC_REQUIRE((((uintptr_t)q | (uintptr_t)workspace) & 15) == 0, FC_EINVAL, "%s: q/workspace not 16-byte aligned", who);
  if (column) {
    // (for a range of 256 tokens or more per workgroup the splits fit what the smallest chunk of 256 needs)
    FC_REQUIRE((csplits == 1 && append) ||
                   workspace_bytes >= fc_decode_attn_workspace_bytes(k_cache->batch, num_q_heads, k_cache->max_seq_len),
               FC_EINVAL, "%s: workspace of %lld bytes is too small", who, (long long)workspace_bytes);
    const int G = num_q_heads / k_cache->num_kv_heads;
    dim3 grid(k_cache->num_kv_heads * ((G + DC_HEADS - 1) / DC_HEADS), k_cache->batch, csplits);
    float* part_o = (float*)workspace;
    float* part_ml = part_o ? part_o + (int64_t)k_cache->batch * num_q_heads * csplits * FC_HEAD_DIM : nullptr;
    const DaAppend ap = append ? *append : DaAppend{nullptr, nullptr, 0, 0, nullptr};
    if ((int64_t)grid.x * grid.y > DC_COLUMNS || csplits > DC_SPLITS || !k_cache->block_tables) {
      turn = -1;
      arrivals = nullptr;
    }
    const bool last_merges = turn >= 0 || arrivals;
    const KvView k = fc_make_view(k_cache), v = fc_make_view(v_cache);
#define DC_LAUNCH3(DT, TERMS, PG, TURN)                                                                            \
  do {                                                                                                             \
    FC_ALLOW_LDS((decode_column_kernel<DT, TERMS, PG, TURN>), DC_LDS);                                              \
    hipLaunchKernelGGL((decode_column_kernel<DT, TERMS, PG, TURN>), grid, dim3(DC_THREADS), DC_LDS, (hipStream_t)stream, \
                       k, v, layer, (const char*)q, num_q_heads, context_lens, scale * DA_LOG2E, (char*)out, ap,    \
                       column, part_o, part_ml, csplits, turn, arrivals);                                                  \
  } while (0)
// (a turn comes with paged caches)
#define DC_LAUNCH(DT, TERMS)                                      \
  if (!k_cache->block_tables) DC_LAUNCH3(DT, TERMS, false, false); \
  else if (!last_merges || csplits == 1) DC_LAUNCH3(DT, TERMS, true, false); \
  else DC_LAUNCH3(DT, TERMS, true, true)
    if (k_cache->dtype == FC_F16) {
      if (G > 4) { DC_LAUNCH(FC_F16, 2); } else { DC_LAUNCH(FC_F16, 3); }
    } else {
      if (G > 4) { DC_LAUNCH(FC_BF16, 2); } else { DC_LAUNCH(FC_BF16, 3); }
    }
#undef DC_LAUNCH3
#undef DC_LAUNCH
    FC_CHECK_LAUNCH(who);
    if (csplits > 1 && !last_merges)
      return da_merge(who, k_cache, part_o, part_ml, context_lens, num_q_heads, csplits, column, DC_ALONE, out, stream);
    return FC_OK;
  }
  const int64_t need = fc_decode_attn_workspace_bytes(k_cache->batch, num_q_heads, k_cache->max_seq_len);
  FC_REQUIRE(workspace_bytes >= need, FC_EINVAL, "%s: workspace of %lld bytes, %lld needed", who,
             (long long)workspace_bytes, (long long)need);
  const int B = k_cache->batch, Hkv = k_cache->num_kv_heads, G = num_q_heads / Hkv;
  const int gt = da_group_tile(G), gtiles = (G + gt - 1) / gt;
  const int chunk = shape.chunk;
  const int splits = (k_cache->max_seq_len + chunk - 1) / chunk;
  float* part_o = (float*)workspace;
  float* part_ml = part_o + (int64_t)B * num_q_heads * (splits > 0 ? splits : 1) * FC_HEAD_DIM;
  KvView k = fc_make_view(k_cache), v = fc_make_view(v_cache);
  hipStream_t st = (hipStream_t)stream;
  const float c = scale * DA_LOG2E;
  const bool bf = k_cache->dtype == FC_BF16;
  if (splits > 0) {
    FC_REQUIRE(Hkv * gtiles <= 65535 && B <= 65535, FC_EUNSUPPORTED, "%s: grid too large", who);
    dim3 grid(splits, Hkv * gtiles, B);
    const bool fast = da_tile_in_page(k_cache) && da_tile_in_page(v_cache), whole = shape.whole;
    const DaAppend ap = append ? *append : DaAppend{nullptr, nullptr, 0, 0, nullptr};
#define DA_LAUNCH(DT, GTV, FA, WH, AP)                                                                                   \
  do {                                                                                                          \
    FC_ALLOW_LDS((decode_attn_kernel<DT, GTV, FA, WH, AP>), DaCfg<GTV>::lds(DA_CHUNK_MAX));                             \
    hipLaunchKernelGGL((decode_attn_kernel<DT, GTV, FA, WH, AP>), grid, dim3(DA_THREADS), DaCfg<GTV>::lds(chunk), st, k, \
                       v, layer, (const char*)q, num_q_heads, context_lens, c, part_o, part_ml, splits, chunk, (char*)out, ap); \
  } while (0)
#define DA_DISPATCH2(DT, FA, WH)                     \
  switch (gt) {                                      \
    case 8: DA_LAUNCH(DT, 8, FA, WH, false); break;  \
    case 4: DA_LAUNCH(DT, 4, FA, WH, false); break;  \
    case 2: DA_LAUNCH(DT, 2, FA, WH, false); break;  \
    default: DA_LAUNCH(DT, 1, FA, WH, false); break; \
  }
#define DA_DISPATCH(DT)                                                                                  \
  if (whole) { DA_DISPATCH2(DT, true, true) } else if (!fast) { DA_DISPATCH2(DT, false, false) }         \
  else if (!ap.k_new) { DA_DISPATCH2(DT, true, false) }                                                  \
  else if (gt == 4) DA_LAUNCH(DT, 4, true, false, true);      /* (da_split_appends: up to 4 heads) */   \
  else if (gt == 2) DA_LAUNCH(DT, 2, true, false, true);                                                 \
  else DA_LAUNCH(DT, 1, true, false, true);
    if (bf) { DA_DISPATCH(FC_BF16) } else { DA_DISPATCH(FC_F16) }
#undef DA_DISPATCH
#undef DA_DISPATCH2
#undef DA_LAUNCH
    FC_CHECK_LAUNCH(who);
    if (whole) return FC_OK;
  }
  return da_merge(who, k_cache, part_o, part_ml, context_lens, num_q_heads, splits, chunk, 0, out, stream);
}

extern "C" int fc_decode_attn(const fc_kv_view* k_cache, const fc_kv_view* v_cache, int32_t layer, const void* q,
                              void* out, int32_t num_q_heads, const int32_t* context_lens, float scale,
                              void* workspace, int64_t workspace_bytes, void* stream) {
  return da_enqueue("fc_decode_attn", k_cache, v_cache, layer, q, out, num_q_heads, context_lens, scale, workspace,
                    workspace_bytes, stream);
}

// The split kernel's workgroups append where one serves a kv head: whole columns, and chunks of groups of up to 4 heads.  us per
// step, 12 captured layers, a launch of its own -> inside: 32 heads, 4 sequences of 600 to 6000 tokens 762 -> 750, 8 of 200 to
// 2000 502 -> 482, 20 of 300 to 2500 1090 -> 1059; 32 on 8, 30 of 400 to 4000 734 -> 706, 60 of 300 to 3000 1105 -> 1076, 90
// of 100 to 1200 863 -> 842 (861 where the slots past the first 64 were asked for in their turn); chunks of 7 heads a group
// lose (90 of 100 to 1000 541 -> 550).  Every workgroup looks at the slots of the whole batch: above 128 sequences that costs
// more than the launch (6 layers: 256 of 60 to 250 inside 1044, apart 911; 200 of 100 to 250 880, 779; 128 of 60 to 120 405, 406).
static bool da_split_appends(const fc_kv_view* k, const fc_kv_view* v, int num_q_heads, const DaPlan& p) {
  const int G = num_q_heads / k->num_kv_heads;
  return k->batch <= 2 * FC_WAVE && G <= 8 && da_tile_in_page(k) && da_tile_in_page(v) && (G <= 4 || p.whole);
}

// Append and attention of one layer.  The workgroup of a column appends its own head's row, so the fused form needs
// one workgroup per kv head (groups of up to 16 query heads, 8 for whole columns of the split kernel) and both caches on one
// block table; otherwise the rows go in first, in a launch of their own.
static bool da_one_table(const fc_kv_view* k, const fc_kv_view* v, int num_q_heads) {
  return num_q_heads / k->num_kv_heads <= DC_HEADS && k->block_tables && k->block_tables == v->block_tables &&
         k->table_stride == v->table_stride && k->block_size == v->block_size && k->max_seq_len > 0;
}
static bool da_appends_inside(const fc_kv_view* k, const fc_kv_view* v, int num_q_heads, const DaPlan& p) {
  return da_one_table(k, v, num_q_heads) && (p.column > 0 || da_split_appends(k, v, num_q_heads, p));
}

extern "C" int64_t fc_decode_layer_workspace_bytes(const fc_kv_view* k_cache, const fc_kv_view* v_cache,
                                                   int32_t num_q_heads) {
  if (!k_cache || !v_cache || num_q_heads <= 0 || k_cache->num_kv_heads <= 0 || k_cache->batch <= 0 ||
      num_q_heads % k_cache->num_kv_heads || k_cache->block_size <= 0 || v_cache->block_size <= 0)
    return -1;
  if (da_one_table(k_cache, v_cache, num_q_heads) && da_column_chunk(k_cache, v_cache, num_q_heads) >= k_cache->max_seq_len)
    return 0;
  return fc_decode_attn_workspace_bytes(k_cache->batch, num_q_heads, k_cache->max_seq_len);
}

extern "C" int fc_decode_layer(const fc_kv_view* k_cache, const fc_kv_view* v_cache, const void* q, const void* k_new,
                               int64_t k_stride, const void* v_new, int64_t v_stride, const int32_t* slot_mapping,
                               void* out, int32_t num_q_heads, const int32_t* context_lens, float scale, void* workspace,
                               int64_t workspace_bytes, void* stream) {
  return fc_decode_layer_turn(k_cache, v_cache, q, k_new, k_stride, v_new, v_stride, slot_mapping, out, num_q_heads,
                              context_lens, scale, workspace, workspace_bytes, -1, stream);
}

static int da_layer(const fc_kv_view* k_cache, const fc_kv_view* v_cache, const void* q, const void* k_new, int64_t k_stride,
                    const void* v_new, int64_t v_stride, const int32_t* slot_mapping, void* out, int32_t num_q_heads,
                    const int32_t* context_lens, float scale, void* workspace, int64_t workspace_bytes, int32_t turn,
                    uint32_t* arrivals, void* stream) {
  const char* who = "fc_decode_layer";
  int rc;
  FC_REQUIRE(turn >= -1 && turn < FC_DECODE_TURNS, FC_EINVAL, "%s: turn %d", who, turn);
  if ((rc = fc_check_view(k_cache, who)) || (rc = fc_check_view(v_cache, who))) return rc;
  FC_REQUIRE(k_new && v_new && slot_mapping, FC_EINVAL, "%s: null pointer", who);
  FC_REQUIRE(k_cache->block_tables && v_cache->block_tables && k_cache->num_layers == 1 && v_cache->num_layers == 1, FC_EINVAL,
             "%s: paged caches of one layer expected", who);
  const int64_t row = (int64_t)k_cache->num_kv_heads * FC_HEAD_DIM;
  for (const fc_kv_view* v : {k_cache, v_cache})
    FC_REQUIRE((v->stride_token == row || v->block_size == 1) && (v->stride_head == FC_HEAD_DIM || v->num_kv_heads == 1) &&
                   (v->stride_block == 0 || v->stride_block == row * v->block_size),
               FC_EINVAL, "%s: a slot counts tokens of a contiguous cache", who);
  FC_REQUIRE(num_q_heads > 0 && num_q_heads % k_cache->num_kv_heads == 0, FC_EINVAL,
             "%s: num_q_heads %d not a multiple of num_kv_heads %d", who, num_q_heads, k_cache->num_kv_heads);
  const int eb = fc_elem_bytes(k_cache->dtype);
  FC_REQUIRE((((uintptr_t)k_new | (uintptr_t)v_new | (uint64_t)(k_stride * eb) | (uint64_t)(v_stride * eb)) & 15) == 0, FC_EINVAL,
             "%s: new rows not 16-byte aligned", who);
  const DaPlan plan = da_plan(k_cache, v_cache, num_q_heads);
  if (da_appends_inside(k_cache, v_cache, num_q_heads, plan)) {
    const DaAppend ap = {(const char*)k_new, (const char*)v_new, k_stride * eb, v_stride * eb, slot_mapping};
    return da_enqueue(who, k_cache, v_cache, 0, q, out, num_q_heads, context_lens, scale, workspace, workspace_bytes,
                      stream, &ap, turn, arrivals, &plan);
  }
  // what the attention would refuse is refused before the rows are written
  FC_REQUIRE(q && out && context_lens && workspace, FC_EINVAL, "%s: null pointer", who);
  FC_REQUIRE(workspace_bytes >= fc_decode_attn_workspace_bytes(k_cache->batch, num_q_heads, k_cache->max_seq_len), FC_EINVAL,
             "%s: workspace too small", who);
  if ((rc = fc_store_kv_slots(k_new, k_stride, v_new, v_stride, k_cache->base, v_cache->base, slot_mapping, k_cache->batch,
                              (int32_t)row, k_cache->dtype, stream)))
    return rc;
  return da_enqueue(who, k_cache, v_cache, 0, q, out, num_q_heads, context_lens, scale, workspace, workspace_bytes, stream, nullptr,
                    -1, nullptr, &plan);
}

extern "C" int fc_decode_layer_turn(const fc_kv_view* k_cache, const fc_kv_view* v_cache, const void* q, const void* k_new,
                                    int64_t k_stride, const void* v_new, int64_t v_stride, const int32_t* slot_mapping,
                                    void* out, int32_t num_q_heads, const int32_t* context_lens, float scale,
                                    void* workspace, int64_t workspace_bytes, int32_t turn, void* stream) {
  return da_layer(k_cache, v_cache, q, k_new, k_stride, v_new, v_stride, slot_mapping, out, num_q_heads, context_lens, scale,
                  workspace, workspace_bytes, turn, nullptr, stream);
}

extern "C" int fc_decode_layer_arrivals(const fc_kv_view* k_cache, const fc_kv_view* v_cache, const void* q, const void* k_new,
                                        int64_t k_stride, const void* v_new, int64_t v_stride, const int32_t* slot_mapping,
                                        void* out, int32_t num_q_heads, const int32_t* context_lens, float scale,
                                        void* workspace, int64_t workspace_bytes, uint32_t* arrivals, void* stream) {
  return da_layer(k_cache, v_cache, q, k_new, k_stride, v_new, v_stride, slot_mapping, out, num_q_heads, context_lens, scale,
                  workspace, workspace_bytes, -1, arrivals, stream);
}

// ---- the same attention for callers that cannot allocate -------------------------------------------------
// The chunk partials live in a file-scope device array instead of a caller workspace.  `scratch` below is the
// host-side handle of that array, not a device address: its address on the current device is looked up once
// per device (every GPU holds its own copy) and only that address is ever handed to a kernel.
#define DA_STATIC_BYTES (16ll << 20)
static __device__ __align__(256) unsigned char scratch[DA_STATIC_BYTES];

#define DA_MAX_DEVICES 64
// filled per device on first use; two threads racing here store the same value
static std::atomic<void*> da_scratch_ptr[DA_MAX_DEVICES];
// Every call on a device shares that device's array, so two calls whose kernels overlap (different streams, or a
// graph replay beside an eager call) corrupt each other's chunk partials.  The library cannot see that in general
// without synchronising; with FC_STATIC_GUARD=1 in the environment it checks the one case it can name cheaply: a
// call on another stream than the previous call's while that stream still has work pending is refused.  The check
// queries the previous stream, so leave it off when streams are being captured.
static std::atomic<void*> da_last_stream[DA_MAX_DEVICES];
static std::atomic<int> da_last_stream_set[DA_MAX_DEVICES];
static bool da_guard_enabled() {
  static const bool on = [] {
    const char* e = getenv("FC_STATIC_GUARD");
    return e && e[0] && e[0] != '0';
  }();
  return on;
}

extern "C" int64_t fc_decode_attn_static_capacity(void) { return DA_STATIC_BYTES; }

extern "C" int fc_decode_attn_static(const fc_kv_view* k_cache, const fc_kv_view* v_cache, int32_t layer,
                                     const void* q, void* out, int32_t num_q_heads, const int32_t* context_lens,
                                     float scale, void* stream) {
  const char* who = "fc_decode_attn_static";
  FC_REQUIRE(k_cache && num_q_heads > 0, FC_EINVAL, "%s: null view or bad head count", who);
  const int64_t need = fc_decode_attn_workspace_bytes(k_cache->batch, num_q_heads, k_cache->max_seq_len);
  FC_REQUIRE(need > 0, FC_EINVAL, "%s: bad sizes", who);
  FC_REQUIRE(need <= DA_STATIC_BYTES, FC_EUNSUPPORTED,
             "%s: batch %d x %d query heads x max_seq_len %d needs %lld bytes of chunk partials, the built-in "
             "buffer holds %lld; use fc_decode_attn with a workspace",
             who, k_cache->batch, num_q_heads, k_cache->max_seq_len, (long long)need, (long long)DA_STATIC_BYTES);
  int dev = -1;
  FC_REQUIRE(hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < DA_MAX_DEVICES, FC_EUNSUPPORTED,
             "%s: no current device below %d", who, DA_MAX_DEVICES);
  void* ws = da_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!ws) {
    const hipError_t e = hipGetSymbolAddress(&ws, HIP_SYMBOL(scratch));
    FC_REQUIRE(e == hipSuccess && ws, FC_ELAUNCH, "%s: hipGetSymbolAddress: %s", who, hipGetErrorString(e));
    da_scratch_ptr[dev].store(ws, std::memory_order_release);
  }
  if (da_guard_enabled()) {
    if (da_last_stream_set[dev].load(std::memory_order_acquire)) {
      void* last = da_last_stream[dev].load(std::memory_order_acquire);
      if (last != stream) {
        const hipError_t q = hipStreamQuery((hipStream_t)last);
        if (q != hipSuccess) (void)hipGetLastError();
        FC_REQUIRE(q != hipErrorNotReady, FC_EINVAL,
                   "%s: the previous call on this device used another stream that still has work pending; calls "
                   "that share the built-in buffer must not overlap", who);
      }
    }
    da_last_stream[dev].store(stream, std::memory_order_release);
    da_last_stream_set[dev].store(1, std::memory_order_release);
  }
  return da_enqueue(who, k_cache, v_cache, layer, q, out, num_q_heads, context_lens, scale, ws, DA_STATIC_BYTES,
                    stream);
}
