// CCM compressor: Linear(cf*128 -> 128) -> ReLU -> Linear(128 -> 128) -> ReLU -> Linear(128 -> 128)
// over rows made of `cf` consecutive tokens of one head, fp16/bf16 storage, fp32 accumulation,
// each Linear's output rounded to the storage dtype.  Reads and writes the caches in place.
//
// Shape of the work: one workgroup of 8 wavefronts (two per SIMD, so that one multiplies while
// the other converts, loads or stores) per group of columns of one layer; a column is one sequence's rows of
// 1 << hsh heads that lie side by side, row r being output token r >> hsh of head r % (1 << hsh); a wavefront owns 32
// rows of one column per iteration.  The three GEMMs are transposed
// (features along the accumulator registers, one token per lane) and chained through registers:
//   layer 1  H1^T = W1 * X^T   A = W1 rows from LDS, B = X token rows;
//   layer 2  H2^T = W2 * H1^T  B = layer 1's accumulators, converted in place;
//   layer 3  Y^T  = W3 * H2^T  B = layer 2's accumulators.
// A 32x32 accumulator block holds, per lane, 16 values of one token column; taking registers
// 0..7 and 8..15 as two k-steps gives a complete, if permuted, set of 16 k indices across the two
// half-waves, so the next layer's weights are stored in LDS with the same permutation
// ([0-3, 8-11 | 4-7, 12-15] inside every group of 16) and no data moves between lanes.
//
// Token rows enter and leave in the layout memory likes, not the one the MFMA wants: four adjacent
// lanes read (write) 64 contiguous bytes of a row, 16 rows per instruction, and the 32 rows x 64
// bytes of two k-steps (of one 32-feature block of the output) are re-laid through 2 KB of LDS
// private to the wavefront.  With one row per lane instead, every 16-byte access of an instruction
// falls into a cache line of its own and the vector memory pipeline, not HBM, sets the pace.
//
// W2 and W3 (permuted) stay in LDS for the life of the workgroup; W1 streams through a double
// buffer one 128-column chunk (one source token) at a time, shared by the wavefronts; each
// wavefront prefetches the X rows of the next chunk into registers while it multiplies the current one.
// In-place safety: output token j lands on token dst_start + j <= seg_start + cf*j; all rows of an
// iteration are read before the workgroup barrier that precedes its stores, and later iterations
// read tokens no earlier iteration writes.
#include <math.h>
#include <algorithm>
#include "fc_common.h"

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

#define ML_WAVES 8                  // wavefronts per workgroup (two per SIMD)
#define ML_ROWS 32                  // rows per wavefront and iteration
#define ML_THREADS (ML_WAVES * 64)
#define ML_ROWB 272                 // LDS bytes per weight row: 128 elements + 16 bytes of padding
#define ML_WBYTES (128 * ML_ROWB)   // one 128 x 128 weight block in LDS
#define ML_TBLTOT 768               // block-table entries cached per workgroup and view, divided among its columns
#define ML_XS 2048                  // per-wavefront LDS bytes for re-laying token rows: 32 rows x 64 bytes
#define ML_LDS (4 * ML_WBYTES + 3 * 128 * 4 + 2 * ML_TBLTOT * 4 + ML_WAVES * ML_XS + ML_WAVES * 4)
// Nothing is scheduled across this point.  Without it the compiler, short of registers, sinks every
// prefetch (weight fragments from LDS, token rows from memory) to just before its use and the
// multiplications wait out the full latency each time.
#define ML_PIN() __builtin_amdgcn_sched_barrier(0)

// two fp32 -> packed storage dtype, round to nearest even
template <int DTYPE>
__device__ __forceinline__ unsigned ml_pack2(float a, float b) {
  f32x2 v = {a, b};
  if constexpr (DTYPE == FC_BF16)
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
  else
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, f16x2));
}

template <int DTYPE>
__device__ __forceinline__ float ml_to_float(unsigned short h) {
  return DTYPE == FC_BF16 ? fc_bf16_to_float(h) : fc_half_to_float(h);
}

// relu + round for 8 consecutive accumulator registers (the bias is already in the accumulator)
// -> one MFMA operand.  ReLU before rounding equals rounding before ReLU.
template <int DTYPE>
__device__ __forceinline__ uint4 ml_act_operand(const f32x16& acc, int i0) {
  unsigned p[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    p[e] = ml_pack2<DTYPE>(fmaxf(acc[i0 + 2 * e], 0.f), fmaxf(acc[i0 + 2 * e + 1], 0.f));
  return make_uint4(p[0], p[1], p[2], p[3]);
}

// accumulator block initialised with the bias of its 16 features: register i holds feature
// fb + (i/4)*8 + lhalf*4 + i%4
__device__ __forceinline__ void ml_bias_init(f32x16& acc, const float* __restrict__ bias, int fb, int lhalf) {
#pragma unroll
  for (int i4 = 0; i4 < 4; ++i4) {
    const float4 bv = *reinterpret_cast<const float4*>(bias + fb + i4 * 8 + lhalf * 4);
    acc[i4 * 4 + 0] = bv.x;
    acc[i4 * 4 + 1] = bv.y;
    acc[i4 * 4 + 2] = bv.z;
    acc[i4 * 4 + 3] = bv.w;
  }
}

// orders a wavefront's LDS writes before its following LDS reads of other lanes' data (the hardware executes
// one wavefront's LDS instructions in order; this only keeps the compiler from moving them)
__device__ __forceinline__ void ml_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The sequence whose segment is the rank-th longest (of equal ones the first); more than 256 sequences are taken as they
// come.  Every wavefront works it out for itself: lane i counts the segments ahead of its own.
__device__ __forceinline__ int ml_ranked_sequence(const int* __restrict__ seg_len_v, int batch, int rank) {
  if (batch <= 1 || batch > 256) return rank;
  const int lane = threadIdx.x & 63;
  int found = rank;
  for (int i0 = 0; i0 < batch; i0 += 64) {
    const int i = i0 + lane, own = seg_len_v[min(i, batch - 1)];
    int ahead = 0;
    for (int j0 = 0; j0 < batch; j0 += 64) {
      const int other = seg_len_v[min(j0 + lane, batch - 1)], m = min(64, batch - j0);
      for (int j = 0; j < m; ++j) {
        const int len = __builtin_amdgcn_readlane(other, j);
        ahead += (len > own || (len == own && j0 + j < i)) ? 1 : 0;
      }
    }
    const unsigned long long who = __ballot(i < batch && ahead == rank);
    if (who) found = i0 + __ffsll((long long)who) - 1;
  }
  return __builtin_amdgcn_readfirstlane(found);
}

// SRC_T / DST_T: 0 = dense view (no table), 1 = paged view whose table row fits the LDS cache,
// 2 = paged view read through global memory.
// W1R: all of W1 fits the two LDS chunk buffers (cf <= 2) and is loaded once; otherwise W1 streams
// through them one chunk per stage, which costs a workgroup barrier per chunk.
// RAG: every sequence has its own segment: seg_start_v / seg_len_v / dst_start_v [batch] in device memory; c_rows is
// then the largest row count any sequence can have (it bounds the loops), and a sequence whose segment gives fewer
// than min_rows rows is left to the copy kernel below.
// FLAT (dense views that do not overlap, nothing to keep in order): there are no columns; the c_rows rows of all
// (sequence, head) pairs are one list of `flat.rows` rows, and the workgroups of a (layer, plane) take 256 of them in turn.
// The body works on ONE layer of one plane: `slayer` / `dlayer` and the weight pointers carry the layer already; a
// workgroup takes the column groups cg0, cg0 + cg_step, ... below ncg.
struct MlFlat { unsigned rows; FcDivisor per_pair, heads; };

template <int DTYPE, int SRC_T, int DST_T, bool W1R, bool RAG, bool FLAT = false>
__device__ __forceinline__ void mlp_body(char* lds, const KvView& src, const KvView& dst, const char* slayer, char* dlayer,
                                         const char* __restrict__ w1l, const char* __restrict__ b1l,
                                         const char* __restrict__ w2l, const char* __restrict__ b2l,
                                         const char* __restrict__ w3l, const char* __restrict__ b3l, int cf,
                                         int seg_start, int c_rows, int dst_start, int hsh, int wpc, int ncols, int ncg, int cg0,
                                         int cg_step, const int* __restrict__ seg_start_v,
                                         const int* __restrict__ seg_len_v, const int* __restrict__ dst_start_v,
                                         int min_rows, MlFlat flat = MlFlat{}) {
  char* w1buf = lds;                       // 2 x ML_WBYTES
  char* w2buf = lds + 2 * ML_WBYTES;       // permuted
  char* w3buf = lds + 3 * ML_WBYTES;       // permuted
  float* bias = reinterpret_cast<float*>(lds + 4 * ML_WBYTES);  // [3][128] fp32
  int* tbls = reinterpret_cast<int*>(lds + 4 * ML_WBYTES + 3 * 128 * 4);  // [2 views][columns of the workgroup][tcap]
  char* xsw = lds + 4 * ML_WBYTES + 3 * 128 * 4 + 2 * ML_TBLTOT * 4 + (threadIdx.x >> 6) * ML_XS;
  int* wave_rows = reinterpret_cast<int*>(lds + 4 * ML_WBYTES + 3 * 128 * 4 + 2 * ML_TBLTOT * 4 + ML_WAVES * ML_XS);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int lq = lane >> 2, lp = lane & 3;   // memory-side layout: row lq (and 16 + lq), 16-byte piece lp of 64 bytes
  const int cols_per_wg = ML_WAVES / wpc;
  const int sub = wave % wpc;
  const int hg_per_seq = src.num_kv_heads >> hsh;   // columns of a sequence
  const int K1 = cf * 128;
  // the column this wavefront works on; set per column group
  int col = 0, b = 0, h = 0;
  bool col_ok = false;

  // this column's block-table rows (source and destination), so that no row address waits on a table read;
  // filled by the wavefronts that share the column
  const int tcap = ML_TBLTOT / cols_per_wg;
  int* stbl = tbls + (wave / wpc) * tcap;
  int* dtbl = stbl + ML_TBLTOT;
  // this wavefront's column: first source token, rows, first destination token (the launch's, or the sequence's own)
  int ss = seg_start, cr = c_rows, ds = dst_start;
  auto fill_tables = [&]() {
    // a column without rows still loads (clamped) rows of its first cf tokens: its table covers them
    const int s_last = min(ss + max(cr, 1) * cf, src.max_seq_len) - 1, d_last = ds + cr - 1;
    // also for a wavefront whose column is past the last one (b = 0): its loads are unconditional and need valid addresses
    if (SRC_T == 1)
      for (int i = sub * 64 + lane; i <= (s_last >> src.block_shift); i += 64 * wpc)
        stbl[i] = src.block_tables[(long long)b * src.table_stride + i];
    if (col_ok && DST_T == 1)
      for (int i = sub * 64 + lane; i <= (d_last >> dst.block_shift); i += 64 * wpc)
        dtbl[i] = dst.block_tables[(long long)b * dst.table_stride + i];
  };
  auto src_off = [&](int s) -> long long {
    if (SRC_T == 0) return (long long)b * src.stride_batch + (long long)s * src.stride_token;
    if (SRC_T == 1) {
      const int blk = stbl[s >> src.block_shift];
      return blk < 0 ? -1 : (long long)blk * src.stride_block + (long long)(s & (src.block_size - 1)) * src.stride_token;
    }
    return fc_token_offset(src, b, s);
  };
  auto dst_off = [&](int s) -> long long {
    if (DST_T == 0) return (long long)b * dst.stride_batch + (long long)s * dst.stride_token;
    if (DST_T == 1) {
      const int blk = dtbl[s >> dst.block_shift];
      return blk < 0 ? -1 : (long long)blk * dst.stride_block + (long long)(s & (dst.block_size - 1)) * dst.stride_token;
    }
    return fc_token_offset(dst, b, s);
  };

  // ---- resident weights: W2, W3 with the k permutation, biases as fp32 ------------------------------
  {
    // 8-byte pieces: piece p of a row holds k = 4p .. 4p+3; inside each group of 4 pieces the order
    // becomes [0, 2, 1, 3]
    for (int i = tid; i < 128 * 32; i += ML_THREADS) {
      const int n = i >> 5, p = i & 31;
      const int q = p & 3;
      const int pp = (p & ~3) | ((q == 1) ? 2 : (q == 2) ? 1 : q);
      *reinterpret_cast<uint2*>(w2buf + n * ML_ROWB + pp * 8) = *reinterpret_cast<const uint2*>(w2l + (n * 128 + p * 4) * 2);
      *reinterpret_cast<uint2*>(w3buf + n * ML_ROWB + pp * 8) = *reinterpret_cast<const uint2*>(w3l + (n * 128 + p * 4) * 2);
    }
    for (int i = tid; i < 384; i += ML_THREADS) {
      const int which = i >> 7, n = i & 127;
      const char* bp = which == 0 ? b1l : which == 1 ? b2l : b3l;
      bias[i] = ml_to_float<DTYPE>(*reinterpret_cast<const unsigned short*>(bp + n * 2));
    }
  }

  // W1 chunk kc covers columns [kc*128, kc*128+128) of W1[l]: 2048 pieces of 16 bytes
  constexpr int WCH = 2048 / ML_THREADS;
  u32x4 wpre[WCH];
  auto w1_load = [&](int kc) {
#pragma unroll
    for (int u = 0; u < WCH; ++u) {
      const int ch = tid + u * ML_THREADS;  // row n = ch / 16, part = ch % 16
      wpre[u] = *reinterpret_cast<const u32x4*>(w1l + ((long long)(ch >> 4) * K1 + kc * 128) * 2 + (ch & 15) * 16);
    }
  };
  auto w1_store = [&](int buf) {
#pragma unroll
    for (int u = 0; u < WCH; ++u) {
      const int ch = tid + u * ML_THREADS;
      *reinterpret_cast<u32x4*>(w1buf + buf * ML_WBYTES + (ch >> 4) * ML_ROWB + (ch & 15) * 16) = wpre[u];
    }
  };

  const int rows_per_iter = ML_ROWS * wpc;
  // FLAT: this workgroup's share of the rows, 256 per iteration, the workgroups' turns interleaved
  const int n_flat = FLAT ? ((int)((flat.rows + ML_ROWS * ML_WAVES - 1) / (ML_ROWS * ML_WAVES)) - cg0 + cg_step - 1) / cg_step : 0;
  auto flat_row = [&](int it) { return (unsigned)(it * cg_step + cg0) * (ML_ROWS * ML_WAVES) + wave * ML_ROWS; };
  auto flat_off = [&](const KvView& v, unsigned r, int start, int per, int kc) -> long long {
    const unsigned pr = flat.per_pair.quotient(r), j = r - pr * flat.per_pair.d;
    const unsigned bb = flat.heads.quotient(pr), hh = pr - bb * flat.heads.d;
    return (long long)bb * v.stride_batch + (long long)hh * v.stride_head + (long long)(start + (int)j * per + kc) * v.stride_token;
  };
  int n_iter = FLAT ? n_flat : ((c_rows << hsh) + rows_per_iter - 1) / rows_per_iter;
  int q_total = n_iter * cf;      // W1 chunk q = (iteration q / cf, token kc = q % cf) sits in buffer q & 1
  const char* sbase = nullptr;   // this lane's piece of token 0 of its head, per column group
  char* dbase = nullptr;
  // X rows of chunk q: xf[2*c4 + rh] holds bytes [64*c4 + 16*lp, +16) of the token row of output row 16*rh + lq
  auto x_load = [&](uint4 (&xf)[8], int q) {
    const int it = q / cf, kc = q - it * cf;
    const int row0 = it * rows_per_iter + sub * ML_ROWS;
    // Every lane always loads (no branch around the loads, so that the compiler keeps exact counts of
    // the loads in flight and the prefetch really overlaps the multiplications): rows past the end, a
    // column past the last one (b = h = 0) and unallocated pages read some valid row instead; what is
    // computed from them is never stored.
#pragma unroll
    for (int rh = 0; rh < 2; ++rh) {
      if constexpr (FLAT) {
        const long long off = flat_off(src, min(flat_row(it) + rh * 16 + lq, flat.rows - 1), seg_start, cf, kc);
#pragma unroll
        for (int c4 = 0; c4 < 4; ++c4) xf[c4 * 2 + rh] = *reinterpret_cast<const uint4*>(sbase + off * 2 + c4 * 64);
        continue;
      }
      int r = min((row0 + rh * 16 + lq) >> hsh, cr - 1);
      int tok = ss + cf * r + kc;
      if constexpr (RAG) {   // a column with no rows, or fewer than the launch's bound, reads some valid token
        r = max(r, 0);
        tok = min(ss + cf * r + kc, src.max_seq_len - 1);
      }
      long long off = src_off(tok);
      off = off < 0 ? 0 : off;
#pragma unroll
      for (int c4 = 0; c4 < 4; ++c4) xf[c4 * 2 + rh] = *reinterpret_cast<const uint4*>(sbase + off * 2 + c4 * 64);
    }
  };
  // Re-laying through this wavefront's 2 KB of LDS: rows of 64 bytes, the four 16-byte pieces of a row XOR-ed
  // with a 2-bit function of the row number chosen so that the operand-side accesses (consecutive rows, same
  // piece) touch every bank once whether 8 rows share a 128-byte bank window or 16 rows a 256-byte one:
  // rows r, r+2, r+4, r+6 and rows r, r+4, r+8, r+12 all get different pieces.
  auto piece_swz = [](int r) { return (unsigned)((((r >> 1) ^ (r >> 3)) & 1) | (((r >> 2) & 1) << 1)); };
  const unsigned mem_at = (unsigned)lq * 64 + ((lp ^ piece_swz(lq)) << 4);   // row lq; row 16 + lq is 1024 further
  const unsigned swz = piece_swz(lrow);
  const unsigned op_at0 = (unsigned)lrow * 64 + (((0 + lhalf) ^ swz) << 4);    // k-step 0 of the pair: pieces 0, 1
  const unsigned op_at1 = (unsigned)lrow * 64 + (((2 + lhalf) ^ swz) << 4);    // k-step 1: pieces 2, 3
  auto relay_put = [&](uint4 lo_rows, uint4 hi_rows) {
    *reinterpret_cast<uint4*>(xsw + mem_at) = lo_rows;
    *reinterpret_cast<uint4*>(xsw + mem_at + 1024) = hi_rows;
    ml_wave_sync();
  };
  auto relay_get = [&](int e) { return *reinterpret_cast<const uint4*>(xsw + (e ? op_at1 : op_at0)); };

  f32x16 acc[4];

  // One pipeline stage: chunk q of layer 1 from `xcur` while chunk q+1's rows load into `xnext`;
  // after the last chunk of an iteration, layers 2 and 3 and the stores.
  auto stage = [&](uint4 (&xcur)[8], uint4 (&xnext)[8], int q) {
    const int it = q / cf, kc = q - it * cf;
    // The prefetches are unconditional (straight-line code keeps the staging registers out of
    // scratch memory): past the last chunk the X rows are clamped to valid ones, and the
    // extra W1 chunk lands in the buffer nobody reads again.
    // Of a streamed W1 the next chunk is asked for ahead of the rows: loads arrive in order, and what waits for it at the
    // end of the stage would wait for the rows as well, which have until the next stage.  us per pass, rows first -> W1 first,
    // factor 5: 28 layers of 4 heads, 16 sequences of 16384 tokens 4191 -> 4130, 14 of 3875 to 11626 2113 -> 2048, 4 of 5840
    // 459 -> 449; 32 of 32, 45 of 640 4193 -> 4127.  A list, whose rows any wavefront may fetch at any time, loses (8 prompts
    // of 6000 tokens 783 -> 815).  Rows two chunks ahead, asked for before layers 2 and 3: no more than this, and 1 % less
    // with W1 resident.
    if (FLAT || W1R) x_load(xnext, q + 1);
    if (!W1R) {
      if (FLAT) ML_PIN();
      __syncthreads();  // chunk q is in w1buf[q & 1]; every wavefront is done with chunk q - 1
      w1_load((kc + 1 < cf) ? kc + 1 : 0);
      if (!FLAT) {
        ML_PIN();
        x_load(xnext, q + 1);
      }
    }
    ML_PIN();   // the prefetch stays ahead of this stage's multiplications
    {
      const char* wa = w1buf + (W1R ? kc : (q & 1)) * ML_WBYTES + lrow * ML_ROWB + lhalf * 16;
      uint4 af[2][4];      // weight fragments of k-step ks+1 are read while k-step ks multiplies
      uint4 bop[2][2];     // token operands of two k-steps (64 bytes of every row), re-laid one pair ahead
      relay_put(xcur[0], xcur[1]);
      bop[0][0] = relay_get(0);
      bop[0][1] = relay_get(1);
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) af[0][mb] = *reinterpret_cast<const uint4*>(wa + mb * 32 * ML_ROWB);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        if ((ks & 1) == 0 && ks + 2 < 8) {
          relay_put(xcur[ks + 2], xcur[ks + 3]);
          bop[((ks >> 1) + 1) & 1][0] = relay_get(0);
          bop[((ks >> 1) + 1) & 1][1] = relay_get(1);
        }
        if (ks + 1 < 8) {
#pragma unroll
          for (int mb = 0; mb < 4; ++mb)
            af[(ks + 1) & 1][mb] = *reinterpret_cast<const uint4*>(wa + mb * 32 * ML_ROWB + (ks + 1) * 32);
        }
        ML_PIN();   // the reads of the next k-step are issued before this k-step's multiplications
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) acc[mb] = fc_mfma<DTYPE>(af[ks & 1][mb], bop[(ks >> 1) & 1][ks & 1], acc[mb]);
        ML_PIN();
      }
    }
    if (!W1R) w1_store((q + 1) & 1);
    if (kc != cf - 1) return;

    // ---- layers 2 and 3: H^T = W * (previous H)^T, B operand taken from the previous layer's accumulators ----
    uint4 hf[8];
#pragma unroll
    for (int layer = 1; layer < 3; ++layer) {
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        hf[2 * mb] = ml_act_operand<DTYPE>(acc[mb], 0);
        hf[2 * mb + 1] = ml_act_operand<DTYPE>(acc[mb], 8);
        ml_bias_init(acc[mb], bias + layer * 128, mb * 32, lhalf);
      }
      const char* wa = (layer == 1 ? w2buf : w3buf) + lrow * ML_ROWB + lhalf * 16;
      uint4 af[2][4];
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) af[0][mb] = *reinterpret_cast<const uint4*>(wa + mb * 32 * ML_ROWB);
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        if (g + 1 < 8) {
#pragma unroll
          for (int mb = 0; mb < 4; ++mb)
            af[(g + 1) & 1][mb] = *reinterpret_cast<const uint4*>(wa + mb * 32 * ML_ROWB + (g + 1) * 32);
        }
        ML_PIN();
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) acc[mb] = fc_mfma<DTYPE>(af[g & 1][mb], hf[g], acc[mb]);
        ML_PIN();
      }
    }
    // every wavefront of the column has consumed this iteration's source rows: stores may alias them
    // (a wavefront that owns its column alone is ordered by its own data dependences)
    if (!FLAT && wpc > 1) __syncthreads();
    {
      // The lane owns output row lrow and, per 32-feature block, features (i/4)*8 + lhalf*4 + i%4: four 8-byte
      // pieces go to the wavefront's LDS rows (64 bytes = one feature block of a row); read back in the
      // memory-side layout, 16 rows x 64 bytes leave per store instruction.
      const int row0 = it * rows_per_iter + sub * ML_ROWS;
      char* rowp[2];
#pragma unroll
      for (int rh = 0; rh < 2; ++rh) {
        const int r = (row0 + rh * 16 + lq) >> hsh;
        long long off = -1;
        if constexpr (FLAT) {
          const unsigned fr = flat_row(it) + rh * 16 + lq;
          if (fr < flat.rows) off = flat_off(dst, fr, dst_start, 1, 0);
        } else if (col_ok && r < cr) {
          off = dst_off(ds + r);
        }
        rowp[rh] = off >= 0 ? dbase + off * 2 : nullptr;
      }
      // (a half-wave writes one 8-byte half per row, so rows that share a piece position in a bank window keep
      // their halves swapped: bit 3 xor bit 4 of the row number)
      const unsigned y_at = (unsigned)lrow * 64 + (((lhalf ^ (lrow >> 3) ^ (lrow >> 4)) & 1) << 3);
      const bool swap0 = (lq >> 3) & 1;     // row lq has its halves swapped; row 16 + lq the opposite
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          uint2 w;
          w.x = ml_pack2<DTYPE>(acc[mb][i4 * 4 + 0], acc[mb][i4 * 4 + 1]);
          w.y = ml_pack2<DTYPE>(acc[mb][i4 * 4 + 2], acc[mb][i4 * 4 + 3]);
          *reinterpret_cast<uint2*>(xsw + y_at + ((i4 ^ swz) << 4)) = w;
        }
        ml_wave_sync();
        const uint4 y0 = *reinterpret_cast<const uint4*>(xsw + mem_at);
        const uint4 y1 = *reinterpret_cast<const uint4*>(xsw + mem_at + 1024);
        if (rowp[0])
          *reinterpret_cast<uint4*>(rowp[0] + mb * 64) = swap0 ? make_uint4(y0.z, y0.w, y0.x, y0.y) : y0;
        if (rowp[1])
          *reinterpret_cast<uint4*>(rowp[1] + mb * 64) = swap0 ? y1 : make_uint4(y1.z, y1.w, y1.x, y1.y);
      }
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) ml_bias_init(acc[mb], bias, mb * 32, lhalf);
  };

  uint4 xa[8], xb[8];
  if (W1R) {
    w1_load(0);
    w1_store(0);
    if (cf > 1) {
      w1_load(1);
      w1_store(1);
    }
  }
  for (int cg = cg0; cg < ncg; cg += cg_step) {
    if (cg != cg0) __syncthreads();   // every wavefront is done with the previous group's tables and W1 buffers
    col = cg * cols_per_wg + wave / wpc;
    col_ok = FLAT || col < ncols;
    b = col_ok ? col / hg_per_seq : 0;
    h = col_ok ? (col - b * hg_per_seq) << hsh : 0;
    if constexpr (RAG) b = ml_ranked_sequence(seg_len_v, src.batch, b);
    // a lane's two rows on the memory side are rows lq and 16 + lq of every 32, of one and the same head
    if constexpr (FLAT) b = h = 0;
    sbase = slayer + (long long)(h + (lq & ((1 << hsh) - 1))) * src.stride_head * 2 + lp * 16;
    dbase = dlayer + (long long)(h + (lq & ((1 << hsh) - 1))) * dst.stride_head * 2 + lp * 16;
    if constexpr (RAG) {
      // The sequence's own segment.  Numbers from device memory are cut to what the host validated: the views'
      // max_seq_len (which their block tables cover) and the launch's row bound.
      ss = min(max(__builtin_amdgcn_readfirstlane(seg_start_v[b]), 0), src.max_seq_len);
      const int sl = min(max(__builtin_amdgcn_readfirstlane(seg_len_v[b]), 0), src.max_seq_len - ss);
      ds = min(max(__builtin_amdgcn_readfirstlane(dst_start_v[b]), 0), dst.max_seq_len);
      cr = sl / cf;
      if (cr < min_rows || !col_ok) cr = 0;
      cr = min(min(cr, c_rows), dst.max_seq_len - ds);
      if (lane == 0) wave_rows[wave] = cr;
    }
    if (!FLAT) fill_tables();
    if (!W1R) {
      w1_load(0);
      w1_store(0);
    }
    __syncthreads();   // block tables, biases and the first weights are in LDS
    if constexpr (RAG) {   // the workgroup walks as many iterations as its longest column needs
      int most = 0;
#pragma unroll
      for (int w = 0; w < ML_WAVES; ++w) most = max(most, wave_rows[w]);
      n_iter = ((most << hsh) + rows_per_iter - 1) / rows_per_iter;
      q_total = n_iter * cf;
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) ml_bias_init(acc[mb], bias, mb * 32, lhalf);
    x_load(xa, 0);
    for (int q = 0; q < q_total; q += 2) {
      stage(xa, xb, q);
      if (q + 1 < q_total) stage(xb, xa, q + 1);
    }
    // the streaming variant is launched with one column group per workgroup (its groups are long, and the
    // loop would cost it registers it does not have)
    if (!W1R || FLAT) break;
  }
}

// K and V of a cache: the same geometry at two places, each with weights of its own (one plane: the first of each).  Both in
// one launch: of few columns a plane alone leaves compute units idle, and every launch ends with some idle.  us per pass of a
// runner, a launch per plane -> one, 28 layers of 4 heads: factor 5, one sequence of 2705 tokens 148 -> 122, 4 of 5840
// 490 -> 463, 14 of 3875 to 11626 2342 -> 2189; factor 2, 14 of 3685 to 11056 2257 -> 2193; 32 layers of 32 heads, image of
// 576: factor 5, 8 of 607 940 -> 823, factor 2, 9 of 590 to 657 1129 -> 1034, 45 of 640 and 24 of 590 to 1158 the same.
struct MlPlanes {
  char* src[2];
  char* dst[2];
  const char* w[2][6];     // w1, b1, w2, b2, w3, b3, all layers stacked
};

// blockIdx.y = plane x layers + layer
template <int DTYPE, int SRC_T, int DST_T, bool W1R, bool RAG>
__global__ __launch_bounds__(ML_THREADS, ML_WAVES / 4) void mlp_kernel(KvView src, KvView dst, MlPlanes a, int cf, int seg_start,
                                                            int c_rows, int dst_start, int hsh, int wpc, int ncols, int ncg,
                                                            const int* __restrict__ seg_start_v,
                                                            const int* __restrict__ seg_len_v,
                                                            const int* __restrict__ dst_start_v, int min_rows) {
  extern __shared__ __align__(16) char lds[];
  int pl = blockIdx.y;
  int group = blockIdx.x;
  if constexpr (RAG) {   // one workgroup per group of columns, the longest sequences' groups of all layers first
    const unsigned id = blockIdx.x + gridDim.x * blockIdx.y;
    group = (int)(id / gridDim.y);
    pl = (int)(id - (unsigned)group * gridDim.y);
  }
  const int p = pl >= src.num_layers;
  const long long l = pl - (p ? src.num_layers : 0);
  mlp_body<DTYPE, SRC_T, DST_T, W1R, RAG>(
      lds, src, dst, a.src[p] + l * src.stride_layer * 2, a.dst[p] + l * dst.stride_layer * 2, a.w[p][0] + l * 128 * cf * 256,
      a.w[p][1] + l * 256, a.w[p][2] + l * 128 * 256, a.w[p][3] + l * 256, a.w[p][4] + l * 128 * 256, a.w[p][5] + l * 256, cf,
      seg_start, c_rows, dst_start, hsh, wpc, ncols, ncg, group, gridDim.x, seg_start_v, seg_len_v, dst_start_v, min_rows);
}

// ---- a list of per-layer tensors, both planes and every segment in ONE launch ---------------------------------
// A HuggingFace cache is a list of (K, V) tensors, one pair per layer; one prompt of it is little work per tensor (32
// columns of 288 rows: 12 us of kernel), so what a launch per (layer, plane, segment) costs is the launches.  The
// addresses travel in the kernel's arguments (no table upload).  blockIdx.y = (segment, plane, layer).  Source and destination
// are different tensors, so nothing has to be ordered: the rows of all columns are one list (FLAT), which leaves no
// wavefront without rows but in the last turn, needs no barrier at the stores and has neighbouring workgroups at
// neighbouring rows; the remainder rows of a segment (or all rows of one too short to compress) are copied behind its
// compressed rows by the same workgroups.  Bound by memory, at 4.4 to 5.1 TB/s.  us per forward, columns of a head each, split
// over wavefronts and walked in groups -> this: 32 layers of 32 heads, factor 2, 2 prompts of 576 + 100 tokens 257 -> 249, 4 of
// 576 + 47 453 -> 439, 8 of 576 + 1500 2836 -> 2808, one of 576 + 47 127 both; factor 5, 3 of 576 + 1000 753 -> 704; 28 layers of
// 4 heads, factor 2, 2 of 3000 129 -> 124, 8 of 6000 920 -> 900; factor 5 the same.
#define ML_LIST_LAYERS 64
#define ML_LIST_SEGS 2
struct MlpList {
  const char* src[2][ML_LIST_LAYERS];           // [plane][layer]
  char* dst[2][ML_LIST_LAYERS];
  const char* w[ML_LIST_SEGS][2][6];            // [segment][plane]: w1, b1, w2, b2, w3, b3, all layers stacked
  int seg_start[ML_LIST_SEGS], c_rows[ML_LIST_SEGS], rem[ML_LIST_SEGS], dst_start[ML_LIST_SEGS];
  int gx[ML_LIST_SEGS];
  MlFlat flat[ML_LIST_SEGS];
};

template <int DTYPE, bool W1R>
__global__ __launch_bounds__(ML_THREADS, ML_WAVES / 4) void mlp_list_kernel(KvView ksrc, KvView vsrc, KvView kdst, KvView vdst,
                                                                           MlpList a, int cf, int ncols) {
  extern __shared__ __align__(16) char lds[];
  const int L = ksrc.num_layers;
  const int job = (int)blockIdx.y / L, l = (int)blockIdx.y - job * L;
  const int seg = job >> 1, p = job & 1;
  const int gx = a.gx[seg];
  if ((int)blockIdx.x >= gx) return;
  const KvView& src = p ? vsrc : ksrc;
  const KvView& dst = p ? vdst : kdst;
  const char* slayer = a.src[p][l];
  char* dlayer = a.dst[p][l];
  const int c = a.c_rows[seg];
  const long long ll = l;
  if (c > 0)
    mlp_body<DTYPE, 0, 0, W1R, false, true>(lds, src, dst, slayer, dlayer, a.w[seg][p][0] + ll * 128 * cf * 256,
                                            a.w[seg][p][1] + ll * 256, a.w[seg][p][2] + ll * 128 * 256, a.w[seg][p][3] + ll * 256,
                                            a.w[seg][p][4] + ll * 128 * 256, a.w[seg][p][5] + ll * 256, cf, a.seg_start[seg], c,
                                            a.dst_start[seg], 0, 1, ncols, 0x7fffffff, blockIdx.x, gx, nullptr, nullptr, nullptr, 0,
                                            a.flat[seg]);
  const int rem = a.rem[seg];
  if (rem > 0) {   // 16 lanes per row
    const int sub = threadIdx.x & 15, s0 = a.seg_start[seg] + c * cf, d0 = a.dst_start[seg] + c;
    for (int i = (int)blockIdx.x * (ML_THREADS / 16) + (threadIdx.x >> 4); i < ncols * rem; i += gx * (ML_THREADS / 16)) {
      const int col = i / rem, t = i - col * rem;
      const int b = col / src.num_kv_heads, h = col - b * src.num_kv_heads;
      const long long so = (long long)b * src.stride_batch + (long long)h * src.stride_head + (long long)(s0 + t) * src.stride_token;
      const long long dof = (long long)b * dst.stride_batch + (long long)h * dst.stride_head + (long long)(d0 + t) * dst.stride_token;
      *reinterpret_cast<uint4*>(dlayer + dof * 2 + sub * 16) = *reinterpret_cast<const uint4*>(slayer + so * 2 + sub * 16);
    }
  }
}

// What the MLP leaves of a segment (the launch's, or with the arrays each sequence's own): the seg_len % cf remainder tokens, or
// the whole segment of a sequence too short to compress, copied to their place behind the compressed rows.  One workgroup per
// (sequence, plane and layer) and heads_per_wg heads, whose rows are one list, tokens ascending; ML_TAIL rows per pass, all
// loaded before any is stored (destination token <= source token).  A workgroup per head is mostly the starting of workgroups
// where a head has a row or two, all heads in one workgroup a chain of passes where it has many, each a table read, a barrier
// and a memory latency: ML_TAIL_ROWS rows a workgroup, in powers of two of heads (3 heads of 18 tokens 36, 4 33, 8 sequences) and
// two heads at least.  us, 32 heads x 64 layers and planes, a workgroup per head / like this / 32 heads in one: 1 token of 1
// sequence 6.2 / 3.2 / 3.1, of 24 58 / 7.0 / 7.0; 4 tokens 6.4 / 4.1 / 5.0, 62 / 26 / 27; 18 8.5 / 6.3 / 14, 129 / 107 / 108;
// 60 19 / 14 / 50, 316 / 312 / 344; 130 32 / 25 / 102, 666 / 674 / 734; 200 43 / 34 / 155, 1007 / 1004 / 1115; 4 heads, 200 tokens
// of 1 sequence 18 / 11 / 19.  (Several rows per thread lose: the table reads of a thread's rows wait for each other, 10 to
// 20 us.)
#define ML_TAIL 32
#define ML_TAIL_ROWS 64
__global__ __launch_bounds__(16 * ML_TAIL) void mlp_tail_copy_kernel(KvView src, KvView dst, MlPlanes a, int cf, int min_rows, int c_max,
                                                            const int* __restrict__ seg_start_v,
                                                            const int* __restrict__ seg_len_v,
                                                            const int* __restrict__ dst_start_v, int seg_start, int seg_len,
                                                            int dst_start, int same_place, int heads_per_wg) {
  const int h0 = blockIdx.x * heads_per_wg, heads = min(heads_per_wg, src.num_kv_heads - h0);
  const int b = blockIdx.y, p = (int)blockIdx.z >= src.num_layers, l = (int)blockIdx.z - (p ? src.num_layers : 0);
  const int ss = min(max(seg_start_v ? seg_start_v[b] : seg_start, 0), src.max_seq_len);
  const int sl = min(max(seg_len_v ? seg_len_v[b] : seg_len, 0), src.max_seq_len - ss);
  const int ds = min(max(dst_start_v ? dst_start_v[b] : dst_start, 0), dst.max_seq_len);
  int c = sl / cf;
  if (c < min_rows) c = 0;
  c = min(min(c, c_max), dst.max_seq_len - ds);
  const int s0 = ss + c * cf, d0 = ds + c;
  const int cnt = min(sl - c * cf, dst.max_seq_len - d0);
  if (cnt <= 0 || (same_place && s0 == d0)) return;
  const int sub = threadIdx.x & 15, tr = threadIdx.x >> 4;
  const char* sb = a.src[p] + (long long)l * src.stride_layer * 2 + sub * 16;
  char* db = a.dst[p] + (long long)l * dst.stride_layer * 2 + sub * 16;
  const unsigned rows = (unsigned)cnt * heads;
  for (unsigned i0 = 0; i0 < rows; i0 += ML_TAIL) {
    const unsigned i = i0 + tr, t = i / heads;
    uint4 row = make_uint4(0, 0, 0, 0);
    long long so = -1, dof = -1, h = h0 + (int)(i - t * heads);
    if (i < rows) {
      so = fc_token_offset(src, b, s0 + (int)t);
      dof = fc_token_offset(dst, b, d0 + (int)t);
    }
    if (so >= 0) row = *reinterpret_cast<const uint4*>(sb + (so + h * src.stride_head) * 2);
    __syncthreads();
    if (so >= 0 && dof >= 0) *reinterpret_cast<uint4*>(db + (dof + h * dst.stride_head) * 2) = row;
  }
}

extern "C" int fc_copy_tokens(const fc_kv_view* src, const fc_kv_view* dst, int32_t seg_start, int32_t count,
                              int32_t dst_start, void* stream);

static int ml_check(const char* who, const fc_kv_view* src, const fc_kv_view* dst, const fc_mlp_weights* w, int cf) {
  int rc;
  if ((rc = fc_check_view(src, who)) || (rc = fc_check_view(dst, who))) return rc;
  FC_REQUIRE(src->dtype == dst->dtype && src->num_layers == dst->num_layers && src->batch == dst->batch &&
                 src->num_kv_heads == dst->num_kv_heads,
             FC_EINVAL, "%s: source and destination views disagree", who);
  FC_REQUIRE(src->dtype == FC_F16 || src->dtype == FC_BF16, FC_EUNSUPPORTED, "%s: fp16/bf16 caches only", who);
  FC_REQUIRE(w && w->w1 && w->b1 && w->w2 && w->b2 && w->w3 && w->b3, FC_EINVAL, "%s: null weights", who);
  FC_REQUIRE(cf >= 1 && cf <= 64, FC_EINVAL, "%s: compression factor %d out of range", who, cf);
  return FC_OK;
}

// How many heads make a column (1 << hsh), how many wavefronts share one, and how many workgroups of a (layer, plane) walk
// its column groups.  One workgroup fills a compute unit (its LDS), so what counts is rounds of workgroups times iterations
// of each, plus the start: loading the weights, about 0.4 of an iteration, 0.7 with resident W1, whose workgroups may walk
// several groups for one start and lose 0.25 between two of them (tables, first rows).  The launch is bound by memory: seven
// eighths of the compute units keep it as busy as all of them, so a last round that is not full costs what it holds, but no
// less than 0.85.  Of equal splits the one with fewer wavefronts per column, which wait for each other at every store.
// Heads in one column make columns of more rows, so that fewer rows of the last iteration are idle and fewer groups are
// walked; what a wavefront reads and writes is a contiguous piece of the page whichever way.  us per launch, one head
// per column -> this split: 32 layers of 32 heads, factor 2, 45 sequences of 576 tokens 2080 -> 2017, of 64 322 -> 287;
// 3 of 576 178 -> 158, of 64 36 -> 30; factor 5, 20 of 576 886 -> 863, of 524 855 -> 769; 28 layers of 4 heads, factor 5,
// 16 of 16384 2090 -> 2050, of 700 114 -> 113; factor 2, 16 of 8000 1271 -> 1153.
//
// Sequences of different lengths (`rag`): a workgroup takes one group, the longest sequences' groups start first, and the
// compute units are busy until about half a group's time before the end; no split ends before its longest column does.
// Lengths are on the device: columns are taken to be two thirds of the longest on average (a third to the whole of it).
// Of equal splits the one with more heads per column.  us per launch, as many wavefronts as make 1024 workgroups in the
// order of the batch -> this: 28 layers of 4 heads, factor 5, 16 sequences of 5461 to 16384 tokens 1680 -> 1455, 5 of 2666
// to 8000 331 -> 284, 9 of 700 to 2100 163 -> 131, 16 of 300 to 900 164 -> 125; factor 2, 16 of 3000 to 9000 1342 -> 920, 16 of
// 300 to 900 158 -> 120; 32 layers of 32 heads, factor 5, 20 of 14 to 824 870 -> 658, factor 2 854 -> 793.
struct MlSplit { int hsh, wpc, gx; double cost; };   // cost in iterations
template <typename Fits>
static MlSplit ml_split(int batch, int heads, int max_hsh, int jobs, int c, int cf, bool rag, Fits fits) {
  const double ncu = fc_compute_units();
  MlSplit best{0, ML_WAVES, batch * heads, 0.0};      // what is left when no split fits
  double best_cost = -1.0;
  for (int i = 0; i <= max_hsh; ++i) {
    const int hsh = rag ? max_hsh - i : i;
    const int per_seq = heads >> hsh, ncols = batch * per_seq;
    const int64_t rows = (int64_t)c << hsh;
    for (int wpc = 1; wpc <= ML_WAVES && (wpc == 1 || ML_ROWS * wpc < 2 * rows); wpc *= 2) {
      if (!fits(wpc)) continue;
      const int cpw = ML_WAVES / wpc, groups = (ncols + cpw - 1) / cpw;
      const double most = (double)((rows + ML_ROWS * wpc - 1) / (ML_ROWS * wpc));
      const double iters = rag ? 0.67 * (double)rows / (ML_ROWS * wpc) + 0.5 : most;
      int last = 0;
      for (int per = 1; per <= groups && per <= (cf <= 2 && !rag ? 64 : 1); ++per) {   // groups a workgroup walks
        const int g = (groups + per - 1) / per;
        if (g == last) continue;
        last = g;
        const double wgs = (double)g * jobs / ncu, whole = (double)(int64_t)wgs, part = wgs - whole;
        const double one = cf <= 2 ? (double)((groups + g - 1) / g) * (iters + 0.25) + 0.7 : iters + 0.4;
        const double rounds = whole + (part <= 0.0 ? 0.0 : part > 0.85 ? part : 0.85);
        const double cost = !rag ? rounds * one : fmax(one - iters + most, wgs * one + 0.5 * iters);
        if (best_cost < 0 || cost < best_cost) {
          best_cost = cost;
          best = {hsh, wpc, g, cost};
        }
      }
    }
  }
  return best;
}

// The MLP launch for c > 0 rows per column: c rows for every sequence from (seg_start, dst_start), or, with the
// three arrays, every sequence's own segment with at most c rows.  `a`: the planes, in views of src's and dst's geometry.
static int ml_launch(const char* who, const fc_kv_view* src, const fc_kv_view* dst, const MlPlanes& a, int planes, int cf,
                     int seg_start, int c, int dst_start, const int32_t* seg_start_v, const int32_t* seg_len_v,
                     const int32_t* dst_start_v, int min_rows, hipStream_t st, const MlSplit* given = nullptr) {
  const bool rag = seg_len_v != nullptr;
  // heads whose rows of a token lie side by side, in both views, may share a column, up to 16 (a lane's two rows of every
  // 32 are then of one head; 32 heads to a column were never the faster split)
  int max_hsh = 0;
  if (src->stride_head < src->stride_token && dst->stride_head < dst->stride_token)
    while (max_hsh < 4 && src->num_kv_heads % (2 << max_hsh) == 0 && c < (1 << 29) >> max_hsh) ++max_hsh;
  const auto tables_fit = [&](int wpc_) {     // in LDS, else every row waits for its entry
    const int cap = ML_TBLTOT / (ML_WAVES / wpc_);
    const auto fit = [&](const fc_kv_view* v, int64_t last) { return !v->block_tables || v->block_size <= 0 || last / v->block_size < cap; };
    return rag ? fit(src, src->max_seq_len - 1) && fit(dst, dst->max_seq_len - 1)
               : fit(src, (int64_t)seg_start + (int64_t)c * cf - 1) && fit(dst, (int64_t)dst_start + c - 1);
  };
  const MlSplit sp = given ? *given : ml_split(src->batch, src->num_kv_heads, max_hsh, planes * src->num_layers, c, cf, rag, tables_fit);
  // Workgroups with resident W1 walk many columns each, and both planes' at a time are up to 3 % slower than one plane's after
  // the other: together only where that saves 1.6 % of the iterations.  us per pass, together / a launch per plane, factor 2,
  // saving: 32 layers of 32 heads, 24 of 640 tokens (0.7 %) 2639 / 2619, 45 4970 / 4927, 9 (12 %) 1049 / 1113; 28 of 4, 8 of
  // 8000 (1.5 %) 1301 / 1262, 16 of 16384 (0.2 %) 4872 / 4837, 2 of 8000 (2.9 %) 353 / 384.  Factor 5, 45 of 640 4269 / 4297,
  // 16 of 16384 4197 / 4252, 9 of 640 991 / 1059; different lengths, factor 2, 8 of 2666 to 8000 972 / 1035, 16 of 5461 to
  // 16384 3397 / 3399.
  if (planes == 2 && !rag && cf <= 2) {
    const MlSplit one = ml_split(src->batch, src->num_kv_heads, max_hsh, src->num_layers, c, cf, false, tables_fit);
    if (2.0 * one.cost < 1.016 * sp.cost) {
      MlPlanes v{};
      v.src[0] = a.src[1];
      v.dst[0] = a.dst[1];
      for (int i = 0; i < 6; ++i) v.w[0][i] = a.w[1][i];
      int rc = ml_launch(who, src, dst, a, 1, cf, seg_start, c, dst_start, nullptr, nullptr, nullptr, min_rows, st, &one);
      return rc ? rc : ml_launch(who, src, dst, v, 1, cf, seg_start, c, dst_start, nullptr, nullptr, nullptr, min_rows, st, &one);
    }
  }
  const int hsh = sp.hsh, wpc = sp.wpc, gx = sp.gx;
  const int ncols = src->batch * (src->num_kv_heads >> hsh);
  const int cols_per_wg = ML_WAVES / wpc, ncg = (ncols + cols_per_wg - 1) / cols_per_wg;
  dim3 grid(gx, planes * src->num_layers);
  const size_t lds = ML_LDS;
  KvView s = fc_make_view(src), d = fc_make_view(dst);
  auto table_mode = [&](const KvView& v, int last_token) {
    if (!v.block_tables) return 0;
    return (v.block_shift >= 0 && (last_token >> v.block_shift) < ML_TBLTOT / cols_per_wg) ? 1 : 2;
  };
  // ragged segments may end anywhere inside the views
  const int sm = table_mode(s, rag ? src->max_seq_len - 1 : seg_start + c * cf - 1);
  const int dm = table_mode(d, rag ? dst->max_seq_len - 1 : dst_start + c - 1);
  // dense/dense, LDS-cached tables, or the general path through global tables (which also serves dense views)
  int mode = (sm == 0 && dm == 0) ? 0 : (sm == 1 && dm == 1) ? 1 : (sm == 0 && dm == 1) ? 2 : (sm == 1 && dm == 0) ? 3 : 4;
  if (rag && mode != 1) mode = 4;
#define ML_LAUNCH(DT, ST, DTT, WR, RG)                                                                                 \
  do {                                                                                                             \
    FC_ALLOW_LDS((mlp_kernel<DT, ST, DTT, WR, RG>), (int)lds);                                                    \
    hipLaunchKernelGGL((mlp_kernel<DT, ST, DTT, WR, RG>), grid, dim3(ML_THREADS), lds, st, s, d, a, cf, seg_start, c, \
                       dst_start, hsh, wpc, ncols, ncg, seg_start_v, seg_len_v, dst_start_v, min_rows);            \
  } while (0)
#define ML_DISPATCH(DT, WR)                                                         \
  if (rag) {                                                                        \
    if (mode == 1) ML_LAUNCH(DT, 1, 1, WR, true); else ML_LAUNCH(DT, 2, 2, WR, true); \
  } else switch (mode) {                                                            \
    case 0: ML_LAUNCH(DT, 0, 0, WR, false); break;                                  \
    case 1: ML_LAUNCH(DT, 1, 1, WR, false); break;                                  \
    case 2: ML_LAUNCH(DT, 0, 1, WR, false); break;                                  \
    case 3: ML_LAUNCH(DT, 1, 0, WR, false); break;                                  \
    default: ML_LAUNCH(DT, 2, 2, WR, false); break;                                 \
  }
  if (src->dtype == FC_BF16) {
    if (cf <= 2) { ML_DISPATCH(FC_BF16, true) } else { ML_DISPATCH(FC_BF16, false) }
  } else {
    if (cf <= 2) { ML_DISPATCH(FC_F16, true) } else { ML_DISPATCH(FC_F16, false) }
  }
#undef ML_DISPATCH
#undef ML_LAUNCH
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}

// One or two planes of one geometry (strides, tables, lengths), each with weights of its own.
static int ml_planes(const char* who, const fc_kv_view* const src[2], const fc_kv_view* const dst[2], const fc_mlp_weights* w,
                     int planes, int cf, MlPlanes& a) {
  int rc;
  for (int p = 0; p < planes; ++p) {
    if ((rc = ml_check(who, src[p], dst[p], w ? w + p : nullptr, cf))) return rc;
    for (const fc_kv_view* const* v : {src, dst}) {
      const fc_kv_view& moved = *v[p];
      FC_REQUIRE(moved.block_tables == v[0]->block_tables && moved.dtype == v[0]->dtype &&
                     moved.num_layers == v[0]->num_layers && moved.batch == v[0]->batch &&
                     moved.num_kv_heads == v[0]->num_kv_heads && moved.max_seq_len == v[0]->max_seq_len &&
                     moved.stride_layer == v[0]->stride_layer && moved.stride_block == v[0]->stride_block &&
                     moved.stride_batch == v[0]->stride_batch && moved.stride_token == v[0]->stride_token &&
                     moved.stride_head == v[0]->stride_head && moved.block_size == v[0]->block_size &&
                     moved.table_stride == v[0]->table_stride,
                 FC_EINVAL, "%s: the planes' views differ in more than their place", who);
    }
    a.src[p] = (char*)src[p]->base;
    a.dst[p] = (char*)dst[p]->base;
    const void* ws[6] = {w[p].w1, w[p].b1, w[p].w2, w[p].b2, w[p].w3, w[p].b3};
    for (int i = 0; i < 6; ++i) a.w[p][i] = (const char*)ws[i];
  }
  FC_REQUIRE(planes * src[0]->num_layers <= 65535, FC_EUNSUPPORTED, "%s: too many layers", who);
  return FC_OK;
}

// remainders and pass-through segments (of the arrays' segments seg_len is the longest); nothing to move when a pass-through
// segment already lies at its place
static void ml_tails(const fc_kv_view* const src[2], const fc_kv_view* const dst[2], const MlPlanes& a, int planes, int cf,
                     int min_rows, int c, const int32_t* seg_start_v, const int32_t* seg_len_v, const int32_t* dst_start_v,
                     int seg_start, int seg_len, int dst_start, hipStream_t st) {
  int same = 1;
  for (int p = 0; p < planes; ++p)
    same = same && src[p]->base == dst[p]->base && src[p]->block_tables == dst[p]->block_tables &&
           src[p]->stride_layer == dst[p]->stride_layer && src[p]->stride_batch == dst[p]->stride_batch;
  // what a sequence leaves at most: a remainder, or a segment of too few rows
  const int64_t most = seg_len_v ? std::min<int64_t>(seg_len, std::max<int64_t>(min_rows, 1) * cf - 1) : seg_len - (int64_t)c * cf;
  int want = 2;
  while (want < 32 && want * most < ML_TAIL_ROWS) want *= 2;
  const int heads = src[0]->num_kv_heads, per = heads < want ? heads : want;
  hipLaunchKernelGGL(mlp_tail_copy_kernel, dim3((heads + per - 1) / per, src[0]->batch, planes * src[0]->num_layers),
                     dim3(16 * ML_TAIL), 0, st, fc_make_view(src[0]), fc_make_view(dst[0]), a, cf, min_rows, c, seg_start_v, seg_len_v, dst_start_v,
                     seg_start, seg_len, dst_start, same, per);
}

static int ml_uniform(const char* who, const fc_kv_view* const src[2], const fc_kv_view* const dst[2], const fc_mlp_weights* w,
                      int planes, int cf, int seg_start, int seg_len, int dst_start, void* stream) {
  MlPlanes a{};
  int rc = ml_planes(who, src, dst, w, planes, cf, a);
  if (rc) return rc;
  FC_REQUIRE(seg_start >= 0 && seg_len >= 0 && dst_start >= 0, FC_EINVAL, "%s: negative range", who);
  FC_REQUIRE((int64_t)seg_start + seg_len <= src[0]->max_seq_len, FC_EINVAL,
             "%s: segment [%d, %d) exceeds the source view's max_seq_len %d", who, seg_start, seg_start + seg_len,
             src[0]->max_seq_len);
  const int c = seg_len / cf;
  const int rem = seg_len - c * cf;
  FC_REQUIRE((int64_t)dst_start + c + rem <= dst[0]->max_seq_len, FC_EINVAL,
             "%s: output [%d, %d) exceeds the destination view's max_seq_len %d", who, dst_start,
             dst_start + c + rem, dst[0]->max_seq_len);
  if (c > 0 && (rc = ml_launch(who, src[0], dst[0], a, planes, cf, seg_start, c, dst_start, nullptr, nullptr, nullptr, 0,
                               (hipStream_t)stream)))
    return rc;
  if (rem > 0 && (planes == 1 || src[0]->batch > 65535)) {     // (more sequences than the tails' grid takes)
    for (int p = 0; p < planes && !rc; ++p) rc = fc_copy_tokens(src[p], dst[p], seg_start + c * cf, rem, dst_start + c, stream);
    return rc;
  }
  if (rem > 0) ml_tails(src, dst, a, planes, cf, 0, c, nullptr, nullptr, nullptr, seg_start, seg_len, dst_start, (hipStream_t)stream);
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}

static int ml_ragged(const char* who, const fc_kv_view* const src[2], const fc_kv_view* const dst[2], const fc_mlp_weights* w,
                     int planes, int cf, const int32_t* seg_start, const int32_t* seg_len, const int32_t* dst_start,
                     int max_seg_len, int min_rows, void* stream) {
  MlPlanes a{};
  int rc = ml_planes(who, src, dst, w, planes, cf, a);
  if (rc) return rc;
  FC_REQUIRE(seg_start && seg_len && dst_start, FC_EINVAL, "%s: null segment arrays", who);
  FC_REQUIRE(max_seg_len >= 0 && max_seg_len <= src[0]->max_seq_len, FC_EINVAL,
             "%s: max_seg_len %d outside [0, max_seq_len %d]", who, max_seg_len, src[0]->max_seq_len);
  FC_REQUIRE(min_rows >= 0, FC_EINVAL, "%s: negative min_rows", who);
  FC_REQUIRE(src[0]->num_kv_heads <= 65535, FC_EUNSUPPORTED, "%s: too many heads", who);
  if (max_seg_len == 0) return FC_OK;
  hipStream_t st = (hipStream_t)stream;
  const int c = max_seg_len / cf;
  if (c > 0 && c >= min_rows &&
      (rc = ml_launch(who, src[0], dst[0], a, planes, cf, 0, c, 0, seg_start, seg_len, dst_start, min_rows, st)))
    return rc;
  ml_tails(src, dst, a, planes, cf, min_rows, c, seg_start, seg_len, dst_start, 0, max_seg_len, 0, st);
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}

extern "C" int fc_ccm_mlp(const fc_kv_view* src, const fc_kv_view* dst, const fc_mlp_weights* w, int32_t cf,
                          int32_t seg_start, int32_t seg_len, int32_t dst_start, void* stream) {
  const fc_kv_view *s[2] = {src, src}, *d[2] = {dst, dst};
  return ml_uniform("fc_ccm_mlp", s, d, w, 1, cf, seg_start, seg_len, dst_start, stream);
}

extern "C" int fc_ccm_mlp_kv(const fc_kv_view* k_src, const fc_kv_view* k_dst, const fc_kv_view* v_src, const fc_kv_view* v_dst,
                             const fc_mlp_weights* weights, int32_t cf, int32_t seg_start, int32_t seg_len, int32_t dst_start,
                             void* stream) {
  const fc_kv_view *s[2] = {k_src, v_src}, *d[2] = {k_dst, v_dst};
  return ml_uniform("fc_ccm_mlp_kv", s, d, weights, 2, cf, seg_start, seg_len, dst_start, stream);
}

extern "C" int fc_ccm_mlp_ragged(const fc_kv_view* src, const fc_kv_view* dst, const fc_mlp_weights* w, int32_t cf,
                                 const int32_t* seg_start, const int32_t* seg_len, const int32_t* dst_start,
                                 int32_t max_seg_len, int32_t min_rows, void* stream) {
  const fc_kv_view *s[2] = {src, src}, *d[2] = {dst, dst};
  return ml_ragged("fc_ccm_mlp_ragged", s, d, w, 1, cf, seg_start, seg_len, dst_start, max_seg_len, min_rows, stream);
}

extern "C" int fc_ccm_mlp_kv_ragged(const fc_kv_view* k_src, const fc_kv_view* k_dst, const fc_kv_view* v_src,
                                    const fc_kv_view* v_dst, const fc_mlp_weights* weights, int32_t cf,
                                    const int32_t* seg_start, const int32_t* seg_len, const int32_t* dst_start,
                                    int32_t max_seg_len, int32_t min_rows, void* stream) {
  const fc_kv_view *s[2] = {k_src, v_src}, *d[2] = {k_dst, v_dst};
  return ml_ragged("fc_ccm_mlp_kv_ragged", s, d, weights, 2, cf, seg_start, seg_len, dst_start, max_seg_len, min_rows, stream);
}

// k_out / v_out null: all layers of a plane in one allocation, a layer stride apart
static int ml_list(const char* who, const void* const* k_layers, const void* const* v_layers, void* const* k_out, void* const* v_out,
                   const fc_kv_view* k_src, const fc_kv_view* v_src, const fc_kv_view* k_dst, const fc_kv_view* v_dst,
                   const fc_mlp_weights* weights, int32_t num_segments, const int32_t* seg_start, const int32_t* seg_len,
                   const int32_t* dst_start, int32_t cf, int32_t min_rows, void* stream) {
  FC_REQUIRE(k_layers && v_layers && k_src && v_src && k_dst && v_dst && weights && seg_start && seg_len && dst_start,
             FC_EINVAL, "%s: null pointer", who);
  FC_REQUIRE(num_segments >= 1 && num_segments <= ML_LIST_SEGS, FC_EINVAL, "%s: %d segments (1 or 2)", who, num_segments);
  FC_REQUIRE(min_rows >= 0, FC_EINVAL, "%s: negative min_rows", who);
  FC_REQUIRE(k_src->num_layers <= ML_LIST_LAYERS, FC_EUNSUPPORTED, "%s: %d layers (at most %d)", who, k_src->num_layers,
             ML_LIST_LAYERS);
  const fc_kv_view* views[2][2] = {{k_src, k_dst}, {v_src, v_dst}};
  int rc;
  for (int p = 0; p < 2; ++p)
    for (int s = 0; s < num_segments; ++s)
      if ((rc = ml_check(who, views[p][0], views[p][1], &weights[s * 2 + p], cf))) return rc;
  FC_REQUIRE(!k_src->block_tables && !v_src->block_tables && !k_dst->block_tables && !v_dst->block_tables, FC_EINVAL,
             "%s: dense tensors only", who);
  FC_REQUIRE(k_src->dtype == v_src->dtype && k_src->num_layers == v_src->num_layers && k_src->batch == v_src->batch &&
                 k_src->num_kv_heads == v_src->num_kv_heads,
             FC_EINVAL, "%s: K and V disagree", who);
  MlpList a;
  for (int p = 0; p < 2; ++p)
    for (int l = 0; l < k_src->num_layers; ++l) {
      const fc_kv_view* dv = views[p][1];
      void* const* out = p ? v_out : k_out;
      a.src[p][l] = (const char*)(p ? v_layers : k_layers)[l];
      a.dst[p][l] = out ? (char*)out[l] : (char*)dv->base + (int64_t)l * dv->stride_layer * 2;
      FC_REQUIRE(a.src[p][l] && a.dst[p][l] && (((uintptr_t)a.src[p][l] | (uintptr_t)a.dst[p][l]) & 15) == 0, FC_EINVAL,
                 "%s: layer %d not 16-byte aligned", who, l);
    }
  const int ncols = k_src->batch * k_src->num_kv_heads;
  const int lp = 2 * k_src->num_layers;     // (plane, layer) pairs per segment
  int gmax = 0;
  for (int s = 0; s < num_segments; ++s) {
    const int64_t n = seg_len[s], c0 = n / cf;
    const int c = c0 < min_rows ? 0 : (int)c0;
    FC_REQUIRE(n >= 0 && seg_start[s] >= 0 && dst_start[s] >= 0 && seg_start[s] + n <= k_src->max_seq_len &&
                   seg_start[s] + n <= v_src->max_seq_len,
               FC_EINVAL, "%s: segment %d outside the source", who, s);
    a.rem[s] = (int)(n - (int64_t)c * cf);
    FC_REQUIRE((int64_t)dst_start[s] + c + a.rem[s] <= k_dst->max_seq_len &&
                   (int64_t)dst_start[s] + c + a.rem[s] <= v_dst->max_seq_len,
               FC_EINVAL, "%s: segment %d outside the destination", who, s);
    a.seg_start[s] = seg_start[s];
    a.dst_start[s] = dst_start[s];
    a.c_rows[s] = c;
    for (int p = 0; p < 2; ++p) {
      const fc_mlp_weights& w = weights[s * 2 + p];
      const void* ws[6] = {w.w1, w.b1, w.w2, w.b2, w.w3, w.b3};
      for (int i = 0; i < 6; ++i) a.w[s][p][i] = (const char*)ws[i];
    }
    // Workgroups per (layer, plane): the fewest rounds times (iterations and the start, as in ml_split).
    const double ncu = fc_compute_units();
    const int64_t rows = (int64_t)ncols * c, turns = (rows + ML_ROWS * ML_WAVES - 1) / (ML_ROWS * ML_WAVES);
    FC_REQUIRE(rows < (1LL << 31) && (int64_t)ncols * a.rem[s] < (1LL << 31), FC_EUNSUPPORTED, "%s: too many rows", who);
    a.flat[s] = MlFlat{(unsigned)rows, fc_divisor(c > 0 ? c : 1), fc_divisor(k_src->num_kv_heads)};
    double best = -1.0;
    a.gx[s] = (int)std::min<int64_t>(8, ((int64_t)ncols * a.rem[s] + 31) / 32);     // a segment that is copied whole
    for (int64_t g = 1; g <= turns && (g == 1 || (double)(g * lp) <= 8.0 * ncu); ++g) {
      const double wgs = (double)g * lp / ncu, whole = floor(wgs), part = wgs - whole;
      const double rounds = whole + (part <= 0.0 ? 0.0 : part > 0.85 ? part : 0.85);
      const double cost = rounds * ((double)((turns + g - 1) / g) + (cf <= 2 ? 0.7 : 0.4));
      if (best < 0 || cost < best) {
        best = cost;
        a.gx[s] = (int)g;
      }
    }
    if (c + a.rem[s] > 0 && a.gx[s] > gmax) gmax = a.gx[s];
  }
  if (gmax == 0) return FC_OK;
  FC_REQUIRE(lp * num_segments <= 65535, FC_EUNSUPPORTED, "%s: grid too large", who);
  dim3 grid(gmax, lp * num_segments);
  KvView ks = fc_make_view(k_src), vs = fc_make_view(v_src), kd = fc_make_view(k_dst), vd = fc_make_view(v_dst);
#define ML_LIST(DT, WR)                                                                                              \
  do {                                                                                                               \
    FC_ALLOW_LDS((mlp_list_kernel<DT, WR>), ML_LDS);                                                                 \
    hipLaunchKernelGGL((mlp_list_kernel<DT, WR>), grid, dim3(ML_THREADS), ML_LDS, (hipStream_t)stream, ks, vs, kd, vd, a, \
                       cf, ncols);                                                                                   \
  } while (0)
  if (k_src->dtype == FC_BF16) {
    if (cf <= 2) ML_LIST(FC_BF16, true); else ML_LIST(FC_BF16, false);
  } else {
    if (cf <= 2) ML_LIST(FC_F16, true); else ML_LIST(FC_F16, false);
  }
#undef ML_LIST
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}

extern "C" int fc_ccm_mlp_layers(const void* const* k_layers, const void* const* v_layers, const fc_kv_view* k_src,
                                 const fc_kv_view* v_src, const fc_kv_view* k_dst, const fc_kv_view* v_dst,
                                 const fc_mlp_weights* weights, int32_t num_segments, const int32_t* seg_start,
                                 const int32_t* seg_len, const int32_t* dst_start, int32_t cf, int32_t min_rows,
                                 void* stream) {
  return ml_list("fc_ccm_mlp_layers", k_layers, v_layers, nullptr, nullptr, k_src, v_src, k_dst, v_dst, weights, num_segments,
                 seg_start, seg_len, dst_start, cf, min_rows, stream);
}

extern "C" int fc_ccm_mlp_layers_into(const void* const* k_layers, const void* const* v_layers, void* const* k_out,
                                      void* const* v_out, const fc_kv_view* k_src, const fc_kv_view* v_src,
                                      const fc_kv_view* k_dst, const fc_kv_view* v_dst, const fc_mlp_weights* weights,
                                      int32_t num_segments, const int32_t* seg_start, const int32_t* seg_len,
                                      const int32_t* dst_start, int32_t cf, int32_t min_rows, void* stream) {
  const char* who = "fc_ccm_mlp_layers_into";
  FC_REQUIRE(k_out && v_out, FC_EINVAL, "%s: null pointer", who);
  return ml_list(who, k_layers, v_layers, k_out, v_out, k_src, v_src, k_dst, v_dst, weights, num_segments, seg_start, seg_len,
                 dst_start, cf, min_rows, stream);
}
