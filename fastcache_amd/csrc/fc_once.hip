// SnapKV per-key sums with every logit formed once (fp16/bf16 caches, up to 16 blocks of 32 window queries per kv head).
//
// A softmax needs all keys of a row before any probability is final, and fc_snapkv.hip sweeps the keys twice for it: QK^T and
// the exponentials a second time, and where columns are cut into key ranges a second launch, which starts as cold as the first.
// Here the exponentials wait in registers.  A workgroup takes a chunk of 256 keys of a column (layer, sequence, kv head)
// against a group of four blocks of 32 window queries, one block per wavefront:
//   1. e = exp2(q.k * c), 128 registers a lane, and every query's sum over the chunk's keys;
//   2. the sums go to memory, past the L2, where the workgroups that hold the column's other chunks look for them;
//   3. when all of the column's sums are there: the queries' totals (in the chunks' order, so every workgroup gets the same
//      bits) and the per-key sums of e / total over the group's queries, which the selection adds up over the groups.
// 256 registers a lane hold the exponentials, the queries and what the matrix instructions need, so two wavefronts share a
// SIMD and two workgroups a compute unit: one computes while the other waits.  The next chunk's first keys and queries travel
// meanwhile; a chunk's second 128 keys travel while the first are multiplied.
//
// Bound by latency, not by the matrix pipes (18 % busy on 2304 columns of 4096 keys) or memory: a turn of a workgroup is about
// 20 000 cycles, 6400 of them the two halves, 3000 the loads' issue, the rest the way of the sums through memory, the wait for
// the column's slowest workgroup and the reductions.  What that buys against the two sweeps stands at fc_once_pays.
// Tried and not kept: 8 wavefronts and 128 keys, the exponentials of two chunks in registers (1590 us against 1400 for 2304
// columns of 4096 keys); looking for the sums in the L2 first (a line that was looked at stays as it was: 382 us against 269
// for 13 sequences of 200 to 2300 tokens); looking at one of the missing sums only (1760 against 1360: a second way through
// memory per wait); knowing two chunks ahead (10 % faster there, 5 to 20 % slower where lengths differ).
//
// Who waits for whom.  A workgroup waits for the sums of a column only while the next chunk it holds is of another column.
// Handed a second chunk of the column it would have to wait for, it gives the exponentials up (`later`), goes on, and forms
// them again when no further chunk of that column is in its hands.  Chunks are handed out in order, one at a time, so: whoever
// waits has written its sums of all chunks it was handed of that column and before; a chunk that is not handed out yet is behind
// the one the waiting workgroup holds, of a later column; and a chunk that another workgroup holds is computed before that one
// waits for its own or for a later column.  The wait therefore ends whatever number of workgroups the chip runs at a time, and
// with one workgroup as well.  It is bounded all the same; a bound that is reached leaves NaN sums.
//
// Offsets.  exp2 needs no maximum subtracted while a chunk's sums stay within 2^-60 .. 2^60 (fp32 rounds relative to the value,
// and terms that underflow are below 2^-60 of the sum); a wavefront that finds one outside forms its chunk again with the
// queries' largest logits as offsets and hands these on beside its sums, whose sign bit says so.  Error of the sums against 64
// bits (2-norm): 5e-8, two sweeps 1.7e-7 to 4.7e-7; queries and keys four times as large, where offsets are needed, 1.1e-6,
// two sweeps 2.7e-6.
#include "fc_common.h"
#include "fc_once.h"

#define SO_WAVES 4                   // wavefronts, and blocks of 32 window queries, of a workgroup
#define SO_THREADS (SO_WAVES * 64)
#define SO_HOOK_KEYS 32768           // see fc_once_pays
#define SO_KEPT_ROWS 1100000         // likewise
#define SO_SLOT (128 * 256)          // 128 keys, or the queries of a group, in LDS: rows of 256 bytes, 16-byte pieces XOR-swizzled
#define SO_RING 4
#define SO_NONE 0xffffffffu          // a sum that is not there yet
#define SO_NEG (-1.0e30f)
#define SO_PATIENCE (1 << 20)        // looks at the sums before a wait is given up (more than a second)
#define SO_EXP_FROM 23
#define SO_INLINE __attribute__((always_inline))   // (the exponentials' arrays must stay in registers)

struct SoChunk {   // one chunk of keys against one group of query blocks
  int sub;         // column * groups + group
  int s0;          // its first key
  int S;           // tokens of the sequence
  int group;
  unsigned long long keys[4];   // addresses of the first rows of its quarters (past the end: the last one there is)
  unsigned long long queries;   // address of the column's first query row
  unsigned long long pad;
};
#define SO_WORDS ((int)(sizeof(SoChunk) / 4))

struct SoArgs {
  KvView kv;
  const char* q;
  int Hq, W, causal, groups;
  float c;
  float* raw;        // [group][column][raw_stride]
  int raw_stride;
  long long raw_group;
  float* sums;       // [column][group][block][chunk][32]; SO_NONE: not there yet
  float* offs;       // the same shape: offsets of the chunks whose sums are negative
  SoChunk* table;    // [list][per_list] in the order they are handed out
  int per_list;
  unsigned* tickets; // [lists] 32 words apart: handed out so far, and how many there are
  int chunks;        // of the longest column
  int lists;
};

// What the kernel below starts from: no sum is there, no chunk handed out, and the list of every chunk with its addresses.
// Chunks of a list go sequence by sequence, column by column (those whose number is the list's modulo their count), group by
// group.
__global__ __launch_bounds__(256) void snapkv_once_setup_kernel(SoArgs a, long long vecs, int items) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i < vecs) reinterpret_cast<uint4*>(a.sums)[i] = make_uint4(SO_NONE, SO_NONE, SO_NONE, SO_NONE);
  const KvView& kv = a.kv;
  const int B = kv.batch, LH = kv.num_layers * kv.num_kv_heads;
  auto chunks_of = [&](int S) { return S > a.W ? (S + SO_KEYS - 1) / SO_KEYS : 0; };
  auto below = [&](int x, int list) { return x > list ? (x - list + a.lists - 1) / a.lists : 0; };   // columns of the list below x
  auto before = [&](int b, int list) {   // chunks of the list of sequences before b
    int n = 0;
    for (int k = 0; k < b; ++k) n += chunks_of(fc_seq_len(kv, k)) * (below((k + 1) * LH, list) - below(k * LH, list));
    return n * a.groups;
  };
  if (i < a.lists * 32) {
    const int list = (int)i >> 5, w = (int)i & 31;
    if (w < 2) a.tickets[i] = w == 0 ? 0u : (unsigned)before(B, list);
  }
  if (i >= items) return;
  const int chunk = (int)i % a.chunks, subs = (int)i / a.chunks, group = subs % a.groups, g = subs / a.groups;   // g: b, l, h
  const int b = g / LH, lh = g - b * LH, l = lh / kv.num_kv_heads, h = lh - l * kv.num_kv_heads, list = g % a.lists;
  const int S = fc_seq_len(kv, b), n = chunks_of(S);
  if (chunk >= n) return;
  SoChunk r;
  r.sub = ((l * B + b) * kv.num_kv_heads + h) * a.groups + group;
  r.s0 = chunk * SO_KEYS;
  r.S = S;
  r.group = group;
  const long long at = (long long)l * kv.stride_layer + (long long)h * kv.stride_head;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int s = r.s0 + 64 * j;
    r.keys[j] = j > 0 ? r.keys[j - 1] : 0;
    if (s < S) r.keys[j] = (unsigned long long)(kv.base + (at + max(fc_token_offset(kv, b, s), 0ll)) * 2);
  }
  r.queries = (unsigned long long)(a.q + ((long long)(l * B + b) * a.Hq + (long long)h * (a.Hq / kv.num_kv_heads)) * a.W * 256);
  r.pad = 0;
  const int rank = below(g, list) - below(b * LH, list);   // of the column among the sequence's in the list
  a.table[(long long)list * a.per_list + before(b, list) + (rank * a.groups + group) * n + chunk] = r;
}

__device__ __forceinline__ float so_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// a + its neighbour 16 (32) lanes away, for two registers at once: the low rows (half) get the sum of a, the high ones of b
__device__ __forceinline__ float so_fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float so_fold32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float so_max16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float so_max32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// Sums (maxima) of 16 registers over the 32 lanes of each half: lane l gets register so_reg(l) of its half.  Every step halves the
// registers and doubles the lanes that hold different ones: 38 instructions, 80 for 16 reductions by themselves.
__device__ __forceinline__ int so_reg(int lane) {
  return ((lane >> 4) & 1) * 8 + ((lane >> 3) & 1) * 4 + ((lane >> 2) & 1) * 2 + ((lane >> 1) & 1);
}
template <bool MAX>
__device__ __forceinline__ float so_reduce(const float (&v)[16], int lane) {
  auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
  float w[8], x[4], y[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) w[i] = MAX ? so_max16(v[i], v[i + 8]) : so_fold16(v[i], v[i + 8]);
  const bool b3 = lane & 8, b2 = lane & 4, b1 = lane & 2;
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = op(b3 ? w[i + 4] : w[i], fc_dpp<0x128>(b3 ? w[i] : w[i + 4]));   // row_ror:8
#pragma unroll
  for (int i = 0; i < 2; ++i) y[i] = op(b2 ? x[i + 2] : x[i], fc_dpp<0x141>(b2 ? x[i] : x[i + 2]));   // row_half_mirror
  float z = op(b1 ? y[1] : y[0], fc_dpp<0x4E>(b1 ? y[0] : y[1]));   // quad_perm [2,3,0,1]
  return op(z, fc_dpp<0xB1>(z));                                     // quad_perm [1,0,3,2]
}

struct SoYes { static constexpr bool value = true; };
struct SoNo { static constexpr bool value = false; };

template <int DTYPE>
__global__ __launch_bounds__(SO_THREADS, 2) void snapkv_once_kernel(SoArgs a) {
  extern __shared__ __align__(16) char smem_raw[];
  char* smem = smem_raw + ((256u - (fc_lds_addr(smem_raw) & 255u)) & 255u);
  // two slots, which change places with every chunk: one takes the chunk's queries, then the second half of its keys, the other
  // the first half, then the next chunk's queries
  float(*vpart)[SO_WAVES][SO_KEYS] = reinterpret_cast<float(*)[SO_WAVES][SO_KEYS]>(smem + 2 * SO_SLOT);   // [2]
  float(*wbuf)[32] = reinterpret_cast<float(*)[32]>(vpart + 2);                                         // [SO_WAVES]
  SoChunk* ring = reinterpret_cast<SoChunk*>(wbuf + SO_WAVES);                                          // [SO_RING]
  int* pending = reinterpret_cast<int*>(ring + SO_RING);   // [SO_CHUNKS_MAX]: tickets

  const int tid = threadIdx.x, lane = tid & 63, lrow = lane & 31, lhalf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = a.W;
  const float c = a.c;
  // what is formed from it is formed again every time, not kept in registers from before the loop
  auto fresh = [](int x) {
    asm volatile("" : "+v"(x));
    return x;
  };
  auto chunks_of = [&](int S) { return (S + SO_KEYS - 1) / SO_KEYS; };

  // ---- tickets: one wavefront takes them, and brings the chunks they stand for ------------------------------------
  const int list = (int)blockIdx.x % a.lists;
  const SoChunk* table = a.table + (long long)list * a.per_list;
  unsigned* tickets = a.tickets + list * 32;
  const int total = (int)tickets[1];
  auto take = [&]() SO_INLINE {
    unsigned t = 0;
    if (lane == 0) t = __hip_atomic_fetch_add(tickets, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return t;
  };
  auto word_of = [&](int t) SO_INLINE {   // (word `lane` of the chunk; none: -1 as its column)
    return t < total ? reinterpret_cast<const int*>(table + t)[lane & (SO_WORDS - 1)] : -1;
  };
  auto put = [&](int word, SoChunk* to) SO_INLINE {
    if (lane < SO_WORDS) reinterpret_cast<int*>(to)[lane] = word;
  };

  // ---- a chunk as a wavefront sees it -----------------------------------------------------------------------------------
  struct Chunk { int sub, s0, S, qi; bool active; const char* keys[2]; const char* queries; };
  auto scalar64 = [](unsigned long long u) {
    return reinterpret_cast<const char*>(((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32) |
                                         (unsigned)__builtin_amdgcn_readfirstlane((int)(u & 0xffffffffu)));
  };
  const int WB = (W + 31) / 32, blocks = a.Hq / a.kv.num_kv_heads * WB;
  auto read_chunk = [&](const SoChunk* from) SO_INLINE {
    Chunk k;
    k.sub = __builtin_amdgcn_readfirstlane(from->sub);
    k.s0 = __builtin_amdgcn_readfirstlane(from->s0);
    k.S = __builtin_amdgcn_readfirstlane(from->S);
    const int block = __builtin_amdgcn_readfirstlane(from->group) * SO_WAVES + wave;
    k.active = k.sub >= 0 && block < blocks;
    const int qg = WB == 1 ? block : WB == 2 ? block >> 1 : block / WB;
    k.qi = (block - qg * WB) * 32;   // first of its queries, of query head qg of the column's
    k.keys[0] = scalar64(from->keys[wave >> 1]);
    k.keys[1] = scalar64(from->keys[2 + (wave >> 1)]);
    k.queries = scalar64(from->queries) + (long long)qg * W * 256;
    return k;
  };

  // ---- loads ---------------------------------------------------------------------------------------------------------
  // Lane i of a wave-load writes LDS piece i of 64 (4 rows) and fetches piece (i & 15) ^ (row & 15) of its row, so that the
  // operand reads (32 rows, one piece each) fall on distinct banks.  Rows past the sequence end (the window's) are clamped.
  const unsigned slots = __builtin_amdgcn_readfirstlane(fc_lds_addr(smem)), mine_at = wave * 8192;
  const unsigned tok_bytes = (unsigned)a.kv.stride_token * 2;
  // rows 32 wave + 4 u .. of half `half`
  auto load_keys = [&](const Chunk& k, int half, unsigned slot, int u) SO_INLINE {
    const int ln = fresh(lane), g = ln >> 4, quarter = min(2 * half + (wave >> 1), (k.S - 1 - k.s0) >> 6);
    const int most = k.S - 1 - k.s0 - 64 * quarter;   // last row of the quarter that exists
    const unsigned piece = (unsigned)(((ln & 15) ^ g ^ (4 * (u & 3))) << 4);
    fc_load_lds(k.keys[half], (unsigned)min((wave & 1) * 32 + 4 * u + g, most) * tok_bytes + piece, slot + mine_at + u * 1024);
  };
  auto load_queries = [&](const Chunk& k, unsigned slot, int u) SO_INLINE {
    const int ln = fresh(lane), g = ln >> 4;
    const unsigned piece = (unsigned)(((ln & 15) ^ g ^ (4 * (u & 3))) << 4);
    fc_load_lds(k.queries, (unsigned)min(k.qi + 4 * u + g, W - 1) * 256 + piece, slot + mine_at + u * 1024);
  };

  int turn_slot = 0;   // (the chunk's place in the ring)
  const unsigned xs = (unsigned)((lhalf ^ (lrow & 15)) << 4) + lrow * 256;
  uint4 qf[8];
  auto settle = [&]() SO_INLINE {   // (what is on its way to these registers is waited for here and not in the loops)
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) asm volatile("" : "+v"(qf[ks].x), "+v"(qf[ks].y), "+v"(qf[ks].z), "+v"(qf[ks].w));
  };
  // C[query][key]: the lane owns one key and 16 queries per 32 keys.  Operand reads run four ahead of the matrix instructions
  // (left to the scheduler each one was waited for by itself), and with_exp the exponentials follow nine
  // instructions behind, two registers at a time (exp_pairs from SO_EXP_FROM on forms the rest of them).
  auto exp_pairs = [&](f32x16* e, float (&rs)[16], int from, int to, bool first) SO_INLINE {
#pragma unroll
    for (int m = from; m < to; ++m) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int cb = m >> 3, i = (m & 7) * 2 + j;
        e[cb][i] = so_exp2(e[cb][i] * c);
        rs[i] = first && cb == 0 ? e[cb][i] : rs[i] + e[cb][i];
      }
    }
  };
  auto logits = [&](unsigned kaddr, f32x16* e, float (&rs)[16], bool first, auto with_exp, auto beside) SO_INLINE {
    unsigned ad[8];
    const unsigned x0 = kaddr + (unsigned)fresh((int)xs);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) ad[ks] = x0 ^ (unsigned)(ks * 32);
    uint4 kf[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) kf[n] = fc_lds_read128(ad[n]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 32; ++n) {
      const int cb = n >> 3, ks = n & 7;
      if (ks == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) e[cb][i] = 0.f;
      }
      e[cb] = fc_mfma<DTYPE>(qf[ks], kf[n & 3], e[cb]);
      if (n + 4 < 32) kf[n & 3] = fc_lds_read128(ad[(n + 4) & 7] + (unsigned)(((n + 4) >> 3) * 8192));
      if constexpr (decltype(with_exp)::value) {
        if (n >= 9) exp_pairs(e, rs, n - 9, n - 8, first);
      }
      beside(n);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // key s of the lane's half against register i's query (qi + half * 4 + place(i)): seen when behind(s) <= place(i)
  auto place = [](int i) { return (i >> 2) * 8 + (i & 3); };
  auto behind = [&](int s, const Chunk& k, int half) {
    const int d = s - (k.S - W);   // place in the window
    return d >= W ? 64 : a.causal ? d - k.qi - half * 4 : -64;
  };
  auto sums_at = [&](const Chunk& k) { return (unsigned)((k.sub * SO_WAVES + wave) * a.chunks) * 32u; };   // of chunk 0

  // exponentials of one half of a chunk into e, added up over its keys per register; `beside` is called between the matrix
  // instructions
  auto half_of = [&](const Chunk& k, int half, unsigned kaddr, f32x16* e, float (&rs)[16], auto beside) SO_INLINE {
    const int s0 = k.s0 + half * 128;
    if (s0 + 128 <= (a.causal ? k.S - W + 1 : k.S)) {
      logits(kaddr, e, rs, half == 0, SoYes{}, beside);
      exp_pairs(e, rs, SO_EXP_FROM, 32, half == 0);
    } else {
      logits(kaddr, e, rs, half == 0, SoNo{}, beside);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const int x = behind(s0 + cb * 32 + fresh(lrow), k, lhalf);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          e[cb][i] = x <= place(i) ? so_exp2(e[cb][i] * c) : 0.f;
          rs[i] = half == 0 && cb == 0 ? e[cb][i] : rs[i] + e[cb][i];
        }
      }
    }
  };
  // the chunk again with the queries' largest logits as offsets, from keys in memory (their places in LDS have been given to
  // others); the offsets go to memory when `write`, and the sums come back negative
  auto with_offsets = [&](const Chunk& k, f32x16 (&e)[8], bool write) SO_INLINE {
    float m[16], rs[16];
#pragma unroll
    for (int cb = 0; cb < 8; ++cb) {
      const int row = min(cb * 32 + fresh(lrow), k.S - 1 - k.s0);
      const unsigned long long* at4 = ring[turn_slot & (SO_RING - 1)].keys;
      const char* kp = reinterpret_cast<const char*>(at4[row >> 6]) + (unsigned long long)(row & 63) * tok_bytes + lhalf * 16;
#pragma unroll
      for (int i = 0; i < 16; ++i) e[cb][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) e[cb] = fc_mfma<DTYPE>(qf[ks], *reinterpret_cast<const uint4*>(kp + ks * 32), e[cb]);
      const int x = behind(k.s0 + cb * 32 + fresh(lrow), k, lhalf);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        e[cb][i] = x <= place(i) ? e[cb][i] * c : SO_NEG;
        m[i] = cb == 0 ? e[cb][i] : fmaxf(m[i], e[cb][i]);
      }
    }
    const float mx = fmaxf(so_reduce<true>(m, lane), SO_NEG);   // (all of the chunk's logits may be -inf)
    const int reg = so_reg(fresh(lane)), q = place(reg) + lhalf * 4;
    __builtin_amdgcn_wave_barrier();
    wbuf[wave][q] = mx;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float mi = wbuf[wave][place(i) + lhalf * 4];
#pragma unroll
      for (int cb = 0; cb < 8; ++cb) {
        e[cb][i] = e[cb][i] == SO_NEG ? 0.f : so_exp2(e[cb][i] - mi);
        rs[i] = cb == 0 ? e[cb][i] : rs[i] + e[cb][i];
      }
    }
    if (write) {
      if (!(lane & 1))
        __hip_atomic_store(a.offs + sums_at(k) + (unsigned)(k.s0 / SO_KEYS * 32 + q), mx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      fc_wait_vm<0>();   // there before the sums that speak of them
    }
    const float z = so_reduce<false>(rs, lane);
    return z == z ? -z : __uint_as_float(0xffc00000u);
  };
  // the chunk's sums into memory
  auto hand_on = [&](const Chunk& k, f32x16 (&e)[8], const float (&rs)[16], bool write) SO_INLINE {
    float z = so_reduce<false>(rs, lane);
    const int reg = so_reg(fresh(lane)), q = place(reg) + lhalf * 4;
    const bool empty = behind(k.s0, k, lhalf) > place(reg);   // the query sees none of these keys
    const bool bad = !empty && !(z >= 0x1p-60f && z <= 0x1p60f);
    if (__builtin_expect(__any(bad), 0)) z = with_offsets(k, e, write);
    if (write && !(lane & 1))
      __hip_atomic_store(a.sums + sums_at(k) + (unsigned)(k.s0 / SO_KEYS * 32 + q), z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };

  // totals of the chunk's queries -> per-key sums of its probabilities into out[SO_KEYS]
  int patience = SO_PATIENCE;
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  // lane: four queries (lane & 7) * 4 + 0..3 of chunk g + 8 j + lane / 8; of chunks that are not there, 0
  auto ask = [&](const Chunk& k, int g, u32x4 (&v)[4]) SO_INLINE {   // (past the L2, which does not see them change)
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.sums + sums_at(k), 0, chunks_of(k.S) * 128, 0x00027000);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, (g + 8 * j) * 128 + lane * 16, 0, 16);
  };
  auto finish = [&](const Chunk& k, const f32x16 (&e)[8], u32x4 (&v)[4], float* out) SO_INLINE {
    const int n = chunks_of(k.S);
    float tot[4] = {0.f, 0.f, 0.f, 0.f};
    unsigned sign = 0;
    for (int g = 0; g < n; g += 32) {
      if (g > 0) ask(k, g, v);
      unsigned top;
      for (int tries = 0;; ++tries) {
        // SO_NONE is the largest number there is, and any sign puts a number above those without
        top = max(max(max(v[0].x, v[0].y), max(v[0].z, v[0].w)), max(max(v[1].x, v[1].y), max(v[1].z, v[1].w)));
        top = max(top, max(max(max(v[2].x, v[2].y), max(v[2].z, v[2].w)), max(max(v[3].x, v[3].y), max(v[3].z, v[3].w))));
        if (__all(top != SO_NONE)) break;
        if (tries >= patience) {   // (does not happen; the sums that are not there are NaN as numbers)
          patience = 0;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
        ask(k, g, v);
      }
      sign |= top;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        tot[0] += __uint_as_float(v[j].x);
        tot[1] += __uint_as_float(v[j].y);
        tot[2] += __uint_as_float(v[j].z);
        tot[3] += __uint_as_float(v[j].w);
      }
    }
    float w[4] = {0.f, 0.f, 0.f, 0.f};
    const int q0 = (lane & 7) * 4;
    auto all_chunks = [&](float t) {
      t += fc_dpp<0x128>(t);
      t = so_fold16(t, t);
      return so_fold32(t, t);
    };
    if (__builtin_expect(!__any((int)sign < 0), 1)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = __builtin_amdgcn_rcpf(all_chunks(tot[i]));   // (1 ulp)
    } else {   // chunks with offsets of their own among them
      float* zs = a.sums + sums_at(k) + fresh(q0);
      float* os = a.offs + sums_at(k) + fresh(q0);
      auto offset_at = [&](int chunk, int i, float z) {
        return (__float_as_uint(z) >> 31) ? __hip_atomic_load(os + chunk * 32 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.f;
      };
      auto sum_at = [&](int chunk, int i) {
        return __hip_atomic_load(zs + chunk * 32 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
#pragma unroll 1
      for (int i = 0; i < 4; ++i) {
        float mx = SO_NEG;
        for (int j = lane >> 3; j < n; j += 8) {
          const float z = sum_at(j, i);
          if (!(z == 0.f)) mx = fmaxf(mx, offset_at(j, i, z));
        }
        mx = fmaxf(mx, fc_dpp<0x128>(mx));
        mx = so_max16(mx, mx);
        mx = so_max32(mx, mx);
        float t = 0.f;
        for (int j = lane >> 3; j < n; j += 8) {
          const float z = sum_at(j, i);
          if (!(z == 0.f)) t += fabsf(z) * so_exp2(offset_at(j, i, z) - mx);
        }
        t = all_chunks(t);
        const float z = sum_at(k.s0 / SO_KEYS, i);
        const float wi = z == 0.f ? 0.f : so_exp2(offset_at(k.s0 / SO_KEYS, i, z) - mx) / t;
        w[0] = i == 0 ? wi : w[0];
        w[1] = i == 1 ? wi : w[1];
        w[2] = i == 2 ? wi : w[2];
        w[3] = i == 3 ? wi : w[3];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (k.qi + q0 + i >= W) w[i] = 0.f;
    __builtin_amdgcn_wave_barrier();
    if (lane < 8) *reinterpret_cast<float4*>(&wbuf[wave][q0]) = make_float4(w[0], w[1], w[2], w[3]);
    __builtin_amdgcn_wave_barrier();
    float vs[8];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 wq = *reinterpret_cast<const float4*>(&wbuf[wave][g * 8 + lhalf * 4]);
#pragma unroll
      for (int cb = 0; cb < 8; ++cb) {
        vs[cb] = g == 0 ? e[cb][0] * wq.x : fmaf(e[cb][4 * g], wq.x, vs[cb]);
        vs[cb] = fmaf(e[cb][4 * g + 1], wq.y, vs[cb]);
        vs[cb] = fmaf(e[cb][4 * g + 2], wq.z, vs[cb]);
        vs[cb] = fmaf(e[cb][4 * g + 3], wq.w, vs[cb]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) out[64 * j + lane] = so_fold32(vs[2 * j], vs[2 * j + 1]);
  };
  // the wavefronts' sums of a chunk added up, in their order, one key per thread
  auto emit = [&](const Chunk& k, const float (*part)[SO_KEYS]) SO_INLINE {
    const int col = a.groups == 1 ? k.sub : a.groups == 2 ? k.sub >> 1 : k.sub / a.groups, group = k.sub - col * a.groups;
    const int n = min(blocks - group * SO_WAVES, SO_WAVES);   // (of the last group fewer than four have queries)
    float t = part[0][tid];
#pragma unroll
    for (int w = 1; w < SO_WAVES; ++w)
      if (w < n) t += part[w][tid];
    if (k.s0 + tid < k.S - W) a.raw[group * a.raw_group + (long long)col * a.raw_stride + k.s0 + tid] = t;
  };

  // ---- start ------------------------------------------------------------------------------------------------------------
  const bool taker = wave == SO_WAVES - 1;   // (where blocks are no multiple of four it has the least to do)
  int ticket = 0, word = -1;   // of the chunk after `cur` (the taker's)
  if (taker) {
    ticket = __builtin_amdgcn_readfirstlane((int)take());
    put(word_of(ticket), ring);
  }
  __syncthreads();
  const Chunk none = {-1, 0, 0, 0, false, {nullptr, nullptr}, nullptr};
  Chunk cur = read_chunk(ring), done = none;
  unsigned first = slots, second = slots + SO_SLOT;   // of the keys' halves
  if (cur.sub >= 0) {
#pragma unroll
    for (int u = 0; u < 8; ++u) load_keys(cur, 0, first, u);
    if (cur.active) {
#pragma unroll
      for (int u = 0; u < 8; ++u) load_queries(cur, second, u);
    }
  }
  int turn = 0, waiting = 0;   // chunks taken up so far; chunks of cur's column in `pending`
  unsigned asked = ~0u;
  f32x16 e[8];
  float rs[16];

  while (cur.sub >= 0) {
    turn_slot = turn;
    const int par = turn & 1;
    fc_wait_barrier<0>();   // queries and first keys of `cur` have landed, the sums of `done` are in LDS
    if (cur.active) {
      const unsigned qa = second + mine_at + (unsigned)fresh((int)xs);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) qf[ks] = fc_lds_read128(qa ^ (unsigned)(ks * 32));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the queries are in registers: their place is free
    settle();
    if (taker) asked = take();   // (nothing is waited for: the ticket comes with what the next barrier waits for)
    const bool two = cur.s0 + 128 < cur.S;
    // one load beside every fourth matrix instruction: issued together they hold the wavefronts up
    if (cur.active) {
      half_of(cur, 0, first, e, rs, [&](int n) SO_INLINE { if ((n & 3) == 1 && two) load_keys(cur, 1, second, n >> 2); });
    } else if (two) {
#pragma unroll
      for (int u = 0; u < 8; ++u) load_keys(cur, 1, second, u);
    }
    fc_wait_barrier<0>();   // the second half has landed, the first has been read
    const int held = ticket;
    if (taker) {
      ticket = __builtin_amdgcn_readfirstlane((int)asked);
      word = word_of(ticket);
    }
    if (cur.active && two) {
      half_of(cur, 1, second, e + 4, rs, [](int) {});
    } else {
#pragma unroll
      for (int cb = 4; cb < 8; ++cb)
#pragma unroll
        for (int i = 0; i < 16; ++i) e[cb][i] = 0.f;
    }
    if (taker) put(word, ring + ((turn + 1) & (SO_RING - 1)));
    fc_lds_barrier();       // the second half has been read
    const Chunk next = read_chunk(ring + ((turn + 1) & (SO_RING - 1)));
    __builtin_amdgcn_s_setprio(1);   // others wait for what comes next
    const bool later = next.sub == cur.sub, again = waiting > 0 && !later;
    const bool load = next.sub >= 0 && !again;
    if (cur.active) hand_on(cur, e, rs, true);   // (ahead of the loads, which hold the wavefront up)
    __builtin_amdgcn_s_setprio(0);
    if (load) {
#pragma unroll
      for (int u = 0; u < 8; ++u) load_keys(next, 0, second, u);
      if (next.active) {
#pragma unroll
        for (int u = 0; u < 8; ++u) load_queries(next, first, u);
      }
    }
    u32x4 v[4];
    if (cur.active && !later) ask(cur, 0, v);
    if (done.sub >= 0) emit(done, vpart[par ^ 1]);
    if (__builtin_expect(later, 0)) {
      if (taker && lane == 0) pending[waiting] = held;
      ++waiting;
      done = none;
    } else {
      if (cur.active) finish(cur, e, v, vpart[par][wave]);
      done = cur;
    }
    if (__builtin_expect(again, 0)) {   // the chunks given up, now that no further one of their column is to come
      fc_lds_barrier();
      emit(cur, vpart[par]);
      fc_lds_barrier();
      done = none;
      turn_slot = turn + 3;   // (its place in the ring is not in use)
      SoChunk* const slot = ring + (turn_slot & (SO_RING - 1));
      for (int w = 0; w < waiting; ++w) {
        if (taker) put(word_of(pending[w]), slot);
        fc_lds_barrier();
        const Chunk k = read_chunk(slot);
        if (k.active) {
#pragma unroll
          for (int ks = 0; ks < 8; ++ks)
            qf[ks] = *reinterpret_cast<const uint4*>(k.queries + (long long)min(k.qi + lrow, W - 1) * 256 + ks * 32 + lhalf * 16);
          settle();
        }
#pragma unroll
        for (int half = 0; half < 2; ++half) {
#pragma unroll
          for (int u = 0; u < 8; ++u) load_keys(k, half, second, u);
          fc_wait_barrier<0>();
          if (k.active) half_of(k, half, second, e + 4 * half, rs, [](int) {});
          fc_lds_barrier();
        }
        if (k.active) {
          hand_on(k, e, rs, false);
          ask(k, 0, v);
          finish(k, e, v, vpart[0][wave]);
        }
        fc_lds_barrier();
        emit(k, vpart[0]);
        fc_lds_barrier();
      }
      waiting = 0;
      if (next.sub >= 0) {
#pragma unroll
        for (int u = 0; u < 8; ++u) load_keys(next, 0, second, u);
        if (next.active) {
#pragma unroll
          for (int u = 0; u < 8; ++u) load_queries(next, first, u);
        }
      }
    }
    cur = next;
    ++turn;
    const unsigned t = first;
    first = second;
    second = t;
  }
  fc_lds_barrier();
  if (done.sub >= 0) emit(done, vpart[(turn & 1) ^ 1]);
}

static int so_groups(int32_t num_q_heads, int32_t num_kv_heads, int32_t window) {
  return (num_q_heads / num_kv_heads * ((window + 31) / 32) + SO_WAVES - 1) / SO_WAVES;
}
static int64_t so_chunks(int32_t max_seq_len) { return (max_seq_len + SO_KEYS - 1) / SO_KEYS; }

int fc_once_groups(const fc_kv_view* keys, int32_t num_q_heads, int32_t window) {
  return so_groups(num_q_heads, keys->num_kv_heads, window);
}

int64_t fc_once_workspace_bytes(int32_t num_layers, int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t window,
                                int32_t max_seq_len) {
  const int64_t cols = (int64_t)num_layers * batch * num_kv_heads, chunks = so_chunks(max_seq_len);
  const int64_t items = cols * so_groups(num_q_heads, num_kv_heads, window) * chunks;
  return 2 * items * SO_WAVES * 128 + (items + SO_LISTS * so_groups(num_q_heads, num_kv_heads, window) * chunks) * (int64_t)sizeof(SoChunk) +
         SO_LISTS * 128;
}

// Lists of columns, and with them how many workgroups share a list's L2 for the queries (8: those of an XCD).  A column that
// is handed out in part while the workgroups are busy keeps those that have its first chunks waiting for a turn: the fewer
// lists, the fewer of them there are.  us for scoring and selection by 1, 2, 4 and 8 lists: one turn or two each, 32 columns of 3000
// keys 46.5 41.7 39.7 39.9, of 4096 53.0 46.5 44.8 43.4, of 6000 67.8 62.0 61.8 69.3; many turns, 2304 columns of 4096 keys
// 1362 1341 1425 1454, 13 sequences of 200 to 2300 tokens 304 287 297 299, 576 columns of 6000 keys 550 570 793 1483.
static int so_lists(int64_t columns, int64_t items, int64_t chunks) {
  const bool few = items / (2 * fc_compute_units()) <= 4;
  const int n = chunks <= 16 ? (few ? SO_LISTS : 2) : (few ? 4 : 1);
  return (int)(columns < n ? columns : n);
}

bool fc_once_takes(const fc_kv_view* keys, int32_t num_q_heads, int32_t window) {
  if (!keys || keys->num_kv_heads <= 0 || window <= 0 || (keys->dtype != FC_F16 && keys->dtype != FC_BF16)) return false;
  const int64_t chunks = so_chunks(keys->max_seq_len), groups = so_groups(num_q_heads, keys->num_kv_heads, window);
  if (chunks < 1 || chunks > SO_CHUNKS_MAX || groups > 4) return false;
  if (keys->stride_token < 0 || keys->stride_token >= (1 << 24)) return false;
  if (keys->block_tables && (keys->block_size < 64 || (keys->block_size & (keys->block_size - 1)))) return false;
  // (the kernel addresses the sums with 32 bits)
  return (int64_t)keys->num_layers * keys->batch * keys->num_kv_heads * groups * chunks < (1ll << 22);
}

// Whether one pass beats two sweeps.  mean_len: the sequences' mean length, the view's max_seq_len their largest.
//
// A dense layer is a hook (scoring, selection, gather).  us, half kept, two sweeps -> one pass; where the rule says no as well:
//  32 query heads on 8, window 64: 8 columns of 4096 keys 30.2 -> 24.7, of 1000 20.4 -> 19.4; window 32: 8 of 700 16.7 -> 18.0
//  (no), of 4096 27.2 -> 23.7.  28 on 4, window 64 (14 blocks): 4 columns of 400 25.4 -> 18.4, of 4096 39.6 -> 24.7; 16 of 2000
//  33.5 -> 26.2.  More than SO_HOOK_KEYS keys in all keep the sweeps, faster or not (32 of 4096 47.5 -> 41.8): the two forms' sums
//  differ by their fp32 roundings, and two keys that all but tie at the threshold are then ranked the other way, which moves the
//  rows between them (26 of 12 800 columns of 4096 keys, 4 of 8000 of 2000, one in two to four million keys; against 64 bits
//  the sweeps are off in 25 and 6, one pass in 23 and 6).  Within the bound one call in 60 to 100 returns other rows than the
//  sweeps do; hooks of more keys, where it would be one in 15 and more, return what they did before there was one pass.  This
//  is a line drawn for unchanged results, not for time or precision.
//
// Everything else is a paged pass (selection in a launch of its own and compaction), against what fc_snapkv_rows_route says:
// key ranges, followed by the same launches, or (whole) one launch per column, which moves a column's kept rows while others
// are scored.  There the kept rows of both planes count as well: beyond SO_KEPT_ROWS of them, more than the caches hold,
// compaction as a launch is slower than what the scoring saves, unless few of a column's rows stay; lengths that differ start longest
// first in one launch, which takes most of the gain away.  us, the other form -> one pass, at 25, 50 or 70 % kept:
//  ranges.  4 blocks: 288 columns of 4201 keys, 25 %, 225 -> 189, 576 of 5870, 25 %, 630 -> 489, 1152 of 7629, 70 %, 2413 -> 2125;
//  14: 336 of 1752, 50 %, 270 -> 221, 784 of 3530, 70 %, 1272 -> 1189; 8: 288 of 2527, 25 %, 190 -> 150, 576 of 4062, 50 %, 654 -> 601, of 8212
//  1278 -> 1421 (no); 7: 112 of 964, 70 %, 60 -> 51.
//  one launch.  4 blocks: 576 of 608, 25 %, 88 -> 67, of 2332, 70 %, 392 -> 340, 1728 of 935, 25 %, 267 -> 232, of 1951, 70 %, 706 -> 786 (no);
//  1 and 2: 3072 of 943, 25 %, 407 -> 355, 4096 of 1941, 70 %, 1499 -> 1712 (no), 8192 of 604, 70 %, 1020 -> 1087 (no), of 724, 25 %, 855 ->
//  741; 14: 784 of 456, 25 %, 225 -> 136, 336 of 1270, 50 %, 232 -> 165, 1456 of 1968, 70 %, 1156 -> 1181 (no); 8: 288 of 1879, 25 %, 146 -> 113,
//  of 651, 70 %, 83 -> 76, 576 of 3245, 70 %, 558 -> 582 (no); 7: 672 of 590, 70 %, 124 -> 141 (no).
// One round of workgroups, or two of up to 4 blocks, nearly full, is where one launch is at its best: 480 columns of 671 keys, 2 blocks,
// 60 %, 75 -> 85, 224 of 809, 14 blocks, 60 %, 91 -> 97.
static bool so_whole_pays(int blocks, int64_t cols, int64_t n, int64_t mean_len, int64_t kept) {
  const bool equal = 16 * mean_len >= 15 * n, few = 3 * kept <= n;
  if (blocks > 4 && blocks <= 8) return cols <= 112 || (equal && (few || (cols <= 340 && n >= 640)));
  if (blocks > 8 ? n > 2304 : !equal && n > 600 && !(few && 10 * mean_len >= 9 * n)) return false;
  const int64_t slots = fc_compute_units() * (blocks > 4 ? 1 : 2), rounds = (cols + slots - 1) / slots;
  if (rounds <= (blocks > 4 ? 1 : 2) && 4 * cols >= 3 * rounds * slots) return few && blocks <= 4;
  return few ? blocks > 2 || n <= 1300 || 2 * cols * kept <= 3 * SO_KEPT_ROWS : cols * kept <= SO_KEPT_ROWS;
}
bool fc_once_pays(const fc_kv_view* keys, int32_t num_q_heads, int32_t window, int32_t mean_len, int32_t kept, bool whole) {
  if (!fc_once_takes(keys, num_q_heads, window)) return false;
  const int blocks = num_q_heads / keys->num_kv_heads * ((window + 31) / 32), n = keys->max_seq_len;
  const int64_t cols = (int64_t)keys->num_layers * keys->batch * keys->num_kv_heads;
  if (!keys->block_tables && keys->num_layers == 1) {
    if (cols * n > SO_HOOK_KEYS || n > 8192) return false;
    if (blocks > 8) return true;
    return blocks > 4 ? cols <= 8 || n >= (blocks == 8 ? 600 : 1500) : n >= 2700;
  }
  if (whole && !so_whole_pays(blocks, cols, n, mean_len, kept)) return false;
  const bool equal = 16LL * mean_len >= 15LL * n;
  if (blocks > 8) return n <= 1536 || (n <= 2304 && cols <= 1500) || (n <= 4096 && (cols < 400 || (equal && cols < 1000)));
  if (n < 450) return false;
  const int64_t round = 2 * fc_compute_units();      // 5 to 8 blocks: where whole columns leave the chip part empty in their last round
  if (blocks > 4) return n <= 4096 && 10 * ((cols + round - 1) / round * round) >= 14 * cols && (equal || cols <= 340);
  if (blocks > 2) return n <= 9216 && (equal || cols <= 2400);
  return equal ? n <= 4096 : n <= 768;
}

int fc_once_sums(const char* who, const fc_kv_view* keys, const void* queries, int32_t num_q_heads, int32_t window,
                 int32_t causal_window, float scale, float* raw, int32_t raw_stride, void* workspace, int32_t workgroups,
                 void* stream) {
  const int64_t cols = (int64_t)keys->num_layers * keys->batch * keys->num_kv_heads;
  const int64_t chunks = so_chunks(keys->max_seq_len), groups = so_groups(num_q_heads, keys->num_kv_heads, window);
  const int64_t items = cols * groups * chunks, n = items * SO_WAVES * 32;
  SoArgs a;
  a.kv = fc_make_view(keys);
  a.q = (const char*)queries;
  a.Hq = num_q_heads;
  a.W = window;
  a.causal = causal_window;
  a.groups = (int)groups;
  a.c = scale * 1.4426950408889634f;
  a.raw = raw;
  a.raw_stride = raw_stride;
  a.raw_group = cols * raw_stride;
  a.chunks = (int)chunks;
  a.lists = so_lists(cols, items, chunks);
  if (workgroups > 0 && a.lists > workgroups) a.lists = workgroups;
  a.per_list = (int)((cols + a.lists - 1) / a.lists * groups * chunks);
  a.sums = (float*)workspace;
  a.offs = a.sums + n;
  a.table = (SoChunk*)(a.offs + n);
  a.tickets = (unsigned*)(a.table + (int64_t)a.lists * a.per_list);
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(snapkv_once_setup_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, st, a, (long long)(n / 4),
                     (int)items);   // (n / 4 = 32 * items threads: enough for the lists' words as well)
  const int64_t want = workgroups > 0 ? workgroups : 2 * fc_compute_units(), most = (int64_t)a.lists * a.per_list;
  const int64_t wgs = (want < most ? want : most) / a.lists * a.lists;
  constexpr int lds = 256 + 2 * SO_SLOT + 2 * SO_WAVES * SO_KEYS * 4 + SO_WAVES * 128 + SO_RING * (int)sizeof(SoChunk) +
                      SO_CHUNKS_MAX * 4;
  static_assert(lds <= 80 * 1024 && sizeof(SoChunk) == 64, "two workgroups share a compute unit's LDS");
  if (keys->dtype == FC_BF16) {
    FC_ALLOW_LDS((snapkv_once_kernel<FC_BF16>), lds);
    hipLaunchKernelGGL((snapkv_once_kernel<FC_BF16>), dim3((unsigned)wgs), dim3(SO_THREADS), lds, st, a);
  } else {
    FC_ALLOW_LDS((snapkv_once_kernel<FC_F16>), lds);
    hipLaunchKernelGGL((snapkv_once_kernel<FC_F16>), dim3((unsigned)wgs), dim3(SO_THREADS), lds, st, a);
  }
  FC_CHECK_LAUNCH(who);
  return FC_OK;
}
