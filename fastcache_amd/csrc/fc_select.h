// Exact top-k selection of one row by one workgroup, shared by the kernels that select: MSB-first radix select over
// order-preserving 32-bit keys, then an ordered pass that emits the kept positions in ascending order.
#pragma once
#include "fc_common.h"

#define TK_BINS 256

// order-preserving key of a score: larger score, larger key
__device__ __forceinline__ unsigned tk_key(float f) {
  unsigned u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0xffffffffu;  // NaN ranks above +inf
  if ((u & 0x7fffffffu) == 0u) u = 0u;                      // -0 == +0
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// LDS words the selection needs beside the keys
template <int THREADS>
struct TkShared {
  unsigned hist[TK_BINS];
  unsigned wave_tot[TK_BINS / FC_WAVE];
  unsigned sel_bin, sel_remaining;
  unsigned w_eq[THREADS / FC_WAVE], w_gt[THREADS / FC_WAVE];
};

// The kk largest of the n keys key_at(0..n-1), 0 < kk < n, ties to the lowest index: emit(position, index) is called
// once per kept index, positions 0..kk-1 in ascending index order.  Every thread of the workgroup (THREADS of them,
// at least 256) calls this; it synchronises the workgroup several times, the first time before it touches `sh`.
template <int THREADS, typename KeyAt, typename Emit>
__device__ __forceinline__ void tk_select_row(TkShared<THREADS>& sh, KeyAt key_at, int n, int kk, Emit emit) {
  constexpr int WAVES = THREADS / FC_WAVE;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  unsigned prefix = 0, mask = 0, remaining = (unsigned)kk;
  for (int shift = 24; shift >= 0; shift -= 8) {
    if (tid < TK_BINS) sh.hist[tid] = 0;
    __syncthreads();
    for (int i0 = 0; i0 < n; i0 += THREADS) {
      const int i = i0 + tid;
      const unsigned u = i < n ? key_at(i) : 0u;
      bool todo = i < n && (u & mask) == prefix;
      const unsigned bin = (u >> shift) & 255u;
      // Scores of one row share their leading bits, so most lanes of a wavefront hit the same bin in the
      // first passes and their atomics would serialise: the two most common bins are counted with a
      // ballot and one atomic each, what is left goes through per-lane atomics.
#pragma unroll
      for (int rep = 0; rep < 2; ++rep) {
        const unsigned long long act = __ballot(todo);
        if (act == 0ull) break;
        const int leader = __ffsll((long long)act) - 1;
        const unsigned lb = __shfl(bin, leader, 64);
        const unsigned long long same = __ballot(todo && bin == lb);
        if (lane == leader) atomicAdd(&sh.hist[lb], (unsigned)__popcll(same));
        todo = todo && bin != lb;
      }
      if (todo) atomicAdd(&sh.hist[bin], 1u);
    }
    __syncthreads();
    // suffix sums over bins: thread t < 256 owns bin 255 - t
    unsigned h = 0, incl = 0;
    if (tid < TK_BINS) {
      h = sh.hist[TK_BINS - 1 - tid];
      incl = h;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        unsigned up = __shfl_up(incl, o, 64);
        if (lane >= o) incl += up;
      }
      if (lane == 63) sh.wave_tot[wave] = incl;
    }
    __syncthreads();
    if (tid < TK_BINS) {
      unsigned base = 0;
      for (int w = 0; w < wave; ++w) base += sh.wave_tot[w];
      incl += base;
      const unsigned excl = incl - h;  // elements in strictly larger bins
      if (excl < remaining && remaining <= incl) {
        sh.sel_bin = (unsigned)(TK_BINS - 1 - tid);
        sh.sel_remaining = remaining - excl;
      }
    }
    __syncthreads();
    prefix |= sh.sel_bin << shift;
    mask |= 255u << shift;
    remaining = sh.sel_remaining;
    __syncthreads();
  }
  const unsigned T = prefix;
  const unsigned need = remaining;  // how many keys == T to keep (>= 1)

  // each wave owns a contiguous segment, walked 64 keys at a time
  const int seg = (((n + WAVES - 1) / WAVES) + 63) & ~63;
  const int beg = wave * seg;
  const int end = min(n, beg + seg);
  unsigned eq_cnt = 0, gt_cnt = 0;
  for (int i0 = beg; i0 < end; i0 += 64) {
    int i = i0 + lane;
    unsigned u = (i < end) ? key_at(i) : 0u;
    bool live = i < end;
    eq_cnt += __popcll(__ballot(live && u == T));
    gt_cnt += __popcll(__ballot(live && u > T));
  }
  if (lane == 0) { sh.w_eq[wave] = eq_cnt; sh.w_gt[wave] = gt_cnt; }
  __syncthreads();
  unsigned eq_seen = 0, out_pos = 0;
  {
    unsigned eq_run = 0;
    for (int w = 0; w < wave; ++w) {
      unsigned take = need > eq_run ? min(need - eq_run, sh.w_eq[w]) : 0u;
      out_pos += sh.w_gt[w] + take;
      eq_run += sh.w_eq[w];
    }
    eq_seen = eq_run;
  }
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int i0 = beg; i0 < end; i0 += 64) {
    int i = i0 + lane;
    bool live = i < end;
    unsigned u = live ? key_at(i) : 0u;
    bool is_eq = live && u == T;
    unsigned long long eqb = __ballot(is_eq);
    unsigned my_rank = eq_seen + __popcll(eqb & lt_mask);
    bool sel = live && (u > T || (is_eq && my_rank < need));
    unsigned long long sb = __ballot(sel);
    if (sel) emit((int)(out_pos + __popcll(sb & lt_mask)), i);
    eq_seen += __popcll(eqb);
    out_pos += __popcll(sb);
  }
}

// orders a wavefront's LDS writes before its following LDS reads of other lanes' data, and the other way round
__device__ __forceinline__ void tk_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lane exchanges are steps of a selection's chain, and one of two digit passes has 26 of them: as DPP steps and lane reads
// instead of permutes through LDS (and the counts of the wavefronts ahead summed by lanes instead of one after the other) a
// hook takes 0.9 to 1.8 us less: Knorm, 8 columns of 1000 keys 11.4 -> 10.5, 16 of 4000 19.6 -> 18.0, 4 of 9000 24.8 -> 23.0;
// SnapKV, 8 of 1000 24.4 -> 22.9, 32 of 4096 50.5 -> 49.3.
// `v` of the lane CTRL names, `none` where CTRL names no lane or ROWS (a bit per row of 16 lanes) excludes this one
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ unsigned tk_dpp(unsigned none, unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp((int)none, (int)v, CTRL, ROWS, 0xf, false);
}
// op over lanes 0 .. own: the rows of 16 lanes by shifts, then the last lane of row 0 and 2 into the row behind, of row 1 into
// the two rows behind
template <typename Op>
__device__ __forceinline__ unsigned tk_wave_scan(unsigned none, unsigned v, Op op) {
  v = op(v, tk_dpp<0x111>(none, v));         // row_shr:1
  v = op(v, tk_dpp<0x112>(none, v));
  v = op(v, tk_dpp<0x114>(none, v));
  v = op(v, tk_dpp<0x118>(none, v));
  v = op(v, tk_dpp<0x142, 0xa>(none, v));    // row_bcast:15
  v = op(v, tk_dpp<0x143, 0xc>(none, v));    // row_bcast:31
  return v;
}
__device__ __forceinline__ unsigned tk_read_lane(unsigned v, int lane) {
  return (unsigned)__builtin_amdgcn_readlane((int)v, lane);
}

// Smallest and largest of an unsigned value over the wavefront, wave-uniform.
__device__ __forceinline__ void tk_wave_range(unsigned& lo, unsigned& hi) {
  lo = tk_read_lane(tk_wave_scan(0xffffffffu, lo, [](unsigned a, unsigned b) { return min(a, b); }), 63);
  hi = tk_read_lane(tk_wave_scan(0u, hi, [](unsigned a, unsigned b) { return max(a, b); }), 63);
}

// The same selection with the row's keys held in registers: every wavefront owns a contiguous segment of the row and
// its lane l the keys segment + e * 64 + l, e < KPT, read and converted ONCE (key_at is called once per key), so the
// digit passes and the ordered pass cost a handful of vector instructions per key instead of an LDS read and a
// conversion each.  Needs n <= THREADS * KPT.
// A column's selection is a chain of short steps between workgroup barriers, and inside a kernel whose other
// workgroups keep the compute unit busy every barrier costs about a microsecond, so the passes are arranged for few
// of them: one per digit pass (every wavefront scans the 256 bins for itself instead of sharing a scan through LDS;
// three histograms in rotation, so that clearing the next one needs no barrier of its own) and one before the
// ordered pass.  The digits are those of the key's distance from the row's smallest key, counted from the highest bit
// that differs within the row: the scores of a row share their leading bits, and digits cut at fixed places would put
// most keys of the first passes into one or two bins, where their LDS atomics queue up.  The digit passes stop as
// soon as every key left in the threshold bin is kept (then no tie has to be ranked): rows of distinct scores end
// after two passes.
// Keys never produced by tk_key (0) stand for "no key here".
template <int THREADS>
struct TkSharedRegs {
  unsigned hist[3][TK_BINS];
  unsigned w_eq[THREADS / FC_WAVE], w_gt[THREADS / FC_WAVE];
  unsigned w_lo[THREADS / FC_WAVE], w_hi[THREADS / FC_WAVE];
};

// Where the keys of a row lie: key e of this lane is row position pos(e), if e < live and pos(e) < end.
template <int THREADS>
struct TkSegment {
  int beg, end, live;
  __device__ __forceinline__ explicit TkSegment(int n) {
    constexpr int WAVES = THREADS / FC_WAVE;
    const int seg = (((n + WAVES - 1) / WAVES) + 63) & ~63;   // <= KPT * 64 by the caller's bound
    beg = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) * seg;
    end = min(n, beg + seg);
    live = end > beg ? (end - beg + 63) >> 6 : 0;             // wave-uniform: 64-key groups of this wavefront
  }
  __device__ __forceinline__ int pos(int e) const { return beg + e * 64 + ((int)threadIdx.x & 63); }
};

// A lane's keys: REGS in registers and, of more, the rest in LDS (`rest`, TK_LDS_KEYS(THREADS, KPT) words).  Loops over
// the keys are unrolled, so which of the two a key is in is decided at compile time.
#define TK_REGS(KPT) ((KPT) <= 40 ? (KPT) : 40)
#define TK_LDS_KEYS(THREADS, KPT) (((KPT) - TK_REGS(KPT)) * (THREADS))
template <int THREADS, int KPT>
struct TkKeys {
  unsigned reg[TK_REGS(KPT)];
  unsigned* mine;
  __device__ __forceinline__ explicit TkKeys(unsigned* rest) {
    mine = rest + ((int)threadIdx.x >> 6) * (KPT - TK_REGS(KPT)) * 64 + ((int)threadIdx.x & 63);
  }
  __device__ __forceinline__ unsigned get(int e) const { return e < TK_REGS(KPT) ? reg[e < TK_REGS(KPT) ? e : 0] : mine[(e - TK_REGS(KPT)) * 64]; }
  __device__ __forceinline__ void set(int e, unsigned v) {
    if (e < TK_REGS(KPT)) reg[e < TK_REGS(KPT) ? e : 0] = v;
    else mine[(e - TK_REGS(KPT)) * 64] = v;
  }
};

// The number of live key groups as a value of its own, for one unrolled loop: taken from the common variable, the compiler
// would keep a lane mask for each of the comparisons from loop to loop, in spilled registers.
__device__ __forceinline__ int tk_live_here(int live) {
  asm volatile("" : "+s"(live));
  return live;
}

// Ends every eighth key of an unrolled loop of a long row: loads of more keys at once than that would be kept in registers
// that the keys need.
#define TK_EIGHT(KPT, e) do { if ((KPT) > TK_REGS(KPT) && ((e) & 7) == 7) __builtin_amdgcn_sched_barrier(0); } while (0)

// ... with the keys already there (0 where there is none)
template <int THREADS, int KPT, typename Emit>
__device__ __forceinline__ void tk_select_loaded(TkSharedRegs<THREADS>& sh, const TkSegment<THREADS>& sg, TkKeys<THREADS, KPT>& key,
                                                 int kk, Emit emit) {
  constexpr int WAVES = THREADS / FC_WAVE;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  unsigned lo = 0xffffffffu, hi = 0;
#pragma unroll
  for (int e = 0; e < KPT; ++e) {
    const unsigned u = key.get(e);
    if (u != 0u) lo = min(lo, u);
    hi = max(hi, u);
    TK_EIGHT(KPT, e);
  }
  tk_wave_range(lo, hi);
  for (int i = tid; i < 2 * TK_BINS; i += THREADS) (&sh.hist[0][0])[i] = 0;   // histograms of the first two passes
  if (lane == 0) { sh.w_lo[wave] = lo; sh.w_hi[wave] = hi; }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    lo = min(lo, sh.w_lo[w]);
    hi = max(hi, sh.w_hi[w]);
  }
  // from here on a key stands as its distance from the smallest one, plus one (0 stays "no key"); the largest key is
  // below 2^32 - 1 above the smallest, whose own distance is at least tk_key(-inf), so nothing wraps
#pragma unroll
  for (int e = 0; e < KPT; ++e) {
    const unsigned u = key.get(e);
    key.set(e, u != 0u ? u - lo + 1u : 0u);
    TK_EIGHT(KPT, e);
  }
  const unsigned span = hi - lo + 1u;
  unsigned prefix = 0, mask = 0, remaining = (unsigned)kk;
  bool whole_bin = false;   // every key that matches the prefix so far is kept
  int top = 32 - __clz((int)span);   // bits not yet looked at
  for (int pass = 0; top > 0 && !whole_bin; ++pass) {
    const int shift = max(top - 8, 0);
    const unsigned dmask = (1u << (top - shift)) - 1u;
    top = shift;
    unsigned* hist = sh.hist[pass % 3];
    if (pass >= 1)   // the histogram of the pass after this one; its last readers are two barriers back
      for (int i = tid; i < TK_BINS; i += THREADS) sh.hist[(pass + 1) % 3][i] = 0;
    const int live_e = tk_live_here(sg.live);
#pragma unroll
    for (int e = 0; e < KPT; ++e) {
      if (e < live_e) {
        const unsigned u = key.get(e);
        if (u != 0u && (u & mask) == prefix) atomicAdd(&hist[(u >> shift) & dmask], 1u);
      }
      TK_EIGHT(KPT, e);
    }
    __syncthreads();
    // every wavefront for itself: lane t holds bins 255 - 4t .. 252 - 4t (descending), suffix sums over the 256 bins
    unsigned h4[4], incl = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      h4[r] = hist[TK_BINS - 1 - (4 * lane + r)];
      incl += h4[r];
    }
    const unsigned own = incl;
    incl = tk_wave_scan(0u, incl, [](unsigned a, unsigned b) { return a + b; });
    unsigned excl = incl - own;   // keys in bins above this lane's four
    int found = -1;
    unsigned left = 0, size = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (found < 0 && excl < remaining && remaining <= excl + h4[r]) {
        found = TK_BINS - 1 - (4 * lane + r);
        left = remaining - excl;
        size = h4[r];
      }
      excl += h4[r];
    }
    const unsigned long long who = __ballot(found >= 0);   // exactly one lane
    const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)who) - 1);
    const unsigned bin = tk_read_lane((unsigned)found, src);
    remaining = tk_read_lane(left, src);
    whole_bin = tk_read_lane(size, src) == remaining;
    prefix |= bin << shift;
    mask |= dmask << shift;
  }
  // kept: keys whose masked bits exceed the prefix, and of those that equal it the first `remaining` by index
  // (all of them when whole_bin; after the last pass the masked bits are the whole key)
  const unsigned T = prefix;
  const unsigned need = remaining;
  unsigned eq_cnt = 0, gt_cnt = 0;
  const int live_c = tk_live_here(sg.live);
#pragma unroll
  for (int e = 0; e < KPT; ++e) {
    if (e < live_c) {
      const unsigned u = key.get(e), m = u & mask;
      eq_cnt += __popcll(__ballot(u != 0u && m == T));
      gt_cnt += __popcll(__ballot(u != 0u && m > T));
    }
    TK_EIGHT(KPT, e);
  }
  if (lane == 0) { sh.w_eq[wave] = eq_cnt; sh.w_gt[wave] = gt_cnt; }
  __syncthreads();
  // what the wavefronts before this one hold, a lane each: of their equal keys all are kept while there is need
  static_assert(WAVES <= 16, "one row of lanes holds the wavefronts' counts");
  unsigned eq_seen = lane < wave ? sh.w_eq[lane & (WAVES - 1)] : 0u, out_pos = lane < wave ? sh.w_gt[lane & (WAVES - 1)] : 0u;
  const auto add = [](unsigned a, unsigned b) { return a + b; };
  eq_seen = tk_read_lane(tk_wave_scan(0u, eq_seen, add), 15);
  out_pos = tk_read_lane(tk_wave_scan(0u, out_pos, add), 15) + min(need, eq_seen);
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int live_o = tk_live_here(sg.live);
  int first = sg.pos(0);
  asm volatile("" : "+v"(first));   // likewise: the positions are computed again, not kept from when the keys were read
#pragma unroll
  for (int e = 0; e < KPT; ++e) {
    if (e < live_o) {
      const unsigned u = key.get(e), m = u & mask;
      const bool is_eq = u != 0u && m == T;
      const unsigned long long eqb = __ballot(is_eq);
      const unsigned my_rank = eq_seen + __popcll(eqb & lt_mask);
      const bool sel = u != 0u && (m > T || (is_eq && my_rank < need));
      const unsigned long long sb = __ballot(sel);
      if (sel) emit((int)(out_pos + __popcll(sb & lt_mask)), first + e * 64);
      eq_seen += __popcll(eqb);
      out_pos += __popcll(sb);
    }
    TK_EIGHT(KPT, e);
  }
}

template <int THREADS, int KPT, typename KeyAt, typename Emit>
__device__ __forceinline__ void tk_select_row_regs(TkSharedRegs<THREADS>& sh, unsigned* rest, KeyAt key_at, int n, int kk, Emit emit) {
  const TkSegment<THREADS> sg(n);
  TkKeys<THREADS, KPT> key(rest);
#pragma unroll
  for (int e = 0; e < KPT; ++e) {
    const int i = sg.pos(e);
    if constexpr (KPT > TK_REGS(KPT)) {   // always a load, of an existing key: 72 lane masks would not fit the registers
      const unsigned u = key_at(min(i, n - 1));
      key.set(e, e < sg.live && i < sg.end ? u : 0u);
    } else {
      key.set(e, (e < sg.live && i < sg.end) ? key_at(i) : 0u);
    }
    TK_EIGHT(KPT, e);
  }
  tk_select_loaded<THREADS, KPT>(sh, sg, key, kk, emit);
}

// LDS of whichever form of the selection a kernel ends up calling
template <int THREADS>
union TkArea {
  TkShared<THREADS> lds_keys;
  TkSharedRegs<THREADS> reg_keys;
};
