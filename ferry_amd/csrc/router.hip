// Router: fp32 softmax + top-k (+ renormalisation, scale, bf16 cast), one wavefront per row.
//
// Reference: ferry/model.py:141-146 (Qwen3 hook) and the greedy DeepSeek-V2 gate feeding
// ferry/model.py:151-157.  torch.topk there selects on the fp32 probabilities with torch's
// CPU algorithm (std::nth_element + std::sort of the first k-1 entries when k*64 > E, else
// std::partial_sort; comparator on values only, NaN first).  Two distinct logits can round to
// the same probability, which torch then treats as a tie, so the selection must run on the
// probabilities themselves, bit for bit.  The kernel therefore computes them exactly as
// torch's CPU softmax does (ATen/native/cpu/SoftMaxKernel.cpp, vectorized last-dim path):
//   m = max of the row; e_i = exp(x_i - m) with SLEEF's expf_u10 (the exp of
//   Vectorized<float>, ATen/cpu/vec/vec512/vec512_float.h:307-309), restated in sleef_expf;
//   s = their sum in vec::reduce_all's order for 16-lane vectors (ATen/cpu/vec/
//   functional_base.h:185-203 and the AVX-512 VecReduceAllSIMD at :78-98); p_i = e_i * (1/s).
// The renormalising sum of the Qwen3 hook, w.sum(-1), follows torch's CPU sum kernel for a
// short contiguous last dimension (see topk_weight_sum).  Both orders were identified on
// torch 2.10's CPU build and are checked against it bit for bit by the tests.  A row holding
// a NaN or +inf logit has all-NaN probabilities, i.e. all elements compare equal.
// Selection runs on order-preserving uint32 keys of the probabilities.
//
// Sorted rows without ties have one possible result, which k wavefront arg-max rounds find
// (distinct_select; taken first where ties are rare, see ferry_router_topk).  Every other row
// replays the CPU algorithm exactly, on a whole wavefront:
//  * introselect: the row is held 1, 2 or 4 keys per lane (position p = 64 * slot + lane); each
//    median-of-3 / Hoare partition step is evaluated in one pass -- the j-th left stop (ascending
//    position holding a key <= pivot) is exchanged with the j-th right stop (descending position
//    holding a key >= pivot) while left < right, which every lane decides from the two ranks of
//    its position (ballots), so a step costs one LDS round trip instead of a serial scan;
//  * the final std::sort of the first k-1 entries (k - 1 <= 16) is an insertion sort, i.e.
//    a stable descending sort, computed by ranking;
//  * the rare remainder (introselect depth limit reached -> heap select; partial_sort regime
//    k*64 <= n; k - 1 > 16) runs the sequential algorithm on lane 0 over the row in LDS.
//
// A decode call is bound by this chain's latency (one wavefront a row, a step of it about 1,000
// clocks), a large batch by its instruction issue.  With the stops' ranks staged in LDS and the
// arg-max rounds first for every sorted row, 16 rows (k = 8 of 128, bf16) took 10.7 us, 8192 rows 24.0
// and, unsorted (k = 6 of 64, fp32), 256 rows 7.4 us and 65,536 rows 108 us; now 7.6, 19.7, 5.4 and
// 68.8 us.
#include "common.h"

#include <type_traits>

// every rounding step below is the reference's: no contraction of a*b+c into one FMA
#pragma clang fp contract(off)

namespace ferry {
namespace {

constexpr int kMaxE = 256;  // 4 keys per lane
constexpr int kMaxK = 32;
constexpr int kWaves = 4;

struct Pair {
  uint32_t v;  // ordered key: larger key = "before" in the torch comparator
  int32_t i;
};

__device__ __forceinline__ bool before(const Pair& x, const Pair& y) { return x.v > y.v; }

// order-preserving key of a float: -0 == +0, NaN above +inf (all NaNs equal)
__device__ __forceinline__ uint32_t ordered_key(float f) {
  if (f != f) return 0xffffffffu;
  if (f == 0.f) f = 0.f;
  uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// ---------------------------------------------------------------------------------------------
// Sequential restatement (lane 0, row in LDS): libstdc++ introselect / introsort / heap select
// ---------------------------------------------------------------------------------------------
__device__ void push_heap_(Pair* a, int hole, int top, Pair value) {
  int parent = (hole - 1) / 2;
  while (hole > top && before(a[parent], value)) {
    a[hole] = a[parent];
    hole = parent;
    parent = (hole - 1) / 2;
  }
  a[hole] = value;
}
__device__ void adjust_heap_(Pair* a, int hole, int len, Pair value) {
  const int top = hole;
  int child = hole;
  while (child < (len - 1) / 2) {
    child = 2 * (child + 1);
    if (before(a[child], a[child - 1])) child--;
    a[hole] = a[child];
    hole = child;
  }
  if ((len & 1) == 0 && child == (len - 2) / 2) {
    child = 2 * (child + 1);
    a[hole] = a[child - 1];
    hole = child - 1;
  }
  push_heap_(a, hole, top, value);
}
__device__ void make_heap_(Pair* a, int len) {
  if (len < 2) return;
  int parent = (len - 2) / 2;
  for (;;) {
    Pair value = a[parent];
    adjust_heap_(a, parent, len, value);
    if (parent == 0) return;
    parent--;
  }
}
__device__ void pop_heap_(Pair* a, int len, int result) {
  Pair value = a[result];
  a[result] = a[0];
  adjust_heap_(a, 0, len, value);
}
__device__ void heap_select_(Pair* a, int middle, int last) {
  make_heap_(a, middle);
  for (int i = middle; i < last; ++i)
    if (before(a[i], a[0])) pop_heap_(a, middle, i);
}
__device__ void sort_heap_(Pair* a, int len) {
  while (len > 1) {
    --len;
    pop_heap_(a, len, len);
  }
}
__device__ void unguarded_linear_insert_(Pair* a, int last) {
  Pair val = a[last];
  int next = last - 1;
  while (before(val, a[next])) {
    a[last] = a[next];
    last = next;
    --next;
  }
  a[last] = val;
}
__device__ void insertion_sort_(Pair* a, int first, int last) {
  if (first == last) return;
  for (int i = first + 1; i != last; ++i) {
    if (before(a[i], a[first])) {
      Pair val = a[i];
      for (int j = i; j > first; --j) a[j] = a[j - 1];
      a[first] = val;
    } else {
      unguarded_linear_insert_(a, i);
    }
  }
}
__device__ __forceinline__ void swap_(Pair* a, int x, int y) {
  Pair t = a[x];
  a[x] = a[y];
  a[y] = t;
}
__device__ void move_median_to_first_(Pair* a, int result, int x, int y, int z) {
  if (before(a[x], a[y])) {
    if (before(a[y], a[z]))
      swap_(a, result, y);
    else if (before(a[x], a[z]))
      swap_(a, result, z);
    else
      swap_(a, result, x);
  } else if (before(a[x], a[z])) {
    swap_(a, result, x);
  } else if (before(a[y], a[z])) {
    swap_(a, result, z);
  } else {
    swap_(a, result, y);
  }
}
__device__ int unguarded_partition_(Pair* a, int first, int last, int pivot) {
  const Pair p = a[pivot];
  for (;;) {
    while (before(a[first], p)) ++first;
    --last;
    while (before(p, a[last])) --last;
    if (!(first < last)) return first;
    swap_(a, first, last);
    ++first;
  }
}
__device__ int partition_pivot_(Pair* a, int first, int last) {
  const int mid = first + (last - first) / 2;
  move_median_to_first_(a, first, first + 1, mid, last - 1);
  return unguarded_partition_(a, first + 1, last, first);
}
__device__ __forceinline__ int lg2_(int n) { return 31 - __clz(n); }

// std::sort of a[first, last): introsort loop down to ranges of 16, then insertion sort.
// stk holds 3 * kStack ints of LDS for the pending right-hand ranges.
constexpr int kStack = 16;
__device__ void sort_(Pair* a, int first, int last, int* stk) {
  if (last - first <= 1) return;
  int sp = 0;
  stk[0] = first;
  stk[1] = last;
  stk[2] = lg2_(last - first) * 2;
  ++sp;
  while (sp > 0) {
    --sp;
    int f = stk[3 * sp], l = stk[3 * sp + 1], depth = stk[3 * sp + 2];
    while (l - f > 16) {
      if (depth == 0) {
        heap_select_(a + f, l - f, l - f);
        sort_heap_(a + f, l - f);
        break;
      }
      --depth;
      const int cut = partition_pivot_(a, f, l);
      // the reference recurses on [cut, l) and loops on [f, cut): disjoint ranges, so the
      // processing order does not change the result.  Ranges here hold at most kMaxK - 1
      // elements, so the pending stack stays far below kStack entries.
      if (sp < kStack) {
        stk[3 * sp] = cut;
        stk[3 * sp + 1] = l;
        stk[3 * sp + 2] = depth;
        ++sp;
      }
      l = cut;
    }
  }
  if (last - first > 16) {
    insertion_sort_(a, first, first + 16);
    for (int i = first + 16; i != last; ++i) unguarded_linear_insert_(a, i);
  } else {
    insertion_sort_(a, first, last);
  }
}

// ---------------------------------------------------------------------------------------------
// Wavefront-parallel restatement
// ---------------------------------------------------------------------------------------------
struct WaveScratch {
  Pair stage[kMaxE];
  float prob[kMaxE];
  int32_t sel[kMaxK];
  int32_t stack[3 * kStack];
};

__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// value at uniform position p = 64 * slot + lane: read lane (p & 63) of each of the four
// registers and select by slot (selecting between register values, not array elements, keeps
// the arrays out of scratch memory)
template <int NS>
__device__ __forceinline__ uint32_t key_at(const uint32_t (&k)[NS], int p) {
  const int l = p & 63, s = p >> 6;
  uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)k[0], l);
#pragma unroll
  for (int q = 1; q < NS; ++q) {
    const uint32_t rq = (uint32_t)__builtin_amdgcn_readlane((int)k[q], l);
    r = s == q ? rq : r;
  }
  return r;
}
template <int NS>
__device__ __forceinline__ int32_t idx_at(const int32_t (&ix)[NS], int p) {
  const int l = p & 63, s = p >> 6;
  int32_t r = __builtin_amdgcn_readlane(ix[0], l);
#pragma unroll
  for (int q = 1; q < NS; ++q) {
    const int32_t rq = __builtin_amdgcn_readlane(ix[q], l);
    r = s == q ? rq : r;
  }
  return r;
}
template <int NS>
__device__ __forceinline__ void set_at(uint32_t (&k)[NS], int32_t (&ix)[NS], int p, uint32_t kv,
                                       int32_t iv) {
  const int s = p >> 6;
  // per-slot selects by a scalar mask (no indexed store, which would move the arrays to scratch)
#pragma unroll
  for (int q = 0; q < NS; ++q) {
    const bool hit = __builtin_amdgcn_inverse_ballot_w64(NS == 1 || q == s ? 1ull << (p & 63) : 0ull);
    k[q] = hit ? kv : k[q];
    ix[q] = hit ? iv : ix[q];
  }
}

// bits of the positions [lo, hi) that lie in slot s (lo, hi wave-uniform)
__device__ __forceinline__ uint64_t slot_mask(int lo, int hi, int s) {
  const int a = lo - 64 * s, b = hi - 64 * s;
  const uint64_t below_b = b >= 64 ? ~0ull : (b <= 0 ? 0ull : (1ull << b) - 1);
  const uint64_t below_a = a >= 64 ? ~0ull : (a <= 0 ? 0ull : (1ull << a) - 1);
  return below_b & ~below_a;
}
__device__ __forceinline__ int lane_rank(uint64_t m) {   // set bits of m below this lane
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}

// One std::__unguarded_partition_pivot step on [first, last); returns the cut.
//
// The j-th left stop L_j (ascending position in [first + 1, last) holding a key <= pivot) is
// exchanged with the j-th right stop R_j (descending position in [first, last) holding a key >=
// pivot) while L_j < R_j.  A left stop of rank j at position p is exchanged iff more than j right
// stops lie above p (R_j > p), a right stop of rank j iff more than j left stops lie below it, so
// every lane decides from two ranks, with ballots and scalar bit operations only; the exchanged
// keys meet in LDS at their rank.  The cut is the first left stop not exchanged or the last right
// stop exchanged, whichever is lower.
template <int NS>
__device__ __forceinline__ int wave_partition_pivot(uint32_t (&k)[NS], int32_t (&ix)[NS], int first, int last,
                                    int lane, WaveScratch& ws) {
  const int mid = first + (last - first) / 2;
  uint32_t piv;
  {
    // __move_median_to_first(first, first + 1, mid, last - 1)
    const int a = first + 1, b = mid, c = last - 1;
    const uint32_t ka = key_at(k, a), kb = key_at(k, b), kc = key_at(k, c);
    int m;
    if (ka > kb) {
      m = (kb > kc) ? b : (ka > kc) ? c : a;
    } else {
      m = (ka > kc) ? a : (kb > kc) ? c : b;
    }
    piv = m == a ? ka : (m == b ? kb : kc);
    const uint32_t kf = key_at(k, first);
    const int32_t xf = idx_at(ix, first), xm = idx_at(ix, m);
    set_at(k, ix, m, kf, xf);
    set_at(k, ix, first, piv, xm);
  }
  uint64_t bl[NS], bg[NS];
  int ng = 0;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    bl[s] = __ballot(k[s] <= piv) & slot_mask(first + 1, last, s);
    bg[s] = __ballot(k[s] >= piv) & slot_mask(first, last, s);
    ng += __popcll(bg[s]);
  }
  uint64_t sl[NS], sr[NS];   // exchanged left / right stops
  int rank[NS];              // of an exchanged stop, on its side
  int below_l = 0, below_g = 0;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int left = below_l + lane_rank(bl[s]);              // left stops below
    const int upto = below_g + lane_rank(bg[s]);              // right stops below
    const bool le = __builtin_amdgcn_inverse_ballot_w64(bl[s]), ge = __builtin_amdgcn_inverse_ballot_w64(bg[s]);
    const int right = ng - upto - (ge ? 1 : 0);               // right stops above
    sl[s] = __ballot(le && right > left);
    sr[s] = __ballot(ge && left > right);
    rank[s] = left < right ? left : right;
    below_l += __popcll(bl[s]);
    below_g += __popcll(bg[s]);
  }
  int lnext = 0x7fffffff, rprev = 0x7fffffff;
#pragma unroll
  for (int s = NS - 1; s >= 0; --s) {
    const uint64_t l = bl[s] & ~sl[s];
    if (l) lnext = 64 * s + __ffsll((long long)l) - 1;
    if (sr[s]) rprev = 64 * s + __ffsll((long long)sr[s]) - 1;
  }
  int cut = lnext < rprev ? lnext : rprev;
  // the median-of-3 pivot guarantees a left stop inside the range, so cut lies in
  // [first + 1, last - 1]; the clamp only keeps indices in range should that ever fail
  cut = cut < first + 1 ? first + 1 : (cut > last - 1 ? last - 1 : cut);
  if (rprev != 0x7fffffff) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const bool l = __builtin_amdgcn_inverse_ballot_w64(sl[s]), r = __builtin_amdgcn_inverse_ballot_w64(sr[s]);
      if (l || r) ws.stage[rank[s] + (r ? 32 * NS : 0)] = Pair{k[s], ix[s]};
    }
    wave_sync_lds();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const bool l = __builtin_amdgcn_inverse_ballot_w64(sl[s]), r = __builtin_amdgcn_inverse_ballot_w64(sr[s]);
      if (l || r) {
        const Pair p = ws.stage[rank[s] + (l ? 32 * NS : 0)];
        k[s] = p.v;
        ix[s] = p.i;
      }
    }
    wave_sync_lds();
  }
  return cut;
}

// stable descending sort of the uniform positions [first, last) (last - first <= 16):
// the result of std::__insertion_sort on that range
template <int NS>
__device__ __forceinline__ void wave_insertion_sort(uint32_t (&k)[NS], int32_t (&ix)[NS], int first, int last,
                                    int lane, WaveScratch& ws) {
  if (last - first <= 1) return;
  int dest[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) dest[s] = 0;
  for (int q = first; q < last; ++q) {
    const uint32_t kq = key_at(k, q);
#pragma unroll
    for (int s = 0; s < NS; ++s) dest[s] += (kq > k[s]) || (kq == k[s] && q < s * 64 + lane);
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int pos = s * 64 + lane;
    if (pos >= first && pos < last) ws.stage[dest[s]] = Pair{k[s], ix[s]};
  }
  wave_sync_lds();
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int pos = s * 64 + lane;
    if (pos >= first && pos < last) {
      const Pair p = ws.stage[pos - first];
      k[s] = p.v;
      ix[s] = p.i;
    }
  }
  wave_sync_lds();
}

// The partition step and the insertion sort on slot 0 alone when [first, last) lies within
// positions 0..63 (the keys of the other slots are outside the range and stay as they are): the
// same steps, with half (or a quarter) of the per-slot work.  introselect narrows the range
// around position k - 1 < 64 within a step or two.
template <int NS>
__device__ __forceinline__ int partition_step(uint32_t (&k)[NS], int32_t (&ix)[NS], int first, int last,
                                              int lane, WaveScratch& ws) {
  if constexpr (NS > 1) {
    if (last <= 64) {
      uint32_t k0[1] = {k[0]};
      int32_t i0[1] = {ix[0]};
      const int cut = wave_partition_pivot(k0, i0, first, last, lane, ws);
      k[0] = k0[0];
      ix[0] = i0[0];
      return cut;
    }
  }
  return wave_partition_pivot(k, ix, first, last, lane, ws);
}
template <int NS>
__device__ __forceinline__ void insertion_step(uint32_t (&k)[NS], int32_t (&ix)[NS], int first, int last,
                                               int lane, WaveScratch& ws) {
  if constexpr (NS > 1) {
    if (last <= 64) {
      uint32_t k0[1] = {k[0]};
      int32_t i0[1] = {ix[0]};
      wave_insertion_sort(k0, i0, first, last, lane, ws);
      k[0] = k0[0];
      ix[0] = i0[0];
      return;
    }
  }
  wave_insertion_sort(k, ix, first, last, lane, ws);
}

// Exact CPU top-k selection of the row (n keys, position p = 64*s + lane): lane j < kk returns
// the j-th chosen index.
template <int NS>
__device__ __forceinline__ int exact_select(uint32_t (&k)[NS], int32_t (&ix)[NS], int n, int kk, bool sorted,
                             int lane, WaveScratch& ws) {
  const bool partial = kk * 64 <= n;                  // partial_sort regime
  const bool long_sort = sorted && kk - 1 > 16;       // a final sort longer than 16
  int first = 0, last = n, depth = lg2_(n) * 2;
  if (!partial && !long_sort) {
    // std::nth_element(first, first + kk - 1, last)
    const int nth = kk - 1;
    while (last - first > 3 && depth > 0) {
      --depth;
      const int cut = partition_step(k, ix, first, last, lane, ws);
      if (cut <= nth)
        first = cut;
      else
        last = cut;
    }
    if (last - first <= 3) {
      insertion_step(k, ix, first, last, lane, ws);
      if (sorted) insertion_step(k, ix, 0, kk - 1, lane, ws);
      return ix[0];
    }
  }
  // sequential on lane 0, from the state reached: the depth limit's heap select on [first, last),
  // or the whole of a partial_sort or of a selection with a long final sort
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int pos = s * 64 + lane;
    if (pos < n) ws.stage[pos] = Pair{k[s], ix[s]};
  }
  wave_sync_lds();
  if (lane == 0) {
    Pair* a = ws.stage;
    const int nth = kk - 1;
    if (partial) {
      heap_select_(a, kk, n);
      sort_heap_(a, kk);
    } else {
      while (last - first > 3 && depth > 0) {
        --depth;
        const int cut = partition_pivot_(a, first, last);
        if (cut <= nth)
          first = cut;
        else
          last = cut;
      }
      if (last - first > 3) {
        heap_select_(a + first, nth + 1 - first, last - first);
        swap_(a, first, nth);
      } else {
        insertion_sort_(a, first, last);
      }
      if (sorted) sort_(a, 0, kk - 1, ws.stack);
    }
    for (int j = 0; j < kk; ++j) ws.sel[j] = a[j].i;
  }
  wave_sync_lds();
  return ws.sel[lane < kk ? lane : 0];
}

// Wavefront reductions through DPP lane moves (a few cycles each, against an LDS round trip
// per step for __shfl_xor): quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror and row_mirror
// combine each row of 16 lanes in every lane; row_bcast:15 and row_bcast:31 then carry rows 0-2
// into the last row, and lane 63 holds the result, which readlane makes wave-uniform.
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ uint32_t dpp_u(uint32_t old, uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROW_MASK, 0xf, false);
}
__device__ __forceinline__ float dpp_asf(uint32_t v) { return __uint_as_float(v); }
__device__ __forceinline__ float wave_max(float v) {
  uint32_t u = __float_as_uint(v);
  v = fmaxf(v, dpp_asf(dpp_u<0xB1>(u, u)));
  u = __float_as_uint(v);
  v = fmaxf(v, dpp_asf(dpp_u<0x4E>(u, u)));
  u = __float_as_uint(v);
  v = fmaxf(v, dpp_asf(dpp_u<0x141>(u, u)));
  u = __float_as_uint(v);
  v = fmaxf(v, dpp_asf(dpp_u<0x140>(u, u)));
  u = __float_as_uint(v);
  v = fmaxf(v, dpp_asf(dpp_u<0x142, 0xa>(u, u)));
  u = __float_as_uint(v);
  v = fmaxf(v, dpp_asf(dpp_u<0x143, 0xc>(u, u)));
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), 63));
}
__device__ __forceinline__ uint32_t umax_(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t wave_max_u(uint32_t v) {
  v = umax_(v, dpp_u<0xB1>(v, v));
  v = umax_(v, dpp_u<0x4E>(v, v));
  v = umax_(v, dpp_u<0x141>(v, v));
  v = umax_(v, dpp_u<0x140>(v, v));
  v = umax_(v, dpp_u<0x142, 0xa>(v, v));
  v = umax_(v, dpp_u<0x143, 0xc>(v, v));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The selection where order and membership do not depend on the algorithm: kk arg-max rounds, lane
// j < kk receives the j-th largest key's index.  False (e undefined) where a round's largest key is
// not the only one, i.e. two of the kk + 1 largest are equal.  Keys of elements are above 0, the
// padding's 0.
template <int NS>
__device__ __forceinline__ bool distinct_select(const uint32_t (&k)[NS], int kk, int lane, int& e) {
  uint32_t cur[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) cur[s] = k[s];
  for (int r = 0; r < kk; ++r) {
    uint32_t most = cur[0];
#pragma unroll
    for (int s = 1; s < NS; ++s) most = umax_(most, cur[s]);
    most = wave_max_u(most);
    int hits = 0, pos = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const uint64_t hit = __ballot(cur[s] == most);
      hits += __popcll(hit);
      if (hit) pos = 64 * s + __ffsll((long long)hit) - 1;
      cur[s] = cur[s] == most ? 0u : cur[s];
    }
    if (hits != 1) return false;
    e = lane == r ? pos : e;
  }
  return true;
}

// SLEEF's single-precision exp with 1.0-ulp bound (xexpf of SLEEF 3, sleefsimdsp.c; the
// published Cody-Waite reduction by ln 2 in two parts, a degree-6 polynomial for e^s - 1 - s in
// Horner form with fused multiply-adds, and a two-step scaling by 2^q).  Restated from that
// method; checked against the SLEEF routine torch calls on all 2^32 fp32 inputs.
__device__ __forceinline__ float pow2i_(int q) { return __uint_as_float((uint32_t)(q + 0x7f) << 23); }
__device__ __forceinline__ float sleef_expf(float d) {
  if (d != d) return d;
  if (d < -104.f) return 0.f;
  if (d > 100.f) return INFINITY;
  const float kRln2 = 1.442695040888963407359924681001892137f;
  const float kL2U = 0.693145751953125f, kL2L = 1.428606765330187045e-06f;
  const int q = (int)__builtin_rintf(d * kRln2);
  float s = __builtin_fmaf((float)q, -kL2U, d);
  s = __builtin_fmaf((float)q, -kL2L, s);
  float u = 0.000198527617612853646278381f;
  u = __builtin_fmaf(u, s, 0.00139304355252534151077271f);
  u = __builtin_fmaf(u, s, 0.00833336077630519866943359f);
  u = __builtin_fmaf(u, s, 0.0416664853692054748535156f);
  u = __builtin_fmaf(u, s, 0.166666671633720397949219f);
  u = __builtin_fmaf(u, s, 0.5f);
  u = 1.0f + __builtin_fmaf(s * s, u, s);
  return u * pow2i_(q >> 1) * pow2i_(q - (q >> 1));
}

// Sum of e[0..n) (in LDS) in the order of torch's vec::reduce_all(+) for 16-lane vectors:
// n < 16: left to right; otherwise lane l of an accumulator vector adds e[16c + l] over the
// full chunks c in order, the tail chunk adds into its first n % 16 lanes, and the 16 lanes are
// combined by the halving butterfly (l + 8, then l + 4, l + 2, l + 1).  The chunks are read
// into registers at once; the butterfly moves lanes with DPP row shifts (row_shl:h, lane l
// reads lane l + h of its row of 16), and lane 0 holds the sum.  Wave-uniform result.
template <int NS>
__device__ __forceinline__ float torch_softmax_sum(const float* e, int n, int lane) {
  float acc = 0.f;
  if (n < 16) {
    if (lane == 0) {
      acc = e[0];
      for (int i = 1; i < n; ++i) acc += e[i];
    }
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(acc), 0));
  }
  const int full = n - n % 16;
  const int l16 = lane & 15;
  float v[4 * NS];
#pragma unroll
  for (int c = 0; c < 4 * NS; ++c) v[c] = 16 * c < full ? e[16 * c + l16] : 0.f;
  const float tail = l16 < n - full ? e[full + l16] : 0.f;
  acc = v[0];
#pragma unroll
  for (int c = 1; c < 4 * NS; ++c)
    if (16 * c < full) acc += v[c];
  if (l16 < n - full) acc += tail;
  uint32_t u = __float_as_uint(acc);
  acc += dpp_asf(dpp_u<0x108>(u, u));
  u = __float_as_uint(acc);
  acc += dpp_asf(dpp_u<0x104>(u, u));
  u = __float_as_uint(acc);
  acc += dpp_asf(dpp_u<0x102>(u, u));
  u = __float_as_uint(acc);
  acc += dpp_asf(dpp_u<0x101>(u, u));
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(acc), 0));
}

// torch's CPU sum over a contiguous last dimension of k <= 32 fp32 values (the renormalising
// w.sum(-1) of the Qwen3 hook), w_j held by lane j.  torch runs its 8-lane (AVX2) reduction
// kernel here: for k < 8 a scalar sum with four interleaved partial sums (partial j takes
// w[4i + j], the tail w[4 * (k / 4)..] goes into partial 0, then partial 0 + 1 + 2 + 3); for
// k >= 8, lane l of an 8-lane vector sums w[8i + l] over the k / 8 full vectors, and the result
// is the sum, left to right, of the scalar tail w[8 * (k / 8)..] followed by the 8 lanes.
// Identified by testing against torch's CPU sum for every k <= 32; wave-uniform result.
__device__ __forceinline__ float topk_weight_sum(float wv, int kk) {
  auto at = [&](int j) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(wv), j));
  };
  if (kk < 8) {
    float p0 = 0.f, p1 = 0.f, p2 = 0.f, p3 = 0.f;
    int i = 0;
    if (kk >= 4) {
      p0 = at(0);
      p1 = at(1);
      p2 = at(2);
      p3 = at(3);
      i = 4;
    }
    for (; i < kk; ++i) p0 += at(i);
    return ((p0 + p1) + p2) + p3;
  }
  const int nv = kk / 8;
  float acc = 0.f;
  for (int i = 8 * nv; i < kk; ++i) acc += at(i);
  for (int l = 0; l < 8; ++l) {
    float lane_sum = at(l);
    for (int v = 1; v < nv; ++v) lane_sum += at(8 * v + l);
    acc += lane_sum;
  }
  return acc;
}

template <typename T>
__device__ __forceinline__ float load_logit(const T* p);
template <>
__device__ __forceinline__ float load_logit<float>(const float* p) {
  return *p;
}
template <>
__device__ __forceinline__ float load_logit<bf16_t>(const bf16_t* p) {
  return bf16_to_f32(*p);
}

// ARGMAX: sorted rows of the introselect regime, which distinct_select tries first
template <typename T, int NS, bool ARGMAX>
__global__ __launch_bounds__(64 * kWaves) void router_kernel(
    const T* __restrict__ logits, int64_t tokens, int n, int kk, int renorm, float scale,
    int sorted, int64_t* __restrict__ idx_out, bf16_t* __restrict__ w_out,
    float* __restrict__ probs_out, int32_t* __restrict__ tie_rows) {
  __shared__ WaveScratch scratch[kWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  WaveScratch& ws = scratch[wave];
  for (int64_t row = (int64_t)blockIdx.x * kWaves + wave; row < tokens;
       row += (int64_t)gridDim.x * kWaves) {
    const T* src = logits + row * n;
    float x[NS];
    bool bad = false;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int e = s * 64 + lane;
      x[s] = e < n ? load_logit<T>(src + e) : -INFINITY;
      bad |= (e < n) && (x[s] != x[s] || x[s] == INFINITY);
    }
    const bool row_bad = __any(bad);  // softmax of this row is all NaN
    // softmax in fp32, rounding step for rounding step as torch's CPU kernel
    float m = x[0];
#pragma unroll
    for (int s = 1; s < NS; ++s) m = fmaxf(m, x[s]);
    m = wave_max(m);
    float ex[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int e = s * 64 + lane;
      ex[s] = e < n ? sleef_expf(x[s] - m) : 0.f;
      if (e < n) ws.prob[e] = ex[s];
    }
    wave_sync_lds();
    const float sum = torch_softmax_sum<NS>(ws.prob, n, lane);
    wave_sync_lds();
    const float inv = 1.0f / sum;
    uint32_t key[NS];
    int32_t ix[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int e = s * 64 + lane;
      const float p = row_bad ? __builtin_nanf("") : ex[s] * inv;
      if (e < n) {
        ws.prob[e] = p;
        if (probs_out) probs_out[row * n + e] = p;
      }
      key[s] = e < n ? (row_bad ? 0xffffffffu : ordered_key(p)) : 0u;
      ix[s] = e;
    }
    int e = 0;
    if (!ARGMAX || row_bad || !distinct_select(key, kk, lane, e))
      e = exact_select(key, ix, n, kk, sorted != 0, lane, ws);
    if (tie_rows) {
      // rows whose result depends on the algorithm's order: unsorted, NaN and partial_sort rows, and
      // those with a chosen key that another element has too
      bool tie = !sorted || row_bad || kk * 64 <= n;
      for (int j = 0; j < kk && !tie; ++j) {
        const uint32_t kj = ordered_key(ws.prob[__builtin_amdgcn_readlane(e, j)]);
        int same = 0;
#pragma unroll
        for (int s = 0; s < NS; ++s)
          same += __popcll(__ballot(s * 64 + lane < n && ordered_key(ws.prob[s * 64 + lane]) == kj));
        tie = same != 1;
      }
      if (tie && lane == 0) atomicAdd(tie_rows, 1);
    }
    wave_sync_lds();
    // weights: lanes 0..kk-1 each own one selected expert
    const float wv = lane < kk ? ws.prob[e] : 0.f;
    const float tot = renorm ? topk_weight_sum(wv, kk) : 0.f;
    if (lane < kk) {
      float w = renorm ? wv / tot : wv;
      w = w * scale;
      idx_out[row * kk + lane] = e;
      w_out[row * kk + lane] = f32_to_bf16(w);
    }
    wave_sync_lds();
  }
}

}  // namespace
}  // namespace ferry

using namespace ferry;

extern "C" int ferry_router_topk(const void* logits, int32_t logits_dtype, int64_t tokens,
                                 int64_t experts, int64_t topk, int32_t renorm, float scale,
                                 int32_t sorted, int64_t* idx_out, void* w_out_bf16,
                                 float* probs_out, int32_t* tie_rows, void* stream) {
  clear_error();
  FERRY_CHECK_ARG(tokens >= 0, "tokens must be >= 0 (got %lld)", (long long)tokens);
  FERRY_CHECK_ARG(experts >= 1 && experts <= kMaxE, "experts must be in [1, %d] (got %lld)",
                  kMaxE, (long long)experts);
  FERRY_CHECK_ARG(topk >= 1 && topk <= experts && topk <= kMaxK,
                  "topk must be in [1, min(experts, %d)] (got %lld)", kMaxK, (long long)topk);
  FERRY_CHECK_ARG(logits_dtype == FERRY_BF16 || logits_dtype == FERRY_F32,
                  "logits dtype must be bf16 or fp32");
  FERRY_CHECK_ARG(tokens == 0 || (logits && idx_out && w_out_bf16), "null pointer argument");
  if (tokens == 0) return 0;
  const int64_t want = ceil_div(tokens, kWaves);
  const int grid = (int)(want < 65535 ? want : 65535);
  hipStream_t s = (hipStream_t)stream;
  // NS = 64-key slots per lane: the exact path's wave-parallel steps scale with it
  auto go = [&](auto kernel, const auto* lg) {
    launch("router_kernel", kernel, dim3(grid), dim3(64 * kWaves), 0, s, lg, tokens, (int)experts,
           (int)topk, renorm, scale, sorted, idx_out, (bf16_t*)w_out_bf16, probs_out, tie_rows);
  };
  auto pick = [&](auto argmax, const auto* lg) {
    typedef std::decay_t<decltype(*lg)> T;
    constexpr bool A = decltype(argmax)::value;
    if (experts <= 64) go(router_kernel<T, 1, A>, lg);
    else if (experts <= 128) go(router_kernel<T, 2, A>, lg);
    else go(router_kernel<T, 4, A>, lg);
  };
  // Arg-max rounds first where most rows have no ties: fp32 logits, and few bf16 rows (about a quarter
  // of the rows of 128 bf16 logits has one among its 9 largest, and the rows of a small call are done
  // when the slowest is).  us, rounds first / replay at once: fp32, k = 8 of 128, 1 row 4.8 / 6.7,
  // 8192 rows 13 / 20, k = 24 of 128 8.5 / 43 and 25 / 98; bf16 (mean of 100 inputs), k = 8 of 128,
  // 1 row 4.9 / 6.2, 4 rows 6.4 / 7.1, 8 rows 7.5 / 7.3, 16 rows 7.8 / 7.6.
  const bool argmax = sorted && topk * 64 > experts && (logits_dtype == FERRY_F32 || tokens <= 4);
  auto typed = [&](const auto* lg) {
    if (argmax)
      pick(std::true_type{}, lg);
    else
      pick(std::false_type{}, lg);
  };
  if (logits_dtype == FERRY_BF16)
    typed((const bf16_t*)logits);
  else
    typed((const float*)logits);
  FERRY_LAUNCHED("router_kernel");
  return 0;
}
