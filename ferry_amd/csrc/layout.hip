// Dispatch layout at world = 1: per-token ID sort, per-expert histogram, exclusive scan and a
// stable token permutation.
//
// Reference: ferry/layout.py:12-94.  At world = 1 every route is local, so build_layout
// reduces to: send_idx = arange(T); send_ids[t] = sorted(selected[t]) (insertion sort,
// :28-33); counts = histogram of send_ids; starts = exclusive prefix (:61-63); (rows, cols)
// = a stable counting sort of all (token, position) pairs by expert, tokens ascending within
// an expert (:64-74).  The packet weights of pack_dispatch (ferry/csrc/expert_ops.cpp:57-60)
// are the routing weights reordered into send_ids order.
//
// Design: one token per lane.  Within a wavefront the rank of a token among the earlier tokens that
// chose the same expert is a popcount of a 64-bit per-expert lane mask built with LDS atomic ORs;
// the wavefront and block offsets come from exclusive scans.  No global atomics are used, so the
// permutation is deterministic.  For few tokens a single block (of as many wavefronts as the
// tokens need) does everything in one launch; more take two: per-block histograms, then the
// scatter, in which every block sums the histograms before its own.
//
// Both are bound by latency: a chain of LDS and L2 round trips on few wavefronts.  Hence the ID sort
// in registers over 8 slots when k <= 8 (16 otherwise), scans across lanes rather than by one thread,
// and blocks of 256 tokens where the histograms then stay small (256 blocks at 65,536 tokens
// instead of 64 of 1024).  us, with one sort width, a one-thread scan, 1024-token blocks and a scan
// launch of its own -> now: 16 tokens (k = 8, 128 experts) 10.2 -> 6.5; 512 tokens 15.8 -> 12.1; 1024
// tokens 25.0 -> 13.4; 8192 tokens 34.9 -> 14.4; 65,536 tokens (k = 6, 64 experts) 39 -> 16.
//
// The one launch is bound by one CU's scattered stores, so its line is drawn in (token, expert) pairs:
// us, one launch - two, 8 IDs of 128: 400 tokens 10.2 - 10.8, 512 tokens 11.8 - 10.9, 1024 tokens 21 -
// 11.5; 6 of 64: 512 tokens 7.8 - 9.0, 640 tokens 9.1 - 9.0; 2 of 8: 768 tokens 5.7 - 7.5, 1024 tokens
// 6.6 - 7.8; 16 of 256, where the two launches sort twice as much: 300 tokens 20.5 - 23.2, 400 tokens
// 25.2 - 23.2.
#include "common.h"

#include <mutex>

namespace ferry {
namespace {

constexpr int kMaxE = 512;
constexpr int kMaxK = 16;
constexpr int kSingleTokens = 1024;   // most tokens of the one-launch layout
constexpr int kSinglePairs8 = 3200;   // ... and of (token, expert) pairs, for up to 8 IDs a token
constexpr int kSinglePairs16 = 5120;  // ... and for up to 16
constexpr int kMaxBlock = 1024;       // most tokens of a block of the two-launch layout

template <int KM>
struct TokenIds {
  int32_t id[KM];
  bf16_t w[KM];
};

// Load one token's k <= KM IDs and weights and sort them by ID (IDs of a token are distinct, so any
// sort gives the insertion-sort result); out-of-range entries carry the key kMaxE, padding
// entries kMaxE + 1.  `bad` is set for a token with an out-of-range or a repeated ID: such a
// token breaks the layout's contract (its entries would share one permutation slot).
template <int KM>
__device__ __forceinline__ void load_sorted(const int64_t* __restrict__ selected,
                                            const bf16_t* __restrict__ weights, int64_t t, int k,
                                            int E, TokenIds<KM>& s, bool& bad) {
#pragma unroll
  for (int j = 0; j < KM; ++j) {
    if (j < k) {
      int64_t e = selected[t * k + j];
      bad |= (e < 0 || e >= E);
      s.id[j] = (e < 0 || e >= E) ? kMaxE : (int32_t)e;
      s.w[j] = weights ? weights[t * k + j] : (bf16_t)0;
    } else {
      s.id[j] = kMaxE + 1;
      s.w[j] = 0;
    }
  }
  // odd-even transposition sort over KM slots (static indices keep it in registers)
#pragma unroll
  for (int r = 0; r < KM; ++r) {
#pragma unroll
    for (int j = r & 1; j + 1 < KM; j += 2) {
      if (s.id[j] > s.id[j + 1]) {
        int32_t ti = s.id[j];
        s.id[j] = s.id[j + 1];
        s.id[j + 1] = ti;
        bf16_t tw = s.w[j];
        s.w[j] = s.w[j + 1];
        s.w[j + 1] = tw;
      }
    }
  }
#pragma unroll
  for (int j = 0; j + 1 < KM; ++j) bad |= (j + 1 < k && s.id[j] < E && s.id[j] == s.id[j + 1]);
}

// LDS of a block of `waves` wavefronts, E experts: lane masks (the wavefront's lanes that chose
// expert e), exclusive prefixes over the wavefronts, and two per-expert arrays
struct BlockLds {
  unsigned long long* mask;   // [waves][E]
  int32_t* wave_base;         // [waves][E]
  int32_t* count;             // [E]
  int32_t* base;              // [E]
  __device__ BlockLds(char* p, int waves, int E) {
    mask = reinterpret_cast<unsigned long long*>(p);
    wave_base = reinterpret_cast<int32_t*>(mask + waves * E);
    count = wave_base + waves * E;
    base = count + E;
  }
  static size_t bytes(int waves, int E) { return (size_t)E * (waves * 12 + 8); }
};

// Phase 1 of a block: the lane masks of its tokens and the per-wavefront prefixes; count[e] (with
// COUNT) is the number of the block's tokens per expert.
template <int KM, bool COUNT>
__device__ __forceinline__ void block_masks(const BlockLds& sh, const int64_t* __restrict__ selected,
                                            const bf16_t* __restrict__ weights, int64_t tokens,
                                            int k, int E, int64_t t, TokenIds<KM>& s, bool& valid,
                                            bool& bad) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  valid = t < tokens;
  if (valid) load_sorted(selected, weights, t, k, E, s, bad);
  for (int i = threadIdx.x; i < waves * E; i += blockDim.x) sh.mask[i] = 0ull;
  __syncthreads();
  if (valid) {
#pragma unroll
    for (int j = 0; j < KM; ++j)
      if (j < k && s.id[j] < E) atomicOr(&sh.mask[wave * E + s.id[j]], 1ull << lane);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    int32_t run = 0;
    for (int w = 0; w < waves; ++w) {
      sh.wave_base[w * E + e] = run;
      run += __popcll(sh.mask[w * E + e]);
    }
    if (COUNT) sh.count[e] = run;
  }
  __syncthreads();
}

// Wavefront 0: exclusive prefix of count[0 .. E) into base (added to it with ADD), and into starts
// (with its total at E) when given.
template <bool ADD>
__device__ __forceinline__ void scan_experts(const int32_t* count, int32_t* base, int E,
                                             int64_t* __restrict__ starts) {
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  int32_t carry = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int32_t c = e < E ? count[e] : 0;
    int32_t incl = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    if (e < E) {
      base[e] = (ADD ? base[e] : 0) + carry + incl - c;
      if (starts) starts[e] = carry + incl - c;
    }
    carry += __shfl(incl, 63, 64);
  }
  if (lane == 0 && starts) starts[E] = carry;
}

// Phase 2 of a block: write the sorted IDs, packet weights and the permutation entries.
// base[e] = grouped position of the block's first entry of expert e.
template <int KM>
__device__ __forceinline__ void block_scatter(const BlockLds& sh, int64_t t, int k,
                                              const TokenIds<KM>& s, int64_t* __restrict__ send_ids,
                                              bf16_t* __restrict__ w_sorted,
                                              int64_t* __restrict__ rows, int64_t* __restrict__ cols,
                                              int32_t* __restrict__ pair_pos, int E) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int j = 0; j < KM; ++j) {
    if (j < k) {
      const int32_t e = s.id[j];
      send_ids[t * k + j] = e < E ? e : -1;
      if (w_sorted) w_sorted[t * k + j] = s.w[j];
      if (e < E) {
        const int64_t pos = (int64_t)sh.base[e] + sh.wave_base[wave * E + e] +
                            __popcll(sh.mask[wave * E + e] & below);
        rows[pos] = t;
        cols[pos] = j;
        if (pair_pos) pair_pos[t * k + j] = (int32_t)pos;
      } else if (pair_pos) {
        pair_pos[t * k + j] = -1;
      }
    }
  }
}

template <int KM>
__global__ __launch_bounds__(kSingleTokens) void layout_single(
    const int64_t* __restrict__ selected, const bf16_t* __restrict__ weights, int64_t tokens,
    int k, int E, int64_t* __restrict__ send_ids, bf16_t* __restrict__ w_sorted,
    int64_t* __restrict__ starts, int64_t* __restrict__ rows, int64_t* __restrict__ cols,
    int32_t* __restrict__ pair_pos, int32_t* __restrict__ err) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const BlockLds sh(lds, blockDim.x >> 6, E);
  TokenIds<KM> s;
  bool valid, bad = false;
  if (threadIdx.x == 0) *err = 0;  // ordered before the atomics by the barriers below
  block_masks<KM, true>(sh, selected, weights, tokens, k, E, threadIdx.x, s, valid, bad);
  scan_experts<false>(sh.count, sh.base, E, starts);
  __syncthreads();
  if (valid) {
    block_scatter(sh, threadIdx.x, k, s, send_ids, w_sorted, rows, cols, pair_pos, E);
    if (bad) atomicAdd(err, 1);
  }
}

// Per-expert counts of each block of block_tokens tokens; an expert that a token names twice
// counts once (as its lane mask holds it once), IDs outside [0, E) do not count.
constexpr int kCountThreads = 256;
template <int KM>
__global__ __launch_bounds__(kCountThreads) void layout_count(
    const int64_t* __restrict__ selected, int64_t tokens, int k, int E, int block_tokens,
    int32_t* __restrict__ block_hist, int32_t* __restrict__ err) {
  __shared__ int32_t hist[kMaxE];
  if (blockIdx.x == 0 && threadIdx.x == 0) *err = 0;
  for (int e = threadIdx.x; e < E; e += kCountThreads) hist[e] = 0;
  __syncthreads();
  const int64_t t0 = (int64_t)blockIdx.x * block_tokens;
  for (int i = threadIdx.x; i < block_tokens; i += kCountThreads) {
    const int64_t t = t0 + i;
    if (t >= tokens) break;
    int64_t id[KM];
#pragma unroll
    for (int j = 0; j < KM; ++j) id[j] = j < k ? selected[t * k + j] : -1;
#pragma unroll
    for (int j = 0; j < KM; ++j) {
      bool count = id[j] >= 0 && id[j] < E;
#pragma unroll
      for (int q = 0; q < j; ++q) count &= id[q] != id[j];
      if (count) atomicAdd(&hist[id[j]], 1);
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += kCountThreads) block_hist[(int64_t)blockIdx.x * E + e] = hist[e];
}

template <int KM>
__global__ __launch_bounds__(kMaxBlock) void layout_scatter(
    const int64_t* __restrict__ selected, const bf16_t* __restrict__ weights, int64_t tokens,
    int k, int E, const int32_t* __restrict__ block_hist, int64_t* __restrict__ starts,
    int64_t* __restrict__ send_ids, bf16_t* __restrict__ w_sorted, int64_t* __restrict__ rows,
    int64_t* __restrict__ cols, int32_t* __restrict__ pair_pos, int32_t* __restrict__ err) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const BlockLds sh(lds, blockDim.x >> 6, E);
  const int nblk = gridDim.x, b = blockIdx.x;
  // per expert: the entries of the blocks before this one (base) and of all blocks (count); the
  // blocks are dealt to the threads of a column of experts (four a thread where E allows)
  for (int e = threadIdx.x; e < E; e += blockDim.x) sh.count[e] = sh.base[e] = 0;
  __syncthreads();
  const bool vec = E % 4 == 0 && ((uintptr_t)block_hist & 15) == 0;
  const int cols_n = vec ? E / 4 : E;
  const int parts = (int)blockDim.x / cols_n > 1 ? (int)blockDim.x / cols_n : 1;
  for (int c = threadIdx.x; c < cols_n * parts; c += blockDim.x) {
    const int col = c % cols_n, part = c / cols_n;
    if (vec) {
      typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
      i32x4 pre = {0, 0, 0, 0}, all = {0, 0, 0, 0};
#pragma unroll 4
      for (int q = part; q < nblk; q += parts) {
        const i32x4 h = *reinterpret_cast<const i32x4*>(block_hist + (int64_t)q * E + 4 * col);
        all += h;
        if (q < b) pre += h;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        atomicAdd(&sh.base[4 * col + i], pre[i]);
        atomicAdd(&sh.count[4 * col + i], all[i]);
      }
    } else {
      int32_t pre = 0, all = 0;
#pragma unroll 4
      for (int q = part; q < nblk; q += parts) {
        const int32_t h = block_hist[(int64_t)q * E + col];
        all += h;
        if (q < b) pre += h;
      }
      atomicAdd(&sh.base[col], pre);
      atomicAdd(&sh.count[col], all);
    }
  }
  __syncthreads();
  scan_experts<true>(sh.count, sh.base, E, b == 0 ? starts : nullptr);
  TokenIds<KM> s;
  bool valid, bad = false;
  const int64_t t = (int64_t)b * blockDim.x + threadIdx.x;
  block_masks<KM, false>(sh, selected, weights, tokens, k, E, t, s, valid, bad);
  if (valid) {
    block_scatter(sh, t, k, s, send_ids, w_sorted, rows, cols, pair_pos, E);
    if (bad) atomicAdd(err, 1);
  }
}

// starts[0 .. n] from n sizes that come with the launch (no copy from host memory)
struct Sizes {
  int32_t v[kMaxE];
};
__global__ __launch_bounds__(64) void starts_kernel(Sizes sizes, int n, int64_t* __restrict__ starts) {
  const int lane = threadIdx.x;
  int64_t carry = 0;
  for (int e0 = 0; e0 < n; e0 += 64) {
    const int e = e0 + lane;
    const int64_t c = e < n ? sizes.v[e] : 0;
    int64_t incl = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int64_t v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    if (e < n) starts[e] = carry + incl - c;
    carry += __shfl(incl, 63, 64);
  }
  if (lane == 0) starts[n] = carry;
}

// The workspace of ferry_layout_noalloc: a file-scope device array instead of caller memory.
// Each GPU holds its own copy for the life of the process; its device address is looked up
// once per device (hipGetSymbolAddress) and only that address is handed to kernels.  Nothing in
// it needs clearing between calls: the error counter is zeroed by the layout kernels themselves
// and the per-block histograms are fully rewritten by every multi-block call.
constexpr int64_t kScratchBytes = 256 + 128 * (int64_t)kMaxE * (int64_t)sizeof(int32_t);
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_dev[kMaxDevices];  // device address of `scratch` on each device, or null

// Device address of `scratch` on the current device (resolved on first use per device).
int scratch_address(void** out) {
  int dev = -1;
  FERRY_HIP(hipGetDevice(&dev));
  FERRY_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_dev[dev] == nullptr) {
    void* p = nullptr;
    FERRY_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_dev[dev] = p;
  }
  *out = g_scratch_dev[dev];
  return 0;
}

}  // namespace
}  // namespace ferry

using namespace ferry;

// Bytes of the error counter (256 B aligned) and of one histogram per block of block_tokens tokens.
static int64_t layout_bytes(int64_t tokens, int64_t experts, int64_t block_tokens) {
  return 256 + ceil_div(tokens > 0 ? tokens : 1, block_tokens) * experts * (int64_t)sizeof(int32_t);
}
// A workspace holds at least the histograms of 1024-token blocks.  Smaller blocks need more of them:
// the recommended size has room for 256-token blocks as long as the histograms stay within 256 KiB
// (which every block of the scatter reads); it grows with the number of tokens.
extern "C" int64_t ferry_layout_workspace_bytes(int64_t tokens, int64_t topk, int64_t experts) {
  (void)topk;
  const int64_t need = layout_bytes(tokens, experts, kMaxBlock);
  const int64_t fine = layout_bytes(tokens, experts, 256);
  const int64_t room = fine < kScratchBytes ? fine : kScratchBytes;
  return need > room ? need : room;
}

extern "C" int ferry_layout(const int64_t* selected, const void* weights_bf16, int64_t tokens,
                            int64_t topk, int64_t experts, int64_t* send_ids,
                            void* w_sorted_bf16, int64_t* starts, int64_t* rows, int64_t* cols,
                            int32_t* pair_pos, void* workspace, int64_t workspace_bytes,
                            void* stream) {
  clear_error();
  FERRY_CHECK_ARG(tokens >= 0, "tokens must be >= 0");
  FERRY_CHECK_ARG(experts >= 1 && experts <= kMaxE, "experts must be in [1, %d]", kMaxE);
  FERRY_CHECK_ARG(topk >= 1 && topk <= kMaxK && topk <= experts,
                  "topk must be in [1, min(experts, %d)]", kMaxK);
  FERRY_CHECK_ARG(tokens * topk < (int64_t)1 << 31, "tokens*topk must be < 2^31");
  FERRY_CHECK_ARG(starts && workspace, "null pointer argument");
  FERRY_CHECK_ARG(workspace_bytes >= layout_bytes(tokens, experts, kMaxBlock),
                  "workspace too small (%lld < %lld bytes)", (long long)workspace_bytes,
                  (long long)layout_bytes(tokens, experts, kMaxBlock));
  FERRY_CHECK_ARG(tokens == 0 || (selected && send_ids && rows && cols), "null pointer argument");
  hipStream_t s = (hipStream_t)stream;
  int32_t* err = (int32_t*)workspace;
  int32_t* hist = (int32_t*)((char*)workspace + 256);
  const int k = (int)topk, E = (int)experts;
  const bf16_t* w = (const bf16_t*)weights_bf16;
  bf16_t* ws = (bf16_t*)w_sorted_bf16;
  if (tokens <= kSingleTokens && tokens * topk <= (topk <= 8 ? kSinglePairs8 : kSinglePairs16)) {
    const int waves = (int)ceil_div(tokens > 0 ? tokens : 1, 64);
    launch("layout_single", k <= 8 ? layout_single<8> : layout_single<16>, dim3(1), dim3(64 * waves),
           (uint32_t)BlockLds::bytes(waves, E), s, selected, w, tokens, k, E, send_ids, ws, starts,
           rows, cols, pair_pos, err);
    FERRY_LAUNCHED("layout_single");
    return 0;
  }
  // the smallest blocks whose histograms fit the workspace and 256 KiB
  int block = 256;
  while (block < kMaxBlock && (layout_bytes(tokens, experts, block) > workspace_bytes ||
                                   layout_bytes(tokens, experts, block) > kScratchBytes))
    block *= 2;
  const int nblk = (int)ceil_div(tokens, block);
  launch("layout_count", k <= 8 ? layout_count<8> : layout_count<16>, dim3(nblk), dim3(kCountThreads),
         0, s, selected, tokens, k, E, block, hist, err);
  FERRY_LAUNCHED("layout_count");
  launch("layout_scatter", k <= 8 ? layout_scatter<8> : layout_scatter<16>, dim3(nblk), dim3(block),
         (uint32_t)BlockLds::bytes(block / 64, E), s, selected, w, tokens, k, E, hist, starts, send_ids,
         ws, rows, cols, pair_pos, err);
  FERRY_LAUNCHED("layout_scatter");
  return 0;
}

extern "C" int ferry_layout_noalloc(const int64_t* selected, const void* weights_bf16,
                                    int64_t tokens, int64_t topk, int64_t experts,
                                    int64_t* send_ids, void* w_sorted_bf16, int64_t* starts,
                                    int64_t* rows, int64_t* cols, int32_t* pair_pos,
                                    void* stream) {
  clear_error();
  FERRY_CHECK_ARG(tokens >= 0, "tokens must be >= 0");
  FERRY_CHECK_ARG(experts >= 1 && experts <= kMaxE, "experts must be in [1, %d]", kMaxE);
  const int64_t need = layout_bytes(tokens, experts, kMaxBlock);
  FERRY_CHECK_ARG(need <= kScratchBytes,
                  "layout_noalloc: %lld tokens x %lld experts need %lld scratch bytes, the static "
                  "buffer holds %lld (at most %lld tokens at this expert count)",
                  (long long)tokens, (long long)experts, (long long)need, (long long)kScratchBytes,
                  (long long)((kScratchBytes - 256) / (experts * (int64_t)sizeof(int32_t)) *
                              kMaxBlock));
  void* ws = nullptr;
  const int rc = scratch_address(&ws);
  if (rc != 0) return rc;
  return ferry_layout(selected, weights_bf16, tokens, topk, experts, send_ids, w_sorted_bf16,
                      starts, rows, cols, pair_pos, ws, kScratchBytes, stream);
}

extern "C" int ferry_starts(const int32_t* sizes, int32_t n, int64_t* starts, void* stream) {
  clear_error();
  FERRY_CHECK_ARG(n >= 0 && n <= kMaxE, "n must be in [0, %d]", kMaxE);
  FERRY_CHECK_ARG(starts && (n == 0 || sizes), "null pointer argument");
  Sizes s;
  for (int i = 0; i < n; ++i) {
    FERRY_CHECK_ARG(sizes[i] >= 0, "sizes[%d] = %d is negative", i, sizes[i]);
    s.v[i] = sizes[i];
  }
  for (int i = n; i < kMaxE; ++i) s.v[i] = 0;
  launch("starts_kernel", starts_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, s, (int)n, starts);
  FERRY_LAUNCHED("starts_kernel");
  return 0;
}
