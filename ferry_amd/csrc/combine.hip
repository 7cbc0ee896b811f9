// Combine: gate-weighted expert outputs summed per token in fp32, cast to bf16.
//
// Reference: ferry/csrc/expert_ops.cpp:75-92.  reduce_partials builds an fp32 [R, H] zero
// tensor, index_add_s every expert's bf16 output (already multiplied by its routing weight)
// in ascending expert order and casts to bf16; at world = 1 scatter_returned is an fp32
// round trip of that bf16 tensor, i.e. the identity.  A token's k entries are stored in
// ascending-ID order, so summing j = 0..k-1 reproduces the reference order exactly.
//
// DeepSeek-V2 adds the shared experts' bf16 output to the routed bf16 output
// (transformers modeling_deepseek_v2.py:136, `hidden_states + self.shared_experts(residuals)`):
// with `addend` the bf16 combine result is added to it in fp32 and rounded again, which is
// torch's bf16 addition.
//
// One block per token row chunk: each thread owns 8 consecutive hidden elements (one 16-byte
// load per entry), so a token row of H = 2048 is one 256-thread block.
#include "common.h"

namespace ferry {
namespace {

constexpr int kThreads = 256;
constexpr int kVec = 8;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(kThreads) void combine_kernel(const bf16_t* __restrict__ part,
                                                           const int32_t* __restrict__ pair_pos,
                                                           const bf16_t* __restrict__ addend,
                                                           int64_t tokens, int k, int64_t H,
                                                           bf16_t* __restrict__ out) {
  const int64_t chunks_per_row = H / kVec;
  const int64_t total = tokens * chunks_per_row;
  for (int64_t c = (int64_t)blockIdx.x * kThreads + threadIdx.x; c < total;
       c += (int64_t)gridDim.x * kThreads) {
    const int64_t t = c / chunks_per_row;
    const int64_t h0 = (c % chunks_per_row) * kVec;
    float acc[kVec];
#pragma unroll
    for (int i = 0; i < kVec; ++i) acc[i] = 0.f;
    for (int j = 0; j < k; ++j) {
      const int64_t src = pair_pos ? (int64_t)pair_pos[t * k + j] : t * k + j;
      if (src < 0) continue;
      const u32x4 v = *reinterpret_cast<const u32x4*>(part + src * H + h0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] += bf16_to_f32((bf16_t)(v[i] & 0xffffu));
        acc[2 * i + 1] += bf16_to_f32((bf16_t)(v[i] >> 16));
      }
    }
    if (addend) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(addend + t * H + h0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] = bf16r(acc[2 * i]) + bf16_to_f32((bf16_t)(v[i] & 0xffffu));
        acc[2 * i + 1] = bf16r(acc[2 * i + 1]) + bf16_to_f32((bf16_t)(v[i] >> 16));
      }
    }
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = (uint32_t)f32_to_bf16(acc[2 * i]) | ((uint32_t)f32_to_bf16(acc[2 * i + 1]) << 16);
    *reinterpret_cast<u32x4*>(out + t * H + h0) = o;
  }
}

// ---------------------------------------------------------------------------------------------
// reduce_rows: fp32 sums of the rows p of part with row_of[p] == r, p ascending, for every r
// ---------------------------------------------------------------------------------------------

// reduce_partials on lists of expert outputs, whose rows come in any order and number.  Three small
// launches: the counters are cleared; every entry p takes one of its row's 16 slots (a layout gives a
// row at most 16 entries), and those after the 16th are chained; a workgroup per row puts its entries
// in order and sums.  Bound by latency (three dependent launches) for decode-sized calls, by the reads
// of part in the last launch for large ones.
// Building the inverse of row_of with a concatenation of part, a sort, a histogram, a scan and
// gathers took 24 launches, two of them waited for, 108 us of GPU time for 64 rows of 8 entries
// (H = 2048) and 170 us for 2000 of 6; these three take 12.4 and 22.1 us.
//
// A row of up to 1024 entries walks its chain with one lane (half a microsecond a step, rows side by
// side) and ranks the entries in LDS.  It looks for them in row_of instead, 256 at a time, in order,
// where that is no longer (fewer than 128 entries of the call for each step: few rows can be so), where
// it has more, or where the workspace has no room for chains.  Looking in row_of for every row of more
// than 16 entries grows with rows * entries: 20,000 rows of 20 (H = 512) took 7480 us and take 164, 8192
// of 32 (H = 2048) 2140 us and 265.
constexpr int kSlots = 16;            // entries of a row with a place of their own
constexpr int kListed = 1024;         // most entries of a row listed in LDS
constexpr int kEntriesPerStep = 128;  // entries of the call per step of a chain

// head (nullable): 0, or 1 + the first entry of row r's chain; next[p] likewise the one after p
__global__ __launch_bounds__(kThreads) void reduce_clear(int32_t* __restrict__ count, int64_t rows,
                                                         int32_t* __restrict__ head) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i <= rows;
       i += (int64_t)gridDim.x * kThreads) {
    count[i] = 0;
    if (head && i < rows) head[i] = 0;
  }
}
// count[r]: entries of row r; count[rows]: entries outside [0, rows) (left out)
__global__ __launch_bounds__(kThreads) void reduce_slots(const int64_t* __restrict__ row_of,
                                                         int64_t entries, int64_t rows,
                                                         int32_t* __restrict__ count,
                                                         int32_t* __restrict__ slots,
                                                         int32_t* __restrict__ head,
                                                         int32_t* __restrict__ next) {
  for (int64_t p = (int64_t)blockIdx.x * kThreads + threadIdx.x; p < entries;
       p += (int64_t)gridDim.x * kThreads) {
    const int64_t r = row_of[p];
    if (r < 0 || r >= rows) {
      atomicAdd(&count[rows], 1);
    } else {
      const int32_t c = atomicAdd(&count[r], 1);
      if (c < kSlots)
        slots[r * kSlots + c] = (int32_t)p;
      else if (head)
        next[p] = atomicExch(&head[r], (int32_t)p + 1);
    }
  }
}
__device__ __forceinline__ void add8(float (&acc)[kVec], const bf16_t* p) {
  const u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    acc[2 * i] += bf16_to_f32((bf16_t)(v[i] & 0xffffu));
    acc[2 * i + 1] += bf16_to_f32((bf16_t)(v[i] >> 16));
  }
}
__global__ __launch_bounds__(kThreads) void reduce_rows_kernel(
    const bf16_t* __restrict__ part, const int64_t* __restrict__ row_of, int64_t entries,
    int64_t rows, int64_t H, const int32_t* __restrict__ count, const int32_t* __restrict__ slots,
    const int32_t* __restrict__ head, const int32_t* __restrict__ next, bf16_t* __restrict__ out) {
  __shared__ int32_t order[kListed], found[kListed];
  __shared__ int32_t wave_n[kThreads / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const int n = count[r];
    if (n <= kSlots && threadIdx.x < 64) {
      const int32_t mine = lane < n ? slots[r * kSlots + lane] : 0x7fffffff;
      int rank = 0;
      for (int j = 0; j < n; ++j) rank += __shfl(mine, j) < mine;
      if (lane < n) order[rank] = mine;
    }
    const bool listed =
        n > kSlots && n <= kListed && head && (int64_t)(n - kSlots) * kEntriesPerStep <= entries;
    if (listed) {
      if (threadIdx.x < kSlots) found[threadIdx.x] = slots[r * kSlots + threadIdx.x];
      if (threadIdx.x == 64) {
        int32_t p = head[r];
        for (int i = kSlots; i < n; ++i) {
          found[i] = p - 1;
          p = next[p - 1];
        }
      }
      __syncthreads();
      for (int i = threadIdx.x; i < n; i += kThreads) {
        const int32_t mine = found[i];
        int rank = 0;
        for (int j = 0; j < n; ++j) rank += found[j] < mine;
        order[rank] = mine;
      }
    }
    __syncthreads();
    for (int64_t h0 = 0; h0 < H; h0 += kThreads * kVec) {
      const int64_t h = h0 + threadIdx.x * kVec;
      float acc[kVec];
#pragma unroll
      for (int i = 0; i < kVec; ++i) acc[i] = 0.f;
      if (n <= kSlots) {
        if (h < H)
          for (int j = 0; j < n; ++j) add8(acc, part + (int64_t)order[j] * H + h);
      } else if (listed) {
        if (h < H)
#pragma unroll 4
          for (int j = 0; j < n; ++j) add8(acc, part + (int64_t)order[j] * H + h);
      } else {
        for (int64_t p0 = 0; p0 < entries; p0 += kThreads) {
          const int64_t p = p0 + threadIdx.x;
          const bool hit = p < entries && row_of[p] == r;
          const uint64_t hits = __ballot(hit);
          if (lane == 0) wave_n[wave] = __popcll(hits);
          __syncthreads();
          int before = 0, all = 0;
          for (int w = 0; w < kThreads / 64; ++w) {
            before += w < wave ? wave_n[w] : 0;
            all += wave_n[w];
          }
          if (hit) order[before + __popcll(hits & ((1ull << lane) - 1))] = (int32_t)p;
          __syncthreads();
          if (h < H)
#pragma unroll 4
            for (int j = 0; j < all; ++j) add8(acc, part + (int64_t)order[j] * H + h);
          __syncthreads();
        }
      }
      if (h < H) {
        u32x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = (uint32_t)f32_to_bf16(acc[2 * i]) | ((uint32_t)f32_to_bf16(acc[2 * i + 1]) << 16);
        *reinterpret_cast<u32x4*>(out + r * H + h) = o;
      }
    }
    __syncthreads();   // order is free again
  }
}

}  // namespace
}  // namespace ferry

using namespace ferry;

extern "C" int64_t ferry_reduce_rows_workspace_bytes(int64_t rows) {
  return (rows * (kSlots + 1) + 1) * (int64_t)sizeof(int32_t);
}

extern "C" int64_t ferry_reduce_rows_full_workspace_bytes(int64_t rows, int64_t entries) {
  return ferry_reduce_rows_workspace_bytes(rows) + (rows + entries) * (int64_t)sizeof(int32_t);
}

extern "C" int ferry_reduce_rows(const void* part, int64_t entries, int64_t hidden,
                                 const int64_t* row_of, int64_t rows, void* out, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
  clear_error();
  FERRY_CHECK_ARG(entries >= 0 && entries < ((int64_t)1 << 31) && rows >= 0, "bad sizes");
  FERRY_CHECK_ARG(hidden > 0 && hidden % kVec == 0, "hidden must be a positive multiple of %d", kVec);
  FERRY_CHECK_ARG(rows == 0 || out, "null pointer argument");
  FERRY_CHECK_ARG(entries == 0 || (part && row_of), "null pointer argument");
  FERRY_CHECK_ARG(((uintptr_t)part % 16) == 0 && ((uintptr_t)out % 16) == 0,
                  "part/out must be 16-byte aligned");
  FERRY_CHECK_ARG(workspace && workspace_bytes >= ferry_reduce_rows_workspace_bytes(rows),
                  "workspace too small (%lld < %lld bytes)", (long long)workspace_bytes,
                  (long long)ferry_reduce_rows_workspace_bytes(rows));
  hipStream_t s = (hipStream_t)stream;
  // words: [count of each row | entries outside the rows | slots | chain heads | chains]
  int32_t* count = (int32_t*)workspace;
  int32_t* slots = count + rows + 1;
  int32_t* head = workspace_bytes >= ferry_reduce_rows_full_workspace_bytes(rows, entries)
                      ? slots + rows * kSlots
                      : nullptr;
  int32_t* next = head ? head + rows : nullptr;
  auto blocks = [](int64_t n) { return dim3((unsigned)(n < 1 ? 1 : (ceil_div(n, kThreads) < 4096 ? ceil_div(n, kThreads) : 4096))); };
  launch("reduce_clear", reduce_clear, blocks(rows + 1), dim3(kThreads), 0, s, count, rows, head);
  FERRY_LAUNCHED("reduce_clear");
  if (entries > 0) {
    launch("reduce_slots", reduce_slots, blocks(entries), dim3(kThreads), 0, s, row_of, entries, rows,
           count, slots, head, next);
    FERRY_LAUNCHED("reduce_slots");
  }
  if (rows > 0) {
    launch("reduce_rows_kernel", reduce_rows_kernel, dim3((unsigned)(rows < kMaxGrid ? rows : kMaxGrid)),
           dim3(kThreads), 0, s, (const bf16_t*)part, row_of, entries, rows, hidden, count, slots,
           head, next, (bf16_t*)out);
    FERRY_LAUNCHED("reduce_rows_kernel");
  }
  return 0;
}

namespace {
int combine_impl(const void* part, const int32_t* pair_pos, int64_t tokens, int64_t topk,
                 int64_t hidden, const void* addend, void* out, void* stream) {
  clear_error();
  FERRY_CHECK_ARG(tokens >= 0 && topk >= 1, "bad sizes");
  FERRY_CHECK_ARG(hidden > 0 && hidden % kVec == 0, "hidden must be a positive multiple of %d",
                  kVec);
  FERRY_CHECK_ARG(tokens == 0 || (part && out), "null pointer argument");
  FERRY_CHECK_ARG(((uintptr_t)part % 16) == 0 && ((uintptr_t)out % 16) == 0 &&
                      ((uintptr_t)addend % 16) == 0,
                  "part/addend/out must be 16-byte aligned");
  if (tokens == 0) return 0;
  const int64_t work = tokens * (hidden / kVec);
  int64_t grid = ceil_div(work, kThreads);
  if (grid > 65536) grid = 65536;
  launch("combine_kernel", combine_kernel, dim3((unsigned)grid), dim3(kThreads), 0, (hipStream_t)stream,
                     (const bf16_t*)part, pair_pos, (const bf16_t*)addend, tokens, (int)topk, hidden,
                     (bf16_t*)out);
  FERRY_LAUNCHED("combine_kernel");
  return 0;
}
}  // namespace

extern "C" int ferry_combine(const void* part, const int32_t* pair_pos, int64_t tokens,
                             int64_t topk, int64_t hidden, void* out, void* stream) {
  return combine_impl(part, pair_pos, tokens, topk, hidden, nullptr, out, stream);
}

extern "C" int ferry_combine_add(const void* part, const int32_t* pair_pos, int64_t tokens,
                                 int64_t topk, int64_t hidden, const void* addend, void* out,
                                 void* stream) {
  if (!addend && tokens > 0) {
    clear_error();
    FERRY_CHECK_ARG(false, "addend must not be null");
  }
  return combine_impl(part, pair_pos, tokens, topk, hidden, addend, out, stream);
}
