// Grouped SwiGLU expert FFN over cache slots (bf16 in, fp32 accumulate, bf16 out).
//
// Reference: ferry/csrc/expert_ops.cpp:13-45 (execute_experts) and expert_ops.cu:6-25
// (silu_mul).  For each expert e with rows p in [starts[e], starts[e+1]):
//   x = in[rows[p]];  g = bf16(x Wg^T);  u = bf16(x Wu^T);  a = bf16(silu(g) * u) (fp32 math)
//   y = bf16(a Wd^T);  out = bf16(y * w[rows[p], cols[p]])
// with cache[slot] = [Wg (I x H) | Wu (I x H) | Wd (H x I)], all row-major bf16.  Both GEMMs
// are "NT" (both operands contiguous along K), which is the native operand order of the
// CDNA4 MFMA instructions used here.  The bf16 rounding points of the reference are kept.
//
// Three kernel schemes, selected per expert by its row count n_e:
//  * skinny (n_e <= 16, decode): bandwidth-bound.  A workgroup owns 16 (phase 1) or 64
//    (phase 2) weight rows and splits K over its four wavefronts; the partial sums meet in
//    LDS.  The weights are loaded 8 rows x 128 B per instruction and turned into MFMA B
//    fragments through a small per-wavefront LDS tile; x rows come from L2.
//    v_mfma_f32_16x16x32_bf16.  For the decode shapes (H = 2048 up, I = 768 down) the K walk
//    is software-pipelined with inline-asm loads: the next batch is in flight while the
//    current one is multiplied.
//  * mid (16 < n_e <= 64, prefill): bandwidth-bound.  A workgroup owns 64 output columns over
//    the full K; the expert's token rows are staged once per workgroup in LDS, the weights
//    stream into MFMA B registers.  Launched together with the skinny experts of a list.
//  * tiled (n_e > 64, prefill): MFMA-bound.  Persistent workgroups walk a device-computed
//    list of output tiles; A (gathered x rows / activation rows) and B (weight rows) tiles of 64
//    along K are staged by direct global->LDS loads into a swizzled LDS layout.
//    v_mfma_f32_16x16x32_bf16.  Tiles of 256x256 (ffn_tiled: two stages in LDS, eight wavefronts,
//    the two of a SIMD taking turns on the matrix core and on memory), or, for lists that leave CUs
//    idle with those, one of five from 256x128 down to 64x64 (ffn_tile: a ring of three to nine
//    stages); choose_tile picks one for the list.
// Phase 1 ("up") computes the gate and up projections together and applies silu(g)*u in the
// epilogue; phase 2 ("down") applies the routing weight in the epilogue and writes the
// per-(token, expert) row that the combine kernel sums.

#include "common.h"

#include <atomic>
#include <cstdint>
#include <mutex>
#include <type_traits>
#include <vector>

namespace ferry {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kListMax = 256;   // experts per launch (longer lists are split by the host)
constexpr int kSkinnyMax = 64;  // rows handled by the skinny and mid kernels (4 tiles of 16)

struct ExpertList {
  int32_t n;
  int32_t n_mid;   // small-expert up launch: the first n_mid entries take 64-column workgroups
  int16_t expert[kListMax];
  int32_t slot[kListMax];
};

struct FfnArgs {
  const bf16_t* cache;
  const bf16_t* x;        // [R, H]
  const bf16_t* w;        // [R, k] routing weights in sorted-ID order
  const int64_t* starts;  // [E+1]
  const int64_t* rows;    // [R*k]
  const int64_t* cols;    // [R*k]
  bf16_t* act;            // [R*k, I]
  bf16_t* out;            // [R*k, H]
  int64_t H, I, k;
  int32_t out_mode;
  ExpertList list;
};


__device__ __forceinline__ float silu_mul(float g, float u) {
  // silu(g) * u in fp32 on the bf16-rounded GEMM outputs: g * u / (1 + e^-g) with the
  // hardware exp2 and reciprocal (relative error ~1e-6, far below the bf16 rounding that
  // follows); a large negative g gives e^-g = inf and a zero result, the exact formula's limit
  return g * u * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
}

// two floats rounded to bf16 (round to nearest even, as f32_to_bf16) in one instruction,
// packed as lo | hi << 16
__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, b16x2));
}

__device__ __forceinline__ bf16x8 load8(const bf16_t* p) {
  return *reinterpret_cast<const bf16x8*>(p);
}

// Activation rows of the one-launch decode kernel (ffn_skinny_fused) are written by one
// workgroup and read by others, on any XCD, inside one launch.  With COH their stores and loads
// are agent-coherent (relaxed agent-scope atomic accesses: sc1), so that no L2 write-back or
// invalidate is needed between the two phases; the other kernels use plain accesses.
template <bool COH>
__device__ __forceinline__ void store_act(bf16_t* p, bf16_t v) {
  if constexpr (COH)
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else
    *p = v;
}
template <bool COH>
__device__ __forceinline__ bf16x8 load_act8(const bf16_t* p) {
  if constexpr (COH) {
    const uint64_t* q = reinterpret_cast<const uint64_t*>(p);
    const uint64_t lo = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t hi = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    struct { uint64_t a, b; } both = {lo, hi};
    return __builtin_bit_cast(bf16x8, both);
  } else {
    return load8(p);
  }
}

// =============================================================================================
// Memory helpers shared by the kernels below
// =============================================================================================

// a wave-uniform value / pointer moved to scalar registers
__device__ __forceinline__ int64_t uniform64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
template <typename T>
__device__ __forceinline__ const T* uniform_ptr(const T* p) {
  return (const T*)(uintptr_t)uniform64((int64_t)(uintptr_t)p);
}
// 16-byte global->LDS direct load of each lane: global address sbase + voff (wave-uniform base
// in scalar registers, 32-bit lane byte offset), LDS byte address lds + 16 * lane.  Issued as
// inline asm so that the address keeps this form wherever the load is scheduled; the compiler
// does not track these loads, their completion is awaited with wait_cnt / wait_vmcnt.  The asm writes
// m0 (the LDS base of the direct load); nothing else in these kernels uses m0.  An LDS direct
// load needs one wait state between the SALU write of m0 and its issue (the s_nop), which the
// compiler's hazard pass would add for its own instructions but cannot see inside the asm.
__device__ __forceinline__ void dma16(const char* sbase, uint32_t voff, uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, %1"
      :
      : "v"(voff), "s"(sbase), "s"(lds)
      : "memory", "m0");
}

typedef __attribute__((address_space(3))) char lds_char;
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(lds_char*)p;
}
// 4-byte global->LDS direct load of each lane (LDS byte address lds + 4 * lane), as dma16
__device__ __forceinline__ void dma4(const char* sbase, uint32_t voff, uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dword %0, %1"
      :
      : "v"(voff), "s"(sbase), "s"(lds)
      : "memory", "m0");
}
// 2-byte load of each lane, zero-extended to 4 bytes in LDS (address lds + 4 * lane)
__device__ __forceinline__ void dma2(const char* sbase, uint32_t voff, uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_ushort %0, %1"
      :
      : "v"(voff), "s"(sbase), "s"(lds)
      : "memory", "m0");
}
// 16 bytes at LDS byte address addr (constant parts of it go into the instruction's offset)
__device__ __forceinline__ bf16x8 lds_read16(uint32_t addr) {
  return *reinterpret_cast<__attribute__((address_space(3))) const bf16x8*>((uintptr_t)addr);
}
// wait until at most VM vector-memory operations (the direct loads among them) and no LDS reads
// of this wavefront are outstanding, in a form whose LDS part the compiler knows of
template <int VM>
__device__ __forceinline__ void wait_cnt() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((VM >> 4) << 14));
  asm volatile("" ::: "memory");
}
// workgroup barrier without the release/acquire fence of __syncthreads (which would drain
// the direct loads of the later stages); LDS visibility is established by the explicit waits
__device__ __forceinline__ void wg_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// =============================================================================================
// Skinny kernels
// =============================================================================================

// Skinny kernels (experts with at most 16 rows: decode, and the smallest experts of a prefill).
// They are bound by the weight bytes.  The four wavefronts of a workgroup split K into
// contiguous ranges of 32-element steps; their partial sums are added in LDS in a fixed order.
// up_skinny / down_skinny below load the weights in MFMA fragment order (each lane 16 bytes
// straight into B-operand registers, the loads of UNR K steps issued before their MFMAs); they
// serve shapes whose per-wavefront K range is not a multiple of 64.  up_skinny_t /
// down_skinny_t load 128 bytes of a row per 8 lanes instead, which the memory system serves
// at a higher rate (every 128-byte line fetched by one instruction, not two), and reorder the
// data into fragments through LDS.

template <int U, int MT, int NB, bool COH = false>
__device__ __forceinline__ void skinny_batch(const bf16_t* const (&pb)[NB], const bf16_t* const (&px)[MT],
                                             const bool (&okx)[MT], int k0,
                                             floatx4 (&acc)[MT][NB]) {
  const bf16x8 zero8 = {};
  bf16x8 b[NB][U], ax[MT][U];
#pragma unroll
  for (int s = 0; s < U; ++s)
#pragma unroll
    for (int j = 0; j < NB; ++j) b[j][s] = load8(pb[j] + k0 + s * 32);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int s = 0; s < U; ++s) ax[mt][s] = okx[mt] ? load_act8<COH>(px[mt] + k0 + s * 32) : zero8;
#pragma unroll
  for (int s = 0; s < U; ++s)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax[mt][s], b[j][s], acc[mt][j], 0, 0, 0);
}
// K steps [k0, kend) (multiples of 32) in batches of U, then of 2 and 1 for the remainder
template <int U, int MT, int NB, bool COH = false>
__device__ __forceinline__ void skinny_k_range(const bf16_t* const (&pb)[NB], const bf16_t* const (&px)[MT],
                                               const bool (&okx)[MT], int k0, int kend,
                                               floatx4 (&acc)[MT][NB]) {
  for (; k0 + U * 32 <= kend; k0 += U * 32) skinny_batch<U, MT, NB, COH>(pb, px, okx, k0, acc);
  for (; k0 + 2 * 32 <= kend; k0 += 2 * 32) skinny_batch<2, MT, NB, COH>(pb, px, okx, k0, acc);
  if (k0 < kend) skinny_batch<1, MT, NB, COH>(pb, px, okx, k0, acc);
}
// the fixed-order K reduction over the KS wavefronts of a column group nt, through the LDS
// buffer red (KS*NT*MT*NB*64 entries); the wavefront with ks = 0 returns true with the sums
template <int KS, int NT, int MT, int NB>
__device__ __forceinline__ bool skinny_reduce(floatx4 (&acc)[MT][NB], int ks, int nt, int lane,
                                              floatx4* red) {
  if constexpr (KS == 1) return true;
  auto at = [&](int q, int mt, int j) -> floatx4& {
    return red[(((q * NT + nt) * MT + mt) * NB + j) * 64 + lane];
  };
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NB; ++j) at(ks, mt, j) = acc[mt][j];
  __syncthreads();
  if (ks != 0) return false;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      acc[mt][j] = at(0, mt, j);
#pragma unroll
      for (int q = 1; q < KS; ++q) acc[mt][j] += at(q, mt, j);
    }
  return true;
}

// Phase 1, skinny: one workgroup = (expert, 16*NT*NC intermediate columns): NT column groups of
// NC tiles, each group's K split over KS = 4/NT wavefronts.  MT = number of 16-row M tiles
// (rows of the expert, <= 16*MT).  B operands j < NC: gate tiles, j >= NC: up tiles.
template <int NT, int NC, int MT, bool COH = false>
__device__ __forceinline__ void up_skinny(const FfnArgs& a, int li, int64_t start, int n, int bx,
                                          floatx4* red) {
  constexpr int KS = 4 / NT;
  constexpr int UNR = NC == 1 && MT == 1 ? 8 : 4;
  const int H = (int)a.H;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nt = wave % NT, ks = wave / NT;
  const int i0 = (bx * NT + nt) * 16 * NC;
  const bf16_t* wg = a.cache + (int64_t)a.list.slot[li] * 3 * a.H * a.I;
  const bf16_t* wu = wg + a.H * a.I;
  const int r16 = lane & 15, kg = (lane >> 4) * 8;
  const bf16_t* pb[2 * NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    pb[c] = wg + (int64_t)(i0 + 16 * c + r16) * H + kg;
    pb[NC + c] = wu + (int64_t)(i0 + 16 * c + r16) * H + kg;
  }
  const bf16_t* px[MT];
  bool okx[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = mt * 16 + r16;
    okx[mt] = r < n;
    const int64_t t = okx[mt] ? a.rows[start + r] : 0;
    px[mt] = a.x + t * a.H + kg;
  }
  floatx4 acc[MT][2 * NC];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < 2 * NC; ++j) acc[mt][j] = floatx4{0, 0, 0, 0};
  const int steps = H / 32;
  skinny_k_range<UNR>(pb, px, okx, ks * steps / KS * 32, (ks + 1) * steps / KS * 32, acc);
  if (!skinny_reduce<KS, NT>(acc, ks, nt, lane, red)) return;
  // 16x16 accumulator layout: column = lane & 15, rows (lane >> 4) * 4 + [0, 4)
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int col = i0 + 16 * c + (lane & 15);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = mt * 16 + (lane >> 4) * 4 + q;
        if (r < n) {
          const float g = bf16r(acc[mt][c][q]), u = bf16r(acc[mt][NC + c][q]);
          store_act<COH>(&a.act[(start + r) * a.I + col], f32_to_bf16(silu_mul(g, u)));
        }
      }
    }
  }
}
// Phase 1, skinny, at most 16 rows (decode): one workgroup = (expert, 16 intermediate columns),
// K split over the four wavefronts as above, but the weights are loaded 128 bytes of a row per
// lane group (8 rows x 128 B per instruction, every 128-byte line fetched by one instruction)
// rather than in the MFMA fragment order (16 rows x 64 B, each line fetched by two).  Each
// wavefront turns them into B fragments through its own 4 KiB LDS tile, one K chunk of 64 at a
// time: 32 rows (gate 0-15, up 16-31) x 128 B, chunk c of row r at slot c ^ ((r >> 1) & 7), which
// keeps the fragment reads free of bank conflicts.  NCH chunks of loads are in flight.
template <int NCH, bool COH = false>
__device__ __forceinline__ void up_skinny_t(const FfnArgs& a, int li, int64_t start, int n, int bx,
                                            floatx4* red, char* tile) {
  const int H = (int)a.H;
  const int lane = threadIdx.x & 63, ks = threadIdx.x >> 6;
  const int i0 = bx * 16;
  const bf16_t* wg = a.cache + (int64_t)a.list.slot[li] * 3 * a.H * a.I;
  const bf16_t* wu = wg + a.H * a.I;
  const int lr = lane >> 3, lc = lane & 7, r16 = lane & 15, kg = (lane >> 4) * 8;
  // row group g: rows 8g + lr of the tile (g = 0, 1 gate, 2, 3 up)
  const bf16_t* prow[4];
  uint32_t woff[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    prow[g] = (g < 2 ? wg : wu) + (int64_t)(i0 + 8 * (g & 1) + lr) * H + lc * 8;
    const int row = 8 * g + lr;
    woff[g] = (uint32_t)(row * 128 + ((lc ^ ((row >> 1) & 7)) << 4));
  }
  // fragment reads, K step s of a chunk: row r16 (gate) or 16 + r16 (up), chunk 4s + lane/16
  uint32_t roff[2][2];
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = 16 * j + r16;
      roff[st][j] = (uint32_t)(row * 128 + (((4 * st + (lane >> 4)) ^ ((row >> 1) & 7)) << 4));
    }
  const bool okx = r16 < n;
  const bf16_t* px = a.x + (okx ? a.rows[start + r16] : 0) * a.H + kg;
  floatx4 acc[2] = {floatx4{0, 0, 0, 0}, floatx4{0, 0, 0, 0}};
  const bf16x8 zero8 = {};
  auto batch = [&](int k0, auto nch) {
    constexpr int N = decltype(nch)::value;
    u32x4 w[N][4];
#pragma unroll
    for (int ch = 0; ch < N; ++ch)
#pragma unroll
      for (int g = 0; g < 4; ++g) w[ch][g] = *reinterpret_cast<const u32x4*>(prow[g] + k0 + 64 * ch);
    bf16x8 xa[2 * N];
#pragma unroll
    for (int st = 0; st < 2 * N; ++st) xa[st] = okx ? load8(px + k0 + 32 * st) : zero8;
#pragma unroll
    for (int ch = 0; ch < N; ++ch) {
#pragma unroll
      for (int g = 0; g < 4; ++g) *reinterpret_cast<u32x4*>(tile + woff[g]) = w[ch][g];
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bf16x8 bg = *reinterpret_cast<const bf16x8*>(tile + roff[st][0]);
        const bf16x8 bu = *reinterpret_cast<const bf16x8*>(tile + roff[st][1]);
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[2 * ch + st], bg, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[2 * ch + st], bu, acc[1], 0, 0, 0);
      }
    }
  };
  const int kb = ks * (H / 4), ke = kb + H / 4;   // H / 4 is a multiple of 64
  int k0 = kb;
  for (; k0 + 64 * NCH <= ke; k0 += 64 * NCH) batch(k0, std::integral_constant<int, NCH>{});
  for (; k0 < ke; k0 += 64) batch(k0, std::integral_constant<int, 1>{});
  floatx4 accm[1][2] = {{acc[0], acc[1]}};
  if (!skinny_reduce<4, 1>(accm, ks, 0, lane, red)) return;
  const int col = i0 + (lane & 15);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = (lane >> 4) * 4 + q;
    if (r < n) {
      const float g = bf16r(accm[0][0][q]), u = bf16r(accm[0][1][q]);
      store_act<COH>(&a.act[(start + r) * a.I + col], f32_to_bf16(silu_mul(g, u)));
    }
  }
}

// Phase 2, skinny: one workgroup = (expert, 16*NT*NC hidden rows), laid out as phase 1.
template <int NT, int NC, int MT, bool COH = false>
__device__ __forceinline__ void down_skinny(const FfnArgs& a, int li, int64_t start, int n, int bx,
                                            floatx4* red) {
  constexpr int KS = 4 / NT;
  constexpr int UNR = NC == 1 ? 8 : 4;
  const int I = (int)a.I;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nt = wave % NT, ks = wave / NT;
  const int h0 = (bx * NT + nt) * 16 * NC;
  const bf16_t* wd = a.cache + (int64_t)a.list.slot[li] * 3 * a.H * a.I + 2 * a.H * a.I;
  const int r16 = lane & 15, kg = (lane >> 4) * 8;
  const bf16_t* pb[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) pb[c] = wd + (int64_t)(h0 + 16 * c + r16) * I + kg;
  const bf16_t* pa[MT];
  bool oka[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = mt * 16 + r16;
    oka[mt] = r < n;
    pa[mt] = a.act + (start + (oka[mt] ? r : 0)) * a.I + kg;
  }
  floatx4 acc[MT][NC];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[mt][c] = floatx4{0, 0, 0, 0};
  const int steps = I / 32;
  skinny_k_range<UNR, MT, NC, COH>(pb, pa, oka, ks * steps / KS * 32, (ks + 1) * steps / KS * 32,
                                   acc);
  if (!skinny_reduce<KS, NT>(acc, ks, nt, lane, red)) return;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = mt * 16 + (lane >> 4) * 4 + q;
      if (r < n) {
        const int64_t p = start + r;
        const int64_t t = a.rows[p], j = a.cols[p];
        const float wt = bf16_to_f32(a.w[t * a.k + j]);
        const int64_t orow = a.out_mode == 0 ? t * a.k + j : p;
#pragma unroll
        for (int c = 0; c < NC; ++c)
          a.out[orow * a.H + h0 + 16 * c + (lane & 15)] = f32_to_bf16(bf16r(acc[mt][c][q]) * wt);
      }
    }
  }
}
// Phase 2, skinny, at most 16 rows (decode): one workgroup = (expert, 64 hidden rows), K split
// over the four wavefronts; the weights go through the wavefront's LDS tile as in up_skinny_t,
// 32 rows (two 16-row column tiles) at a time.
template <int NCH, bool COH = false>
__device__ __forceinline__ void down_skinny_t(const FfnArgs& a, int li, int64_t start, int n, int bx,
                                              floatx4* red, char* tile) {
  const int I = (int)a.I;
  const int lane = threadIdx.x & 63, ks = threadIdx.x >> 6;
  const int h0 = bx * 64;
  const bf16_t* wd = a.cache + (int64_t)a.list.slot[li] * 3 * a.H * a.I + 2 * a.H * a.I;
  const int lr = lane >> 3, lc = lane & 7, r16 = lane & 15, kg = (lane >> 4) * 8;
  // row group g (< 8): rows h0 + 8g + lr, at p0 + g * gstride; tile row (8g + lr) % 32
  const bf16_t* p0 = wd + (int64_t)(h0 + lr) * I + lc * 8;
  const int64_t gstride = (int64_t)8 * I;
  uint32_t woff[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int row = 8 * g + lr;
    woff[g] = (uint32_t)(row * 128 + ((lc ^ ((row >> 1) & 7)) << 4));
  }
  uint32_t roff[2][2];
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = 16 * j + r16;
      roff[st][j] = (uint32_t)(row * 128 + (((4 * st + (lane >> 4)) ^ ((row >> 1) & 7)) << 4));
    }
  const bool oka = r16 < n;
  const bf16_t* pa = a.act + (start + (oka ? r16 : 0)) * a.I + kg;
  // the token and slot index of the expert's row lane % 16, loaded ahead of the weights by the
  // wavefront that writes the output (the epilogue takes them from that lane by a shuffle)
  int32_t row_t = 0, row_j = 0;
  if (ks == 0) {
    const int64_t p = start + (r16 < n ? r16 : 0);
    row_t = (int32_t)a.rows[p];
    row_j = (int32_t)a.cols[p];
  }
  floatx4 acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = floatx4{0, 0, 0, 0};
  const bf16x8 zero8 = {};
  auto batch = [&](int k0, auto nch) {
    constexpr int N = decltype(nch)::value;
    u32x4 w[N][8];
#pragma unroll
    for (int ch = 0; ch < N; ++ch)
#pragma unroll
      for (int g = 0; g < 8; ++g) w[ch][g] = *reinterpret_cast<const u32x4*>(p0 + g * gstride + k0 + 64 * ch);
    bf16x8 xa[2 * N];
#pragma unroll
    for (int st = 0; st < 2 * N; ++st) xa[st] = oka ? load_act8<COH>(pa + k0 + 32 * st) : zero8;
#pragma unroll
    for (int ch = 0; ch < N; ++ch) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int g = 0; g < 4; ++g) *reinterpret_cast<u32x4*>(tile + woff[g]) = w[ch][4 * h + g];
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const bf16x8 b0 = *reinterpret_cast<const bf16x8*>(tile + roff[st][0]);
          const bf16x8 b1 = *reinterpret_cast<const bf16x8*>(tile + roff[st][1]);
          acc[2 * h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[2 * ch + st], b0, acc[2 * h], 0, 0, 0);
          acc[2 * h + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[2 * ch + st], b1, acc[2 * h + 1], 0, 0, 0);
        }
      }
    }
  };
  const int kb = ks * (I / 4), ke = kb + I / 4;   // I / 4 is a multiple of 64
  int k0 = kb;
  for (; k0 + 64 * NCH <= ke; k0 += 64 * NCH) batch(k0, std::integral_constant<int, NCH>{});
  for (; k0 < ke; k0 += 64) batch(k0, std::integral_constant<int, 1>{});
  floatx4 accm[1][4] = {{acc[0], acc[1], acc[2], acc[3]}};
  // the routing weight of each output row, loaded before the K reduction (whose barrier waits
  // for the other wavefronts)
  int32_t lane_orow = 0;
  float lane_wt = 0.0f;
  if (ks == 0) {
    const int64_t tj = (int64_t)row_t * a.k + row_j;
    lane_wt = bf16_to_f32(a.w[tj]);
    lane_orow = a.out_mode == 0 ? (int32_t)tj : (int32_t)(start + (r16 < n ? r16 : 0));
  }
  if (!skinny_reduce<4, 1>(accm, ks, 0, lane, red)) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = (lane >> 4) * 4 + q;
    const int64_t orow = __shfl(lane_orow, r);
    const float wt = __shfl(lane_wt, r);
    if (r < n) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        a.out[orow * a.H + h0 + 16 * c + (lane & 15)] = f32_to_bf16(bf16r(accm[0][c][q]) * wt);
    }
  }
}

// 16-byte global load into registers (saddr + 32-bit lane byte offset) as inline asm: the
// compiler does not track it, so the registers are read only after vmcnt_tie names them.
__device__ __forceinline__ void gload16(bf16x8& v, const void* sbase, uint32_t voff) {
  asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(v) : "v"(voff), "s"(sbase) : "memory");
}
// wait until at most N vector loads are outstanding; the registers named are those loads'
// destinations, tied so that no use of them is scheduled before the wait
template <int N>
__device__ __forceinline__ void vmcnt_tie(bf16x8 (&r)[8]) {
  asm volatile("s_waitcnt vmcnt(%8)"
               : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]),
                 "+v"(r[6]), "+v"(r[7])
               : "n"(N)
               : "memory");
}
template <int N>
__device__ __forceinline__ void vmcnt_tie(bf16x8 (&r)[2]) {
  asm volatile("s_waitcnt vmcnt(%2)" : "+v"(r[0]), "+v"(r[1]) : "n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void vmcnt_tie(bf16x8 (&r)[4]) {
  asm volatile("s_waitcnt vmcnt(%4)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]) : "n"(N) : "memory");
}

// f(integral_constant<int, i>) for i = B .. E - 1, unrolled at compile time
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}
template <int OFF>
__device__ __forceinline__ void gload16o(bf16x8& v, const void* sbase, uint32_t voff) {
  asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3"
               : "=v"(v)
               : "v"(voff), "s"(sbase), "n"(OFF)
               : "memory");
}
// gload16o for activation rows: agent-coherent (sc1) under COH, see store_act
template <int OFF, bool COH>
__device__ __forceinline__ void gload16o_act(bf16x8& v, const void* sbase, uint32_t voff) {
  if constexpr (COH)
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3 sc1"
                 : "=v"(v)
                 : "v"(voff), "s"(sbase), "n"(OFF)
                 : "memory");
  else
    gload16o<OFF>(v, sbase, voff);
}

// Phase 1, skinny, at most 16 rows, H = 512 * NB: up_skinny_t's tile scheme with the K range of
// each wavefront walked in NB batches of two 64-element chunks, software-pipelined -- the loads
// of batch b + 1 are issued before batch b goes through the tile and the matrix cores, so that a
// wavefront always has a batch in flight.  All loads are inline asm (saddr + 32-bit lane offset:
// two registers per batch set instead of a 64-bit address per load), 12 per batch in a fixed
// order (8 weight loads, then 4 token-row loads; padding rows load token row 0 and are zeroed
// after the wait), so each wait has a fixed count of younger loads.  The batch loop is fully
// unrolled: no loop-carried register holds a load in flight.
template <int NB, bool COH = false>
__device__ __forceinline__ void up_skinny_p(const FfnArgs& a, int li, int64_t start, int n, int bx,
                                            floatx4* red, char* tile) {
  static_assert(NB >= 2 && NB % 2 == 0, "an even number of batches");
  constexpr int H = 512 * NB;
  const int lane = threadIdx.x & 63, ks = threadIdx.x >> 6;
  const int i0 = bx * 16;
  const bf16_t* wg = uniform_ptr(a.cache + (int64_t)a.list.slot[li] * 3 * H * a.I);
  const bf16_t* xs = uniform_ptr(a.x);
  const int lr = lane >> 3, lc = lane & 7, r16 = lane & 15, kg = (lane >> 4) * 8;
  // byte offsets of the wavefront's K range: row group g = rows 8 (g & 1) + lr of the gate
  // (g < 2) or up (g >= 2) projection; the group offsets are wavefront-uniform
  const int kb = ks * (H / 4);
  const uint32_t wrow = (uint32_t)(((i0 + lr) * H + lc * 8 + kb) * 2);
  const uint32_t gup = (uint32_t)(H * a.I * 2);
  uint32_t woff[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int row = 8 * g + lr;
    woff[g] = (uint32_t)(row * 128 + ((lc ^ ((row >> 1) & 7)) << 4));
  }
  uint32_t roff[2][2];
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = 16 * j + r16;
      roff[st][j] = (uint32_t)(row * 128 + (((4 * st + (lane >> 4)) ^ ((row >> 1) & 7)) << 4));
    }
  const bool okx = r16 < n;
  floatx4 acc[2] = {floatx4{0, 0, 0, 0}, floatx4{0, 0, 0, 0}};
  const bf16x8 zero8 = {};
  // batch b: weights w[4 ch + g] (chunk ch of row group g), token rows xa[st] (K step st)
  uint32_t xrow;
  auto load_w = [&](auto b, bf16x8 (&w)[8]) {
    constexpr uint32_t kbyte = decltype(b)::value * 256;
    gload16o<0>(w[0], wg, wrow + kbyte);
    gload16o<0>(w[1], wg, wrow + kbyte + 16 * H);
    gload16o<0>(w[2], wg, wrow + kbyte + gup);
    gload16o<0>(w[3], wg, wrow + kbyte + gup + 16 * H);
    gload16o<128>(w[4], wg, wrow + kbyte);
    gload16o<128>(w[5], wg, wrow + kbyte + 16 * H);
    gload16o<128>(w[6], wg, wrow + kbyte + gup);
    gload16o<128>(w[7], wg, wrow + kbyte + gup + 16 * H);
  };
  auto load_x = [&](auto b, bf16x8 (&xa)[4]) {
    constexpr uint32_t kbyte = decltype(b)::value * 256;
    gload16o<0>(xa[0], xs, xrow + kbyte);
    gload16o<64>(xa[1], xs, xrow + kbyte);
    gload16o<128>(xa[2], xs, xrow + kbyte);
    gload16o<192>(xa[3], xs, xrow + kbyte);
  };
  auto mma = [&](bf16x8 (&w)[8], bf16x8 (&xa)[4]) {
#pragma unroll
    for (int st = 0; st < 4; ++st) xa[st] = okx ? xa[st] : zero8;
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) {
#pragma unroll
      for (int g = 0; g < 4; ++g) *reinterpret_cast<bf16x8*>(tile + woff[g]) = w[4 * ch + g];
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bf16x8 bg = *reinterpret_cast<const bf16x8*>(tile + roff[st][0]);
        const bf16x8 bu = *reinterpret_cast<const bf16x8*>(tile + roff[st][1]);
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[2 * ch + st], bg, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[2 * ch + st], bu, acc[1], 0, 0, 0);
      }
    }
  };
  auto load = [&](auto b, bf16x8 (&w)[8], bf16x8 (&xa)[4]) {
    load_w(b, w);
    load_x(b, xa);
  };
  // the token row of each lane (padding rows: row 0) is loaded ahead of the first weights and
  // awaited behind them, so the first batch keeps the fixed order of 8 weight and 4 row loads
  // (the low word suffices: token indices times H stay below 2^31)
  uint32_t trow;
  asm volatile("global_load_dword %0, %1, %2"
               : "=v"(trow)
               : "v"((uint32_t)((okx ? r16 : 0) * 8)), "s"(uniform_ptr(a.rows + start))
               : "memory");
  bf16x8 wA[8], wB[8], xA[4], xB[4];
  load_w(std::integral_constant<int, 0>{}, wA);
  asm volatile("s_waitcnt vmcnt(8)" : "+v"(trow) : : "memory");
  xrow = (trow * H + kg + kb) * 2;
  load_x(std::integral_constant<int, 0>{}, xA);
  static_for<0, NB / 2 - 1>([&](auto j) {
    load(std::integral_constant<int, 2 * decltype(j)::value + 1>{}, wB, xB);
    vmcnt_tie<12>(wA);
    vmcnt_tie<12>(xA);
    mma(wA, xA);
    load(std::integral_constant<int, 2 * decltype(j)::value + 2>{}, wA, xA);
    vmcnt_tie<12>(wB);
    vmcnt_tie<12>(xB);
    mma(wB, xB);
  });
  load(std::integral_constant<int, NB - 1>{}, wB, xB);
  vmcnt_tie<12>(wA);
  vmcnt_tie<12>(xA);
  mma(wA, xA);
  vmcnt_tie<0>(wB);
  vmcnt_tie<0>(xB);
  mma(wB, xB);
  floatx4 accm[1][2] = {{acc[0], acc[1]}};
  if (!skinny_reduce<4, 1>(accm, ks, 0, lane, red)) return;
  const int col = i0 + (lane & 15);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = (lane >> 4) * 4 + q;
    if (r < n) {
      const float g = bf16r(accm[0][0][q]), u = bf16r(accm[0][1][q]);
      store_act<COH>(&a.act[(start + r) * a.I + col], f32_to_bf16(silu_mul(g, u)));
    }
  }
}

// Phase 2, skinny, at most 16 rows, I = 256 * NC: down_skinny_t's tile scheme with each
// wavefront's K range walked one 64-element chunk at a time, software-pipelined over two register
// sets -- chunk c + 1 is loaded while chunk c goes through the tile and the matrix cores.  Ten
// asm loads per chunk in a fixed order (eight 8-row weight groups, then two activation loads;
// padding rows load the expert's first row and are zeroed after the wait).  Fully unrolled.
template <int NC, bool COH = false>
__device__ __forceinline__ void down_skinny_p(const FfnArgs& a, int li, int64_t start, int n, int bx,
                                              floatx4* red, char* tile) {
  constexpr int I = 256 * NC;
  const int lane = threadIdx.x & 63, ks = threadIdx.x >> 6;
  const int h0 = bx * 64;
  const bf16_t* wd =
      uniform_ptr(a.cache + (int64_t)a.list.slot[li] * 3 * a.H * I + 2 * a.H * I);
  const bf16_t* as = uniform_ptr(a.act + start * I);
  const int lr = lane >> 3, lc = lane & 7, r16 = lane & 15, kg = (lane >> 4) * 8;
  const int kb = ks * (I / 4);
  // row group g (< 8): rows h0 + 8g + lr, byte offset wrow + g * 16 I; tile row (8g + lr) % 32
  const uint32_t wrow = (uint32_t)(((h0 + lr) * I + lc * 8 + kb) * 2);
  uint32_t woff[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int row = 8 * g + lr;
    woff[g] = (uint32_t)(row * 128 + ((lc ^ ((row >> 1) & 7)) << 4));
  }
  uint32_t roff[2][2];
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = 16 * j + r16;
      roff[st][j] = (uint32_t)(row * 128 + (((4 * st + (lane >> 4)) ^ ((row >> 1) & 7)) << 4));
    }
  const bool oka = r16 < n;
  const uint32_t arow = (uint32_t)(((oka ? r16 : 0) * I + kg + kb) * 2);
  floatx4 acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = floatx4{0, 0, 0, 0};
  const bf16x8 zero8 = {};
  auto load = [&](auto c, bf16x8 (&w)[8], bf16x8 (&xa)[2]) {
    constexpr uint32_t kbyte = decltype(c)::value * 128;
#pragma unroll
    for (int g = 0; g < 8; ++g) gload16o<0>(w[g], wd, wrow + kbyte + g * 16 * I);
    gload16o_act<0, COH>(xa[0], as, arow + kbyte);
    gload16o_act<64, COH>(xa[1], as, arow + kbyte);
  };
  auto mma = [&](bf16x8 (&w)[8], bf16x8 (&xa)[2]) {
#pragma unroll
    for (int st = 0; st < 2; ++st) xa[st] = oka ? xa[st] : zero8;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int g = 0; g < 4; ++g) *reinterpret_cast<bf16x8*>(tile + woff[g]) = w[4 * h + g];
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bf16x8 b0 = *reinterpret_cast<const bf16x8*>(tile + roff[st][0]);
        const bf16x8 b1 = *reinterpret_cast<const bf16x8*>(tile + roff[st][1]);
        acc[2 * h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[st], b0, acc[2 * h], 0, 0, 0);
        acc[2 * h + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[st], b1, acc[2 * h + 1], 0, 0, 0);
      }
    }
  };
  // the token and slot index of the expert's row lane % 16, loaded ahead of the weights by the
  // wavefront that writes the output (the epilogue takes them from that lane by a shuffle)
  int32_t row_t = 0, row_j = 0;
  if (ks == 0) {
    const int64_t p = start + (r16 < n ? r16 : 0);
    row_t = (int32_t)a.rows[p];
    row_j = (int32_t)a.cols[p];
  }
  bf16x8 wA[8], wB[8], xA[2], xB[2];
  load(std::integral_constant<int, 0>{}, wA, xA);
  static_for<0, NC>([&](auto c) {
    constexpr int C = decltype(c)::value;
    auto& wc = (C % 2 == 0) ? wA : wB;
    auto& xc = (C % 2 == 0) ? xA : xB;
    auto& wn = (C % 2 == 0) ? wB : wA;
    auto& xn = (C % 2 == 0) ? xB : xA;
    if constexpr (C + 1 < NC) {
      load(std::integral_constant<int, C + 1>{}, wn, xn);
      vmcnt_tie<10>(wc);
      vmcnt_tie<10>(xc);
    } else {
      vmcnt_tie<0>(wc);
      vmcnt_tie<0>(xc);
    }
    mma(wc, xc);
  });
  floatx4 accm[1][4] = {{acc[0], acc[1], acc[2], acc[3]}};
  // the routing weight of each output row, loaded before the K reduction (whose barrier waits
  // for the other wavefronts)
  int32_t lane_orow = 0;
  float lane_wt = 0.0f;
  if (ks == 0) {
    const int64_t tj = (int64_t)row_t * a.k + row_j;
    lane_wt = bf16_to_f32(a.w[tj]);
    lane_orow = a.out_mode == 0 ? (int32_t)tj : (int32_t)(start + (r16 < n ? r16 : 0));
  }
  if (!skinny_reduce<4, 1>(accm, ks, 0, lane, red)) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = (lane >> 4) * 4 + q;
    const int64_t orow = __shfl(lane_orow, r);
    const float wt = __shfl(lane_wt, r);
    if (r < n) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        a.out[orow * a.H + h0 + 16 * c + (lane & 15)] = f32_to_bf16(bf16r(accm[0][c][q]) * wt);
    }
  }
}

// Phase 2, skinny, short lists: one workgroup = (expert, 16 hidden rows), K split over the four
// wavefronts as in down_skinny, walked in chunks of 64 elements (up to NC each).  With 64 hidden rows a workgroup, a list of one
// to eight experts starts 32 to 256 workgroups, each a chain of load latencies over its K range; here
// a wavefront loads all of its weights at once, before the workgroup waits for the activation rows
// (which they do not depend on), and what is left after the wait is one load of the rows and the
// products.  The weights go through the wavefront's 2 KiB LDS tile (16 rows x 128 B) as in
// down_skinny_t.  load() takes the weights, the output rows and the routing weights, finish() the rest.
template <int NC, bool COH>
struct DownRows16 {
  bf16x8 w[2 * NC];
  int k0, ns;           // first element, 32-element steps (an odd count ends with half a chunk)
  int32_t lane_orow;    // of the expert's row lane % 16
  float lane_wt;
  __device__ __forceinline__ void load(const FfnArgs& a, int li, int64_t start, int n, int bx) {
    const int lane = threadIdx.x & 63, ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = (int)a.I / 32, s0 = ks * steps / 4;
    k0 = 32 * s0;
    ns = (ks + 1) * steps / 4 - s0;
    const char* wd = reinterpret_cast<const char*>(
        uniform_ptr(a.cache + (int64_t)a.list.slot[li] * 3 * a.H * a.I + 2 * a.H * a.I +
                    (int64_t)bx * 16 * a.I + k0));
    const uint32_t r8 = (uint32_t)((lane >> 3) * (int)a.I * 2), half = (uint32_t)(16 * a.I);
    const uint32_t row = r8 + (lane & 7) * 16, row_half = r8 + (lane & 3) * 16;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      // the second half of a half chunk is its first again, a chunk past the last the first half
      // chunk: no load leaves the wavefront's range
      const char* b = wd + (2 * c < ns ? 128 * c : 0);
      const uint32_t at = 2 * c + 1 < ns ? row : row_half;
      w[2 * c] = *reinterpret_cast<const bf16x8*>(b + at);
      w[2 * c + 1] = *reinterpret_cast<const bf16x8*>(b + at + half);
    }
    const int64_t p = start + ((lane & 15) < n ? lane & 15 : 0);
    const int64_t tj = a.rows[p] * a.k + a.cols[p];
    lane_wt = bf16_to_f32(a.w[tj]);
    lane_orow = a.out_mode == 0 ? (int32_t)tj : (int32_t)p;
    // all landed here: not sunk below the wait
#pragma unroll
    for (int c = 0; c < 2 * NC; ++c) asm volatile("" : "+v"(w[c]));
    asm volatile("" : "+v"(lane_wt), "+v"(lane_orow));
  }
  __device__ __forceinline__ void finish(const FfnArgs& a, int64_t start, int n, int bx, floatx4* red,
                                         char* tile) {
    const int lane = threadIdx.x & 63, ks = threadIdx.x >> 6;
    const int lr = lane >> 3, lc = lane & 7, r16 = lane & 15, kg = (lane >> 4) * 8;
    const bool ok = r16 < n;
    // 16-byte loads through a buffer descriptor of the expert's activation rows, agent-coherent
    // (sc1) under COH; steps past the wavefront's last load what it does not use, or zero past the rows
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(uniform_ptr(a.act + start * a.I)), 0, (int)(n * a.I * 2), 0x00020000);
    const int off = ((ok ? r16 : 0) * (int)a.I + k0 + kg) * 2;
    bf16x8 xa[2 * NC];
#pragma unroll
    for (int st = 0; st < 2 * NC; ++st)
      xa[st] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rows, off + 64 * st, 0, COH ? 16 : 0));
    const bf16x8 zero8 = {};
    floatx4 acc[1][1] = {{floatx4{0, 0, 0, 0}}};
    uint32_t woff[2], roff[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int row = 8 * g + lr;
      woff[g] = (uint32_t)(row * 128 + ((lc ^ ((row >> 1) & 7)) << 4));
      roff[g] = (uint32_t)(r16 * 128 + (((4 * g + (lane >> 4)) ^ ((r16 >> 1) & 7)) << 4));
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (2 * c < ns) {
#pragma unroll
        for (int g = 0; g < 2; ++g) *reinterpret_cast<bf16x8*>(tile + woff[g]) = w[2 * c + g];
#pragma unroll
        for (int st = 0; st < 2; ++st)
          if (2 * c + st < ns) {
            const bf16x8 b = *reinterpret_cast<const bf16x8*>(tile + roff[st]);
            acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ok ? xa[2 * c + st] : zero8, b, acc[0][0], 0, 0, 0);
          }
      }
    if (!skinny_reduce<4, 1>(acc, ks, 0, lane, red)) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = (lane >> 4) * 4 + q;
      const int64_t orow = __shfl(lane_orow, r);
      const float wt = __shfl(lane_wt, r);
      if (r < n) a.out[orow * a.H + bx * 16 + (lane & 15)] = f32_to_bf16(bf16r(acc[0][0][q]) * wt);
    }
  }
};

// =============================================================================================
// Mid kernels
// =============================================================================================

// Mid scheme (experts with 17-64 rows, prefill).  The skinny kernels read an expert's token rows
// once per 16 output columns, which at 64 rows is twice the weight bytes; here a workgroup covers
// 64 columns and reads them once.  One workgroup = (expert, 64 output columns), four wavefronts,
// each a 16-column group over the full K (phase 1: its 16 gate and 16 up columns).  Rows are held
// in 16-row M tiles (MT of them).  K is walked in chunks of 64:
//  * the token rows go through a ring of three 8 KiB LDS buffers, staged by direct loads (8 rows
//    x 128 B each, XD per wavefront) two chunks ahead; 128-byte rows, chunk j of row r at slot
//    j ^ ((r >> 1) & 7), so that the A-fragment reads are free of bank conflicts;
//  * the weights, read exactly once, are loaded 8 rows x 128 B per instruction (every 128-byte
//    line fetched by one instruction) into a ring of three register sets three chunks ahead, and
//    each chunk goes through the wavefront's 2 KiB LDS tile (16 rows x 128 B) into B fragments.
// Per wavefront and chunk the loads are issued in a fixed order -- XD token-row loads at the top
// of the chunk, NW weight loads after the tile writes -- so every wait has a fixed count of
// younger loads.
constexpr int kMidXBuf = 64 * 128;                    // token-row ring buffer (64 rows x 128 B)
constexpr int kMidLds = 3 * kMidXBuf + 4 * 2048;      // ring + four wavefront tiles: 32 KiB

template <int N>
__device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

template <int MODE, int MT>
__device__ __forceinline__ void ffn_mid_body_t(const FfnArgs& a, int li, int64_t start, int n,
                                               int bx, char* sm) {
  static_assert(MT == 1 || MT == 2 || MT == 4, "MT 16-row tiles");
  // token-row direct loads per wavefront and chunk (MT = 1 stages 32 rows, of which 16 are used)
  constexpr int XD = MT >= 2 ? MT / 2 : 1;
  constexpr int NB = MODE == 0 ? 2 : 1;
  constexpr int NW = 2 * NB;                 // weight loads per wavefront and chunk
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = (int)(MODE == 0 ? a.H : a.I);
  const int C = K / 64;
  const int lr = lane >> 3, lc = lane & 7, r16 = lane & 15;
  const uint32_t lds0 = lds_addr(sm);
  char* tile = sm + 3 * kMidXBuf + wave * 2048;
  // token rows: direct load i of this wavefront moves rows 8 (XD wave + i) + lr
  const char* xbase = reinterpret_cast<const char*>(MODE == 0 ? a.x : a.act);
  uint32_t xoff[XD];
#pragma unroll
  for (int i = 0; i < XD; ++i) {
    const int r = 8 * (XD * wave + i) + lr;
    const int rr = r < n ? r : 0;   // rows past the expert's last load a valid row
    const uint32_t t = MODE == 0 ? (uint32_t)a.rows[start + rr] : (uint32_t)(start + rr);
    xoff[i] = t * (uint32_t)(K * 2) + (uint32_t)((lc ^ ((r >> 1) & 7)) << 4);
  }
  auto stage = [&](int c) {   // chunks past the last restage it into a buffer nobody reads
    const int cc = c < C ? c : C - 1;
    const uint32_t dst = lds0 + (uint32_t)((c % 3) * kMidXBuf + XD * wave * 1024);
#pragma unroll
    for (int i = 0; i < XD; ++i) dma16(xbase + cc * 128, xoff[i], dst + (uint32_t)(i * 1024));
  };
  // weights: row group g (< NW) = rows 8 (g & 1) + lr of gate (g < 2) or up / down, 128 B of
  // the chunk per lane group
  const int col0 = bx * 64 + wave * 16;
  const bf16_t* slot = a.cache + (int64_t)a.list.slot[li] * 3 * a.H * a.I;
  const bf16_t* wbase = uniform_ptr(slot + (MODE == 0 ? (int64_t)col0 * a.H
                                                      : 2 * a.H * a.I + (int64_t)col0 * a.I));
  uint32_t woff[NW];
#pragma unroll
  for (int g = 0; g < NW; ++g)
    woff[g] = (uint32_t)(((g >= 2 ? a.H * a.I : 0) + (int64_t)(8 * (g & 1) + lr) * K + lc * 8) * 2);
  bf16x8 wb[3][NW];
  auto wload = [&](int c, bf16x8 (&w)[NW]) {   // chunks past the last reload it
    const int cc = c < C ? c : C - 1;
    const char* b = reinterpret_cast<const char*>(wbase) + cc * 128;
#pragma unroll
    for (int g = 0; g < NW; ++g) gload16(w[g], b, woff[g]);
  };
  // tile rows: write row group g2 (< 2) at rows 8 g2 + lr; fragment read of K step st: row r16,
  // chunk 4 st + lane / 16
  uint32_t twoff[2], troff[2], aoff[2];
#pragma unroll
  for (int g2 = 0; g2 < 2; ++g2) {
    const int row = 8 * g2 + lr;
    twoff[g2] = (uint32_t)(row * 128 + ((lc ^ ((row >> 1) & 7)) << 4));
  }
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    troff[st] = (uint32_t)(r16 * 128 + (((4 * st + (lane >> 4)) ^ ((r16 >> 1) & 7)) << 4));
    aoff[st] = troff[st];   // token-row fragments: the same layout, rows mt*16 + r16
  }
  floatx4 acc[MT][NB];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[mt][j] = floatx4{0, 0, 0, 0};
  auto chunk = [&](int c, auto par) {
    constexpr int P = decltype(par)::value;   // c % 3
    wg_barrier();             // chunk c staged by every wavefront; chunk c-1's buffer free
    stage(c + 2);
    // this chunk's weights: older than x(c), w(c+1), x(c+1), w(c+2), x(c+2)
    vmcnt_tie<3 * XD + 2 * NW>(wb[P]);
    bf16x8 bfr[NB][2];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
#pragma unroll
      for (int g2 = 0; g2 < 2; ++g2) *reinterpret_cast<bf16x8*>(tile + twoff[g2]) = wb[P][2 * j + g2];
#pragma unroll
      for (int st = 0; st < 2; ++st) bfr[j][st] = *reinterpret_cast<const bf16x8*>(tile + troff[st]);
    }
    wload(c + 3, wb[P]);
    const char* xb = sm + P * kMidXBuf;
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      bf16x8 xa[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        xa[mt] = *reinterpret_cast<const bf16x8*>(xb + mt * 16 * 128 + aoff[st]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[mt], bfr[j][st], acc[mt][j], 0, 0, 0);
    }
    // token rows of chunk c+1 landed: older than w(c+2), x(c+2), w(c+3)
    wait_vmcnt<2 * NW + XD>();
  };
  // phase 2: lane l loads the token and slot index of the expert's row l ahead of the weights,
  // so that after the K loop only the routing weight's load (which depends on them) is left;
  // the epilogue takes each row's output offset and weight from its lane by a shuffle
  int32_t row_t = 0, row_j = 0;
  if (MODE == 1) {
    const int64_t p = start + (lane < n ? lane : 0);
    row_t = (int32_t)a.rows[p];
    row_j = (int32_t)a.cols[p];
  }
  // prologue in the steady-state order: w(0), x(0), w(1), x(1), w(2)
  wload(0, wb[0]);
  stage(0);
  wload(1, wb[1]);
  stage(1);
  wload(2, wb[2]);
  wait_vmcnt<2 * NW + XD>();   // x(0) landed
  for (int c = 0; c < C; c += 3) {
    chunk(c, std::integral_constant<int, 0>{});
    if (c + 1 < C) chunk(c + 1, std::integral_constant<int, 1>{});
    if (c + 2 < C) chunk(c + 2, std::integral_constant<int, 2>{});
  }
  // the loads past the last chunk are never used: hold their registers (and the LDS) until
  // they landed
  wait_vmcnt<0>();
  vmcnt_tie<0>(wb[0]);
  vmcnt_tie<0>(wb[1]);
  vmcnt_tie<0>(wb[2]);
  // 16x16 accumulator layout: column = lane & 15, rows (lane >> 4) * 4 + [0, 4)
  const int col = col0 + (lane & 15);
  int32_t lane_orow = 0;
  float lane_wt = 0.0f;
  if (MODE == 1) {
    const int64_t tj = (int64_t)row_t * a.k + row_j;
    lane_wt = bf16_to_f32(a.w[tj]);
    lane_orow = a.out_mode == 0 ? (int32_t)tj : (int32_t)(start + (lane < n ? lane : 0));
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = mt * 16 + (lane >> 4) * 4 + q;
      if (MODE == 0) {
        if (r < n) {
          const float g = bf16r(acc[mt][0][q]), u = bf16r(acc[mt][NB - 1][q]);
          a.act[(start + r) * a.I + col] = f32_to_bf16(silu_mul(g, u));
        }
      } else {
        const int64_t orow = __shfl(lane_orow, r);
        const float wt = __shfl(lane_wt, r);
        if (r < n) a.out[orow * a.H + col] = f32_to_bf16(bf16r(acc[mt][0][q]) * wt);
      }
    }
  }
}

// Small experts (at most 64 rows), one launch for a list of mixed sizes so that together they
// fill the GPU: up to 16 rows the skinny scheme, 17-64 rows the mid scheme.  MTMAX = 1 when no
// expert of the list has more than 16 rows: then only the skinny scheme is compiled in and a
// phase-1 workgroup covers 16 intermediate columns (grid (I / 16, list)).  Otherwise the grid
// is one-dimensional: the list's first n_mid entries (those the host knows to have 17-64 rows)
// take I / 64 workgroups of 64 columns each, the rest I / 16 workgroups of 16 columns each, so
// that the larger workgroups are dispatched first.  A workgroup whose expert turns out to have
// the other scheme's row count still covers its columns: a 64-column workgroup of an expert with
// at most 16 rows runs four 16-column skinny passes (a one-tile mid workgroup when H is not a
// multiple of 256); of the four 16-column workgroups of a 64-column block of an expert with more
// than 16 rows, the first runs the block's mid workgroup and the others return.  Phase 2: 64
// hidden rows per workgroup in both schemes (grid (H / 64, list)).
template <int MTMAX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void ffn_up_skinny(FfnArgs a) {
  // MTMAX = 1: the K-reduction buffer (8 KiB) and four 4 KiB weight tiles
  __shared__ __attribute__((aligned(1024))) char sm[MTMAX > 1 ? kMidLds : 8192 + 4 * 4096];
  int li = blockIdx.y, bx = blockIdx.x;
  bool wide = false;   // a 64-column workgroup
  if (MTMAX > 1) {
    const int per_mid = (int)(a.I / 64), per_sk = (int)(a.I / 16);
    const int mid_wgs = a.list.n_mid * per_mid;
    const int b = blockIdx.x;
    wide = b < mid_wgs;
    li = wide ? b / per_mid : a.list.n_mid + (b - mid_wgs) / per_sk;
    bx = wide ? b % per_mid : (b - mid_wgs) % per_sk;
  }
  if (li >= a.list.n) return;
  const int e = a.list.expert[li];
  const int64_t start = a.starts[e];
  const int n = (int)(a.starts[e + 1] - start);
  if (n == 0 || n > 16 * MTMAX) return;
  if (MTMAX == 1 || (!wide && n <= 16)) {
    if (a.H == 2048)
      up_skinny_p<4>(a, li, start, n, bx, reinterpret_cast<floatx4*>(sm),
                  sm + 8192 + (threadIdx.x >> 6) * 4096);
    else if (a.H % 256 == 0)
      up_skinny_t<4>(a, li, start, n, bx, reinterpret_cast<floatx4*>(sm),
                     sm + 8192 + (threadIdx.x >> 6) * 4096);
    else
      up_skinny<1, 1, 1>(a, li, start, n, bx, reinterpret_cast<floatx4*>(sm));
    return;
  }
  if constexpr (MTMAX > 1) {
    if (!wide) {   // 16-column workgroup of an expert with more than 16 rows
      if (bx % 4 != 0) return;
      bx /= 4;
    }
    if (n > 32) {
      ffn_mid_body_t<0, 4>(a, li, start, n, bx, sm);
    } else if (n > 16) {
      ffn_mid_body_t<0, 2>(a, li, start, n, bx, sm);
    } else if (a.H % 256 == 0) {
#pragma unroll 1
      for (int j = 0; j < 4; ++j) {
        up_skinny_t<2>(a, li, start, n, bx * 4 + j, reinterpret_cast<floatx4*>(sm),
                       sm + 8192 + (threadIdx.x >> 6) * 4096);
        __syncthreads();   // the K-reduction buffer is free again
      }
    } else {
      ffn_mid_body_t<0, 1>(a, li, start, n, bx, sm);
    }
  }
}
template <int MTMAX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void ffn_down_skinny(FfnArgs a) {
  // the K-reduction buffer (16 KiB) and four 4 KiB weight tiles
  __shared__ __attribute__((aligned(1024))) char sm[MTMAX > 1 ? kMidLds : 16384 + 4 * 4096];
  const int li = blockIdx.y;
  if (li >= a.list.n) return;
  const int e = a.list.expert[li];
  const int64_t start = a.starts[e];
  const int n = (int)(a.starts[e + 1] - start);
  if (n == 0 || n > 16 * MTMAX) return;
  if (MTMAX == 1 || n <= 16) {
    if (a.I == 768)
      down_skinny_p<3>(a, li, start, n, blockIdx.x, reinterpret_cast<floatx4*>(sm),
                       sm + 16384 + (threadIdx.x >> 6) * 4096);
    else if (a.I % 256 == 0)
      down_skinny_t<2>(a, li, start, n, blockIdx.x, reinterpret_cast<floatx4*>(sm),
                       sm + 16384 + (threadIdx.x >> 6) * 4096);
    else
      down_skinny<1, 4, 1>(a, li, start, n, blockIdx.x, reinterpret_cast<floatx4*>(sm));
    return;
  }
  if constexpr (MTMAX > 1) {
    if (n > 32)
      ffn_mid_body_t<1, 4>(a, li, start, n, blockIdx.x, sm);
    else
      ffn_mid_body_t<1, 2>(a, li, start, n, blockIdx.x, sm);
  }
}

// =============================================================================================
// Decode: both phases of every expert (at most 16 rows each) in one launch
// =============================================================================================

// The workgroups of ffn_up_skinny<1> (I/16 per expert) come first in the grid, those of
// ffn_down_skinny<1> (H/64 per expert; H/16 with DownRows16) after them.  A down workgroup needs every intermediate
// column of its expert's activation rows, so it waits for all of that expert's up workgroups:
// each up workgroup, once its rows are stored, sets its arrival flag; a down workgroup's first
// wavefront waits for all flags of its expert.  The L2s of the XCDs are not coherent with
// each other, and a release / acquire pair would write back and invalidate a whole L2 for every
// workgroup (measured: 550 us per launch instead of 30): instead the activation rows themselves
// are stored and loaded agent-coherently (sc1, see store_act), each wavefront waits for its
// stores to complete before the workgroup arrives, and the flags are relaxed agent-scope
// atomic words.  Workgroups are dispatched in index order, so every producer a down
// workgroup waits for has been dispatched before it: the wait ends.  It is still bounded
// (kSyncSpinLimit sleeps, about a second); a down workgroup that runs out counts a timeout and
// skips its expert rather than read unfinished rows.  The count lives in device memory
// (g_sync_timeouts); the history kernel copies it into the caller's mapped host buffer at the
// start of every layer call, so that the runtime raises on the next call's routing readback
// instead of returning unwritten rows as output.
//
// Arrival flags: one 32-bit word per up workgroup, holding the epoch (a number unique to the
// call) once that workgroup's rows are stored.  A down workgroup's first wavefront checks all
// flags of its expert at once (a lane takes every 64th) until every one holds the call's epoch.  Flags
// from earlier calls hold older epochs, so nothing is ever cleared, and no word is written by
// two workgroups (no read-modify-write contention).  The flags live in a static per-device ring
// of kSyncSets sets (set = epoch % kSyncSets); calls that run at the same time on one GPU use
// different sets unless kSyncSets of them overlap.
constexpr int kSyncSets = 8;
constexpr int kMaxUpWgs = 176;   // up workgroups per expert (I / 16): I <= 2816
constexpr int kSyncSpinLimit = 1 << 21;
static __device__ __align__(256) uint32_t g_sync[kSyncSets][kListMax][kMaxUpWgs];
static __device__ int32_t g_sync_timeouts;

struct FusedSync {
  uint32_t* flags;   // the call's flag set (device address of g_sync[epoch % kSyncSets])
  int32_t* timeouts;
  uint32_t epoch;
  int32_t up_wgs;    // up workgroups per expert (I / 16)
  int32_t down_wgs;  // down workgroups per expert (H / 64, or H / 16 with DownRows16)
  int32_t spin_limit;  // polls before a down workgroup gives up (0: gives up at once)
};

__device__ __forceinline__ void sync_arrive(const FusedSync& fs, int li, int bx) {
  __hip_atomic_store(fs.flags + li * kMaxUpWgs + bx, fs.epoch, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// wavefront 0 of a down workgroup: true once every up workgroup of list entry li has arrived,
// false on timeout
__device__ __forceinline__ bool sync_wait(const FusedSync& fs, int li) {
  const int lane = threadIdx.x & 63;
  const uint32_t* f = fs.flags + li * kMaxUpWgs;
  for (int spins = 0;; ++spins) {
    if (spins >= fs.spin_limit) {
      if (lane == 0) atomicAdd(fs.timeouts, 1);
      return false;
    }
    bool mine = true;
    for (int j = lane; j < fs.up_wgs; j += 64)
      mine &= __hip_atomic_load(f + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == fs.epoch;
    if (__all(mine)) return true;
    __builtin_amdgcn_s_sleep(8);
  }
}

template <int NC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NC > 6 ? 2 : (NC > 3 ? 3 : 4)))) void ffn_skinny_fused(
    FfnArgs a, FusedSync fs) {
  // phase 2's K-reduction buffer (16 KiB; phase 1 uses 8) and four 4 KiB weight tiles
  __shared__ __attribute__((aligned(1024))) char sm[16384 + 4 * 4096];
  __shared__ int ok_s;
  const int nup = fs.up_wgs * a.list.n;
  const bool up = (int)blockIdx.x < nup;
  const int b = up ? (int)blockIdx.x : (int)blockIdx.x - nup;
  const int per = up ? fs.up_wgs : fs.down_wgs;
  const int li = b / per, bx = b % per;
  const int e = a.list.expert[li];
  const int64_t start = a.starts[e];
  const int n = (int)(a.starts[e + 1] - start);
  if (n == 0 || n > 16) return;   // up and down workgroups of such an expert both skip it
  if (up) {
    if (a.H == 2048)
      up_skinny_p<4, true>(a, li, start, n, bx, reinterpret_cast<floatx4*>(sm),
                     sm + 16384 + (threadIdx.x >> 6) * 4096);
    else if (a.H % 256 == 0)
      up_skinny_t<4, true>(a, li, start, n, bx, reinterpret_cast<floatx4*>(sm),
                     sm + 16384 + (threadIdx.x >> 6) * 4096);
    else
      up_skinny<1, 1, 1, true>(a, li, start, n, bx, reinterpret_cast<floatx4*>(sm));
    // the agent-coherent activation stores of every wavefront complete before the arrival
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) sync_arrive(fs, li, bx);
    return;
  }
  auto wait = [&]() {
    if (threadIdx.x < 64) {
      const bool ok = sync_wait(fs, li);
      if (threadIdx.x == 0) ok_s = ok ? 1 : 0;
    }
    __syncthreads();
    return ok_s != 0;
  };
  if constexpr (NC > 0) {
    DownRows16<NC, true> d;
    d.load(a, li, start, n, bx);
    if (!wait()) return;
    d.finish(a, start, n, bx, reinterpret_cast<floatx4*>(sm), sm + 16384 + (threadIdx.x >> 6) * 4096);
    return;
  }
  if (!wait()) return;
  if (a.I == 768)
    down_skinny_p<3, true>(a, li, start, n, bx, reinterpret_cast<floatx4*>(sm),
                     sm + 16384 + (threadIdx.x >> 6) * 4096);
  else if (a.I % 256 == 0)
    down_skinny_t<2, true>(a, li, start, n, bx, reinterpret_cast<floatx4*>(sm),
                     sm + 16384 + (threadIdx.x >> 6) * 4096);
  else
    down_skinny<1, 4, 1, true>(a, li, start, n, bx, reinterpret_cast<floatx4*>(sm));
}

// =============================================================================================
// Tiled kernels
// =============================================================================================

// Output tile 256 x 256 per workgroup, eight wavefronts, two per SIMD.  Bound by the matrix cores
// (and, under them, by the clock that the power limit leaves: 1.6-1.7 GHz).
//
// Halves and quadrants.  A stage holds BK = 64 columns of K: 256 A rows and 256 B rows of 128
// bytes, each operand cut into two halves of 128 rows (16 KiB).  Wavefront (wm, wn) = (w / 4,
// w % 4) computes in each of the four quadrants (A half, B half) the 64 rows 32 i + 16 wm + [0, 16)
// (i < 4) by the 32 columns 32 wn + [0, 32): 16 v_mfma_f32_16x16x32_bf16, 256 cycles.  In phase 1
// the B halves are 128 gate rows and the 128 up rows of the same intermediate columns, so every
// wavefront owns matching gate / up accumulators and the SwiGLU runs in registers.
//
// Ping-pong.  A stage is four phases, each a memory segment (the LDS reads of one half's
// fragments, the direct loads of another half) and a matrix segment (one quadrant's products), a
// barrier after each.  The wavefronts wm = 1 run one segment behind those of wm = 0, the other
// wavefront of the same SIMD: while one multiplies, its partner reads fragments and issues loads,
// and the two never compete for the matrix core or for the LDS.
//
//   phase            1        2        3        4
//   reads            A0(k)    B1(k)    A1(k)    B0(k+1)
//   loads            B0(k+2)  A0(k+2)  B1(k+2)  A1(k+2)    (into the half read one phase before)
//   multiplies       A0 B0    A0 B1    A1 B0    A1 B1
//
// Loads in flight.  Each half is loaded seven phases (about 2.2 us) before it is read, into the
// buffer that the previous phase read: two stages of LDS (128 KiB) hold up to seven halves in
// flight.  A wavefront issues two loads a phase, so "at most 12 outstanding" before the barrier
// says that its share of the half read next has landed; nothing in the loop waits for all loads.
// Before this schedule (one barrier and a full drain of the loads per stage, both wavefronts of a
// SIMD waiting together) a stage took 1.7 us, now 1.31.  One dense expert of 65,536 rows, H x I = 2048
// x 768, both timed in turn: up 372-391 -> 308-321 us (1060-1110 -> 1280-1340 TFLOP/s), down 255-271
// -> 209-214 us (760-810 -> 960-990); launched back to back, at the clock that the power limit then
// leaves, 430-455 -> 371-400 and 265-283 -> 216-227 (the card before: up 352 -> 299, down 233 -> 197
// after idling).  2048 x 1408: up 1177 -> 1411, down 1048 -> 1232 TFLOP/s; 2048 x 4096 down 1240 -> 1488.
// Of that, running on across tiles gives 2 % (up) and 2-6 % (down); each tile still spends about 6.5 us
// outside its stages, most of it the SwiGLU of the up epilogue (two quarter-rate transcendentals for
// each of a lane's 64 outputs).
// The same products are summed in the same K order as before: results are bit-identical.
//
// Operand staging: global -> LDS direct loads (global_load_lds_dwordx4, no VGPR round trip).  One
// load moves 8 full rows (64 lanes x 16 B, lane l -> row l / 8, LDS slot l % 8), fully coalesced.
// Inside a row the 16-byte chunk c is stored at slot c ^ swizzle(row); with two 128-byte rows per
// 256-byte bank line, the 16 rows that a quarter of a wavefront reads then touch 16 distinct
// 16-byte bank groups.  The rows are 16 consecutive ones for A, and {8 g + 4 c + [0, 4)} for B
// (below), hence the two swizzles.
//
// The products take the weight rows as first operand and the token rows as second: a lane then
// holds four consecutive weight rows (output columns) of one token row.  The B fragments of the
// column tiles c = 0, 1 take the weight rows 8 g + 4 c + [0, 4) (g < 4), so that the two tiles
// give a lane eight consecutive columns: the epilogue packs them into one 16-byte store, with no
// LDS staging, one row address and one routing weight per 16-row tile.
constexpr int BM = 256, BN = 256, BK = 64;
constexpr int kRowBytes = BK * 2;                  // 128
constexpr int kHalfBytes = 128 * kRowBytes;        // half an operand tile of one stage: 16 KiB
__device__ __forceinline__ int swz_a(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ int swz_b(int row) { return ((row >> 1) & 1) | (((row >> 3) & 3) << 1); }

struct TileTable {
  __attribute__((aligned(16))) int32_t cum[kListMax + 1];  // cumulative M tiles over list entries
  int32_t total;
  int64_t start[kListMax];    // per list entry: its expert's first grouped row, and row count
  int32_t rows[kListMax];
};

// Wavefront 0 builds the cumulative counts of M tiles of ROWS rows of the big experts of the list.
template <int ROWS>
__device__ void build_tile_table(const FfnArgs& a, TileTable& tt) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int cnt[4];
    int local = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int li = lane * 4 + q;
      int c = 0;
      if (li < a.list.n) {
        const int e = a.list.expert[li];
        const int64_t s0 = a.starts[e];
        const int64_t n = a.starts[e + 1] - s0;
        c = n > kSkinnyMax ? (int)((n + ROWS - 1) / ROWS) : 0;
        tt.start[li] = s0;
        tt.rows[li] = (int32_t)n;
      }
      cnt[q] = c;
      local += c;
    }
    int incl = local;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    int run = incl - local;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      tt.cum[lane * 4 + q] = run;
      run += cnt[q];
    }
    if (lane == 63) {
      tt.cum[kListMax] = incl;
      tt.total = incl;
    }
  }
  __syncthreads();
}

// largest li with cum[li] <= m (cum is non-decreasing), by a whole wavefront: the entries that hold
// at most m, counted with ballots over four entries a lane
__device__ __forceinline__ int find_entry(const TileTable& tt, int m) {
  const u32x4 c = *reinterpret_cast<const u32x4*>(&tt.cum[(threadIdx.x & 63) * 4]);
  int le = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) le += __popcll(__ballot((int)c[q] <= m));
  return le - 1;
}

// MODE 0: A = gathered x rows (K = H); B half 0 = gate rows i0 .. +128, half 1 = the up rows of
//         the same columns; epilogue act[p, i0 + c] = bf16(silu(bf16(g)) * bf16(u)).
// MODE 1: A = activation rows (K = I); B half h = down rows h0 + 128 h .. +128;
//         epilogue out[row(p), h0 + c] = bf16(bf16(y) * w(p)).
constexpr int kTiledThreads = 512;
template <int MODE>
__global__ __launch_bounds__(kTiledThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void ffn_tiled(FfnArgs a) {
  __shared__ TileTable tt;
  __shared__ __attribute__((aligned(1024))) char smem[8 * kHalfBytes];
  // per tile row, two sets taken in turn: phase 1 the token (source row), phase 2 the token and
  // slot index, and from them the output row and the routing weight (bf16 bits)
  __shared__ __attribute__((aligned(256))) int32_t row_s[2][BM], col_s[MODE == 1 ? 2 : 1][MODE == 1 ? BM : 1];
  __shared__ __attribute__((aligned(256))) int32_t orow_s[MODE == 1 ? 2 : 1][MODE == 1 ? BM : 1],
      wt_s[MODE == 1 ? 2 : 1][MODE == 1 ? BM : 1];
  build_tile_table<BM>(a, tt);
  const int64_t K = MODE == 0 ? a.H : a.I;
  const int ntn = MODE == 0 ? (int)(a.I / 128) : (int)(a.H / BN);
  const int total = __builtin_amdgcn_readfirstlane(tt.total) * ntn;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int KT = (int)(K / BK);   // even: H and I are multiples of 128
  const int j16 = lane & 15, g4 = lane >> 4;

  // fragment reads (byte address of K step ks; tile i / c, half and slot go into the offset)
  const uint32_t smem0 = lds_addr(smem);
  uint32_t a_addr[2], b_addr[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int arow = 16 * wm + j16, brow = 32 * wn + 8 * (j16 >> 2) + (j16 & 3);
    a_addr[ks] = smem0 + (uint32_t)(arow * kRowBytes + (((4 * ks + g4) ^ swz_a(arow)) << 4));
    b_addr[ks] = smem0 + (uint32_t)(4 * kHalfBytes + brow * kRowBytes + (((4 * ks + g4) ^ swz_b(brow)) << 4));
  }
  // Direct loads: of each half this wavefront moves rows 16 wave + 8 q + lane / 8 (q < 2), lane
  // slot lane % 8 holding the row's chunk (lane % 8) ^ swizzle(row).  Rows past the expert's last
  // row load its first row instead: each output row depends only on its own A row, and those rows
  // are never stored.
  const int r8 = lane >> 3, slot8 = lane & 7;
  uint32_t aoff[2][2], boff[2];   // byte offsets: < 2^32 (host-checked sizes)
  const char* const abase = reinterpret_cast<const char*>(MODE == 0 ? a.x : a.act);
#pragma unroll
  for (int q = 0; q < 2; ++q)
    boff[q] = ((uint32_t)(8 * q + r8) * (uint32_t)K + (uint32_t)((slot8 ^ swz_b(16 * wave + 8 * q + r8)) * 8)) * 2u;

  const int64_t bhalf = MODE == 0 ? a.H * a.I * 2 : 128 * a.I * 2;   // bytes from B half 0 to half 1
  struct Tile {
    int64_t start;       // the expert's first grouped row
    int m0, vrows, ntile;
    const char* bbase;   // B half 0, rows 16 wave ...
  };
  auto locate = [&](int tile) {
    Tile t;
    const int mt_global = tile / ntn;
    t.ntile = tile - mt_global * ntn;
    const int li = __builtin_amdgcn_readfirstlane(find_entry(tt, mt_global));
    t.start = uniform64(tt.start[li]);
    t.m0 = (mt_global - __builtin_amdgcn_readfirstlane(tt.cum[li])) * BM;
    t.vrows = __builtin_amdgcn_readfirstlane(tt.rows[li]) - t.m0;   // > 0
    const bf16_t* slot = a.cache + (int64_t)a.list.slot[li] * 3 * a.H * a.I;
    t.bbase = reinterpret_cast<const char*>(uniform_ptr(
        MODE == 0 ? slot + (int64_t)(t.ntile * 128 + 16 * wave) * a.H
                  : slot + 2 * a.H * a.I + (int64_t)(t.ntile * BN + 16 * wave) * a.I));
    return t;
  };
  // the tile rows' indices (low words; rows past the last: the first row's) into set p, direct
  // loads of the wavefronts 0 .. 3, 64 rows each
  auto load_rows = [&](const Tile& t, int p) {
    if (wave < 4) {
      const int r = 64 * wave + lane;
      const uint32_t off = (uint32_t)((r < t.vrows ? r : 0) * 8);
      const int64_t at = t.start + t.m0;
      dma4(reinterpret_cast<const char*>(uniform_ptr(a.rows + at)), off, lds_addr(row_s[p]) + 256 * wave);
      if constexpr (MODE == 1)
        dma4(reinterpret_cast<const char*>(uniform_ptr(a.cols + at)), off, lds_addr(col_s[p]) + 256 * wave);
    }
  };
  auto dma_a = [&](int kt, int h, int s) {
    const uint32_t dst = smem0 + (uint32_t)((2 * h + s) * kHalfBytes + 16 * wave * kRowBytes);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      dma16(abase + kt * BK * 2, aoff[h][q], dst + (uint32_t)(8 * q * kRowBytes));
  };
  auto dma_b = [&](const char* b, int h, int s) {   // b: the stage's columns of B half 0
    const uint32_t dst = smem0 + (uint32_t)((4 + 2 * h + s) * kHalfBytes + 16 * wave * kRowBytes);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      dma16(b + (h ? bhalf : 0), boff[q], dst + (uint32_t)(8 * q * kRowBytes));
  };
  // A offsets of a tile whose row indices are in set p
  auto set_aoff = [&](const Tile& t, int p) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = 16 * wave + 8 * q + r8, r = 128 * h + row;
        const uint32_t src = MODE == 0 ? (uint32_t)row_s[p][r]
                                       : (uint32_t)(t.start + t.m0 + (r < t.vrows ? r : 0));
        aoff[h][q] = (src * (uint32_t)K + (uint32_t)((slot8 ^ swz_a(row)) * 8)) * 2u;
      }
  };

  // XCD-aware order: workgroup b runs on XCD b % 8 (round-robin dispatch), so in each round
  // of gridDim tiles the workgroups of one XCD take a contiguous run of tiles.  Tiles of one
  // expert are consecutive with N fastest, so a run covers a compact block of M x N tiles whose
  // A and B slices are shared in that XCD's L2.
  const int per_xcd = gridDim.x % 8 == 0 ? (int)gridDim.x / 8 : 0;
  const int lslot = per_xcd ? (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  if (lslot >= total) return;
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  bf16x8 ft[4][2], fw[2][2][2];
  auto read_a = [&](auto h, auto s) {
    constexpr int off = (2 * decltype(h)::value + decltype(s)::value) * kHalfBytes;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i) ft[i][ks] = lds_read16(a_addr[ks] + off + i * 32 * kRowBytes);
  };
  auto read_b = [&](auto h, auto s) {
    constexpr int H = decltype(h)::value, off = (2 * H + decltype(s)::value) * kHalfBytes;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int c = 0; c < 2; ++c) fw[H][c][ks] = lds_read16(b_addr[ks] + off + c * 4 * kRowBytes);
  };
  // the first tile's first two stages, halves in the order in which they are read
  Tile cur = locate(lslot);
  load_rows(cur, 0);
  wait_cnt<0>();
  wg_barrier();
  set_aoff(cur, 0);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    dma_b(cur.bbase + k * BK * 2, 0, k);
    dma_a(k, 0, k);
    dma_b(cur.bbase + k * BK * 2, 1, k);
    dma_a(k, 1, k);
  }
  wait_cnt<12>();   // B half 0 and A half 0 of stage 0 have landed
  wg_barrier();
  read_b(I0{}, I0{});
  // every wavefront has read B half 0 of stage 0 before stage 0's first loads replace it
  wait_cnt<12>();
  wg_barrier();
  if (wm == 1) wg_barrier();   // the second group runs one segment behind the first
  int set = 0;
  for (int tile = lslot; tile < total; tile += gridDim.x, set ^= 1) {
    // the tile after this one; after the last tile its own first stages are loaded again
    const bool more = tile + (int)gridDim.x < total;
    Tile next = cur;
    if (more) next = locate(tile + gridDim.x);
    load_rows(next, set ^ 1);
    if constexpr (MODE == 1) {
      // output row and routing weight of tile row tid, in LDS before the epilogue reads them
      if (wave < 4) {
        const int64_t tj = (int64_t)row_s[set][tid] * a.k + col_s[set][tid];
        dma2(reinterpret_cast<const char*>(a.w), (uint32_t)(tj * 2), lds_addr(wt_s[set]) + 256 * wave);
        orow_s[set][tid] = a.out_mode == 0 ? (int32_t)tj : (int32_t)(cur.start + cur.m0 + tid);
      }
    }
    const int vrows = cur.vrows, ntile = cur.ntile;
    const int64_t row0 = cur.start + cur.m0;

    // 16-row tiles of each A half that hold rows of the expert (the others' products are skipped
    // in a partial tile: their output rows are never stored)
    int nf[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int v = vrows - 128 * h - 16 * wm;
      nf[h] = __builtin_amdgcn_readfirstlane(v >= 128 ? 4 : (v > 0 ? (v + 31) / 32 : 0));
    }

    auto pipeline = [&](auto part) {
      constexpr bool PARTIAL = decltype(part)::value;
      floatx4 acc[2][2][4][2];   // [A half][B half][16-row tile][16-column tile]
#pragma unroll
      for (int ha = 0; ha < 2; ++ha)
#pragma unroll
        for (int hb = 0; hb < 2; ++hb)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < 2; ++c) acc[ha][hb][i][c] = floatx4{0, 0, 0, 0};
      auto mma = [&](auto ha, auto hb) {
        constexpr int A = decltype(ha)::value, B = decltype(hb)::value;
        auto tile_row = [&](int i, int ks) {
#pragma unroll
          for (int c = 0; c < 2; ++c)
            acc[A][B][i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[B][c][ks], ft[i][ks],
                                                                     acc[A][B][i][c], 0, 0, 0);
        };
        __builtin_amdgcn_s_setprio(1);
        if constexpr (!PARTIAL) {
#pragma unroll
          for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i) tile_row(i, ks);
        } else {
#pragma unroll
          for (int i = 0; i < 4; i += 2)
            if (i < nf[A]) {
#pragma unroll
              for (int ks = 0; ks < 2; ++ks) {
                tile_row(i, ks);
                tile_row(i + 1, ks);
              }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        wg_barrier();
      };
      // end of a memory segment: the loads of the next segment's half have landed (the 12 loads of
      // the six halves after it may be in flight), this segment's fragments are in registers
      auto mem_end = [&]() {
        wait_cnt<12>();
        wg_barrier();
      };
      // a stage in slot S; its loads are those of stage kl (A) and at bl (B)
      auto stage = [&](const char* bl, int kl, auto ss) {
        constexpr int S = decltype(ss)::value;
        typedef std::integral_constant<int, S> IS;
        typedef std::integral_constant<int, 1 - S> IO;
        read_a(I0{}, IS{});
        dma_b(bl, 0, S);
        mem_end();
        mma(I0{}, I0{});
        read_b(I1{}, IS{});
        dma_a(kl, 0, S);
        mem_end();
        mma(I0{}, I1{});
        read_a(I1{}, IS{});
        dma_b(bl, 1, S);
        mem_end();
        mma(I1{}, I0{});
        read_b(I0{}, IO{});
        dma_a(kl, 1, S);
        mem_end();
        mma(I1{}, I1{});
      };
      const char* bnext = cur.bbase + 2 * BK * 2;   // B half 0 of the stage loaded next
      int kl = 2;
      for (int k = 0; k < KT; k += 2) {
        if (k + 2 == KT) {   // the last two stages load the next tile's first two
          set_aoff(next, set ^ 1);
          bnext = next.bbase;
          kl = 0;
        }
        bnext = uniform_ptr(bnext);
        stage(bnext, kl, I0{});
        stage(bnext + BK * 2, kl + 1, I1{});
        bnext += 2 * BK * 2;
        kl += 2;
      }
    // 16x16 accumulator layout (first operand: weight rows): column = token row lane & 15, rows
    // (lane >> 4) * 4 + q.  The weight rows of tiles c = 0, 1 interleave in groups of four (see
    // b_addr), so a lane holds 8 consecutive output columns of one token row: one 16-byte store.
    // the lane's row, opaque here so that the stores' addresses are computed now and not kept in
    // registers through the loop
    int erow = 16 * wm + j16;
    asm volatile("" : "+v"(erow));
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 128 * h + 32 * i + erow;
        if constexpr (MODE == 0) {
          u32x4 y;
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int q = 0; q < 4; q += 2) {
              const floatx4& g = acc[h][0][i][c];
              const floatx4& u = acc[h][1][i][c];
              const uint32_t gp = pk_bf16(g[q], g[q + 1]), up = pk_bf16(u[q], u[q + 1]);
              const float s0 = silu_mul(__uint_as_float(gp << 16), __uint_as_float(up << 16));
              const float s1 = silu_mul(__uint_as_float(gp & 0xffff0000u), __uint_as_float(up & 0xffff0000u));
              y[2 * c + q / 2] = pk_bf16(s0, s1);
            }
          if (r < vrows)
            *reinterpret_cast<u32x4*>(&a.act[(row0 + r) * a.I + ntile * 128 + wn * 32 + 8 * g4]) = y;
        } else {
          const float wt = __uint_as_float((uint32_t)wt_s[set][r] << 16);
          bf16_t* const o = a.out + (int64_t)orow_s[set][r] * a.H + ntile * BN + wn * 32 + 8 * g4;
#pragma unroll
          for (int hb = 0; hb < 2; ++hb) {
            u32x4 y;
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
              for (int q = 0; q < 4; q += 2) {
                const uint32_t v = pk_bf16(acc[h][hb][i][c][q], acc[h][hb][i][c][q + 1]);
                y[2 * c + q / 2] = pk_bf16(__uint_as_float(v << 16) * wt,
                                           __uint_as_float(v & 0xffff0000u) * wt);
              }
            if (r < vrows) *reinterpret_cast<u32x4*>(o + 128 * hb) = y;
          }
        }
      }
    };
    if (vrows >= BM)
      pipeline(std::false_type{});
    else
      pipeline(std::true_type{});
    cur = next;
  }
  if (wm == 0) wg_barrier();
  wait_cnt<0>();   // no load may write this workgroup's LDS after its end
}

// Smaller tiles, for lists that leave CUs idle (or a nearly empty last round) with 256 x 256 ones
// (choose_tile): TM = 16 WM MI rows by TN = 16 WN NI weight rows per workgroup of WM x WN
// wavefronts, each with MI x NI 16 x 16 accumulators.  Such a launch is one or two rounds of tiles,
// so a tile's latency is what counts: its stages (64 columns of K) stream through an LDS ring as
// deep as 144 KiB allows (3 to 9 stages for the five shapes below), the loads of a stage spread
// between the matrix instructions; a wavefront's fragments of the next 32 columns are read while
// the current ones are multiplied.  The loads of one CU reach it at about 64 bytes a clock, which a
// 64 x 64 tile needs for 256 clocks of 128 clocks of products a stage: below that size nothing is
// gained.  Stage time at full occupancy, us (256 x 256: 1.3): 256 x 128 and 128 x 256 0.8,
// 128 x 128 0.5, 64 x 128 0.38, 64 x 64 0.3.  128 x 128 with four wavefronts of 64 x 64 took 0.6
// (a wavefront alone on its SIMD stalls on its loads' issue), with eight of 64 x 32 0.52.
// Products, K order, operand layout in LDS and roundings are those of ffn_tiled, so the outputs
// do not depend on the tile.

// wait until at most y groups of LPS vector-memory operations are outstanding (y wave-uniform,
// values above V count as V)
template <int V, int LPS>
__device__ __forceinline__ void wait_groups(int y) {
  if constexpr (V == 0) {
    wait_cnt<0>();
  } else {
    if (y >= V)
      wait_cnt<V * LPS>();
    else
      wait_groups<V - 1, LPS>(y);
  }
}

template <int MODE, int WM, int WN, int MI, int NI>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(WM * WN / 4, WM * WN / 4))) void ffn_tile(FfnArgs a) {
  constexpr int W = WM * WN;
  constexpr int TM = 16 * WM * MI, TN = 16 * WN * NI;    // tile rows and weight rows
  constexpr int kStage = (TM + TN) * kRowBytes;
  constexpr int SST = 147456 / kStage;                   // stages: 128 or 144 KiB
  constexpr int LA = TM / (8 * W), LB = TN / (8 * W);    // direct loads per wavefront and stage
  constexpr int LPS = LA + LB;
  // phase 1 with one gate and one up tile per wavefront: weight rows in order (else interleaved)
  constexpr bool INORD = MODE == 0 && NI == 2;
  __shared__ TileTable tt;
  __shared__ __attribute__((aligned(1024))) char smem[SST * kStage];
  __shared__ __attribute__((aligned(256))) int32_t row_s[MODE == 1 ? TM : 1], col_s[MODE == 1 ? TM : 1];
  __shared__ int32_t orow_s[MODE == 1 ? TM : 1];
  __shared__ float wt_s[MODE == 1 ? TM : 1];
  build_tile_table<TM>(a, tt);
  const int64_t K = MODE == 0 ? a.H : a.I;
  const int ntn = MODE == 0 ? (int)(a.I / (TN / 2)) : (int)(a.H / TN);
  const int total = tt.total * ntn;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int KT = (int)(K / BK);   // at least 2
  const int j16 = lane & 15, g4 = lane >> 4;
  const uint32_t smem0 = lds_addr(smem);
  auto swz_w = [](int row) { return INORD ? swz_a(row) : swz_b(row); };
  // fragment reads: K step ks of A tile i (rows 32 i + 16 wm + j16) and of weight tile c.  Phase 1:
  // gate columns (TN / 4) wn + ... for c < NI / 2, the same up columns for the others; phase 2:
  // columns (TN / 2) wn + ...; pairs of tiles interleaved as in ffn_tiled
  uint32_t a_addr[2], b_addr[2];
  constexpr int kPair = (MODE == 0 ? TN / 2 : 32) * kRowBytes;   // from tiles c < NI / 2 to the others
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int arow = 16 * wm + j16;
    const int brow = INORD ? 16 * wn + j16 : 16 * (MODE == 0 ? NI / 2 : NI) * wn + 8 * (j16 >> 2) + (j16 & 3);
    a_addr[ks] = (uint32_t)(arow * kRowBytes + (((4 * ks + g4) ^ swz_a(arow)) << 4));
    b_addr[ks] = (uint32_t)((TM + brow) * kRowBytes + (((4 * ks + g4) ^ swz_w(brow)) << 4));
  }
  const int per_xcd = gridDim.x % 8 == 0 ? (int)gridDim.x / 8 : 0;
  const int lslot = per_xcd ? (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  for (int tile = lslot; tile < total; tile += gridDim.x) {
    const int mt_global = tile / ntn, ntile = tile % ntn;
    const int li = find_entry(tt, mt_global);
    const int64_t start = tt.start[li];
    const int n = tt.rows[li];
    const int m0 = (mt_global - tt.cum[li]) * TM;
    const int vrows = n - m0;   // > 0
    const bf16_t* slot = a.cache + (int64_t)a.list.slot[li] * 3 * a.H * a.I;
    // direct loads: this wavefront moves A rows 8 MI wave + 8 q + lane / 8 (q < MI) and weight rows
    // 8 NI wave + 8 q + lane / 8 (q < NI)
    const int r8 = lane >> 3, slot8 = lane & 7;
    uint32_t aoff[LA], boff[LB];
    const char* abase = reinterpret_cast<const char*>(MODE == 0 ? a.x : a.act);
    const uint32_t lda = (uint32_t)K;
#pragma unroll
    for (int q = 0; q < LA; ++q) {
      const int row = 8 * LA * wave + 8 * q + r8;
      const int r = m0 + row;
      const bool ok = r < n;
      const uint32_t t = MODE == 0 ? (uint32_t)a.rows[start + (ok ? r : 0)]
                                   : (uint32_t)(start + (ok ? r : 0));
      aoff[q] = (t * lda + (uint32_t)((slot8 ^ swz_a(row)) * 8)) * 2u;
    }
#pragma unroll
    for (int q = 0; q < LB; ++q) {
      const int row = 8 * LB * wave + 8 * q + r8;
      boff[q] = (uint32_t)(((uint32_t)(8 * q + r8) * (uint32_t)K + (uint32_t)((slot8 ^ swz_w(row)) * 8)) * 2u);
    }
    // phase 1: the first TN / 2 weight rows are gate, the others up columns (TN / 2) ntile + ...
    const int brow0 = 8 * LB * wave;
    const char* bbase = reinterpret_cast<const char*>(uniform_ptr(
        MODE == 0 ? slot + (brow0 < TN / 2 ? (int64_t)(ntile * (TN / 2) + brow0) * a.H
                                           : a.H * a.I + (int64_t)(ntile * (TN / 2) + brow0 - TN / 2) * a.H)
                  : slot + 2 * a.H * a.I + (int64_t)(ntile * TN + brow0) * a.I));
    if (MODE == 1 && 64 * wave < TM) {
      // the tile rows' token and slot indices (low words) of rows 64 wave + lane: the oldest loads
      // of the tile, so they have landed when the first stage has
      const int r = 64 * wave + lane;
      const int64_t p = start + m0;
      const uint32_t off = (uint32_t)((r < vrows ? r : 0) * 8);
      dma4(reinterpret_cast<const char*>(uniform_ptr(a.rows + p)), off, lds_addr(row_s) + 256 * wave);
      dma4(reinterpret_cast<const char*>(uniform_ptr(a.cols + p)), off, lds_addr(col_s) + 256 * wave);
    }
    floatx4 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int c = 0; c < NI; ++c) acc[i][c] = floatx4{0, 0, 0, 0};
    // 16-row tiles of this wavefront that hold rows of the expert
    const int v = vrows - 16 * wm;
    const int nf = __builtin_amdgcn_readfirstlane(v <= 0 ? 0 : ((v + 16 * WM - 1) / (16 * WM) < MI ? (v + 16 * WM - 1) / (16 * WM) : MI));
    auto dma = [&](int kt, int sl, auto qq) {   // load q of stage kt into slot sl: A rows for q < MI
      constexpr int q = decltype(qq)::value;
      const uint32_t dst = smem0 + (uint32_t)(sl * kStage);
      if constexpr (q < LA)
        dma16(abase + kt * BK * 2, aoff[q], dst + (uint32_t)((8 * LA * wave + 8 * q) * kRowBytes));
      else
        dma16(bbase + kt * BK * 2, boff[q - LA], dst + (uint32_t)((TM + 8 * LB * wave + 8 * (q - LA)) * kRowBytes));
    };
    auto read = [&](int sl, int ks, bf16x8 (&ft)[MI], bf16x8 (&fw)[NI]) {
      const char* st = smem + sl * kStage;
#pragma unroll
      for (int c = 0; c < NI; ++c)
        fw[c] = *reinterpret_cast<const bf16x8*>(
            st + b_addr[ks] + (INORD ? c * kPair : (c >> 1) * kPair + (c & 1) * 4 * kRowBytes));
#pragma unroll
      for (int i = 0; i < MI; ++i)
        ft[i] = *reinterpret_cast<const bf16x8*>(st + a_addr[ks] + i * 16 * WM * kRowBytes);
    };
    auto mma = [&](int i, const bf16x8 (&ft)[MI], const bf16x8 (&fw)[NI]) {
      if (i < nf) {
#pragma unroll
        for (int c = 0; c < NI; ++c)
          acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[c], ft[i], acc[i][c], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    bf16x8 t0[MI], w0[NI], t1[MI], w1[NI];
    for (int k = 0; k < (SST < KT ? SST : KT); ++k)
      static_for<0, LPS>([&](auto q) { dma(k, k, q); });
    wait_groups<SST - 1, LPS>(KT - 1);
    wg_barrier();
    // phase 2: the output row and routing weight of row tid, loaded under the K loop
    int32_t my_orow = 0;
    float my_wt = 0.f;
    if (MODE == 1 && tid < TM) {
      const int64_t tj = (int64_t)row_s[tid] * a.k + col_s[tid];
      my_wt = bf16_to_f32(a.w[tj]);
      my_orow = a.out_mode == 0 ? (int32_t)tj : (int32_t)(start + m0 + tid);
    }
    read(0, 0, t0, w0);
    int cur = 0;   // slot of stage k
    for (int k = 0; k < KT; ++k) {
      const int nxt = cur + 1 == SST ? 0 : cur + 1;
      read(cur, 1, t1, w1);
#pragma unroll
      for (int i = 0; i < MI; ++i) mma(i, t0, w0);
      // stage k is read by this wavefront, its loads of stage k + 1 have landed
      wait_groups<SST - 2, LPS>(KT - 2 - k);
      wg_barrier();
      if (k + 1 < KT) read(nxt, 0, t0, w0);
      const bool more = k + SST < KT;
      static_for<0, MI>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        if (more)   // a share of the loads into the buffer of stage k
          static_for<i * LPS / MI, (i + 1) * LPS / MI>([&](auto q) { dma(k + SST, cur, q); });
        mma(i, t1, w1);
      });
      cur = nxt;
    }
    if (MODE == 1) {
      if (tid < TM) {
        orow_s[tid] = my_orow;
        wt_s[tid] = my_wt;
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int r = 16 * WM * i + 16 * wm + j16;
      if constexpr (MODE == 0) {
        uint32_t y[NI];
#pragma unroll
        for (int c = 0; c < NI / 2; ++c)
#pragma unroll
          for (int q = 0; q < 4; q += 2) {
            const uint32_t gp = pk_bf16(acc[i][c][q], acc[i][c][q + 1]);
            const uint32_t up = pk_bf16(acc[i][NI / 2 + c][q], acc[i][NI / 2 + c][q + 1]);
            const float s0 = silu_mul(__uint_as_float(gp << 16), __uint_as_float(up << 16));
            const float s1 = silu_mul(__uint_as_float(gp & 0xffff0000u), __uint_as_float(up & 0xffff0000u));
            y[2 * c + q / 2] = pk_bf16(s0, s1);
          }
        bf16_t* const o = a.act + (start + m0 + r) * a.I + ntile * (TN / 2) + wn * (8 * NI) + 2 * NI * g4;
        if (r < vrows) {
          if constexpr (NI == 4)
            *reinterpret_cast<u32x4*>(o) = u32x4{y[0], y[1], y[2], y[3]};
          else
            *reinterpret_cast<u32x2*>(o) = u32x2{y[0], y[1]};
        }
      } else {
        const float wt = wt_s[r];
        bf16_t* const o = a.out + (int64_t)orow_s[r] * a.H + ntile * TN + wn * (16 * NI) + 8 * g4;
#pragma unroll
        for (int hb = 0; hb < NI / 2; ++hb) {
          u32x4 y;
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int q = 0; q < 4; q += 2) {
              const uint32_t v2 = pk_bf16(acc[i][2 * hb + c][q], acc[i][2 * hb + c][q + 1]);
              y[2 * c + q / 2] = pk_bf16(__uint_as_float(v2 << 16) * wt,
                                         __uint_as_float(v2 & 0xffff0000u) * wt);
            }
          if (r < vrows) *reinterpret_cast<u32x4*>(o + 32 * hb) = y;
        }
      }
    }
    if (MODE == 1) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      wg_barrier();
    }
  }
}

int g_num_cus = 0;

// Device addresses of g_sync / g_sync_timeouts on each device (resolved on first use there).
constexpr int kMaxDevices = 64;
std::mutex g_sync_mu;
uint32_t* g_sync_dev[kMaxDevices];
int32_t* g_timeouts_dev[kMaxDevices];
std::atomic<uint32_t> g_epoch{0};
std::atomic<int32_t> g_spin_limit{kSyncSpinLimit};

int sync_addresses(uint32_t** sync, int32_t** timeouts) {
  int dev = -1;
  FERRY_HIP(hipGetDevice(&dev));
  FERRY_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_sync_mu);
  if (g_sync_dev[dev] == nullptr) {
    void* ps = nullptr;
    void* pt = nullptr;
    FERRY_HIP(hipGetSymbolAddress(&ps, HIP_SYMBOL(g_sync)));
    FERRY_HIP(hipGetSymbolAddress(&pt, HIP_SYMBOL(g_sync_timeouts)));
    g_sync_dev[dev] = (uint32_t*)ps;
    g_timeouts_dev[dev] = (int32_t*)pt;
  }
  *sync = g_sync_dev[dev];
  *timeouts = g_timeouts_dev[dev];
  return 0;
}

}  // namespace

// device address of the fused decode kernel's timeout counter on the current device (for the
// history kernel's copy of it)
int ffn_timeouts_address(int32_t** timeouts) {
  uint32_t* sync = nullptr;
  return sync_addresses(&sync, timeouts);
}

}  // namespace ferry

using namespace ferry;

// M tiles of a list's experts with more than 64 rows, for tiles of 64 << i rows (0: row counts
// unknown)
struct MTiles {
  int64_t n[3] = {0, 0, 0};
};
static int ffn_launch_list(FfnArgs& args, const int32_t* expert_list, const int32_t* slot_of,
                           int32_t n_list, int32_t n_mid, int64_t maxn, int64_t min_rows,
                           int64_t pairs, const MTiles& mt, int32_t phases, int64_t hidden,
                           int64_t inter, int64_t tiled_cus, hipStream_t s);

static int expert_ffn_call(const void* cache, int64_t cache_rows, int64_t hidden,
                                int64_t inter, const void* x, int64_t rows_in, int64_t topk,
                                const void* w_sorted, const int64_t* starts, const int64_t* rows,
                                const int64_t* cols, const int32_t* expert_list, int32_t n_list,
                                const int32_t* slot_of, int64_t experts,
                                int64_t max_rows_per_expert, int64_t min_rows_per_expert,
                                const int32_t* list_rows, void* act, void* out,
                                int32_t out_mode, int32_t phases, int32_t spare_cus, void* stream) {
  clear_error();
  FERRY_CHECK_ARG(phases >= 1 && phases <= 3, "phases must be 1 (up), 2 (down) or 3 (both)");
  FERRY_CHECK_ARG(hidden > 0 && hidden % 128 == 0, "hidden must be a positive multiple of 128");
  FERRY_CHECK_ARG(inter > 0 && inter % 128 == 0, "intermediate must be a positive multiple of 128");
  FERRY_CHECK_ARG(topk >= 1 && rows_in >= 0 && n_list >= 0 && max_rows_per_expert >= 0,
                  "bad sizes");
  FERRY_CHECK_ARG(min_rows_per_expert >= 0 && min_rows_per_expert <= max_rows_per_expert,
                  "min_rows_per_expert must be in [0, max_rows_per_expert]");
  FERRY_CHECK_ARG(experts >= 1 && experts <= FERRY_MAX_EXPERTS, "experts must be in [1, %d]",
                  FERRY_MAX_EXPERTS);
  FERRY_CHECK_ARG(out_mode == 0 || out_mode == 1, "out_mode must be 0 or 1");
  FERRY_CHECK_ARG(spare_cus >= 0 && spare_cus <= 128, "spare_cus must be in [0, 128]");
  // the tiled down projection covers the hidden dimension in 256-column tiles
  FERRY_CHECK_ARG(hidden % 256 == 0 || max_rows_per_expert <= kSkinnyMax,
                  "hidden must be a multiple of 256 when an expert has more than %d rows",
                  kSkinnyMax);
  FERRY_CHECK_ARG(rows_in * topk < (int64_t)1 << 31, "rows*topk must be < 2^31");
  // the kernels address weights with 32-bit byte offsets from the expert's cache row
  FERRY_CHECK_ARG(3 * hidden * inter * 2 < ((int64_t)1 << 32),
                  "an expert's cache row (3 * hidden * intermediate bf16) must be under 4 GiB");
  // the tiled kernels address A rows with 32-bit byte offsets
  FERRY_CHECK_ARG(rows_in * hidden < ((int64_t)1 << 31) &&
                      rows_in * topk * inter < ((int64_t)1 << 31),
                  "x / act must hold fewer than 2^31 elements");
  if (n_list == 0 || rows_in == 0) return 0;
  FERRY_CHECK_ARG(cache && x && w_sorted && starts && rows && cols && expert_list && slot_of &&
                      act && out,
                  "null pointer argument");
  for (int32_t i = 0; i < n_list; ++i) {
    const int32_t e = expert_list[i];
    FERRY_CHECK_ARG(e >= 0 && e < experts, "expert_list[%d] = %d out of range", i, e);
    const int32_t s = slot_of[e];
    FERRY_CHECK_ARG(s >= 0 && s < cache_rows, "expert %d is not cached (slot %d)", e, s);
    if (list_rows)
      FERRY_CHECK_ARG(list_rows[i] >= min_rows_per_expert && list_rows[i] <= max_rows_per_expert,
                      "list_rows[%d] = %d outside [min_rows_per_expert, max_rows_per_expert]", i,
                      list_rows[i]);
  }
  if (g_num_cus == 0) {
    int dev = 0, cus = 0;
    FERRY_HIP(hipGetDevice(&dev));
    FERRY_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    g_num_cus = cus > 0 ? cus : 256;
  }
  hipStream_t s = (hipStream_t)stream;
  FfnArgs args;
  args.cache = (const bf16_t*)cache;
  args.x = (const bf16_t*)x;
  args.w = (const bf16_t*)w_sorted;
  args.starts = starts;
  args.rows = rows;
  args.cols = cols;
  args.act = (bf16_t*)act;
  args.out = (bf16_t*)out;
  args.H = hidden;
  args.I = inter;
  args.k = topk;
  args.out_mode = out_mode;
  const int64_t tiled_cus = g_num_cus > 2 * spare_cus ? g_num_cus - spare_cus : g_num_cus;
  // max_rows_per_expert must bound every n_e from above (rows_in does for a layout from
  // ferry_layout) and min_rows_per_expert from below (0 when unknown); the kernels size their
  // work from the device starts, the bounds only select and gate the launches.  With the
  // entries' row counts (list_rows) the list is issued as two lists with exact bounds: the
  // small experts (1-64 rows; those with 17-64 rows first), then the tiled ones (the small
  // launches measured slower after the tiled ones, whose output writes they then meet); experts
  // without rows are left out.
  if (!list_rows)
    return ffn_launch_list(args, expert_list, slot_of, n_list, n_list, max_rows_per_expert,
                           min_rows_per_expert, rows_in * topk, MTiles{}, phases, hidden, inter, tiled_cus, s);
  std::vector<int32_t> small, big;
  int32_t n_mid = 0;
  MTiles mt;
  int64_t small_max = 0, small_min = kSkinnyMax, big_max = 0, big_min = INT64_MAX;
  for (int pass = 0; pass < 2; ++pass)   // 17-64 rows, then 1-16 rows
    for (int32_t i = 0; i < n_list; ++i) {
      const int64_t r = list_rows[i];
      if (r > 16 && r <= kSkinnyMax && pass == 0) small.push_back(expert_list[i]), ++n_mid;
      if (r >= 1 && r <= 16 && pass == 1) small.push_back(expert_list[i]);
      if (r >= 1 && r <= kSkinnyMax && pass == 0) {
        small_max = r > small_max ? r : small_max;
        small_min = r < small_min ? r : small_min;
      }
      if (r > kSkinnyMax && pass == 0) {
        big.push_back(expert_list[i]);
        big_max = r > big_max ? r : big_max;
        big_min = r < big_min ? r : big_min;
        for (int i = 0; i < 3; ++i) mt.n[i] += ceil_div(r, 64 << i);
      }
    }
  if (!small.empty()) {
    const int rc = ffn_launch_list(args, small.data(), slot_of, (int32_t)small.size(), n_mid,
                                   small_max, small_min, rows_in * topk, MTiles{}, phases, hidden,
                                   inter, tiled_cus, s);
    if (rc != 0) return rc;
  }
  if (!big.empty())
    return ffn_launch_list(args, big.data(), slot_of, (int32_t)big.size(), 0, big_max, big_min,
                           rows_in * topk, mt, phases, hidden, inter, tiled_cus, s);
  return 0;
}

extern "C" int ferry_expert_ffn(const void* cache, int64_t cache_rows, int64_t hidden,
                                int64_t inter, const void* x, int64_t rows_in, int64_t topk,
                                const void* w_sorted, const int64_t* starts, const int64_t* rows,
                                const int64_t* cols, const int32_t* expert_list, int32_t n_list,
                                const int32_t* slot_of, int64_t experts,
                                int64_t max_rows_per_expert, int64_t min_rows_per_expert,
                                const int32_t* list_rows, void* act, void* out,
                                int32_t out_mode, int32_t phases, void* stream) {
  return expert_ffn_call(cache, cache_rows, hidden, inter, x, rows_in, topk, w_sorted, starts, rows, cols,
                         expert_list, n_list, slot_of, experts, max_rows_per_expert,
                         min_rows_per_expert, list_rows, act, out, out_mode, phases, 0, stream);
}

extern "C" int ferry_expert_ffn_spare(const void* cache, int64_t cache_rows, int64_t hidden,
                                      int64_t inter, const void* x, int64_t rows_in, int64_t topk,
                                      const void* w_sorted, const int64_t* starts,
                                      const int64_t* rows, const int64_t* cols,
                                      const int32_t* expert_list, int32_t n_list,
                                      const int32_t* slot_of, int64_t experts,
                                      int64_t max_rows_per_expert, int64_t min_rows_per_expert,
                                      const int32_t* list_rows, void* act, void* out,
                                      int32_t out_mode, int32_t phases, int32_t spare_cus,
                                      void* stream) {
  return expert_ffn_call(cache, cache_rows, hidden, inter, x, rows_in, topk, w_sorted, starts, rows, cols,
                         expert_list, n_list, slot_of, experts, max_rows_per_expert,
                         min_rows_per_expert, list_rows, act, out, out_mode, phases, spare_cus, stream);
}

// Which tile a list's tiled experts take: the one whose rounds of one tile per CU cost least.  A
// tile costs kt stages of K plus a fixed part (tile table, row indices, first loads, epilogue); the
// figures are fitted to launches of 1-64 experts of 65-4096 rows, H x I = 2048 x 768 / 1408 / 2816.
// Over 2 x 97 of those the choice costs 0.8 % more than the best tile on average, 14 % at worst (64
// experts of 65 rows: 1.5 rounds).  A small tile has less latency, a large one less traffic per
// product; so a list that leaves CUs idle with large tiles takes smaller ones.  us, 256 x 256 ->
// chosen: shared expert (2048 x 2816) of 256 rows 36.6 -> 17.2 up, 47.0 -> 18.2 down, of 777 rows
// 37.8 -> 30.8 and 47.9 -> 20.8; 8 experts (2048 x 1408) of 128 rows 36.3 -> 24.6 and 24.5 -> 13.8;
// 24 experts (2048 x 768) of 100 rows 43.8 -> 41.9.  No choice beats reading the list's weights at
// 4.5 TB/s, and the 256 x 256 tile is preferred by 5 % (its loop is the better one when full).
// The whole list takes one tile.  Lists without row counts take 256 x 256 tiles.
struct TileCost {
  int rows_log, cols;    // 64 << rows_log rows, weight rows
  double stage, fixed;   // us
};
static const TileCost kTiles[] = {{2, 256, 1.3, 7.0}, {2, 128, 0.8, 6.0}, {1, 256, 0.8, 6.0},
                                  {1, 128, 0.5, 5.0}, {0, 128, 0.38, 4.0}, {0, 64, 0.3, 3.5}};
static int choose_tile(const MTiles& mt, int64_t experts, int64_t cols, int64_t k, int64_t cus) {
  const double read = (double)(experts * cols * k * 2) / 4.5e6 + 1.0;
  int best = 0;
  double least = 0;
  for (int i = 0; i < 6; ++i) {
    const int64_t tiles = mt.n[kTiles[i].rows_log] * (cols / kTiles[i].cols);
    const double t = (double)ceil_div(tiles, cus) * ((double)(k / BK) * kTiles[i].stage + kTiles[i].fixed);
    const double cost = (t > read ? t : read) * (i == 0 ? 0.95 : 1.0);
    if (i == 0 || cost < least) best = i, least = cost;
  }
  return best;
}

// The tiled experts of a list, one phase (MODE 0: up, 1: down).
template <int MODE>
static int tiled_launch(const FfnArgs& args, const MTiles& mt, int64_t pairs, int64_t cus, hipStream_t s) {
  const char* name = MODE == 0 ? "ffn_tiled_up" : "ffn_tiled_down";
  const int64_t cols = MODE == 0 ? 2 * args.I : args.H;   // weight rows of an expert
  const int c = mt.n[0] == 0 ? 0 : choose_tile(mt, args.list.n, cols, MODE == 0 ? args.H : args.I, cus);
  auto go = [&](auto kernel, int threads, int64_t tiles) {
    launch(name, kernel, dim3((unsigned)(tiles < cus ? tiles : cus)), dim3(threads), 0, s, args);
  };
  const int64_t tiles = mt.n[kTiles[c].rows_log] * (cols / kTiles[c].cols);
  switch (c) {
    case 0:
      // M tiles over experts with > 64 rows when the row counts are unknown:
      // sum ceil(n/BM) <= pairs/BM + (experts with > 64 rows), and those are <= pairs/65
      go(ffn_tiled<MODE>, kTiledThreads,
         mt.n[0] ? tiles : (pairs / BM + pairs / (kSkinnyMax + 1) + 1) * (cols / BN));
      break;
    case 1: go(ffn_tile<MODE, 4, 2, 4, 4>, 512, tiles); break;
    case 2: go(ffn_tile<MODE, 2, 4, 4, 4>, 512, tiles); break;
    case 3: go(ffn_tile<MODE, 4, 2, 2, 4>, 512, tiles); break;
    case 4: go(ffn_tile<MODE, 2, 4, 2, 2>, 512, tiles); break;
    default: go(ffn_tile<MODE, 2, 2, 2, 2>, 256, tiles);
  }
  FERRY_LAUNCHED(name);
  return 0;
}

// One-launch decode: down workgroups of 16 hidden rows (DownRows16) instead of 64 for a list of cnt
// experts?  They shorten each workgroup's chain of loads, and pay while the workgroups of 64 rows
// (wgs) leave CUs idle; past that, four times as many workgroups read the activation rows.  The limit
// also depends on what they replace: workgroups of 64 rows, which read whole 128-byte pieces of the
// weight rows only where I is a multiple of 256, and above kWideInter two launches.  Measured for 32
// H x I of 512-7168 x 512-2816, 1 to 16 experts of 1 and of 16 rows, time relative to those, 1 row an
// expert - 16 rows:
//   K range of up to 3 chunks (of 64 columns, per wavefront): 0.87-0.95 up to an eighth of the CUs,
//     768 x 2048 then 1.02-1.10
//   I a multiple of 256, up to 2048: at half the CUs 0.87-0.92 (H = 2048), 0.93-1.00 (4096); at 3/4
//     0.97-1.03 and 0.95-1.04, at all of them 1.03-1.14 and 0.96-1.04
//   I of 2304 to 2816: below half the CUs 0.75-1.00, at half 0.85-0.99 (H = 2048) and 0.93-1.07
//     (4096); 8 experts 0.83-1.02, 12 experts 0.93-1.07 (H = 512)
//   other I: at 5/8 of the CUs 0.79-1.02; 1152 to 1920 at all of them 0.84-1.01 (H up to 5120), 7168 x
//     1408 already 1.00-1.05 at 7/8; 896 at 3/4 0.97-1.05; 2688 at all of them 0.94-1.04
// e.g. us, 64 -> 16 rows, 16 rows an expert, H = 2048: I = 1408, 1 expert 17.9 -> 12.7, 3 experts 26.4
// -> 21.4, 8 experts 37.0 -> 34.4; I = 768, 1 expert 11.0 -> 10.5; the 2048 x 2816 shared expert, from
// two launches, 20.7 -> 17.2 (1 row: 19.8 -> 14.4).  I = 3072 to 4096 in one launch of 64-row workgroups
// took 1.04 to 1.23 times the two launches (1 to 6 experts of 16 rows), so they keep those.
constexpr int kNarrowChunks = 11;    // the longest K range of DownRows16: I <= 2816
constexpr int kWideInter = 2048;     // largest I of a launch with workgroups of 64 rows
static bool narrow_down(int64_t cnt, int64_t hidden, int64_t inter) {
  const int64_t chunks = ceil_div(ceil_div(inter / 32, 4), 2), wgs = cnt * (hidden / 64), cus = g_num_cus;
  if (chunks <= 3) return wgs <= cus / 8;
  if (chunks > kNarrowChunks) return false;
  if (inter % 256 == 0 && inter <= kWideInter) return wgs <= cus / 2;
  if (inter % 256 == 0) return wgs <= (hidden <= 2048 ? cus / 2 : cus / 2 - 1) && cnt <= 8;
  return wgs <= (chunks >= 5 && chunks <= 8 && hidden <= 5120 ? cus : cus * 5 / 8);
}

// Is work on s being captured into a graph?  (The null stream cannot be captured, and is not asked.)
static bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (s == nullptr) return false;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();   // the launch that follows reports what is wrong with the stream
    return false;
  }
  return st != hipStreamCaptureStatusNone;
}

// The launches of one list: n_mid of its leading entries are known to hold 17-64 rows (the
// small-expert up launch gives them 64-column workgroups; the others get 16-column ones unless
// the bounds allow no expert of more than 16 rows, n_mid = n_list when unknown).
static int ffn_launch_list(FfnArgs& args, const int32_t* expert_list, const int32_t* slot_of,
                           int32_t n_list, int32_t n_mid, int64_t maxn, int64_t min_rows,
                           int64_t pairs, const MTiles& mt, int32_t phases, int64_t hidden,
                           int64_t inter, int64_t tiled_cus, hipStream_t s) {
  const bool any_small = min_rows <= kSkinnyMax;
  for (int32_t off = 0; off < n_list; off += kListMax) {
    const int32_t cnt = (n_list - off) < kListMax ? (n_list - off) : kListMax;
    args.list.n = cnt;
    const int32_t mid_left = n_mid - off;
    args.list.n_mid = mid_left < 0 ? 0 : (mid_left < cnt ? mid_left : cnt);
    for (int32_t i = 0; i < kListMax; ++i) {
      args.list.expert[i] = (int16_t)(i < cnt ? expert_list[off + i] : 0);
      args.list.slot[i] = i < cnt ? slot_of[expert_list[off + i]] : 0;
    }
    const bool any_big = maxn > kSkinnyMax;
    const int64_t grid_cap = tiled_cus;  // one tiled workgroup per CU
    // Decode: both phases in one launch, each expert's down projection as soon as its up projection is
    // stored.  Not in a graph: its replays would all carry the captured epoch, whose flags the first
    // of them leaves set, so a later one's down projections would not wait.
    const bool narrow = narrow_down(cnt, hidden, inter);
    if (phases == 3 && any_small && !any_big && maxn <= 16 && (inter <= kWideInter || narrow) && !capturing(s)) {
      FusedSync fs;
      uint32_t* sync = nullptr;
      const int rc = sync_addresses(&sync, &fs.timeouts);
      if (rc != 0) return rc;
      uint32_t epoch = ++g_epoch;
      if (epoch == 0) epoch = ++g_epoch;   // epoch 0 would match never-used words
      fs.epoch = epoch;
      fs.flags = sync + (int64_t)(epoch % kSyncSets) * kListMax * kMaxUpWgs;
      fs.up_wgs = (int32_t)(inter / 16);
      fs.spin_limit = g_spin_limit.load();
      const int64_t chunks = ceil_div(ceil_div(inter / 32, 4), 2);
      fs.down_wgs = (int32_t)(hidden / (narrow ? 16 : 64));
      launch("ffn_skinny_fused",
             !narrow ? ffn_skinny_fused<0>
                     : (chunks <= 3 ? ffn_skinny_fused<3> : (chunks <= 6 ? ffn_skinny_fused<6> : ffn_skinny_fused<11>)),
             dim3((unsigned)((fs.up_wgs + fs.down_wgs) * cnt)), dim3(256), 0, s, args, fs);
      FERRY_LAUNCHED("ffn_skinny_fused");
      continue;
    }
    if (phases & 1) {
      // 16 intermediate columns per workgroup, K split over the four wavefronts
      if (any_small) {
        const dim3 g1((unsigned)(inter / 16), cnt);
        const int64_t wgs = args.list.n_mid * (inter / 64) + (cnt - args.list.n_mid) * (inter / 16);
        if (maxn <= 16)
          launch("ffn_up_skinny", ffn_up_skinny<1>, g1, dim3(256), 0, s, args);
        else
          launch("ffn_up_skinny", ffn_up_skinny<4>, dim3((unsigned)wgs), dim3(256), 0, s, args);
        FERRY_LAUNCHED("ffn_up_skinny");
      }
      if (any_big) {
        const int rc = tiled_launch<0>(args, mt, pairs, grid_cap, s);
        if (rc != 0) return rc;
      }
    }
    if (phases & 2) {
      // 64 hidden rows per workgroup
      if (any_small) {
        const dim3 g2((unsigned)(hidden / 64), cnt);
        if (maxn <= 16)
          launch("ffn_down_skinny", ffn_down_skinny<1>, g2, dim3(256), 0, s, args);
        else
          launch("ffn_down_skinny", ffn_down_skinny<4>, g2, dim3(256), 0, s, args);
        FERRY_LAUNCHED("ffn_down_skinny");
      }
      if (any_big) {
        const int rc = tiled_launch<1>(args, mt, pairs, grid_cap, s);
        if (rc != 0) return rc;
      }
    }
  }
  return 0;
}

// Number of fused decode launches whose down phase gave up waiting for its up phase (each such
// workgroup left its rows unwritten); 0 unless workgroups were not dispatched in index order.
extern "C" int ferry_expert_ffn_sync_timeouts(int64_t* count) {
  clear_error();
  FERRY_CHECK_ARG(count, "null pointer argument");
  uint32_t* sync = nullptr;
  int32_t* timeouts = nullptr;
  const int rc = sync_addresses(&sync, &timeouts);
  if (rc != 0) return rc;
  int32_t v = 0;
  FERRY_HIP(hipMemcpy(&v, timeouts, sizeof(v), hipMemcpyDeviceToHost));
  *count = v;
  return 0;
}

// How many times a fused decode launch's down workgroup polls its up workgroups' flags before
// giving up (limit < 0: the default, about a second of polling; 0: it gives up without polling,
// so that a caller can check how a timeout is reported).  Applies to launches made after it.
extern "C" int ferry_expert_ffn_set_sync_spin_limit(int64_t limit) {
  clear_error();
  FERRY_CHECK_ARG(limit < ((int64_t)1 << 30), "spin limit must be below 2^30");
  g_spin_limit.store(limit < 0 ? kSyncSpinLimit : (int32_t)limit);
  return 0;
}
