// Router logits of a gate with bf16 weights, in fp32: out[T, E] = fp32(x) fp32(w)^T.
//
// Reference: the DeepSeek-V2 gate that feeds ferry/model.py:151-158 (HF's
// F.linear(hidden.float(), weight.float())).  A product of two bf16 values is exact in fp32, so
// the bf16 matrix instructions with fp32 accumulators give the sums of the fp32 product without
// the fp32 copies of x and w; only the order of the additions differs.
#include "common.h"

namespace ferry {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// One workgroup computes 16*MI rows x 16*NI experts; its WAVES wavefronts take every WAVES-th
// 64-element chunk of the hidden dimension and their partial tiles are added through LDS, in
// wavefront order.  Operands go from global memory to registers, one chunk ahead: lane l holds
// 16 consecutive values of row l % 16, from (l / 16) * 16 of the chunk on, so that a row's 128
// bytes are read by one instruction pair; both operands place their values alike, which is all
// the matrix instruction needs of the order along K.
// Small calls are bound by the latency of the loads and the LDS sum, large ones by reading x.  At
// 65,536 x 2048 x 64 the library's fp32 copies and product took 290 us and this takes 70; at 256
// rows 29 and 5.4.  Error of the sums against 64 bits, relative: 0.6e-7 to 0.8e-7 over 1 to 65,536
// rows, where the library's was 0.9e-7 to 4.6e-7.
template <int MI, int NI, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void gate_kernel(const bf16_t* __restrict__ x,
                                                          int64_t tokens, int hidden,
                                                          const bf16_t* __restrict__ w,
                                                          int experts, float* __restrict__ out) {
  constexpr int M = 16 * MI, N = 16 * NI, LD = N + 4;   // + 4: a tile's 4 row groups on 4 x 16 banks
  __shared__ float part[WAVES][M][LD];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t t0 = (int64_t)blockIdx.x * M;
  const int e0 = blockIdx.y * N;
  const int row = lane & 15, k0 = (lane >> 4) * 16;
  const bf16_t* a[MI];
  const bf16_t* b[NI];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int64_t t = t0 + 16 * i + row;
    a[i] = x + (t < tokens ? t : tokens - 1) * hidden + k0;
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int e = e0 + 16 * i + row;
    b[i] = w + (int64_t)(e < experts ? e : experts - 1) * hidden + k0;
  }
  f32x4 acc[MI][NI] = {};
  bf16x8 av[MI][2], bv[NI][2], an[MI][2], bn[NI][2];
  const int chunks = hidden >> 6;
  auto load = [&](int c, bf16x8 (&pa)[MI][2], bf16x8 (&pb)[NI][2]) {
    const int k = c * 64;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      pa[i][0] = *(const bf16x8*)(a[i] + k);
      pa[i][1] = *(const bf16x8*)(a[i] + k + 8);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      pb[i][0] = *(const bf16x8*)(b[i] + k);
      pb[i][1] = *(const bf16x8*)(b[i] + k + 8);
    }
  };
  if (wave < chunks) load(wave, av, bv);
  for (int c = wave; c < chunks; c += WAVES) {
    const bool more = c + WAVES < chunks;
    if (more) load(c + WAVES, an, bn);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i][s], bv[j][s], acc[i][j], 0, 0, 0);
    if (more) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int i = 0; i < MI; ++i) av[i][s] = an[i][s];
#pragma unroll
        for (int i = 0; i < NI; ++i) bv[i][s] = bn[i][s];
      }
    }
  }
  // lane l holds rows (l / 16) * 4 + r of column l % 16
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[wave][16 * i + (lane >> 4) * 4 + r][16 * j + row] = acc[i][j][r];
  __syncthreads();
  for (int p = threadIdx.x; p < M * N; p += 64 * WAVES) {
    const int m = p / N, n = p % N;
    if (t0 + m >= tokens || e0 + n >= experts) continue;
    float s = part[0][m][n];
#pragma unroll
    for (int v = 1; v < WAVES; ++v) s += part[v][m][n];
    out[(t0 + m) * experts + e0 + n] = s;
  }
}

template <int MI, int NI, int WAVES>
void gate_launch(const bf16_t* x, int64_t tokens, int hidden, const bf16_t* w, int experts,
                 float* out, hipStream_t s) {
  launch("gate_kernel", gate_kernel<MI, NI, WAVES>,
         dim3((unsigned)ceil_div(tokens, 16 * MI), (unsigned)ceil_div(experts, 16 * NI)),
         dim3(64 * WAVES), 0, s, x, tokens, hidden, w, experts, out);
}

}  // namespace
}  // namespace ferry

using namespace ferry;

extern "C" int ferry_gate_logits(const void* x, int64_t tokens, int64_t hidden, const void* w,
                                 int64_t experts, float* out, void* stream) {
  clear_error();
  FERRY_CHECK_ARG(tokens >= 0 && experts >= 1 && experts <= 65536, "bad sizes");
  FERRY_CHECK_ARG(hidden >= 64 && hidden % 64 == 0 && hidden <= (1 << 24),
                  "hidden must be a multiple of 64 in [64, 2^24]");
  FERRY_CHECK_ARG(tokens < (int64_t)1 << 30, "too many tokens");   // 256 threads for each 64 of them
  if (tokens == 0) return 0;
  FERRY_CHECK_ARG(x && w && out, "null pointer argument");
  FERRY_CHECK_ARG(((uintptr_t)x | (uintptr_t)w) % 16 == 0, "x and w must be 16-byte aligned");
  const bf16_t* xb = (const bf16_t*)x;
  const bf16_t* wb = (const bf16_t*)w;
  const int h = (int)hidden, e = (int)experts;
  hipStream_t s = (hipStream_t)stream;
  // The smallest tile that gives each of the 256 CUs at most one workgroup: a workgroup's time is
  // the latency of its loads until the CUs are full (5.3, 7.2, 9.2, 13, 18 us for the five tiles at
  // hidden 2048), and from there on the tile's re-reads of x and w cost most.  us, by tile, with the
  // library product and its fp32 copies first; 64 experts: 256 rows 29.4: 5.4 7.1 9.0 13.1 17.8;
  // 2048 rows 29.4: 9.3 7.6 9.5 13.5 17.9; 4096 rows 32.6: 16.7 12.8 9.6 13.5 18.0; 8192 rows 41.9:
  // 31.7 23.7 17.3 14.3 18.1; 65,536 rows 290: 235 175 128 94 70 (3.8 TB/s of x).
  auto groups = [&](int mi, int ni) { return ceil_div(tokens, 16 * mi) * ceil_div(experts, 16 * ni); };
  if (groups(1, 1) <= 256)
    gate_launch<1, 1, 8>(xb, tokens, h, wb, e, out, s);
  else if (groups(1, 2) <= 256)
    gate_launch<1, 2, 8>(xb, tokens, h, wb, e, out, s);
  else if (groups(2, 2) <= 256)
    gate_launch<2, 2, 8>(xb, tokens, h, wb, e, out, s);
  else if (groups(2, 4) <= 256)
    gate_launch<2, 4, 4>(xb, tokens, h, wb, e, out, s);
  else
    gate_launch<4, 4, 4>(xb, tokens, h, wb, e, out, s);
  FERRY_LAUNCHED("gate_kernel");
  return 0;
}
