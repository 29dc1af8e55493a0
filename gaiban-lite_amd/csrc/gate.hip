// Router logits = x . Wg^T on bf16 MFMA with fp32 accumulation.
// Restates F.linear(x.float(), weight.float()) of the learned gate
// (runtime/dsv4_direct/moe_forward.py:80, reference/inference/model.py:565):
// bf16 x bf16 products are exact in fp32, so only the summation order differs.
// Every summation order here is fixed, so the logits of a token do not depend
// on the other tokens of the batch or on the run; they can differ in the last
// bits between batch sizes that run different kernels (as a vendor GEMM changes
// its algorithm by M).
//
// Three kernels by batch size and shape (Wg is [experts, hidden], experts = 256 at
// the Flash shape: 2 MiB of bf16):
//  * gate_logits_gemv_kernel (gate_gemv, up to 16 tokens): one expert per workgroup,
//    the tokens' dot products on the VALU (exact bf16 products, fp32 FMAs), so the
//    weights come through 256 CUs instead of the 16 that 16-expert MFMA tiles
//    occupy: T=1 6.2 -> 2.3 us, T=8 7.5 -> 4.5, T=16 8.8 -> 7.0;
//  * gate_logits_split_kernel (up to 512 tokens, and any shape the others do not
//    take): one workgroup of 8 wavefronts per 16-expert x 16-token output tile;
//    wavefront w sums K range w of 8 (8 loads of each operand in flight), and the
//    8 partial tiles are added through LDS in wavefront order: bound by the latency
//    of those loads (T=64 8.8 us, T=240 9.7 against 10.1 with the tiles below);
//  * gate_logits_tile_kernel (gate_tiles, prefill): 64 x 64 or 32 x 32 tokens x
//    experts per workgroup, K in chunks of 128 copied into LDS by buffer_load ... lds
//    (XOR-swizzled rows for conflict-free ds_read_b128) in a ring that holds 128
//    KiB: with two buffers every chunk waits for a whole read latency (22 us for
//    any batch up to ~2000).  32 x 32 tiles while one round of 256 workgroups holds
//    them (T=400 16.9 -> 10.8 us, T=1000 22.2 -> 10.7; two rounds at T=2000 29.3),
//    then 64 x 64 (T=3000 25.4 -> 22.1), with two buffers and two workgroups per CU
//    once one round does not hold those (T=8192 36 us, 41 with four buffers) or
//    where hidden is too short to fill four (H=1024, T=2048 8.3 us, 9.0 with four).
#include <type_traits>

#include "common.h"
#include "experts_common.h"
#include "../../include/dsv4moe.h"

namespace dsv4 {

constexpr int kGateSplitWaves = 8;
constexpr int kGateSplitBatch = 8;          // K steps (32 K each) loaded ahead per batch

__global__ __launch_bounds__(64 * kGateSplitWaves) void gate_logits_split_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ wg, int64_t tokens, int hidden, int experts,
    float* __restrict__ logits) {
  __shared__ f32x4 part[kGateSplitWaves][64];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t t0 = (int64_t)blockIdx.x * 16;
  const int e0 = blockIdx.y * 16;
  const int e = e0 + (lane & 15);
  const int64_t t = t0 + (lane & 15);
  const bool e_ok = e < experts;
  const bool t_ok = t < tokens;
  // K steps of 32 (hidden % 32 == 0): wavefront w takes steps [w*per, min(steps, (w+1)*per))
  const int steps = hidden / 32;
  const int per = (steps + kGateSplitWaves - 1) / kGateSplitWaves;
  const int s_begin = wave * per;
  const int s_end = min(steps, s_begin + per);
  const int koff = 8 * (lane >> 4);
  const uint16_t* arow = wg + (int64_t)(e_ok ? e : 0) * hidden + koff;
  const uint16_t* brow = x + (t_ok ? t : 0) * hidden + koff;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = s_begin; s0 < s_end; s0 += kGateSplitBatch) {
    u32x4 a[kGateSplitBatch], b[kGateSplitBatch];
#pragma unroll
    for (int j = 0; j < kGateSplitBatch; ++j) {
      const bool in = s0 + j < s_end;
      a[j] = e_ok && in ? load16(arow + (s0 + j) * 32) : u32x4{0u, 0u, 0u, 0u};
      b[j] = t_ok && in ? load16(brow + (s0 + j) * 32) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int j = 0; j < kGateSplitBatch; ++j)
      acc = mfma_bf16(__builtin_bit_cast(bf16x8, a[j]), __builtin_bit_cast(bf16x8, b[j]), acc);
  }
  part[wave][lane] = acc;
  __syncthreads();
  if (wave == 0) {
    f32x4 s = part[0][lane];
#pragma unroll
    for (int w = 1; w < kGateSplitWaves; ++w) {
      const f32x4 v = part[w][lane];
      s[0] += v[0]; s[1] += v[1]; s[2] += v[2]; s[3] += v[3];
    }
    if (t_ok) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int er = e0 + 4 * (lane >> 4) + i;
        if (er < experts) logits[t * experts + er] = s[i];
      }
    }
  }
}

constexpr int64_t kGateGemvMaxTokens = 16;

// logits[t][e] for expert e = blockIdx.x and NT >= tokens tokens: thread i sums K
// 8i .. 8i+7 of every 2048 columns, then a fixed tree over the wavefront and the
// four wavefronts.
template <int NT>
__global__ __launch_bounds__(256) void gate_logits_gemv_kernel(const uint16_t* __restrict__ x,
                                                               const uint16_t* __restrict__ wg, int tokens, int hidden,
                                                               int experts, float* __restrict__ logits) {
  __shared__ float part[4][NT];
  const int e = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  float acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = 0.0f;
#pragma unroll 2
  for (int k = threadIdx.x * 8; k < hidden; k += 2048) {
    const u32x4 w = load16(wg + (int64_t)e * hidden + k);
    u32x4 v[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) v[t] = load16(x + (int64_t)min(t, tokens - 1) * hidden + k);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        acc[t] = __builtin_fmaf(__uint_as_float(w[q] << 16), __uint_as_float(v[t][q] << 16), acc[t]);
        acc[t] = __builtin_fmaf(__uint_as_float(w[q] & 0xFFFF0000u), __uint_as_float(v[t][q] & 0xFFFF0000u), acc[t]);
      }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc[t] += __shfl_xor(acc[t], off, 64);
    if (lane == 0) part[wave][t] = acc[t];
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < tokens && t < NT) logits[(int64_t)t * experts + e] = ((part[0][t] + part[1][t]) + part[2][t]) + part[3][t];
}

constexpr int kGateChunk = 128;  // K per LDS stage

// TILE tokens x TILE experts (64 or 32) per workgroup, RING chunks in LDS.
template <int TILE, int RING>
__global__ __launch_bounds__(256, 1) void gate_logits_tile_kernel(const uint16_t* __restrict__ x,
                                                                  const uint16_t* __restrict__ wg,
                                                                  int64_t tokens, int hidden, int experts,
                                                                  float* __restrict__ logits) {
  constexpr int kStrips = TILE / 16;                  // 16-expert strips, 16-token columns
  constexpr int kCols = kStrips * kStrips / 4;        // token columns per wavefront
  constexpr int kCopies = TILE / 16;                  // copies per wavefront and operand
  constexpr int kStage = TILE * 256;
  static_assert(kStrips == 4 || kStrips == 2, "64 or 32");
  // row r of a stage: 16 parts of 16 B (8 K each); part q stored at q ^ (r & 15)
  __shared__ __attribute__((aligned(16))) uint8_t xs[RING * kStage];
  __shared__ __attribute__((aligned(16))) uint8_t ws[RING * kStage];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t t0 = (int64_t)blockIdx.x * TILE;
  const int e0 = blockIdx.y * TILE;
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)x, (short)0, (int)(tokens * hidden * 2), kRsrcFlags);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)wg, (short)0, (int)((int64_t)experts * hidden * 2), kRsrcFlags);
  // copy q of wave w fills rows 4 (kCopies w + q) + lane/16 of both tiles
  uint32_t xoff[kCopies], woff[kCopies];
#pragma unroll
  for (int q = 0; q < kCopies; ++q) {
    const int row = 4 * (kCopies * wave + q) + (lane >> 4);
    const int part = (lane & 15) ^ (row & 15);
    const int64_t t = t0 + row;
    const int e = e0 + row;
    xoff[q] = t < tokens ? (uint32_t)(t * hidden * 2 + part * 16) : kOobOffset;
    woff[q] = e < experts ? (uint32_t)((int64_t)e * hidden * 2 + part * 16) : kOobOffset;
  }
  const uint32_t xs_lds = __builtin_amdgcn_readfirstlane(lds_addr(&xs[kCopies * wave * 1024]));
  const uint32_t ws_lds = __builtin_amdgcn_readfirstlane(lds_addr(&ws[kCopies * wave * 1024]));
  const int chunks = hidden / kGateChunk;
  // chunks past the end repeat the last one into a buffer that nothing reads
  // again (the copies in flight stay countable)
  auto issue = [&](int c, uint32_t buf) {
    const uint32_t k = (uint32_t)min(c, chunks - 1) * kGateChunk * 2;
#pragma unroll
    for (int q = 0; q < kCopies; ++q) {
      lds_copy16(x_rsrc, xs_lds + buf + q * 1024, xoff[q], k);
      lds_copy16(w_rsrc, ws_lds + buf + q * 1024, woff[q], k);
    }
  };
  const int sw = lane & 15;
  const int strip = wave % kStrips;
  const int col0 = wave / kStrips * kCols;
  // one accumulator per K step of a chunk or, in the deeper rings, of a pair of chunks:
  // shorter rounding chains, and no MFMA waits for the one before it
  constexpr int kAccs = RING > 2 ? 8 : 4;
  f32x4 acc[kCols][kAccs];
#pragma unroll
  for (int ct = 0; ct < kCols; ++ct)
#pragma unroll
    for (int d = 0; d < kAccs; ++d) acc[ct][d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < RING - 1; ++c) issue(c, c * kStage);
  uint32_t cur = 0, fill = (RING - 1) * kStage;
  auto step = [&](int c, auto u_c) {
    constexpr int u = decltype(u_c)::value;
    lds_dma_wait_keep<(RING - 2) * 2 * kCopies>();  // this wavefront's copies of chunk c have landed
    __syncthreads();  // ... and everyone's; every wavefront has read chunk c - 1
    if (RING > 2 || c + 1 < chunks) issue(c + RING - 1, fill);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int part = ((4 * d + (lane >> 4)) ^ sw) * 16;
      const bf16x8 a =
          __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&ws[cur + (16 * strip + sw) * 256 + part]));
#pragma unroll
      for (int ct = 0; ct < kCols; ++ct) {
        const bf16x8 b = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const u32x4*>(&xs[cur + (16 * (col0 + ct) + sw) * 256 + part]));
        constexpr int first = kAccs > 4 ? 4 * u : 0;
        acc[ct][first + d] = mfma_bf16(a, b, acc[ct][first + d]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    fill = cur;
    cur = cur + kStage < RING * kStage ? cur + kStage : 0;
  };
  for (int c = 0; c < chunks; c += 2) {
    step(c, std::integral_constant<int, 0>{});
    if (c + 1 < chunks) step(c + 1, std::integral_constant<int, 1>{});
  }
  lds_dma_wait_all();
  // acc[ct] lane l: expert e0 + 16 strip + 4(l/16) + i, token t0 + 16 (col0 + ct) + l%16
#pragma unroll
  for (int ct = 0; ct < kCols; ++ct) {
    const int64_t t = t0 + 16 * (col0 + ct) + sw;
    if (t >= tokens) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = e0 + 16 * strip + 4 * (lane >> 4) + i;
      float sum = (acc[ct][0][i] + acc[ct][1][i]) + (acc[ct][2][i] + acc[ct][3][i]);
      if constexpr (kAccs > 4) sum += (acc[ct][4][i] + acc[ct][5][i]) + (acc[ct][6][i] + acc[ct][7][i]);
      if (e < experts) logits[t * experts + e] = sum;
    }
  }
}

}  // namespace dsv4

using namespace dsv4;

// Per token a gemv workgroup does more work and reads all tokens again, so it needs
// a longer K the more tokens, and few experts: 256 experts, against the split kernel,
// T=4 H=512 2.5 -> 2.8 us, H=1024 3.1 -> 2.8; T=8 H=1024 3.3 -> 3.8, H=2048 4.8 ->
// 4.0; T=16 H=2048 5.3 -> 6.0, H=4096 8.8 -> 6.9; T=16 H=4096 1024 experts 9.4 ->
// 10.7.  Under 32 experts the split kernel reads as little (T=9 H=4096 8 experts 5.9
// -> 6.7).
static bool gate_gemv(int64_t tokens, int hidden, int experts) {
  if (tokens <= 2) return tokens == 1 || hidden >= 1024;
  if (tokens <= 4) return hidden >= (experts >= 32 ? 1024 : 2048);
  return tokens <= kGateGemvMaxTokens && experts >= 32 && experts <= 512 && hidden >= (tokens <= 8 ? 2048 : 4096);
}

// Up to 512 tokens the split kernel is the faster one while one round of 256 holds its
// workgroups (T=512 H=4096, 128 experts 9.5 us, tiles 10.4; 160 experts 16.4, tiles
// 10.4) and for short K (T=300 H=256 256 experts 2.9, tiles 3.3; H=1024 5.4, 4.7).
static bool gate_tiles(int64_t tokens, int hidden, int experts) {
  if (tokens > 512) return true;
  return tokens > 256 && hidden >= 1024 && ((tokens + 15) / 16) * ((experts + 15) / 16) > 256;
}

int dsv4_launch_gate_logits(const uint16_t* x, const uint16_t* wg, int64_t tokens, int hidden,
                            int experts, float* logits, hipStream_t stream) {
  if (tokens == 0) return DSV4MOE_OK;
  if (gate_gemv(tokens, hidden, experts)) {
    const dim3 grid((unsigned)experts);
#define DSV4_GATE_GEMV(NT)                                                                                          \
  hipLaunchKernelGGL(gate_logits_gemv_kernel<NT>, grid, dim3(256), 0, stream, x, wg, (int)tokens, hidden, experts, \
                     logits)
    if (tokens <= 1) DSV4_GATE_GEMV(1);
    else if (tokens <= 2) DSV4_GATE_GEMV(2);
    else if (tokens <= 4) DSV4_GATE_GEMV(4);
    else if (tokens <= 8) DSV4_GATE_GEMV(8);
    else DSV4_GATE_GEMV(16);
#undef DSV4_GATE_GEMV
    DSV4_CHECK_LAUNCH("gate_logits_gemv_kernel");
    return DSV4MOE_OK;
  }
  const bool tiled = gate_tiles(tokens, hidden, experts) && hidden % kGateChunk == 0 &&
                     tokens * hidden * 2 < 0x7FFFFFFFLL && (int64_t)experts * hidden * 2 < 0x7FFFFFFFLL;
  if (!tiled) {
    const dim3 grid((unsigned)((tokens + 15) / 16), (unsigned)((experts + 15) / 16));
    hipLaunchKernelGGL(gate_logits_split_kernel, grid, dim3(64 * kGateSplitWaves), 0, stream, x, wg, tokens, hidden,
                       experts, logits);
    DSV4_CHECK_LAUNCH("gate_logits_split_kernel");
    return DSV4MOE_OK;
  }
  const int64_t small = ((tokens + 31) / 32) * ((experts + 31) / 32);
  const int64_t large = ((tokens + 63) / 64) * ((experts + 63) / 64);
  const dim3 grid32((unsigned)((tokens + 31) / 32), (unsigned)((experts + 31) / 32));
  const dim3 grid64((unsigned)((tokens + 63) / 64), (unsigned)((experts + 63) / 64));
#define DSV4_GATE_TILE(TILE, RING)                                                                             \
  hipLaunchKernelGGL((gate_logits_tile_kernel<TILE, RING>), grid##TILE, dim3(256), 0, stream, x, wg, tokens, \
                     hidden, experts, logits)
  if (small <= 256) DSV4_GATE_TILE(32, 8);
  else if (large <= 256 && hidden >= 3072) DSV4_GATE_TILE(64, 4);
  else DSV4_GATE_TILE(64, 2);
#undef DSV4_GATE_TILE
  DSV4_CHECK_LAUNCH("gate_logits_tile_kernel");
  return DSV4MOE_OK;
}
