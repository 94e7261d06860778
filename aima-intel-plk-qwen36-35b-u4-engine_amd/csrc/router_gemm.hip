// Batched router for the grouped prefill (the reference runtime's
// native_router, grouped_s8_u4_prefill_runtime.cpp:1085-1101): router logits
// for every token with one f32 GEMM, then the per-token top-k selection of
// aima_router_topk.
//
// logits[T][E] = X[T][H] . W[E][H]^T in f32 (2 T E H flops: 2.1 GFLOP at
// T = 2048, E = 256, H = 2048) on the f32 matrix cores
// (v_mfma_f32_32x32x2_f32: f32 operands, f32 accumulation).  An f16 input is
// widened in registers.
#include "common.h"

namespace aima {

int router_topk_launch(const float* logits, int64_t tokens, int experts, int k,
                       float min_weight_sum, int32_t* ids, float* weights, hipStream_t st,
                       float* probs);

namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kRgWaves = 8;
constexpr int kRgThreads = 64 * kRgWaves;
constexpr int kRgChunk = 128;  // k per step

// 8 consecutive values of a row in LDS as f32 (row: its chunk, 16-byte piece
// p at slot p ^ (row index % pieces); k0: first value)
__device__ __forceinline__ void rg_read(const float* row, int swz, int k0, float (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const u32x4 d = *reinterpret_cast<const u32x4*>(row + (((k0 / 4 + i) ^ swz) * 4));
#pragma unroll
    for (int j = 0; j < 4; ++j) v[4 * i + j] = as_f32(d[j]);
  }
}
__device__ __forceinline__ void rg_read(const uint16_t* row, int swz, int k0, float (&v)[8]) {
  const u32x4 d = *reinterpret_cast<const u32x4*>(row + (((k0 / 8) ^ (swz & 15)) * 8));
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t w = d[j];
    v[2 * j] = h2f((uint16_t)(w & 0xffffu));
    v[2 * j + 1] = h2f((uint16_t)(w >> 16));
  }
}

// A block of 8 waves owns 32 NA tokens x 32 experts.  K runs in steps of 128
// through two LDS buffers (the next step's rows are loaded into registers
// while this one is multiplied); wave w multiplies k 16 w .. 16 w + 15 of
// every step, lane half h the 8 from 8 h (MFMA j sees k0 + 8 h + j in both
// operands), and the eight partial tiles are added through LDS in wave order,
// the same every call.
//
// Bound: the f32 MFMAs (13 us at the 163 TFLOP/s peak for T = 2048, E = 256,
// H = 2048).  The output has only 512 32 x 32 tiles there, two per CU: K split
// over the waves of a block fills the chip.  Rows read straight into the
// operands' lanes (32 rows per load) made T = 4096 f32 88 us a call with its
// selection, against 55 here; 64 x 64 tiles with two K halves, read the
// same way, took 68 us at T = 2048 where this takes 28 (f16 input).
// Blocks are mapped XCD-aware: a token tile's expert blocks run on one XCD.
// The grid is 8 token tiles x the expert tiles, by the rest of the token tiles:
// in one dimension 2^24 tokens of 1024 experts would pass 2^32 threads.
//
// Rows past T (tokens) or E (experts) load the last row (valid memory) and
// are never stored; k past H load as zeros.  H % 16 == 0 and both matrices
// 16-byte aligned (checked on the host).
template <typename X, int NA>
__global__ __launch_bounds__(kRgThreads, 2) void router_gemm_kernel(
    const X* __restrict__ x, const float* __restrict__ w, int64_t T, int E, int H,
    float* __restrict__ logits) {
  constexpr int kXVals = 16 / sizeof(X);         // values of a 16-byte piece
  constexpr int kXPieces = kRgChunk / kXVals;    // pieces of a token row's step
  constexpr int kWPieces = kRgChunk / 4;
  constexpr int kXPer = NA * 32 * kXPieces / kRgThreads, kWPer = 32 * kWPieces / kRgThreads;
  constexpr int kXBytes = NA * 32 * kRgChunk * sizeof(X), kWBytes = 32 * kRgChunk * 4;
  constexpr int kPartBytes = kRgWaves * NA * 16 * 64 * 4;
  constexpr int kSmem = 2 * (kXBytes + kWBytes) > kPartBytes ? 2 * (kXBytes + kWBytes) : kPartBytes;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kSmem];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int p = blockIdx.x;
  const int64_t t0 = ((int64_t)blockIdx.y * 8 + (p & 7)) * (32 * NA);
  const int e0 = (p >> 3) * 32;
  if (t0 >= T) return;

  const X* xp[kXPer];
  const float* wp[kWPer];
  const int xk = (tid % kXPieces) * kXVals, wk = (tid % kWPieces) * 4;
  const int xr = tid / kXPieces, wr = tid / kWPieces;
#pragma unroll
  for (int i = 0; i < kXPer; ++i) {
    const int64_t t = t0 + xr + i * (kRgThreads / kXPieces);
    xp[i] = x + (t < T ? t : T - 1) * H + xk;
  }
#pragma unroll
  for (int i = 0; i < kWPer; ++i) {
    const int e = e0 + wr + i * (kRgThreads / kWPieces);
    wp[i] = w + (int64_t)(e < E ? e : E - 1) * H + wk;
  }
  struct Regs {
    u32x4 x[kXPer], w[kWPer];
  };
  auto load = [&](int k, Regs& d) {
    const bool xin = k + xk < H, win = k + wk < H;  // whole pieces: H % 16 == 0
    const int xo = xin ? k : -xk, wo = win ? k : -wk;
#pragma unroll
    for (int i = 0; i < kXPer; ++i) {
      d.x[i] = *reinterpret_cast<const u32x4*>(xp[i] + xo);
      d.x[i] = xin ? d.x[i] : u32x4{};
    }
#pragma unroll
    for (int i = 0; i < kWPer; ++i) {
      d.w[i] = *reinterpret_cast<const u32x4*>(wp[i] + wo);
      d.w[i] = win ? d.w[i] : u32x4{};
    }
  };
  auto store = [&](const Regs& d, uint8_t* buf) {
#pragma unroll
    for (int i = 0; i < kXPer; ++i) {
      const int r = xr + i * (kRgThreads / kXPieces);
      *reinterpret_cast<u32x4*>(buf + (r * kXPieces + ((tid % kXPieces) ^ (r & (kXPieces - 1)))) * 16) =
          d.x[i];
    }
#pragma unroll
    for (int i = 0; i < kWPer; ++i) {
      const int r = wr + i * (kRgThreads / kWPieces);
      *reinterpret_cast<u32x4*>(buf + kXBytes +
                                (r * kWPieces + ((tid % kWPieces) ^ (r & (kWPieces - 1)))) * 16) = d.w[i];
    }
  };

  f32x16_t acc[NA];
#pragma unroll
  for (int a = 0; a < NA; ++a) acc[a] = f32x16_t{};
  const int row = lane & 31, k0 = 16 * wave + 8 * (lane >> 5);
  auto multiply = [&](const uint8_t* buf) {
    float b[8], av[NA][8];
    rg_read(reinterpret_cast<const float*>(buf + kXBytes) + row * kRgChunk, row, k0, b);
#pragma unroll
    for (int a = 0; a < NA; ++a)
      rg_read(reinterpret_cast<const X*>(buf) + (32 * a + row) * kRgChunk, row, k0, av[a]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
      for (int a = 0; a < NA; ++a)
        acc[a] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[a][j], b[j], acc[a], 0, 0, 0);
    }
  };
  // two steps of rows in flight: a step's loads have the next two
  // multiplications to land
  uint8_t* const buf0 = smem;
  uint8_t* const buf1 = smem + kXBytes + kWBytes;
  Regs r0, r1;
  load(0, r0);
  load(kRgChunk, r1);
  store(r0, buf0);
  __syncthreads();
  for (int k = 0; k < H; k += 2 * kRgChunk) {
    load(k + 2 * kRgChunk, r0);
    multiply(buf0);
    store(r1, buf1);  // zeros past K
    __syncthreads();
    load(k + 3 * kRgChunk, r1);
    multiply(buf1);
    store(r0, buf0);
    __syncthreads();
  }

  // partial tiles [wave][frag][acc][lane]; every wave adds its share of them
  float* part = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int i = 0; i < 16; ++i) part[((wave * NA + a) * 16 + i) * 64 + lane] = acc[a][i];
  __syncthreads();
#pragma unroll
  for (int f = 0; f < 2 * NA; ++f) {
    const int c = wave * 2 * NA + f, a = c >> 4, i = c & 15;
    float v = part[c * 64 + lane];
#pragma unroll
    for (int q = 1; q < kRgWaves; ++q) v += part[(q * NA * 16 + c) * 64 + lane];
    // lane l holds expert e0 + l % 32 of token rows 8 (i / 4) + 4 (l / 32) + i % 4
    const int64_t t = t0 + 32 * a + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
    const int e = e0 + (lane & 31);
    if (t < T && e < E) logits[t * E + e] = v;
  }
}

// Short rows (rows_short): a block of 8 waves owns 64 tokens x 64 experts; wave
// w computes the 32 x 32 quarter w % 4 over the K half w / 4, and the two halves
// are added through LDS (half 0 + half 1, the same order every call).  Each lane
// loads 4 consecutive k of its token row and of its expert row per 8 k straight
// into the operands.
//
// Bound: the logits' bytes.  There are too few k to split over eight waves, and
// a block of the kernel above holds 64 KB or more of LDS whatever they are, so
// that one or two per CU wait for their few loads.
constexpr int kRgShortTile = 64;

__device__ __forceinline__ float4 rg_load4(const float* p) {
  return *reinterpret_cast<const float4*>(p);
}
__device__ __forceinline__ float4 rg_load4(const uint16_t* p) {
  const u32x2 d = *reinterpret_cast<const u32x2*>(p);
  const uint32_t a = d[0], b = d[1];
  return make_float4(h2f((uint16_t)(a & 0xffffu)), h2f((uint16_t)(a >> 16)),
                     h2f((uint16_t)(b & 0xffffu)), h2f((uint16_t)(b >> 16)));
}

template <typename X>
__global__ __launch_bounds__(kRgThreads) void router_gemm_short_kernel(
    const X* __restrict__ x, const float* __restrict__ w, int64_t T, int E, int H,
    float* __restrict__ logits) {
  __shared__ float part[4][16][64];  // K-half 1 partial sums, [quarter][acc][lane]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = wave & 3, kh = wave >> 2;
  const int64_t t0 = (int64_t)blockIdx.x * kRgShortTile + 32 * (q >> 1);
  const int e0 = (int)blockIdx.y * kRgShortTile + 32 * (q & 1);
  const int64_t tr = t0 + (lane & 31) < T ? t0 + (lane & 31) : T - 1;
  const int er = e0 + (lane & 31) < E ? e0 + (lane & 31) : E - 1;
  const int half = H / 2;
  const X* xp = x + tr * H + kh * half + 4 * (lane >> 5);
  const float* wp = w + (int64_t)er * H + kh * half + 4 * (lane >> 5);
  f32x16_t acc = f32x16_t{};
  for (int k = 0; k < half; k += 8) {
    const float4 a = rg_load4(xp + k), b = rg_load4(wp + k);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, acc, 0, 0, 0);
  }
  if (kh == 1) {
#pragma unroll
    for (int i = 0; i < 16; ++i) part[q][i][lane] = acc[i];
  }
  __syncthreads();
  if (kh == 1) return;
  const int e = e0 + (lane & 31);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int64_t t = t0 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
    const float v = acc[i] + part[q][i][lane];
    if (t < T && e < E) logits[t * E + e] = v;
  }
}

// Where short rows pay, direct against through LDS, us a call with its
// selection: hidden 128, f16, E = 512, T = 16384 73 against 97, f32 73 against
// 107; hidden 192 85 against 97, f32 85 against 107; hidden 256, f16 97 against
// 97, E = 64, T = 8192 19 against 16, f32 100 against 105 and 20 against 19.
// In the largest calls that goes on to hidden 384 for f32 rows, which take more
// LDS: E = 1024, T = 16384 248 against 272 (f16 236 against 237), T = 65536 1012
// against 1085 (f16 945 against 925); hidden 512, E = 512 84 against 77.  One
// rule for both types: an f16 input has the bits of its f32 copy.
bool rows_short(int64_t tokens, int experts, int64_t hidden) {
  return hidden <= (tokens * experts >= (1 << 23) ? 384 : 192);
}

// 64 tokens per block (fewer reads of the router's rows) for f16 tokens, once
// that leaves more than one block per CU: T = 2048, E = 256 (256 such blocks)
// 35.3 us a call against 33.3 in 512 blocks of 32 tokens; T = 4096 52.6 against
// 55.5.  With f32 tokens such a block takes 96 KB of LDS, one per CU instead of
// two: T = 2500, E = 256 58.0 against 43.2, T = 4096 59.8 against 54.9, T =
// 16384 222 against 197.
template <typename X>
int router_gemm_launch(const X* x, int64_t tokens, int experts, int64_t hidden, const float* w,
                       float* logits, hipStream_t st) {
  constexpr bool kWide = sizeof(X) == 2;
  const int ey = (experts + 31) / 32;
  const int64_t wide = (tokens + 63) / 64, narrow = (tokens + 31) / 32;
  if (rows_short(tokens, experts, hidden)) {
    const dim3 grid((unsigned)((tokens + kRgShortTile - 1) / kRgShortTile),
                    (unsigned)((experts + kRgShortTile - 1) / kRgShortTile));
    hipLaunchKernelGGL(router_gemm_short_kernel<X>, grid, dim3(kRgThreads), 0, st, x, w, tokens,
                       experts, (int)hidden, logits);
  } else if (kWide && wide * ey > 256) {
    hipLaunchKernelGGL((router_gemm_kernel<X, kWide ? 2 : 1>),
                       dim3((unsigned)(8 * ey), (unsigned)(round_up(wide, 8) / 8)),
                       dim3(kRgThreads), 0, st, x, w, tokens, experts, (int)hidden, logits);
  } else {
    hipLaunchKernelGGL((router_gemm_kernel<X, 1>),
                       dim3((unsigned)(8 * ey), (unsigned)(round_up(narrow, 8) / 8)),
                       dim3(kRgThreads), 0, st, x, w, tokens, experts, (int)hidden, logits);
  }
  return launch_check("router_gemm");
}

}  // namespace
}  // namespace aima

using namespace aima;

extern "C" int aima_router_gemm_workspace_size(int64_t tokens, int64_t hidden,
                                               int32_t /*input_f32*/, size_t* bytes) {
  AIMA_REQUIRE(bytes, "router_gemm_workspace_size: null pointer");
  AIMA_REQUIRE(tokens > 0 && hidden > 0, "router_gemm_workspace_size: sizes must be positive");
  *bytes = 0;  // an f16 input is widened in registers
  return AIMA_OK;
}

extern "C" int aima_router_gemm_topk(const void* hidden_states, int32_t input_f32, int64_t tokens,
                                     int64_t hidden, const float* router_weight, int32_t experts,
                                     int32_t k, float min_weight_sum, float* logits, int32_t* ids,
                                     float* weights, void* /*workspace*/,
                                     size_t /*workspace_bytes*/, void* stream) {
  AIMA_REQUIRE(hidden_states && router_weight && logits && ids && weights,
               "router_gemm_topk: null pointer");
  AIMA_REQUIRE(tokens > 0 && hidden > 0 && tokens <= (1 << 24) && hidden <= (1 << 20),
               "router_gemm_topk: tokens must be in [1, 2^24] and hidden in [1, 2^20]");
  AIMA_REQUIRE(hidden % 16 == 0, "router_gemm_topk: hidden must be a multiple of 16");
  AIMA_REQUIRE(aligned(hidden_states, 16) && aligned(router_weight, 16),
               "router_gemm_topk: hidden_states and router_weight must be 16-byte aligned");
  AIMA_REQUIRE(experts > 0 && experts <= 1024, "router_gemm_topk: experts must be in [1, 1024]");
  AIMA_REQUIRE(k > 0 && k <= 16 && k <= experts,
               "router_gemm_topk: k must be in [1, min(16, experts)]");
  AIMA_REQUIRE(min_weight_sum > 0.f, "router_gemm_topk: minimum weight sum must be positive");
  const hipStream_t st = (hipStream_t)stream;
  const int rc = input_f32 ? router_gemm_launch(static_cast<const float*>(hidden_states), tokens,
                                                experts, hidden, router_weight, logits, st)
                           : router_gemm_launch(static_cast<const uint16_t*>(hidden_states), tokens,
                                                experts, hidden, router_weight, logits, st);
  if (rc != AIMA_OK) return rc;
  return router_topk_launch(logits, tokens, experts, k, min_weight_sum, ids, weights, st,
                            nullptr);
}
