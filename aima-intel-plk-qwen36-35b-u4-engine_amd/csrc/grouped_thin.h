// Grouped GEMM of the prefill for thin tiles (at most 32 token rows of one
// expert), where the packed weights and their dequantization, not the matrix
// cores, set the time.
//
// The weights enter as the integers q - z, exact in f16: a code OR-ed into
// bits 0..3 of 0x6400 is 1024 + q, into bits 4..7 of 0x5400 64 + q, and one
// subtraction leaves q - z, nine VALU instructions for the eight nibbles of a
// word and no rounding (f16 (q - z) * s operands: 17 and one).  Each 128-wide
// quantization group is folded into the f32 result as
//   acc += s * sum((q - z) x)
// Error of a layer's output against 64 bits: 3.6e-4 (f16 operands: 4.9e-4; the
// rest is the f16 intermediates), with a few channels 2^4 .. 2^12 times the
// rest too (3.0e-4 and 4.6e-4 with f32 outputs).  An infinite x keeps its sign
// through q - z, as in the products with (q - z) * s.
// The z must be subtracted before the product: sum(q x) - z sum(x), with the
// codes alone as (subnormal) operands, takes two instructions less a word, but
// an infinite x makes it inf - inf, sum(x) takes MFMAs of its own, and its
// extra fold and registers cost more than they save: T = 777 (24 rows an
// expert) 167 us a call against 151 here, T = 96 109.5 against 107.4.
//
// A block of NW waves owns one tile and 32 NW weight rows (gate/up: 16 NW
// gate and the matching 16 NW up rows).  v_mfma_f32_16x16x32_f16: the tokens
// are the A operand, the weights B (lane l: weight row l % 16, the 32 k of
// quarter l / 16 of the group: one 16-byte load per row and group), so a
// lane's results all belong to its own weight row, whose scale and zero point
// it loads itself.  Each wave runs 2 x 16 weight rows against NB x 16 tokens.
// Tokens reach LDS through registers, 4 groups at a time in two buffers,
// already in the operands' order (low nibbles' k, then high nibbles' k of
// each 16), with 16-byte piece p of row r in slot p ^ (r & 15) of its 256
// bytes: no bank conflicts.  The next 4 groups of weights are in flight while
// the current ones are used.
//
// Bound: the weights' bytes.  T = 96 over 256 experts (hidden 2048, inter
// 512; about 245 experts active: 267 and 133 MB of weights): gate/up 59.9 us,
// down 35.7 (4.5 and 3.7 TB/s, in a kernel trace; a bare read in the same
// pattern reaches 6.1).  The call takes 108 us; with f16 (q - z) * s operands in
// 512-thread blocks and three schedule launches it took 160.
#ifndef AIMA_GROUPED_THIN_H_
#define AIMA_GROUPED_THIN_H_

#include "common.h"

namespace aima {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThinThreads = 256;
constexpr int kThinTurn = 4;  // groups per turn of the weight registers and token buffers

__host__ __device__ constexpr int thin_buf_bytes(int nb) { return nb * 16 * kThinTurn * 256; }
inline size_t thin_lds_bytes(int nb, int64_t GK) {
  return (size_t)(GK > kThinTurn ? 2 : 1) * thin_buf_bytes(nb);
}

struct ThinArgs {
  const uint16_t* src;        // token rows: x [T][H], or the SwiGLU rows [rows][I]
  const int32_t* tiles;       // [tile_count][4]: expert, first row, rows, 0
  const int32_t* tile_count;
  const int32_t* token_map;
  const float* row_weight;
  int64_t A;                  // routed rows (the shared expert's follow)
  int ntiles_n;               // blocks per tile
  uint16_t* act_out;
  uint16_t* contrib_out;
  float* act32;               // optional f32 copies (GemmCapture)
  float* contrib32;
};

// Tokens of one thread's 32-byte piece (x0 | x1: 16 consecutive k of a row)
// into the group buffer `row` (256 bytes of that row and group), in operand
// order.
__device__ __forceinline__ void thin_store_piece(const u32x4 x0, const u32x4 x1, uint8_t* row, int r,
                                                 int piece) {
  const uint32_t a0 = x0[0], a1 = x0[1], a2 = x0[2], a3 = x0[3];
  const uint32_t b0 = x1[0], b1 = x1[1], b2 = x1[2], b3 = x1[3];
  const u32x4 lo{__builtin_amdgcn_perm(a2, a0, 0x05040100u), __builtin_amdgcn_perm(a3, a1, 0x05040100u),
                 __builtin_amdgcn_perm(b2, b0, 0x05040100u), __builtin_amdgcn_perm(b3, b1, 0x05040100u)};
  const u32x4 hi{__builtin_amdgcn_perm(a2, a0, 0x07060302u), __builtin_amdgcn_perm(a3, a1, 0x07060302u),
                 __builtin_amdgcn_perm(b2, b0, 0x07060302u), __builtin_amdgcn_perm(b3, b1, 0x07060302u)};
  *reinterpret_cast<u32x4*>(row + ((piece ^ (r & 15)) * 16)) = lo;
  *reinterpret_cast<u32x4*>(row + (((piece + 1) ^ (r & 15)) * 16)) = hi;
}

// The halves 0x6400 and 0x5400 in VGPRs (as u4_magic): a code OR-ed into bits
// 0..3 or 4..7 of them is the f16 value 1024 + q or 64 + q.
struct ThinMagic {
  uint32_t lo, hi;
};
__device__ __forceinline__ ThinMagic thin_magic() {
  ThinMagic m{u4_magic(), 0x54005400u};
  asm volatile("" : "+v"(m.hi));
  return m;
}

// 1024 + z and 64 + z of one weight row and group, and the exact operands
// q - z of a word (k 0..7): `lo` holds k 0, 4, 2, 6 (bits 0..3 of each byte),
// `hi` k 1, 5, 3, 7.
struct ThinZero {
  f16x2 lo, hi;
};
__device__ __forceinline__ ThinZero thin_zero(uint32_t z, const ThinMagic& m) {
  const uint32_t zz = z * 0x00010001u;
  return ThinZero{as_h2(zz | m.lo), as_h2((zz << 4) | m.hi)};
}
__device__ __forceinline__ void thin_word(uint32_t v, const ThinZero& z, const ThinMagic& m,
                                          uint32_t (&lo)[2], uint32_t (&hi)[2]) {
  const uint32_t v8 = v >> 8;
  lo[0] = h2_bits(as_h2((v & 0x000F000Fu) | m.lo) - z.lo);
  hi[0] = h2_bits(as_h2((v & 0x00F000F0u) | m.hi) - z.hi);
  lo[1] = h2_bits(as_h2((v8 & 0x000F000Fu) | m.lo) - z.lo);
  hi[1] = h2_bits(as_h2((v8 & 0x00F000F0u) | m.hi) - z.hi);
}

// Scales and zero points of one weight row for a turn's 4 groups.  V4: one
// 8-byte and one 2-byte load (whole turns, aligned rows); else value by value.
template <bool V4>
struct ThinSz {
  u32x2 s;
  uint32_t z;
  __device__ __forceinline__ void load(const uint16_t* sc, const uint8_t* zp, int64_t at, int g,
                                       int GK) {
    const int gc = g < GK ? g : 0;  // past the last turn: any valid group
    s = *reinterpret_cast<const AIMA_GLOBAL u32x2*>((const AIMA_GLOBAL uint16_t*)sc + at + gc);
    z = *reinterpret_cast<const AIMA_GLOBAL uint16_t*>((const AIMA_GLOBAL uint8_t*)zp +
                                                       ((at + gc) >> 1));
  }
  __device__ __forceinline__ float scale(int i) const {
    const f16x2 v = as_h2(s[i >> 1]);
    return i & 1 ? (float)v.y : (float)v.x;
  }
  __device__ __forceinline__ uint32_t zero(int i) const { return (z >> (4 * i)) & 0xfu; }
};
template <>
struct ThinSz<false> {
  uint32_t s[4], z[4];
  __device__ __forceinline__ void load(const uint16_t* sc, const uint8_t* zp, int64_t at, int g,
                                       int GK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t j = at + (g + i < GK ? g + i : GK - 1);
      s[i] = ((const AIMA_GLOBAL uint16_t*)sc)[j];
      z[i] = (uint32_t)((const AIMA_GLOBAL uint8_t*)zp)[j >> 1] | ((uint32_t)(j & 1) << 16);
    }
  }
  __device__ __forceinline__ float scale(int i) const { return h2f((uint16_t)s[i]); }
  __device__ __forceinline__ uint32_t zero(int i) const {
    return (z[i] >> ((z[i] >> 16) * 4)) & 0xfu;
  }
};

// The value rounded to f32: the compiler would fold a product into the f16
// conversion behind it (one rounding), and the f16 rows would no longer be
// the f32 capture's values rounded.
__device__ __forceinline__ float as_f32_value(float v) {
  asm volatile("" : "+v"(v));
  return v;
}

template <bool GATEUP, int NB, bool V4, bool CAP, int TH>
__device__ __forceinline__ void thin_tile(const ThinArgs& a, const aima_moe_layer& L, uint8_t* smem,
                                          int e, int64_t row0, int rows, int ntile) {
  constexpr int WD = kThinTurn, NW = TH / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, q = lane >> 4;
  const int64_t H = L.hidden, I = L.inter;
  const int64_t K = GATEUP ? H : I;
  const int GK = (int)(K >> 7);
  const bool routed = e < L.experts;
  const int64_t eoff = routed ? e : 0;
  constexpr int kBuf = thin_buf_bytes(NB);

  // this lane's two weight rows: gate and up row of unit ntile * 64 +
  // wave * 16 + n, or output columns ntile * 128 + wave * 32 + n and + 16
  const uint8_t* wp[2];
  const uint16_t* sp[2];
  const uint8_t* zp[2];
  int64_t zat[2];
  if (GATEUP) {
    const GateUpView V = routed ? routed_gate_up(L) : shared_gate_up(L);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t row = V.row(eoff, h, (int64_t)ntile * (16 * NW) + wave * 16 + n);
      wp[h] = V.q[h] + row * (K / 2) + q * 16;
      sp[h] = V.s[h];
      zp[h] = V.z[h];
      zat[h] = row * GK;
    }
  } else {
    const aima_u4_tensor& W = routed ? L.down : L.shared_down;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t row = eoff * H + (int64_t)ntile * (32 * NW) + wave * 32 + 16 * h + n;
      wp[h] = W.qweight + row * (K / 2) + q * 16;
      sp[h] = W.scale;
      zp[h] = W.zp;
      zat[h] = row * GK;
    }
  }
  u32x4 w[WD][2];
  ThinSz<V4> sz[2], sn[2];
  auto load_w = [&](int g, u32x4 (&d)[2]) {
    const int gc = g < GK ? g : GK - 1;
    d[0] = gload16(wp[0] + gc * 64);
    d[1] = gload16(wp[1] + gc * 64);
  };

  // token rows staged by this thread: rows tid / (8 WD) + ..., 32 bytes each
  constexpr int kPairs = WD * 8;                 // 32-byte pieces of a row per turn
  constexpr int kPer = NB * 16 * kPairs / TH;
  constexpr int kRowStep = TH / kPairs;
  const int tp = tid % kPairs, trow = tid / kPairs;
  uint32_t soff[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int r = trow + i * kRowStep;
    const int64_t grow = row0 + (r < rows ? r : 0);  // rows past the tile: its first row
    const int64_t s = GATEUP ? (routed ? (int64_t)a.token_map[grow] : grow - a.A) : grow;
    soff[i] = (uint32_t)(s * K * 2);
  }
  const char* src = reinterpret_cast<const char*>(a.src);
  u32x4 tk[kPer][2];
  auto load_tokens = [&](int t) {
    // groups past K (a last, partial turn) reload the turn's first group
    const int g = t * WD + tp / 8;
    const uint32_t off = (uint32_t)(t * WD * 256 + (g < GK ? tp * 32 : (tp & 7) * 32));
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      tk[i][0] = *reinterpret_cast<const u32x4*>(src + soff[i] + off);
      tk[i][1] = *reinterpret_cast<const u32x4*>(src + soff[i] + off + 16);
    }
  };
  auto store_tokens = [&](uint8_t* buf) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int r = trow + i * kRowStep;
      thin_store_piece(tk[i][0], tk[i][1], buf + ((tp >> 3) * NB * 16 + r) * 256, r, (tp & 7) * 2);
    }
  };

  // first loads, nothing waited for in between but the token map
  sz[0].load(sp[0], zp[0], zat[0], 0, GK);
  sz[1].load(sp[1], zp[1], zat[1], 0, GK);
#pragma unroll
  for (int g = 0; g < WD; ++g) load_w(g, w[g]);
  load_tokens(0);
  store_tokens(smem);
  __syncthreads();

  f32x4 acc[2][NB];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[h][b] = f32x4{};
  const ThinMagic magic = thin_magic();

  // one group: its token rows at grp, this wave's weights wg, group i of the turn
  auto group = [&](const uint8_t* grp, const u32x4 (&wg)[2], int i) {
    f16x8 tf[NB][4];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int p = 0; p < 4; ++p)
        tf[b][p] = *reinterpret_cast<const f16x8*>(grp + (b * 16 + n) * 256 +
                                                   (((q * 4 + p) ^ n) * 16));
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const ThinZero z = thin_zero(sz[h].zero(i), magic);
      f16x8 lo[2], hi[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        uint32_t l0[2], l1[2], h0[2], h1[2];
        thin_word(wg[h][2 * m], z, magic, l0, h0);
        thin_word(wg[h][2 * m + 1], z, magic, l1, h1);
        lo[m] = __builtin_bit_cast(f16x8, (u32x4{l0[0], l0[1], l1[0], l1[1]}));
        hi[m] = __builtin_bit_cast(f16x8, (u32x4{h0[0], h0[1], h1[0], h1[1]}));
      }
      const float s = sz[h].scale(i);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        f32x4 al = f32x4{};
        al = __builtin_amdgcn_mfma_f32_16x16x32_f16(tf[b][0], lo[0], al, 0, 0, 0);
        al = __builtin_amdgcn_mfma_f32_16x16x32_f16(tf[b][1], hi[0], al, 0, 0, 0);
        al = __builtin_amdgcn_mfma_f32_16x16x32_f16(tf[b][2], lo[1], al, 0, 0, 0);
        al = __builtin_amdgcn_mfma_f32_16x16x32_f16(tf[b][3], hi[1], al, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[h][b][j] = fmaf(s, al[j], acc[h][b][j]);
      }
    }
  };

  // The tokens of the next turn are loaded while this one's are used and stored
  // behind them.  Every turn but the last is straight-line code: a branch
  // around a load would make the compiler wait for the loads before it.
  const int turns = (GK + WD - 1) / WD;
  int g0 = 0;
  for (int t = 0; t + 1 < turns; ++t, g0 += WD) {
    sn[0].load(sp[0], zp[0], zat[0], g0 + WD, GK);
    sn[1].load(sp[1], zp[1], zat[1], g0 + WD, GK);
    load_tokens(t + 1);
    const uint8_t* buf = smem + (t & 1) * kBuf;
#pragma unroll
    for (int gi = 0; gi < WD; gi += 2) {
      group(buf + gi * NB * 16 * 256, w[gi], gi);
      group(buf + (gi + 1) * NB * 16 * 256, w[gi + 1], gi + 1);
      // two groups are one 128-byte line of a row: asked for together
      load_w(g0 + gi + WD, w[gi]);
      load_w(g0 + gi + WD + 1, w[gi + 1]);
    }
    store_tokens(smem + ((t + 1) & 1) * kBuf);
    __syncthreads();
    sz[0] = sn[0];
    sz[1] = sn[1];
  }
  const uint8_t* last = smem + ((turns - 1) & 1) * kBuf;
#pragma unroll
  for (int gi = 0; gi < WD; ++gi) {
    if (g0 + gi < GK) group(last + gi * NB * 16 * 256, w[gi], gi);
  }

  // lane (n, q): weight rows n (of each 16) and token rows 16 b + 4 q + j.
  // The wave's outputs pass through LDS, [token row][32 or 16 columns], so
  // that a lane writes 16 bytes of a row.
  constexpr int kCols = GATEUP ? 16 : 32;
  __syncthreads();  // every wave is done with the token buffers
  uint16_t* stage = reinterpret_cast<uint16_t*>(smem) + wave * (NB * 16 * (kCols + 8));
  const int64_t ld = GATEUP ? I : H;
  const int64_t col0 = (int64_t)ntile * (NW * kCols) + wave * kCols;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = b * 16 + 4 * q + j;
      if (GATEUP) {
        const float g = acc[0][b][j], u = acc[1][b][j];
        const float o = as_f32_value(g * u * __builtin_amdgcn_rcpf(1.0f + __expf(-g)));
        stage[m * (kCols + 8) + n] = f2h(o);
        if (CAP && a.act32 && m < rows) a.act32[(row0 + m) * ld + col0 + n] = o;
      } else {
        const float wt = routed && m < rows ? a.row_weight[row0 + m] : 1.0f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float o = as_f32_value(wt * acc[h][b][j]);
          stage[m * (kCols + 8) + 16 * h + n] = f2h(o);
          if (CAP && a.contrib32 && m < rows) a.contrib32[(row0 + m) * ld + col0 + 16 * h + n] = o;
        }
      }
    }
  }
  wave_lds_sync();
  uint16_t* out = GATEUP ? a.act_out : a.contrib_out;
  constexpr int kLanes = kCols / 8;  // lanes of 16 bytes per row
#pragma unroll
  for (int r0 = 0; r0 < NB * 16; r0 += 64 / kLanes) {
    const int m = r0 + lane / kLanes, c = lane % kLanes;
    if (m < NB * 16 && m < rows) {
      *reinterpret_cast<u32x4*>(out + (row0 + m) * ld + col0 + c * 8) =
          *reinterpret_cast<const u32x4*>(stage + m * (kCols + 8) + c * 8);
    }
  }
}

// Tiles of at most 16 rows, several small blocks per CU: one block's first
// loads and epilogue pass under another's stream (blocks of 512 threads:
// T = 96 119 against 108 us per call).  Blocks are mapped XCD-aware, as in
// grouped_gemm_kernel: tile i on XCD i % 8, its blocks consecutive there.
template <bool GATEUP, bool V4, bool CAP>
__global__ __launch_bounds__(kThinThreads, V4 ? 3 : 2) void grouped_thin_kernel(aima_moe_layer L,
                                                                                ThinArgs a) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t thin_smem[];
  const int p = blockIdx.x;
  const int slot = p >> 3;
  const int mt = (slot / a.ntiles_n) * 8 + (p & 7);
  if (mt >= *a.tile_count) return;
  thin_tile<GATEUP, 1, V4, CAP, kThinThreads>(a, L, thin_smem, a.tiles[4 * mt + 0],
                                              a.tiles[4 * mt + 1], a.tiles[4 * mt + 2],
                                              slot % a.ntiles_n);
}

}  // namespace aima

#endif  // AIMA_GROUPED_THIN_H_
