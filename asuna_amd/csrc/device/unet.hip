// Learned denoiser (include/asuna_denoise.h): a 5-level U-Net trained and
// run by hand-written gfx950 kernels.
//
// Every 3x3 convolution is an implicit GEMM on v_mfma_f32_16x16x32_bf16
// (BF16 operands, FP32 accumulation):
//   forward      Y[p][co]  = b[co] + sum_tap sum_ci X[p + d(tap)][ci] W[tap][co][ci]
//                GEMM rows = cout, cols = pixels, K = 9 x cin
//   backward-x   dX[p][ci] = sum_tap sum_co dY[p - d(tap)][co] W[tap][co][ci]
//                the same kernels on dY with the taps reversed and the roles
//                of cin and cout exchanged in the packed weights
//   backward-w   dW[tap][co][ci] = sum_p dY[p][co] X[p + d(tap)][ci]
//                GEMM rows = cout, cols = cin, K = pixels (split over blocks;
//                each split writes its partial sums, which a second kernel
//                adds in a fixed order, so gradients are reproducible)
// Activations are NHWC BF16 with the channel count padded to a multiple of
// 32 (padding channels hold zeros and their weights stay zero), so an
// operand row is one 16-byte load.  Decoder convolutions read their input
// as two sources -- the half-resolution tensor below, nearest-upsampled on
// the fly, then the skip tensor -- so neither the upsampled tensor nor the
// concatenation is materialised.  Gradients are summed in FP32 and rounded to
// BF16 once, where they are complete, as the operand of the next products;
// bias gradients and the weight gradients' partial sums are FP32.
//
// MFMA 16x16x32 operand layout (lane l of 64, q = l / 16):
//   A (16 x 32)  row l % 16, k = 8q .. 8q+7
//   B (32 x 16)  col l % 16, k = 8q .. 8q+7
//   D (16 x 16)  col l % 16, rows 4q .. 4q+3
// With weights as A and pixels as B a lane ends with 4 channels of one pixel
// per tile.  Row m of tile t (of a 32-channel group's two) is channel
// 8 (m / 4) + 4 t + m % 4, so the lane's 8 values are channels 8q .. 8q+7 of
// its pixel and a wave stores 16 pixels x 64 bytes without a transpose.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../../include/asuna_denoise.h"
#include "ctx_internal.h"
#include "log1p.h"

namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kLevels = 5;
constexpr uint32_t kWidths[kLevels] = {32, 48, 64, 96, 128};
constexpr uint32_t kInCh = 10, kOutCh = 3;
constexpr int kNumLayers = 2 * kLevels + 2 * (kLevels - 1) + 1;
constexpr uint32_t kMaxChunks = 7;  // 224 / 32: widest input in 32-channel chunks

__host__ __device__ inline uint32_t pad32(uint32_t c) { return (c + 31) & ~31u; }

struct Src {
  const bf16* a;  // activations (or a gradient) [N][h][w][C]
  uint32_t C;     // stored channels (multiple of 32)
  uint32_t up;    // 1: half-resolution tensor read nearest-upsampled
};

// What a convolution computes: a layer's activations, the last layer's
// prediction, or a backward-x product.
enum ConvMode { kModeAct, kModeLast, kModeGrad };

// Where a backward-x convolution's output goes, by the tensor its forward
// convolution read.
enum GradKind : uint32_t {
  kGradFinal,  // the tensor's only reader: ReLU mask, BF16
  kGradUp,     // read upsampled: sum of the 2 x 2 pixels, ReLU mask, BF16 at half resolution
  kGradPool,   // a pooled tensor: a quarter to each of the 4 pixels of the unpooled one, added to
               // its skip gradient, ReLU mask, BF16 at full resolution
  kGradSkip,   // a skip tensor, whose pooled branch follows: FP32
};
struct GradDst {
  uint32_t kind;
  uint32_t C;       // channels of the tensor
  bf16* g;          // its complete gradient, masked
  const bf16* act;  // its activations (the mask)
  float* skip;      // FP32 skip gradient (written by kGradSkip, read by kGradPool)
  float* bPart;     // bias-gradient partial sums of the layer that made it: [pixel tile][C]
};

struct ConvArgs {
  Src s0, s1;  // s1.C == 0: one source
  uint32_t N, H, W;
  uint32_t nCh, nCg;  // 32-channel input chunks and output groups
  const bf16* Wp;     // packed weights [group][chunk][tap][2 tiles][64 lanes][8]
  // forward
  const float* bias;  // [32 nCg]
  bf16* Y;            // BF16 output [N][H][W][32 nCg] after ReLU, or null: the last layer
  bf16* pool;         // 2 x 2 average of Y, or null
  float* Yf;          // last layer (training): FP32 prediction [pixel][4] (log space)
  float* rgb;         // last layer (inference): expm1 of it, [pixel][3], or
  float4* film;       // max(expm1, 0) as RGBA of the filmW x filmH part
  uint32_t filmW, filmH;
  // backward-x: groups [0, cg0) belong to d0, the rest to d1
  uint32_t cg0;
  GradDst d0, d1;
};

__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
  for (int i = 0; i < 8; ++i) z[i] = bf16(0.0f);
  return z;
}

// One 32-channel chunk of one image of a convolution's input (uniform over
// the block: sources hold whole chunks).
struct ChunkSrc {
  const bf16* p;
  uint32_t C, w, up;  // channels per pixel, pixels per row, coordinate shift
};
__device__ __forceinline__ ChunkSrc chunkSrc(const Src& s0, const Src& s1, uint32_t H, uint32_t W, uint32_t n, uint32_t ch) {
  const bool first = 32 * ch < s0.C;
  const Src& s = first ? s0 : s1;
  ChunkSrc k;
  k.C = s.C, k.up = s.up, k.w = W >> s.up;
  k.p = s.a + size_t(n) * (H >> s.up) * k.w * s.C + (32 * ch - (first ? 0u : s0.C));
  return k;
}
// 8 BF16 channels [c, c + 8) of the chunk at pixel (y, x); zeros outside the H x W image.
__device__ __forceinline__ u32x4 loadIn(const ChunkSrc& k, uint32_t H, uint32_t W, int y, int x, uint32_t c) {
  u32x4 v = {0, 0, 0, 0};
  if (uint32_t(y) < H && uint32_t(x) < W)
    v = *reinterpret_cast<const u32x4*>(k.p + (uint64_t((uint32_t(y) >> k.up) * k.w + (uint32_t(x) >> k.up)) * k.C + c));
  return v;
}

// The value of the lane whose index differs in bit 0 (the horizontally
// neighbouring pixel of a pair).
__device__ __forceinline__ float pairLane(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));
}

// Bias, activation, store and what follows a convolution, for ROWS pixels
// (n, y0 .. y0 + ROWS - 1, x) of the lane and the 8 channels 32 cg + 8q + j
// (y0 even, ROWS = 2, lane pairs hold even and odd x).  All lanes of the wave
// call it; pixels outside the image are dropped here.  b: the lane's biases
// (forward), read once per block; bs: its sums of the complete gradient
// (backward).
template <int ROWS, ConvMode MODE>
__device__ __forceinline__ void emit(const ConvArgs& a, uint32_t cg, uint32_t n, int y0, int x, uint32_t q,
                                     float (&v)[ROWS][8], const float (&b)[8], float (&bs)[8]) {
  const int H = int(a.H), W = int(a.W);
  if (MODE != kModeGrad) {
    const uint32_t C = 32 * a.nCg, c0 = 32 * cg + 8 * q;
    if (MODE == kModeLast) {  // channels 0..2, no ReLU
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        const int y = y0 + i;
        if (!q && !cg && y < H && x < W)
          *reinterpret_cast<float4*>(a.Yf + 4 * ((size_t(n) * a.H + y) * a.W + x)) =
              make_float4(v[i][0] + b[0], v[i][1] + b[1], v[i][2] + b[2], 0.f);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        o[j] = bf16(fmaxf(v[i][j] + b[j], 0.f));
        v[i][j] = float(o[j]);
      }
      const int y = y0 + i;
      if (y < H && x < W) *reinterpret_cast<bf16x8*>(a.Y + ((size_t(n) * a.H + y) * a.W + x) * C + c0) = o;
    }
    if (a.pool) {
#pragma unroll
      for (int i = 0; i < ROWS; i += 2) {
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float right0 = pairLane(v[i][j]), right1 = pairLane(v[i + 1][j]);
          o[j] = bf16(0.25f * (v[i][j] + right0 + v[i + 1][j] + right1));
        }
        const int y = y0 + i;
        if (!(x & 1) && y < H && x < W)
          *reinterpret_cast<bf16x8*>(a.pool + ((size_t(n) * (a.H / 2) + y / 2) * (a.W / 2) + x / 2) * C + c0) = o;
      }
    }
    return;
  }
  const GradDst& d = cg < a.cg0 ? a.d0 : a.d1;
  const uint32_t c0 = 32 * (cg < a.cg0 ? cg : cg - a.cg0) + 8 * q;
  auto put = [&](size_t e, const float (&g)[8]) {  // masked gradient of elements e .. e + 7
    const bf16x8 act = *reinterpret_cast<const bf16x8*>(d.act + e);
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float m = float(act[j]) > 0.f ? g[j] : 0.f;
      o[j] = bf16(m);
      bs[j] += m;
    }
    *reinterpret_cast<bf16x8*>(d.g + e) = o;
  };
  if (d.kind == kGradUp) {
#pragma unroll
    for (int i = 0; i < ROWS; i += 2) {
      float s[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] = v[i][j] + pairLane(v[i][j]) + v[i + 1][j] + pairLane(v[i + 1][j]);
      const int y = y0 + i;
      if (!(x & 1) && y < H && x < W) put(((size_t(n) * (a.H / 2) + y / 2) * (a.W / 2) + x / 2) * d.C + c0, s);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int y = y0 + i;
    if (y >= H || x >= W) continue;
    if (d.kind == kGradPool) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const size_t e = ((size_t(n) * (2 * a.H) + 2 * y + k / 2) * (2 * a.W) + 2 * x + k % 2) * d.C + c0;
        float s[8];
        *reinterpret_cast<float4*>(s) = *reinterpret_cast<const float4*>(d.skip + e);
        *reinterpret_cast<float4*>(s + 4) = *reinterpret_cast<const float4*>(d.skip + e + 4);
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] += 0.25f * v[i][j];
        put(e, s);
      }
    } else {
      const size_t e = ((size_t(n) * a.H + y) * a.W + x) * d.C + c0;
      if (d.kind == kGradFinal) {
        put(e, v[i]);
      } else {
        *reinterpret_cast<float4*>(d.skip + e) = make_float4(v[i][0], v[i][1], v[i][2], v[i][3]);
        *reinterpret_cast<float4*>(d.skip + e + 4) = make_float4(v[i][4], v[i][5], v[i][6], v[i][7]);
      }
    }
  }
}

// The lane's 8 biases of an output group (zeros in backward-x).
template <ConvMode MODE> __device__ __forceinline__ void laneBias(const float* bias, uint32_t cg, uint32_t q, float (&b)[8]) {
  if (MODE == kModeGrad) {
    for (int j = 0; j < 8; ++j) b[j] = 0.f;
    return;
  }
  *reinterpret_cast<float4*>(b) = *reinterpret_cast<const float4*>(bias + 32 * cg + 8 * q);
  *reinterpret_cast<float4*>(b + 4) = *reinterpret_cast<const float4*>(bias + 32 * cg + 8 * q + 4);
}

// Sums the lanes' bias-gradient parts over the wave's 16 pixel columns (a
// fixed tree) into row[8q + j].
__device__ __forceinline__ void waveBias(float (&bs)[8], uint32_t q, uint32_t r16, float* row) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float s = bs[j];
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    s += __shfl_xor(s, 4);
    s += __shfl_xor(s, 8);
    if (r16 == 0) row[8 * q + j] = s;
  }
}
// Writes a 32-channel group's bias-gradient sums of one pixel tile (thread c
// of 32; rows: the waves' sums, added in wave order).
__device__ __forceinline__ void tileBias(const ConvArgs& a, uint32_t cg, uint32_t tile, uint32_t c, const float* rows,
                                         uint32_t nRows) {
  const GradDst& d = cg < a.cg0 ? a.d0 : a.d1;
  if (d.kind == kGradSkip) return;
  float s = 0.f;
  for (uint32_t w = 0; w < nRows; ++w) s += rows[32 * w + c];
  d.bPart[size_t(tile) * d.C + 32 * (cg < a.cg0 ? cg : cg - a.cg0) + c] = s;
}

// Convolution from LDS, for levels with work for the whole chip: a block of
// 4 waves owns a tile of 2R rows x 32 columns (CW = 1: four pixel waves) or
// 2R x 16 columns (CW = 2: two pixel waves for each of two output groups)
// and walks the input in chunks of 32 channels.  Per chunk it holds in LDS
// the input tile with its halo (64 bytes per pixel) and the chunk's weights
// of its output groups, in fragment order (a fragment is 1 KB in lane order).
// Each wave computes R rows x 16 columns x 32 channels: an input fragment
// (one row, one column shift) is read once and feeds the three taps of its
// column shift, i.e. up to 6 MFMAs, so that per chunk a wave reads 3 (R + 2)
// input and 18 weight fragments for 18 R MFMAs and the LDS asks for less time
// than the matrix cores (R = 8: the block's four waves read 192 KB, 1536 cycles of
// the CU's 128 bytes per cycle, against 2304 cycles of 16 per MFMA on each SIMD).
// The loads of the next chunk (or the next tile's first) are in flight in registers during
// the MFMAs.  Blocks are persistent; with one chunk the weights stay in LDS.
//
// A pixel's four 16-byte slots are swizzled by its column (slot ^ column / 4),
// which spreads a fragment's 16 pixels over all banks and leaves the
// row's offset an immediate.
//
// The MFMAs of one staged chunk for a wave's R rows x 16 columns from (row0,
// col0) of a tile of `Pitch` staged pixels per row; wAt: the lane's place in the
// first weight fragment.
template <int R, int NT, uint32_t Pitch>
__device__ __forceinline__ void chunkMfma(const bf16* tile, uint32_t row0, uint32_t col0, uint32_t q, uint32_t r16,
                                          const bf16* wAt, f32x4 (&acc)[R][NT]) {
#pragma unroll 1  // unrolled, the reads of all three shifts are hoisted together and spill
  for (int dx = 0; dx < 3; ++dx) {
    const uint32_t col = col0 + r16 + dx;  // rows are immediate offsets from here
    const bf16* xAt = tile + ((row0 * Pitch + col) * 4 + (q ^ ((col >> 2) & 3))) * 8;
    bf16x8 wf[3][NT];
#pragma unroll
    for (int dy = 0; dy < 3; ++dy)
#pragma unroll
      for (int t = 0; t < NT; ++t) wf[dy][t] = *reinterpret_cast<const bf16x8*>(wAt + ((dy * 3 + dx) * 2 + t) * 512);
#pragma unroll
    for (int r = 0; r < R + 2; ++r) {
      const bf16x8 xf = *reinterpret_cast<const bf16x8*>(xAt + r * Pitch * 32);
#pragma unroll
      for (int dy = 0; dy < 3; ++dy) {
        const int o = r - dy;
        if (o < 0 || o >= R) continue;
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[o][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[dy][t], xf, acc[o][t], 0, 0, 0);
      }
    }
  }
}
template <int R, int CW> struct ConvTile {
  static constexpr uint32_t PW = 4 / CW;              // pixel waves
  static constexpr uint32_t TR = 2 * R, TC = CW == 1 ? 32 : 16;
  static constexpr uint32_t P = (TR + 2) * (TC + 2);  // staged pixels
  static constexpr uint32_t LX = (P * 4 + 255) / 256;           // 16-byte input loads per thread
  static constexpr uint32_t LW = (CW * 18 * 64 + 255) / 256;    // weight loads per thread
  static constexpr size_t lds = size_t(P) * 64 + size_t(CW) * 18 * 1024;
};
template <int R, int CW, int NT, ConvMode MODE>
__global__ __launch_bounds__(256, R == 8 ? 2 : 3) void kConvLds(ConvArgs a, uint32_t tilesX, uint32_t tilesY, uint32_t items) {
  using T = ConvTile<R, CW>;
  extern __shared__ __align__(16) bf16 lds[];
  __shared__ float sB[4 * 32];
  bf16* tile = lds;               // [T::P][4 slots][8]
  bf16* wts = lds + T::P * 32;    // [CW][9 taps][2][64][8]
  const uint32_t tid = threadIdx.x, lane = tid & 63, q = lane >> 4, r16 = lane & 15, wv = tid >> 6;
  const uint32_t cw = wv / T::PW, pw = wv % T::PW;
  const uint32_t row0 = CW == 1 ? (pw >> 1) * R : pw * R, col0 = CW == 1 ? (pw & 1) * 16 : 0;
  const uint32_t cgb = a.nCg / CW;  // gridDim.x is a multiple: a block keeps its output groups
  uint32_t item = blockIdx.x;
  const uint32_t cgBase = (item % cgb) * CW;
  u32x4 px[T::LX], pwt[T::LW];
  auto origin = [&](uint32_t it, uint32_t& n, int& ty, int& tx) {
    const uint32_t t = it / cgb;
    tx = int((t % tilesX) * T::TC);
    ty = int(((t / tilesX) % tilesY) * T::TR);
    n = t / (tilesX * tilesY);
  };
  // the thread index through an opaque copy: the staging coordinates are recomputed where they are used instead of
  // being held in registers through the loops (10 loads of 2 coordinates spilled 100 registers)
  auto fresh = [&]() {
    uint32_t t = tid;
    asm volatile("" : "+v"(t));
    return t;
  };
  auto fetch = [&](uint32_t it, uint32_t ch, bool weights) {
    const uint32_t tid = fresh();
    uint32_t n;
    int ty, tx;
    origin(it, n, ty, tx);
    const ChunkSrc src = chunkSrc(a.s0, a.s1, a.H, a.W, n, ch);
#pragma unroll
    for (uint32_t j = 0; j < T::LX; ++j) {
      const uint32_t k = tid + 256 * j, pix = k >> 2;
      if (k < T::P * 4) {
        const int y = ty - 1 + int(pix / (T::TC + 2)), x = tx - 1 + int(pix % (T::TC + 2));
        px[j] = loadIn(src, a.H, a.W, y, x, 8 * (k & 3));
      }
    }
    if (weights) {
#pragma unroll
      for (uint32_t j = 0; j < T::LW; ++j) {
        const uint32_t k = tid + 256 * j, g = k / (18 * 64), f = k % (18 * 64);
        if (k < CW * 18 * 64)
          pwt[j] = *reinterpret_cast<const u32x4*>(a.Wp + ((size_t(cgBase + g) * a.nCh + ch) * (18 * 64) + f) * 8);
      }
    }
  };
  auto put = [&](bool weights) {
    const uint32_t tid = fresh();
#pragma unroll
    for (uint32_t j = 0; j < T::LX; ++j) {
      const uint32_t k = tid + 256 * j, pix = k >> 2, col = pix % (T::TC + 2);
      if (k < T::P * 4) *reinterpret_cast<u32x4*>(tile + (pix * 4 + ((k & 3) ^ ((col >> 2) & 3))) * 8) = px[j];
    }
    if (weights) {
#pragma unroll
      for (uint32_t j = 0; j < T::LW; ++j) {
        const uint32_t k = tid + 256 * j;
        if (k < CW * 18 * 64) *reinterpret_cast<u32x4*>(wts + k * 8) = pwt[j];
      }
    }
  };
  const bf16* wAt = wts + (cw * 18 * 64 + lane) * 8;
  bool w = true;
  fetch(item, 0, true);
  for (;;) {
    f32x4 acc[R][NT];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (uint32_t ch = 0; ch < a.nCh; ++ch) {
      __syncthreads();  // the previous chunk's fragments are consumed
      put(w);
      __syncthreads();
      w = a.nCh > 1;
      if (ch + 1 < a.nCh) fetch(item, ch + 1, w);
      else if (item + gridDim.x < items) fetch(item + gridDim.x, 0, w);
      __builtin_amdgcn_sched_barrier(0);  // the loads are issued before the MFMAs
      chunkMfma<R, NT, T::TC + 2>(tile, row0, col0, q, r16, wAt, acc);
    }
    uint32_t n;
    int ty, tx;
    origin(item, n, ty, tx);
    float bs[8] = {};
#pragma unroll
    for (int i = 0; i < R; i += 2) {
      __builtin_amdgcn_sched_barrier(0);
      float v[2][8];
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int j = 0; j < 8; ++j) v[k][j] = j / 4 < NT ? acc[i + k][j / 4 < NT ? j / 4 : 0][j % 4] : 0.f;
      float bias[8];
      laneBias<MODE>(a.bias, cgBase + cw, q, bias);
      emit<2, MODE>(a, cgBase + cw, n, ty + int(row0) + i, tx + int(col0 + r16), q, v, bias, bs);
    }
    if (MODE == kModeGrad) {
      waveBias(bs, q, r16, sB + 32 * wv);
      __syncthreads();
      if (tid < 32 * CW) tileBias(a, cgBase + tid / 32, item / cgb, tid & 31, sB + 32 * T::PW * (tid / 32), T::PW);
    }
    item += gridDim.x;
    if (item >= items) break;
  }
}

// Two 32-channel convolutions of the finest level in one pass, for inference:
// the first two layers (from the film's planes or packed features; the second
// one's output and its pooled copy are written), or the last two (the prediction
// is written).  At 1920 x 1088 a 32-channel tensor is 134 MB and the layers
// alone are bound by moving it; here the tensor between the two stays in LDS.  A
// block stages 18 x 34 input pixels, computes 16 x 32 of the first layer (four
// waves of 8 rows x 16 columns), puts them in the input's place (zeros outside
// the image) and computes the 14 x 30 pixels of the second whose neighbours it
// holds: 1.22 times the MFMAs for one read and one write less.  Both layers'
// weights stay in LDS.  1080p film: features and the two layers 60 + 80 + 85 us
// before, the last two 88 + 68; 133 and 112 us in one.
struct FilmSrc {
  const float4 *rad, *alb, *nrm, *dep;  // planes of W x H pixels; all but rad may be null
  uint32_t W, H;
};
struct PairArgs {
  ConvArgs c;        // the second layer; its input is the first layer's: c.s0, or the film
  const bf16* Wp1;
  const float* bias1;
  FilmSrc film;
};
constexpr uint32_t kPairRows = 14, kPairCols = 30, kPairPitch = 34, kPairPix = 18 * kPairPitch;
constexpr size_t kPairLds = size_t(kPairPix) * 64 + 2 * 18 * 1024;

// The network's ten input features of a pixel.
__device__ __forceinline__ void featuresOf(const float (&v)[10], bf16x8& lo, bf16x8& hi) {
  lo = hi = zero8();
#pragma unroll
  for (int c = 0; c < 10; ++c) {
    const float f = c < 3 || c == 9 ? ashd::log1pPos(fmaxf(v[c], 0.f), [](float d) { return __builtin_amdgcn_rcpf(d); }) : v[c];
    if (c < 8) lo[c] = bf16(f);
    else hi[c - 8] = bf16(f);
  }
}

template <ConvMode MODE, bool FILM>
__global__ __launch_bounds__(256, 2) void kConvPair(PairArgs p, uint32_t tilesX, uint32_t tilesY, uint32_t tiles) {
  constexpr int R = 8, NT = MODE == kModeLast ? 1 : 2;
  constexpr uint32_t LX = (kPairPix * 4 + 255) / 256, LF = (kPairPix + 255) / 256;
  extern __shared__ __align__(16) bf16 lds[];
  bf16* tile = lds;                      // [kPairPix][4 slots][8], swizzled by column as in kConvLds
  bf16* wts = lds + kPairPix * 32;       // [2 layers][18 fragments][64][8]
  const ConvArgs& a = p.c;
  const uint32_t tid = threadIdx.x, lane = tid & 63, q = lane >> 4, r16 = lane & 15, wv = tid >> 6;
  const uint32_t row0 = (wv >> 1) * R, col0 = (wv & 1) * 16;
  for (uint32_t k = tid; k < 18 * 64; k += 256) {
    *reinterpret_cast<u32x4*>(wts + k * 8) = *reinterpret_cast<const u32x4*>(p.Wp1 + k * 8);
    *reinterpret_cast<u32x4*>(wts + (18 * 64 + k) * 8) = *reinterpret_cast<const u32x4*>(a.Wp + k * 8);
  }
  auto fresh = [&]() {  // as in kConvLds
    uint32_t t = tid;
    asm volatile("" : "+v"(t));
    return t;
  };
  auto origin = [&](uint32_t t, uint32_t& n, int& ty, int& tx) {
    tx = int((t % tilesX) * kPairCols);
    ty = int(((t / tilesX) % tilesY) * kPairRows);
    n = t / (tilesX * tilesY);
  };
  u32x4 px[FILM ? 1 : LX];
  float pf[FILM ? LF : 1][10];
  auto fetch = [&](uint32_t t) {
    const uint32_t tid = fresh();
    uint32_t n;
    int ty, tx;
    origin(t, n, ty, tx);
    if (FILM) {
#pragma unroll
      for (uint32_t j = 0; j < LF; ++j) {
        const uint32_t pix = tid + 256 * j;
        const int y = ty - 2 + int(pix / kPairPitch), x = tx - 2 + int(pix % kPairPitch);
        float4 r = make_float4(0.f, 0.f, 0.f, 0.f), al = r, no = r;
        float de = 0.f;
        if (pix < kPairPix && uint32_t(y) < p.film.H && uint32_t(x) < p.film.W) {
          const size_t k = size_t(y) * p.film.W + x;
          r = p.film.rad[k];
          if (p.film.alb) al = p.film.alb[k];
          if (p.film.nrm) no = p.film.nrm[k];
          if (p.film.dep) de = p.film.dep[k].x;
        }
        pf[j][0] = r.x, pf[j][1] = r.y, pf[j][2] = r.z, pf[j][3] = al.x, pf[j][4] = al.y, pf[j][5] = al.z;
        pf[j][6] = no.x, pf[j][7] = no.y, pf[j][8] = no.z, pf[j][9] = de;
      }
    } else {
      const ChunkSrc src = chunkSrc(a.s0, a.s0, a.H, a.W, n, 0);
#pragma unroll
      for (uint32_t j = 0; j < LX; ++j) {
        const uint32_t k = tid + 256 * j, pix = k >> 2;
        if (k < kPairPix * 4)
          px[j] = loadIn(src, a.H, a.W, ty - 2 + int(pix / kPairPitch), tx - 2 + int(pix % kPairPitch), 8 * (k & 3));
      }
    }
  };
  auto at = [&](uint32_t pix, uint32_t col, uint32_t s) { return tile + (pix * 4 + (s ^ ((col >> 2) & 3))) * 8; };
  auto put = [&]() {
    const uint32_t tid = fresh();
    if (FILM) {
#pragma unroll
      for (uint32_t j = 0; j < LF; ++j) {
        const uint32_t pix = tid + 256 * j, col = pix % kPairPitch;
        bf16x8 lo, hi;
        featuresOf(pf[j], lo, hi);
        if (pix < kPairPix) {
          *reinterpret_cast<bf16x8*>(at(pix, col, 0)) = lo;
          *reinterpret_cast<bf16x8*>(at(pix, col, 1)) = hi;
          *reinterpret_cast<bf16x8*>(at(pix, col, 2)) = zero8();
          *reinterpret_cast<bf16x8*>(at(pix, col, 3)) = zero8();
        }
      }
    } else {
#pragma unroll
      for (uint32_t j = 0; j < LX; ++j) {
        const uint32_t k = tid + 256 * j, pix = k >> 2;
        if (k < kPairPix * 4) *reinterpret_cast<u32x4*>(at(pix, pix % kPairPitch, k & 3)) = px[j];
      }
    }
  };
  uint32_t t = blockIdx.x;
  if (t < tiles) fetch(t);
  float b1[8], b2[8];
  laneBias<kModeAct>(p.bias1, 0, q, b1);
  laneBias<MODE>(a.bias, 0, MODE == kModeLast ? 0 : q, b2);
  while (t < tiles) {
    __syncthreads();  // the previous tile's fragments are consumed
    put();
    __syncthreads();
    const uint32_t next = t + gridDim.x;
    if (next < tiles) fetch(next);  // in flight during both layers
    __builtin_amdgcn_sched_barrier(0);
    uint32_t n;
    int ty, tx;
    origin(t, n, ty, tx);
    {
      f32x4 acc[R][2];
#pragma unroll
      for (int i = 0; i < R; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      chunkMfma<R, 2, kPairPitch>(tile, row0, col0, q, r16, wts + lane * 8, acc);
      __syncthreads();  // the input's fragments are consumed: the first layer takes its place
      const uint32_t col = col0 + r16;
      const bool inX = uint32_t(tx - 1 + int(col)) < a.W;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const bool in = inX && uint32_t(ty - 1 + int(row0) + i) < a.H;
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = bf16(in ? fmaxf(acc[i][j / 4][j % 4] + b1[j], 0.f) : 0.f);
        *reinterpret_cast<bf16x8*>(at((row0 + i) * kPairPitch + col, col, q)) = o;
      }
    }
    __syncthreads();
    f32x4 acc[R][NT];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int k = 0; k < NT; ++k) acc[i][k] = f32x4{0.f, 0.f, 0.f, 0.f};
    // rows 16, 17 and columns 32, 33 still hold input pixels: only dropped outputs read them
    chunkMfma<R, NT, kPairPitch>(tile, row0, col0, q, r16, wts + (18 * 64 + lane) * 8, acc);
    const uint32_t col = col0 + r16;
    const int x = col < kPairCols ? tx + int(col) : int(a.W);  // at the image's edge or past it: dropped
    if (MODE == kModeAct) {
      float bs[8] = {};
#pragma unroll
      for (int i = 0; i < R; i += 2) {
        __builtin_amdgcn_sched_barrier(0);
        if (row0 + i >= kPairRows) continue;
        float v[2][8];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int j = 0; j < 8; ++j) v[k][j] = acc[i + k][j / 4 < NT ? j / 4 : 0][j % 4];
        emit<2, MODE>(a, 0, n, ty + int(row0) + i, x, q, v, b2, bs);
      }
    } else {
      // The 3 channels of a pixel lie in its q = 0 lane: lane group q takes row i + q, so that the
      // exponentials run on all lanes (on a quarter of them they were a third of the kernel's time).
#pragma unroll
      for (int i = 0; i < R; i += 4) {
        __builtin_amdgcn_sched_barrier(0);
        float f[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float g0 = __shfl(acc[i][0][c], int(r16)), g1 = __shfl(acc[i + 1][0][c], int(r16)),
                      g2 = __shfl(acc[i + 2][0][c], int(r16)), g3 = __shfl(acc[i + 3][0][c], int(r16));
          f[c] = expm1f((q < 2 ? (q ? g1 : g0) : (q == 2 ? g2 : g3)) + b2[c]);
        }
        const uint32_t row = row0 + i + q;
        const int y = ty + int(row);
        if (row >= kPairRows || y >= int(a.H) || x >= int(a.W)) continue;
        if (a.rgb) {
          float* o = a.rgb + 3 * ((size_t(n) * a.H + y) * a.W + x);
          o[0] = f[0], o[1] = f[1], o[2] = f[2];
        } else if (y < int(a.filmH) && x < int(a.filmW)) {
          a.film[size_t(y) * a.filmW + x] = make_float4(fmaxf(f[0], 0.f), fmaxf(f[1], 0.f), fmaxf(f[2], 0.f), 1.f);
        }
      }
    }
    t = next;
  }
}

// Convolution of small levels, whose pixels do not fill the chip: a block
// owns 4 rows x 16 columns x 32 output channels and has one wave per
// 32-channel input chunk (K split over the waves), so a layer lasts about one
// round trip to L2 instead of a serial walk over its chunks: a wave loads its
// chunk's 18 weight and 18 input fragments straight from memory, all in
// flight together, and the partial sums are added in chunk order in LDS.
constexpr int kSplitRows = 4;
template <ConvMode MODE>
__global__ __launch_bounds__(64 * kMaxChunks) void kConvSplit(ConvArgs a, uint32_t tilesX, uint32_t tilesY) {
  extern __shared__ __align__(16) float red[];  // [chunk][row][lane][8]
  __shared__ float sB[2 * 32];
  constexpr int R = kSplitRows;
  const uint32_t tid = threadIdx.x, lane = tid & 63, q = lane >> 4, r16 = lane & 15, wv = tid >> 6;
  const uint32_t cg = blockIdx.x % a.nCg, t0 = blockIdx.x / a.nCg;
  const int tx = int((t0 % tilesX) * 16), ty = int(((t0 / tilesX) % tilesY) * R);
  const uint32_t n = t0 / (tilesX * tilesY);
  const int x = tx + int(r16);
  bf16x8 xf[R + 2][3], wf[9][2];
  const ChunkSrc src = chunkSrc(a.s0, a.s1, a.H, a.W, n, __builtin_amdgcn_readfirstlane(wv));
#pragma unroll
  for (int r = 0; r < R + 2; ++r)
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) xf[r][dx] = __builtin_bit_cast(bf16x8, loadIn(src, a.H, a.W, ty + r - 1, x + dx - 1, 8 * q));
  const bf16* wp = a.Wp + ((size_t(cg) * a.nCh + wv) * (18 * 64) + lane) * 8;
#pragma unroll
  for (int k = 0; k < 18; ++k) wf[k / 2][k % 2] = *reinterpret_cast<const bf16x8*>(wp + k * 512);
  f32x4 acc[R][2];
#pragma unroll
  for (int i = 0; i < R; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[tap][t], xf[i + tap / 3][tap % 3], acc[i][t], 0, 0, 0);
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t) *reinterpret_cast<f32x4*>(red + ((wv * R + i) * 64 + lane) * 8 + 4 * t) = acc[i][t];
  __syncthreads();
  float bias[8];
  laneBias<MODE>(a.bias, cg, q, bias);
  for (uint32_t pair = wv; pair < R / 2; pair += a.nCh) {
    float v[2][8] = {};
    for (uint32_t w = 0; w < a.nCh; ++w)
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const f32x4 p = *reinterpret_cast<const f32x4*>(red + ((w * R + 2 * pair + k) * 64 + lane) * 8 + 4 * t);
#pragma unroll
          for (int j = 0; j < 4; ++j) v[k][4 * t + j] += p[j];
        }
    float bs[8] = {};
    emit<2, MODE>(a, cg, n, ty + 2 * int(pair), x, q, v, bias, bs);
    if (MODE == kModeGrad) waveBias(bs, q, r16, sB + 32 * pair);
  }
  if (MODE == kModeGrad) {
    __syncthreads();
    if (tid < 32) tileBias(a, cg, t0, tid, sB, R / 2);
  }
}

// ---------------------------------------------------------- backward-w
// A block (4 waves) owns the 9 taps of a 32 cout x 32 cin block of one
// layer's weights and walks every splits-th pixel tile (TC columns, 256 / TC
// rows).  A tile's output gradient and its input with the halo are staged in
// LDS as they are in memory (64 bytes per pixel, loads of the next tile in
// flight in registers); both operands need 8 consecutive pixels of one channel
// per lane, which ds_read_b64_tr_b16 reads transposed (16 lanes read 4 pixels
// x 16 channels), at any pixel offset, so the nine taps read the one staged
// tile.  Each wave takes 2 of the tile's 8 steps of 32 pixels and keeps all 36
// output tiles in registers: 20 fragments read for 36 MFMAs.  The waves' sums
// are added in wave order through LDS.
//
// One launch does every layer once all output gradients are there: alone, a
// small level's layer cannot fill the chip and lasts as long as a large one.
// A batch of 8 x 128 x 128: 319 us per layer with one wave per tap, 32 x 32
// block and split gathering 2-byte values from memory, 12 us per layer as 19
// launches of this kernel (230 us), 74 us for all layers in one.
struct BwdWLayer {
  Src s0, s1;
  const bf16* dY;  // [N][H][W][32 nCo], masked
  float* part;     // [splits][9][32 nCo][32 nCi]
  uint32_t H, W, tilesX, tilesY, tiles;
  uint16_t nCo, nCi, splits, tc;
  uint32_t block0;  // first block of the layer
};
struct BwdWArgs {
  BwdWLayer l[kNumLayers];
};
static_assert(sizeof(BwdWArgs) <= 4096, "kernel argument limit");
template <int TC> struct BwdWTile {
  static constexpr uint32_t TR = 256 / TC, P = (TR + 2) * (TC + 2);
  static constexpr uint32_t LX = (P * 4 + 255) / 256;
  static constexpr size_t lds = (size_t(P) + 256) * 64;
};
typedef __attribute__((address_space(3))) bf16x4* LdsTr;
// 8 pixels (two groups of 4) x 16 channels, transposed: lane l holds channel l % 16.
__device__ __forceinline__ bf16x8 readTr(const bf16* p0, const bf16* p1) {
  const bf16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((LdsTr)(p0));
  const bf16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((LdsTr)(p1));
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
template <int TC>
__device__ __forceinline__ void bwdW(const BwdWLayer& a, uint32_t block, bf16* lds) {
  using T = BwdWTile<TC>;
  static_assert(T::lds >= 4 * 9 * 1024, "the reduction reuses the staging space");
  bf16* xs = lds;              // [T::P][4 slots][8]
  bf16* ys = lds + T::P * 32;  // [256][4 slots][8]
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint32_t pairs = a.nCo * a.nCi, split = block / pairs;
  const uint32_t cob = (block % pairs) / a.nCi, cib = (block % pairs) % a.nCi;
  u32x4 px[T::LX], py[4];
  auto fresh = [&]() {  // as in kConvLds
    uint32_t i = tid;
    asm volatile("" : "+v"(i));
    return i;
  };
  auto fetch = [&](uint32_t t) {
    const uint32_t tid = fresh();
    const int tx = int((t % a.tilesX) * TC), ty = int(((t / a.tilesX) % a.tilesY) * T::TR);
    const uint32_t n = t / (a.tilesX * a.tilesY);
    const ChunkSrc src = chunkSrc(a.s0, a.s1, a.H, a.W, n, cib);
#pragma unroll
    for (uint32_t j = 0; j < T::LX; ++j) {
      const uint32_t k = tid + 256 * j, pix = k >> 2;
      if (k < T::P * 4)
        px[j] = loadIn(src, a.H, a.W, ty - 1 + int(pix / (TC + 2)), tx - 1 + int(pix % (TC + 2)), 8 * (k & 3));
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t k = tid + 256 * j, pix = k >> 2;
      const uint32_t y = uint32_t(ty) + pix / TC, x = uint32_t(tx) + pix % TC;
      py[j] = u32x4{0, 0, 0, 0};
      if (y < a.H && x < a.W)
        py[j] = *reinterpret_cast<const u32x4*>(a.dY + ((size_t(n) * a.H + y) * a.W + x) * (32 * a.nCo) + 32 * cob + 8 * (k & 3));
    }
  };
  // 16-byte slots swapped in halves by bit 3 of the column: the lane groups of one read use different banks
  auto slot = [](uint32_t col, uint32_t s) { return s ^ (((col >> 3) & 1) << 1); };
  auto put = [&]() {
    const uint32_t tid = fresh();
#pragma unroll
    for (uint32_t j = 0; j < T::LX; ++j) {
      const uint32_t k = tid + 256 * j, pix = k >> 2;
      if (k < T::P * 4) *reinterpret_cast<u32x4*>(xs + (pix * 4 + slot(pix % (TC + 2), k & 3)) * 8) = px[j];
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t k = tid + 256 * j, pix = k >> 2;
      *reinterpret_cast<u32x4*>(ys + (pix * 4 + slot(pix, k & 3)) * 8) = py[j];
    }
  };
  // The lane's addresses in the wave's first step of 32 pixels: pixel group h (of 4 pixels), channel tile c.  The second
  // step and the taps' rows are immediate offsets.
  const uint32_t kp = 8 * (lane >> 4) + ((lane & 15) >> 2), sub = lane & 3;
  constexpr uint32_t stepRows = TC >= 32 ? 1 : 32 / TC;
  uint32_t yAt[2][2], xAt[3][2][2];
#pragma unroll
  for (uint32_t h = 0; h < 2; ++h)
#pragma unroll
    for (uint32_t c = 0; c < 2; ++c) {
      const uint32_t p = 64 * wv + kp + 4 * h, row = 2 * wv * stepRows + (kp + 4 * h) / TC;
      yAt[h][c] = T::P * 32 + p * 32 + slot(p, 2 * c + (sub >> 1)) * 8 + (sub & 1) * 4;
#pragma unroll
      for (uint32_t dx = 0; dx < 3; ++dx) {
        const uint32_t col = (kp + 4 * h) % TC + dx;
        xAt[dx][h][c] = (row * (TC + 2) + col) * 32 + slot(col, 2 * c + (sub >> 1)) * 8 + (sub & 1) * 4;
      }
    }
  f32x4 acc[9][2][2];
#pragma unroll
  for (int k = 0; k < 9; ++k)
#pragma unroll
    for (int i = 0; i < 2; ++i) acc[k][i][0] = acc[k][i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t t = split;
  if (t < a.tiles) fetch(t);
  while (t < a.tiles) {
    __syncthreads();
    put();
    __syncthreads();
    t += a.splits;
    if (t < a.tiles) fetch(t);
#pragma unroll
    for (uint32_t s = 0; s < 2; ++s) {
      bf16x8 A[2];
#pragma unroll
      for (uint32_t c = 0; c < 2; ++c) A[c] = readTr(lds + yAt[0][c] + s * 1024, lds + yAt[1][c] + s * 1024);
#pragma unroll
      for (uint32_t tap = 0; tap < 9; ++tap) {
        const uint32_t off = (s * stepRows + tap / 3) * (TC + 2) * 32;
        if (tap % 3 == 0) __builtin_amdgcn_sched_barrier(0);  // later rows' reads would spill
        bf16x8 B[2];
#pragma unroll
        for (uint32_t c = 0; c < 2; ++c) B[c] = readTr(lds + xAt[tap % 3][0][c] + off, lds + xAt[tap % 3][1][c] + off);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[tap][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[i], B[j], acc[tap][i][j], 0, 0, 0);
      }
    }
  }
  // waves' sums in wave order, one (cout tile, cin tile) of the nine taps at a time
  float* red = reinterpret_cast<float*>(lds);  // [4 waves][9 taps][64 lanes][4]
  const uint32_t Co = 32 * a.nCo, Ci = 32 * a.nCi;
  float* out = a.part + size_t(split) * 9 * Co * Ci;
#pragma unroll
  for (uint32_t ij = 0; ij < 4; ++ij) {
    __syncthreads();
#pragma unroll
    for (uint32_t tap = 0; tap < 9; ++tap)
      *reinterpret_cast<f32x4*>(red + ((wv * 9 + tap) * 64 + lane) * 4) = acc[tap][ij / 2][ij % 2];
    __syncthreads();
    for (uint32_t e = tid; e < 9 * 64; e += 256) {
      f32x4 s = *reinterpret_cast<const f32x4*>(red + e * 4);
      for (uint32_t w = 1; w < 4; ++w) s += *reinterpret_cast<const f32x4*>(red + (w * 9 * 64 + e) * 4);
      const uint32_t tap = e / 64, l = e % 64;
      const uint32_t co = 32 * cob + 16 * (ij / 2) + 4 * (l >> 4), ci = 32 * cib + 16 * (ij % 2) + (l & 15);
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r) out[(size_t(tap) * Co + co + r) * Ci + ci] = s[r];
    }
  }
}

__global__ __launch_bounds__(256, 2) void kConvBwdW(BwdWArgs a) {
  __shared__ __align__(16) bf16 lds[std::max({BwdWTile<32>::lds, BwdWTile<16>::lds, BwdWTile<8>::lds}) / 2];
  int k = 0;
  while (k + 1 < kNumLayers && blockIdx.x >= a.l[k + 1].block0) ++k;
  const BwdWLayer& l = a.l[k];
  const uint32_t block = blockIdx.x - l.block0;
  if (l.tc == 32) bwdW<32>(l, block, lds);
  else if (l.tc == 16) bwdW<16>(l, block, lds);
  else bwdW<8>(l, block, lds);
}

// ------------------------------------------------- parameters (all layers)
// One layer's place in the parameter vector, the packed weights and the
// gradient partial sums.
struct LayerTab {
  struct Row {
    uint32_t CoS, CinS;             // stored channels
    uint32_t co, ca, CaS, cin;      // real output, source-0 and input channels, stored source-0 channels
    uint32_t wOff, bOff;            // FP32 parameters: W[9][CoS][CinS], bias[CoS]
    uint32_t fOff;                  // packed BF16 weights (both layouts)
    uint32_t rOff;                  // real-channel flat order
    uint32_t splits, nbk;           // weight and bias partial sums per element
    size_t wPart, bPart;            // their offsets in the partial-sum buffer
  } r[kNumLayers];
};
// The layer that holds parameter i of the padded vector.
__device__ __forceinline__ const LayerTab::Row& layerOf(const LayerTab& T, uint32_t i) {
  int k = 0;
  while (k + 1 < kNumLayers && i >= T.r[k + 1].wOff) ++k;
  return T.r[k];
}
// Stores weight e of a layer in both fragment orders.  A fragment holds,
// per lane, 8 input channels of one output row; row m of tile t of a
// 32-channel output group is channel 8 (m / 4) + 4 t + m % 4.
__device__ __forceinline__ uint32_t fragIndex(uint32_t out, uint32_t in, uint32_t nIn, uint32_t tap) {
  const uint32_t g = out / 32, c = out % 32, t = (c / 4) & 1, m = 4 * (c / 8) + c % 4;
  return ((((g * (nIn / 32) + in / 32) * 9 + tap) * 2 + t) * 64 + ((in % 32) / 8) * 16 + m) * 8 + in % 8;
}
__device__ __forceinline__ void packWeight(const LayerTab::Row& l, uint32_t e, float w, bf16* wf, bf16* wb) {
  const uint32_t ci = e % l.CinS, co = (e / l.CinS) % l.CoS, tap = e / (l.CinS * l.CoS);
  wf[l.fOff + fragIndex(co, ci, l.CinS, tap)] = bf16(w);
  wb[l.fOff + fragIndex(ci, co, l.CoS, 8 - tap)] = bf16(w);  // backward-x: taps reversed, roles exchanged
}
__global__ __launch_bounds__(256) void kPackW(LayerTab T, const float* theta, uint32_t n, bf16* wf, bf16* wb) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const LayerTab::Row& l = layerOf(T, i);
  if (i < l.bOff) packWeight(l, i - l.wOff, theta[i], wf, wb);
}

// Parameter gradients from the partial sums, and (ADAM) the optimiser step
// and the packed weights, for 32 parameters per block: eight groups of 32
// threads each add an eighth of a parameter's partial sums in order, then the
// groups' sums are added in group order.  One launch of 45 us for a batch of
// 8 x 128 x 128, where per-layer reductions of weights (8 us) and biases (one
// block, 41 us), the Adam pass and 19 packing launches took 1.1 ms.
struct AdamArgs {
  float *theta, *m, *v;
  float lr, b1, b2, eps, c1, c2;
};
template <bool ADAM>
__global__ __launch_bounds__(256) void kGradients(LayerTab T, const float* part, float* grad, AdamArgs o, bf16* wf, bf16* wb) {
  __shared__ float red[8][32];
  const uint32_t c = threadIdx.x & 31, g = threadIdx.x >> 5;
  const uint32_t i = blockIdx.x * 32 + c;  // every layer's weights and biases are whole blocks of 32
  const LayerTab::Row& l = layerOf(T, blockIdx.x * 32);
  const bool isW = blockIdx.x * 32 < l.bOff;
  const uint32_t e = isW ? i - l.wOff : i - l.bOff, n = isW ? l.splits : l.nbk;
  const size_t stride = isW ? size_t(9) * l.CoS * l.CinS : l.CoS;
  const float* p = part + (isW ? l.wPart : l.bPart) + e;
  const uint32_t k0 = uint32_t(uint64_t(n) * g / 8), k1 = uint32_t(uint64_t(n) * (g + 1) / 8);
  float s = 0.f;
#pragma unroll 8
  for (uint32_t k = k0; k < k1; ++k) s += p[k * stride];
  red[g][c] = s;
  __syncthreads();
  if (g) return;
  for (uint32_t k = 1; k < 8; ++k) s += red[k][c];
  grad[i] = s;
  if (ADAM) {
    const float mi = o.b1 * o.m[i] + (1.f - o.b1) * s;
    const float vi = o.b2 * o.v[i] + (1.f - o.b2) * s * s;
    o.m[i] = mi;
    o.v[i] = vi;
    const float w = o.theta[i] - o.lr * (mi / o.c1) / (sqrtf(vi / o.c2) + o.eps);
    o.theta[i] = w;
    if (isW) packWeight(l, e, w, wf, wb);
  }
}

// Padded parameter vector -> real-channel flat order.
__global__ __launch_bounds__(256) void kRealOrder(LayerTab T, const float* pad, float* real, uint32_t n) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  int k = 0;
  while (k + 1 < kNumLayers && i >= T.r[k + 1].rOff) ++k;
  const LayerTab::Row& l = T.r[k];
  const uint32_t e = i - l.rOff, nw = 9 * l.co * l.cin;
  if (e >= nw) {
    real[i] = pad[l.bOff + (e - nw)];
    return;
  }
  const uint32_t r = e % l.cin, co = (e / l.cin) % l.co, tap = e / (l.cin * l.co);
  const uint32_t s = r < l.ca ? r : l.CaS + (r - l.ca);
  real[i] = pad[l.wOff + (tap * l.CoS + co) * l.CinS + s];
}

// --------------------------------------------------------- elementwise
// Raw (P, 10) FP32 -> features (P, 32) BF16
__global__ __launch_bounds__(256) void kFeatures(const float* raw, bf16* x, uint32_t P) {
  const uint32_t p = blockIdx.x * 256 + threadIdx.x;
  if (p >= P) return;
  float v[10];
  const float2* r = reinterpret_cast<const float2*>(raw + size_t(p) * 10);
#pragma unroll
  for (int k = 0; k < 5; ++k) v[2 * k] = r[k].x, v[2 * k + 1] = r[k].y;
  bf16x8* o = reinterpret_cast<bf16x8*>(x + size_t(p) * 32);
  featuresOf(v, o[0], o[1]);
  o[2] = o[3] = zero8();
}

// Mean L1 in log space: per pixel the gradient sign / (3P) of the three
// channels as the last layer's BF16 output gradient, per block of 256 pixels
// the partial loss and bias-gradient sums (trees of fixed order).
__global__ __launch_bounds__(256) void kLoss(const float4* y, const float* target, uint32_t P, bf16* dY, float* partial,
                                             float* bPart) {
  __shared__ float4 red[256];
  const uint32_t p = blockIdx.x * 256 + threadIdx.x;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);  // gradients of the three channels, loss
  if (p < P) {
    const float4 v = y[p];
    const float d[3] = {v.x - log1pf(fmaxf(target[3 * size_t(p)], 0.f)), v.y - log1pf(fmaxf(target[3 * size_t(p) + 1], 0.f)),
                        v.z - log1pf(fmaxf(target[3 * size_t(p) + 2], 0.f))};
    float g[3];
    for (int c = 0; c < 3; ++c) {
      s.w += fabsf(d[c]);
      g[c] = (d[c] > 0.f ? 1.f : (d[c] < 0.f ? -1.f : 0.f)) / float(3.0 * double(P));
    }
    s.x = g[0], s.y = g[1], s.z = g[2];
    bf16x8 o = zero8();
    bf16x8* row = reinterpret_cast<bf16x8*>(dY + size_t(p) * 32);
    row[1] = row[2] = row[3] = o;
    o[0] = bf16(g[0]), o[1] = bf16(g[1]), o[2] = bf16(g[2]);
    row[0] = o;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (int(threadIdx.x) < k) {
      const float4 b = red[threadIdx.x + k];
      float4& a = red[threadIdx.x];
      a.x += b.x, a.y += b.y, a.z += b.z, a.w += b.w;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0].w;
  if (threadIdx.x < 32) {
    const float4 r = red[0];
    bPart[size_t(blockIdx.x) * 32 + threadIdx.x] =
        threadIdx.x == 0 ? r.x : threadIdx.x == 1 ? r.y : threadIdx.x == 2 ? r.z : 0.f;
  }
}

template <class T> struct Buf {
  T* p = nullptr;
  size_t n = 0;
  size_t cap = 0;
  hipError_t alloc(size_t count) {
    release();
    n = cap = count;
    return hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T));
  }
  // Keeps the allocation when it is large enough: a shape change then costs
  // no hipFree, which would wait for the whole device.
  hipError_t reserve(size_t count) {
    if (p && count <= cap) {
      n = count;
      return hipSuccess;
    }
    return alloc(count);
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = cap = 0;
  }
};

struct Layer {
  uint32_t ca, cb, co;     // real channels (source 0, skip source, out)
  uint32_t CaS, CbS, CoS;  // stored channels
  bool relu;
  size_t wOff, bOff;  // into the FP32 parameter vector
  size_t fOff;        // into the BF16 packed weights (Wf and Wb each)
};

struct Act {
  uint32_t N, H, W, C;
  int layer = -1;   // the layer that writes it
  Buf<bf16> a;
  Buf<bf16> g;      // training: its complete gradient, ReLU mask applied
  Buf<float> skip;  // training: the skip branch's part of the gradient (encoder outputs)
  size_t count() const { return size_t(N) * H * W * C; }
};

}  // namespace

struct ash_denoiser {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  std::vector<Layer> L;
  size_t nParams = 0;  // padded FP32 parameter count
  size_t nPacked = 0;  // BF16 weights per layout
  Buf<float> theta, grad, m, v;
  Buf<bf16> wf, wb;
  uint64_t step = 0;
  // activations for the current batch shape
  uint32_t N = 0, H = 0, W = 0;
  Act x, out;
  Act enc[kLevels][2], pooled[kLevels], dec[kLevels][2];
  Buf<float> outF, lossPart, raw, target, rgb;
  Buf<float> part;  // weight and bias gradient partial sums of all layers
  Buf<float> real;  // parameters or gradient in the real-channel order
  int numCU = 256;
  bool wDirty = true;
};

static int dfail(ash_denoiser* d, int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  d->err = buf;
  return code;
}

#define DH(d, x)                                                                              \
  do {                                                                                        \
    hipError_t e_ = (x);                                                                      \
    if (e_ != hipSuccess) return dfail(d, ASH_E_HIP, "%s: %s", #x, hipGetErrorString(e_));   \
  } while (0)

static unsigned blocks(size_t n, unsigned b = 256) { return unsigned((n + b - 1) / b); }

static void buildLayers(ash_denoiser* d) {
  auto add = [&](uint32_t ca, uint32_t cb, uint32_t co, bool relu) {
    Layer l;
    l.ca = ca, l.cb = cb, l.co = co;
    l.CaS = pad32(ca), l.CbS = cb ? pad32(cb) : 0, l.CoS = pad32(co);
    l.relu = relu;
    d->L.push_back(l);
  };
  uint32_t c = kInCh;
  for (int lv = 0; lv < kLevels; ++lv) {
    add(c, 0, kWidths[lv], true);
    add(kWidths[lv], 0, kWidths[lv], true);
    c = kWidths[lv];
  }
  for (int lv = kLevels - 2; lv >= 0; --lv) {
    add(c, kWidths[lv], kWidths[lv], true);
    add(kWidths[lv], 0, kWidths[lv], true);
    c = kWidths[lv];
  }
  add(c, 0, kOutCh, false);
  size_t off = 0, foff = 0;
  for (auto& l : d->L) {
    uint32_t cin = l.CaS + l.CbS;
    l.wOff = off;
    off += size_t(9) * l.CoS * cin;
    l.bOff = off;
    off += l.CoS;
    l.fOff = foff;
    foff += size_t(9) * l.CoS * cin;
  }
  d->nParams = off;
  d->nPacked = foff;
}

// Real-channel index of stored input channel `s` of a layer, or -1 (padding).
static int realIn(const Layer& l, uint32_t s) {
  if (s < l.CaS) return s < l.ca ? int(s) : -1;
  s -= l.CaS;
  return s < l.cb ? int(l.ca + s) : -1;
}

static size_t realCount(const ash_denoiser* d) {
  size_t n = 0;
  for (auto& l : d->L) n += size_t(9) * l.co * (l.ca + l.cb) + l.co;
  return n;
}

// real-channel flat order -> padded device layout
static void toPadded(const ash_denoiser* d, const float* real, std::vector<float>& pad) {
  pad.assign(d->nParams, 0.f);
  size_t k = 0;
  for (auto& l : d->L) {
    uint32_t cin = l.CaS + l.CbS, rin = l.ca + l.cb;
    for (uint32_t t = 0; t < 9; ++t)
      for (uint32_t co = 0; co < l.co; ++co)
        for (uint32_t s = 0; s < cin; ++s) {
          int r = realIn(l, s);
          if (r >= 0) pad[l.wOff + (size_t(t) * l.CoS + co) * cin + s] = real[k + (size_t(t) * l.co + co) * rin + r];
        }
    k += size_t(9) * l.co * rin;
    for (uint32_t co = 0; co < l.co; ++co) pad[l.bOff + co] = real[k + co];
    k += l.co;
  }
}

// Every layer's offsets; the partial-sum fields are filled by the backward pass.
static LayerTab layerTab(const ash_denoiser* d) {
  LayerTab T;
  std::memset(&T, 0, sizeof T);
  size_t k = 0;
  for (size_t i = 0; i < d->L.size(); ++i) {
    const Layer& l = d->L[i];
    LayerTab::Row& r = T.r[i];
    r.CoS = l.CoS, r.CinS = l.CaS + l.CbS, r.co = l.co, r.ca = l.ca, r.CaS = l.CaS, r.cin = l.ca + l.cb;
    r.wOff = uint32_t(l.wOff), r.bOff = uint32_t(l.bOff), r.fOff = uint32_t(l.fOff), r.rOff = uint32_t(k);
    k += size_t(9) * l.co * (l.ca + l.cb) + l.co;
  }
  return T;
}

static int packWeights(ash_denoiser* d) {
  if (!d->wDirty) return ASH_OK;
  kPackW<<<blocks(d->nParams), 256, 0, d->stream>>>(layerTab(d), d->theta.p, uint32_t(d->nParams), d->wf.p, d->wb.p);
  DH(d, hipGetLastError());
  d->wDirty = false;
  return ASH_OK;
}

// Copies a padded parameter-sized vector to the host in the real-channel order.
static int readReal(ash_denoiser* d, const float* pad, float* host) {
  const size_t n = realCount(d);
  DH(d, d->real.reserve(n));
  kRealOrder<<<blocks(n), 256, 0, d->stream>>>(layerTab(d), pad, d->real.p, uint32_t(n));
  DH(d, hipGetLastError());
  DH(d, hipMemcpyAsync(host, d->real.p, n * sizeof(float), hipMemcpyDeviceToHost, d->stream));
  DH(d, hipStreamSynchronize(d->stream));
  return ASH_OK;
}

static int allocAct(ash_denoiser* d, Act& t, uint32_t N, uint32_t H, uint32_t W, uint32_t C) {
  t.N = N, t.H = H, t.W = W, t.C = C;
  DH(d, t.a.reserve(t.count()));
  return ASH_OK;
}

static int ensureShape(ash_denoiser* d, uint32_t N, uint32_t H, uint32_t W) {
  if (H % 16 || W % 16 || !N) return dfail(d, ASH_E_INVALID, "batch spatial size must be a multiple of 16");
  if (d->N == N && d->H == H && d->W == W) return ASH_OK;
  int rc;
#define CK(x) \
  if ((rc = (x))) return rc
  CK(allocAct(d, d->x, N, H, W, 32));
  for (int lv = 0; lv < kLevels; ++lv) {
    uint32_t h = H >> lv, w = W >> lv, c = pad32(kWidths[lv]);
    if (lv) CK(allocAct(d, d->pooled[lv], N, h, w, pad32(kWidths[lv - 1])));
    CK(allocAct(d, d->enc[lv][0], N, h, w, c));
    CK(allocAct(d, d->enc[lv][1], N, h, w, c));
    if (lv < kLevels - 1) {
      CK(allocAct(d, d->dec[lv][0], N, h, w, c));
      CK(allocAct(d, d->dec[lv][1], N, h, w, c));
    }
  }
  CK(allocAct(d, d->out, N, H, W, 32));
#undef CK
  d->N = N, d->H = H, d->W = W;
  return ASH_OK;
}

// Layer schedule: the conv inputs of every layer in network order.
struct Step {
  int layer;
  Act* s0;
  bool up;
  Act* s1;
  Act* out;
  Act* pool;  // the pooled copy of the output, or null
};

static std::vector<Step> schedule(ash_denoiser* d) {
  std::vector<Step> s;
  int li = 0;
  Act* h = &d->x;
  auto add = [&](Act* s0, bool up, Act* s1, Act* out, Act* pool) {
    out->layer = li;
    s.push_back({li++, s0, up, s1, out, pool});
    h = out;
  };
  for (int lv = 0; lv < kLevels; ++lv) {
    add(lv ? &d->pooled[lv] : h, false, nullptr, &d->enc[lv][0], nullptr);
    add(h, false, nullptr, &d->enc[lv][1], lv + 1 < kLevels ? &d->pooled[lv + 1] : nullptr);
  }
  for (int lv = kLevels - 2; lv >= 0; --lv) {
    add(h, true, &d->enc[lv][1], &d->dec[lv][0], nullptr);
    add(h, false, nullptr, &d->dec[lv][1], nullptr);
  }
  add(h, false, nullptr, &d->out, nullptr);
  return s;
}

// Which kernel runs a convolution and its pixel tiles.
enum ConvKind { kKindSplit, kKind4, kKind8, kKind8x2 };
struct ConvPlan {
  ConvKind kind;
  uint32_t tilesX, tilesY, tiles;  // tiles = N tilesX tilesY
};
// The larger a block's tile, the less it reads per product, so the largest that gives every CU a block is taken: waiting
// for two blocks a CU costs 1024 -> 984 us at 1920 x 1080, 403 -> 367 at 960 x 540 and 265 -> 239 at 640 x 360 (two
// blocks -> one).  16 x 16 pixels by two output groups before 16 x 32 by one: without it 984 -> 1086 us.  8 rows are for
// images the 16-row tiles leave CUs idle at: taken for the finest level of 1920 x 1080 instead they cost 1033 -> 1180 us.
// Below one such block a CU the input channels are split over a block's waves: with 8-row tiles from half a block a CU on,
// 1920 x 1080 goes 984 -> 997 us and 317 x 179 166 -> 183.  (Whole passes, before the first and last pairs were fused.)
static ConvPlan convPlan(const ash_denoiser* d, uint32_t N, uint32_t H, uint32_t W, uint32_t nCg) {
  auto make = [&](ConvKind k, uint32_t tr, uint32_t tc) {
    ConvPlan p{k, (W + tc - 1) / tc, (H + tr - 1) / tr, 0};
    p.tiles = N * p.tilesX * p.tilesY;
    return p;
  };
  const uint32_t cus = uint32_t(d->numCU);
  if (nCg % 2 == 0) {
    const ConvPlan p = make(kKind8x2, 16, 16);
    if (uint64_t(p.tiles) * (nCg / 2) >= cus) return p;
  }
  const ConvPlan p8 = make(kKind8, 16, 32);
  if (uint64_t(p8.tiles) * nCg >= cus) return p8;
  const ConvPlan p4 = make(kKind4, 8, 32);
  if (uint64_t(p4.tiles) * nCg >= cus) return p4;
  return make(kKindSplit, kSplitRows, 16);
}

template <int R, int CW, int NT, ConvMode MODE>
static void convLds(const ash_denoiser* d, const ConvArgs& a, const ConvPlan& p) {
  const uint32_t cgb = a.nCg / CW, items = p.tiles * cgb;
  const uint32_t cap = std::max<uint32_t>(uint32_t(d->numCU) * (R == 8 ? 2 : 3) / cgb, 1) * cgb;  // whole sets of output groups
  kConvLds<R, CW, NT, MODE><<<std::min(items, cap), 256, ConvTile<R, CW>::lds, d->stream>>>(a, p.tilesX, p.tilesY, items);
}
template <ConvMode MODE>
static void launchConv(const ash_denoiser* d, const ConvArgs& a, const ConvPlan& p) {
  constexpr int NT = MODE == kModeLast ? 1 : 2;  // the last layer's 3 channels lie in the first of the group's two tiles
  if (p.kind == kKindSplit) {
    const size_t lds = size_t(a.nCh) * kSplitRows * 64 * 8 * sizeof(float);
    kConvSplit<MODE><<<p.tiles * a.nCg, 64 * a.nCh, lds, d->stream>>>(a, p.tilesX, p.tilesY);
  } else if (p.kind == kKind4) {
    convLds<4, 1, NT, MODE>(d, a, p);
  } else if (p.kind == kKind8) {
    convLds<8, 1, NT, MODE>(d, a, p);
  } else if constexpr (MODE != kModeLast) {  // that layer has one output group
    convLds<8, 2, NT, MODE>(d, a, p);
  }
}

// What the last layer writes (null: not wanted).
struct Output {
  float* pred = nullptr;    // training: [pixel][4], log space
  float* rgb = nullptr;     // inference: [pixel][3], or
  float4* film = nullptr;   // filmW x filmH RGBA
  uint32_t filmW = 0, filmH = 0;
};

static int checkLayer(ash_denoiser* d, const Step& st) {
  const Layer& l = d->L[st.layer];
  const Act& o = *st.out;
  const bool fits = st.s0->C == l.CaS && (st.s1 ? st.s1->C : 0) == l.CbS && o.C == l.CoS && l.CaS + l.CbS <= 32 * kMaxChunks &&
                    l.CoS <= 32 * kMaxChunks && st.s0->H * (st.up ? 2 : 1) == o.H && st.s0->W * (st.up ? 2 : 1) == o.W &&
                    (!st.s1 || (st.s1->H == o.H && st.s1->W == o.W));
  return fits ? ASH_OK : dfail(d, ASH_E_INVALID, "layer %d: shape or channel layout mismatch", st.layer);
}

// Two layers of the finest level in one launch (see kConvPair): steps a and b.
template <ConvMode MODE>
static void launchPair(ash_denoiser* d, const Step& a, const Step& b, const Output& out, const FilmSrc* film) {
  PairArgs p;
  std::memset(&p, 0, sizeof p);
  const Layer &la = d->L[a.layer], &lb = d->L[b.layer];
  p.c.s0 = Src{a.s0->a.p, a.s0->C, 0};
  p.c.N = b.out->N, p.c.H = b.out->H, p.c.W = b.out->W;
  p.c.nCh = p.c.nCg = 1;
  p.c.Wp = d->wf.p + lb.fOff;
  p.c.bias = d->theta.p + lb.bOff;
  if (MODE == kModeAct) p.c.Y = b.out->a.p, p.c.pool = b.pool->a.p;
  else p.c.rgb = out.rgb, p.c.film = out.film, p.c.filmW = out.filmW, p.c.filmH = out.filmH;
  p.Wp1 = d->wf.p + la.fOff;
  p.bias1 = d->theta.p + la.bOff;
  if (film) p.film = *film;
  const uint32_t tx = (p.c.W + kPairCols - 1) / kPairCols, ty = (p.c.H + kPairRows - 1) / kPairRows, tiles = p.c.N * tx * ty;
  const uint32_t grid = std::min(tiles, 2 * uint32_t(d->numCU));
  if (film) kConvPair<kModeAct, true><<<grid, 256, kPairLds, d->stream>>>(p, tx, ty, tiles);
  else kConvPair<MODE, false><<<grid, 256, kPairLds, d->stream>>>(p, tx, ty, tiles);
}

// out.pred: a training batch, every layer's output is kept; else the finest
// level's first and last two layers run as pairs, the first ones straight
// from `film` where given (else from the packed features).
static int forwardPass(ash_denoiser* d, const Output& out, const FilmSrc* film = nullptr) {
  int rc = packWeights(d);
  if (rc) return rc;
  const std::vector<Step> sched = schedule(d);
  for (const Step& st : sched)
    if ((rc = checkLayer(d, st))) return rc;
  for (size_t k = 0; k < sched.size(); ++k) {
    const Step& st = sched[k];
    if (!out.pred && k == 0) {
      launchPair<kModeAct>(d, st, sched[++k], out, film);
      continue;
    }
    if (!out.pred && k + 2 == sched.size()) {
      launchPair<kModeLast>(d, st, sched[++k], out, nullptr);
      continue;
    }
    const Layer& l = d->L[st.layer];
    const Act& o = *st.out;
    ConvArgs a;
    std::memset(&a, 0, sizeof a);
    a.s0 = Src{st.s0->a.p, st.s0->C, st.up ? 1u : 0u};
    if (st.s1) a.s1 = Src{st.s1->a.p, st.s1->C, 0};
    a.N = o.N, a.H = o.H, a.W = o.W;
    a.nCh = (l.CaS + l.CbS) / 32, a.nCg = l.CoS / 32;
    a.Wp = d->wf.p + l.fOff;
    a.bias = d->theta.p + l.bOff;
    if (l.relu) {
      a.Y = o.a.p;
      if (st.pool) a.pool = st.pool->a.p;
    } else {
      a.Yf = out.pred;
    }
    const ConvPlan plan = convPlan(d, a.N, a.H, a.W, a.nCg);
    if (l.relu) launchConv<kModeAct>(d, a, plan);
    else launchConv<kModeLast>(d, a, plan);
  }
  DH(d, hipGetLastError());
  return ASH_OK;
}

// Forward pass of a training batch: prediction kept in outF, gradient buffers made.
static int trainForward(ash_denoiser* d) {
  const size_t P = size_t(d->N) * d->H * d->W;
  DH(d, d->outF.reserve(P * 4));
  DH(d, d->lossPart.reserve(blocks(P)));
  DH(d, d->out.g.reserve(d->out.count()));
  for (int lv = 0; lv < kLevels; ++lv)
    for (int k = 0; k < 2; ++k) {
      DH(d, d->enc[lv][k].g.reserve(d->enc[lv][k].count()));
      if (lv < kLevels - 1) DH(d, d->dec[lv][k].g.reserve(d->dec[lv][k].count()));
      if (lv < kLevels - 1 && k) DH(d, d->enc[lv][k].skip.reserve(d->enc[lv][k].count()));
    }
  Output o;
  o.pred = d->outF.p;
  return forwardPass(d, o);
}

// Pixel tiles of a layer's weight gradient: 32, 16 or 8 columns by the
// image's width, kBwdWTiles of them per block (fewer partial sums to write and
// add than with a block per tile, more blocks than with one per CU).  2, 4 and
// 8 a block: 3.62, 3.45 and 3.42 ms for 4 steps on 8 crops of 128 x 128, 680,
// 684 and 707 us for a gradient of 2 images of 80 x 48.
constexpr uint32_t kBwdWTiles = 4;
static void bwdWPlan(const Layer& l, uint32_t N, uint32_t H, uint32_t W, BwdWLayer& p) {
  p.tc = uint16_t(W > 16 ? 32 : W > 8 ? 16 : 8);
  const uint32_t tr = 256 / p.tc;
  p.H = H, p.W = W;
  p.nCo = uint16_t(l.CoS / 32), p.nCi = uint16_t((l.CaS + l.CbS) / 32);
  p.tilesX = (W + p.tc - 1) / p.tc, p.tilesY = (H + tr - 1) / tr;
  p.tiles = N * p.tilesX * p.tilesY;
  p.splits = uint16_t(std::min<uint32_t>((p.tiles + kBwdWTiles - 1) / kBwdWTiles, 512));
}

// Loss, then the gradient of the loss w.r.t. all parameters into d->grad;
// with `adam`, the optimiser step too.
static int backwardPass(ash_denoiser* d, const AdamArgs* adam) {
  const std::vector<Step> sched = schedule(d);
  const uint32_t N = d->N;
  const size_t P = size_t(N) * d->H * d->W;
  // a convolution's backward-x plan, and the partial sums' places
  auto xPlan = [&](const Step& st) { return convPlan(d, N, st.out->H, st.out->W, (d->L[st.layer].CaS + d->L[st.layer].CbS) / 32); };
  LayerTab T = layerTab(d);
  BwdWArgs w;
  std::memset(&w, 0, sizeof w);
  uint32_t wBlocks = 0;
  for (const Step& st : sched) {
    const Layer& l = d->L[st.layer];
    BwdWLayer& wl = w.l[st.layer];
    bwdWPlan(l, N, st.out->H, st.out->W, wl);
    T.r[st.layer].splits = wl.splits;
    wl.block0 = wBlocks;
    wBlocks += uint32_t(wl.splits) * wl.nCo * wl.nCi;
    // the bias gradient is summed where the output's gradient is completed: by the layer that reads it
    // (its pooled copy, where there is one), or by the loss
    int made = -1;
    if (st.layer > 0) {
      const Act* src = st.s0;
      for (int lv = 1; lv < kLevels; ++lv)
        if (src == &d->pooled[lv]) src = &d->enc[lv - 1][1];
      made = src->layer;
    }
    if (made >= 0) T.r[made].nbk = xPlan(st).tiles;
  }
  T.r[sched.back().layer].nbk = blocks(P);
  size_t off = 0;
  for (auto& r : T.r) {
    r.wPart = off;
    off += size_t(r.splits) * 9 * r.CoS * r.CinS;
    r.bPart = off;
    off += size_t(r.nbk) * r.CoS;
  }
  DH(d, d->part.reserve(off));
  kLoss<<<blocks(P), 256, 0, d->stream>>>(reinterpret_cast<const float4*>(d->outF.p), d->target.p, uint32_t(P), d->out.g.p,
                                          d->lossPart.p, d->part.p + T.r[sched.back().layer].bPart);
  for (int k = int(sched.size()) - 1; k >= 0; --k) {
    const Step& st = sched[k];
    const Layer& l = d->L[st.layer];
    const Act& o = *st.out;
    BwdWLayer& wl = w.l[st.layer];
    wl.s0 = Src{st.s0->a.p, st.s0->C, st.up ? 1u : 0u};
    if (st.s1) wl.s1 = Src{st.s1->a.p, st.s1->C, 0};
    wl.dY = o.g.p;
    wl.part = d->part.p + T.r[st.layer].wPart;
    if (st.s0 == &d->x) continue;  // no gradient for the input features
    ConvArgs a;
    std::memset(&a, 0, sizeof a);
    a.s0 = Src{o.g.p, o.C, 0};
    a.N = N, a.H = o.H, a.W = o.W;
    a.nCh = l.CoS / 32, a.nCg = (l.CaS + l.CbS) / 32;
    a.Wp = d->wb.p + l.fOff;
    a.cg0 = l.CaS / 32;
    Act* dst = st.s0;
    a.d0.kind = st.up ? kGradUp : kGradFinal;
    for (int lv = 1; lv < kLevels; ++lv)
      if (dst == &d->pooled[lv]) {
        dst = &d->enc[lv - 1][1];
        a.d0.kind = kGradPool;
        a.d0.skip = dst->skip.p;
      }
    a.d0.C = dst->C, a.d0.g = dst->g.p, a.d0.act = dst->a.p;
    a.d0.bPart = d->part.p + T.r[dst->layer].bPart;
    if (st.s1) a.d1.kind = kGradSkip, a.d1.C = st.s1->C, a.d1.skip = st.s1->skip.p;
    launchConv<kModeGrad>(d, a, xPlan(st));
  }
  kConvBwdW<<<wBlocks, 256, 0, d->stream>>>(w);
  const uint32_t nb = uint32_t(d->nParams / 32);
  if (adam) kGradients<true><<<nb, 256, 0, d->stream>>>(T, d->part.p, d->grad.p, *adam, d->wf.p, d->wb.p);
  else kGradients<false><<<nb, 256, 0, d->stream>>>(T, d->part.p, d->grad.p, AdamArgs{}, nullptr, nullptr);
  DH(d, hipGetLastError());
  if (adam) ++d->step;
  return ASH_OK;
}

static int uploadBatch(ash_denoiser* d, uint32_t n, uint32_t h, uint32_t w, const float* input, const float* target) {
  int rc = ensureShape(d, n, h, w);
  if (rc) return rc;
  size_t P = size_t(n) * h * w;
  if (d->raw.n < P * kInCh) DH(d, d->raw.alloc(P * kInCh));
  DH(d, hipMemcpyAsync(d->raw.p, input, P * kInCh * sizeof(float), hipMemcpyHostToDevice, d->stream));
  kFeatures<<<blocks(P), 256, 0, d->stream>>>(d->raw.p, d->x.a.p, uint32_t(P));
  if (target) {
    if (d->target.n < P * kOutCh) DH(d, d->target.alloc(P * kOutCh));
    DH(d, hipMemcpyAsync(d->target.p, target, P * kOutCh * sizeof(float), hipMemcpyHostToDevice, d->stream));
  }
  DH(d, hipGetLastError());
  return ASH_OK;
}

static int lossAndBackward(ash_denoiser* d, float* loss, const AdamArgs* adam) {
  size_t P = size_t(d->N) * d->H * d->W;
  unsigned nb = blocks(P);
  std::vector<float> part(nb);
  int rc = backwardPass(d, adam);
  if (rc) return rc;
  DH(d, hipMemcpyAsync(part.data(), d->lossPart.p, nb * sizeof(float), hipMemcpyDeviceToHost, d->stream));
  DH(d, hipStreamSynchronize(d->stream));
  double s = 0;
  for (float v : part) s += v;
  if (loss) *loss = float(s / (3.0 * double(P)));
  return ASH_OK;
}

extern "C" {

int ash_denoiser_create(int device, uint32_t seed, ash_denoiser** out) {
  if (!out) return ASH_E_INVALID;
  *out = nullptr;
  int nd = 0;
  if (hipGetDeviceCount(&nd) != hipSuccess || device < 0 || device >= nd) return ASH_E_HIP;
  ash_denoiser* d = new ash_denoiser();
  d->device = device;
  if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess) {
    delete d;
    return ASH_E_HIP;
  }
  // the pair kernels hold 74 KB of LDS per block, above the default limit
  for (const void* f : {reinterpret_cast<const void*>(kConvPair<kModeAct, true>),
                        reinterpret_cast<const void*>(kConvPair<kModeAct, false>),
                        reinterpret_cast<const void*>(kConvPair<kModeLast, false>)})
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, int(kPairLds)) != hipSuccess) (void)hipGetLastError();
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cus > 0) d->numCU = cus;
  buildLayers(d);
  if (d->theta.alloc(d->nParams) || d->grad.alloc(d->nParams) || d->m.alloc(d->nParams) || d->v.alloc(d->nParams) ||
      d->wf.alloc(d->nPacked) || d->wb.alloc(d->nPacked)) {
    ash_denoiser_destroy(d);
    return ASH_E_NOMEM;
  }
  // He-normal initialisation over the real fan-in, zero bias
  std::mt19937_64 rng(seed ? seed : 1);
  std::normal_distribution<double> nd01(0.0, 1.0);
  std::vector<float> real(realCount(d));
  size_t k = 0;
  for (auto& l : d->L) {
    size_t fan = size_t(9) * (l.ca + l.cb);
    double sd = std::sqrt((l.relu ? 2.0 : 1.0) / double(fan));
    for (size_t i = 0; i < fan * l.co; ++i) real[k++] = float(nd01(rng) * sd);
    for (uint32_t i = 0; i < l.co; ++i) real[k++] = 0.f;
  }
  int rc = ash_denoiser_set_params(d, real.data());
  if (rc) {
    ash_denoiser_destroy(d);
    return rc;
  }
  *out = d;
  return ASH_OK;
}

void ash_denoiser_destroy(ash_denoiser* d) {
  if (!d) return;
  (void)hipSetDevice(d->device);
  if (d->stream) (void)hipStreamSynchronize(d->stream);
  for (auto* b : {&d->theta, &d->grad, &d->m, &d->v, &d->outF, &d->lossPart, &d->raw, &d->target, &d->rgb, &d->part, &d->real})
    b->release();
  d->wf.release(), d->wb.release();
  auto rel = [](Act& t) { t.a.release(), t.g.release(), t.skip.release(); };
  rel(d->x), rel(d->out);
  for (int lv = 0; lv < kLevels; ++lv) {
    rel(d->enc[lv][0]), rel(d->enc[lv][1]), rel(d->pooled[lv]), rel(d->dec[lv][0]), rel(d->dec[lv][1]);
  }
  if (d->stream) (void)hipStreamDestroy(d->stream);
  delete d;
}

const char* ash_denoiser_last_error(ash_denoiser* d) { return d ? d->err.c_str() : "null denoiser"; }

int ash_denoiser_num_params(ash_denoiser* d, uint64_t* n) {
  if (!d || !n) return ASH_E_INVALID;
  *n = realCount(d);
  return ASH_OK;
}

int ash_denoiser_get_params(ash_denoiser* d, float* host) {
  if (!d || !host) return ASH_E_INVALID;
  DH(d, hipSetDevice(d->device));
  return readReal(d, d->theta.p, host);
}

int ash_denoiser_set_params(ash_denoiser* d, const float* host) {
  if (!d || !host) return ASH_E_INVALID;
  std::vector<float> pad;
  toPadded(d, host, pad);
  DH(d, hipSetDevice(d->device));
  DH(d, hipMemcpyAsync(d->theta.p, pad.data(), d->nParams * sizeof(float), hipMemcpyHostToDevice, d->stream));
  DH(d, hipMemsetAsync(d->m.p, 0, d->nParams * sizeof(float), d->stream));
  DH(d, hipMemsetAsync(d->v.p, 0, d->nParams * sizeof(float), d->stream));
  DH(d, hipStreamSynchronize(d->stream));
  d->step = 0;
  d->wDirty = true;
  return ASH_OK;
}

int ash_denoiser_forward(ash_denoiser* d, uint32_t n, uint32_t h, uint32_t w, const float* input, float* out) {
  if (!d || !input || !out) return ASH_E_INVALID;
  DH(d, hipSetDevice(d->device));
  size_t P = size_t(n) * h * w;
  if (d->rgb.n < P * 3) DH(d, d->rgb.alloc(P * 3));
  Output o;
  o.rgb = d->rgb.p;
  int rc = uploadBatch(d, n, h, w, input, nullptr);
  if (!rc) rc = forwardPass(d, o);
  if (rc) return rc;
  DH(d, hipMemcpyAsync(out, d->rgb.p, P * 3 * sizeof(float), hipMemcpyDeviceToHost, d->stream));
  DH(d, hipStreamSynchronize(d->stream));
  return ASH_OK;
}

int ash_denoiser_gradient(ash_denoiser* d, uint32_t n, uint32_t h, uint32_t w, const float* input, const float* target,
                          float* loss, float* grad) {
  if (!d || !input || !target || !grad) return ASH_E_INVALID;
  DH(d, hipSetDevice(d->device));
  int rc = uploadBatch(d, n, h, w, input, target);
  if (!rc) rc = trainForward(d);
  if (!rc) rc = lossAndBackward(d, loss, nullptr);
  if (rc) return rc;
  return readReal(d, d->grad.p, grad);
}

int ash_denoiser_train_step(ash_denoiser* d, uint32_t n, uint32_t h, uint32_t w, const float* input,
                            const float* target, float lr, float* loss) {
  if (!d || !input || !target || !(lr > 0.f)) return ASH_E_INVALID;
  DH(d, hipSetDevice(d->device));
  int rc = uploadBatch(d, n, h, w, input, target);
  if (!rc) rc = trainForward(d);
  if (rc) return rc;
  const float b1 = 0.9f, b2 = 0.999f, step = float(d->step + 1);
  const AdamArgs adam{d->theta.p, d->m.p, d->v.p, lr, b1, b2, 1e-8f, 1.f - std::pow(b1, step), 1.f - std::pow(b2, step)};
  return lossAndBackward(d, loss, &adam);
}

}  // extern "C"

namespace ashd {
int denoisePlanesAsync(ash_denoiser* d, const void* radiance, const void* albedo, const void* normal,
                       const void* depth, uint32_t W, uint32_t H, void* out, hipEvent_t start, hipEvent_t done) {
  if (!d || !radiance || !out || !W || !H) return ASH_E_INVALID;
  DH(d, hipSetDevice(d->device));
  const uint32_t Hp = (H + 15) & ~15u, Wp = (W + 15) & ~15u;
  int rc = ensureShape(d, 1, Hp, Wp);
  if (rc) return rc;
  DH(d, hipEventRecord(start, d->stream));
  const FilmSrc film{static_cast<const float4*>(radiance), static_cast<const float4*>(albedo),
                     static_cast<const float4*>(normal), static_cast<const float4*>(depth), W, H};
  Output o;
  o.film = static_cast<float4*>(out);
  o.filmW = W, o.filmH = H;
  rc = forwardPass(d, o, &film);
  if (rc) return rc;
  DH(d, hipEventRecord(done, d->stream));
  return ASH_OK;
}
}  // namespace ashd

extern "C" {

int ash_denoise_planes(ash_denoiser* d, const void* radiance, const void* albedo, const void* normal,
                       const void* depth, uint32_t W, uint32_t H, void* out, double* ms) {
  if (!d || !radiance || !out || !W || !H) return ASH_E_INVALID;
  DH(d, hipSetDevice(d->device));
  hipEvent_t e0, e1;
  DH(d, hipEventCreate(&e0));
  DH(d, hipEventCreate(&e1));
  int rc = ashd::denoisePlanesAsync(d, radiance, albedo, normal, depth, W, H, out, e0, e1);
  if (rc) {
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
  }
  DH(d, hipEventSynchronize(e1));
  float t = 0;
  DH(d, hipEventElapsedTime(&t, e0, e1));
  if (ms) *ms = t;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return ASH_OK;
}

int ash_denoise_film(ash_denoiser* d, ash_ctx* ctx, int32_t albedoCh, int32_t normalCh, int32_t depthCh, int32_t outImage,
                     double* ms) {
  if (!d || !ctx || outImage < 0 || outImage >= ASH_NUM_OUTPUT_IMAGES) return ASH_E_INVALID;
  uint32_t W = 0, H = 0;
  ashd::ctxFilm(ctx, &W, &H);
  if (!W || !H) return dfail(d, ASH_E_STATE, "context has no film");
  auto plane = [&](int32_t ch) -> const void* {
    if (ch < 0 || ch >= ASH_NUM_OUTPUT_IMAGES - 1) return nullptr;
    void* p = nullptr;
    return ash_output_device_ptr(ctx, ch + 1, &p) == ASH_OK ? p : nullptr;
  };
  void* rad = nullptr;
  void* outp = nullptr;
  if (ash_output_device_ptr(ctx, 0, &rad) || ash_output_device_ptr(ctx, outImage, &outp))
    return dfail(d, ASH_E_STATE, "film planes unavailable");
  DH(d, hipSetDevice(d->device));
  // the denoiser works on its own stream after the context's pending renders
  hipEvent_t ready;
  DH(d, hipEventCreate(&ready));
  DH(d, hipEventRecord(ready, ashd::ctxStream(ctx)));
  DH(d, hipStreamWaitEvent(d->stream, ready, 0));
  int rc = ash_denoise_planes(d, rad, plane(albedoCh), plane(normalCh), plane(depthCh), W, H, outp, ms);
  (void)hipEventDestroy(ready);
  return rc;
}

}  // extern "C"
