// net.hip -- BF16 MFMA kernels of the learned preconditioner network (net.h).

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "device_common.h"
#include "net.h"

#define HG_CHECK(x)                                                                  \
  do {                                                                               \
    hipError_t e_ = (x);                                                             \
    if (e_ != hipSuccess) throw std::runtime_error(std::string("HIP: ") +            \
                                                   hipGetErrorString(e_) + " at " #x); \
  } while (0)

namespace hg {

namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));  // one lane's 16x16x32 operand
using bf = uint16_t;

__device__ __forceinline__ bool Done(const int* d) { return d && *d; }

// FP32 -> BF16, round to nearest even.
__device__ __forceinline__ bf F2B(float f) {
  unsigned u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return bf(0x7fc0);
  u += 0x7fffu + ((u >> 16) & 1u);
  return bf(u >> 16);
}
__device__ __forceinline__ float B2F(bf b) { return __uint_as_float(unsigned(b) << 16); }

__device__ __forceinline__ void Unpack8(const uint4 u, float f[8]) {
  const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    f[2 * k] = __uint_as_float(w[k] << 16);
    f[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
  }
}
__device__ __forceinline__ uint4 Pack8(const float f[8]) {
  unsigned w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) w[k] = unsigned(F2B(f[2 * k])) | (unsigned(F2B(f[2 * k + 1])) << 16);
  return uint4{w[0], w[1], w[2], w[3]};
}
__device__ __forceinline__ uint4 Ld8(const bf* p) { return *reinterpret_cast<const uint4*>(p); }
// 8 BF16 values (16 bytes, 16-byte aligned) as an MFMA operand
__device__ __forceinline__ b8 LdOp(const bf* p) { return __builtin_bit_cast(b8, Ld8(p)); }
__device__ __forceinline__ void St8(bf* p, uint4 v) { *reinterpret_cast<uint4*>(p) = v; }

// ---------------------------------------------------------------------------
// 3x3 'same' convolution, CIN, COUT multiples of 16, as an implicit GEMM on
// gfx950's MFMA 16x16x32 BF16 (FP32 accumulate).  A block of 4 waves
// computes a 16 SEG x 4 pixel tile (one row per wave) for all output channels.
// The input tile with its one-pixel halo is staged once in LDS (16-byte
// global loads and LDS stores; pixels padded to CIN + 8 channels, a 16-byte
// multiple, so every operand read is one aligned 16-byte LDS load).  The
// GEMM's K runs over (tap, input channel), k = tap * CIN + ci, 32 at a time:
// per chunk a wave multiplies each weight block (M = 16 output channels,
// read once and used SEG times) by SEG input blocks from LDS (N = 16
// pixels each); with CIN = 16 a chunk spans two taps, and the chunk past
// the ninth tap is zero.  Operand lane layouts (checked on the device):
// A[i][k] in lane i + 16*(k/8), element k%8 (8 consecutive channels of one
// tap: 16 contiguous bytes of wt[tap][co][ci]); B[k][j] in lane j +
// 16*(k/8), element k%8; D[i][j] in lane j + 16*(i/4), element i%4, so each
// lane ends with 4 consecutive output channels of one pixel and stores them
// as one 8-byte word.  Used for the forward pass and, with tap-flipped
// weights, for dgrad.
//
// SEG input blocks per wave (a tile is 16 SEG pixels wide): four use a weight
// block most often, but leave the coarse levels with fewer blocks than CUs;
// there a wave's weight loads, from L2 or memory once per chunk, are what takes
// the time, so they are issued kAhead chunks ahead and the tiles are narrower
// (64 -> 64 at 64 x 128 pixels: 17.0 us with 32 blocks of 64 x 4, 12.1 with 128
// of 16 x 4; 64 -> 32 at 128 x 256: 12.6 with 128, 10.1 with 256 of 32 x 4).
constexpr int kCTY = 4;           // tile height (one row per wave)
constexpr int kAhead = 4;

template <int CIN, int COUT, bool RELU, int SEG>
__global__ void __launch_bounds__(256)
KConvMfma(int W, int H, const bf* __restrict__ in, const bf* __restrict__ wt,
          bf* __restrict__ out, const int* done) {
  if (Done(done)) return;
  static_assert(CIN % 16 == 0 && COUT % 16 == 0, "channel counts");
  constexpr int CP = CIN + 8;  // padded channel stride in LDS (16-byte multiple)
  constexpr int kCTX = 16 * SEG, HX = kCTX + 2, HY = kCTY + 2;
  __shared__ __attribute__((aligned(16))) bf sin_[HY * HX * CP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles_x = (W + kCTX - 1) / kCTX;
  const int bx = blockIdx.x % tiles_x, by = blockIdx.x / tiles_x;
  const int x0 = bx * kCTX, y0 = by * kCTY;
  const int pj = lane & 15, kq = lane >> 4;
  constexpr int NQ = (9 * CIN + 31) / 32, NC = COUT / 16;  // K chunks, channel blocks
  const b8 zero = __builtin_bit_cast(b8, uint4{0u, 0u, 0u, 0u});
  // this lane's 8 values of chunk q: channels ci0..ci0+7 of tap t
  b8 bw[kAhead][NC];
  auto Weights = [&](int q) {
    const int kk = 32 * q + 8 * kq, t = kk / CIN, ci0 = kk % CIN;
#pragma unroll
    for (int n = 0; n < NC; ++n)
      bw[q % kAhead][n] = t < 9 ? LdOp(wt + size_t(t * COUT + n * 16 + pj) * CIN + ci0) : zero;
  };
#pragma unroll
  for (int q = 0; q < kAhead - 1; ++q) Weights(q);
  // stage the input tile + halo: 8 channels (16 bytes) per load
  constexpr int G = CIN / 8;
  for (int q = threadIdx.x; q < HX * HY * G; q += 256) {
    const int g = q % G, pix = q / G;
    const int hx = pix % HX, hy = pix / HX;
    const int xx = x0 + hx - 1, yy = y0 + hy - 1;
    uint4 v = uint4{0u, 0u, 0u, 0u};
    if (xx >= 0 && xx < W && yy >= 0 && yy < H) v = Ld8(in + (size_t(yy) * W + xx) * CIN + g * 8);
    St8(sin_ + pix * CP + g * 8, v);
  }
  __syncthreads();
  const int ty = y0 + wave;
  if (ty >= H) return;
  f4 acc[SEG][NC];
#pragma unroll
  for (int s = 0; s < SEG; ++s)
#pragma unroll
    for (int n = 0; n < NC; ++n) acc[s][n] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (q + kAhead - 1 < NQ) Weights(q + kAhead - 1);
    const int kk = 32 * q + 8 * kq;
    const int t = kk / CIN, ci0 = kk % CIN;
    const bool live = t < 9;
    const int hy = wave + t / 3;
#pragma unroll
    for (int s = 0; s < SEG; ++s) {
      const int hx = 16 * s + pj + t % 3;
      const b8 xin = live ? LdOp(sin_ + (hy * HX + hx) * CP + ci0) : zero;
#pragma unroll
      for (int n = 0; n < NC; ++n)
        acc[s][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[q % kAhead][n], xin, acc[s][n], 0,
                                                            0, 0);
    }
  }
#pragma unroll
  for (int s = 0; s < SEG; ++s) {
    const int px = x0 + 16 * s + pj;
    if (px >= W) continue;
#pragma unroll
    for (int n = 0; n < COUT / 16; ++n) {
      s4 o;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float r = acc[s][n][v];
        if (RELU) r = fmaxf(r, 0.f);
        o[v] = short(F2B(r));
      }
      *reinterpret_cast<s4*>(out + (size_t(ty) * W + px) * COUT + n * 16 + kq * 4) = o;
    }
  }
}

// Weight gradient dW[tap][ci][co] += sum_p in[p + off(tap)][ci] g[p][co]:
// per tap an implicit GEMM with M = 16 input channels, N = 16 output channels,
// K = pixels, 32 pixels per MFMA 16x16x32 BF16.  A block of 4 waves walks
// tiles of 64 x TR pixels: it stages the input tile with its one-pixel halo and
// the output gradients in LDS as they lie in memory (pixel by pixel, 16-byte
// loads and stores), once for all nine taps.  An operand -- 8 consecutive
// pixels of one channel per lane -- is two transposing LDS reads of 4 pixels x
// 16 channels per 16 lanes (ds_read_b64_tr_b16: lane i reads channels 4 (i % 4)
// .. of pixel i / 4, and gets channel i of the four pixels; checked on the
// device), so that a tap is an address offset.  Wave w holds all taps and output
// channels of input channels 16 (w % MW) .. and takes every KW-th 32 pixels.
// Each (block, pixel share) writes its sums to `part`, which KSumParts adds in
// order.
//
// What bounds it is latency: a tile's loads, a few hundred MFMAs per wave, and
// the partial sums' way through memory.  One tap and 16 input channels per
// block, with both operands transposed by 2-byte LDS stores, took (64 -> 64 at
// 64 x 128 pixels, 32 -> 64 at 128 x 256, 16 -> 32 at 256 x 512) 188, 114 and
// 75 us; this takes 14, 19 and 16, and KSumParts 5 more.
constexpr int kWgX = 64;            // tile width
constexpr int kWgHX = kWgX + 2;     // with halo
constexpr long kWgPartFloats = 4L << 20;  // of one layer's partial sums
template <int CIN, int COUT>
struct WgShape {
  static constexpr int MW = CIN / 16, KW = 4 / MW;
  static constexpr int CP = CIN + 8, GP = COUT + 8;  // pixel strides in LDS (16-byte multiples)
  static constexpr int Lds(int tr) { return (kWgHX * (tr + 2) * CP + kWgX * tr * GP) * 2; }
  static constexpr int TR = Lds(4) <= 65536 ? 4 : 2;  // tile height
  static_assert(CIN % 16 == 0 && COUT % 16 == 0 && 4 % MW == 0 && Lds(TR) <= 65536, "channels");
  // blocks for a W x H layer: one per tile up to 256 and to kWgPartFloats
  static int Blocks(int W, int H) {
    const long tiles = long((W + kWgX - 1) / kWgX) * ((H + TR - 1) / TR);
    return int(std::min({tiles, 256L, kWgPartFloats / (KW * 9L * CIN * COUT)}));
  }
};

template <int CIN, int COUT>
__global__ void __launch_bounds__(256)
KConvWgrad(int W, int H, int tiles_x, int tiles, const bf* __restrict__ in,
           const bf* __restrict__ g, float* __restrict__ part) {
  using S = WgShape<CIN, COUT>;
  constexpr int TR = S::TR, CP = S::CP, GP = S::GP, NC = COUT / 16;
  __shared__ __attribute__((aligned(16))) bf sin_[kWgHX * (TR + 2) * CP];
  __shared__ __attribute__((aligned(16))) bf sg[kWgX * TR * GP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int mt = wave % S::MW, kw = wave / S::MW;
  // this lane's pixel and channels of an operand's first transposing read
  const int px = 8 * (lane >> 4) + ((lane & 15) >> 2), ch = 4 * (lane & 3);
  auto Operand = [&](const bf* p, int stride) {
    using L4 = __attribute__((address_space(3))) s4;
    const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L4*)p);
    const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L4*)(p + 4 * stride));
    return __builtin_bit_cast(b8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  f4 acc[9][NC];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int n = 0; n < NC; ++n) acc[t][n] = f4{0.f, 0.f, 0.f, 0.f};
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const int x0 = tile % tiles_x * kWgX, y0 = tile / tiles_x * TR;
    constexpr int GI = CIN / 8, GO = COUT / 8;
    for (int q = threadIdx.x; q < kWgHX * (TR + 2) * GI; q += 256) {
      const int c8 = q % GI, p = q / GI;
      const int xx = x0 + p % kWgHX - 1, yy = y0 + p / kWgHX - 1;
      uint4 v = uint4{0u, 0u, 0u, 0u};
      if (xx >= 0 && xx < W && yy >= 0 && yy < H) v = Ld8(in + (size_t(yy) * W + xx) * CIN + c8 * 8);
      St8(sin_ + p * CP + c8 * 8, v);
    }
    for (int q = threadIdx.x; q < kWgX * TR * GO; q += 256) {
      const int c8 = q % GO, p = q / GO;
      const int xx = x0 + p % kWgX, yy = y0 + p / kWgX;
      uint4 v = uint4{0u, 0u, 0u, 0u};
      if (xx < W && yy < H) v = Ld8(g + (size_t(yy) * W + xx) * COUT + c8 * 8);
      St8(sg + p * GP + c8 * 8, v);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2 * TR / S::KW; ++k) {
      const int ks = k * S::KW + kw;  // 32 pixels of row ks / 2
      const int row = ks >> 1, col = (ks & 1) * 32 + px;
      b8 bg[NC];
#pragma unroll
      for (int n = 0; n < NC; ++n) bg[n] = Operand(sg + (row * kWgX + col) * GP + n * 16 + ch, GP);
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const b8 a =
            Operand(sin_ + ((row + t / 3) * kWgHX + col + t % 3) * CP + mt * 16 + ch, CP);
#pragma unroll
        for (int n = 0; n < NC; ++n)
          acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bg[n], acc[t][n], 0, 0, 0);
      }
    }
    __syncthreads();  // the tile's LDS is restaged next
  }
  // D[i][j]: i = 4 (lane / 16) + v (input channel), j = lane % 16 (output channel)
  float* const out = part + size_t(blockIdx.x * S::KW + kw) * (9 * CIN * COUT);
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        out[(t * CIN + mt * 16 + 4 * (lane >> 4) + v) * COUT + n * 16 + (lane & 15)] = acc[t][n][v];
}

// dw[i] += part[0][i] + part[1][i] + ... of np arrays of 4 n4 floats: a block
// sums 64 weights, 16 shares of the arrays side by side, the shares in order.
__global__ void __launch_bounds__(256)
KSumParts(int n4, int np, const float4* __restrict__ part, float4* __restrict__ dw) {
  __shared__ float4 red[16][16];
  const int l = threadIdx.x & 15, share = threadIdx.x >> 4;
  const int i = blockIdx.x * 16 + l;
  float4 s = {0.f, 0.f, 0.f, 0.f};
  if (i < n4) {
#pragma unroll 8
    for (int p = share; p < np; p += 16) {
      const float4 v = part[size_t(p) * n4 + i];
      s.x += v.x;
      s.y += v.y;
      s.z += v.z;
      s.w += v.w;
    }
  }
  red[share][l] = s;
  __syncthreads();
  if (share == 0 && i < n4) {
    float4 o = dw[i];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float4 v = red[k][l];
      o.x += v.x;
      o.y += v.y;
      o.z += v.z;
      o.w += v.w;
    }
    dw[i] = o;
  }
}

// E0: 1 -> 16 channels, FP32 input, ReLU, BF16 output; w[tap][co].
__global__ void __launch_bounds__(256)
KConvE0(int W, int H, const float* __restrict__ x, const float* __restrict__ w,
        bf* __restrict__ out, bool relu, const int* done) {
  if (Done(done)) return;
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= W * H) return;
  const int px = p % W, py = p / W;
  float acc[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) acc[c] = 0.f;
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int xx = px + t % 3 - 1, yy = py + t / 3 - 1;
    if (xx < 0 || xx >= W || yy < 0 || yy >= H) continue;
    const float v = x[yy * W + xx];
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[c] += v * w[t * 16 + c];
  }
  if (relu)
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[c] = fmaxf(acc[c], 0.f);
  St8(out + size_t(p) * 16, Pack8(acc));
  St8(out + size_t(p) * 16 + 8, Pack8(acc + 8));
}

// D0: 16 -> 1 channel, FP32 output y = base + conv(in); w[tap][ci].  y may
// alias base (each thread reads its base value before writing it).
__global__ void __launch_bounds__(256)
KConvD0(int W, int H, const bf* __restrict__ in, const float* __restrict__ w,
        const float* base, float* y, const int* done) {
  if (Done(done)) return;
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= W * H) return;
  const int px = p % W, py = p / W;
  float acc = 0.f;
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int xx = px + t % 3 - 1, yy = py + t / 3 - 1;
    if (xx < 0 || xx >= W || yy < 0 || yy >= H) continue;
    const bf* q = in + (size_t(yy) * W + xx) * 16;
    float f[16];
    Unpack8(Ld8(q), f);
    Unpack8(Ld8(q + 8), f + 8);
#pragma unroll
    for (int c = 0; c < 16; ++c) acc += f[c] * w[t * 16 + c];
  }
  y[p] = base ? base[p] + acc : acc;
}

// D0 dgrad: gin[p][ci] = sum_t gy[p - off(t)] w[t][ci].
__global__ void __launch_bounds__(256)
KConvD0Dgrad(int W, int H, const float* __restrict__ gy, const float* __restrict__ w,
             bf* __restrict__ gin) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= W * H) return;
  const int px = p % W, py = p / W;
  float acc[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) acc[c] = 0.f;
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int xx = px - (t % 3 - 1), yy = py - (t / 3 - 1);
    if (xx < 0 || xx >= W || yy < 0 || yy >= H) continue;
    const float g = gy[yy * W + xx];
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[c] += g * w[t * 16 + c];
  }
  St8(gin + size_t(p) * 16, Pack8(acc));
  St8(gin + size_t(p) * 16 + 8, Pack8(acc + 8));
}

// Weight gradients of the 1-channel ends, with s the 1-channel and f the
// 16-channel field:  E0: dw[t][co] += s[p + off(t)] f[p][co], f the gradient;
// D0: dw[t][ci] += f[p][ci] s[p - off(t)], s the gradient.  Each thread sums its
// pixels (f in two 16-byte loads), a wave its lanes, and each block writes its
// sums for KSumParts.  (16 threads that added 256 rows of LDS per tap, behind
// 16 two-byte loads per pixel, took 45 us at 512 x 1024; this takes 18.)
constexpr int kEndBlocks = 256;
template <bool E0>
__global__ void __launch_bounds__(256)
KEndWgrad(int W, int H, const float* __restrict__ s, const bf* __restrict__ f,
          float* __restrict__ part) {
  __shared__ float red[4][9 * 16];
  float acc[9][16];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[t][c] = 0.f;
  for (int p = blockIdx.x * 256 + threadIdx.x; p < W * H; p += gridDim.x * 256) {
    const int px = p % W, py = p / W;
    float v[16];
    Unpack8(Ld8(f + size_t(p) * 16), v);
    Unpack8(Ld8(f + size_t(p) * 16 + 8), v + 8);
    float a[9];
    bool in[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const int dx = t % 3 - 1, dy = t / 3 - 1;
      const int xx = E0 ? px + dx : px - dx, yy = E0 ? py + dy : py - dy;
      in[t] = xx >= 0 && xx < W && yy >= 0 && yy < H;
      a[t] = s[in[t] ? yy * W + xx : p];
    }
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      if (!in[t]) continue;
#pragma unroll
      for (int c = 0; c < 16; ++c) acc[t][c] += a[t] * v[c];
    }
  }
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const float w = DppSum<6>(acc[t][c]);
      if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6][t * 16 + c] = w;
    }
  __syncthreads();
  for (int q = threadIdx.x; q < 9 * 16; q += 256)
    part[blockIdx.x * (9 * 16) + q] = ((red[0][q] + red[1][q]) + red[2][q]) + red[3][q];
}

// ---- elementwise ops on BF16 NHWC tensors ----------------------------------
// Channel counts are multiples of 16: every thread moves groups of 8 channels
// (16 bytes).  Sums are formed in FP32 in a fixed order and rounded once.
__global__ void KPool(int W, int H, int C, const bf* __restrict__ in, bf* __restrict__ out,
                      const int* done) {
  if (Done(done)) return;
  const int Wc = W / 2, Hc = H / 2, G = C / 8;
  const long n = long(Wc) * Hc * G;
  for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L) {
    const int c = int(q % G) * 8;
    const long p = q / G;
    const int X = int(p % Wc), Y = int(p / Wc);
    const bf* b = in + (size_t(2 * Y) * W + 2 * X) * C + c;
    float f0[8], f1[8], f2[8], f3[8], o[8];
    Unpack8(Ld8(b), f0);
    Unpack8(Ld8(b + C), f1);
    Unpack8(Ld8(b + size_t(W) * C), f2);
    Unpack8(Ld8(b + size_t(W) * C + C), f3);
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = 0.25f * (f0[k] + f1[k] + f2[k] + f3[k]);
    St8(out + p * C + c, Pack8(o));
  }
}
// out = up(d) + e (fine grid W x H, C channels)
__global__ void KUpAdd(int W, int H, int C, const bf* __restrict__ d, const bf* __restrict__ e,
                       bf* __restrict__ out, const int* done) {
  if (Done(done)) return;
  const int Wc = W / 2, G = C / 8;
  const long n = long(W) * H * G;
  for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L) {
    const int c = int(q % G) * 8;
    const long p = q / G;
    const int x = int(p % W), y = int(p / W);
    float fd[8], fe[8], o[8];
    Unpack8(Ld8(d + (size_t(y / 2) * Wc + x / 2) * C + c), fd);
    Unpack8(Ld8(e + p * C + c), fe);
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = fd[k] + fe[k];
    St8(out + p * C + c, Pack8(o));
  }
}
// g_coarse = sum of the four children of g_fine
__global__ void KUpBwd(int Wc, int Hc, int C, const bf* __restrict__ gf, bf* __restrict__ gc) {
  const int W = 2 * Wc, G = C / 8;
  const long n = long(Wc) * Hc * G;
  for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L) {
    const int c = int(q % G) * 8;
    const long p = q / G;
    const int X = int(p % Wc), Y = int(p / Wc);
    const bf* b = gf + (size_t(2 * Y) * W + 2 * X) * C + c;
    float f0[8], f1[8], f2[8], f3[8], o[8];
    Unpack8(Ld8(b), f0);
    Unpack8(Ld8(b + C), f1);
    Unpack8(Ld8(b + size_t(W) * C), f2);
    Unpack8(Ld8(b + size_t(W) * C + C), f3);
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = f0[k] + f1[k] + f2[k] + f3[k];
    St8(gc + p * C + c, Pack8(o));
  }
}
// g_fine (+)= 0.25 * g_coarse at each child
__global__ void KPoolBwdAdd(int W, int H, int C, const bf* __restrict__ gc, bf* __restrict__ gf) {
  const int Wc = W / 2, G = C / 8;
  const long n = long(W) * H * G;
  for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L) {
    const int c = int(q % G) * 8;
    const long p = q / G;
    const int x = int(p % W), y = int(p / W);
    float ff[8], fc[8], o[8];
    Unpack8(Ld8(gf + p * C + c), ff);
    Unpack8(Ld8(gc + (size_t(y / 2) * Wc + x / 2) * C + c), fc);
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = ff[k] + 0.25f * fc[k];
    St8(gf + p * C + c, Pack8(o));
  }
}
// out = g * (act > 0); n is a multiple of 8
__global__ void KMask(long n, const bf* __restrict__ g, const bf* __restrict__ act,
                      bf* __restrict__ out) {
  for (long q = blockIdx.x * 256L + threadIdx.x; q < n / 8; q += gridDim.x * 256L) {
    const uint4 gv = Ld8(g + q * 8), av = Ld8(act + q * 8);
    const unsigned gw[4] = {gv.x, gv.y, gv.z, gv.w}, aw[4] = {av.x, av.y, av.z, av.w};
    unsigned ow[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const unsigned lo = __uint_as_float(aw[k] << 16) > 0.f ? (gw[k] & 0xffffu) : 0u;
      const unsigned hi = __uint_as_float(aw[k] & 0xffff0000u) > 0.f ? (gw[k] & 0xffff0000u) : 0u;
      ow[k] = lo | hi;
    }
    St8(out + q * 8, uint4{ow[0], ow[1], ow[2], ow[3]});
  }
}

// loss = mean((y - t)^2) (partials), gy = 2 (y - t) / N
__global__ void __launch_bounds__(256)
KLoss(long n, const float* __restrict__ y, const float* __restrict__ t, float* __restrict__ gy,
      double* __restrict__ part) {
  double s = 0.;
  for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L) {
    const float d = y[q] - t[q];
    gy[q] = 2.f * d / float(n);
    s += double(d) * double(d);
  }
  s = WaveSum(s);
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// Energy-norm loss: d = o*y - t (o: optional per-cell output scale), q = A d
// (face-form operator, FP32 coefficients kx[(nx+1)*ny], ky[nx*(ny+1)]);
// loss = d.q / n (partials), gy = o * 2 q / n.
__global__ void KDiff(long n, float* __restrict__ y, const float* __restrict__ t,
                      const float* __restrict__ o) {
  for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L)
    y[q] = (o ? o[q] * y[q] : y[q]) - t[q];
}

__global__ void __launch_bounds__(256)
KEnergyLoss(int nx, int ny, const float* __restrict__ kx, const float* __restrict__ ky,
            const float* __restrict__ d, const float* __restrict__ o, float* __restrict__ gy,
            double* __restrict__ part) {
  const long n = long(nx) * ny;
  double s = 0.;
  for (long c = blockIdx.x * 256L + threadIdx.x; c < n; c += gridDim.x * 256L) {
    const int i = int(c % nx), j = int(c / nx);
    const float kw = kx[i + long(nx + 1) * j], ke = kx[i + 1 + long(nx + 1) * j];
    const float ks = ky[i + long(nx) * j], kn = ky[i + long(nx) * (j + 1)];
    float q = (((kw + ke) + ks) + kn) * d[c];
    if (i > 0) q -= kw * d[c - 1];
    if (i < nx - 1) q -= ke * d[c + 1];
    if (j > 0) q -= ks * d[c - nx];
    if (j < ny - 1) q -= kn * d[c + nx];
    gy[c] = (o ? o[c] : 1.f) * (2.f * q / float(n));
    s += double(d[c]) * double(q);
  }
  s = WaveSum(s);
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

__global__ void KAdam(int n, float* __restrict__ w, const float* __restrict__ g,
                      float* __restrict__ m, float* __restrict__ v, float lr, float b1, float b2,
                      float c1, float c2) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  const float gg = g[q];
  const float mm = b1 * m[q] + (1.f - b1) * gg;
  const float vv = b2 * v[q] + (1.f - b2) * gg * gg;
  m[q] = mm;
  v[q] = vv;
  w[q] -= lr * (mm / c1) / (sqrtf(vv / c2) + 1e-8f);
}

// Scale-free energy loss: u = o*y, c = u.(A t), Y = u.(A u), T = t.(A t)
// (per-block partials part[3b..3b+2]; qu = A u and qt = A t kept).
__global__ void __launch_bounds__(256)
KCosDots(int nx, int ny, const float* __restrict__ kx, const float* __restrict__ ky,
         const float* __restrict__ y, const float* __restrict__ o, const float* __restrict__ t,
         float* __restrict__ qu, float* __restrict__ qt, double* __restrict__ part) {
  const long n = long(nx) * ny;
  double sc = 0., sy = 0., st = 0.;
  auto U = [&](long c) { return o ? o[c] * y[c] : y[c]; };
  for (long c = blockIdx.x * 256L + threadIdx.x; c < n; c += gridDim.x * 256L) {
    const int i = int(c % nx), j = int(c / nx);
    const float kw = kx[i + long(nx + 1) * j], ke = kx[i + 1 + long(nx + 1) * j];
    const float ks = ky[i + long(nx) * j], kn = ky[i + long(nx) * (j + 1)];
    const float dg = ((kw + ke) + ks) + kn;
    const float uc = U(c), tc = t[c];
    float au = dg * uc, at = dg * tc;
    if (i > 0) au -= kw * U(c - 1), at -= kw * t[c - 1];
    if (i < nx - 1) au -= ke * U(c + 1), at -= ke * t[c + 1];
    if (j > 0) au -= ks * U(c - nx), at -= ks * t[c - nx];
    if (j < ny - 1) au -= kn * U(c + nx), at -= kn * t[c + nx];
    qu[c] = au;
    qt[c] = at;
    sc += double(uc) * at;
    sy += double(uc) * au;
    st += double(tc) * at;
  }
  sc = WaveSum(sc);
  sy = WaveSum(sy);
  st = WaveSum(st);
  __shared__ double red[3][4];
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = sc;
    red[1][threadIdx.x >> 6] = sy;
    red[2][threadIdx.x >> 6] = st;
  }
  __syncthreads();
  if (threadIdx.x < 3)
    part[3 * blockIdx.x + threadIdx.x] =
        red[threadIdx.x][0] + red[threadIdx.x][1] + red[threadIdx.x][2] + red[threadIdx.x][3];
}

// Gradient of L = 1 - c^2 / (Y T) (one minus the squared energy-cosine of u
// and t, i.e. the relative energy error of the best multiple alpha = c/Y of
// u): dL/du = (2 c / (Y T)) (alpha A u - A t); gy = o * dL/du.  Every block
// folds the partials in the same order; block 0 stores (L, alpha) in stat.
__global__ void __launch_bounds__(256)
KCosGrad(long n, int nb, const double* __restrict__ part, const float* __restrict__ o,
         const float* __restrict__ qu, const float* __restrict__ qt, float* __restrict__ gy,
         double* __restrict__ stat) {
  __shared__ double red[3][4];
  double a[3] = {0., 0., 0.};
  for (int b = threadIdx.x; b < nb; b += 256)
    for (int k = 0; k < 3; ++k) a[k] += part[3 * b + k];
  for (int k = 0; k < 3; ++k) {
    const double v = WaveSum(a[k]);
    if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = v;
  }
  __syncthreads();
  const double c = red[0][0] + red[0][1] + red[0][2] + red[0][3];
  const double Y = red[1][0] + red[1][1] + red[1][2] + red[1][3];
  const double T = red[2][0] + red[2][1] + red[2][2] + red[2][3];
  const bool ok = Y > 0. && T > 0.;
  const double alpha = ok ? c / Y : 0.;
  const float f = ok ? float(2. * c / (Y * T)) : 0.f, al = float(alpha);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    stat[0] = ok ? 1. - c * c / (Y * T) : 1.;
    stat[1] = alpha;
  }
  for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L)
    gy[q] = (o ? o[q] : 1.f) * (f * (al * qu[q] - qt[q]));
}

// w[0..n) *= a
__global__ void KScaleW(int n, float* __restrict__ w, float a) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q < n) w[q] *= a;
}

// Tied decoder of the first layer: wd0[t][c] = wE0[8 - t][c].
__global__ void KFlipE0(const float* __restrict__ w, float* __restrict__ wd0) {
  const int q = threadIdx.x;
  if (q < 144) wd0[q] = w[(8 - q / 16) * 16 + q % 16];
}

// Gradient of a tied decoder layer (layout [t][a][b], a < cout, b < cin of
// the encoder layer it mirrors) added to the encoder layer's gradient
// gE[8 - t][b][a].
__global__ void KFoldTied(int cin, int cout, const float* __restrict__ gd, float* __restrict__ ge) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= 9 * cin * cout) return;
  const int t = q / (cin * cout), r = q % (cin * cout), a = r / cin, b = r % cin;
  ge[(size_t(8 - t) * cin + b) * cout + a] += gd[q];
}

// Master W[tap][ci][co] -> forward wf[tap][co][ci] and dgrad
// wb[tap][ci][co] = W[8 - tap][ci][co] (BF16).
__global__ void KConvertW(int cin, int cout, const float* __restrict__ w, bf* __restrict__ wf,
                          bf* __restrict__ wb) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  const int n = 9 * cin * cout;
  if (q >= n) return;
  const int t = q / (cin * cout), r = q % (cin * cout), ci = r / cout, co = r % cout;
  const bf v = F2B(w[q]);
  wf[(size_t(t) * cout + co) * cin + ci] = v;
  wb[(size_t(8 - t) * cin + ci) * cout + co] = v;
}

inline unsigned Blk(long n) { return unsigned(std::min<long>((n + 255) / 256, 65535)); }

// Dispatch of the MFMA conv for the (cin, cout) pairs of the network.
void ConvFwd(int cin, int cout, bool relu, int W, int H, const bf* in, const bf* wt, bf* out,
             hipStream_t st, const int* done) {
  auto blocks = [&](int seg) { return ((W + 16 * seg - 1) / (16 * seg)) * ((H + kCTY - 1) / kCTY); };
  // at least a block per CU, if the grid has them (figures at KConvMfma)
  const int seg = blocks(4) >= 256 ? 4 : blocks(2) >= 256 ? 2 : 1;
  const unsigned grid = unsigned(blocks(seg));
  auto launch = [&](auto k4, auto k2, auto k1) {
    (seg == 4 ? k4 : seg == 2 ? k2 : k1)<<<grid, 256, 0, st>>>(W, H, in, wt, out, done);
  };
#define HG_CONV(CI, CO)                                                                  \
  if (cin == CI && cout == CO) {                                                         \
    if (relu)                                                                            \
      launch(KConvMfma<CI, CO, true, 4>, KConvMfma<CI, CO, true, 2>,                     \
             KConvMfma<CI, CO, true, 1>);                                                \
    else                                                                                 \
      launch(KConvMfma<CI, CO, false, 4>, KConvMfma<CI, CO, false, 2>,                   \
             KConvMfma<CI, CO, false, 1>);                                               \
    return;                                                                              \
  }
  HG_CONV(16, 32) HG_CONV(32, 64) HG_CONV(64, 64) HG_CONV(64, 32) HG_CONV(32, 16)
  HG_CONV(16, 16) HG_CONV(32, 32) HG_CONV(16, 64) HG_CONV(64, 16)
#undef HG_CONV
  throw std::runtime_error("no MFMA conv for this channel pair");
}

// the channel pairs of the weight gradient
#define HG_WG_PAIRS                                                                      \
  HG_WG(16, 32) HG_WG(32, 64) HG_WG(64, 64) HG_WG(64, 32) HG_WG(32, 16)                  \
  HG_WG(16, 16) HG_WG(32, 32) HG_WG(16, 64) HG_WG(64, 16)

void SumParts(int n, int np, const float* part, float* dw, hipStream_t st) {
  KSumParts<<<unsigned((n / 4 + 15) / 16), 256, 0, st>>>(
      n / 4, np, reinterpret_cast<const float4*>(part), reinterpret_cast<float4*>(dw));
}

// dw += the weight gradient; part: WgradPartFloats(cin, cout, W, H) floats.
void ConvWgrad(int cin, int cout, int W, int H, const bf* in, const bf* g, float* part,
               float* dw, hipStream_t st) {
#define HG_WG(CI, CO)                                                                     \
  if (cin == CI && cout == CO) {                                                          \
    using S = WgShape<CI, CO>;                                                            \
    const int tx = (W + kWgX - 1) / kWgX, tiles = tx * ((H + S::TR - 1) / S::TR);         \
    const int nb = S::Blocks(W, H);                                                       \
    KConvWgrad<CI, CO><<<unsigned(nb), 256, 0, st>>>(W, H, tx, tiles, in, g, part);       \
    SumParts(9 * CI * CO, nb * S::KW, part, dw, st);                                      \
    return;                                                                               \
  }
  HG_WG_PAIRS
#undef HG_WG
  throw std::runtime_error("no MFMA wgrad for this channel pair");
}

long WgradPartFloats(int cin, int cout, int W, int H) {
#define HG_WG(CI, CO)                                                                     \
  if (cin == CI && cout == CO) {                                                          \
    using S = WgShape<CI, CO>;                                                            \
    return long(S::Blocks(W, H)) * S::KW * 9 * CI * CO;                                   \
  }
  HG_WG_PAIRS
#undef HG_WG
  return 0;
}

}  // namespace

// ---------------------------------------------------------------------------

UNet::UNet(int nx, int ny) : nx_(nx), ny_(ny) {
  if (!Supported(nx, ny)) throw std::runtime_error("UNet: grid dimensions must be multiples of 8");
  for (int l = 0; l < kLevels; ++l) {
    lw_[l] = nx >> l;
    lh_[l] = ny >> l;
    ch_[l] = std::min(16 << l, 64);
  }
  ch_[kLevels - 1] = ch_[kLevels - 2];
  int off = 0, k = 0;
  layer_[k++] = {off, 1, ch_[0], 0};
  off += 9 * 1 * ch_[0];
  for (int l = 1; l < kLevels; ++l) {
    layer_[k++] = {off, ch_[l - 1], ch_[l], l};
    off += 9 * ch_[l - 1] * ch_[l];
  }
  for (int l = kLevels - 1; l >= 1; --l) {
    layer_[k++] = {off, ch_[l], ch_[l - 1], l};
    off += 9 * ch_[l] * ch_[l - 1];
  }
  layer_[k++] = {off, ch_[0], 1, 0};
  off += 9 * ch_[0];
  nw_ = off;
  auto A = [](void** p, size_t bytes) {
    HG_CHECK(hipMalloc(p, std::max<size_t>(bytes, 16)));
    HG_CHECK(hipMemset(*p, 0, std::max<size_t>(bytes, 16)));
  };
  A((void**)&w_, size_t(nw_) * 4);
  A((void**)&g_, size_t(nw_) * 4);
  A((void**)&m_, size_t(nw_) * 4);
  A((void**)&v_, size_t(nw_) * 4);
  A((void**)&wf_, size_t(nw_) * 2);
  A((void**)&wb_, size_t(nw_) * 2);
  A((void**)&wd0_, 9 * 16 * 4);
  A((void**)&gtie_, size_t(9) * 64 * 64 * 4);
  for (int l = 0; l < kLevels; ++l) {
    const size_t px = size_t(lw_[l]) * lh_[l];
    A((void**)&enc_[l], px * ch_[l] * 2);
    A((void**)&genc_[l], px * ch_[l] * 2);
    A((void**)&gin_[l], px * 64 * 2);
    A((void**)&gpre_[l], px * 64 * 2);
    if (l > 0) {
      A((void**)&pin_[l], px * ch_[l - 1] * 2);
      A((void**)&dout_[l], px * ch_[l - 1] * 2);
      A((void**)&gtmp_[l], px * ch_[l - 1] * 2);
    }
    if (l < kLevels - 1) A((void**)&din_[l], px * ch_[l] * 2);
  }
  A((void**)&yb_, size_t(nx) * ny * 4);
  A((void**)&qu_, size_t(nx) * ny * 4);
  A((void**)&qt_, size_t(nx) * ny * 4);
  A((void**)&gy_, size_t(nx) * ny * 4);
  A((void**)&part_, 65536 * 8);
  long np = kEndBlocks * 9 * 16;
  for (const Layer& L : layer_)
    np = std::max(np, WgradPartFloats(L.cin, L.cout, lw_[L.level], lh_[L.level]));
  A((void**)&wpart_, size_t(np) * 4);
  HG_CHECK(hipHostMalloc((void**)&loss_h_, 65536 * 8));
}

UNet::~UNet() {
  std::vector<void*> ps = {w_, g_, m_, v_, wf_, wb_, wd0_, gtie_, yb_, qu_, qt_, gy_, part_, wpart_};
  for (int l = 0; l < kLevels; ++l)
    for (void* p : {(void*)enc_[l], (void*)genc_[l], (void*)gin_[l], (void*)gpre_[l],
                    (void*)pin_[l], (void*)dout_[l], (void*)gtmp_[l], (void*)din_[l]})
      ps.push_back(p);
  for (void* p : ps)
    if (p) (void)hipFree(p);
  if (loss_h_) (void)hipHostFree(loss_h_);
}

void UNet::ConvertWeights(hipStream_t st) {
  for (const Layer& L : layer_) {
    const int n = 9 * L.cin * L.cout;
    KConvertW<<<Blk(n), 256, 0, st>>>(L.cin, L.cout, w_ + L.off, wf_ + L.off, wb_ + L.off);
  }
  KFlipE0<<<1, 256, 0, st>>>(w_ + layer_[0].off, wd0_);
}

void UNet::SetWeights(const float* host, hipStream_t st) {
  HG_CHECK(hipMemcpyAsync(w_, host, size_t(nw_) * 4, hipMemcpyHostToDevice, st));
  HG_CHECK(hipMemsetAsync(m_, 0, size_t(nw_) * 4, st));
  HG_CHECK(hipMemsetAsync(v_, 0, size_t(nw_) * 4, st));
  adam_t_ = 0;
  ConvertWeights(st);
  HG_CHECK(hipStreamSynchronize(st));
}

void UNet::GetWeights(float* host, hipStream_t st) {
  HG_CHECK(hipMemcpyAsync(host, w_, size_t(nw_) * 4, hipMemcpyDeviceToHost, st));
  HG_CHECK(hipStreamSynchronize(st));
}

void UNet::InitWeights(uint64_t seed, hipStream_t st) {
  std::mt19937_64 rng(seed);
  std::vector<float> w(nw_, 0.f);
  for (int k = 0; k < 2 * kLevels; ++k) {
    const Layer& L = layer_[k];
    const bool last = (k == 2 * kLevels - 1);
    std::normal_distribution<float> nd(0.f, std::sqrt(2.f / (9.f * L.cin)));
    for (int q = 0; q < 9 * L.cin * L.cout; ++q) w[L.off + q] = last ? 0.f : nd(rng);
  }
  SetWeights(w.data(), st);
}

void UNet::Forward(const float* x, float* y, const float* base, hipStream_t st, const int* done) {
  // encoder
  const bool relu = !linear_;
  KConvE0<<<Blk(long(lw_[0]) * lh_[0]), 256, 0, st>>>(lw_[0], lh_[0], x, w_ + layer_[0].off,
                                                      enc_[0], relu, done);
  for (int l = 1; l < kLevels; ++l) {
    const int W = lw_[l], H = lh_[l];
    KPool<<<Blk(long(W) * H * ch_[l - 1]), 256, 0, st>>>(lw_[l - 1], lh_[l - 1], ch_[l - 1],
                                                        enc_[l - 1], pin_[l], done);
    const Layer& L = layer_[l];
    ConvFwd(L.cin, L.cout, relu, W, H, pin_[l], wf_ + L.off, enc_[l], st, done);
  }
  // decoder: D3 on enc3, then up + skip + conv down to level 1; tied
  // decoder layers are the transposes of the encoder layers (the encoder's
  // dgrad-form weights)
  for (int l = kLevels - 1; l >= 1; --l) {
    const Layer& L = layer_[kLevels + (kLevels - 1 - l)];
    const int W = lw_[l], H = lh_[l];
    const bf* src = (l == kLevels - 1) ? enc_[l] : din_[l];
    if (l < kLevels - 1)
      KUpAdd<<<Blk(long(W) * H * ch_[l]), 256, 0, st>>>(W, H, ch_[l], dout_[l + 1], enc_[l],
                                                        din_[l], done);
    const bf* wt = tied_ ? wb_ + layer_[l].off : wf_ + L.off;
    ConvFwd(L.cin, L.cout, relu, W, H, src, wt, dout_[l], st, done);
  }
  KUpAdd<<<Blk(long(lw_[0]) * lh_[0] * ch_[0]), 256, 0, st>>>(lw_[0], lh_[0], ch_[0], dout_[1],
                                                              enc_[0], din_[0], done);
  KConvD0<<<Blk(long(lw_[0]) * lh_[0]), 256, 0, st>>>(lw_[0], lh_[0], din_[0], D0Weights(), base,
                                                      y, done);
}

const float* UNet::D0Weights() const {
  return tied_ ? wd0_ : w_ + layer_[2 * kLevels - 1].off;
}

void UNet::ZeroGrad(hipStream_t st) { HG_CHECK(hipMemsetAsync(g_, 0, size_t(nw_) * 4, st)); }

void UNet::GetGrad(float* host, hipStream_t st) {
  HG_CHECK(hipMemcpyAsync(host, g_, size_t(nw_) * 4, hipMemcpyDeviceToHost, st));
  HG_CHECK(hipStreamSynchronize(st));
}

void UNet::Backward(const float* x, const float* gy, hipStream_t st) {
  const int W0 = lw_[0], H0 = lh_[0];
  const long n0 = long(W0) * H0;
  // D0: dgrad into gin0 (grad of din0), wgrad
  const Layer& D0 = layer_[2 * kLevels - 1];
  KConvD0Dgrad<<<Blk(n0), 256, 0, st>>>(W0, H0, gy, D0Weights(), gin_[0]);
  if (tied_) {
    HG_CHECK(hipMemsetAsync(gtie_, 0, 9 * 16 * 4, st));
    KEndWgrad<false><<<kEndBlocks, 256, 0, st>>>(W0, H0, gy, din_[0], wpart_);
    SumParts(9 * 16, kEndBlocks, wpart_, gtie_, st);
    KFoldTied<<<1, 256, 0, st>>>(1, ch_[0], gtie_, g_ + layer_[0].off);
  } else {
    KEndWgrad<false><<<kEndBlocks, 256, 0, st>>>(W0, H0, gy, din_[0], wpart_);
    SumParts(9 * 16, kEndBlocks, wpart_, g_ + D0.off, st);
  }
  // din0 = up(dout1) + enc0: grad to enc0 and (summed over children) to dout1
  HG_CHECK(hipMemcpyAsync(genc_[0], gin_[0], size_t(n0) * ch_[0] * 2, hipMemcpyDeviceToDevice, st));
  KUpBwd<<<Blk(long(lw_[1]) * lh_[1] * ch_[0]), 256, 0, st>>>(lw_[1], lh_[1], ch_[0], gin_[0],
                                                              gtmp_[1]);
  // decoder D1 .. D_{L-1}
  for (int l = 1; l < kLevels; ++l) {
    const Layer& L = layer_[kLevels + (kLevels - 1 - l)];
    const int W = lw_[l], H = lh_[l];
    const long np = long(W) * H;
    const bf* gp = gtmp_[l];
    if (!linear_) {
      KMask<<<Blk(np * L.cout), 256, 0, st>>>(np * L.cout, gtmp_[l], dout_[l], gpre_[l]);
      gp = gpre_[l];
    }
    const bf* src = (l == kLevels - 1) ? enc_[l] : din_[l];
    if (tied_) {
      const Layer& E = layer_[l];
      HG_CHECK(hipMemsetAsync(gtie_, 0, size_t(9) * E.cin * E.cout * 4, st));
      ConvWgrad(L.cin, L.cout, W, H, src, gp, wpart_, gtie_, st);
      KFoldTied<<<Blk(9L * E.cin * E.cout), 256, 0, st>>>(E.cin, E.cout, gtie_, g_ + E.off);
      ConvFwd(L.cout, L.cin, false, W, H, gp, wf_ + E.off, gin_[l], st, nullptr);
    } else {
      ConvWgrad(L.cin, L.cout, W, H, src, gp, wpart_, g_ + L.off, st);
      ConvFwd(L.cout, L.cin, false, W, H, gp, wb_ + L.off, gin_[l], st, nullptr);
    }
    HG_CHECK(hipMemcpyAsync(genc_[l], gin_[l], size_t(np) * ch_[l] * 2, hipMemcpyDeviceToDevice,
                            st));
    if (l < kLevels - 1)
      KUpBwd<<<Blk(long(lw_[l + 1]) * lh_[l + 1] * ch_[l]), 256, 0, st>>>(
          lw_[l + 1], lh_[l + 1], ch_[l], gin_[l], gtmp_[l + 1]);
  }
  // encoder from the top
  for (int l = kLevels - 1; l >= 1; --l) {
    const Layer& L = layer_[l];
    const int W = lw_[l], H = lh_[l];
    const long np = long(W) * H;
    const bf* gp = genc_[l];
    if (!linear_) {
      KMask<<<Blk(np * L.cout), 256, 0, st>>>(np * L.cout, genc_[l], enc_[l], gpre_[l]);
      gp = gpre_[l];
    }
    ConvWgrad(L.cin, L.cout, W, H, pin_[l], gp, wpart_, g_ + L.off, st);
    ConvFwd(L.cout, L.cin, false, W, H, gp, wb_ + L.off, gin_[l], st, nullptr);
    KPoolBwdAdd<<<Blk(long(lw_[l - 1]) * lh_[l - 1] * ch_[l - 1]), 256, 0, st>>>(
        lw_[l - 1], lh_[l - 1], ch_[l - 1], gin_[l], genc_[l - 1]);
  }
  const bf* gp0 = genc_[0];
  if (!linear_) {
    KMask<<<Blk(n0 * ch_[0]), 256, 0, st>>>(n0 * ch_[0], genc_[0], enc_[0], gpre_[0]);
    gp0 = gpre_[0];
  }
  KEndWgrad<true><<<kEndBlocks, 256, 0, st>>>(W0, H0, x, gp0, wpart_);
  SumParts(9 * 16, kEndBlocks, wpart_, g_ + layer_[0].off, st);
}

void UNet::AdamStep(float lr, hipStream_t st) {
  ++adam_t_;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, float(adam_t_)), c2 = 1.f - std::pow(b2, float(adam_t_));
  KAdam<<<Blk(nw_), 256, 0, st>>>(nw_, w_, g_, m_, v_, lr, b1, b2, c1, c2);
  ConvertWeights(st);
}

void UNet::TrainStep(const float* x, const float* target, float lr, hipStream_t st,
                     double* loss) {
  Forward(x, yb_, nullptr, st, nullptr);
  const long n = long(nx_) * ny_;
  const int nb = 1024;
  if (mkx_ && scale_free_) {
    KCosDots<<<nb, 256, 0, st>>>(nx_, ny_, mkx_, mky_, yb_, oscale_, target, qu_, qt_, part_);
    KCosGrad<<<nb, 256, 0, st>>>(n, nb, part_, oscale_, qu_, qt_, gy_, part_ + 3 * nb);
    if (loss) HG_CHECK(hipMemcpyAsync(loss_h_, part_ + 3 * nb, 16, hipMemcpyDeviceToHost, st));
  } else {
    if (mkx_) {
      KDiff<<<nb, 256, 0, st>>>(n, yb_, target, oscale_);
      KEnergyLoss<<<nb, 256, 0, st>>>(nx_, ny_, mkx_, mky_, yb_, oscale_, gy_, part_);
    } else {
      KLoss<<<nb, 256, 0, st>>>(n, yb_, target, gy_, part_);
    }
    if (loss) HG_CHECK(hipMemcpyAsync(loss_h_, part_, nb * 8, hipMemcpyDeviceToHost, st));
  }
  ZeroGrad(st);
  Backward(x, gy_, st);
  AdamStep(lr, st);
  if (loss) {
    HG_CHECK(hipStreamSynchronize(st));
    if (mkx_ && scale_free_) {
      *loss = loss_h_[0];
      last_alpha_ = loss_h_[1];
    } else {
      double s = 0.;
      for (int b = 0; b < nb; ++b) s += loss_h_[b];
      *loss = s / double(n);
    }
  }
}

void UNet::ScaleOutput(float a, hipStream_t st) {
  if (!(a > 0.f)) throw std::runtime_error("UNet::ScaleOutput: factor must be positive");
  // the tied network is quadratic in the first layer, the untied one linear
  // in the last
  const Layer& L = tied_ ? layer_[0] : layer_[2 * kLevels - 1];
  const int n = 9 * L.cin * L.cout;
  KScaleW<<<Blk(n), 256, 0, st>>>(n, w_ + L.off, tied_ ? std::sqrt(a) : a);
  ConvertWeights(st);
}

double UNet::ForwardFlops() const {
  double f = 0.;
  for (const Layer& L : layer_)
    f += 18. * L.cin * L.cout * double(lw_[L.level]) * lh_[L.level];
  return f;
}

double UNet::MfmaForwardFlops() const {
  double f = 0.;
  for (const Layer& L : layer_)
    if (L.cin % 16 == 0 && L.cout % 16 == 0)
      f += 18. * L.cin * L.cout * double(lw_[L.level]) * lh_[L.level];
  return f;
}

// forward + weight gradients of every layer + input gradients of every
// layer but the first
double UNet::TrainFlops() const {
  double f = 2. * ForwardFlops();
  const Layer& E0 = layer_[0];
  f += ForwardFlops() - 18. * E0.cin * E0.cout * double(lw_[0]) * lh_[0];
  return f;
}

}  // namespace hg
