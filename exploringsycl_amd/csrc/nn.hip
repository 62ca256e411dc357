// libteahip.so: the learned preconditioner's network (no counterpart in the
// reference).  Six 3x3 convolutions, 32 hidden channels, ReLU after the
// first five; inputs (residual, kx feature, ky feature), one output channel.
// 38,177 parameters, FP32 master copy; BF16 weights and activations with
// FP32 accumulation on the MFMA units (v_mfma_f32_32x32x16_bf16).
//
// Tensors are NHWC with a one-pixel zero border: [B][H+2][W+2][C], C = 8
// for the input (3 used) and 32 for hidden activations, so a pixel's 8 or
// 32 channels are one or four 16-byte vectors.  W must be a multiple of 32.
//
// A 32->32 convolution is an implicit GEMM per row tile of 32 pixels:
// D[co][pixel] = sum over k = (tap, ci) of Wt[co][k] * In[pixel + tap][ci],
// K = 9*32 = 288 = 18 MFMA steps of 16.  A (32 x 16) is the weights (lane l:
// co = l%32, k = step slice + 8*(l/32) + 0..7), B (16 x 32) the input patch
// (lane l: pixel l%32, same k), D (32 x 32): lane l holds pixel l%32 and
// channels 8*(v/4) + 4*(l/32) + v%4 for v = 0..15 (layout checked on the
// device).  The backward-data pass is the same kernel with the weights
// flipped and transposed, times the ReLU mask of the layer's input.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "tea_hip_impl.h"

namespace tea {
namespace nn {

constexpr int kC = 32;   // hidden channels
constexpr int kC0 = 8;   // input channels in memory (3 used)
constexpr int kIn = 3;   // real input channels
constexpr int kTaps = 9;
constexpr int kFwdRows = 4;  // output rows per block of the multi-row forward kernel

// FP32 master parameters, in the order W1 (32,3,3,3), b1 (32), W2..W5
// (32,32,3,3) with b2..b5 (32), W6 (1,32,3,3), b6 (1); W[co][ci][ky][kx].
constexpr int kW1 = kC * kIn * kTaps;  // 864
constexpr int kWh = kC * kC * kTaps;   // 9216
constexpr int kWf1 = 5 * 64 * 8;       // layer 1 in fragment order, taps and channels padded
constexpr int kW6 = kC * kTaps;        // 288
constexpr int kNumParams = (kW1 + kC) + 4 * (kWh + kC) + (kW6 + 1);  // 38177
constexpr int kWgradMaxW = 128;  // widest row the weight-gradient kernel stages

__host__ __device__ inline int w_offset(int layer) {  // layer 0..5
  return layer == 0 ? 0 : (kW1 + kC) + (layer - 1) * (kWh + kC);
}
__host__ __device__ inline int b_offset(int layer) {
  return layer == 0 ? kW1 : layer < 5 ? w_offset(layer) + kWh : w_offset(5) + kW6;
}

// ---- forward / backward-data convolution on MFMA ---------------------------

// k slice of MFMA step t for lane half hf: CIN = 32 -> tap t/2, channels
// 16*(t%2) + 8*hf; CIN = 8 -> tap 2t + hf (tap 9 is padding), channels 0..7.
template <int CIN>
__device__ inline void kmap(int t, int hf, int& tap, int& ci) {
  if (CIN == kC) {
    tap = t >> 1;
    ci = ((t & 1) << 4) + 8 * hf;
  } else {
    tap = 2 * t + hf;
    ci = 0;
  }
}

// Orders a wave's own LDS stores and loads (other lanes' data, no barrier).
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int CIN>
constexpr int nsteps() {
  return CIN == kC ? 18 : 5;
}

// LDS place (in 16-byte chunks) of chunk ch of staged pixel px.  The chunks of
// a pixel are swapped by px / 4 % 4, so that one chunk of 16 consecutive
// pixels, a 16-lane part of an LDS read, lies in 16 distinct bank groups
// (a padded fifth chunk did the same with a quarter more LDS: two instead of
// three blocks of the four-row kernel per CU).
template <int CPC>
__device__ inline int px_slot(int px, int ch) {
  return CPC == 1 ? px : px * CPC + (ch ^ ((px >> 2) & 3));
}

// 16-byte LDS chunks of a forward block by R (conv_fwd_block).
template <int CIN, int R>
constexpr int conv_lds() {
  return CIN / 8 * (R == 0 ? 4 * 3 * 34 : (R + 2) * 130);
}

// MODE 0: out = relu(D + bias).  MODE 1: out = D * (mask > 0).
// One 32-pixel tile per wave and round, the tiles of all rows and samples
// numbered in one sequence, so that every wave of a block has work at any
// width (a block per row left three of four waves idle at width 32: 8.8 us
// per hidden layer at 64 x 32 x 32); the weights a wave holds in registers
// serve its further tiles.  A wave stages the three 34-pixel input rows of its
// tile in its own part of LDS (7 loads of consecutive 16-byte chunks, where
// the fragments of all taps took 18, each pixel up to 9 times: 64 x 32 x 32
// 6.6 -> 5.6 us forward, 8.4 -> 6.1 backward).
template <int CIN, int MODE>
__device__ inline void conv_mfma_tiles(
    bf16x8* sm, const bf16* __restrict__ in, const bf16* __restrict__ wt,
    const float* __restrict__ bias, const bf16* __restrict__ mask,
    bf16* __restrict__ out, int H, int W, int B, int block, int blocks) {
  constexpr int NS = nsteps<CIN>();
  constexpr int CPC = CIN / 8;  // 16-byte chunks per pixel
  constexpr int kPx = 34, kChunks = 3 * kPx * CPC, kIt = (kChunks + 63) / 64;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  bf16x8* sw = sm + wv * kChunks;
  const int hf = lane >> 5, col = lane & 31;
  const int Wp = W + 2;
  const size_t plane = (size_t)(H + 2) * Wp;
  bf16x8 A[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) A[t] = weight_frag(wt, t, lane);
  float bco[16];
  if (MODE == 0) {
#pragma unroll
    for (int v = 0; v < 16; ++v) bco[v] = bias[8 * (v >> 2) + 4 * hf + (v & 3)];
  }
  const int per_row = W / 32;
  const int tiles = B * H * per_row;
  // Contiguous tiles per XCD (xcd_span): neighbouring rows share its L2.
  for (int tile = xcd_span(block, blocks) * 4 + wv; tile < tiles; tile += 4 * blocks) {
    const int row = tile / per_row, b = row / H, y = row - b * H;
    const int x0 = (tile - row * per_row) * 32, xo = x0 + col;
    const bf16* src = in + ((size_t)b * plane + (size_t)y * Wp + x0) * CIN;
    bf16x8 v[kIt];
#pragma unroll
    for (int k = 0; k < kIt; ++k) {
      const int q = min(lane + 64 * k, kChunks - 1), r = q / (kPx * CPC);
      v[k] = *reinterpret_cast<const bf16x8*>(src + (size_t)r * Wp * CIN + 8 * (q - r * kPx * CPC));
    }
    const size_t pix = (size_t)b * plane + (size_t)(y + 1) * Wp + (xo + 1);
    bf16x4 m[4];
    if (MODE == 1) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        m[g] = *reinterpret_cast<const bf16x4*>(mask + pix * kC + 8 * g + 4 * hf);
    }
    wave_lds_fence();  // the tile before has read its pixels
#pragma unroll
    for (int k = 0; k < kIt; ++k) {
      const int q = lane + 64 * k;
      if (q < kChunks) sw[px_slot<CPC>(q / CPC, q % CPC)] = v[k];
    }
    wave_lds_fence();
    bf16x8 Bv[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
      int tap, ci;
      kmap<CIN>(t, hf, tap, ci);
      if (tap < kTaps)
        Bv[t] = sw[px_slot<CPC>(tap / 3 * kPx + col + tap % 3, ci / 8)];
      else
        Bv[t] = bf16x8{};
    }
    f32x16 acc = {};
#pragma unroll
    for (int t = 0; t < NS; ++t)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[t], Bv[t], acc, 0, 0, 0);
    if (MODE == 0) {
      store_out_row(out + pix * kC, acc, bco, hf);
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        bf16x4 o;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          o[q] = (bf16)((float)m[g][q] > 0.0f ? acc[4 * g + q] : 0.0f);
        *reinterpret_cast<bf16x4*>(out + pix * kC + 8 * g + 4 * hf) = o;
      }
    }
  }
}

template <int CIN, int MODE>
__global__ __launch_bounds__(256) void conv_mfma_kernel(
    const bf16* __restrict__ in, const bf16* __restrict__ wt,
    const float* __restrict__ bias, const bf16* __restrict__ mask,
    bf16* __restrict__ out, int H, int W, int B) {
  __shared__ bf16x8 sm[conv_lds<CIN, 0>()];
  conv_mfma_tiles<CIN, MODE>(sm, in, wt, bias, mask, out, H, W, B, blockIdx.x, gridDim.x);
}

// Stages NROWS padded input rows (from row y0) of a 130-pixel segment
// (from padded column x0) into LDS, CPC 16-byte chunks per pixel (px_slot):
// every thread issues all its loads before its first LDS
// store (a load-store loop waited for each load in turn: 13 global-memory
// latencies per thread of the four-row kernel).
template <int NROWS, int CPC, int kPx>
__device__ inline void stage_rows(bf16x8* sm, const bf16* __restrict__ inb, int y0, int Wp,
                                  int x0) {
  constexpr int kTotal = NROWS * kPx * CPC;
  constexpr int kIt = (kTotal + 255) / 256;
  constexpr int CIN = CPC * 8;
  bf16x8 v[kIt];
  int slot[kIt];
#pragma unroll
  for (int k = 0; k < kIt; ++k) {
    const int q = threadIdx.x + 256 * k;
    const int qq = q < kTotal ? q : 0;
    const int row = qq / (kPx * CPC), rem = qq - row * (kPx * CPC);
    const int px = rem / CPC, ch = rem - px * CPC;
    slot[k] = row * (kPx * CPC) + px_slot<CPC>(px, ch);
    v[k] = *reinterpret_cast<const bf16x8*>(inb + ((size_t)(y0 + row) * Wp + (x0 + px)) * CIN +
                                            ch * 8);
  }
#pragma unroll
  for (int k = 0; k < kIt; ++k)
    if (threadIdx.x + 256 * k < kTotal) sm[slot[k]] = v[k];
}

// The (segment, row group, sample) of block `block` of a (W / 128, H / R, B)
// grid in linear order, numbered so that each XCD takes one contiguous range of row groups:
// the hardware deals blocks round-robin to the 8 XCDs, which put the row
// groups above and below a block on other XCDs, so the input rows two
// blocks share were fetched into two L2s (1.27x the activations per hidden
// layer at 512^2 with four rows per block).
__device__ inline void xcd_tile(int block, int segs, int groups, int samples, int& seg, int& grp,
                                int& b) {
  const int L = xcd_span(block, segs * groups * samples);
  seg = L % segs;
  const int rest = L / segs;
  grp = rest % groups;
  b = rest / groups;
}

// Forward layer for rows of 128 pixels or more: a block takes a 128-pixel
// segment of row y, stages input rows y-1..y+1 over the segment plus its
// 1-pixel ring in LDS once (130 pixels x CIN channels x 3 rows, in 16-byte
// chunks),
// and each wave computes one 32-pixel tile from LDS.  Same arithmetic and
// output as conv_mfma_kernel<CIN, 0>.  W / 128 x H x B blocks.
template <int CIN>
__device__ inline void conv_fwd_lds_block(
    bf16x8* sm, const bf16* __restrict__ in, const bf16* __restrict__ wt,
    const float* __restrict__ bias, bf16* __restrict__ out, int H, int W, int B, int block) {
  constexpr int NS = nsteps<CIN>();
  constexpr int CPC = CIN / 8;  // 16-byte chunks per pixel
  constexpr int kPx = 130;
  int seg, y, b;
  xcd_tile(block, W / 128, H, B, seg, y, b);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int hf = lane >> 5, col = lane & 31;
  const int Wp = W + 2;
  const size_t plane = (size_t)(H + 2) * Wp;
  const bf16* inb = in + (size_t)b * plane * CIN;
  const int x0 = seg * 128;  // padded column of the segment's left ring pixel
  // Weights and biases first: loaded after the staged rows' LDS stores, they
  // were a second global-memory latency before the first MFMA.
  bf16x8 A[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) A[t] = weight_frag(wt, t, lane);
  float bco[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) bco[v] = bias[8 * (v >> 2) + 4 * hf + (v & 3)];
  stage_rows<3, CPC, kPx>(sm, inb, y, Wp, x0);
  __syncthreads();
  const int xl = wv * 32 + col;  // pixel within the segment
  bf16x8 Bv[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) {
    int tap, ci;
    kmap<CIN>(t, hf, tap, ci);
    if (tap < kTaps) {
      const int dy = tap / 3 - 1, dx = tap % 3 - 1;
      Bv[t] = sm[(dy + 1) * kPx * CPC + px_slot<CPC>(xl + 1 + dx, ci / 8)];
    } else {
      Bv[t] = bf16x8{};
    }
  }
  f32x16 acc = {};
#pragma unroll
  for (int t = 0; t < NS; ++t)
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[t], Bv[t], acc, 0, 0, 0);
  const size_t pix = (size_t)b * plane + (size_t)(y + 1) * Wp + (x0 + xl + 1);
  store_out_row(out + pix * kC, acc, bco, hf);
}

// conv_fwd_lds_block over R output rows per block: the block stages R + 2
// input rows once (instead of 3 per output row) and each wave keeps its
// weight fragments in registers across the R rows (instead of reloading
// them per 32-pixel tile).  Each tile's MFMA sequence, bias and ReLU are
// those of conv_fwd_lds_block, so the output is bitwise the same.
// W / 128 x H / R x B blocks.
template <int CIN, int R>
__device__ inline void conv_fwd_rows_block(
    bf16x8* sm, const bf16* __restrict__ in, const bf16* __restrict__ wt,
    const float* __restrict__ bias, bf16* __restrict__ out, int H, int W, int B, int block) {
  constexpr int NS = nsteps<CIN>();
  constexpr int CPC = CIN / 8;
  constexpr int kPx = 130;
  int seg, grp, b;
  xcd_tile(block, W / 128, H / R, B, seg, grp, b);
  const int y0 = grp * R;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int hf = lane >> 5, col = lane & 31;
  const int Wp = W + 2;
  const size_t plane = (size_t)(H + 2) * Wp;
  const bf16* inb = in + (size_t)b * plane * CIN;
  const int x0 = seg * 128;
  // Weights and biases first (as conv_fwd_lds_block).
  bf16x8 A[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) A[t] = weight_frag(wt, t, lane);
  float bco[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) bco[v] = bias[8 * (v >> 2) + 4 * hf + (v & 3)];
  stage_rows<R + 2, CPC, kPx>(sm, inb, y0, Wp, x0);
  __syncthreads();
  const int xl = wv * 32 + col;
#pragma unroll 1
  for (int r = 0; r < R; ++r) {
    bf16x8 Bv[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
      int tap, ci;
      kmap<CIN>(t, hf, tap, ci);
      if (tap < kTaps) {
        const int dy = tap / 3 - 1, dx = tap % 3 - 1;
        Bv[t] = sm[(r + dy + 1) * kPx * CPC + px_slot<CPC>(xl + 1 + dx, ci / 8)];
      } else {
        Bv[t] = bf16x8{};
      }
    }
    f32x16 acc = {};
#pragma unroll
    for (int t = 0; t < NS; ++t)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[t], Bv[t], acc, 0, 0, 0);
    const size_t pix = (size_t)b * plane + (size_t)(y0 + r + 1) * Wp + (x0 + xl + 1);
    store_out_row(out + pix * kC, acc, bco, hf);
  }
}

// The forward kernel R selects: 0 a tile per wave (conv_mfma_tiles), 1 a row
// per block, 2 or 4 rows per block.
template <int CIN, int R>
__device__ inline void conv_fwd_block(bf16x8* sm, const bf16* in, const bf16* wt, const float* bias, bf16* out,
                                      int H, int W, int B, int block, int blocks) {
  if (R == 0)
    conv_mfma_tiles<CIN, 0>(sm, in, wt, bias, nullptr, out, H, W, B, block, blocks);
  else if (R == 1)
    conv_fwd_lds_block<CIN>(sm, in, wt, bias, out, H, W, B, block);
  else
    conv_fwd_rows_block<CIN, R ? R : 1>(sm, in, wt, bias, out, H, W, B, block);
}

template <int CIN, int R>
__global__ __launch_bounds__(256, 3) void conv_fwd_kernel(
    const bf16* __restrict__ in, const bf16* __restrict__ wt,
    const float* __restrict__ bias, bf16* __restrict__ out, int H, int W, int B) {
  __shared__ bf16x8 sm[conv_lds<CIN, R>()];
  conv_fwd_block<CIN, R>(sm, in, wt, bias, out, H, W, B, blockIdx.x, gridDim.x);
}

// One hidden layer of two networks of one sample each (two levels of the
// learned preconditioner), the first nb0 blocks the first network's by R and
// the others the second's, a tile per wave: the second level's 32 blocks ran
// on a stream of their own before, whose fork and join cost more (about 17 us
// per application at 4096^2) than its five short launches.  Three blocks per
// CU (px_slot, 168 registers): the 640 blocks of 512^2 and 128^2 are one round
// (14.2 us with two per CU, 12.4 now).
struct ConvArgs {
  const bf16* in;
  const bf16* wt;
  const float* bias;
  bf16* out;
  int H, W;
};
template <int R>
__global__ __launch_bounds__(256, 3) void conv_fwd_pair_kernel(ConvArgs a, ConvArgs b, int nb0) {
  __shared__ bf16x8 sm[conv_lds<kC, R>() > conv_lds<kC, 0>() ? conv_lds<kC, R>()
                                                             : conv_lds<kC, 0>()];
  if ((int)blockIdx.x < nb0)
    conv_fwd_block<kC, R>(sm, a.in, a.wt, a.bias, a.out, a.H, a.W, 1, blockIdx.x, nb0);
  else
    conv_mfma_tiles<kC, 0>(sm, b.in, b.wt, b.bias, nullptr, b.out, b.H, b.W, 1, blockIdx.x - nb0,
                           gridDim.x - nb0);
}

// ---- output layer (32 -> 1), FP32 on the vector units ------------------------

// out[b][y][x] = b6 + sum_{tap,ci} w6[tap][ci] * a5[b][y+1+dy][x+1+dx][ci].
__global__ __launch_bounds__(256) void out_layer_kernel(
    const bf16* __restrict__ a5, const float* __restrict__ w6,
    const float* __restrict__ bias, float* __restrict__ out, int B, int H,
    int W) {
  const float b6 = bias[5 * kC];
  // Rows in one contiguous range per XCD (xcd_span): the rows above and
  // below a block's pixels are then in its XCD's L2.
  const long idx = (long)xcd_span(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  const long total = (long)B * H * W;
  if (idx >= total) return;
  const int x = (int)(idx % W);
  const int y = (int)((idx / W) % H);
  const int b = (int)(idx / ((long)W * H));
  const int Wp = W + 2;
  const size_t plane = (size_t)(H + 2) * Wp;
  float acc = 0.0f;
#pragma unroll
  for (int tap = 0; tap < kTaps; ++tap) {
    const int dy = tap / 3 - 1, dx = tap % 3 - 1;
    const bf16* p = a5 + ((size_t)b * plane + (size_t)(y + 1 + dy) * Wp + (x + 1 + dx)) * kC;
#pragma unroll
    for (int c8 = 0; c8 < kC; c8 += 8) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(p + c8);
#pragma unroll
      for (int q = 0; q < 8; ++q) acc += w6[tap * kC + c8 + q] * (float)v[q];
    }
  }
  out[idx] = acc + b6;
}

// ---- loss: mean squared error, and its gradient -----------------------------

// dout = 2 (out - t) / n; per-block partial sums of (out - t)^2 in FP32.
__global__ __launch_bounds__(256) void mse_kernel(const float* __restrict__ out,
                                                  const float* __restrict__ t,
                                                  float* __restrict__ dout,
                                                  float* __restrict__ partial,
                                                  long n) {
  __shared__ float s[256];
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  float e2 = 0.0f;
  if (i < n) {
    const float d = out[i] - t[i];
    dout[i] = 2.0f * d / (float)n;
    e2 = d * d;
  }
  s[threadIdx.x] = e2;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (threadIdx.x < st) s[threadIdx.x] += s[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// ---- output layer backward ---------------------------------------------------

// delta5[p][ci] = (a5[p][ci] > 0) * sum_tap dout[p - tap] * w6[tap][ci].
__global__ __launch_bounds__(256) void out_layer_bwd_data_kernel(
    const float* __restrict__ dout, const float* __restrict__ w6,
    const bf16* __restrict__ a5, bf16* __restrict__ d5, int B, int H, int W) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  const long total = (long)B * H * W;
  if (idx >= total) return;
  const int x = (int)(idx % W);
  const int y = (int)((idx / W) % H);
  const int b = (int)(idx / ((long)W * H));
  float g[kC];
#pragma unroll
  for (int c = 0; c < kC; ++c) g[c] = 0.0f;
#pragma unroll
  for (int tap = 0; tap < kTaps; ++tap) {
    const int dy = tap / 3 - 1, dx = tap % 3 - 1;
    const int ys = y - dy, xs = x - dx;  // output pixel that reads p at tap
    if (ys < 0 || ys >= H || xs < 0 || xs >= W) continue;
    const float d = dout[((long)b * H + ys) * W + xs];
#pragma unroll
    for (int c = 0; c < kC; ++c) g[c] += d * w6[tap * kC + c];
  }
  const int Wp = W + 2;
  const size_t pix = (size_t)b * (H + 2) * Wp + (size_t)(y + 1) * Wp + (x + 1);
#pragma unroll
  for (int c8 = 0; c8 < kC; c8 += 8) {
    const bf16x8 m = *reinterpret_cast<const bf16x8*>(a5 + pix * kC + c8);
    bf16x8 o;
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = (bf16)((float)m[q] > 0.0f ? g[c8 + q] : 0.0f);
    *reinterpret_cast<bf16x8*>(d5 + pix * kC + c8) = o;
  }
}

// Partial dW6[tap][ci] and db6 per block of rows: thread t < 288 handles
// (tap, ci) = (t / 32, t % 32); thread 288 accumulates db6.  Block blk of nblk
// handles rows [blk*rows_per, ...) of the B*H rows.
__device__ inline void out_layer_wgrad_rows(
    const float* __restrict__ dout, const bf16* __restrict__ a5,
    float* __restrict__ partial, int B, int H, int W, int rows_per) {
  const int t = threadIdx.x;
  if (t > kW6) return;
  const int Wp = W + 2;
  const size_t plane = (size_t)(H + 2) * Wp;
  float acc = 0.0f;
  const int r0 = blockIdx.x * rows_per;
  const int r1 = min(r0 + rows_per, B * H);
  const int tap = t / kC, ci = t % kC;
  const int dy = tap / 3 - 1, dx = tap % 3 - 1;
  for (int row = r0; row < r1; ++row) {
    const int b = row / H, y = row % H;
    const float* d = dout + (long)row * W;
    if (t == kW6) {
      for (int x = 0; x < W; ++x) acc += d[x];
    } else {
      // 32 pixels' loads before any is used (W is a multiple of 32).
      const bf16* a = a5 + ((size_t)b * plane + (size_t)(y + 1 + dy) * Wp + 1 + dx) * kC + ci;
      for (int x = 0; x < W; x += 32) {
        bf16 v[32];
        float e[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) {
          v[k] = a[(size_t)(x + k) * kC];
          e[k] = d[x + k];
        }
#pragma unroll
        for (int k = 0; k < 32; ++k) acc += e[k] * (float)v[k];
      }
    }
  }
  partial[(size_t)blockIdx.x * (kW6 + 1) + t] = acc;
}

// ---- hidden-layer weight gradient on MFMA ------------------------------------
//
// dW[co][n] = sum over pixels p of delta[p][co] * In[p + tap(n)][ci(n)],
// n = tap*CIN + ci, and db[co] = sum_p delta[p][co].  One block per group of
// rows; the delta row and the three input rows it needs are staged in LDS,
// then each wave accumulates its share of the 32-wide n blocks over all
// pixels with MFMA steps of 16 pixels (A: lane co, 8 pixels; B: lane n,
// the same 8 pixels).  Per-block partials are summed by reduce_grad_kernel.
constexpr int kWgradThreads = 320;     // 5 waves: 9 n blocks as 2, 2, 2, 2, 1
template <int CIN>
__device__ inline void wgrad_rows(
    bf16* __restrict__ sd, bf16* __restrict__ sa, const bf16* __restrict__ delta,
    const bf16* __restrict__ in, float* __restrict__ partial, int B, int H, int W,
    int rows_per) {
  constexpr int kT = kWgradThreads, kWv = kT / 64;
  constexpr int kQ = CIN == kC ? 2 : 1;  // n blocks per wave
  constexpr int N = kTaps * CIN;         // 288 or 72
  constexpr int NB = (N + 31) / 32;      // 9 or 3 blocks of 32
  constexpr int kMaxW = kWgradMaxW;      // staged row width limit
  // sd: delta row; sa: input rows y-1..y+1.
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int hf = lane >> 5, col = lane & 31;
  const int Wp = W + 2;
  const size_t plane = (size_t)(H + 2) * Wp;
  f32x16 acc[kQ];
#pragma unroll
  for (int q = 0; q < kQ; ++q) acc[q] = f32x16{};
  float dbias = 0.0f;
  const int r0 = blockIdx.x * rows_per;
  const int r1 = min(r0 + rows_per, B * H);
  // delta[b][y+1][1..W][*] and in[b][y..y+2][0..W+1][*] of one row, in 16-byte
  // chunks: row r + 1's are loaded into registers while row r is computed
  // from LDS (waiting for each row's loads in turn took 17.6 us per hidden
  // layer at 64 x 32 x 32, 13.0 us without).
  constexpr int kD = (kMaxW * kC / 8 + kT - 1) / kT;
  constexpr int kA = (3 * (kMaxW + 2) * CIN / 8 + kT - 1) / kT;
  const int nd = W * kC / 8, na = 3 * Wp * CIN / 8;
  bf16x8 vd[kD], va[kA];
  auto load_row = [&](int row) {
    const int b = row / H, y = row % H;
    const bf16* d = delta + ((size_t)b * plane + (size_t)(y + 1) * Wp + 1) * kC;
    const bf16* a = in + ((size_t)b * plane + (size_t)y * Wp) * CIN;
#pragma unroll
    for (int k = 0; k < kD; ++k) {
      const int i = threadIdx.x + kT * k;
      if (i < nd) vd[k] = *reinterpret_cast<const bf16x8*>(d + 8 * i);
    }
#pragma unroll
    for (int k = 0; k < kA; ++k) {
      const int i = threadIdx.x + kT * k;
      if (i < na) va[k] = *reinterpret_cast<const bf16x8*>(a + 8 * i);
    }
  };
  if (r0 < r1) load_row(r0);
  for (int row = r0; row < r1; ++row) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kD; ++k) {
      const int i = threadIdx.x + kT * k;
      if (i < nd) *reinterpret_cast<bf16x8*>(sd + 8 * i) = vd[k];
    }
#pragma unroll
    for (int k = 0; k < kA; ++k) {
      const int i = threadIdx.x + kT * k;
      if (i < na) *reinterpret_cast<bf16x8*>(sa + 8 * i) = va[k];
    }
    __syncthreads();
    if (row + 1 < r1) load_row(row + 1);
    for (int x0 = 0; x0 < W; x0 += 16) {
      bf16x8 a;
#pragma unroll
      for (int s = 0; s < 8; ++s) a[s] = sd[(x0 + 8 * hf + s) * kC + col];
      if (wv == 0) {
#pragma unroll
        for (int s = 0; s < 8; ++s) dbias += (float)a[s];
      }
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        const int nb = wv + kWv * q;
        if (nb >= NB) break;
        const int n = nb * 32 + col;
        bf16x8 bv;
        if (n < N) {
          const int tap = n / CIN, ci = n % CIN;
          const int dy = tap / 3 - 1, dx = tap % 3 - 1;
#pragma unroll
          for (int s = 0; s < 8; ++s)
            bv[s] = sa[((1 + dy) * Wp + (x0 + 8 * hf + s + 1 + dx)) * CIN + ci];
        } else {
          bv = bf16x8{};
        }
        acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bv, acc[q], 0, 0, 0);
      }
    }
  }
  // D[co][n]: lane l holds n = nb*32 + l%32 and co = 8*(v/4) + 4*hf + v%4.
  float* pb = partial + (size_t)blockIdx.x * (kC * N + kC);
#pragma unroll
  for (int q = 0; q < kQ; ++q) {
    const int nb = wv + kWv * q;
    if (nb >= NB) break;
    const int n = nb * 32 + col;
    if (n >= N) continue;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int co = 8 * (v >> 2) + 4 * hf + (v & 3);
      pb[co * N + n] = acc[q][v];
    }
  }
  if (wv == 0) {
    // Lanes l and l+32 hold the two halves of channel l%32.
    const float other = __shfl_xor(dbias, 32);
    if (hf == 0) pb[kC * N + col] = dbias + other;
  }
}

// A layer's input gradients' and activations' pointers (0 the first layer).
struct WgradArgs {
  const bf16* delta[5];
  const bf16* in[5];
  const float* dout;  // output layer
  const bf16* a5;
  float* partial;
};

// Length of a block's partial row of layer l (5: the output layer), and the
// rows of the layers before it per block.
__host__ __device__ inline int wgrad_len(int l) {
  return l == 0 ? kC * kTaps * kC0 + kC : l < 5 ? kC * kTaps * kC + kC : kW6 + 1;
}
__host__ __device__ inline int wgrad_offset(int l) {
  return l == 0 ? 0 : wgrad_len(0) + (l - 1) * wgrad_len(1);
}

// The weight gradients of all six layers in one launch, after the backward
// data pass, which none of them waits for: a layer alone is one four-wave
// block per CU whose rows are a chain of load, LDS and MFMA latencies (64 x 32
// x 32: 13.1 us per hidden layer, 14.0 and 7.9 us the last and first, 74 us in
// all); together they fill the chip.
// Grid (nblk, 6), the longest layers first.
__global__ __launch_bounds__(kWgradThreads) void wgrad_kernel(WgradArgs a, int B, int H, int W,
                                                              int rows_per) {
  __shared__ bf16 sd[kWgradMaxW * kC];
  __shared__ bf16 sa[3 * (kWgradMaxW + 2) * kC];
  const int l = blockIdx.y < 4 ? 4 - blockIdx.y : blockIdx.y == 4 ? 5 : 0;
  float* part = a.partial + (size_t)gridDim.x * wgrad_offset(l);
  if (l == 5)
    out_layer_wgrad_rows(a.dout, a.a5, part, B, H, W, rows_per);
  else if (l == 0)
    wgrad_rows<kC0>(sd, sa, a.delta[0], a.in[0], part, B, H, W, rows_per);
  else
    wgrad_rows<kC>(sd, sa, a.delta[l], a.in[l], part, B, H, W, rows_per);
}

// Sums each layer's nblk partial rows ([co][tap][ci_pad] then db) in block
// order into the master-layout gradient ([co][ci][ky][kx], then b).  One column
// per thread; kReduceBatch rows are loaded before any is added, or each load's
// latency would be waited for in turn (a plain loop took 60 us for 256 rows
// of 9248 columns, 9.5 MB).  All layers in one launch: blockIdx.y is the layer.
constexpr int kReduceBatch = 64;
__global__ __launch_bounds__(64) void reduce_grad_kernel(const float* __restrict__ partials,
                                                         int nblk, float* __restrict__ grad) {
  const int i = blockIdx.x * 64 + threadIdx.x, l = blockIdx.y;
  const int cin_pad = l == 0 ? kC0 : kC, cin = l == 0 ? kIn : kC, cout = l == 5 ? 1 : kC;
  const int nw = cout * kTaps * cin_pad, len = nw + cout;
  const float* __restrict__ partial = partials + (size_t)nblk * wgrad_offset(l);
  float* gw = grad + w_offset(l);
  float* gb = grad + b_offset(l);
  if (i >= len) return;
  float s = 0.0f;
  int b = 0;
  for (; b + kReduceBatch <= nblk; b += kReduceBatch) {
    float v[kReduceBatch];
#pragma unroll
    for (int k = 0; k < kReduceBatch; ++k) v[k] = partial[(size_t)(b + k) * len + i];
#pragma unroll
    for (int k = 0; k < kReduceBatch; ++k) s += v[k];
  }
  for (; b < nblk; ++b) s += partial[(size_t)b * len + i];
  if (i >= nw) {
    gb[i - nw] = s;
    return;
  }
  const int co = i / (kTaps * cin_pad), rem = i % (kTaps * cin_pad);
  const int tap = rem / cin_pad, ci = rem % cin_pad;
  if (ci < cin) gw[(co * cin + ci) * kTaps + tap] = s;
}

// ---- parameters ------------------------------------------------------------

// BF16 kernel layouts from the FP32 master: the hidden layers' forward and
// backward-data weights and the first layer's in fragment order (weight_frag),
// output-layer w6 [tap][ci] (FP32) and the biases.  Row col and K-value k of
// the forward fragments are output channel and (tap, input channel), of the
// backward ones input channel and (flipped tap, output channel).
__global__ __launch_bounds__(256) void pack_params_kernel(
    const float* __restrict__ master, bf16* __restrict__ wf1,
    bf16* __restrict__ wfh, bf16* __restrict__ wbh, float* __restrict__ w6,
    float* __restrict__ bias) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int j = i & 7, hf = (i >> 8) & 1, col = (i >> 3) & 31;
  if (i < kWf1) {
    int tap, ci;
    kmap<kC0>(i >> 9, hf, tap, ci);
    wf1[i] = (bf16)(j < kIn && tap < kTaps ? master[(col * kIn + j) * kTaps + tap] : 0.0f);
  }
  // Hidden layers 2..5.
  if (i < 4 * kWh) {
    const int l = i / kWh;
    const float* W = master + w_offset(l + 1);
    int tap, c0;
    kmap<kC>((i - l * kWh) >> 9, hf, tap, c0);
    wfh[i] = (bf16)W[(col * kC + c0 + j) * kTaps + tap];
    wbh[i] = (bf16)W[((c0 + j) * kC + col) * kTaps + (kTaps - 1 - tap)];
  }
  if (i < kW6) {
    const int tap = i / kC, ci = i % kC;
    w6[i] = (float)(bf16)master[w_offset(5) + ci * kTaps + tap];
  }
  if (i < 5 * kC + 1) bias[i] = i < 5 * kC ? master[b_offset(i / kC) + i % kC] : master[b_offset(5)];
}

__global__ __launch_bounds__(256) void adam_kernel(float* __restrict__ p,
                                                   const float* __restrict__ g,
                                                   float* __restrict__ m,
                                                   float* __restrict__ v, int n,
                                                   float lr, float b1, float b2,
                                                   float eps, float c1, float c2) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// Input tensor from FP32 planes [b][y][x][3] (already scaled).
__global__ __launch_bounds__(256) void pack_input_kernel(const float* __restrict__ src,
                                                         bf16* __restrict__ dst, int B,
                                                         int H, int W) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long)B * H * W) return;
  const int x = (int)(idx % W), y = (int)((idx / W) % H), b = (int)(idx / ((long)W * H));
  const size_t pix = (size_t)b * (H + 2) * (W + 2) + (size_t)(y + 1) * (W + 2) + (x + 1);
  bf16x8 o = bf16x8{};
  for (int c = 0; c < kIn; ++c) o[c] = (bf16)src[idx * kIn + c];
  *reinterpret_cast<bf16x8*>(dst + pix * kC0) = o;
}

}  // namespace nn
}  // namespace tea

// ---- host side -----------------------------------------------------------------

using namespace tea;
using namespace tea::nn;

struct tea_nn {
  int device = 0;
  int max_batch = 0, H = 0, W = 0;
  hipStream_t stream = nullptr;
  int fwd_rows = kFwdRows;  // rows per block of the forward kernel (0: one-row kernel)
  // parameters
  float *master = nullptr, *grad = nullptr, *adam_m = nullptr, *adam_v = nullptr;
  long adam_t = 0;
  bf16 *wf1 = nullptr, *wfh = nullptr, *wbh = nullptr;
  float *w6 = nullptr, *bias = nullptr;
  // activations and gradients
  float* in_f32 = nullptr;   // [B][H][W][3]
  bf16* in0 = nullptr;       // [B][H+2][W+2][8]
  bf16* act[5] = {};         // a1..a5 [B][H+2][W+2][32]
  bf16* del[5] = {};         // delta1..delta5
  float *out = nullptr, *target = nullptr, *dout = nullptr;
  float *partial = nullptr, *loss_part = nullptr;
  size_t loss_len = 0;       // floats loss_part holds
  size_t partial_len = 0;
  int wg_blocks = 0;
  // device-resident training set
  float *ds_in = nullptr, *ds_tgt = nullptr;
  int ds_n = 0;
  int* ds_order = nullptr;
  int order_len = 0;         // samples that ds_order holds
};

namespace {

size_t act_elems(const tea_nn* n, int c) {
  return (size_t)n->max_batch * (n->H + 2) * (n->W + 2) * c;
}

int nn_alloc(void** p, size_t bytes, hipStream_t st) {
  if (hipMalloc(p, bytes) != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    set_error("hipMalloc failed in the network workspace");
    return TEA_HIP_ENOMEM;
  }
  TEA_HIP_TRY(hipMemsetAsync(*p, 0, bytes, st));
  return TEA_HIP_OK;
}

int pack_params(tea_nn* n) {
  hipLaunchKernelGGL(pack_params_kernel, dim3((4 * kWh + 255) / 256), dim3(256), 0,
                     n->stream, n->master, n->wf1, n->wfh, n->wbh, n->w6, n->bias);
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}

// conv_mfma_kernel's grid: a tile per wave, at most 2048 blocks (the chip
// holds about that many at once).
dim3 conv_grid(const tea_nn* n, int batch) {
  const long tiles = (long)batch * n->H * (n->W / 32);
  return dim3((unsigned)std::min(2048L, (tiles + 3) / 4));
}
unsigned flat_blocks(long count) { return (unsigned)((count + 255) / 256); }

// The forward kernel for a batch: several rows per block only while the grid
// keeps at least 512 blocks (on small grids the one-row kernel's parallelism
// matters more than the saved weight and row loads), a tile per wave where
// rows are not whole 128-pixel segments.
int fwd_variant(const tea_nn* n, int batch) {
  const int H = n->H, W = n->W, R = n->fwd_rows;
  if (W % 128 != 0) return 0;
  if ((R == 2 || R == 4) && H % R == 0 && (long)(W / 128) * (H / R) * batch >= 512) return R;
  return 1;
}
unsigned fwd_blocks(const tea_nn* n, int batch, int variant) {
  return variant == 0 ? conv_grid(n, batch).x
                      : (unsigned)((n->W / 128) * (n->H / variant) * batch);
}

template <int CIN>
void launch_fwd(tea_nn* n, int batch, hipStream_t st, const bf16* in, const bf16* wt,
                const float* bias, bf16* out) {
  const int v = fwd_variant(n, batch);
  const auto kernel = v == 0   ? conv_fwd_kernel<CIN, 0>
                      : v == 1 ? conv_fwd_kernel<CIN, 1>
                      : v == 2 ? conv_fwd_kernel<CIN, 2>
                               : conv_fwd_kernel<CIN, 4>;
  hipLaunchKernelGGL(kernel, dim3(fwd_blocks(n, batch, v)), dim3(256), 0, st, in, wt, bias, out,
                     n->H, n->W, batch);
}

// Forward pass over `batch` samples whose packed input is in n->in0, on
// stream `st` (the network's own, or a solver's); without the output layer
// unless with_output (its caller then runs it on the last activations); from
// hidden layer `first` on (0-based: the caller has written the activations
// of the layers before it).
int forward_on(tea_nn* n, int batch, hipStream_t st, bool with_output = true,
               int first = 0) {
  const int H = n->H, W = n->W;
  if (first == 0) launch_fwd<kC0>(n, batch, st, n->in0, n->wf1, n->bias, n->act[0]);
  for (int l = first > 1 ? first : 1; l < 5; ++l)
    launch_fwd<kC>(n, batch, st, n->act[l - 1], n->wfh + (size_t)(l - 1) * kWh, n->bias + l * kC,
                   n->act[l]);
  if (with_output)
    hipLaunchKernelGGL(out_layer_kernel, dim3(flat_blocks((long)batch * H * W)), dim3(256),
                       0, st, n->act[4], n->w6, n->bias, n->out, batch, H, W);
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}

int forward(tea_nn* n, int batch) { return forward_on(n, batch, n->stream); }

// Blocks of mse_kernel, each leaving one partial of a batch's squared error.
unsigned loss_blocks(const tea_nn* n, int batch) {
  return flat_blocks((long)batch * n->H * n->W);
}

// The losses of `batches` batches from their partials, one batch after the
// other in n->loss_part (waits for the stream).
int read_losses(tea_nn* n, int batch, int batches, float* loss) {
  const size_t nb = loss_blocks(n, batch);
  const long cnt = (long)batch * n->H * n->W;
  std::vector<float> lp(nb * batches);
  TEA_HIP_TRY(hipMemcpyAsync(lp.data(), n->loss_part, lp.size() * sizeof(float),
                             hipMemcpyDeviceToHost, n->stream));
  TEA_HIP_TRY(hipStreamSynchronize(n->stream));
  for (int k = 0; k < batches; ++k) {
    double s = 0.0;
    for (size_t i = 0; i < nb; ++i) s += lp[k * nb + i];
    loss[k] = (float)(s / (double)cnt);
  }
  return TEA_HIP_OK;
}

// Queues the loss partials (batch k's in n->loss_part) and gradients for
// `batch` samples (input packed, targets in place).
int loss_and_grad(tea_nn* n, int batch, int k = 0) {
  const int H = n->H, W = n->W;
  TEA_RETURN_IF(forward(n, batch));
  const long cnt = (long)batch * H * W;
  const unsigned nb = loss_blocks(n, batch);
  hipLaunchKernelGGL(mse_kernel, dim3(nb), dim3(256), 0, n->stream, n->out, n->target,
                     n->dout, n->loss_part + (size_t)k * nb, cnt);
  // Backward data, output layer to layer 1.
  hipLaunchKernelGGL(out_layer_bwd_data_kernel, dim3(nb), dim3(256), 0, n->stream,
                     n->dout, n->w6, n->act[4], n->del[4], batch, H, W);
  for (int l = 4; l >= 1; --l)
    hipLaunchKernelGGL((conv_mfma_kernel<kC, 1>), conv_grid(n, batch), dim3(256), 0,
                       n->stream, n->del[l], n->wbh + (size_t)(l - 1) * kWh, nullptr,
                       n->act[l - 1], n->del[l - 1], H, W, batch);
  // Weight gradients.
  const int rows = batch * H;
  const int rows_per = (rows + n->wg_blocks - 1) / n->wg_blocks;
  const int nblk = (rows + rows_per - 1) / rows_per;
  WgradArgs a{};
  for (int l = 0; l < 5; ++l) {
    a.delta[l] = n->del[l];
    a.in[l] = l == 0 ? n->in0 : n->act[l - 1];
  }
  a.dout = n->dout;
  a.a5 = n->act[4];
  a.partial = n->partial;
  hipLaunchKernelGGL(wgrad_kernel, dim3(nblk, 6), dim3(kWgradThreads), 0, n->stream, a, batch, H,
                     W, rows_per);
  hipLaunchKernelGGL(reduce_grad_kernel, dim3((wgrad_len(1) + 63) / 64, 6), dim3(64), 0,
                     n->stream, n->partial, nblk, n->grad);
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}

int adam_step(tea_nn* n, float lr) {
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  n->adam_t += 1;
  // Bias corrections 1 - beta^t of the FP32 betas, formed in double: in FP32,
  // 1 - powf(0.999f, t) loses about 1e-5 of its value to cancellation.
  const float c1 = (float)(1.0 - pow((double)b1, (double)n->adam_t));
  const float c2 = (float)(1.0 - pow((double)b2, (double)n->adam_t));
  hipLaunchKernelGGL(adam_kernel, dim3((kNumParams + 255) / 256), dim3(256), 0,
                     n->stream, n->master, n->grad, n->adam_m, n->adam_v, kNumParams,
                     lr, b1, b2, eps, c1, c2);
  TEA_HIP_TRY(hipGetLastError());
  return pack_params(n);
}

int upload_batch(tea_nn* n, int batch, const float* input, const float* target) {
  const long px = (long)batch * n->H * n->W;
  TEA_HIP_TRY(hipMemcpyAsync(n->in_f32, input, px * kIn * sizeof(float),
                             hipMemcpyHostToDevice, n->stream));
  if (target)
    TEA_HIP_TRY(hipMemcpyAsync(n->target, target, px * sizeof(float),
                               hipMemcpyHostToDevice, n->stream));
  hipLaunchKernelGGL(pack_input_kernel, dim3(flat_blocks(px)), dim3(256), 0, n->stream,
                     n->in_f32, n->in0, batch, n->H, n->W);
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}

// Gathers samples order[0..batch) of the resident training set: the packed
// input (as pack_input_kernel) and the targets.
__global__ __launch_bounds__(256) void gather_kernel(const float* __restrict__ ds_in,
                                                     const float* __restrict__ ds_tgt,
                                                     const int* __restrict__ order,
                                                     bf16* __restrict__ in0,
                                                     float* __restrict__ tgt, int batch,
                                                     int H, int W) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  const int px = H * W;
  if (i >= (long)batch * px) return;
  const int b = (int)(i / px), p = (int)(i % px), y = p / W, x = p % W;
  const long src = (long)order[b] * px + p;
  tgt[i] = ds_tgt[src];
  bf16x8 o = bf16x8{};
  for (int c = 0; c < kIn; ++c) o[c] = (bf16)ds_in[src * kIn + c];
  const size_t pix = (size_t)b * (H + 2) * (W + 2) + (size_t)(y + 1) * (W + 2) + (x + 1);
  *reinterpret_cast<bf16x8*>(in0 + pix * kC0) = o;
}

#define NN_CHECK(n) TEA_CHECK_ARG((n) != nullptr, "null network handle")

}  // namespace

namespace tea {
namespace nn {
// Used by the flexible-CG preconditioner (fcg.hip).
int forward_hidden_on_stream(tea_nn* n, hipStream_t st, int first) {
  return forward_on(n, 1, st, false, first);
}
int forward_hidden_pair(tea_nn* n0, tea_nn* n1, hipStream_t st, int first) {
  const int v = fwd_variant(n0, 1);
  const unsigned nb0 = fwd_blocks(n0, 1, v), nb1 = conv_grid(n1, 1).x;
  const auto kernel = v == 0   ? conv_fwd_pair_kernel<0>
                      : v == 1 ? conv_fwd_pair_kernel<1>
                      : v == 2 ? conv_fwd_pair_kernel<2>
                               : conv_fwd_pair_kernel<4>;
  auto args = [](tea_nn* n, int l) {
    return ConvArgs{n->act[l - 1], n->wfh + (size_t)(l - 1) * kWh, n->bias + l * kC, n->act[l],
                    n->H, n->W};
  };
  for (int l = first; l < 5; ++l)
    hipLaunchKernelGGL(kernel, dim3(nb0 + nb1), dim3(256), 0, st, args(n0, l), args(n1, l),
                       (int)nb0);
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}
const bf16* last_hidden(tea_nn* n) { return n->act[4]; }
bf16* hidden(tea_nn* n, int l) { return n->act[l]; }
bf16* input_tensor(tea_nn* n) { return n->in0; }
PackedWeights packed_weights(const tea_nn* n) {
  return PackedWeights{n->wf1, n->wfh, n->w6, n->bias};
}
const float* output(tea_nn* n) { return n->out; }
int sync(tea_nn* n) {
  TEA_HIP_TRY(hipStreamSynchronize(n->stream));
  return TEA_HIP_OK;
}
}  // namespace nn
}  // namespace tea

extern "C" {

int tea_nn_num_params(void) { return kNumParams; }

int tea_nn_create(int device, int max_batch, int height, int width, tea_nn** out) {
  TEA_CHECK_ARG(out != nullptr, "null output handle");
  *out = nullptr;
  TEA_CHECK_ARG(max_batch >= 1 && height >= 1 && width >= 32 && width % 32 == 0,
                "need batch >= 1, height >= 1 and width a multiple of 32");
  TEA_HIP_TRY(hipSetDevice(device));
  tea_nn* n = new tea_nn();
  n->device = device;
  n->max_batch = max_batch;
  n->H = height;
  n->W = width;
  if (const char* v = getenv("TEA_NN_FWD_ROWS")) n->fwd_rows = atoi(v);
  auto fail = [&](int code) {
    tea_nn_destroy(n);
    return code;
  };
  if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess) {
    set_error("hipStreamCreateWithFlags failed");
    return fail(TEA_HIP_EHIP);
  }
  const size_t px = (size_t)max_batch * height * width;
  n->wg_blocks = 256;
  n->loss_len = px / 256 + 2;
  n->partial_len = (size_t)n->wg_blocks * (wgrad_offset(5) + wgrad_len(5));
  struct {
    void** p;
    size_t bytes;
  } bufs[] = {
      {(void**)&n->master, kNumParams * sizeof(float)},
      {(void**)&n->grad, kNumParams * sizeof(float)},
      {(void**)&n->adam_m, kNumParams * sizeof(float)},
      {(void**)&n->adam_v, kNumParams * sizeof(float)},
      {(void**)&n->wf1, (size_t)kWf1 * sizeof(bf16)},
      {(void**)&n->wfh, (size_t)4 * kWh * sizeof(bf16)},
      {(void**)&n->wbh, (size_t)4 * kWh * sizeof(bf16)},
      {(void**)&n->w6, kW6 * sizeof(float)},
      {(void**)&n->bias, (5 * kC + 1) * sizeof(float)},
      {(void**)&n->in_f32, px * kIn * sizeof(float)},
      {(void**)&n->in0, act_elems(n, kC0) * sizeof(bf16)},
      {(void**)&n->out, px * sizeof(float)},
      {(void**)&n->target, px * sizeof(float)},
      {(void**)&n->dout, px * sizeof(float)},
      {(void**)&n->partial, n->partial_len * sizeof(float)},
      {(void**)&n->loss_part, n->loss_len * sizeof(float)},
  };
  for (auto& b : bufs) {
    const int st = nn_alloc(b.p, b.bytes, n->stream);
    if (st != TEA_HIP_OK) return fail(st);
  }
  for (int l = 0; l < 5; ++l) {
    int st = nn_alloc((void**)&n->act[l], act_elems(n, kC) * sizeof(bf16), n->stream);
    if (st == TEA_HIP_OK && width <= kWgradMaxW)
      st = nn_alloc((void**)&n->del[l], act_elems(n, kC) * sizeof(bf16), n->stream);
    if (st != TEA_HIP_OK) return fail(st);
  }
  if (hipStreamSynchronize(n->stream) != hipSuccess) {
    set_error("hipStreamSynchronize failed");
    return fail(TEA_HIP_EHIP);
  }
  *out = n;
  return TEA_HIP_OK;
}

int tea_nn_destroy(tea_nn* n) {
  if (!n) return TEA_HIP_OK;
  (void)hipSetDevice(n->device);
  if (n->stream) (void)hipStreamSynchronize(n->stream);
  void* ptrs[] = {n->master, n->grad, n->adam_m, n->adam_v, n->wf1, n->wfh, n->wbh,
                  n->w6, n->bias, n->in_f32, n->in0, n->out, n->target, n->dout,
                  n->partial, n->loss_part, n->ds_in, n->ds_tgt, n->ds_order};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  for (int l = 0; l < 5; ++l) {
    if (n->act[l]) (void)hipFree(n->act[l]);
    if (n->del[l]) (void)hipFree(n->del[l]);
  }
  if (n->stream) (void)hipStreamDestroy(n->stream);
  delete n;
  return TEA_HIP_OK;
}

int tea_nn_set_params(tea_nn* n, const float* host, size_t count) {
  NN_CHECK(n);
  TEA_CHECK_ARG(host && count == (size_t)kNumParams, "need exactly tea_nn_num_params() values");
  TEA_HIP_TRY(hipSetDevice(n->device));
  TEA_HIP_TRY(hipMemcpyAsync(n->master, host, count * sizeof(float),
                             hipMemcpyHostToDevice, n->stream));
  TEA_HIP_TRY(hipMemsetAsync(n->adam_m, 0, count * sizeof(float), n->stream));
  TEA_HIP_TRY(hipMemsetAsync(n->adam_v, 0, count * sizeof(float), n->stream));
  n->adam_t = 0;
  TEA_RETURN_IF(pack_params(n));
  TEA_HIP_TRY(hipStreamSynchronize(n->stream));
  return TEA_HIP_OK;
}

int tea_nn_get_params(tea_nn* n, float* host, size_t count) {
  NN_CHECK(n);
  TEA_CHECK_ARG(host && count == (size_t)kNumParams, "need exactly tea_nn_num_params() values");
  TEA_HIP_TRY(hipSetDevice(n->device));
  TEA_HIP_TRY(hipMemcpyAsync(host, n->master, count * sizeof(float),
                             hipMemcpyDeviceToHost, n->stream));
  TEA_HIP_TRY(hipStreamSynchronize(n->stream));
  return TEA_HIP_OK;
}

int tea_nn_forward(tea_nn* n, int batch, const float* input, float* output) {
  NN_CHECK(n);
  TEA_CHECK_ARG(batch >= 1 && batch <= n->max_batch, "batch out of range");
  TEA_CHECK_ARG(input && output, "null arrays");
  TEA_HIP_TRY(hipSetDevice(n->device));
  TEA_RETURN_IF(upload_batch(n, batch, input, nullptr));
  TEA_RETURN_IF(forward(n, batch));
  TEA_HIP_TRY(hipMemcpyAsync(output, n->out, (size_t)batch * n->H * n->W * sizeof(float),
                             hipMemcpyDeviceToHost, n->stream));
  TEA_HIP_TRY(hipStreamSynchronize(n->stream));
  return TEA_HIP_OK;
}

int tea_nn_loss_grad(tea_nn* n, int batch, const float* input, const float* target,
                     float* loss, float* grad) {
  NN_CHECK(n);
  TEA_CHECK_ARG(batch >= 1 && batch <= n->max_batch, "batch out of range");
  TEA_CHECK_ARG(input && target, "null arrays");
  TEA_CHECK_ARG(n->del[0] != nullptr, "training needs width <= 128");
  TEA_HIP_TRY(hipSetDevice(n->device));
  TEA_RETURN_IF(upload_batch(n, batch, input, target));
  TEA_RETURN_IF(loss_and_grad(n, batch));
  if (grad)
    TEA_HIP_TRY(hipMemcpyAsync(grad, n->grad, kNumParams * sizeof(float),
                               hipMemcpyDeviceToHost, n->stream));
  float l = 0.0f;
  TEA_RETURN_IF(read_losses(n, batch, 1, &l));
  if (loss) *loss = l;
  return TEA_HIP_OK;
}

int tea_nn_train_step(tea_nn* n, int batch, const float* input, const float* target,
                      float lr, float* loss) {
  TEA_RETURN_IF(tea_nn_loss_grad(n, batch, input, target, loss, nullptr));
  TEA_RETURN_IF(adam_step(n, lr));
  TEA_HIP_TRY(hipStreamSynchronize(n->stream));
  return TEA_HIP_OK;
}

int tea_nn_adam_step(tea_nn* n, const float* grad, float lr) {
  NN_CHECK(n);
  TEA_CHECK_ARG(grad != nullptr, "null gradient");
  TEA_HIP_TRY(hipSetDevice(n->device));
  TEA_HIP_TRY(hipMemcpyAsync(n->grad, grad, kNumParams * sizeof(float),
                             hipMemcpyHostToDevice, n->stream));
  TEA_RETURN_IF(adam_step(n, lr));
  TEA_HIP_TRY(hipStreamSynchronize(n->stream));
  return TEA_HIP_OK;
}

int tea_nn_get_adam_state(tea_nn* n, float* m, float* v, size_t count, long long* step) {
  NN_CHECK(n);
  TEA_CHECK_ARG(m && v && step && count == (size_t)kNumParams,
                "need two arrays of tea_nn_num_params() values and a step counter");
  TEA_HIP_TRY(hipSetDevice(n->device));
  TEA_HIP_TRY(hipMemcpyAsync(m, n->adam_m, count * sizeof(float), hipMemcpyDeviceToHost,
                             n->stream));
  TEA_HIP_TRY(hipMemcpyAsync(v, n->adam_v, count * sizeof(float), hipMemcpyDeviceToHost,
                             n->stream));
  TEA_HIP_TRY(hipStreamSynchronize(n->stream));
  *step = n->adam_t;
  return TEA_HIP_OK;
}

int tea_nn_load_dataset(tea_nn* n, int count, const float* inputs, const float* targets) {
  NN_CHECK(n);
  TEA_CHECK_ARG(count >= 1 && inputs && targets, "empty dataset");
  TEA_HIP_TRY(hipSetDevice(n->device));
  if (n->ds_in) (void)hipFree(n->ds_in);
  if (n->ds_tgt) (void)hipFree(n->ds_tgt);
  if (n->ds_order) (void)hipFree(n->ds_order);
  n->ds_in = n->ds_tgt = nullptr;
  n->ds_order = nullptr;
  n->ds_n = 0;
  const size_t px = (size_t)n->H * n->W;
  TEA_RETURN_IF(nn_alloc((void**)&n->ds_in, (size_t)count * px * kIn * sizeof(float), n->stream));
  TEA_RETURN_IF(nn_alloc((void**)&n->ds_tgt, (size_t)count * px * sizeof(float), n->stream));
  TEA_RETURN_IF(nn_alloc((void**)&n->ds_order, (size_t)count * sizeof(int), n->stream));
  n->order_len = count;
  TEA_HIP_TRY(hipMemcpyAsync(n->ds_in, inputs, (size_t)count * px * kIn * sizeof(float),
                             hipMemcpyHostToDevice, n->stream));
  TEA_HIP_TRY(hipMemcpyAsync(n->ds_tgt, targets, (size_t)count * px * sizeof(float),
                             hipMemcpyHostToDevice, n->stream));
  TEA_HIP_TRY(hipStreamSynchronize(n->stream));
  n->ds_n = count;
  return TEA_HIP_OK;
}

// One pass over order[0..count) in batches of `batch` (a short last batch is
// dropped); Adam with learning rate lr; mean batch loss to *mean_loss.
int tea_nn_train_epoch(tea_nn* n, const int* order, int count, int batch, float lr,
                       float* mean_loss) {
  NN_CHECK(n);
  TEA_CHECK_ARG(n->ds_n > 0, "no dataset loaded");
  TEA_CHECK_ARG(n->del[0] != nullptr, "training needs width <= 128");
  TEA_CHECK_ARG(batch >= 1 && batch <= n->max_batch && count >= batch, "bad batch");
  TEA_HIP_TRY(hipSetDevice(n->device));
  for (int i = 0; i < count; ++i)
    TEA_CHECK_ARG(order[i] >= 0 && order[i] < n->ds_n, "sample index out of range");
  // An epoch may be longer than the set (samples drawn with repetition).
  if (count > n->order_len) {
    int* more = nullptr;
    TEA_RETURN_IF(nn_alloc((void**)&more, (size_t)count * sizeof(int), n->stream));
    (void)hipFree(n->ds_order);
    n->ds_order = more;
    n->order_len = count;
  }
  TEA_HIP_TRY(hipMemcpyAsync(n->ds_order, order, (size_t)count * sizeof(int),
                             hipMemcpyHostToDevice, n->stream));
  // The batches' loss partials stay on the device until the epoch's end: a
  // read back per batch left the GPU idle for 52 us of each 650 us step.
  const int steps = count / batch;
  const size_t need = (size_t)steps * loss_blocks(n, batch);
  if (need > n->loss_len) {
    float* more = nullptr;
    TEA_RETURN_IF(nn_alloc((void**)&more, need * sizeof(float), n->stream));
    (void)hipFree(n->loss_part);
    n->loss_part = more;
    n->loss_len = need;
  }
  const int px = n->H * n->W;
  for (int k = 0; k < steps; ++k) {
    hipLaunchKernelGGL(gather_kernel, dim3(flat_blocks((long)batch * px)), dim3(256), 0,
                       n->stream, n->ds_in, n->ds_tgt, n->ds_order + (size_t)k * batch, n->in0,
                       n->target, batch, n->H, n->W);
    TEA_HIP_TRY(hipGetLastError());
    TEA_RETURN_IF(loss_and_grad(n, batch, k));
    TEA_RETURN_IF(adam_step(n, lr));
  }
  std::vector<float> losses(steps);
  TEA_RETURN_IF(read_losses(n, batch, steps, losses.data()));
  double total = 0.0;
  for (float l : losses) total += l;
  if (mean_loss) *mean_loss = (float)(total / (steps ? steps : 1));
  return TEA_HIP_OK;
}

}  // extern "C"
