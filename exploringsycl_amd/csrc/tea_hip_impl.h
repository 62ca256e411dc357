// Internal declarations of libteahip.so: the chunk handle, launch helpers
// and the device-side reduction machinery shared by the kernel files.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <unordered_map>
#include <vector>

#include "tea_hip.h"

namespace tea {

// ---------------------------------------------------------------------------
// Errors

void set_error(const std::string& msg);

#define TEA_HIP_TRY(call)                                                     \
  do {                                                                        \
    hipError_t err_ = (call);                                                 \
    if (err_ != hipSuccess) {                                                 \
      ::tea::set_error(std::string(#call) + " failed: " +                     \
                       hipGetErrorString(err_) + " (" + __FILE__ + ":" +      \
                       std::to_string(__LINE__) + ")");                       \
      return TEA_HIP_EHIP;                                                    \
    }                                                                         \
  } while (0)

#define TEA_CHECK_ARG(cond, msg)                                              \
  do {                                                                        \
    if (!(cond)) {                                                            \
      ::tea::set_error(std::string(__func__) + ": " + (msg));                 \
      return TEA_HIP_EINVAL;                                                  \
    }                                                                         \
  } while (0)

#define TEA_RETURN_IF(status)                                                 \
  do {                                                                        \
    int st_ = (status);                                                       \
    if (st_ != TEA_HIP_OK) return st_;                                        \
  } while (0)

// ---------------------------------------------------------------------------
// Geometry of a chunk and fast division by its row length.

// Division by a runtime constant d (1 <= d < 2^31) for n < 2^31 with one
// multiply-high: q = (umulhi(n, m) + n) >> s, s = ceil(log2 d),
// m = floor(2^32 (2^s - d) / d) + 1 (Granlund & Montgomery 1994, sec. 4).
struct FastDiv {
  uint32_t d = 1, m = 0, s = 0;
  FastDiv() = default;
  explicit FastDiv(uint32_t divisor) : d(divisor) {
    s = 0;
    while ((uint64_t(1) << s) < d) ++s;
    m = uint32_t(((uint64_t(1) << 32) * ((uint64_t(1) << s) - d)) / d + 1);
  }
  __host__ __device__ inline uint32_t div(uint32_t n) const {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t t = __umulhi(n, m);
#else
    const uint32_t t = uint32_t((uint64_t(n) * m) >> 32);
#endif
    return uint32_t((uint64_t(t) + n) >> s);
  }
};

struct Geo {
  int x, y, h;
  int n;      // x*y
  FastDiv dx; // division by x
  int nt = 1, nt_half = 1;  // streaming access (kStreamCells)
  int bands = 0;  // FP64 passes in XCD bands (band_index)
};

__device__ inline bool interior(const Geo& g, int kk, int jj) {
  return kk >= g.h && kk < g.x - g.h && jj >= g.h && jj < g.y - g.h;
}

// ---------------------------------------------------------------------------
// Launch shape.  A "span" is 4096 consecutive linear cells = 64 groups of 64:
// exactly one level-2 partial of the reference's reduction tree.  A span is
// processed by one 256-thread block (4 wave64s), 16 cells per thread, with
// cell index base + k*256 + threadIdx.x, so wave w's k-th cell set is group
// 4k+w of the span.

constexpr int kWave = 64;
constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;
constexpr int kItems = 16;
constexpr int kSpan = kBlock * kItems;  // 4096
constexpr int kNumXcd = 8;              // MI355X: 8 XCDs, one L2 each

// Blocks are dispatched round-robin over the XCDs (block b -> XCD b % 8).
// Renumber them so each XCD walks one contiguous range of spans: the rows a
// stencil reads above and below were then fetched by the same XCD, into the
// same L2, moments earlier.
__device__ inline int xcd_span(int b, int nb) {
  const int xcd = b % kNumXcd, idx = b / kNumXcd;
  const int per = nb / kNumXcd, rem = nb % kNumXcd;
  return xcd * per + (xcd < rem ? xcd : rem) + idx;
}

// From how many cells on the passes stream (ld2_nt): where an iteration's
// arrays outgrow the 256 MB Infinity Cache.  FP64 CG (about 80 bytes per cell)
// per iteration, streaming against plain: 1000^2 22.1, 20.3 us, 1700^2 47.8,
// 46.0, 1800^2 52.5, 52.2, 1900^2 56.6, 57.7, 3000^2 137.4, 149.8.  Jacobi and
// the FP32 passes (half): Jacobi 1000^2 10.5, 8.8, 2400^2 47.2, 44.1, 2800^2
// 60.1, 65.6; mixed precision 1400^2 27.9, 25.9, 2400^2 57.8, 56.6, 2800^2
// 76.4, 79.0.
constexpr int kStreamCells = 3200000, kStreamCellsHalf = 6200000;

// The workgroup's place in a pair- or quad-per-thread pass: in segments of
// 8 * kBandBlocks blocks each XCD takes kBandBlocks consecutive blocks, so a
// row is re-read, as the row above or below, from the L2 that read it first,
// passes find in it what the pass before wrote, and the chip still streams
// through memory as one front (one band per XCD over the whole grid: 4-7%
// slower from 4096^2 on).  In launch order each row comes into up to three
// L2s.  FP64 CG per iteration, launch order against bands of 128 blocks (64
// and 256 within 1%): 1000^2 24.6 -> 21.5 us, 1500^2 50.9 -> 39.8, 3000^2 166.6
// -> 138.6, 6000^2 612 -> 534; Jacobi sweeps 2048^2 44.5 -> 38.7; mixed
// precision 1024^2 22.8 -> 20.9, 3001x2999 119.1 -> 105.2, 4096^2 158.1 ->
// 156.4.
// KS: blocks per workgroup (stacked_block).
constexpr int kBandBlocks = 128;
template <int KS = 1>
__device__ inline int band_index(bool bands = true) {
  if (!bands) return (int)blockIdx.x;
  constexpr int seg_len = kNumXcd * kBandBlocks / KS;
  const int seg = (int)blockIdx.x / seg_len * seg_len, left = (int)gridDim.x - seg;
  return seg + xcd_span((int)blockIdx.x - seg, left < seg_len ? left : seg_len);
}
// FP64 passes keep the launch order where rows are 8 blocks (or a multiple)
// and up to an eighth of a block long: all but that share of the cells above
// and below a block then lie on its own XCD anyway, and the plain front is
// faster.  CG per iteration, launch order against bands: x = 4100 239.1, 240.8
// us, 4156 242.4, 243.4, 8196 476.5, 483.2, 8252 478.9, 486.4; past the line 4176
// 240.1, 240.3, 4200 243.6, 242.6, 8300 481.3, 485.3, 8400 486.5, 480.0, 4352
// 251.1, 240.6; below whole rows 4080 250.7, 236.4.  (The crossing lies at 80 to
// 150 cells, later with longer rows.)
inline int bands_for(int x) {
  const int row = kNumXcd * 512;
  return x < row || x % row > 512 / 8;
}

// Cross-lane moves on the VALU's data-parallel-primitive (DPP) path instead
// of LDS permutes.  CTRL is a DPP control: 0x130 wave_shl:1 (lane l takes
// lane l+1), 0x138 wave_shr:1 (lane l takes lane l-1), 0xB1 and 0x4E
// quad_perm [1,0,3,2] and [2,3,0,1] (lane l takes lane l^1, l^2), 0x141
// row_half_mirror (lane i of each 8 takes lane 7-i), 0x140 row_mirror (lane
// i of each 16 takes lane 15-i).  A lane without a source keeps its value.
template <int CTRL>
__device__ inline float dpp(float v) {
  const int b = __float_as_int(v);
  return __int_as_float(__builtin_amdgcn_update_dpp(b, b, CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ inline double dpp(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xF, 0xF, false),
                          __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xF, 0xF, false));
}
template <class T>
__device__ inline T from_next_lane(T v) { return dpp<0x130>(v); }
template <class T>
__device__ inline T from_prev_lane(T v) { return dpp<0x138>(v); }

// The value of lane `l` (a constant), in every lane.
__device__ inline double lane_value(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Pairwise tree of 64 lanes (lane l <- lane l^m for m = 1..32).  After the
// step with mask m every lane of an aligned block of 2m lanes holds the same
// value, the tree sum of that block, so the result equals the reference's
// "a[2s*l] += a[2s*l+s]" tree bit for bit (IEEE addition commutes exactly).
__device__ inline double wave_tree(double v) {
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) v = v + __shfl_xor(v, m);
  return v;
}

// Level-1 trees of the 16 groups a thread's wave holds (value k of lane l is
// cell l of group k), with the values transposed across lanes as the tree
// goes so each butterfly step moves half as many values as the last: after
// steps m = 1, 2, 4, 8 lane l holds one group, k = bitreverse4(l & 15), and
// steps 16 and 32 finish it.  Each step still adds the two aligned halves of
// a block, so every sum is the reference tree's.  Returns, in lanes 0..15,
// the level-1 partial of group bitreverse4(lane).
__device__ inline double wave_tree16(double (&v)[kItems]) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int step = 0; step < 4; ++step) {
    const int m = 1 << step;
    const int half = kItems >> (step + 1);
    const bool upper = (lane & m) != 0;
#pragma unroll
    for (int i = 0; i < half; ++i) {
      const double send = upper ? v[i] : v[half + i];
      const double keep = upper ? v[half + i] : v[i];
      v[i] = keep + __shfl_xor(send, m);
    }
  }
  double s = v[0];
  s = s + __shfl_xor(s, 16);
  s = s + __shfl_xor(s, 32);
  return s;
}

__device__ inline int bitrev4(int l) {
  return ((l & 1) << 3) | ((l & 2) << 1) | ((l & 4) >> 1) | ((l & 8) >> 3);
}

// Reduces the 16 values per thread of one span (NR independent sums) to the
// span's level-2 partials and stores them at partials[q*nspan + span].
// `single_group` (the whole field is one group of 64) stores the level-1
// value instead, as the reference's reduceArray then runs no pass at all.
template <int NR>
__device__ inline void span_reduce(double (&v)[NR][kItems], double* partials,
                                   int nspan, int span, bool single_group) {
  __shared__ double lds[NR][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave;
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    const double t = wave_tree16(v[q]);
    if (lane < kItems) lds[q][bitrev4(lane) * kWaves + wv] = t;
  }
  __syncthreads();
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const double level1 = lds[q][lane];
      const double t = single_group ? lds[q][0] : wave_tree(level1);
      if (lane == 0) partials[q * nspan + span] = t;
    }
  }
}


// ---- two cells per lane ---------------------------------------------------
//
// Kernels over cell pairs (2m, 2m+1), m = lane index within a 512-cell slot:
// every pair starts on an aligned boundary, so each operand is
// one 8-byte (FP32) or 16-byte (FP64) load, and the left/right neighbours
// come from the adjacent lanes (lane l-1 holds 2m-1, lane l+1 holds 2m+2);
// only lanes 0 and 63 load theirs.  With x even a pair lies in one row and
// the pairs above and below are aligned too.  With x odd every other row's
// pairs are shifted by one cell: the rows above and below are read with
// loads that need only element alignment (ld2u), and a pair may hold the last
// cell of a row and the first of the next, neither of which is interior.
// The last pair of an odd number of cells has no second cell; x*y buffers
// hold room for it (pair_bytes).  A wave covers 128 consecutive cells =
// two groups of the reduction tree (lanes 0-31 and 32-63); a 256-thread
// block covers a 4096-cell span in 8 slots of 512 cells.  The first tree
// level is the in-lane pair sum, then the butterfly runs over each 32-lane
// half.

constexpr int kSlots = kSpan / (2 * kBlock);  // 8

__device__ inline double2 ld2(const double* p, int i) {
  return *reinterpret_cast<const double2*>(p + i);
}

__device__ inline float2 ld2(const float* p, int i) {
  return *reinterpret_cast<const float2*>(p + i);
}

// The same at an index that may be odd (global loads need only 4-byte
// alignment): on an even index the instruction is ld2's.
__device__ inline double2 ld2u(const double* p, int i) {
  typedef double vec2 __attribute__((ext_vector_type(2), aligned(8)));
  const vec2 v = *reinterpret_cast<const vec2*>(p + i);
  return double2{v.x, v.y};
}

__device__ inline float2 ld2u(const float* p, int i) {
  typedef float vec2 __attribute__((ext_vector_type(2), aligned(4)));
  const vec2 v = *reinterpret_cast<const vec2*>(p + i);
  return float2{v.x, v.y};
}

// An even index whose pair, the pairs one row up and down and the cells
// next to it are in range (y >= 3).
__device__ inline int safe_pair(int x) { return (x + 2) & ~1; }

// Bytes of an x*y buffer that pair kernels use.
inline size_t pair_bytes(long n, size_t elem) { return (size_t)((n + 1) & ~1L) * elem; }

// Stores a cell pair with one vector store, or the interior member alone.
template <class T>
__device__ inline void st2(T* p, int i, bool in0, bool in1, T v0, T v1) {
  if (in0 && in1) {
    typedef T vec2 __attribute__((ext_vector_type(2)));
    *reinterpret_cast<vec2*>(p + i) = vec2{v0, v1};
  } else {
    if (in0) p[i] = v0;
    if (in1) p[i + 1] = v1;
  }
}

__device__ inline int bitrev3(int l) {
  return ((l & 1) << 2) | (l & 2) | ((l & 4) >> 2);
}

// Level-1 trees of the 8 slot pair-sums of a lane, transposed across lanes
// as in wave_tree16 (steps 1, 2, 4), then steps 8 and 16 within each 32-lane
// half; stores each group's partial in lds[q][group-in-span] and finishes
// the span's level-2 trees in wave 0 (partials[q * nspan + span]).
template <int NR>
__device__ inline void span_reduce_pairs_n(double (&v)[NR][kSlots], double* partials,
                                           int nspan, int span, bool single_group) {
  __shared__ double lds[NR][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave;
#pragma unroll
  for (int q = 0; q < NR; ++q) {
#pragma unroll
    for (int step = 0; step < 3; ++step) {
      const int m = 1 << step;
      const int half = kSlots >> (step + 1);
      const bool upper = (lane & m) != 0;
#pragma unroll
      for (int i = 0; i < half; ++i) {
        const double send = upper ? v[q][i] : v[q][half + i];
        const double keep = upper ? v[q][half + i] : v[q][i];
        v[q][i] = keep + __shfl_xor(send, m);
      }
    }
    double t = v[q][0];
    t = t + __shfl_xor(t, 8);
    t = t + __shfl_xor(t, 16);
    if ((lane & 31) < kSlots)
      lds[q][bitrev3(lane & 7) * 8 + wv * 2 + (lane >> 5)] = t;
  }
  __syncthreads();
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const double r = single_group ? lds[q][0] : wave_tree(lds[q][lane]);
      if (lane == 0) partials[q * nspan + span] = r;
    }
  }
}
// Streaming (nontemporal) access for data read or written once per pass
// and not read again before the next iteration (u, p_new, and the residual
// pass's r); stencil operands (p, r, kx, ky) use ld2 so the neighbouring rows
// can reuse them from L2, and w, which the residual pass reads next, is
// stored normally so that it can stay in the 256 MB Infinity Cache (storing
// it streaming made that pass 1-12% slower).  With nt = 0 they are plain:
// an iteration's arrays that fit in that cache are read back from it.
typedef double dvec2 __attribute__((ext_vector_type(2)));

__device__ inline double2 ld2_nt(const double* p, int i, int nt = 1) {
  if (!nt) return ld2(p, i);
  const dvec2 v = __builtin_nontemporal_load(reinterpret_cast<const dvec2*>(p + i));
  return double2{v.x, v.y};
}

// Stores a cell pair with one 16-byte streaming store, or the interior
// member alone.
__device__ inline void st2_nt(double* p, int i, bool in0, bool in1, double v0,
                              double v1, int nt = 1) {
  if (!nt) {
    if (in0 && in1) {
      *reinterpret_cast<dvec2*>(p + i) = dvec2{v0, v1};
    } else {
      if (in0) p[i] = v0;
      if (in1) p[i + 1] = v1;
    }
    return;
  }
  if (in0 && in1) {
    __builtin_nontemporal_store(dvec2{v0, v1}, reinterpret_cast<dvec2*>(p + i));
  } else {
    if (in0) __builtin_nontemporal_store(v0, p + i);
    if (in1) __builtin_nontemporal_store(v1, p + i + 1);
  }
}

// The FP32 pair store of the mixed-precision kernels.
typedef float fvec2 __attribute__((ext_vector_type(2)));

__device__ inline void st2_nt(float* p, int i, bool in0, bool in1, float v0,
                              float v1, int nt = 1) {
  if (!nt) {
    if (in0 && in1) {
      *reinterpret_cast<fvec2*>(p + i) = fvec2{v0, v1};
    } else {
      if (in0) p[i] = v0;
      if (in1) p[i + 1] = v1;
    }
    return;
  }
  if (in0 && in1) {
    __builtin_nontemporal_store(fvec2{v0, v1}, reinterpret_cast<fvec2*>(p + i));
  } else {
    if (in0) __builtin_nontemporal_store(v0, p + i);
    if (in1) __builtin_nontemporal_store(v1, p + i + 1);
  }
}

// ---- one pair per thread ---------------------------------------------------
//
// A 256-thread block over 512 consecutive cells = 8 groups of the reduction
// tree, one cell pair per lane.  The reference's level-2 tree over a span's
// 64 level-1 partials (sycl_shared.hpp:59-64: a[2s*l] += a[2s*l + s] for
// s = 1, 2, 4, ...) sums aligned runs of 8 leaves before it combines them, so
// a block's 8-leaf subtree is an exact intermediate of that tree: blocks
// store it in sub[q * sub_stride + block], and span_finish_kernel (or, for
// small grids, the next pass itself: consume_sums) combines them.
//
// Which block a workgroup takes: band_index.

constexpr int kPairBlock = 2 * kBlock;              // 512 cells
constexpr int kSubPerSpan = kSpan / kPairBlock;     // 8
constexpr int kSubMaxNr = 4;                        // dot products per launch

// Length of one dot product's block sums: the blocks rounded up to whole
// groups of 512 (64 spans), the cells past the grid's blocks zero for good.
constexpr int kGroupBlocks = kSubPerSpan * kWave;   // 512
__host__ __device__ inline int sub_stride(int nblk) {
  return (nblk + kGroupBlocks - 1) / kGroupBlocks * kGroupBlocks;
}

// wave_tree with the steps within 16 lanes on the DPP path (after each, every
// lane of an aligned block holds the block's sum; the mirrors pair whole
// blocks of equal lanes); the sum in every lane.
__device__ inline double wave_tree_dpp(double t) {
  t = t + dpp<0xB1>(t);
  t = t + dpp<0x4E>(t);
  t = t + dpp<0x141>(t);
  t = t + dpp<0x140>(t);
  return (lane_value(t, 0) + lane_value(t, 16)) + (lane_value(t, 32) + lane_value(t, 48));
}

// Stores the sum of each of a workgroup's KS blocks of NW waves from the
// lanes' values v (the in-lane sums: tree step 1 for pairs, 1 and 2 for
// quads).  tid is the thread in its block; blk may lie past the grid.  Every
// wave of the workgroup calls it.
template <int NR, int NW, int KS>
__device__ inline void store_block_sums(const double (&v)[NR], double* sub, int nblk, int blk,
                                        int tid) {
  static_assert(NW == 2 || NW == 4, "waves per block");
  __shared__ double ws[KS][NR][NW];
  const int slot = KS == 1 ? 0 : (int)threadIdx.x / (NW * kWave);
  const int wv = tid / kWave;
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    const double t = wave_tree_dpp(v[q]);
    if ((threadIdx.x & (kWave - 1)) == 0) ws[slot][q][wv] = t;
  }
  __syncthreads();
  if (tid >= NR || blk >= nblk) return;
  double s = ws[slot][tid][0] + ws[slot][tid][1];
  if (NW == 4) s = s + (ws[slot][tid][NW - 2] + ws[slot][tid][NW - 1]);
  sub[(size_t)tid * sub_stride(nblk) + blk] = s;
}
template <int NR, int KS = 1>
__device__ inline void block_sums_pairs(const double (&v)[NR], double* sub, int nblk, int blk,
                                        int tid) {
  store_block_sums<NR, kWaves, KS>(v, sub, nblk, blk, tid);
}

// ---- four cells per lane ---------------------------------------------------
//
// A 128-thread block over one 512-cell pair block, four cells per lane (x a
// multiple of 4, so a quad never straddles a row and every quad, and the
// quads one row up and down, are 16-byte aligned).  The block covers the
// cells of a pair block, so that the same XCD has them in both kinds of pass.
// The in-lane sum ((v0 + v1) + (v2 + v3)) is tree steps 1 and 2; the four DPP
// steps of wave_tree_dpp then finish a 64-cell group in each 16-lane row, and (g0 + g1) + (g2 + g3)
// is the sum pair waves 2w and 2w + 1 combine to: the same tree, bit for bit.

constexpr int kQuadThreads = kPairBlock / 4;  // 128
constexpr int kQuadBlock = kPairBlock;        // 512 cells

__device__ inline float4 ld4(const float* p, int i) {
  return *reinterpret_cast<const float4*>(p + i);
}

__device__ inline float q_at(const float4& v, int c) {
  return c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
}

typedef float fvec4 __attribute__((ext_vector_type(4)));

// Stores a quad with one 16-byte store, or its interior members alone.
__device__ inline void st4(float* p, int i, const bool (&in)[4], const float (&v)[4]) {
  if (in[0] && in[1] && in[2] && in[3]) {
    *reinterpret_cast<fvec4*>(p + i) = fvec4{v[0], v[1], v[2], v[3]};
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (in[c]) p[i + c] = v[c];
  }
}

__device__ inline void st4(float* p, int i, const bool (&in)[4], fvec4 v) {
  if (in[0] && in[1] && in[2] && in[3]) {
    *reinterpret_cast<fvec4*>(p + i) = v;
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (in[c]) p[i + c] = v[c];
  }
}

// The same with streaming stores.
__device__ inline void st4_nt(float* p, int i, const bool (&in)[4], fvec4 v,
                              int nt = 1) {
  if (!nt) return st4(p, i, in, v);
  if (in[0] && in[1] && in[2] && in[3]) {
    __builtin_nontemporal_store(v, reinterpret_cast<fvec4*>(p + i));
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (in[c]) __builtin_nontemporal_store(v[c], p + i + c);
  }
}

__device__ inline void st4_nt(float* p, int i, const bool (&in)[4], const float (&v)[4],
                              int nt = 1) {
  if (!nt) return st4(p, i, in, v);
  if (in[0] && in[1] && in[2] && in[3]) {
    __builtin_nontemporal_store(fvec4{v[0], v[1], v[2], v[3]}, reinterpret_cast<fvec4*>(p + i));
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (in[c]) __builtin_nontemporal_store(v[c], p + i + c);
  }
}

template <int NR, int KS = 1>
__device__ inline void block_sums_quads(const double (&v)[NR], double* sub, int nblk, int blk,
                                        int tid) {
  store_block_sums<NR, kQuadThreads / kWave, KS>(v, sub, nblk, blk, tid);
}

// The sums a pass before this one left in sub, formed by every block of this
// pass for itself (up to four waves load, every thread gets the sums):
// with up to 2048 blocks (4 groups) the reference's remaining passes are one
// pairwise tree over the zero-padded block sums.  It saves the finisher's
// launch (3.4-4.2 us) between two dependent passes: an FP64 CG iteration at
// 512^2 takes 17.9 us with it and 22.7 us with finishers.  (Counting the
// blocks done and letting the last one finish the sum inside its own kernel
// took 26 us: the count of 512 blocks on 8 XCDs is a serial chain of about
// 18 ns each.)  Beyond 2048 blocks, more than the chip holds at once, each
// further round of blocks would repeat the sum, and the finisher stays.
constexpr int kConsumeBlocks = 4 * kGroupBlocks;
template <int NR>
__device__ inline void consume_sums(const double* __restrict__ sub, int nblk,
                                    double (&sum)[NR]) {
  __shared__ double gs[NR][4];
  const int lane = threadIdx.x & (kWave - 1);
  const int stride = sub_stride(nblk), waves = blockDim.x / kWave;
  for (int g = threadIdx.x / kWave; g < 4; g += waves) {
    const int i0 = kGroupBlocks * g + kSubPerSpan * lane;
    double t[NR];
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      t[q] = 0.0;
      if (i0 < stride) {
        const double* p = sub + (size_t)q * stride + i0;
        const double2 a = ld2(p, 0), b = ld2(p, 2), c = ld2(p, 4), d = ld2(p, 6);
        t[q] = ((a.x + a.y) + (b.x + b.y)) + ((c.x + c.y) + (d.x + d.y));
      }
    }
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const double s = wave_tree_dpp(t[q]);
      if (lane == 0) gs[q][g] = s;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NR; ++q) sum[q] = (gs[q][0] + gs[q][1]) + (gs[q][2] + gs[q][3]);
}

// The cell pair (e, e + 1) of a pair-per-thread lane, e = 512 b + 2 m for
// lane m of block b.
struct PairAt {
  int e;          // first cell
  bool valid;     // e < x*y
  bool in0, in1;  // interior cells
  int kk, row;    // column and row of e
  int ic;         // e if valid, else a safe even index (safe_pair)
  int ir;         // e if either cell is interior, else the safe index
};

__device__ inline PairAt pair_at(const Geo& g, int e) {
  PairAt q;
  q.e = e;
  q.valid = e < g.n;
  q.row = q.valid ? (int)g.dx.div((uint32_t)e) : 0;
  q.kk = e - q.row * g.x;
  q.in0 = q.valid && interior(g, q.kk, q.row);
  q.in1 = q.valid && interior(g, q.kk + 1, q.row);
  q.ic = q.valid ? e : safe_pair(g.x);
  q.ir = (q.in0 || q.in1) ? e : safe_pair(g.x);
  return q;
}

// The reflection of an interior cell's new value v onto the depth-1 halo
// ring where the cell borders it (kc, rc its column and row).
template <class T>
__device__ inline void ring_store(T* f, int i, int kc, int rc, int x, int xl, int xr, int yb,
                                  int yt, T v) {
  const bool L = kc == xl, Rg = kc == xr, B = rc == yb, Tp = rc == yt;
  if (!(L | Rg | B | Tp)) return;
  if (L) f[i - 1] = v;
  if (Rg) f[i + 1] = v;
  if (B) f[i - x] = v;
  if (Tp) f[i + x] = v;
  if (L && B) f[i - 1 - x] = v;
  if (Rg && B) f[i + 1 - x] = v;
  if (L && Tp) f[i - 1 + x] = v;
  if (Rg && Tp) f[i + 1 + x] = v;
}

// One block per span: each thread evaluates `body` on its 16 cells (only
// interior cells; everything else contributes +0.0, as in the reference) and
// the block stores the span's NR level-2 partials.
template <int NR, class Body>
__global__ __launch_bounds__(kBlock) void span_kernel(Geo g, Body body,
                                                      double* partials,
                                                      int nspan,
                                                      int single_group) {
  const int span = xcd_span(blockIdx.x, gridDim.x);
  const int base = span * kSpan;
  double v[NR][kItems];
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    const int e = base + k * kBlock + threadIdx.x;
    double out[NR];
#pragma unroll
    for (int q = 0; q < NR; ++q) out[q] = 0.0;
    if (e < g.n) {
      const int jj = (int)g.dx.div((uint32_t)e);
      const int kk = e - jj * g.x;
      if (interior(g, kk, jj)) body(e, kk, jj, out);
    }
#pragma unroll
    for (int q = 0; q < NR; ++q) v[q][k] = out[q];
  }
  span_reduce<NR>(v, partials, nspan, span, single_group != 0);
}

// The same sums with one cell pair per thread and the block's sums in sub (for
// a finisher): 16 cells' values of four sums per thread did not fit in
// registers (528 bytes of scratch per lane: 290 us for the field summary at
// 4096^2, and a 140 us wait for the scratch memory before it at any size).
template <int NR, class Body>
__global__ __launch_bounds__(kBlock) void pair_sum_kernel(Geo g, Body body, double* sub,
                                                          int nblk) {
  const int blk = band_index(g.bands);
  const PairAt q = pair_at(g, blk * kPairBlock + 2 * threadIdx.x);
  double a[NR], b[NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) a[k] = b[k] = 0.0;
  if (q.in0) body(q.e, q.kk, q.row, a);
  if (q.in1) body(q.e + 1, q.kk + 1, q.row, b);
#pragma unroll
  for (int k = 0; k < NR; ++k) a[k] = a[k] + b[k];
  block_sums_pairs<NR>(a, sub, nblk, blk, threadIdx.x);
}

// One thread per cell of the padded x*y range.
template <class Body>
__global__ __launch_bounds__(kBlock) void each_kernel(Geo g, Body body) {
  const int e = blockIdx.x * kBlock + threadIdx.x;
  if (e >= g.n) return;
  const int jj = (int)g.dx.div((uint32_t)e);
  const int kk = e - jj * g.x;
  body(e, kk, jj);
}

// ---------------------------------------------------------------------------
// Kernel identifiers for timing.

enum KernelId {
  K_SET_CHUNK_DATA = 0,
  K_SET_CHUNK_STATE,
  K_STORE_ENERGY,
  K_LOCAL_HALOS,
  K_FIELD_SUMMARY,
  K_CG_INIT_U,
  K_CG_INIT_K,
  K_CG_INIT_OTHERS,
  K_CG_CALC_W,
  K_CG_CALC_UR,
  K_CG_CALC_P,
  K_CG_FUSED_W,
  K_CG_FUSED_R,
  K_CG_APPLY_PENDING,
  K_COPY_U,
  K_CALC_RESIDUAL,
  K_CALC_2NORM,
  K_FINALISE,
  K_MP_CONVERT,
  K_MP_W,
  K_MP_R,
  K_MP_APPLY_U,
  K_MP_REFRESH,
  K_FCG_W,
  K_FCG_JACOBI,
  K_FCG_RESTRICT,
  K_FCG_NET,
  K_FCG_PROLONG,
  K_SPAN_FINISH,
  K_JACOBI_INIT,
  K_JACOBI_COPY_U,
  K_JACOBI_ITERATE,
  K_JACOBI_FUSED,
  K_CHEBY_INIT,
  K_CHEBY_ITERATE,
  K_CHEBY_CALC_U,
  K_CHEBY_FUSED,
  K_PPCG_INIT,
  K_PPCG_CALC_UR,
  K_PPCG_CALC_SD,
  K_PPCG_FUSED,
  K_PPCG_TWO_STEP,
  K_CHEBY_TWO_STEP,
  K_FCG_SWEEPS,
  K_CG_RA_FINISH,
  K_NUM
};

extern const char* const kKernelNames[K_NUM];

}  // namespace tea

namespace tea {

// Arguments of the mixed-precision stencil kernel (mpcg.hip), shared with
// flexible CG (fcg.hip).
struct MpArgs {
  const float* p_old;
  float* p_new;
  const float* r;     // added to beta p_old (the residual, or z for FCG)
  double* u;
  float* w;
  const float* kx;
  const float* ky;
  const float* rdot;  // second dot product p.rdot (DOT2 only)
  double alpha, beta;
  int apply_u, apply_p;
  // Held updates applied first (mp_w4_kernel, UM 3): u += alpha_h p_h,
  // then u += alpha_h2 p_h2.
  const float* p_h;
  const float* p_h2;
  double alpha_h, alpha_h2;
  // Pair-per-thread and four-cell kernels: the new u goes to u_out (u, or a
  // spare buffer when the iteration runs ahead).
  double* u_out;
  // Those kernels only: the alpha of u's update, where the device has it.
  const double* alpha_dev;
};

// Arguments of the FP64 w-step kernels (cg.hip).
struct FusedWArgs {
  const double* p_old;
  double* p_new;
  const double* r;
  double* u;
  double* w;
  const double* kx;
  const double* ky;
  double alpha, beta;
  int apply_u, ring;
  // Pair-per-thread kernel only: the new u goes to u_out (u itself for the
  // iteration the host asked for, a spare buffer when it runs ahead); its
  // alpha is *alpha_dev where that is set; held updates made first (UM 3):
  // u += alpha_h p_h, then u += alpha_h2 p_h2.
  double* u_out;
  const double* alpha_dev;
  const double* p_h;
  const double* p_h2;
  double alpha_h, alpha_h2;
};

// Where a pass of the iteration takes its scalar from: the host's value
// (dev null), the device's (dev: a finisher of the run-ahead left it there),
// or, with CONSUME, the block sums sub of the pass before it, which every
// block reduces for itself; the first block then leaves the scalar and the
// sum for the next pass and the host.  alpha = rro / sum (r-step), beta =
// sum / rro (w-step); rro is *rro_dev where that is set, else the value.
// Mixed-precision CG and FCG take two sums: (p.w, p.r) give alpha = p.r /
// p.w, (r.r, r.w or z.w) give beta = -r.w / p.w with p.w in rro.
struct RaScalar {
  const double* dev = nullptr;
  const double* sub = nullptr;
  int nblk = 0, inverse = 0;
  double rro = 0.0;
  const double* rro_dev = nullptr;
  double* sum_dev = nullptr;  // left for the next passes: by the w-step r.r (the
                              // next alpha's rro), by the r-step alpha (with
                              // two sums alpha and p.w)
  double* out = nullptr;      // host slot {sum(s), scalar}
};

template <int kBatch, bool DOT2>
__global__ void mp_w_kernel(Geo g, MpArgs a, double* partials, int nspan,
                            int single_group);
template <bool RW>
__global__ void mp_r_kernel(Geo g, float* r, const float* w, double alpha,
                            double* partials, int nspan, int single_group);
template <bool DOT2, int SB>
__global__ void mp_w2_kernel(Geo g, MpArgs a, double* partials, int nspan,
                             int single_group);
}  // namespace tea

struct tea_nn;

namespace tea {
namespace nn {
typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Stores one 32-pixel row of a layer's MFMA output (bias, ReLU, BF16) at
// px, the row's pixel of lane col: lane (hf, col) holds channels 8 g + 4 hf
// + 0..3, g = 0..3, of pixel col.  Lanes col and col + 32 swap half of
// theirs, so that each holds 16 consecutive channels (32 bytes at 16 hf),
// stored with two 16-byte stores (four 8-byte stores at a 64-byte stride
// each wrote the first layer's output at 1.5 TB/s).  Every lane takes part
// in the exchange; only lanes with ok store.
__device__ inline void store_out_row(bf16* px, const f32x16& acc, const float (&bco)[16],
                                     int hf, bool ok = true) {
  union Pack {
    bf16x4 v;
    unsigned u[2];
  };
  Pack o[4];
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float vv = acc[4 * g + q] + bco[4 * g + q];
      o[g].v[q] = (bf16)(vv > 0.0f ? vv : 0.0f);
    }
  // hf 0 keeps channels 0-3 and 8-11 and takes 4-7 and 12-15 (the
  // partner's g 0, 1); hf 1 keeps 20-23 and 28-31 and takes 16-19 and
  // 24-27 (the partner's g 2, 3).
  Pack in[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int w = 0; w < 2; ++w) in[j].u[w] = __shfl_xor(hf ? o[j].u[w] : o[2 + j].u[w], 32);
  union Pack8 {
    bf16x8 v;
    bf16x4 h[2];
  };
  Pack8 lo, hi;
  lo.h[0] = hf ? in[0].v : o[0].v;
  lo.h[1] = hf ? o[2].v : in[0].v;
  hi.h[0] = hf ? in[1].v : o[1].v;
  hi.h[1] = hf ? o[3].v : in[1].v;
  if (!ok) return;
  *reinterpret_cast<bf16x8*>(px + 16 * hf) = lo.v;
  *reinterpret_cast<bf16x8*>(px + 16 * hf + 8) = hi.v;
}

// The A operand of a layer's K-step t (lane l: output channel l % 32, the
// step's K-values 8 (l / 32) .. + 7), stored as the lanes take it: each load is
// one KiB in a row.  (From [co][tap][ci] a load touched 32 cache lines, and a
// hidden layer's 18 of them a wave: 64 x 32 x 32 8.9 us per layer.)
__device__ inline bf16x8 weight_frag(const bf16* __restrict__ wt, int t, int lane) {
  return *reinterpret_cast<const bf16x8*>(wt + (size_t)(t * kWave + lane) * 8);
}

// The network's device copies of its parameters, in the layouts of its
// forward kernels: layer 1 and the hidden layers in BF16 in fragment order
// (weight_frag), the output layer w6[tap][ci] (BF16 values in FP32) and the
// biases bias[layer * 32 + co], bias[160].
struct PackedWeights {
  const bf16* wf1;
  const bf16* wfh;
  const float* w6;
  const float* bias;
};
PackedWeights packed_weights(const tea_nn* n);
// The hidden layers alone, from layer `first` on (0-based; the caller has
// written layer first - 1's activations at hidden(n, first - 1)); the last
// layer's activations (padded (H + 2) x (W + 2) pixels of 32 BF16 channels,
// zero ring) at last_hidden.
int forward_hidden_on_stream(tea_nn* n, hipStream_t st, int first = 0);
// The same for two networks (one sample each), their layers in one launch;
// first >= 1.
int forward_hidden_pair(tea_nn* n0, tea_nn* n1, hipStream_t st, int first);
const bf16* last_hidden(tea_nn* n);
bf16* hidden(tea_nn* n, int l);
bf16* input_tensor(tea_nn* n);
const float* output(tea_nn* n);
}  // namespace nn
}  // namespace tea

// ---------------------------------------------------------------------------
// The chunk handle.

// The mixed-precision p buffers: a ring of four, so that a w-step can hold
// the u updates of two steps back and a w-step that runs ahead writes a
// buffer no update still needs (three, without the run-ahead, where there is
// no memory for the fourth).
constexpr int kMpRing = 4;

// One FP64 CG w-step on the pair kernels: its arguments, the u update it makes
// (um: none, its own where a.apply_u, or the two held ones and its own) and
// the updates held once it is taken over.
struct CgStep {
  tea::FusedWArgs a{};
  bool apply_p = false;
  int um = 1;
  int hold = 0;
  double* hold_p[2] = {};
  double hold_alpha[2] = {0.0, 0.0};
};

// One mixed-precision (or FCG) w-step on the pair or four-cell kernels: its
// arguments, the u update it makes (um: none, its own, or the two held ones
// and its own) and the updates held once it is taken over.
struct MpStep {
  tea::MpArgs a;
  int um = 0;
  int hold = 0;
  int hold_buf[2] = {0, 0};
  double hold_alpha[2] = {0.0, 0.0};
};

// One coarse level of the learned preconditioner.
struct FcgLevel {
  int c = 0, hc = 0, wc = 0;  // coarsening factor, coarse rows and columns
  tea_nn* net = nullptr;      // the network, sized hc x wc
  float* feat = nullptr;      // [2][hc][wc] normalised features
  float* rbar = nullptr;      // [hc][wc] block means of r
  float* kc = nullptr;        // [2][hc][wc] coarse left / bottom face coefficients
  float* dis = nullptr;       // [hc][wc] D^-1/2 of the coarse operator
  float* sig = nullptr;       // [hc][wc] local input scale of the network
  double* rms = nullptr;      // per-restriction-block sums of (D^-1/2 rbar)^2
  int nrms = 0;
  // The coarse solve's output y (network or Jacobi sweeps) and the
  // per-16x16-tile partials of y.rbar and y.T y (2 * ntiles).
  float* y = nullptr;
  double* tpart = nullptr;
  int ntiles = 0;
};
constexpr int kFcgMaxLevels = 2;

struct tea_hip_chunk {
  int device = 0;
  tea::Geo geo{};
  int nspan = 0;   // spans covering x*y (level-2 partial count)
  int ngroup = 0;  // groups of 64 covering x*y (level-1 partial count)
  hipStream_t stream = nullptr;

  double* field[TEA_NUM_FIELDS] = {};
  size_t field_len[TEA_NUM_FIELDS] = {};

  // Spare p buffers for the fused iteration (p is read as a stencil while the
  // new p is written; the first at creation, the others with the first
  // iteration, for the held updates below).  p_alt_synced: their cells
  // outside the interior and its ring equal p's.
  double* p_alt[3] = {};
  bool p_alt_synced = false;

  // Reduction workspace: up to 4 x nspan level-2 partials in pinned,
  // coherent host memory; kernels write through the device view.
  double* partials = nullptr;       // device view
  double* host_partials = nullptr;  // host view of the same memory
  // Block sums of the pair-per-thread kernels, kSubMaxNr x sub_stride(nblk),
  // device.  sub2: a second set (the same allocation), for a pass that reads
  // the sums of the pass before it while its own blocks write theirs.
  int nblk = 0;                     // 512-cell blocks covering x*y
  double* sub = nullptr;
  double* sub2 = nullptr;
  // Sums of the groups of 512 blocks and the finisher's count of blocks done
  // (zero between launches), for grids of more than 16 groups.
  double* grp_sum = nullptr;
  unsigned* done_count = nullptr;
  int pair_blocks = 3;              // pair-per-thread kernels: bit 0 fused_w,
                                    // bit 1 fused_r

  // Spare FP64 field buffer (x*y, allocated by the first Chebyshev or PPCG
  // call): the fused Chebyshev and PPCG steps write the new u or sd into it
  // and exchange it with the field.
  double* spare = nullptr;
  // Second spare buffer (x*y, allocated by the first two-step pass), which
  // takes the new r (PPCG) or p (Chebyshev) there: neighbouring tiles still
  // read the old values.
  double* spare2 = nullptr;

  // A PPCG inner step or Chebyshev step held back (fused mode) so that it
  // can run in one pass with the next one: which (kHeld*), its
  // coefficients, and whether the depth-1 halo update that follows it (of
  // SD, or U) has been requested and held back too.
  int held = 0;
  bool held_halo = false;
  double held_alpha = 0.0, held_beta = 0.0;
  // A depth-1 reflective update of SD (PPCG) or U (Chebyshev), all faces
  // external, requested with no step held and held back so that the next
  // two-step pass reflects the ring of the field it stages instead (the
  // halo slot, or -1).
  int pre_halo = -1;

  // Device memory of the chunk (dev_alloc), its buffers' sizes, and the most
  // that it may take (TEA_HIP_EXTRA_BYTES beyond what creation took; a refusal
  // is that of a full device).
  std::unordered_map<const void*, size_t> dev_sizes;
  size_t dev_bytes = 0, dev_limit = SIZE_MAX;

  // Deferred CG work (fused mode).
  int fused = 1;
  int batch = 0;   // load batch of the fused stencil kernel (0: default)
  bool pairs = false;  // two-cells-per-lane kernels
  bool quads = false;  // four-cells-per-lane mixed-precision kernels (x % 4 == 0)
  bool pend_u = false, pend_p = false, pend_halo = false;
  double pend_alpha = 0.0, pend_beta = 0.0;
  // Up to two updates u += uh_alpha[i] uh_p[i] (oldest first, uh_p among
  // p_alt), each with the U halo update after it, that passes of the fused
  // iteration have left to a later one (TEA_HIP_HOLD_U=0 turns this off):
  // the third pass makes both and its own in one pass over u.  Older than
  // the deferred work above; any other entry point makes them first.
  int uh = 0;
  double* uh_p[2] = {};
  double uh_alpha[2] = {0.0, 0.0};

  // Mixed-precision CG: FP32 p (a ring of buffers, mp_cur is
  // current; each w-step writes the next), r, w and
  // face coefficients; allocated by the first tea_hip_mpcg_init.
  float* mp_p[kMpRing] = {};
  int mp_cur = 0;
  // Up to two updates u += hold_alpha[i] p, p in mp_p[hold_buf[i]] (oldest
  // first), reported done to the host but held back (TEA_HIP_HOLD_U=0 turns
  // this off): the third four-cells-per-lane w-step reads both held p and
  // makes the held updates and its own
  // in one pass over u; any other entry point makes them first.
  bool hold_ok = true;
  int hold = 0;
  int hold_buf[2] = {0, 0};
  double hold_alpha[2] = {0.0, 0.0};
  float* mp_r = nullptr;
  float* mp_w = nullptr;
  float* mp_kx = nullptr;
  float* mp_ky = nullptr;

  // Flexible CG: the preconditioned residual z (FP32) and, for the learned
  // preconditioner, up to kFcgMaxLevels coarse levels (coarsening c, 4c),
  // each with its network instance, coarse operator and work arrays.
  float* fcg_z = nullptr;
  float fcg_norm[4] = {0.0f, 1.0f, 0.0f, 1.0f};
  int fcg_levels = 0;
  FcgLevel fcg_lv[kFcgMaxLevels];
  // Coarse solve by fcg_sweeps Jacobi sweeps instead of the network (0:
  // network); the level-0 sums of T y over the level-1 blocks (the cross
  // term of two levels), and the factors g of the levels.
  int fcg_sweeps = 0;
  double* fcg_xsum = nullptr;
  float* fcg_g = nullptr;

  // Passes in flight that calls have taken over: FP64 CG, mixed-precision CG and
  // FCG, Jacobi (tea_hip_ahead_taken).
  long taken[3] = {};

  // Run-ahead of the fused CG iteration (cg.hip): the device forms alpha and
  // beta from its own sums and runs the next passes of the iteration, the
  // r-step (ra_r) and the w-step behind it (ra_w), into spare buffers before
  // the host asks for them; the host's call takes a pass over when its scalar
  // is bitwise the device's.
  bool ra_r = false, ra_w = false;
  CgStep ra_step;             // the w-step in flight
  bool ra_enabled = true;     // TEA_HIP_RUN_AHEAD=0 turns it off
  bool ra_off = false;        // a buffer it needs could not be allocated
  bool p_ring_off = false;    // the same of the held updates' p buffers
  // Blocks one row apart per workgroup of the stencil passes mp_w4_kernel,
  // fused_w1_kernel and jacobi_pair_kernel: 1, 2 (the default) or 4
  // (TEA_HIP_STACK).  (fcg_z4_kernel, whose only row above is ky's, took
  // 57.4 us with two against 56.0 us with one.)
  int stack = 2;
  bool ra_dirty = false;      // a discarded run-ahead may still be writing ra_host
  int ra_fail = 0;            // consecutive mismatches (3 turn it off)
  int ra_wi = 0, ra_ri = 0;   // host slots of the newest w-step and r-step
  double ra_rro = 0.0;        // r.r the host was last given (its rro)
  bool ra_rro_known = false;
  double ra_alpha = 0.0;      // the device's alpha of the last w-step the
                              // host asked for
  double ra_beta = 0.0;       // its beta of the last r-step
  double* r_alt = nullptr;    // spare r, u and w (x*y each)
  double* u_alt = nullptr;
  double* w_alt = nullptr;
  double* ra_dev = nullptr;   // device: [0] alpha, [1] beta, [2] r.r
  double* ra_host = nullptr;  // pinned: {w-step, r-step} x 2 slots x {sum, scalar}
  double* ra_host_dev = nullptr;  // device view of ra_host

  // Run-ahead of mixed-precision CG and FCG (mpcg.hip): up to two passes in
  // flight beyond what the host asked for, the next r-step (mra_r; with FCG
  // also z = M(r)) and the next w-step (mra_w), into spare buffers.
  bool mra_r = false, mra_w = false;
  int mra_turn = 0;            // kind of the first one (kMraSlotW or R)
  bool mra_fcg = false;        // the passes belong to FCG
  int mra_coarse = 0;          // use_net of the last preconditioner call
  int mra_fail = 0;            // consecutive mismatches (3 turn it off)
  bool mra_off = false;        // a buffer it needs could not be allocated
  int mra_since = 0, mra_period = 0;  // r-steps since the last refresh, and
                                      // how many the last two were apart
  int mra_wi = 0, mra_ri = 0;  // host slots of the newest w-step and r-step
  bool mra_synced = false;     // u_alt equals u outside the interior
  double mra_alpha = 0.0;      // the device's alpha of the last w-step the
                               // host asked for
  double mra_beta = 0.0;       // its beta of the last r-step
  MpStep mra_step;             // the w-step in flight
  float* mp_r_alt = nullptr;
  float* mp_w_alt = nullptr;
  float* fcg_z_alt = nullptr;
  double* mra_dev = nullptr;   // [0] alpha, [1] beta, [2] p.w
  double* mra_host = nullptr;  // pinned: {w-step, r-step} x 2 slots x {sum,
                               // sum, scalar}
  double* mra_host_dev = nullptr;

  // Run-ahead of the Jacobi sweeps (solvers.hip): up to two sweeps queued
  // beyond the one the host asked for, the first into j_buf[0] (one of the
  // spare buffers), each with the U halo update before it; and whether the
  // ring of r, the u of before the last sweep, still lacks that update.
  int jra = 0;
  bool j_off = false;          // a buffer it needs could not be allocated
  double** j_buf[2] = {};
  bool j_ring = false;
  int j_sub = 0;               // the block sums (sub or sub2) of the newest sweep
  int j_slot = 0;              // host slot of the last sweep the host asked for
  int j_since = 0, j_period = 0;  // sweeps since the last restart, and between
                                  // the last two
  double* j_host = nullptr;    // pinned, 2 slots
  double* j_host_dev = nullptr;

  // Waiting for a reduction by its values: launch_span_finish(..., poll)
  // fills the first partial of arrays 0 .. poll_nr-1 with a sentinel, and the
  // finish waits until the finisher has overwritten them all (or the stream
  // is idle).
  bool poll = true;
  int poll_nr = 0;

  // A depth-1 reflective update also copies the cells of its face lines
  // beyond the ring (e.g. column h-1 at rows below h-1) from other cells
  // outside the interior, which no kernel of the iteration changes.  A
  // U/P update is deferred into a fused pass, which writes only the ring,
  // once a real update of all external faces has made those cells what the
  // update would leave; host writes and initialisations clear the flags.
  bool faces_ok_u = false, faces_ok_p = false;

  // Timing.
  bool timing = false;
  struct Pending {
    int kid;
    hipEvent_t start, stop;
  };
  std::vector<Pending> inflight;
  std::vector<hipEvent_t> event_pool;
  bool time_kernel[tea::K_NUM];     // kernels timed (all, or TEA_HIP_STATS_ONLY)
  long launches[tea::K_NUM] = {};
  double total_ms[tea::K_NUM] = {};
};

namespace tea {

// Records start/stop events around one kernel launch when timing is on.
struct Timed {
  tea_hip_chunk* c;
  int kid;
  hipStream_t stream;  // the chunk's stream unless given
  hipEvent_t start = nullptr, stop = nullptr;
  Timed(tea_hip_chunk* c_, int kid_, hipStream_t s = nullptr);
  ~Timed();
};

// Resolves the recorded events (after the stream has been synchronised).
int resolve_timing(tea_hip_chunk* c);

// Synchronises the stream and resolves timing.
int sync_chunk(tea_hip_chunk* c);

// Resolves the recorded events that have completed, oldest first, without
// waiting.
int resolve_ready(tea_hip_chunk* c);

// Waits for the stream, then finishes nr reductions on the host: the
// reference tree's remaining passes over each array of nspan level-2
// partials; results go to out[0..nr).
int finish_reduction(tea_hip_chunk* c, int nr, double* out);

// The run-ahead's scalar, formed by the finisher: mode 0 (after a w-step)
// alpha = rro / sum into ra[0]; mode 1 (after an r-step) beta = sum / rro into
// ra[1] and sum into ra[2].  rro is ra[2] when from_dev, else the value.  The
// sum and the scalar also go to out[0], out[1] (pinned host memory the host
// polls).
// With two sums (mixed-precision CG, FCG): mode 0 alpha = sum1 / sum0 into
// ra[0] and sum0 (p.w) into ra[2]; mode 1 beta = -sum1 / ra[2] into ra[1];
// out holds both sums and the scalar.
struct RaTail {
  double rro;
  int from_dev, mode;
  double* ra;
};
// The finisher of nr sums (1 or 2) of c->sub with the run-ahead's scalar, into
// out; not waited for.
int launch_span_finish_ra(tea_hip_chunk* c, int nr, double* out, const RaTail& tail);
// Finishes nr sums from their block sums (the first nr arrays of sub, c->sub
// unless given), sum q into the first value of array slot + q of c->partials
// (*len = 1).  With poll (slot 0), the next finish waits for the values
// themselves instead of the stream; only for a finish that follows with no
// other kernel writing the partials in between.
int launch_span_finish(tea_hip_chunk* c, int nr, int* len, int slot = 0,
                       bool poll = false, const double* sub = nullptr);

// finish_reduction over the first len partials of each array (len is what
// launch_span_finish leaves).
int finish_reduction_n(tea_hip_chunk* c, int nr, int len, double* out);
// Values in pinned, mapped host memory that a kernel of the stream writes:
// arm them with the wait sentinel before the launch, then wait until the
// kernel has overwritten all count of them.
void arm_host_values(double* host, int count);
int wait_host_values(tea_hip_chunk* c, const double* host, int count);

// The same with a length per array.
int finish_reduction_lens(tea_hip_chunk* c, int nr, const int* lens, double* out);

// The pair-per-thread kernels apply: pairs and more than one group
// (the reference then runs its level-2 pass; for a single group it stops at
// level 1, which the span-per-block kernels reproduce).
inline bool use_pair_blocks(const tea_hip_chunk* c, int kernel_bit) {
  return c->pairs && (c->pair_blocks & kernel_bit) && c->ngroup > 1;
}

// The four-cells-per-lane variants of the pair-per-thread kernels (same
// results bit for bit) apply where those do and x is a multiple of 4.
inline bool use_quad_blocks(const tea_hip_chunk* c, int kernel_bit) {
  return c->quads && use_pair_blocks(c, kernel_bit);
}

// A body's NR sums over the interior, to out: one pair per thread and a
// finisher where the pair kernels apply, else one block per span and the
// host's passes.
template <int NR, class Body>
int sum_over_cells(tea_hip_chunk* c, int kid, const Body& body, double* out) {
  if (use_pair_blocks(c, 1)) {
    {
      Timed t(c, kid);
      hipLaunchKernelGGL((pair_sum_kernel<NR, Body>), dim3(c->nblk), dim3(kBlock), 0, c->stream,
                         c->geo, body, c->sub, c->nblk);
    }
    TEA_HIP_TRY(hipGetLastError());
    int len;
    TEA_RETURN_IF(launch_span_finish(c, NR, &len, 0, true));
    return finish_reduction_n(c, NR, len, out);
  }
  {
    Timed t(c, kid);
    hipLaunchKernelGGL((span_kernel<NR, Body>), dim3(c->nspan), dim3(kBlock), 0, c->stream,
                       c->geo, body, c->partials, c->nspan, c->ngroup == 1 ? 1 : 0);
  }
  TEA_HIP_TRY(hipGetLastError());
  return finish_reduction(c, NR, out);
}

// Kinds of held-back step.
enum { kHeldNone = 0, kHeldPpcg = 1, kHeldCheby = 2 };

// Applies the deferred CG work (fused mode: u += alpha p, p = beta p + r and
// their halo ring), then runs a held-back step.  Deferred CG work is always
// older than a held step: a step is held with at most u += alpha p pending,
// and the CG entry points run a held step before they defer new work.
int apply_pending(tea_hip_chunk* c);
// Drops Jacobi sweeps in flight and makes r's ring what the halo update of the
// u it was leaves (solvers.hip).
int jacobi_settle(tea_hip_chunk* c);
// The deferred CG work alone (cg.hip).
int apply_cg_pending(tea_hip_chunk* c);
// The held FP64 u updates alone, with their U halo update (cg.hip).
int apply_held_u(tea_hip_chunk* c);
// A held-back halo update before a step, alone (solvers.hip).
int apply_pre_halo(tea_hip_chunk* c);
// Runs what is held back, oldest first: deferred CG work, a held-back halo
// update before a step (pre_halo), a held-back PPCG inner step or Chebyshev
// step and its held-back halo update (solvers.hip).
int flush_held(tea_hip_chunk* c);
// A mixed-precision residual step: r_out = r - alpha w, r.r and, with rw, r.w.
struct MpRStep {
  const float* r;
  float* r_out;
  const float* w;
  double alpha;
  RaScalar sc;
};
// Launches it, its sums left in `sub` (pair and four-cell kernels; the first
// two arrays) or, on the span kernels, its partials in c->partials (mpcg.hip).
int launch_mp_r(tea_hip_chunk* c, const MpRStep& s, bool rw, double* sub);
// The w-step and r-step of mixed-precision CG, and of FCG (fcg), with the
// run-ahead (mpcg.hip).  The r-step returns r.r and r.w (z.w).
int mp_calc_w(tea_hip_chunk* c, bool fcg, double alpha, int apply_u, double beta, int apply_p,
              double* pw, double* pr);
int mp_calc_r(tea_hip_chunk* c, bool fcg, double alpha, int use_net, double* rr, double* rx);
// FCG's z = M(r) and z.w, the block sums in `sub` (pair and four-cell kernels;
// fcg.hip).
int launch_fcg_z(tea_hip_chunk* c, int use_net, const float* r, const float* w, float* z,
                 double* sub);
// The same on any kernels with the partials of z.w in array `slot` of
// c->partials; *len is the number left to finish (fcg.hip).
int launch_precondition(tea_hip_chunk* c, int use_net, int slot, int* len);
// Makes the held-back u updates on their own, oldest first (mpcg.hip).
int apply_mp_hold(tea_hip_chunk* c);

// The depth-1 reflective update of one field's x*y array, all faces external.
int launch_halo_of(tea_hip_chunk* c, double* field);
// One reflective-halo launch (all flagged fields and external faces).
int launch_halos(tea_hip_chunk* c, int depth, const int neighbours[4],
                 const int fields[6]);

// Device memory within the chunk's limit: false (and *p null) where there is
// none.  Buffers of one size may have changed places with a field's.
bool dev_alloc_bytes(tea_hip_chunk* c, void** p, size_t bytes);
void dev_free_bytes(tea_hip_chunk* c, void* p);
template <class T>
bool dev_alloc(tea_hip_chunk* c, T** p, size_t bytes) {
  return dev_alloc_bytes(c, (void**)p, bytes);
}
// Gives back the buffers that solvers only run faster with (those of passes in
// flight and held updates, which end first; the spare field pair unless
// keep_pair) and leaves them out from then on.
int release_spares(tea_hip_chunk* c, bool keep_pair);
// A buffer that a solver cannot do without.
template <class T>
int need_alloc(tea_hip_chunk* c, T** p, size_t bytes, const char* what, bool keep_pair = false) {
  if (dev_alloc(c, p, bytes)) return TEA_HIP_OK;
  TEA_RETURN_IF(release_spares(c, keep_pair));
  if (dev_alloc(c, p, bytes)) return TEA_HIP_OK;
  set_error(std::string("hipMalloc of ") + what + " failed");
  return TEA_HIP_ENOMEM;
}
// `n` doubles of pinned, coherent host memory for values that the device
// leaves (null: there is none), and the device's view of them.
double* host_slots(int n, double** dev);
template <class T>
void dev_free(tea_hip_chunk* c, T*& p) {
  dev_free_bytes(c, p);
  p = nullptr;
}

// Drops a run-ahead of the fused CG iteration (cg.hip): it wrote only
// spare buffers and device scalars, so nothing is undone.
int ra_discard(tea_hip_chunk* c);
// The same for a pass of mixed-precision CG or FCG in flight (mpcg.hip).
int mra_discard(tea_hip_chunk* c);

// Drops the passes in flight of every solver but `keep`, whose entry points
// may take theirs over.  The solvers' passes share the block sums, the spare
// u and the fields themselves, so a call that launches anything, or changes
// what they read, leaves at most its own in flight.
enum { kAheadNone, kAheadCg, kAheadMp, kAheadJacobi };
inline int drop_ahead(tea_hip_chunk* c, int keep) {
  if (keep != kAheadCg) TEA_RETURN_IF(ra_discard(c));
  if (keep != kAheadMp) TEA_RETURN_IF(mra_discard(c));
  if (keep != kAheadJacobi) TEA_RETURN_IF(jacobi_settle(c));
  return TEA_HIP_OK;
}

// Checks the handle and makes its device current, leaving a run-ahead in
// flight (the CG entry points that can take it over); applies a held-back
// mixed-precision u update.
#define TEA_ENTER_RA(c)                                   \
  TEA_CHECK_ARG((c) != nullptr, "null chunk handle");     \
  TEA_HIP_TRY(hipSetDevice((c)->device));                 \
  TEA_RETURN_IF(::tea::drop_ahead(c, ::tea::kAheadCg));   \
  (c)->mra_synced = false;                                \
  if ((c)->hold) TEA_RETURN_IF(::tea::apply_mp_hold(c))

// Checks the handle and makes its device current (entry points); drops a
// run-ahead of the CG iteration.
#define TEA_ENTER_HELD(c)                                 \
  TEA_ENTER_RA(c);                                        \
  TEA_RETURN_IF(::tea::drop_ahead(c, ::tea::kAheadNone))

// Entry points other than the PPCG inner step and the halo update first run
// a held-back halo update and PPCG or Chebyshev step (and drop a run-ahead)
// and apply a held-back mixed-precision u update.
#define TEA_FLUSH_HELD(c)                                                  \
  do {                                                                     \
    TEA_RETURN_IF(::tea::drop_ahead(c, ::tea::kAheadNone));                \
    if ((c)->hold) TEA_RETURN_IF(::tea::apply_mp_hold(c));                 \
    TEA_RETURN_IF(::tea::flush_held(c));                                   \
  } while (0)

// TEA_FLUSH_HELD for the mixed-precision and FCG steps: leaves their own held
// u updates held (the w-step makes them with its own) and their own passes in
// flight, and makes the FP64 iteration's held updates, which are older.
#define TEA_FLUSH_HELD_KEEP_MP(c)                                          \
  do {                                                                     \
    TEA_RETURN_IF(::tea::drop_ahead(c, ::tea::kAheadMp));                  \
    TEA_RETURN_IF(::tea::apply_held_u(c));                                 \
    TEA_RETURN_IF(::tea::flush_held(c));                                   \
  } while (0)

#define TEA_ENTER(c)   \
  TEA_ENTER_HELD(c);   \
  TEA_FLUSH_HELD(c)

inline int mp_next(const tea_hip_chunk* c, int i) {
  return i + 1 == kMpRing || !c->mp_p[i + 1] ? 0 : i + 1;
}

inline dim3 span_grid(const tea_hip_chunk* c) { return dim3(c->nspan); }
inline dim3 pair_grid(const tea_hip_chunk* c) { return dim3(c->nblk); }
inline dim3 quad_grid(const tea_hip_chunk* c) { return dim3(c->nblk); }
inline dim3 flat_grid(long n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); }

// Stacked workgroups of the 512-cell-block stencil kernels: with S = x / 512
// blocks per row, block c + S t holds the cells one row above block c + S
// (t - 1), so a workgroup of KS blocks takes c + S t for t = KS j .. KS j +
// KS - 1 and their rows above and below are mostly each other's own rows,
// loaded on the same CU (L1 hits, not L2 requests).  Each block's cells,
// lanes and wave sums are those of one block per workgroup.  stack_factor is
// c->stack where it applies (1, 2 or 4; 1 for rows shorter than a block).
inline int stack_factor(const tea_hip_chunk* c) {
  const int S = c->geo.x / kPairBlock;
  return (c->stack == 2 || c->stack == 4) && S >= 1 ? c->stack : 1;
}
inline int stack_rows(const tea_hip_chunk* c) { return c->geo.x / kPairBlock; }
inline dim3 stacked_grid(const tea_hip_chunk* c, int ks) {
  if (ks == 1) return dim3(c->nblk);
  const int S = stack_rows(c), tn = (c->nblk + S - 1) / S;
  return dim3((unsigned)(S * ((tn + ks - 1) / ks)));
}
// The block and thread index of the calling thread in a workgroup of KS
// blocks of T threads (blk >= nblk for the unused blocks of the last row).
template <int KS, int T>
__device__ inline int stacked_block(int S, int* tid, bool bands = true) {
  *tid = KS == 1 ? (int)threadIdx.x : (int)threadIdx.x % T;
  if (KS == 1) return band_index(bands);
  // Workgroup w in launch order or, in bands, in place w of the pass.
  if (!bands)
    return (int)(blockIdx.x % S) + S * ((int)(blockIdx.x / S) * KS + (int)threadIdx.x / T);
  const int w = band_index<KS>();
  return w % S + S * (w / S * KS + (int)threadIdx.x / T);
}

}  // namespace tea
