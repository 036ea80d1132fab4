// Operands and device helpers that the quantize kernels share (quant.hip: sixteen
// vectors per work-group, float64 rotation; quant_tile.hip: many vectors per wave).
#pragma once

#include "wn_common.h"

namespace wn {

struct QuantSide {
  const void* x;
  int64_t sb, sh, sn;  // element strides of (B, H, n, D)
  const float* pi;
  const float* bnd;
  int bw;
  uint8_t* pages;  // scatter mode
  int64_t psp, psh;
  uint16_t* norms;
  int64_t nsp, nsh;
  uint8_t* codes_out;  // flat mode
  float* norms_out;
};

template <class Side>
struct QuantArgsOf {
  Side side[2];  // K, V
  const int32_t* table;
  const int32_t* start_pos;
  int64_t tsb;
  int64_t total;  // vectors per side = B*H*n
  int H, n, log2S, num_pages, max_pages, x_dtype, scatter;
};
using QuantArgs = QuantArgsOf<QuantSide>;

// Outlier channels (launch_quantize_split): boundaries, width, rows and norms of the second group.
struct QuantGroup2 {
  const float* bnd;
  int bw;
  uint8_t* pages;
  uint16_t* norms;
};

struct QuantSplitSide : QuantSide {
  QuantGroup2 second;
};

struct QuantSplitArgs : QuantArgsOf<QuantSplitSide> {
  const uint8_t* chan;    // group of each channel
  int split, pos0;        // codes of group 0, first position
  int64_t cap;            // rows per (sequence, head)
};

// pos[k] = #{b < y[k]} over the 2^bw - 1 ascending boundaries (torch.bucketize,
// right=False), for N values at once: the N binary searches advance in lockstep, so
// each level issues N independent LDS reads instead of one dependent read per value.
template <int N>
__device__ __forceinline__ void bucketize_n(const float* bnd, int bw, const float (&y)[N], uint32_t (&pos)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) pos[k] = 0;
  for (int step = 1 << (bw - 1); step > 0; step >>= 1) {
    float b[N];
#pragma unroll
    for (int k = 0; k < N; ++k) b[k] = bnd[pos[k] + step - 1];
#pragma unroll
    for (int k = 0; k < N; ++k) pos[k] += b[k] < y[k] ? step : 0;
  }
}

// The bw bytes of eight bw-bit codes packed LSB-first, stored at p (p is aligned to
// the largest power of two dividing bw).
__device__ __forceinline__ void store_packed8(uint8_t* p, uint64_t v, int bw) {
  if (bw == 8) {
    *reinterpret_cast<uint2*>(p) = make_uint2(uint32_t(v), uint32_t(v >> 32));
  } else if (bw == 4) {
    *reinterpret_cast<uint32_t*>(p) = uint32_t(v);
  } else if (bw == 2) {
    *reinterpret_cast<uint16_t*>(p) = uint16_t(v);
  } else if (bw == 6) {
    reinterpret_cast<uint16_t*>(p)[0] = uint16_t(v);
    reinterpret_cast<uint16_t*>(p)[1] = uint16_t(v >> 16);
    reinterpret_cast<uint16_t*>(p)[2] = uint16_t(v >> 32);
  } else {
    for (int k = 0; k < bw; ++k) p[k] = uint8_t(v >> (8 * k));
  }
}

// quant_tile.hip: whether its kernel serves these operands, and its launch (0: launched).
bool quantize_tiles_ok(const QuantArgs& a, int sides, int D);
int launch_quantize_tiles(const QuantArgs& a, int sides, int D, hipStream_t st);
// The same kernel with two groups of channels, rows of a contiguous cache (quant.hip's
// wn_append_split).
bool quantize_split_ok(const QuantSplitArgs& a, int sides, int D);
int launch_quantize_split(const QuantSplitArgs& a, int sides, int D, hipStream_t st);

}  // namespace wn
