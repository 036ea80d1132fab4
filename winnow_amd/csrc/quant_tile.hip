// quantize for many vectors (prompts, prefill chunks) at head_dim 64 and 128, gfx950:
// the codes and norms of quantize_kernel (quant.hip), bit for bit, with the rotation on
// the fp16 matrix cores.
//
// The float64 matrix cores bound quantize_kernel: 2 D^2 float64 operations per vector
// are 55 us of MFMA time for the 131,056 vectors of an 8,191-token prompt (8 kv heads, K and
// V), and it took 131 us. Here y is first formed with fp16 operands and fp32 sums, to
// within a bound eps of its float64 value, and bucketized. A y closer than eps to a
// bucket boundary (0.2 of a vector's 128 at 4 bits, 2.4 at 8 bits) is then recomputed
// in float64 from the same correctly rounded fp32 x / n that quantize_kernel uses, so
// no code depends on the fp16 products.
//
//   operands  Pi 2^8 = H + L, an fp16 pair per entry (22 bits), in LDS in the order the
//             MFMAs read it, staged once by a persistent work-group of sixteen waves; x
//             2^(8-e), e the exponent of the norm: one fp16 for bf16 and fp16 inputs
//             (exact but for elements below 2^-22 of the norm, which end as fp16 subnormals,
//             2^-33 of it off at most), an fp16 pair for fp32 inputs.
//   product   y^T = Pi x^T on v_mfma_f32_16x16x32_f16, A = rows of Pi, B = sixteen
//             vectors; a wave takes one such tile of vectors at a time (with two, half
//             the LDS reads, the kernel spilled and ran slower: 34 us against 30).
//   eps       |error of y| <= (D 2^-23 + 2^-20) R, R the largest row norm of Pi: the
//             products of fp16 values are exact, each of a sum's D additions errs by at
//             most one ulp (2^-23, truncation allowed) of a partial sum, all of which
//             are below |x / n| R <= R (Cauchy-Schwarz); 2^-20 covers the two splits
//             (2^-22 each), the subnormal elements (sqrt(D) 2^-33), the product with 1 / n
//             and the last rounding.
//   buckets   y's cell of a 512-cell grid over the boundaries gives the number of
//             boundaries below the cell and the one boundary in reach of it: one 8-byte
//             LDS read, against a search of bw reads. A cell with two or more in reach
//             sends its y to the float64 path.
//   exact     the flagged (vector, dim) pairs of a pass go to a list in LDS; sixteen of
//             them at a time, four lanes each form the float64 dot product of x / n with
//             a row of Pi (both read again, from L2) and its code.
// A vector whose norm is not below 2^100, and a Pi that does not fit the operands (row
// norms of 128 or more), take the float64 path for every code. The codes of a pass sit
// in LDS as bytes, so that whole rows are packed and stored by neighbouring lanes.
//
// With outlier channels (G2; the contiguous cache) a vector is two: its regular and its
// outlier channels, each with its own norm, rotation, boundaries and width. Pi is then
// the matrix of both rotations, rows in code order (regular first), columns in channel
// order, zero between the groups; the norms, thresholds, grids and exact dot products
// are taken per group, and the rows are packed byte by byte (a group's codes need not
// fill eights). A prompt of 2,048 tokens (2 sequences, 8 heads; 120 channels at 4 bits, 8 at
// 8) took sixteen launches and copies; now the prompt takes 54 us, a single token 26 (traces).
//
// Measured (K and V of 8 kv heads in one launch, head_dim 128, quantize_kernel -> this):
// 8,191 tokens 4 bits bf16 128 -> 30 us, 8 bits 133 -> 47 us, 4 bits fp32 119 -> 34 us;
// 65,536 tokens 4 bits bf16 947 -> 186 us (1.8 TB/s). The vector ALU bounds it: about
// eleven instructions per code to find its bucket, and the float64 norms and flagged
// dot products; a launch of one pass per wave adds the staging and the latency of its
// loads. Measured without gain: a touch of the next pass's rows ahead of it (40 us).
#include <algorithm>
#include <type_traits>

#include "wn_quant.h"

namespace wn {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

// waves of a work-group (two groups of channels: eight, whose registers they need)
template <bool G2>
constexpr int tile_waves() { return G2 ? 8 : 16; }
constexpr int kTileVecs = 16;    // vectors a wave takes per pass (an MFMA column tile)
constexpr int kCells = 512;      // cells of the boundary grid
constexpr int kListMax = 256;    // flagged pairs a wave lists; with more it recomputes the whole pass

struct Cell {
  float b;        // the boundary in reach of the cell: +inf for none, NaN for several
  uint32_t base;  // boundaries below the cell's reach
};

// Number of the nb ascending boundaries below y.
__device__ __forceinline__ uint32_t count_below(const float* bnd, int bw, float y) {
  uint32_t pos = 0;
  for (int step = 1 << (bw - 1); step > 0; step >>= 1) pos += bnd[pos + step - 1] < y ? step : 0;
  return pos;
}

// Eight elements of a row of x, as they are stored.
template <int DT>
struct Raw8 {
  uint4 w[DT == WN_F32 ? 2 : 1];
};
template <int DT>
__device__ __forceinline__ Raw8<DT> load8(const void* x, int64_t i) {
  Raw8<DT> r;
  if constexpr (DT == WN_F32) {
    const uint4* p = reinterpret_cast<const uint4*>(static_cast<const float*>(x) + i);
    r.w[0] = p[0];
    r.w[1] = p[1];
  } else {
    r.w[0] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(x) + i);
  }
  return r;
}
template <int DT>
__device__ __forceinline__ float elem(const Raw8<DT>& r, int k) {
  const uint4 a = r.w[DT == WN_F32 ? k >> 2 : 0];
  if constexpr (DT == WN_F32) {
    const int j = k & 3;
    return __builtin_bit_cast(float, j == 0 ? a.x : j == 1 ? a.y : j == 2 ? a.z : a.w);
  } else {
    const int j = k >> 1;
    const uint32_t w = j == 0 ? a.x : j == 1 ? a.y : j == 2 ? a.z : a.w;
    if constexpr (DT == WN_BF16) return __builtin_bit_cast(float, k & 1 ? w & 0xffff0000u : w << 16);
    else return f16_to_f32(uint16_t(k & 1 ? w >> 16 : w));
  }
}

// float64 sum of squares of a lane's elements reduced over the four lanes of a vector,
// in quantize_kernel's order: D/16 consecutive elements in turn, then the sixteen
// partial sums by halves.
// G2: the elements of one group only, `in` naming the lane's elements 8s + k in it.
template <int DT, int KS, bool G2>
__device__ __forceinline__ double sum_squares(const Raw8<DT> (&x)[KS], uint32_t in) {
  constexpr int EPT = 2 * KS, PPL = 8 / EPT;  // elements per partial sum, partial sums per eight elements
  double p[KS][PPL];
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int h = 0; h < PPL; ++h) {
      double ss = 0.0;
#pragma unroll
      for (int k = 0; k < EPT; ++k) {
        const double e = double(elem<DT>(x[s], EPT * h + k));
        const double f = !G2 || (in >> (8 * s + EPT * h + k) & 1) ? e : 0.0;
        ss = fma(f, f, ss);
      }
      __builtin_amdgcn_sched_barrier(0);
      p[s][h] = ss;
    }
#pragma unroll
  for (int o = KS / 2; o > 0; o >>= 1)
#pragma unroll
    for (int s = 0; s < o; ++s)
#pragma unroll
      for (int h = 0; h < PPL; ++h) p[s][h] += p[s + o][h];
#pragma unroll
  for (int h = 0; h < PPL; ++h) {
    p[0][h] += __shfl_xor(p[0][h], 32, 64);
    p[0][h] += __shfl_xor(p[0][h], 16, 64);
  }
  return PPL == 1 ? p[0][0] : p[0][0] + p[0][PPL - 1];
}

// One row (vector) of a wave's pass.
struct RowInfo {
  int64_t x;     // element offset of x
  int64_t page;  // byte offset of the packed row, or element offset of its codes; -1: not written
  int64_t norm;  // element offset of the norm
  float n[2];    // the norms of the two groups (one group: the first)
};

template <int D>
struct TileWave {
  RowInfo row[kTileVecs];
  uint16_t list[kListMax];                   // vector D + dim
  __align__(8) uint8_t code[kTileVecs][D];     // code8()
};

// The eight codes of dims 8k .. 8k + 7 of row r (the eights of a row swapped about, so
// that neither the MFMA layout's writes nor the row reads meet in a few banks).
template <int D>
__device__ __forceinline__ uint8_t* code8(TileWave<D>& w, int r, int k) {
  return w.code[r] + 8 * (k ^ ((r >> 1) & (D / 8 - 1)));
}

template <bool G2>
using TileArgs = std::conditional_t<G2, QuantSplitArgs, QuantArgs>;
// The second group of a side that has one; else `none`.
__device__ __forceinline__ const QuantGroup2& second_group(const QuantSplitSide& s, const QuantGroup2&) { return s.second; }
__device__ __forceinline__ const QuantGroup2& second_group(const QuantSide&, const QuantGroup2& none) { return none; }

template <int D, int DT, bool G2>
__global__ __launch_bounds__(64 * tile_waves<G2>()) void quantize_tile_kernel(TileArgs<G2> a) {
  constexpr int WV = tile_waves<G2>();
  constexpr int KS = D / 32;  // K-steps of 32 input dims
  constexpr int U = D / 32;   // eights of output dims per lane (two MFMA row tiles each)
  constexpr int NR = kTileVecs, NTHR = 64 * WV;
  constexpr bool F32 = DT == WN_F32;
  constexpr int NG = G2 ? 2 : 1;
  __shared__ __align__(16) h8 ph[2 * U][KS][64], pl[2 * U][KS][64];
  __shared__ __align__(8) Cell cells[NG][kCells];
  __shared__ float bnd[NG][256];
  __shared__ float rowsq[D];
  __shared__ TileWave<D> waves[WV];

  const auto& sd = a.side[blockIdx.y];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int wig = __builtin_amdgcn_readfirstlane(tid >> 6);
  TileWave<D>& wv = waves[wig];
  const int bw = sd.bw;
  const QuantGroup2 none{};
  const QuantGroup2& s2 = second_group(sd, none);
  int split = D;
  uint32_t outl = 0;  // bit 8s + k: channel 32s + 8g + k is an outlier
  if constexpr (G2) {
    split = a.split;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int k = 0; k < 8; ++k) outl |= (a.chan[32 * s + 8 * g + k] ? 1u : 0u) << (8 * s + k);
  }
  // passes are dealt to the work-groups in turn, so that a launch of few passes still
  // spreads over the CUs
  const int64_t passes = (a.total + NR - 1) / NR, stride = int64_t(gridDim.x) * WV;
  int64_t pass = int64_t(wig) * gridDim.x + blockIdx.x;
#pragma unroll
  for (int q = 0; q < NG; ++q)
    for (int i = tid; i < (1 << (q ? s2.bw : bw)) - 1; i += NTHR) bnd[q][i] = (q ? s2.bnd : sd.bnd)[i];
  for (int i = tid; i < D; i += NTHR) rowsq[i] = 0.f;
  __syncthreads();
  // operand (t, s, lane 16g + c): row r = c of tile t = 2u + h is output dim
  // D/4 (c >> 2) + 8u + 4h + (c & 3), k-slots of group g the input dims 32s + 8g ..
#pragma unroll
  for (int it = 0; it < (2 * U * KS + WV - 1) / WV; ++it) {
    const int item = it * WV + wig, t = item / KS, s = item % KS;
    if (item < 2 * U * KS) {
      const int dim = (D / 4) * (c >> 2) + 8 * (t >> 1) + 4 * (t & 1) + (c & 3);
      const float4* p = reinterpret_cast<const float4*>(sd.pi + dim * D + 32 * s + 8 * g);
      const float4 p0 = p[0], p1 = p[1];
      const float v[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
      h8 hi, lo;
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float z = v[k] * 256.f;
        hi[k] = _Float16(z);
        lo[k] = _Float16(z - float(hi[k]));
        ss = fmaf(v[k], v[k], ss);
      }
      ph[t][s][lane] = hi;
      pl[t][s][lane] = lo;
      atomicAdd(&rowsq[dim], ss);
    }
  }
  __syncthreads();
  float eps[NG], inv_w[NG], at0[NG];
#pragma unroll
  for (int q = 0; q < NG; ++q) {
    const int qbw = q ? s2.bw : bw, nb = (1 << qbw) - 1;
    const float* bd = bnd[q];
    float rmax = 0.f;  // largest squared row norm (a NaN row is left out: its own dims' y are NaN, hence flagged)
#pragma unroll
    for (int i = 0; i < D; i += 64)
      if (!G2 || (i + lane >= split) == (q == 1)) rmax = fmaxf(rmax, rowsq[i + lane]);
    rmax = wave_max(rmax);
    eps[q] = rmax < 16384.f ? (D * 0x1p-23f + 0x1p-20f) * 1.01f * sqrtf(rmax) : NAN;
    // cells of width cw: cell 0 ends at the first boundary, the last one starts at the last
    const float b0 = bd[0], b1 = bd[nb - 1];
    const float cw = (b1 - b0) / float(kCells - 2);
    const bool grid_ok = cw > 0.f && cw < INFINITY && fabsf(b0) < INFINITY && eps[q] < INFINITY;
    inv_w[q] = grid_ok ? 8.f / cw : 0.f;  // 8: bytes of a cell
    const float lo0 = b0 - cw;
    at0[q] = -lo0 * inv_w[q];
    for (int i = tid; i < kCells; i += NTHR) {
      const float reach = eps[q] + 0.05f * cw;  // 0.05 cw: rounding of the cell number and of the edges
      Cell e{NAN, 0};
      if (grid_ok) {
        const uint32_t below = i == 0 ? 0 : count_below(bd, qbw, lo0 + i * cw - reach);
        const uint32_t upto = i == kCells - 1 ? nb : count_below(bd, qbw, lo0 + (i + 1) * cw + reach);
        e.base = below;
        e.b = upto == below ? INFINITY : upto == below + 1 ? bd[below] : NAN;
      }
      cells[q][i] = e;
    }
  }
  __syncthreads();  // the only block-wide barriers: waves run independently from here

  for (; pass < passes; pass += stride) {
    wave_lds_sync();  // the last pass's reads of the wave's LDS area are done
    if (lane < NR) {
      const int64_t vec = pass * NR + lane;
      const uint32_t vc = uint32_t(vec < a.total ? vec : a.total - 1);  // total < 2^31
      const uint32_t bh = vc / uint32_t(a.n), i = vc % uint32_t(a.n), b = bh / uint32_t(a.H), h = bh % uint32_t(a.H);
      RowInfo& o = wv.row[lane];
      o.x = b * sd.sb + h * sd.sh + i * sd.sn;
      int64_t page = -1, norm = 0;
      if (vec < a.total) {
        if constexpr (G2) {
          page = norm = (int64_t(b) * a.H + h) * a.cap + a.pos0 + i;  // the row's number
        } else if (!a.scatter) {
          page = vec * D;
          norm = vec;
        } else {
          const int pos = a.start_pos[b] + int(i), col = pos >> a.log2S;
          const int pid = pos >= 0 && col < a.max_pages ? a.table[b * a.tsb + col] : -1;
          if (pid >= 0 && pid < a.num_pages) {
            const int64_t slot = pos & ((1 << a.log2S) - 1);
            page = pid * sd.psp + h * sd.psh + slot * (D * bw / 8);
            norm = pid * sd.nsp + h * sd.nsh + slot;
          }
        }
      }
      o.page = page;
      o.norm = norm;
    }
    wave_lds_sync();
    float r[NG], thr[NG];
    h8 xh[KS], xl[F32 ? KS : 1];
    {
      Raw8<DT> x[KS];
      const int64_t xo = wv.row[c].x + 8 * g;
#pragma unroll
      for (int s = 0; s < KS; ++s) x[s] = load8<DT>(sd.x, xo + 32 * s);
      float sc[NG];
#pragma unroll
      for (int q = 0; q < NG; ++q) {
        const float n = fmaxf(float(sqrt(sum_squares<DT, KS, G2>(x, q ? outl : ~outl))), 1e-10f);
        if (g == 0) wv.row[c].n[q] = n;
        int e;
        frexpf(n, &e);
        const bool sane = n < 0x1p100f;
        sc[q] = sane ? ldexpf(1.f, 8 - e) : 0.f;
        r[q] = sane ? ldexpf(1.f / n, e - 16) : 0.f;
        thr[q] = sane ? eps[q] : NAN;  // NaN: every code is flagged
      }
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float z = elem<DT>(x[s], k) * (G2 && (outl >> (8 * s + k) & 1) ? sc[NG - 1] : sc[0]);
          xh[s][k] = _Float16(z);
          if constexpr (F32) xl[s][k] = _Float16(z - float(xh[s][k]));
        }
    }
    int flagged = 0;  // wave-uniform
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // the operands are read here, pass after pass: kept in registers over the passes
      // (they do not change) they would spill
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      f32x4 acc[2], low[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) acc[h] = low[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const h8 p = ph[2 * u + h][s][lane], q = pl[2 * u + h][s][lane];
          acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p, xh[s], acc[h], 0, 0, 0);
          low[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(q, xh[s], low[h], 0, 0, 0);
          if constexpr (F32) low[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p, xl[s], low[h], 0, 0, 0);
        }
      }
      float rw[NG];  // inv_w, at0: in bytes of the table
#pragma unroll
      for (int q = 0; q < NG; ++q) rw[q] = r[q] * inv_w[q];
      const int j0 = (D / 4) * g + 8 * u;  // the lane's first code of the eight
      uint32_t word[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        Cell e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[h][i] += low[h][i];
          const int q = G2 && j0 + 4 * h + i >= split;
          // the cell number, below 0 and past the end clamped; a NaN reads some cell
          const float at = __builtin_amdgcn_fmed3f(fmaf(acc[h][i], q ? rw[NG - 1] : rw[0], q ? at0[NG - 1] : at0[0]), 0.f,
                                                   8.f * kCells - 1.f);
          e[i] = *reinterpret_cast<const Cell*>(reinterpret_cast<const char*>(cells[0]) + (uint32_t(at) & (8 * kCells - 8)) +
                                                (q ? 8 * kCells : 0));
        }
        word[h] = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int q = G2 && j0 + 4 * h + i >= split;
          const float d = fmaf(acc[h][i], q ? r[NG - 1] : r[0], -e[i].b);  // y - b
          word[h] |= (e[i].base + (d > 0.f ? 1u : 0u)) << (8 * i);
          const uint64_t near = __ballot(!(fabsf(d) >= (q ? thr[NG - 1] : thr[0])));
          if (near) {  // wave-uniform, taken for one in ten at 4 bits
            const int at = flagged + int(__builtin_amdgcn_mbcnt_hi(uint32_t(near >> 32),
                                                                   __builtin_amdgcn_mbcnt_lo(uint32_t(near), 0)));
            if ((near >> lane & 1) && at < kListMax)
              wv.list[at] = uint16_t(c * D + (D / 4) * g + 8 * u + 4 * h + i);
            flagged += __builtin_popcountll(near);
          }
        }
      }
      *reinterpret_cast<uint2*>(code8<D>(wv, c, (D / 32) * g + u)) = make_uint2(word[0], word[1]);
    }
    wave_lds_sync();  // codes, list, norms
    const bool all = flagged > kListMax;
    const int items = all ? NR * D : flagged;
    for (int j0 = 0; j0 < items; j0 += 16) {
      const int j = min(j0 + c, items - 1);
      const int id = all ? j : int(wv.list[j]);
      const int rr = id / D, dim = id % D;
      const int q2 = G2 && dim >= split;  // the group
      const float n = wv.row[rr].n[q2], rn = 1.f / n;
      const bool divide = __any(!(n < 0x1p100f));  // wave-uniform
      const int64_t xo = wv.row[rr].x + 8 * g;
      const float* prow = sd.pi + dim * D + 8 * g;
      double sum = 0.0;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const Raw8<DT> x = load8<DT>(sd.x, xo + 32 * s);
        const float4 p0 = *reinterpret_cast<const float4*>(prow + 32 * s);
        const float4 p1 = *reinterpret_cast<const float4*>(prow + 32 * s + 4);
        const float p[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
        // the correctly rounded fp32 x / n: rn is the rounded reciprocal, the residual x - q n
        // is exact, and one correction by it rounds right (Markstein, "Computation of
        // elementary functions on the IBM RISC System/6000 processor", 1990). A quotient
        // below the normal range may differ in its last bit: 2^-149 of y.
        float z[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float xv = elem<DT>(x, k), q = xv * rn;
          z[k] = fmaf(fmaf(-q, n, xv), rn, q);
          if (G2 && int(outl >> (8 * s + k) & 1) != q2) z[k] = 0.f;
        }
        if (divide) {
          asm volatile("" ::: "memory");  // a branch: the divisions are not formed for a select
#pragma unroll
          for (int k = 0; k < 8; ++k) z[k] = G2 && int(outl >> (8 * s + k) & 1) != q2 ? 0.f : elem<DT>(x, k) / n;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) sum = fma(double(z[k]), double(p[k]), sum);
      }
      sum += __shfl_xor(sum, 16, 64);
      sum += __shfl_xor(sum, 32, 64);
      if (g == 0) code8<D>(wv, rr, dim >> 3)[dim & 7] = uint8_t(count_below(bnd[q2], q2 ? s2.bw : bw, float(sum)));
    }
    wave_lds_sync();
    if constexpr (G2) {
      // byte by byte: the bytes of both groups' rows, neighbouring lanes neighbouring bytes
      const int nb1 = split * bw / 8, nb2 = (D - split) * s2.bw / 8, nball = nb1 + nb2;
      for (int i = lane; i < NR * nball; i += 64) {
        const int rr = i / nball, k = i % nball, q = k >= nb1;
        const int64_t row = wv.row[rr].page;
        if (row < 0) continue;
        const int w = q ? s2.bw : bw, first = q ? split : 0, end = q ? D : split, bit0 = 8 * (q ? k - nb1 : k);
        uint32_t v = 0;
        for (int d = bit0 / w; first + d < end && d * w < bit0 + 8; ++d) {
          const int j = first + d, sh = d * w - bit0;
          const uint32_t cd = code8<D>(wv, rr, j >> 3)[j & 7];
          v |= sh >= 0 ? cd << sh : cd >> -sh;
        }
        if (q) s2.pages[row * nb2 + k - nb1] = uint8_t(v);
        else sd.pages[row * nb1 + k] = uint8_t(v);
      }
      if (lane < NR && wv.row[lane].page >= 0) {
        sd.norms[wv.row[lane].norm] = f32_to_f16(wv.row[lane].n[0]);
        s2.norms[wv.row[lane].norm] = f32_to_f16(wv.row[lane].n[1]);
      }
      continue;
    }
    // whole rows: D/8 lanes each pack and store eight codes
    constexpr int LPR = D / 8, RPI = 64 / LPR;
#pragma unroll
    for (int it = 0; it < NR / RPI; ++it) {
      const int rr = it * RPI + lane / LPR, part = lane % LPR;
      const int64_t page = wv.row[rr].page;
      if (page < 0) continue;
      const uint2 w = *reinterpret_cast<const uint2*>(code8<D>(wv, rr, part));
      if (!a.scatter) {
        *reinterpret_cast<uint2*>(sd.codes_out + page + 8 * part) = w;
        if (part == 0) sd.norms_out[wv.row[rr].norm] = wv.row[rr].n[0];
        continue;
      }
      uint8_t* dst = sd.pages + page + part * bw;
      if (bw == 4) {  // nibbles of the four bytes of a word, two words to one
        const uint32_t t0 = w.x | w.x >> 4, t1 = w.y | w.y >> 4;
        *reinterpret_cast<uint32_t*>(dst) =
            (t0 & 0xffu) | (t0 >> 8 & 0xff00u) | (t1 & 0xffu) << 16 | (t1 << 8 & 0xff000000u);
      } else {
        uint64_t pk = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) pk |= uint64_t((k < 4 ? w.x : w.y) >> (8 * (k & 3)) & 0xffu) << (bw * k);
        store_packed8(dst, pk, bw);
      }
      if (part == 0) sd.norms[wv.row[rr].norm] = f32_to_f16(wv.row[rr].n[0]);
    }
  }
}

template <bool G2>
using TileFn = void (*)(TileArgs<G2>);

template <int D, bool G2>
TileFn<G2> pick_tile(int dtype) {
  return dtype == WN_F32   ? quantize_tile_kernel<D, WN_F32, G2>
         : dtype == WN_F16 ? quantize_tile_kernel<D, WN_F16, G2>
                           : quantize_tile_kernel<D, WN_BF16, G2>;
}

bool rows_aligned(const QuantSide& s, int es) {
  return aligned(s.x, 16) && s.sb * es % 16 == 0 && s.sh * es % 16 == 0 && s.sn * es % 16 == 0;
}

}  // namespace

// Rows that 16-byte loads can read, vector numbers that fit 31 bits, and enough vectors
// that staging Pi and the grid pays. Measured (us, quantize_kernel -> this; K + V
// vectors, bf16): head_dim 128, 4 bits, 12,288: 17.9 -> 13.0, 16,384: 21.2 -> 13.2 (8,192
// stay, at 13.1); 8 bits, whose longer lists cost a wave more, 16,384: 22.9 -> 20.1;
// head_dim 64, 4 bits, 12,288: 8.5 -> 8.6, 16,384: 9.1 -> 8.3-9.1, 8 bits 10.1 -> 9.5.
bool quantize_tiles_ok(const QuantArgs& a, int sides, int D) {
  if ((D != 64 && D != 128) || a.total >= (int64_t(1) << 31)) return false;
  bool wide = D == 64;
  const int es = a.x_dtype == WN_F32 ? 4 : 2;
  for (int i = 0; i < sides; ++i) {
    if (!rows_aligned(a.side[i], es)) return false;
    wide = wide || a.side[i].bw == 8;
  }
  return a.total * sides >= (wide ? 16384 : 12288);
}

template <bool G2>
static int launch_tiles(TileFn<G2> fn, const TileArgs<G2>& a, int sides, hipStream_t st) {
  // one work-group per CU; its passes are dealt out from there
  const int cus = device_cus();
  if (cus <= 0) return WN_E_LAUNCH;
  const int64_t groups = std::min<int64_t>((a.total + kTileVecs - 1) / kTileVecs, std::max(1, cus / sides));
  hipLaunchKernelGGL(fn, dim3(unsigned(groups), sides), dim3(64 * tile_waves<G2>()), 0, st, a);
  return WN_OK;
}

int launch_quantize_tiles(const QuantArgs& a, int sides, int D, hipStream_t st) {
  return launch_tiles<false>(D == 64 ? pick_tile<64, false>(a.x_dtype) : pick_tile<128, false>(a.x_dtype), a, sides, st);
}

bool quantize_split_ok(const QuantSplitArgs& a, int sides, int D) {
  if ((D != 64 && D != 128) || a.total >= (int64_t(1) << 31)) return false;
  const int es = a.x_dtype == WN_F32 ? 4 : 2;
  for (int i = 0; i < sides; ++i)
    if (!rows_aligned(a.side[i], es)) return false;
  return true;
}

int launch_quantize_split(const QuantSplitArgs& a, int sides, int D, hipStream_t st) {
  return launch_tiles<true>(D == 64 ? pick_tile<64, true>(a.x_dtype) : pick_tile<128, true>(a.x_dtype), a, sides, st);
}

}  // namespace wn
