// Attention of Q query tokens over reconstructed (dense, 16-bit) histories for gfx950:
// the second half of the route that dequantizes each history to the query's type and
// attends to it under the offset causal mask (turboquant_kv/packed_backend.py:211-226,
// mask packed_attention.py:198-206: query i of a sequence of length L sees keys
// j <= L - Q + i; a query that sees none gives 0). It serves the steps that the packed
// prefill (prefill.hip) does not compile: other widths, head_dim 64, 16-bit queries.
//
// The library's attention took these steps through fp32 copies of K, V and the mask (a
// dozen launches, each a pass over a (query, key) matrix in memory): 57 us of softmax, 115
// and 100 us of fp32 products and 300 us of copies for 4 sequences of 64 queries over
// 1,000-4,096 tokens, 28 / 4 heads. Here K and V stay 16 bits wide, both products run on
// v_mfma_f32_16x16x32_{bf16,f16} and no score leaves the work-group.
//
// Precision is that of the fp32 products: q, K and V are exact operands, scores and
// softmax are fp32, and each probability goes to its product as a sum of 16-bit values:
// three for bf16 (24 bits), two for fp16, taken up by 2^7 to the top of fp16's range (22
// bits of those above 2^-10 of the largest, 2^-32 of the largest below). A bf16 pair (16
// bits) took 80.6 us for the call below and left up to three times the error that fp32
// weights have where a sum of both signs cancels.
//
// Work-group: eight waves take eight neighbouring 32-row query blocks (row r = qi n_rep +
// h) of one (sequence, kv head, split) and share its 64-token chunks through two LDS tile
// sets, one barrier per chunk, the next chunk's rows loading a chunk ahead. The tiles and
// the token order are those of the packed prefill's shared-tile scan: K [token][dim] rows
// of 2 D + 16 bytes (16-byte column quads of rows 16-31 and 48-63 swapped), V transposed
// [dim][token] rows of 144 bytes; row c of score tile t is token 32 (t >> 1) + 8 (c >> 2)
// + 4 (t & 1) + (c & 3), so that lane 16g + c ends the scores with the eight tokens that
// are its k-slots of a value K-step.
// Measured (that call, 8-bit K and V): 952 -> 84 us, of which the two batched dequants
// 21 us each, this scan 42 us and the merge 7 us; the same distance from 64 bits.
#include <algorithm>
#include <map>
#include <mutex>
#include <utility>

#include "wn_common.h"
#include "wn_tables.h"

namespace wn {
namespace {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int kHtWaves = 8;
constexpr int kHtBlock = 32;                    // query rows of a wave
constexpr int kHtRows = kHtWaves * kHtBlock;    // query rows of a work-group
constexpr int kHtVRow = 144;                    // bytes of a V tile row
constexpr float kHtRescale = 8.0f;              // the reference maximum moves past this (log2 units)

struct HistArgs {
  const uint16_t* q;
  int64_t qsb, qsh, qsq;  // element strides of (B, Hq, Q, D)
  const uint16_t* k;      // (B, Hkv, Lpad, D) contiguous
  const uint16_t* v;
  const int32_t* seq_lens;
  float* part_acc;  // (rows, D), row = (unit nsplit + s) 256 + row of the unit
  float* part_ml;   // (rows, 2)
  int64_t Lpad;
  float scale;      // of the scores, log2 units
  int B, Hkv, n_rep, Q, ncg, nsplit;  // ncg: work-group blocks of rows per (sequence, kv head)
};

template <int D>
struct HistTile {
  static constexpr int KRow = 2 * D + 16, K = 64 * KRow, V = D * kHtVRow, Set = K + V;
};

template <int D>
__device__ __forceinline__ uint32_t hist_k_off(int r, int q) {
  return uint32_t(r * HistTile<D>::KRow + ((q ^ ((r & 16) >> 2)) << 4));
}

template <bool BF>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
}

// Terms of a probability in the 16-bit type, and the log2 it is taken up by (its largest, 2^8,
// ends below 2^15).
template <bool BF>
constexpr int kHtTerms = BF ? 3 : 2;
template <bool BF>
constexpr float kHtLift = BF ? 0.f : 7.f;

// Two values as 16-bit ones, rounded to nearest, and, term by term, what the rounding left.
template <bool BF>
__device__ __forceinline__ void split_terms(float x, float y, uint32_t (&o)[kHtTerms<BF>]) {
  if constexpr (BF) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < kHtTerms<BF>; ++i) {
      o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x, y}, b2));
      x -= __builtin_bit_cast(float, o[i] << 16);
      y -= __builtin_bit_cast(float, o[i] & 0xffff0000u);
    }
  } else {
    const _Float16 a = _Float16(x), b = _Float16(y);
    o[0] = uint32_t(__builtin_bit_cast(uint16_t, a)) | uint32_t(__builtin_bit_cast(uint16_t, b)) << 16;
    o[1] = tf_word(x - float(a), y - float(b));
  }
}

// The rows one thread brings to the tiles per chunk. K: (token, 8-dim group), the groups
// of a row side by side; V: (token pair, 8-dim group), the pairs side by side.
template <int D>
struct HistRaw {
  static constexpr int G = D / 8, NTHR = 64 * kHtWaves;
  static constexpr int NK = 64 * G / NTHR;
  static constexpr int NV = (32 * G + NTHR - 1) / NTHR;
  u32x4 k[NK], v[NV][2];
};

// Tokens are clamped to the last of the range: real rows, masked.
template <int D>
__device__ __forceinline__ void hist_load(const uint16_t* k, const uint16_t* v, int c0, int t_hi, int tid, HistRaw<D>& o) {
  using R = HistRaw<D>;
#pragma unroll
  for (int j = 0; j < R::NK; ++j) {
    const int it = tid + R::NTHR * j;
    o.k[j] = *reinterpret_cast<const u32x4*>(k + int64_t(min(c0 + it / R::G, t_hi - 1)) * D + 8 * (it % R::G));
  }
#pragma unroll
  for (int j = 0; j < R::NV; ++j) {
    const int it = tid + R::NTHR * j, tp = it & 31, dg = it >> 5;
    if (32 * R::G % R::NTHR == 0 || it < 32 * R::G) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        o.v[j][h] = *reinterpret_cast<const u32x4*>(v + int64_t(min(c0 + 2 * tp + h, t_hi - 1)) * D + 8 * dg);
    }
  }
}

template <int D>
__device__ __forceinline__ void hist_store(const HistRaw<D>& r, char* set, int tid) {
  using R = HistRaw<D>;
#pragma unroll
  for (int j = 0; j < R::NK; ++j) {
    const int it = tid + R::NTHR * j;
    *reinterpret_cast<u32x4*>(set + hist_k_off<D>(it / R::G, it % R::G)) = r.k[j];
  }
  char* vt = set + HistTile<D>::K;
#pragma unroll
  for (int j = 0; j < R::NV; ++j) {
    const int it = tid + R::NTHR * j, tp = it & 31, dg = it >> 5;
    if (32 * R::G % R::NTHR != 0 && it >= 32 * R::G) break;
#pragma unroll
    for (int m = 0; m < 8; ++m)  // dim 8dg + m: tokens 2tp (low half), 2tp + 1
      *reinterpret_cast<uint32_t*>(vt + (8 * dg + m) * kHtVRow + 4 * tp) =
          __builtin_amdgcn_perm(r.v[j][1][m >> 1], r.v[j][0][m >> 1], m & 1 ? 0x07060302u : 0x05040100u);
  }
}

template <int D, bool BF>
__global__ __launch_bounds__(64 * kHtWaves) void history_kernel(HistArgs a) {
  using T = HistTile<D>;
  constexpr int KS = D / 32, MT = D / 16, LA = 4;  // K-steps, value M-tiles, operand reads in flight
  constexpr int NT = kHtTerms<BF>;
  constexpr float lift = kHtLift<BF>;
  __shared__ __align__(16) char lds[2 * T::Set];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int wig = __builtin_amdgcn_readfirstlane(tid >> 6);
  // work-groups go to the XCDs round robin; those of neighbouring units (row blocks and
  // splits of one history) get one XCD's L2
  const int nwg = gridDim.x, p8 = blockIdx.x & 7, per = nwg >> 3;
  int64_t u = p8 * per + min(p8, nwg & 7) + (blockIdx.x >> 3);
  const int cg = int(u % a.ncg);
  u /= a.ncg;
  const int s = int(u % a.nsplit);
  u /= a.nsplit;
  const int kvh = int(u % a.Hkv), b = int(u / a.Hkv);
  const int rows = a.n_rep * a.Q;
  const int r_first = cg * kHtRows + wig * kHtBlock;
  const bool live = r_first < rows;
  const int L = int(min(int64_t(const_view(a.seq_lens)[b]), a.Lpad));  // no row past the histories' own
  // the chunks that the group's last row sees
  const int g_last = min((cg + 1) * kHtRows, rows) - 1;
  const int seen = max(0, min(L, L - a.Q + g_last / a.n_rep + 1));
  const int nch = (seen + 63) >> 6;
  const int ch_lo = int(int64_t(nch) * s / a.nsplit), n = int(int64_t(nch) * (s + 1) / a.nsplit) - ch_lo;
  const int t_lo = 64 * ch_lo, t_hi = min(t_lo + 64 * n, seen);

  f32x4 acc[2][MT];
  float m[2], l[2];
  int lim[2];  // last visible token of column c of column tile ct
  u32x4 qb[2][KS];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[ct][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[ct] = -INFINITY;
    l[ct] = 0.f;
    const int r = min(r_first + 16 * ct + c, rows - 1);  // rows past the end repeat the last one
    lim[ct] = L - a.Q + r / a.n_rep;
    const uint16_t* q = a.q + b * a.qsb + (kvh * a.n_rep + r % a.n_rep) * a.qsh + (r / a.n_rep) * a.qsq + (D / 4) * g;
#pragma unroll
    for (int k = 0; k < KS; ++k) qb[ct][k] = *reinterpret_cast<const u32x4*>(q + 8 * k);
  }
  const int lim_min = L - a.Q + min(r_first, rows - 1) / a.n_rep;

  if (n > 0) {
    const uint16_t* kh = a.k + (int64_t(b) * a.Hkv + kvh) * a.Lpad * D;
    const uint16_t* vh = a.v + (int64_t(b) * a.Hkv + kvh) * a.Lpad * D;
    HistRaw<D> raw;
    hist_load<D>(kh, vh, t_lo, t_hi, tid, raw);
    hist_store<D>(raw, lds, tid);
    if (n > 1) hist_load<D>(kh, vh, t_lo + 64, t_hi, tid, raw);
    int krow[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) krow[t] = 32 * (t >> 1) + 8 * (c >> 2) + 4 * (t & 1) + (c & 3);
    for (int ch = 0; ch < n; ++ch) {
      __syncthreads();  // chunk ch is in set ch & 1; the other set is free
      const char* cur = lds + (ch & 1) * T::Set;
      if (ch + 1 < n) {
        hist_store<D>(raw, lds + ((ch + 1) & 1) * T::Set, tid);
        if (ch + 2 < n) hist_load<D>(kh, vh, t_lo + 64 * (ch + 2), t_hi, tid, raw);
      }
      if (!live) continue;
      const int c0 = t_lo + 64 * ch;
      const bool full = c0 + 63 <= lim_min && c0 + 64 <= t_hi;
      f32x4 d[2][4];
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int t = 0; t < 4; ++t) d[ct][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      {  // step k = 4s + t: dims D/4 g + 8s .. of tile t; the schedule is pinned (prefill.hip)
        u32x4 e[LA + 1];
        auto look = [&](auto kc, u32x4& o) {
          constexpr int k = decltype(kc)::value;
          o = *reinterpret_cast<const u32x4*>(cur + hist_k_off<D>(krow[k & 3], KS * g + (k >> 2)));
        };
        static_for<0, LA>([&](auto kc) { look(kc, e[decltype(kc)::value]); });
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, 4 * KS>([&](auto kc) {
          constexpr int k = decltype(kc)::value, j = k % (LA + 1);
          if constexpr (k + LA < 4 * KS) {
            look(std::integral_constant<int, k + LA>{}, e[(k + LA) % (LA + 1)]);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int ct = 0; ct < 2; ++ct) d[ct][k & 3] = mfma16<BF>(e[j], qb[ct][k >> 2], d[ct][k & 3]);
          __builtin_amdgcn_sched_barrier(0);
        });
      }
      u32x4 pt[NT][2][2];  // value operands, by term: tokens 32 ks + 8g .. + 7 of column tile ct
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const bool fresh = m[ct] == -INFINITY;
        const float m0 = fresh ? 0.f : m[ct];
        const int last = min(lim[ct], t_hi - 1) - (c0 + 8 * g);
        float x[16], top = -INFINITY;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float y = fmaf(d[ct][t][i], a.scale, lift - m0);
            x[4 * t + i] = full || 32 * (t >> 1) + 4 * (t & 1) + i <= last ? y : -INFINITY;
            top = fmaxf(top, x[4 * t + i]);
          }
        top = fmaxf(top, __shfl_xor(top, 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        top -= lift;
        const bool move = top > kHtRescale || (fresh && top > -INFINITY);
        if (__any(move)) {  // wave-uniform
          const float shift = move ? top : 0.f;
          const float alpha = move ? (fresh ? 0.f : __builtin_amdgcn_exp2f(-top)) : 1.f;
          m[ct] = move ? m0 + top : m[ct];
          l[ct] *= alpha;
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[ct][mt] *= alpha;
#pragma unroll
          for (int k = 0; k < 16; ++k) x[k] -= shift;
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int k = 8 * ks + 2 * j;
            const float p0 = __builtin_amdgcn_exp2f(x[k]), p1 = __builtin_amdgcn_exp2f(x[k + 1]);
            l[ct] += p0 + p1;
            uint32_t w[NT];
            split_terms<BF>(p0, p1, w);
#pragma unroll
            for (int i = 0; i < NT; ++i) pt[i][ct][ks][j] = w[i];
          }
      }
      {  // step k = MT ks + mt: tokens 32 ks + 8g .. of dim 16 mt + c
        u32x4 e[LA + 1];
        auto look = [&](auto kc, u32x4& o) {
          constexpr int k = decltype(kc)::value;
          o = *reinterpret_cast<const u32x4*>(cur + T::K + (16 * (k % MT) + c) * kHtVRow + 16 * (4 * (k / MT) + g));
        };
        static_for<0, LA>([&](auto kc) { look(kc, e[decltype(kc)::value]); });
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, 2 * MT>([&](auto kc) {
          constexpr int k = decltype(kc)::value, ks = k / MT, mt = k % MT, j = k % (LA + 1);
          if constexpr (k + LA < 2 * MT) {
            look(std::integral_constant<int, k + LA>{}, e[(k + LA) % (LA + 1)]);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) acc[ct][mt] = mfma16<BF>(e[j], pt[i][ct][ks], acc[ct][mt]);
          __builtin_amdgcn_sched_barrier(0);
        });
      }
    }
  }
  if (!live) return;
  const int64_t row0 = ((((int64_t(b) * a.Hkv + kvh) * a.nsplit + s) * a.ncg + cg) * kHtWaves + wig) * kHtBlock;
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    float sum = l[ct];
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const int64_t row = row0 + 16 * ct + c;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<f32x4*>(a.part_acc + row * D + 16 * mt + 4 * g) = acc[ct][mt];
    if (g == 0) *reinterpret_cast<float2*>(a.part_ml + 2 * row) = make_float2(m[ct], sum);
  }
}

struct HistMergeArgs {
  const float* part_acc;
  const float* part_ml;
  void* out;  // (B, Q, Hq, D) contiguous
  int Hkv, n_rep, Q, ncg, nsplit, D;
  int64_t items;  // B Q Hq D / 8
};

// One thread per eight outputs: the max-stable merge of the row's splits, 1 / l, the cast.
template <bool BF>
__global__ __launch_bounds__(256) void history_merge_kernel(HistMergeArgs a) {
  const int64_t it = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (it >= a.items) return;
  const uint32_t per = uint32_t(a.D) / 8, Hq = uint32_t(a.Hkv * a.n_rep);
  const uint32_t d0 = 8 * uint32_t(it % per);
  const int64_t row = it / per;  // (b, qi, h)
  const uint32_t h = uint32_t(row % Hq);
  const int64_t bq = row / Hq;
  const uint32_t qi = uint32_t(bq % a.Q), b = uint32_t(bq / a.Q), kvh = h / uint32_t(a.n_rep);
  const uint32_t r = qi * uint32_t(a.n_rep) + h % uint32_t(a.n_rep);
  const int64_t step = int64_t(a.ncg) * kHtRows;
  const int64_t first = (int64_t(b) * a.Hkv + kvh) * a.nsplit * step + r;
  float M = -INFINITY;
#pragma unroll 4
  for (int s = 0; s < a.nsplit; ++s) M = fmaxf(M, a.part_ml[2 * (first + s * step)]);
  float den = 0.f;
  f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
#pragma unroll 4
  for (int s = 0; s < a.nsplit; ++s) {
    const int64_t pr = first + s * step;
    const float2 ml = *reinterpret_cast<const float2*>(a.part_ml + 2 * pr);
    // 0 for a split without keys; a row without a maximum saw no key (sums of 0) or only
    // NaN scores (NaN sums, which stay)
    const float w = M == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(ml.x - M);
    den = fmaf(w, ml.y, den);
    const f32x4* src = reinterpret_cast<const f32x4*>(a.part_acc + pr * a.D + d0);
    x += w * src[0];
    y += w * src[1];
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
  x *= inv;
  y *= inv;
  uint16_t o[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float v = k < 4 ? x[k & 3] : y[k & 3];
    o[k] = BF ? f32_to_bf16(v) : f32_to_f16(v);
  }
  uint4 w;
  __builtin_memcpy(&w, o, 16);
  reinterpret_cast<uint4*>(a.out)[it] = w;
}

using HistFn = void (*)(HistArgs);

HistFn pick_history(int D, int dtype) {
  if (D == 128) return dtype == WN_BF16 ? history_kernel<128, true> : history_kernel<128, false>;
  if (D == 64) return dtype == WN_BF16 ? history_kernel<64, true> : history_kernel<64, false>;
  return nullptr;
}

int history_ncg(int n_rep, int Q) { return int((int64_t(n_rep) * Q + kHtRows - 1) / kHtRows); }

int64_t history_rows(int B, int Hkv, int n_rep, int Q, int nsplit) {
  return int64_t(B) * Hkv * nsplit * history_ncg(n_rep, Q) * kHtRows;
}

int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

// Resident work-groups of `fn` on the current device.
int history_slots(HistFn fn) {
  static std::mutex mu;
  static std::map<std::pair<int, HistFn>, int> cache;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lock(mu);
  auto it = cache.find({dev, fn});
  if (it != cache.end()) return it->second;
  int per_cu = 0, cus = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(fn), 64 * kHtWaves, 0) !=
          hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return cache[{dev, fn}] = per_cu * cus;
}

}  // namespace
}  // namespace wn

using namespace wn;

extern "C" int wn_history_plan(int B, int Hq, int Hkv, int Q, int D, int dtype, int max_len, int* num_splits) {
  clear_error();
  WN_REQUIRE(B >= 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && Q > 0 && max_len >= 0 && num_splits, WN_E_INVALID,
             "wn_history_plan: bad sizes B=%d Hq=%d Hkv=%d Q=%d max_len=%d", B, Hq, Hkv, Q, max_len);
  WN_REQUIRE(dtype == WN_F16 || dtype == WN_BF16, WN_E_INVALID, "wn_history_plan: dtype code %d", dtype);
  const HistFn fn = pick_history(D, dtype);
  WN_REQUIRE(fn, WN_E_UNSUPPORTED, "wn_history_plan: head_dim %d (64 or 128)", D);
  const int w = history_slots(fn);
  WN_REQUIRE(w > 0, WN_E_LAUNCH, "wn_history_plan: cannot query the device occupancy");
  // in chunks of one work-group: rounds of work-groups, a split's chunks and about two for
  // its start and end, a tenth of a round for the spread of the ends, and the partials
  // (256 rows written and read per unit and split)
  const int64_t units = int64_t(B > 0 ? B : 1) * Hkv * history_ncg(Hq / Hkv, Q), chunks = (int64_t(max_len) + 63) / 64;
  double best = 0.0;
  for (int64_t ns = 1; ns <= std::max<int64_t>(1, std::min<int64_t>(64, chunks / 2)); ++ns) {
    const int64_t rounds = (units * ns + w - 1) / w;
    const double cost = (double(rounds) + 0.1) * double((chunks + ns - 1) / ns + 2) + 0.018 * double(units * ns);
    if (ns == 1 || cost < best) {
      best = cost;
      *num_splits = int(ns);
    }
  }
  return WN_OK;
}

extern "C" int64_t wn_history_workspace_bytes(int B, int Hq, int Hkv, int Q, int D, int num_splits) {
  if (B < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || Q <= 0 || (D != 64 && D != 128) || num_splits <= 0) return -1;
  const int64_t rows = history_rows(B, Hkv, Hq / Hkv, Q, num_splits);
  return align256(rows * D * 4) + rows * 8;
}

extern "C" int wn_history_attention(const void* q, int dtype, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_q,
                                    const void* k, const void* v, const int32_t* seq_lens, void* out, void* workspace,
                                    int64_t workspace_bytes, int B, int Hq, int Hkv, int Q, int D, int64_t Lpad,
                                    float scale, int num_splits, void* stream) {
  clear_error();
  WN_REQUIRE(B >= 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && Q > 0 && Lpad >= 0, WN_E_INVALID,
             "wn_history_attention: bad sizes B=%d Hq=%d Hkv=%d Q=%d Lpad=%lld", B, Hq, Hkv, Q, (long long)Lpad);
  WN_REQUIRE(dtype == WN_F16 || dtype == WN_BF16, WN_E_INVALID, "wn_history_attention: dtype code %d", dtype);
  const HistFn fn = pick_history(D, dtype);
  WN_REQUIRE(fn, WN_E_UNSUPPORTED, "wn_history_attention: head_dim %d (64 or 128)", D);
  WN_REQUIRE(num_splits > 0 && num_splits <= 4096, WN_E_INVALID, "wn_history_attention: num_splits %d", num_splits);
  const int n_rep = Hq / Hkv;
  WN_REQUIRE(int64_t(n_rep) * Q <= (int64_t(1) << 24), WN_E_INVALID, "wn_history_attention: n_rep * Q too large");
  if (B == 0) return WN_OK;
  WN_REQUIRE(q && k && v && seq_lens && out, WN_E_INVALID, "wn_history_attention: null operand");
  WN_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(out, 16) && q_stride_b % 8 == 0 &&
                 q_stride_h % 8 == 0 && q_stride_q % 8 == 0,
             WN_E_INVALID, "wn_history_attention: operands 16-byte aligned, strides of q multiples of 8");
  const int64_t need = wn_history_workspace_bytes(B, Hq, Hkv, Q, D, num_splits);
  WN_REQUIRE(workspace && workspace_bytes >= need && aligned(workspace, 256), WN_E_WORKSPACE,
             "wn_history_attention: workspace needs %lld bytes, 256-aligned (got %lld)", (long long)need,
             (long long)workspace_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int ncg = history_ncg(n_rep, Q);
  const int64_t rows = history_rows(B, Hkv, n_rep, Q, num_splits), groups = rows / kHtRows;
  WN_REQUIRE(groups < (int64_t(1) << 31), WN_E_INVALID, "wn_history_attention: grid too large");
  HistArgs a{};
  a.q = static_cast<const uint16_t*>(q);
  a.qsb = q_stride_b;
  a.qsh = q_stride_h;
  a.qsq = q_stride_q;
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.seq_lens = seq_lens;
  a.part_acc = static_cast<float*>(workspace);
  a.part_ml = reinterpret_cast<float*>(static_cast<char*>(workspace) + align256(rows * D * 4));
  a.Lpad = Lpad;
  a.scale = float(double(scale) * 1.4426950408889634);
  a.B = B;
  a.Hkv = Hkv;
  a.n_rep = n_rep;
  a.Q = Q;
  a.ncg = ncg;
  a.nsplit = num_splits;
  hipLaunchKernelGGL(fn, dim3(unsigned(groups)), dim3(64 * kHtWaves), 0, st, a);
  HistMergeArgs m{a.part_acc, a.part_ml, out, Hkv, n_rep, Q, ncg, num_splits, D, int64_t(B) * Q * Hq * (D / 8)};
  const int64_t blocks = (m.items + 255) / 256;
  WN_REQUIRE(blocks < (int64_t(1) << 31), WN_E_INVALID, "wn_history_attention: grid too large");
  if (dtype == WN_BF16) hipLaunchKernelGGL(history_merge_kernel<true>, dim3(unsigned(blocks)), dim3(256), 0, st, m);
  else hipLaunchKernelGGL(history_merge_kernel<false>, dim3(unsigned(blocks)), dim3(256), 0, st, m);
  return check_launch("wn_history_attention");
}
