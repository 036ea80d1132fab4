// Dequantization at fp32 accuracy for every head_dim up to 256 (gfx950): byte codes
// (TurboQuantMSE.dequantize_into, turboquant_kv/cache.py:117-131), packed rows of a
// contiguous cache with or without outlier channels (cache.py:221-262), and packed pages
// at the head dims that the fused dequant (dequant.hip, 128) does not take.
//
//   out[r, d] = n_g(d)[r] * sum_j c_g(j)[code(r, j)] M[j][d]
//
// With outlier channels the codes of a row are two groups (regular, then outlier), each
// with its own codebook, width, norm and rotation; M holds both rotations, its rows in
// code order and its columns in channel order, zero where row and column belong to
// different groups, so one product returns the channels in place. g[d] names the
// group of channel d.
//
// One work-group of four waves (eight at 256) per tile of 32 rows (64 at head dims up to
// 64), looping over tiles: all threads unpack the tile's codes, eight at a time, and look
// their centroids up into LDS; then each wave makes 32 output channels on
// v_mfma_f32_16x16x4f32 (fp32 operands and sums) with its part of M in registers for the
// whole launch, as the prefill's merge does. The norm multiplies the sum, so an infinite
// norm gives what it gave.
// Measured: K and V histories of 2,049 tokens (2 sequences, 8 heads, 120 channels at 4 bits
// and 8 at 8; 65,568 rows) 41.6 us in one launch, where 20 launches of one work-group per
// row took 380 us beside their unpacks, copies and masked writes. The fp32 matrix products
// are 14 us of it.
#include <algorithm>

#include "wn_common.h"

namespace wn {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct RowsGroup {
  const float* cb;   // codebook
  int bits, count;   // bits a code takes in a row, codes of the group in a row
  uint32_t mask;     // bits of a code that index the codebook
  int nb;            // bytes of a row
  int wide;          // 4: one dword holds eight codes (4-bit), 8: two (8-bit); rows aligned so. 0: bytes
};

struct RowsSide {  // K, V
  const uint8_t* codes[2];
  const uint16_t* norms[2];  // fp16
  void* out;                 // (rows, D)
};

struct RowsArgs {
  RowsSide side[2];
  RowsGroup grp[2];
  const float* m;        // (D, D)
  const uint8_t* chan;   // group of each channel; null: all group 0
  int64_t rows;
  uint32_t L;            // rows per plane
  int64_t plane_rows;    // rows between planes in codes and norms
  // pages (group 0 only, table not null): plane = sequence H + head
  const int32_t* table;
  const int32_t* lens;   // null: every sequence has L rows
  int64_t tsb, psp, psh, nsp, nsh;
  uint32_t H;
  int log2S, D, out_dtype, vec;
};

template <int KD>
struct RowsShape {
  static constexpr int CW = KD / 32, W = CW > 4 ? CW : 4, TW = W / CW, NR = 32 * TW, S = KD / 16, STRIDE = KD + 4;
};

template <int KD>
__global__ __launch_bounds__(64 * RowsShape<KD>::W) void dequant_rows_kernel(RowsArgs a) {
  using Sh = RowsShape<KD>;
  constexpr int NTHR = 64 * Sh::W, NR = Sh::NR;
  __shared__ __align__(16) float xt[NR * Sh::STRIDE];
  __shared__ float cbs[2][256];
  __shared__ int64_t off[NR];    // row of the tile: its row number in codes and norms (planes), its byte offset (pages)
  __shared__ float nrm[2][NR];
  const RowsSide& sd = a.side[blockIdx.y];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15, w = tid >> 6;
  const int d0 = 32 * (w % Sh::CW);
  const int G0 = (a.grp[0].count + 7) / 8, G1 = (a.grp[1].count + 7) / 8, groups = G0 + G1;
  for (int i = tid; i < 512; i += NTHR) {
    const RowsGroup& gr = a.grp[i >> 8];
    cbs[i >> 8][i & 255] = gr.count && uint32_t(i & 255) <= gr.mask ? gr.cb[i & 255] : 0.f;
  }
  for (int i = tid; i < NR * Sh::STRIDE; i += NTHR) xt[i] = 0.f;  // columns past D stay zero
  f32x4 m[2][Sh::S];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int s = 0; s < Sh::S; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 16 * s + 4 * g + e, d = d0 + 16 * t + c;
        m[t][s][e] = j < a.D && d < a.D ? a.m[j * a.D + d] : 0.f;
      }
  uint32_t chan = 0;  // bit 4t + i: group of channel d0 + 16t + 4g + i
  if (a.chan) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int d = d0 + 16 * (k >> 2) + 4 * g + (k & 3);
      if (d < a.D && a.chan[d]) chan |= 1u << k;
    }
  }
  const int64_t tiles = (a.rows + NR - 1) / NR;
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    if (tid < NR) {
      const int64_t r = tile * NR + tid;
      const uint32_t rc = uint32_t(r < a.rows ? r : a.rows - 1);  // rows < 2^31
      uint32_t plane = rc / a.L, t = rc % a.L;
      int64_t o, no;
      if (a.table) {
        const uint32_t b = plane / a.H;
        plane -= b * a.H;
        if (a.lens) t = min(t, uint32_t(max(a.lens[b], 1) - 1));  // rows past a length repeat the last one
        const int32_t* trow = a.table + b * a.tsb;
        const int64_t page = max(trow[t >> a.log2S], 0), slot = t & ((1u << a.log2S) - 1u);
        o = page * a.psp + plane * a.psh + slot * a.grp[0].nb;
        no = page * a.nsp + plane * a.nsh + slot;
      } else {
        o = no = int64_t(plane) * a.plane_rows + t;
      }
      off[tid] = o;
      nrm[0][tid] = f16_to_f32(sd.norms[0][no]);
      nrm[1][tid] = a.grp[1].count ? f16_to_f32(sd.norms[1][no]) : 0.f;
    }
    __syncthreads();
    for (int i = tid; i < NR * groups; i += NTHR) {
      const int rr = i / groups, q = i % groups;
      const int gi = q >= G0, k = gi ? q - G0 : q;
      const RowsGroup& gr = a.grp[gi];
      const uint8_t* p = sd.codes[gi] + (a.table ? off[rr] : off[rr] * gr.nb) + k * gr.bits;
      uint64_t v = 0;
      if (gr.wide == 4) {
        v = *reinterpret_cast<const uint32_t*>(p);
      } else if (gr.wide == 8) {
        const uint2 x = *reinterpret_cast<const uint2*>(p);
        v = uint64_t(x.y) << 32 | x.x;
      } else {
        const int n = min(gr.bits, gr.nb - k * gr.bits);
#pragma unroll
        for (int z = 0; z < 8; ++z)
          if (z < n) v |= uint64_t(p[z]) << (8 * z);
      }
      const int cnt = min(8, gr.count - 8 * k);
      float* y = xt + rr * Sh::STRIDE + (gi ? a.grp[0].count : 0) + 8 * k;
#pragma unroll
      for (int z = 0; z < 8; ++z) {
        const float cv = cbs[gi][uint32_t(v >> (z * gr.bits)) & gr.mask];
        if (z < cnt) y[z] = cv;
      }
    }
    __syncthreads();
    {
      const int sub = w / Sh::CW;
      f32x4 x[2][Sh::S > 8 ? 1 : Sh::S], acc[2][2];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[rt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      const float* xr = xt + (32 * sub + c) * Sh::STRIDE + 4 * g;
#pragma unroll
      for (int s = 0; s < Sh::S; ++s) {
        const int sx = Sh::S > 8 ? 0 : s;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) x[rt][sx] = *reinterpret_cast<const f32x4*>(xr + 16 * rt * Sh::STRIDE + 16 * s);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int t = 0; t < 2; ++t)
              acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[t][s][e], x[rt][sx][e], acc[rt][t], 0, 0, 0);
      }
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const int rr = 32 * sub + 16 * rt + c;
        const int64_t row = tile * NR + rr;
        if (row >= a.rows) continue;
        const float n0 = nrm[0][rr], n1 = nrm[1][rr];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int d = d0 + 16 * t + 4 * g;
          f32x4 v = acc[rt][t];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] *= chan >> (4 * t + i) & 1 ? n1 : n0;
          const int64_t at = row * a.D + d;
          if (a.vec) {  // D a multiple of four, out aligned to four elements
            if (d >= a.D) continue;
            if (a.out_dtype == WN_F32) {
              *reinterpret_cast<f32x4*>(static_cast<float*>(sd.out) + at) = v;
            } else {
              uint16_t h[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) h[i] = a.out_dtype == WN_BF16 ? f32_to_bf16(v[i]) : f32_to_f16(v[i]);
              *reinterpret_cast<uint2*>(static_cast<uint16_t*>(sd.out) + at) =
                  make_uint2(uint32_t(h[0]) | uint32_t(h[1]) << 16, uint32_t(h[2]) | uint32_t(h[3]) << 16);
            }
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (d + i < a.D) store_elem(sd.out, at + i, a.out_dtype, v[i]);
          }
        }
      }
    }
    __syncthreads();  // the tile is read
  }
}

int launch_rows(RowsArgs& a, int sides, hipStream_t st, const char* what) {
  if (a.rows == 0) return WN_OK;
  WN_REQUIRE(a.rows < (int64_t(1) << 31), WN_E_INVALID, "%s: too many rows", what);
  a.vec = a.D % 4 == 0;
  for (int i = 0; i < sides; ++i) a.vec = a.vec && aligned(a.side[i].out, a.out_dtype == WN_F32 ? 16 : 8);
  const int cus = device_cus();
  WN_REQUIRE(cus > 0, WN_E_LAUNCH, "%s: cannot query the device", what);
  const int KD = a.D <= 64 ? 64 : a.D <= 128 ? 128 : 256, NR = KD == 64 ? 64 : 32;
  // three work-groups of four waves fit a CU (registers): each reads M once
  const int64_t tiles = (a.rows + NR - 1) / NR;
  const dim3 grid(unsigned(std::min<int64_t>(tiles, std::max(1, 3 * cus / sides))), unsigned(sides));
  if (KD == 64) hipLaunchKernelGGL(dequant_rows_kernel<64>, grid, dim3(64 * RowsShape<64>::W), 0, st, a);
  else if (KD == 128) hipLaunchKernelGGL(dequant_rows_kernel<128>, grid, dim3(64 * RowsShape<128>::W), 0, st, a);
  else hipLaunchKernelGGL(dequant_rows_kernel<256>, grid, dim3(64 * RowsShape<256>::W), 0, st, a);
  return check_launch(what);
}

// How a group's rows may be read: eight 4- or 8-bit codes at once where every row starts
// aligned for it (step: bytes between rows, or all strides' common divisor) and no last,
// partial eight reads past its row.
int rows_wide(const uint8_t* p, int bits, int count, int64_t step) {
  if (count % 8) return 0;
  if (bits == 4 && aligned(p, 4) && step % 4 == 0) return 4;
  if (bits == 8 && aligned(p, 8) && step % 8 == 0) return 8;
  return 0;
}

RowsGroup rows_group(const float* cb, int bw, int bits, int count) {
  return RowsGroup{cb, bits, count, (1u << bw) - 1u, int((int64_t(count) * bits + 7) / 8), 0};
}

}  // namespace
}  // namespace wn

using namespace wn;

extern "C" int wn_dequantize(const uint8_t* codes, const uint16_t* norms, int64_t rows, const float* pi,
                             const float* centroids, int bw, int D, void* out, int out_dtype, void* stream) {
  clear_error();
  WN_REQUIRE(rows >= 0 && valid_bw(bw), WN_E_INVALID, "dequantize: rows=%lld bw=%d", (long long)rows, bw);
  WN_REQUIRE(D >= 1 && D <= 256, WN_E_UNSUPPORTED, "dequantize: head_dim %d (1 .. 256)", D);
  WN_REQUIRE(out_dtype >= WN_F32 && out_dtype <= WN_BF16, WN_E_INVALID, "dequantize: dtype %d", out_dtype);
  if (rows == 0) return WN_OK;
  WN_REQUIRE(rows < (int64_t(1) << 31), WN_E_INVALID, "dequantize: too many rows");
  WN_REQUIRE(codes && norms && pi && centroids && out, WN_E_INVALID, "dequantize: null operand");
  RowsArgs a{};
  a.side[0] = RowsSide{{codes, nullptr}, {norms, nullptr}, out};
  a.grp[0] = rows_group(centroids, bw, 8, D);
  a.grp[0].wide = rows_wide(codes, 8, D, D);
  a.m = pi;
  a.rows = rows;
  a.L = uint32_t(rows);
  a.plane_rows = rows;
  a.D = D;
  a.out_dtype = out_dtype;
  return launch_rows(a, 1, static_cast<hipStream_t>(stream), "wn_dequantize");
}

extern "C" int wn_dequantize_rows(const uint8_t* k_codes, const uint8_t* v_codes, const uint16_t* k_norms,
                                  const uint16_t* v_norms, int bw, const float* centroids, const uint8_t* k_codes2,
                                  const uint8_t* v_codes2, const uint16_t* k_norms2, const uint16_t* v_norms2, int bw2,
                                  const float* centroids2, int count2, const float* m, const uint8_t* channel_group,
                                  int64_t planes, int64_t L, int64_t plane_rows, int D, void* k_out, void* v_out,
                                  int out_dtype, void* stream) {
  clear_error();
  WN_REQUIRE(planes >= 0 && L >= 0 && plane_rows >= L, WN_E_INVALID, "dequantize_rows: bad sizes planes=%lld L=%lld",
             (long long)planes, (long long)L);
  WN_REQUIRE(D >= 1 && D <= 256 && count2 >= 0 && count2 < D, WN_E_UNSUPPORTED, "dequantize_rows: head_dim %d (1 .. 256), %d outlier channels",
             D, count2);
  WN_REQUIRE(valid_bw(bw) && (!count2 || valid_bw(bw2)), WN_E_INVALID, "dequantize_rows: bit widths %d/%d", bw, bw2);
  WN_REQUIRE((D - count2) * bw % 8 == 0 && (!count2 || count2 * bw2 % 8 == 0), WN_E_INVALID,
             "dequantize_rows: rows of whole bytes");
  WN_REQUIRE(out_dtype >= WN_F32 && out_dtype <= WN_BF16, WN_E_INVALID, "dequantize_rows: dtype %d", out_dtype);
  if (planes == 0 || L == 0) return WN_OK;
  WN_REQUIRE(planes * L < (int64_t(1) << 31), WN_E_INVALID, "dequantize_rows: too many rows");
  WN_REQUIRE(k_codes && k_norms && centroids && m && k_out && (!v_codes || (v_norms && v_out)), WN_E_INVALID,
             "dequantize_rows: null operand");
  WN_REQUIRE(!count2 || (k_codes2 && k_norms2 && centroids2 && channel_group && (!v_codes || (v_codes2 && v_norms2))),
             WN_E_INVALID, "dequantize_rows: null outlier operand");
  RowsArgs a{};
  a.side[0] = RowsSide{{k_codes, k_codes2}, {k_norms, k_norms2}, k_out};
  a.side[1] = RowsSide{{v_codes, v_codes2}, {v_norms, v_norms2}, v_out};
  a.grp[0] = rows_group(centroids, bw, bw, D - count2);
  const int sides = v_codes ? 2 : 1;
  a.grp[0].wide = rows_wide(k_codes, bw, a.grp[0].count, a.grp[0].nb);
  if (sides == 2 && rows_wide(v_codes, bw, a.grp[0].count, a.grp[0].nb) == 0) a.grp[0].wide = 0;
  if (count2) {
    a.grp[1] = rows_group(centroids2, bw2, bw2, count2);
    a.grp[1].wide = rows_wide(k_codes2, bw2, count2, a.grp[1].nb);
    if (sides == 2 && rows_wide(v_codes2, bw2, count2, a.grp[1].nb) == 0) a.grp[1].wide = 0;
    a.chan = channel_group;
  }
  a.m = m;
  a.rows = planes * L;
  a.L = uint32_t(L);
  a.plane_rows = plane_rows;
  a.D = D;
  a.out_dtype = out_dtype;
  return launch_rows(a, sides, static_cast<hipStream_t>(stream), "wn_dequantize_rows");
}

extern "C" int wn_dequantize_pages(const uint8_t* pages, int64_t page_stride, int64_t head_stride, const uint16_t* norms,
                                   int64_t norm_page_stride, int64_t norm_head_stride, const int32_t* page_table,
                                   int64_t table_stride_b, const int32_t* seq_lens, int B, int Lpad, int Hkv, int S,
                                   const float* centroids, const float* pi, int bw, int D, void* out, int out_dtype,
                                   void* stream) {
  clear_error();
  WN_REQUIRE(B >= 0 && Lpad >= 0 && Hkv > 0 && is_pow2(S), WN_E_INVALID,
             "dequantize_pages: bad sizes B=%d Lpad=%d Hkv=%d S=%d", B, Lpad, Hkv, S);
  WN_REQUIRE(D >= 1 && D <= 256 && valid_bw(bw) && D * bw % 8 == 0, WN_E_UNSUPPORTED, "dequantize_pages: head_dim %d, %d bits", D, bw);
  WN_REQUIRE(out_dtype >= WN_F32 && out_dtype <= WN_BF16, WN_E_INVALID, "dequantize_pages: dtype %d", out_dtype);
  if (B == 0 || Lpad == 0) return WN_OK;
  WN_REQUIRE(int64_t(B) * Hkv * Lpad < (int64_t(1) << 31), WN_E_INVALID, "dequantize_pages: too many rows");
  WN_REQUIRE(pages && norms && page_table && centroids && pi && out, WN_E_INVALID, "dequantize_pages: null operand");
  RowsArgs a{};
  a.side[0] = RowsSide{{pages, nullptr}, {norms, nullptr}, out};
  a.grp[0] = rows_group(centroids, bw, bw, D);
  a.grp[0].wide = rows_wide(pages, bw, D, page_stride | head_stride | a.grp[0].nb);
  a.m = pi;
  a.rows = int64_t(B) * Hkv * Lpad;
  a.L = uint32_t(Lpad);
  a.table = page_table;
  a.lens = seq_lens;
  a.tsb = table_stride_b;
  a.psp = page_stride;
  a.psh = head_stride;
  a.nsp = norm_page_stride;
  a.nsh = norm_head_stride;
  a.H = uint32_t(Hkv);
  a.log2S = ilog2(S);
  a.D = D;
  a.out_dtype = out_dtype;
  return launch_rows(a, 1, static_cast<hipStream_t>(stream), "wn_dequantize_pages");
}
