// conv_weight_mfma.hip -- weight gradients of ungrouped convolutions over large planes on the
// matrix cores (conv_mfma.h; autograd.rs:412-527).
//
// dW[oc][(ic, tap)] = sum over output positions of G[oc][p] * X[ic][p's tap]: a product of
// out_c rows x (in_c * taps) columns over k = (image, oy, ox), k cut into chunks whose partial
// sums a second launch adds in order (chunk_sum.h).
//   * A block takes 32 or 64 rows x 32 CT columns and walks its chunk in groups of whole output
//     rows of one image.  Per group it stages the gradient rows and the source rows the group's
//     taps reach, zero around the plane, in LDS: each source value serves every tap and row of
//     the block.
//   * v_mfma_f32_32x32x2_f32 (lane layout: conv_mfma.hip): per 8 positions, lane (i, h) reads
//     four of its row's gradient values as one 128-bit access and a table entry with the offsets
//     of those positions in the staged rows; its column's offset added, each of the four products
//     per column tile then takes one LDS read.  The position table is the same for every group,
//     so the inner loop has one addition per product.
//   * The waves split the rows (two row tiles) and the positions; the position parts are summed
//     with the chunks.  Two blocks per CU (at most kLdsBytes each): one stages while the other
//     multiplies.
// Fused multiply-adds in a fixed order: within 1e-5 * sum|terms| of the CPU path's running sum,
// the same on every run.  The CPU path skips taps outside the plane where these products have a
// zero: the same for finite gradients; a block that meets an infinity or a NaN among its
// gradients sums its chunk again, one position per product, and keeps the old sum in the columns
// whose tap lies outside (a lane holds one column: a select).
//
// 32 images of 64 x 56 x 56 to 64, 3 x 3: 5212 -> 137 us, 13 of them the chunks' sums (54
// TFLOP/s).  By counters the matrix cores are busy 45 % of the CUs' active cycles and waves wait
// half of their time for their turn to issue; address additions and LDS reads, one of each per
// product, and the staging between barriers take the rest.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "conv_mfma.h"

namespace oxh {
namespace conv_mfma {
namespace {

constexpr uint32_t kNowhere = 0x80000000u;  // past every buffer resource
constexpr uint64_t kMaxBytes = 1ull << 31;
constexpr uint32_t kLdsBytes = 78 * 1024;   // two blocks in a CU's 160 KB
constexpr uint32_t kMaxGroup = 512;         // positions of a group
constexpr uint32_t kBlocks = 2 * kComputeUnits;

struct WeightArgs {
  const float *g, *x;
  float *out;
  uint32_t C, M, H, W, OH, OW, KW, taps, stride;
  int pad;
  uint32_t rows;       // output rows per group
  uint32_t gpos;       // its positions, padded to 8
  uint32_t gp;         // floats between the staged gradient rows
  uint32_t srows, pw;  // staged source rows and columns per channel
  uint32_t ps;         // floats between the staged channels
  uint32_t channels;   // staged channels of a block
  uint32_t wm;         // row tiles of a block (1 or 2); 4 / wm position parts
  uint32_t per_image, groups, per_chunk;  // groups
  uint32_t tiles, row_blocks, out_stride;
  FastDiv tiles_div, row_blocks_div, per_image_div, gpos_div, srows_pw_div, pw_div, ow_div,
      taps_div, kw_div;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(const float *p, uint64_t elements) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0,
                                           static_cast<int>(elements * 4), 0x00020000);
}
__device__ __forceinline__ float load(__amdgpu_buffer_rsrc_t r, uint32_t offset) {
  return __int_as_float(static_cast<int>(
      __builtin_amdgcn_raw_buffer_load_b32(r, static_cast<int>(offset), 0, 0)));
}

template <int CT>
__global__ __launch_bounds__(256, 2) void conv_weight_kernel(WeightArgs a) {
  extern __shared__ float lds[];
  const uint32_t id = xcd_contiguous(blockIdx.x, gridDim.x);
  const uint32_t chunk = fast_div(id, a.tiles_div), tile = id - chunk * a.tiles;
  const uint32_t column_block = fast_div(tile, a.row_blocks_div);
  const uint32_t m0 = (tile - column_block * a.row_blocks) * 32 * a.wm;
  const uint32_t col0 = column_block * 32 * CT, columns = a.C * a.taps;
  const uint32_t ic0 = fast_div(col0, a.taps_div);
  const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 32, h = lane / 32;
  const uint32_t wm = wave % a.wm, part = wave / a.wm, parts = 4 / a.wm;
  const uint32_t plane = a.H * a.W, oplane = a.OH * a.OW;
  int *table = reinterpret_cast<int *>(lds);
  float *gl = lds + a.gpos, *xl = gl + 32 * a.wm * a.gp;
  for (uint32_t p = threadIdx.x; p < a.gpos; p += 256) {
    const uint32_t oy = fast_div(p, a.ow_div), ox = p - oy * a.OW;
    table[p] = static_cast<int>(oy < a.rows ? (oy * a.pw + ox) * a.stride : 0u);
  }
  uint32_t at[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const uint32_t col = min(col0 + 32 * ct + j, columns - 1);
    const uint32_t ic = fast_div(col, a.taps_div), tap = col - ic * a.taps;
    const uint32_t ky = fast_div(tap, a.kw_div);
    at[ct] = (ic - ic0) * a.ps + ky * a.pw + (tap - ky * a.KW);
  }
  f32x16 acc[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[ct][r] = 0.0f;
  const uint32_t first = chunk * a.per_chunk, last = min(first + a.per_chunk, a.groups);
  const uint32_t gcount = 32 * a.wm * a.gpos, xcount = a.channels * a.srows * a.pw;
  bool odd = false;
  for (uint32_t gi = first; gi < last; ++gi) {
    const uint32_t n = fast_div(gi, a.per_image_div);
    const uint32_t oy0 = (gi - n * a.per_image) * a.rows;
    const uint32_t count = min(a.rows, a.OH - oy0) * a.OW;
    const __amdgpu_buffer_rsrc_t gr =
        resource(a.g + static_cast<uint64_t>(n) * a.M * oplane,
                 static_cast<uint64_t>(a.M) * oplane);
    const __amdgpu_buffer_rsrc_t xr = resource(a.x + static_cast<uint64_t>(n) * a.C * plane,
                                               static_cast<uint64_t>(a.C) * plane);
    const int iy0 = static_cast<int>(oy0 * a.stride) - a.pad;
    __syncthreads();  // the previous group's values are read
    constexpr int U = 8;
    for (uint32_t b = threadIdx.x; b < gcount; b += 256 * U) {
      float v[U];
      uint32_t to[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t e = b + 256 * u, oc = fast_div(e, a.gpos_div), p = e - oc * a.gpos;
        const bool ok = e < gcount && p < count && m0 + oc < a.M;
        v[u] = load(gr, ok ? ((m0 + oc) * oplane + oy0 * a.OW + p) * 4u : kNowhere);
        to[u] = oc * a.gp + p;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        odd |= (__float_as_uint(v[u]) & 0x7F800000u) == 0x7F800000u;
        if (b + 256 * u < gcount) gl[to[u]] = v[u];
      }
    }
    for (uint32_t b = threadIdx.x; b < xcount; b += 256 * U) {
      float v[U];
      uint32_t to[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t e = b + 256 * u, ic = fast_div(e, a.srows_pw_div);
        const uint32_t q = e - ic * (a.srows * a.pw), row = fast_div(q, a.pw_div);
        const int iy = iy0 + static_cast<int>(row);
        const int ix = static_cast<int>(q - row * a.pw) - a.pad;
        const bool ok = e < xcount && ic0 + ic < a.C && static_cast<uint32_t>(iy) < a.H &&
                        static_cast<uint32_t>(ix) < a.W;
        v[u] = load(xr, ok ? ((ic0 + ic) * plane + static_cast<uint32_t>(iy) * a.W +
                              static_cast<uint32_t>(ix)) * 4u
                           : kNowhere);
        to[u] = ic * a.ps + q;
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (b + 256 * u < xcount) xl[to[u]] = v[u];
    }
    __syncthreads();
    const float *ga = gl + (32 * wm + j) * a.gp + 4 * h;
    const int *ta = table + 4 * h;
    for (uint32_t p = 8 * part; p < count; p += 8 * parts) {
      const float4 g4 = *reinterpret_cast<const float4 *>(ga + p);
      const int4 t4 = *reinterpret_cast<const int4 *>(ta + p);
      const float gv[4] = {g4.x, g4.y, g4.z, g4.w};
      const int tv[4] = {t4.x, t4.y, t4.z, t4.w};
      if (p + 8 <= count) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
            acc[ct] = __builtin_amdgcn_mfma_f32_32x32x2f32(gv[s], xl[at[ct] + tv[s]], acc[ct], 0,
                                                           0, 0);
      } else {  // positions past the group: zero in both operands
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const bool in = p + 4 * h + s < count;
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            const float b = xl[at[ct] + tv[s]];
            acc[ct] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? gv[s] : 0.0f, in ? b : 0.0f,
                                                           acc[ct], 0, 0, 0);
          }
        }
      }
    }
  }
  float *out = a.out + static_cast<uint64_t>(chunk * parts + part) * a.out_stride;
  const auto store = [&](uint32_t col, const f32x16 &sums) {
    if (col >= columns) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t m = m0 + 32 * wm + 8u * (r / 4) + 4u * h + r % 4;
      if (m < a.M) out[m * columns + col] = sums[r];
    }
  };
  if (__syncthreads_or(odd) == 0) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) store(col0 + 32 * ct + j, acc[ct]);
    return;
  }
  // a position per product and a column tile at a time, both operands from memory
  const uint32_t m = m0 + 32 * wm + j;
#pragma unroll 1
  for (uint32_t c0 = col0; c0 < col0 + 32 * CT && c0 < columns; c0 += 32) {
    const uint32_t col = min(c0 + j, columns - 1);
    const uint32_t ic = fast_div(col, a.taps_div), tap = col - ic * a.taps;
    const uint32_t ky = fast_div(tap, a.kw_div), kx = tap - ky * a.KW;
    f32x16 sums = {};
#pragma unroll 1
    for (uint32_t gi = first; gi < last; ++gi) {
      const uint32_t n = fast_div(gi, a.per_image_div);
      const uint32_t oy0 = (gi - n * a.per_image) * a.rows;
      const uint32_t count = min(a.rows, a.OH - oy0) * a.OW;
      const __amdgpu_buffer_rsrc_t gr =
          resource(a.g + static_cast<uint64_t>(n) * a.M * oplane,
                   static_cast<uint64_t>(a.M) * oplane);
      const __amdgpu_buffer_rsrc_t xr = resource(a.x + static_cast<uint64_t>(n) * a.C * plane,
                                                 static_cast<uint64_t>(a.C) * plane);
      constexpr uint32_t U = 4;  // positions in flight
#pragma unroll 1
      for (uint32_t p0 = part; p0 < count; p0 += U * parts) {
        float gv[U], xv[U];
        bool in[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
          const uint32_t p = p0 + u * parts, row = fast_div(p, a.ow_div);
          const uint32_t iy = (oy0 + row) * a.stride + ky - static_cast<uint32_t>(a.pad);
          const uint32_t ix = (p - row * a.OW) * a.stride + kx - static_cast<uint32_t>(a.pad);
          in[u] = p < count && iy < a.H && ix < a.W;
          const bool mine = h == 0 && p < count;  // the other half's position: +0 both
          gv[u] = load(gr, mine && m < a.M ? (m * oplane + oy0 * a.OW + p) * 4u : kNowhere);
          xv[u] = load(xr, mine && in[u] ? (ic * plane + iy * a.W + ix) * 4u : kNowhere);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) multiply_in(gv[u], xv[u], in[u], sums);
      }
    }
    store(c0 + j, sums);
  }
}

// The launch of a shape: column tiles per block, the group of rows, LDS.  lds == 0: not taken.
struct Plan {
  WeightArgs a{};
  int ct = 0;
  uint32_t chunks = 0, lds = 0;
  double cycles = 0;  // estimated
};

Plan make_plan(const WeightDims &d) {
  Plan best;
  const uint64_t columns = static_cast<uint64_t>(d.in_c) * d.kh * d.kw;
  const uint64_t weights = columns * d.out_c;
  if (static_cast<uint64_t>(d.in_c) * d.h * d.w * 4 >= kMaxBytes ||
      static_cast<uint64_t>(d.out_c) * d.oh * d.ow * 4 >= kMaxBytes || weights >= (1u << 29) ||
      d.ow > kMaxGroup || d.pad > (1u << 12) || d.stride > (1u << 12))
    return best;
  const uint32_t taps = d.kh * d.kw, mtiles = (d.out_c + 31) / 32;
  const uint32_t ntiles = static_cast<uint32_t>((columns + 31) / 32);
  const uint32_t wm = mtiles % 2 == 0 ? 2 : 1;
  // the column tiles and rows per group with the least estimated time, in cycles: per group the
  // products (64 cycles each, the SIMDs shared when a CU has two blocks), the staging (about 14
  // cycles of the block's time per value and thread) and two memory round trips, then the sums
  // of the chunks' partials at 1700 bytes per cycle
  double least = 1e300;
  for (int ct : {9, 5, 3, 2, 1}) {
    const uint32_t tiles = (ntiles + ct - 1) / ct * ((mtiles + wm - 1) / wm);
    uint32_t channels = (32 * ct + taps - 2) / taps + 1;
    if (channels > d.in_c) channels = d.in_c;
    const uint32_t pw = (d.ow - 1) * d.stride + d.kw;
    for (uint32_t rows = 1; rows <= d.oh && rows * d.ow <= kMaxGroup; ++rows) {
      const uint32_t gpos = (rows * d.ow + 7) / 8 * 8, gp = gpos + 4;
      const uint64_t srows = static_cast<uint64_t>(rows - 1) * d.stride + d.kh;
      const uint64_t ps = srows * pw | 1u;
      const uint64_t lds = (gpos + 32ull * wm * gp + channels * ps) * 4;
      if (lds > kLdsBytes) break;
      const double groups = static_cast<double>(d.batch) * ((d.oh + rows - 1) / rows);
      const double chunks = std::min(groups, std::ceil(static_cast<double>(kBlocks) / tiles));
      const double blocks = chunks * tiles;
      const double share = std::min(2.0, std::max(1.0, blocks / kComputeUnits));
      const double multiply = 64.0 * gpos / 2 * ct * wm / 4 * share;
      const double staging = 14.0 * (32.0 * wm * gpos + channels * srows * pw) / 256;
      const double cycles = std::ceil(blocks / kBlocks) * std::ceil(groups / chunks) *
                                (multiply + staging + 4000.0) +
                            chunks * (4 / wm) * weights * 8.0 / 1700.0;
      if (cycles < least) {
        least = cycles;
        best.ct = ct;
        best.lds = static_cast<uint32_t>(lds);
        best.a.rows = rows, best.a.gpos = gpos, best.a.gp = gp;
        best.a.srows = static_cast<uint32_t>(srows), best.a.pw = pw;
        best.a.ps = static_cast<uint32_t>(ps), best.a.channels = channels;
      }
    }
  }
  if (best.lds == 0) return best;
  best.cycles = least;
  WeightArgs &a = best.a;
  a.C = d.in_c, a.M = d.out_c, a.H = d.h, a.W = d.w, a.OH = d.oh, a.OW = d.ow;
  a.KW = d.kw, a.taps = taps, a.stride = d.stride, a.pad = static_cast<int>(d.pad), a.wm = wm;
  a.row_blocks = (mtiles + wm - 1) / wm;
  a.tiles = a.row_blocks * ((ntiles + best.ct - 1) / best.ct);
  a.per_image = (d.oh + a.rows - 1) / a.rows;
  a.out_stride = static_cast<uint32_t>(weights);
  const uint64_t groups = static_cast<uint64_t>(d.batch) * a.per_image;
  if (groups >= (1ull << 31)) return Plan{};
  a.groups = static_cast<uint32_t>(groups);
  // chunks for two blocks on each CU
  uint64_t chunks = (kBlocks + a.tiles - 1) / a.tiles;
  if (chunks > groups) chunks = groups;
  while (chunks > 1 && chunks * (4 / wm) * weights >= (1ull << 31)) --chunks;
  if (chunks * (4 / wm) * weights >= (1ull << 31) || chunks * a.tiles >= (1u << 23))
    return Plan{};
  a.per_chunk = static_cast<uint32_t>((groups + chunks - 1) / chunks);
  best.chunks = static_cast<uint32_t>((groups + a.per_chunk - 1) / a.per_chunk);
  a.tiles_div = make_fastdiv(a.tiles), a.row_blocks_div = make_fastdiv(a.row_blocks);
  a.per_image_div = make_fastdiv(a.per_image), a.gpos_div = make_fastdiv(a.gpos);
  a.srows_pw_div = make_fastdiv(a.srows * a.pw), a.pw_div = make_fastdiv(a.pw);
  a.ow_div = make_fastdiv(a.OW), a.taps_div = make_fastdiv(taps);
  a.kw_div = make_fastdiv(d.kw);
  return best;
}

// make_plan weighs some dozens of layouts (a few us of host time) and a backward asks for the
// same shape's plan several times: each thread keeps its last one, a pure function of the shape.
const Plan &plan_of(const WeightDims &d) {
  thread_local WeightDims last{};
  thread_local Plan plan;
  if (std::memcmp(&last, &d, sizeof d) != 0) {
    plan = make_plan(d);
    last = d;
  }
  return plan;
}

}  // namespace

uint32_t weight_partials(const WeightDims &d) {
  const Plan &p = plan_of(d);
  return p.lds == 0 ? 0 : p.chunks * (4 / p.a.wm);
}

double weight_time(const WeightDims &d) { return 5.0 + 1.8 * plan_of(d).cycles / 2400; }

void weight_backward(hipStream_t s, const WeightDims &d, const float *gradient, const float *x,
                     float *out) {
  Plan p = plan_of(d);
  p.a.g = gradient, p.a.x = x, p.a.out = out;
  const dim3 grid(p.chunks * p.a.tiles), threads(256);
  switch (p.ct) {
    case 9: launch(conv_weight_kernel<9>, grid, threads, p.lds, s, p.a); break;
    case 5: launch(conv_weight_kernel<5>, grid, threads, p.lds, s, p.a); break;
    case 3: launch(conv_weight_kernel<3>, grid, threads, p.lds, s, p.a); break;
    case 2: launch(conv_weight_kernel<2>, grid, threads, p.lds, s, p.a); break;
    default: launch(conv_weight_kernel<1>, grid, threads, p.lds, s, p.a);
  }
}

}  // namespace conv_mfma
}  // namespace oxh
