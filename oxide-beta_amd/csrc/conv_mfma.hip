// conv_mfma.hip -- ungrouped K x K convolutions over large planes as implicit matrix products on
// the matrix cores: the forward and the input gradient of shapes whose planes are too large for
// conv.hip's per-image LDS kernels.
//
// CPU semantics: evaluation.rs:334-445 (forward), autograd.rs:412-527 (backward).
//
// v_mfma_f32_32x32x2_f32 takes A[i][k] from lane i + 32 k and B[k][j] from lane j + 32 k and
// leaves D[i][j] in lane j + 32 ((i / 4) % 2), register i % 4 + 4 (i / 8).  Rows i are output
// channels, columns j output positions (flattened over images, so a tile may span rows and
// images and any plane size fills it), k the source channels of one kernel tap.
//   * B comes straight from global memory: lane (j, h) reads channel c + h at its position's tap,
//     32 neighbouring positions per half wave.  Per tap the byte offset of the lane's position is
//     kept in a register and the channel goes into the buffer load's scalar offset, so the inner
//     loop has no address arithmetic; a tap outside the plane carries an offset past the buffer
//     resource, which loads +0.  The K * K taps of a channel read overlapping lines, served by
//     L1.  A channel pair's loads are issued before the previous pair's products.
//   * A (the weights) is staged through LDS, rows innermost, double buffered in chunks of
//     channels: the four waves of a block share it.
// The products are added by the matrix cores' fused multiply-adds in (channel pair, tap) order:
// within 1e-5 * sum|terms| of the CPU path's serial sum, and the same on every run.
//
// 32 images of 64 x 56 x 56 to 64, 3 x 3: forward 978 -> 91 us, input gradient 995 -> 92 us (81
// TFLOP/s).  Bound by the matrix cores with too little beside them: by counters they are busy 63 %
// of the CUs' active cycles; waves wait two thirds of their time for their turn to issue and a
// fifth for loads, of which L1 serves nine in ten.
//
// The CPU path skips a tap outside the plane; the +0 operand adds 0 * weight in its place, the
// same for finite weights.  A block that meets an infinity or a NaN among its weights sums again
// and keeps, at each product, the old sum in the columns whose tap lies outside (a lane holds one
// column, so that is a select): 32 images of 64 x 56 x 56, 3 x 3, all weights NaN: 310 us.
#include <hip/hip_runtime.h>

#include "conv_mfma.h"

namespace oxh {
namespace conv_mfma {
namespace {

constexpr int kRows = 32;        // output channels of a block
constexpr int kPositions = 128;  // its positions: 32 for each of its four waves
constexpr uint32_t kNowhere = 0x80000000u;  // past every buffer resource
constexpr uint64_t kMaxBytes = 1ull << 31;  // byte offsets of one block's operands

__device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(const float *p, uint64_t elements) {
  const uint64_t bytes = elements * 4;
  return __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(p), 0,
      static_cast<int>(bytes < kMaxBytes ? static_cast<uint32_t>(bytes) : 0x7FFFFFFFu),
      0x00020000);
}
__device__ __forceinline__ float load(__amdgpu_buffer_rsrc_t r, uint32_t offset,
                                      uint32_t scalar_offset) {
  return __int_as_float(static_cast<int>(__builtin_amdgcn_raw_buffer_load_b32(
      r, static_cast<int>(offset), static_cast<int>(scalar_offset), 0)));
}
__device__ __forceinline__ bool not_finite(float v) {
  return (__float_as_uint(v) & 0x7F800000u) == 0x7F800000u;
}
// Row of D held in register r by the lanes of half h.
__device__ __forceinline__ uint32_t tile_row(int r, uint32_t h) {
  return 8u * static_cast<uint32_t>(r / 4) + 4u * h + static_cast<uint32_t>(r % 4);
}

struct TapArgs {
  const float *x, *w, *bias, *addend;  // source planes; weights; per row or null; or null
  float *y;
  uint32_t C, M, H, W;  // source channels and plane, output channels
  uint32_t OH, OW, N;   // output plane; batch * OH * OW
  uint32_t images, stride;
  int pad;              // source row of (oy, ky): oy * stride + ky - pad
  uint32_t w_m, w_c;    // weight strides of an output and of a source channel
  uint32_t row_blocks;  // blocks along M; consecutive blocks take the same positions
  FastDiv oplane_div, ow_div, row_blocks_div;
};

// The grid is row blocks x position blocks, rows fastest, each XCD taking a contiguous run.
struct Tile {
  uint32_t rows, positions;
};
__device__ __forceinline__ Tile this_tile(const TapArgs &g) {
  const uint32_t id = xcd_contiguous(blockIdx.x, gridDim.x);
  const uint32_t n = fast_div(id, g.row_blocks_div);
  return {id - n * g.row_blocks, n};
}

// Weights of CB source channels from c0 for a block's rows from m0, taps innermost in memory:
// loads into registers, then stores as lds[(c * T + tap) * kRow + m].  MFast: memory order
// (channel, row, tap), else (row, channel, tap); Flip: taps turned round.
template <int T, int CB, bool Flip, bool MFast>
struct WeightStage {
  static constexpr int BM = kRows;
  static constexpr int kRow = BM + 1;  // odd: neighbouring taps start in different banks
  static constexpr int kCount = BM * CB * T, kLoads = (kCount + 255) / 256;
  float v[kLoads];
  __device__ __forceinline__ static void at(int u, int &m, int &c, int &t) {
    const int e = static_cast<int>(threadIdx.x) + u * 256;
    t = e % T;
    const int q = e / T;
    m = MFast ? q % BM : q / CB;
    c = MFast ? q / BM : q % CB;
  }
  __device__ __forceinline__ void fetch(const TapArgs &g, __amdgpu_buffer_rsrc_t r, uint32_t m0,
                                        uint32_t c0) {
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      int m, c, t;
      at(u, m, c, t);
      const bool ok = m < BM && c < CB && m0 + m < g.M && c0 + c < g.C;
      v[u] = load(r, ok ? ((m0 + m) * g.w_m + (c0 + c) * g.w_c + t) * 4u : kNowhere, 0);
    }
  }
  __device__ __forceinline__ bool store(float *lds) const {
    bool odd = false;
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      int m, c, t;
      at(u, m, c, t);
      odd |= not_finite(v[u]);
      if (kCount % 256 == 0 || (m < BM && c < CB))
        lds[(c * T + (Flip ? T - 1 - t : t)) * kRow + m] = v[u];
    }
    return odd;
  }
};

// Forward, and input gradient of a stride-1 convolution (Flip: source = the output gradient,
// pad = K - 1 - the convolution's, taps turned round, weights read as (source, output, tap)).
// Block: 32 output channels x 128 positions, wave w the w-th 32 positions.
template <int K, bool Flip, int CB>
__global__ __launch_bounds__(256, K == 1 ? 8 : K == 3 ? 4 : 2) void conv_taps_kernel(TapArgs g) {
  constexpr int T = K * K, Pairs = CB / 2;
  using Stage = WeightStage<T, CB, Flip, Flip>;
  __shared__ float wl[2][CB * T * Stage::kRow];
  const Tile tile = this_tile(g);
  const uint32_t m0 = tile.rows * kRows, wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const uint32_t j = lane % 32, h = lane / 32;
  const uint32_t plane = g.H * g.W, oplane = g.OH * g.OW, image = g.C * plane;
  const uint32_t first = tile.positions * kPositions, n0 = fast_div(first, g.oplane_div);
  const __amdgpu_buffer_rsrc_t xr = resource(g.x + static_cast<uint64_t>(n0) * image,
                                             static_cast<uint64_t>(g.images - n0) * image);
  const __amdgpu_buffer_rsrc_t wr =
      resource(g.w, static_cast<uint64_t>(g.M) * g.C * T);

  const uint32_t pos = first + wave * 32 + j, pc = pos < g.N ? pos : g.N - 1;
  const uint32_t n = fast_div(pc, g.oplane_div), q = pc - n * oplane;
  const uint32_t oy = fast_div(q, g.ow_div), ox = q - oy * g.OW;
  const int by = static_cast<int>(oy * g.stride) - g.pad;
  const int bx = static_cast<int>(ox * g.stride) - g.pad;
  uint32_t off[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int iy = by + t / K, ix = bx + t % K;
    const bool ok = static_cast<uint32_t>(iy) < g.H && static_cast<uint32_t>(ix) < g.W;
    off[t] = ok ? ((n - n0) * image + h * plane + static_cast<uint32_t>(iy) * g.W +
                   static_cast<uint32_t>(ix)) * 4u
                : kNowhere;
  }
  f32x16 acc;
  auto start = [&](const float *bias) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t m = m0 + tile_row(r, h);
      acc[r] = bias != nullptr && m < g.M ? bias[m] : 0.0f;
    }
  };
  start(g.bias);
  // the pair of channels c, c + 1 at every tap (+0 past the channels)
  auto fetch = [&](uint32_t c, float (&b)[T]) {
    const uint32_t past = c + h < g.C ? 0u : kNowhere;
    const uint32_t at = c < g.C ? c * plane * 4u : 0u;
#pragma unroll
    for (int t = 0; t < T; ++t) b[t] = load(xr, off[t] | past, at);
  };
  Stage ws;
  ws.fetch(g, wr, m0, 0);
  float b[2][T];
  fetch(0, b[0]);
  bool odd = ws.store(wl[0]);
  uint32_t buf = 0;
  for (uint32_t c0 = 0; c0 < g.C; c0 += CB, buf ^= 1) {
    __syncthreads();
    const bool more = c0 + CB < g.C;
    if (more) ws.fetch(g, wr, m0, c0 + CB);
    const float *wa = &wl[buf][h * T * Stage::kRow + j];
#pragma unroll
    for (int p = 0; p < Pairs; ++p) {
      if (c0 + 2 * p >= g.C) break;
      fetch(c0 + 2 * p + 2, b[(p + 1) % 2]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < T; ++t)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wa[(2 * p * T + t) * Stage::kRow], b[p % 2][t],
                                                   acc, 0, 0, 0);
    }
    if (more) odd |= ws.store(wl[buf ^ 1]);
  }
  if (__syncthreads_or(odd) != 0) {  // one product at a time, both operands from memory
    const float *bias = g.bias;
    asm volatile("" : "+s"(bias));  // loaded again, not held in registers over the sums
    start(bias);
    const uint32_t row = m0 + j < g.M ? ((m0 + j) * g.w_m + h * g.w_c) * 4u : kNowhere;
#pragma unroll 1
    for (uint32_t c = 0; c < g.C; c += 2) {
      const uint32_t past = c + h < g.C ? 0u : kNowhere;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        multiply_in(load(wr, row | past, (c * g.w_c + (Flip ? T - 1 - t : t)) * 4u),
                    load(xr, off[t] | past, c * plane * 4u), off[t] != kNowhere, acc);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if (pos >= g.N) return;
  const uint64_t at = static_cast<uint64_t>(n) * g.M * oplane + q;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t m = m0 + tile_row(r, h);
    if (m >= g.M) continue;
    const uint64_t o = at + static_cast<uint64_t>(m) * oplane;
    g.y[o] = g.addend != nullptr ? acc[r] + g.addend[o] : acc[r];
  }
}

// Input gradient of a stride-2 convolution.  With yy = y + pad = 2 a + py, the outputs an input
// row feeds are oy = a - i through ky = py + 2 i < K: the four inputs (2 a + py - pad,
// 2 b + px - pad) share their M2 x M2 output positions (M2 = ceil(K / 2)) and each of the K * K
// taps belongs to one of them.  Block: 32 input channels x 128 (a, b) positions, wave w the w-th
// 32; four accumulators (py, px), so an operand load serves up to four products and nothing is
// multiplied that no tap asks for.
struct PhaseArgs {
  TapArgs t;            // x: the output gradient (C channels of H x W); M, OH, OW: the input's
  uint32_t a0, na, nb;  // positions a in [a0, a0 + na), b in [a0, a0 + nb); N = images * na * nb
  FastDiv ab_div, nb_div;
};

template <int K, int CB>
__global__ __launch_bounds__(256, K == 1 ? 8 : 2) void conv_input_s2_kernel(PhaseArgs p) {
  constexpr int T = K * K, Pairs = CB / 2, M2 = (K + 1) / 2, B = M2 * M2;
  constexpr int Ahead = Pairs % 4 == 0 && B <= 4 ? 4 : 2;  // operand register sets
  using Stage = WeightStage<T, CB, false, true>;
  __shared__ float wl[2][CB * T * Stage::kRow];
  const TapArgs &g = p.t;
  const Tile tile = this_tile(g);
  const uint32_t m0 = tile.rows * kRows, wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const uint32_t j = lane % 32, h = lane / 32;
  const uint32_t plane = g.H * g.W, image = g.C * plane, ab = p.na * p.nb;
  const uint32_t first = tile.positions * kPositions, n0 = fast_div(first, p.ab_div);
  const __amdgpu_buffer_rsrc_t xr = resource(g.x + static_cast<uint64_t>(n0) * image,
                                             static_cast<uint64_t>(g.images - n0) * image);
  const __amdgpu_buffer_rsrc_t wr =
      resource(g.w, static_cast<uint64_t>(g.M) * g.C * T);
  const uint32_t pos = first + wave * 32 + j;
  const uint32_t pc = pos < g.N ? pos : g.N - 1;
  const uint32_t n = fast_div(pc, p.ab_div), q = pc - n * ab;
  const uint32_t qa = fast_div(q, p.nb_div);
  const uint32_t a = p.a0 + qa, bcol = p.a0 + (q - qa * p.nb);
  uint32_t off[B];
#pragma unroll
  for (int i = 0; i < B; ++i) {
    const int oy = static_cast<int>(a) - i / M2, ox = static_cast<int>(bcol) - i % M2;
    const bool ok = static_cast<uint32_t>(oy) < g.H && static_cast<uint32_t>(ox) < g.W;
    off[i] = ok ? ((n - n0) * image + h * plane + static_cast<uint32_t>(oy) * g.W +
                   static_cast<uint32_t>(ox)) * 4u
                : kNowhere;
  }
  f32x16 acc[4];
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[f][r] = 0.0f;
  auto fetch = [&](uint32_t c, float (&b)[B]) {
    const uint32_t past = c + h < g.C ? 0u : kNowhere;
    const uint32_t at = c < g.C ? c * plane * 4u : 0u;
#pragma unroll
    for (int i = 0; i < B; ++i) b[i] = load(xr, off[i] | past, at);
  };
  Stage ws;
  ws.fetch(g, wr, m0, 0);
  float b[Ahead][B];
#pragma unroll
  for (int s = 0; s + 1 < Ahead; ++s) fetch(2 * s, b[s]);
  bool odd = ws.store(wl[0]);
  uint32_t buf = 0;
  for (uint32_t c0 = 0; c0 < g.C; c0 += CB, buf ^= 1) {
    __syncthreads();
    const bool more = c0 + CB < g.C;
    if (more) ws.fetch(g, wr, m0, c0 + CB);
    const float *wa = &wl[buf][h * T * Stage::kRow + j];
#pragma unroll
    for (int s = 0; s < Pairs; ++s) {
      if (c0 + 2 * s >= g.C) break;
      fetch(c0 + 2 * s + 2 * (Ahead - 1), b[(s + Ahead - 1) % Ahead]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int ky = t / K, kx = t % K, f = (ky % 2) * 2 + kx % 2;
        acc[f] = __builtin_amdgcn_mfma_f32_32x32x2f32(wa[(2 * s * T + t) * Stage::kRow],
                                                      b[s % Ahead][(ky / 2) * M2 + kx / 2],
                                                      acc[f], 0, 0, 0);
      }
    }
    if (more) odd |= ws.store(wl[buf ^ 1]);
  }
  if (__syncthreads_or(odd) != 0) {  // as in conv_taps_kernel
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[f][r] = 0.0f;
    const uint32_t row = m0 + j < g.M ? ((m0 + j) * g.w_m + h * g.w_c) * 4u : kNowhere;
#pragma unroll 1
    for (uint32_t c = 0; c < g.C; c += 2) {
      const uint32_t past = c + h < g.C ? 0u : kNowhere;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int ky = t / K, kx = t % K, i = (ky / 2) * M2 + kx / 2;
        multiply_in(load(wr, row | past, (c * g.w_c + t) * 4u),
                    load(xr, off[i] | past, c * plane * 4u), off[i] != kNowhere,
                    acc[(ky % 2) * 2 + kx % 2]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if (pos >= g.N) return;
  const uint32_t oplane = g.OH * g.OW;
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const int y = 2 * static_cast<int>(a) + f / 2 - g.pad;
    const int x = 2 * static_cast<int>(bcol) + f % 2 - g.pad;
    if (static_cast<uint32_t>(y) >= g.OH || static_cast<uint32_t>(x) >= g.OW) continue;
    const uint64_t at = static_cast<uint64_t>(n) * g.M * oplane +
                        static_cast<uint32_t>(y) * g.OW + static_cast<uint32_t>(x);
    float *dx = g.y + at;
    const float *add = g.addend != nullptr ? g.addend + at : nullptr;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t m = m0 + tile_row(r, h);
      if (m >= g.M) continue;
      const uint64_t o = static_cast<uint64_t>(m) * oplane;
      dx[o] = add != nullptr ? acc[f][r] + add[o] : acc[f][r];
    }
  }
}

// ---------------------------------------------------------------- host side

// Bytes of the images one block's positions can touch (`per_image` positions each).
bool fits(uint64_t block, uint64_t per_image, uint64_t image_elements) {
  return ((block - 1) / per_image + 2) * image_elements * 4 < kMaxBytes;
}

bool square_kernel(const Dims &d) { return d.k == 1 || d.k == 3 || d.k == 5; }

dim3 set_grid(TapArgs &g) {
  g.row_blocks = (g.M + kRows - 1) / kRows;
  g.row_blocks_div = make_fastdiv(g.row_blocks);
  return dim3(g.row_blocks * ((g.N + kPositions - 1) / kPositions));
}

// Channels per weight stage: 8 (3 x 3), 4 (5 x 5) or 16 (1 x 1), 18 to 26 KB of LDS.
template <bool Flip>
void launch_taps(hipStream_t s, uint32_t k, TapArgs g) {
  const dim3 grid = set_grid(g), threads(256);
  if (k == 3) launch(conv_taps_kernel<3, Flip, 8>, grid, threads, 0, s, g);
  else if (k == 5) launch(conv_taps_kernel<5, Flip, 4>, grid, threads, 0, s, g);
  else launch(conv_taps_kernel<1, Flip, 16>, grid, threads, 0, s, g);
}

void launch_s2(hipStream_t s, uint32_t k, PhaseArgs p) {
  const dim3 grid = set_grid(p.t), threads(256);
  if (k == 3) launch(conv_input_s2_kernel<3, 8>, grid, threads, 0, s, p);
  else if (k == 5) launch(conv_input_s2_kernel<5, 4>, grid, threads, 0, s, p);
  else launch(conv_input_s2_kernel<1, 16>, grid, threads, 0, s, p);
}

// Tiles of 128 positions x 32 rows fit a one-dimensional grid of 256 threads each.
bool grid_fits(uint64_t positions, uint64_t rows) {
  return positions < (1ull << 31) - 512 &&
         (positions + 127) / 128 * ((rows + 31) / 32) < (1ull << 23);
}

PhaseArgs phase_args(const Dims &d) {
  PhaseArgs p{};
  p.a0 = d.pad / 2;
  p.na = (d.h - 1 + d.pad) / 2 - p.a0 + 1;
  p.nb = (d.w - 1 + d.pad) / 2 - p.a0 + 1;
  return p;
}

}  // namespace

bool takes_forward(const Dims &d) {
  const uint64_t positions = static_cast<uint64_t>(d.batch) * d.oh * d.ow;
  const uint64_t weights = static_cast<uint64_t>(d.out_c) * d.in_c * d.k * d.k;
  return square_kernel(d) && !(d.k == 1 && d.stride == 1 && d.pad == 0) &&
         grid_fits(positions, d.out_c) && weights * 4 < kMaxBytes && d.pad < 4 * d.k &&
         fits(kPositions, static_cast<uint64_t>(d.oh) * d.ow,
              static_cast<uint64_t>(d.in_c) * d.h * d.w);
}

bool takes_input_backward(const Dims &d) {
  if (d.stride > 2 || d.pad >= 4 * d.k) return false;
  const uint64_t weights = static_cast<uint64_t>(d.out_c) * d.in_c * d.k * d.k;
  const PhaseArgs p = phase_args(d);
  const uint64_t per_image = d.stride == 1 ? static_cast<uint64_t>(d.h) * d.w
                                           : static_cast<uint64_t>(p.na) * p.nb;
  const uint64_t positions = d.batch * per_image;
  return square_kernel(d) && !(d.k == 1 && d.stride == 1 && d.pad == 0) &&
         grid_fits(positions, d.in_c) && weights * 4 < kMaxBytes &&
         fits(kPositions, per_image, static_cast<uint64_t>(d.out_c) * d.oh * d.ow);
}

void forward(hipStream_t s, const Dims &d, const float *x, const float *weight,
             const float *bias, float *y) {
  TapArgs g{};
  g.x = x, g.w = weight, g.bias = bias, g.y = y;
  g.C = d.in_c, g.M = d.out_c, g.H = d.h, g.W = d.w, g.OH = d.oh, g.OW = d.ow;
  g.N = d.batch * d.oh * d.ow, g.images = d.batch, g.stride = d.stride;
  g.pad = static_cast<int>(d.pad);
  g.w_m = d.in_c * d.k * d.k, g.w_c = d.k * d.k;
  g.oplane_div = make_fastdiv(d.oh * d.ow), g.ow_div = make_fastdiv(d.ow);
  launch_taps<false>(s, d.k, g);
}

void input_backward(hipStream_t s, const Dims &d, const float *gradient, const float *weight,
                    const float *addend, float *dx) {
  TapArgs g{};
  g.x = gradient, g.w = weight, g.addend = addend, g.y = dx;
  g.C = d.out_c, g.M = d.in_c, g.H = d.oh, g.W = d.ow, g.OH = d.h, g.OW = d.w;
  g.images = d.batch, g.stride = 1;
  g.w_m = d.k * d.k, g.w_c = d.in_c * d.k * d.k;
  if (d.stride == 1) {
    g.N = d.batch * d.h * d.w;
    g.pad = static_cast<int>(d.k) - 1 - static_cast<int>(d.pad);
    g.oplane_div = make_fastdiv(d.h * d.w), g.ow_div = make_fastdiv(d.w);
    launch_taps<true>(s, d.k, g);
    return;
  }
  PhaseArgs p = phase_args(d);
  g.N = d.batch * p.na * p.nb;
  g.pad = static_cast<int>(d.pad);
  p.t = g;
  p.ab_div = make_fastdiv(p.na * p.nb), p.nb_div = make_fastdiv(p.nb);
  launch_s2(s, d.k, p);
}

}  // namespace conv_mfma
}  // namespace oxh
