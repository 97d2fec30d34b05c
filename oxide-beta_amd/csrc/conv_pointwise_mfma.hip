// conv_pointwise_mfma.hip -- 1 x 1 convolutions over large planes (stride 1, no padding, one
// group) on the matrix cores: the forward and the input gradient (conv_mfma.h).
//
// Y[m][(n, p)] = bias[m] + sum over k of W[m][k] X[(n, k)][p] (+ addend), or with the weight read
// the other way round the input gradient.  v_mfma_f32_32x32x2_f32 (lane layout: conv_mfma.hip),
// rows m, columns positions:
//   * The operand that streams, X, goes straight from global memory into the matrix cores'
//     registers: lane (j, h) loads NT neighbouring positions of channel k + h as one access and
//     column j of tile t is position NT j + t, so the NT results of a lane are neighbours too
//     and leave as one store.  A chunk of channels is loaded while the previous one is
//     multiplied.
//   * The weights of 32 rows and a chunk of channels go through LDS, double buffered, shared by
//     the block's waves.
//   * Grids that leave the chip idle take a kernel whose blocks split the channels over their
//     waves instead (conv_point_split_kernel).
// Blocks with the same positions are neighbours on one XCD, so the rows' blocks share X in its
// L2.  Fused multiply-adds in a fixed order, within 1e-5 * sum|terms| of the CPU path's sum.
//
// 64 images of 64 x 56 x 56 to 192: forward 237 -> 79 us, input gradient 177 -> 65 us.  Neither
// memory (205 MB: 33 us at the rate of a large copy) nor the matrix cores (33 us) bind alone: by
// counters these are busy 48 and 64 % of the CUs' active cycles, waves wait 56 and 61 % of their
// time for their turn to issue behind each other's products and 29 and 25 % for loads.  X comes
// from L2 once per 32 rows (six times forward, twice in the input gradient).
#include <hip/hip_runtime.h>

#include "conv_mfma.h"

namespace oxh {
namespace conv_mfma {
namespace {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kRows = 32;
constexpr uint32_t kNowhere = 0x80000000u;  // past every buffer resource
constexpr uint64_t kMaxBytes = 1ull << 31;

struct PointArgs {
  const float *x, *w, *bias, *addend;
  float *y;
  uint32_t K, M, N, plane, images;
  uint32_t w_m, w_k;  // weight strides
  uint32_t row_blocks;
  FastDiv plane_div, row_blocks_div;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(const float *p, uint64_t elements) {
  const uint64_t bytes = elements * 4;
  return __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(p), 0,
      static_cast<int>(bytes < kMaxBytes ? static_cast<uint32_t>(bytes) : 0x7FFFFFFFu),
      0x00020000);
}
template <int NT>
__device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t offset, uint32_t scalar,
                                     float (&v)[NT]) {
  const int o = static_cast<int>(offset), s = static_cast<int>(scalar);
  if constexpr (NT == 2) {
    const u32x2 u = __builtin_amdgcn_raw_buffer_load_b64(r, o, s, 0);
    for (int i = 0; i < 2; ++i) v[i] = __uint_as_float(u[i]);
  } else {
    v[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, o, s, 0));
  }
}

// KFast: weights contiguous along k (the forward's rows), else along m.
template <int NT, bool KFast>
__global__ __launch_bounds__(256) void conv_point_kernel(PointArgs g) {
  constexpr int Pairs = NT == 1 ? 16 : 8;     // channel pairs per chunk
  constexpr uint32_t Chunk = 2 * Pairs;
  constexpr uint32_t Row = kRows + 1, Loads = kRows * Chunk / 256;
  constexpr uint32_t Positions = 128 * NT;
  __shared__ float lds[2 * Chunk * Row];
  const uint32_t id = xcd_contiguous(blockIdx.x, gridDim.x);
  const uint32_t block = fast_div(id, g.row_blocks_div);
  const uint32_t m0 = (id - block * g.row_blocks) * kRows;
  const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 32, h = lane / 32;
  const uint32_t first = block * Positions, n0 = fast_div(first, g.plane_div);
  const uint32_t image = g.K * g.plane;
  const __amdgpu_buffer_rsrc_t xr = resource(g.x + static_cast<uint64_t>(n0) * image,
                                             static_cast<uint64_t>(g.images - n0) * image);
  const __amdgpu_buffer_rsrc_t wr = resource(g.w, static_cast<uint64_t>(g.M) * g.K);
  const uint32_t pos = first + wave * (32 * NT) + NT * j;  // NT positions of one plane
  const uint32_t pc = pos < g.N ? pos : g.N - NT;
  const uint32_t n = fast_div(pc, g.plane_div), p = pc - n * g.plane;
  const uint32_t off = ((n - n0) * image + h * g.plane + p) * 4u;

  f32x16 acc[NT];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t m = m0 + 8u * (r / 4) + 4u * h + r % 4;
    const float b = g.bias != nullptr && m < g.M ? g.bias[m] : 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t][r] = b;
  }
  float b[2][Pairs][NT], wv[Loads];
  auto fetch_x = [&](uint32_t k0, float (&v)[Pairs][NT]) {
#pragma unroll
    for (int s = 0; s < Pairs; ++s) {
      const uint32_t ks = k0 + 2 * s;
      load<NT>(xr, ks + h < g.K ? off : kNowhere, ks < g.K ? ks * g.plane * 4u : 0u, v[s]);
    }
  };
  // element e of a weight chunk: row e / Chunk, channel e % Chunk (KFast), or the other way round
  auto fetch_w = [&](uint32_t k0) {
#pragma unroll
    for (uint32_t u = 0; u < Loads; ++u) {
      const uint32_t e = threadIdx.x + u * 256;
      const uint32_t m = m0 + (KFast ? e / Chunk : e % kRows);
      const uint32_t k = k0 + (KFast ? e % Chunk : e / kRows);
      const bool ok = m < g.M && k < g.K;
      wv[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          wr, static_cast<int>(ok ? (m * g.w_m + k * g.w_k) * 4u : kNowhere), 0, 0));
    }
  };
  auto store_w = [&](float *to) {
#pragma unroll
    for (uint32_t u = 0; u < Loads; ++u) {
      const uint32_t e = threadIdx.x + u * 256;
      to[(KFast ? e % Chunk : e / kRows) * Row + (KFast ? e / Chunk : e % kRows)] = wv[u];
    }
  };
  auto multiply = [&](const float *w, const float (&v)[Pairs][NT]) {
    w += h * Row + j;
#pragma unroll
    for (int s = 0; s < Pairs; ++s) {
      const float a = w[2 * s * Row];
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, v[s][t], acc[t], 0, 0, 0);
    }
  };
  fetch_w(0);
  fetch_x(0, b[0]);
  store_w(lds);
  // two chunks a turn, so that the register sets keep their names
  for (uint32_t k0 = 0; k0 < g.K; k0 += 2 * Chunk) {
    __syncthreads();
    if (k0 + Chunk < g.K) {
      fetch_w(k0 + Chunk);
      fetch_x(k0 + Chunk, b[1]);
    }
    __builtin_amdgcn_sched_barrier(0);
    multiply(lds, b[0]);
    if (k0 + Chunk >= g.K) break;
    store_w(lds + Chunk * Row);
    __syncthreads();
    if (k0 + 2 * Chunk < g.K) {
      fetch_w(k0 + 2 * Chunk);
      fetch_x(k0 + 2 * Chunk, b[0]);
    }
    __builtin_amdgcn_sched_barrier(0);
    multiply(lds + Chunk * Row, b[1]);
    if (k0 + 2 * Chunk < g.K) store_w(lds);
  }
  if (pos >= g.N) return;
  const uint64_t at = static_cast<uint64_t>(n) * g.M * g.plane + p;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t m = m0 + 8u * (r / 4) + 4u * h + r % 4;
    if (m >= g.M) continue;
    const uint64_t o = at + static_cast<uint64_t>(m) * g.plane;
    float v[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) v[t] = acc[t][r];
    if constexpr (NT == 2) {
      float2 *y = reinterpret_cast<float2 *>(g.y + o);
      if (g.addend != nullptr) {
        const float2 d = *reinterpret_cast<const float2 *>(g.addend + o);
        v[0] += d.x, v[1] += d.y;
      }
      *y = make_float2(v[0], v[1]);
    } else {
      g.y[o] = g.addend != nullptr ? v[0] + g.addend[o] : v[0];
    }
  }
}

// Grids that leave the chip idle: a block takes 32 rows x 32 positions and each of its four waves
// every fourth group of eight channels, the sums added in wave order.  No operand is shared, so
// both come straight from global memory: per group, lane (i, h) loads four positions' worth --
// its position at channels k + 4 h + s, s < 4 -- and its row's four weights there, for four
// products (channels k + s and k + 4 + s each).  Without barriers kAhead groups stay in flight.
template <bool KFast>
__global__ __launch_bounds__(256) void conv_point_split_kernel(PointArgs g) {
  constexpr int KS = 4, kAhead = 6;
  __shared__ float sums[KS - 1][16][64];
  const uint32_t id = xcd_contiguous(blockIdx.x, gridDim.x);
  const uint32_t block = fast_div(id, g.row_blocks_div);
  const uint32_t m0 = (id - block * g.row_blocks) * kRows;
  const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 32, h = lane / 32;
  const uint32_t first = block * 32, n0 = fast_div(first, g.plane_div);
  const uint32_t image = g.K * g.plane;
  const __amdgpu_buffer_rsrc_t xr = resource(g.x + static_cast<uint64_t>(n0) * image,
                                             static_cast<uint64_t>(g.images - n0) * image);
  const __amdgpu_buffer_rsrc_t wr = resource(g.w, static_cast<uint64_t>(g.M) * g.K);
  const uint32_t pos = first + j, pc = pos < g.N ? pos : g.N - 1;
  const uint32_t n = fast_div(pc, g.plane_div), p = pc - n * g.plane;
  const uint32_t xo = ((n - n0) * image + 4 * h * g.plane + p) * 4u;
  const uint32_t m = m0 + j < g.M ? m0 + j : g.M - 1;  // rows past M are not stored
  const uint32_t wo = (m * g.w_m + 4 * h * g.w_k) * 4u;
  const uint32_t groups = (g.K + 7) / 8, mine = groups > wave ? (groups - wave - 1) / KS + 1 : 0;

  float a[kAhead][4], b[kAhead][4];
  auto fetch = [&](uint32_t i, float (&av)[4], float (&bv)[4]) {
    const uint32_t k = 8 * (wave + i * KS);
    if (KFast && k + 8 <= g.K) {
      const u32x4 u = __builtin_amdgcn_raw_buffer_load_b128(wr, static_cast<int>(wo),
                                                            static_cast<int>(k * 4), 0);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        av[s] = __uint_as_float(u[s]);
        load<1>(xr, xo, (k + s) * g.plane * 4u, reinterpret_cast<float(&)[1]>(bv[s]));
      }
      return;
    }
#pragma unroll
    for (uint32_t s = 0; s < 4; ++s) {  // +0 past the channels
      const uint32_t past = k + 4 * h + s < g.K ? 0u : kNowhere, ks = k + s < g.K ? k + s : 0;
      load<1>(wr, wo | past, ks * g.w_k * 4u, reinterpret_cast<float(&)[1]>(av[s]));
      load<1>(xr, xo | past, ks * g.plane * 4u, reinterpret_cast<float(&)[1]>(bv[s]));
    }
  };
#pragma unroll
  for (int s = 0; s < kAhead; ++s)
    if (static_cast<uint32_t>(s) < mine) fetch(s, a[s], b[s]);
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t row = m0 + 8u * (r / 4) + 4u * h + r % 4;
    acc[r] = wave == 0 && g.bias != nullptr && row < g.M ? g.bias[row] : 0.0f;
  }
  for (uint32_t i0 = 0; i0 < mine; i0 += kAhead) {
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      if (i0 + s >= mine) break;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s][q], b[s][q], acc, 0, 0, 0);
      if (i0 + s + kAhead < mine) fetch(i0 + s + kAhead, a[s], b[s]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sums[wave - 1][r][lane] = acc[r];
  }
  __syncthreads();
  if (wave > 0 || pos >= g.N) return;
  for (int q = 0; q < KS - 1; ++q)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] += sums[q][r][lane];
  const uint64_t at = static_cast<uint64_t>(n) * g.M * g.plane + p;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t row = m0 + 8u * (r / 4) + 4u * h + r % 4;
    if (row >= g.M) continue;
    const uint64_t o = at + static_cast<uint64_t>(row) * g.plane;
    g.y[o] = g.addend != nullptr ? acc[r] + g.addend[o] : acc[r];
  }
}

template <int NT>
void launch_tiles(hipStream_t s, const PointArgs &g, bool k_fast) {
  constexpr uint32_t positions = 128 * NT;
  const dim3 grid(g.row_blocks * ((g.N + positions - 1) / positions)), threads(256);
  if (k_fast)
    launch(conv_point_kernel<NT, true>, grid, threads, 0, s, g);
  else
    launch(conv_point_kernel<NT, false>, grid, threads, 0, s, g);
}

void launch_split(hipStream_t s, const PointArgs &g, bool k_fast) {
  const dim3 grid(g.row_blocks * ((g.N + 31) / 32)), threads(256);
  if (k_fast)
    launch(conv_point_split_kernel<true>, grid, threads, 0, s, g);
  else
    launch(conv_point_split_kernel<false>, grid, threads, 0, s, g);
}

// Pairs of positions where planes and pointers allow and leave two blocks per CU (192 channels to
// 64, 64 images of 56 x 56: 66 us, 70 with four positions, 73 with one), else single ones.  The
// split kernel where a wave's walk over the channels, about 37 ns each, would outlast the split
// kernel's pass over all products (6.5 us per 2^27, operands unshared): 64 images of 7 x 7, 512
// channels to 128: 15 against 24 us; 128 to 512: 15 against 12 us.
void launch_point(hipStream_t s, PointArgs g, bool k_fast) {
  g.row_blocks = (g.M + kRows - 1) / kRows;
  g.row_blocks_div = make_fastdiv(g.row_blocks);
  g.plane_div = make_fastdiv(g.plane);
  uintptr_t bits = reinterpret_cast<uintptr_t>(g.x) | reinterpret_cast<uintptr_t>(g.y) |
                   reinterpret_cast<uintptr_t>(g.addend);
  bits |= static_cast<uintptr_t>(g.plane) * 4;
  const auto blocks = [&](uint64_t positions) {
    return (g.N + positions - 1) / positions * g.row_blocks;
  };
  const double products = static_cast<double>(g.N) * g.M * g.K;
  if (bits % 8 == 0 && blocks(256) >= 2 * kComputeUnits)
    launch_tiles<2>(s, g, k_fast);
  else if (0.037 * g.K > 6.5 * products / (1 << 27))
    launch_split(s, g, k_fast);
  else
    launch_tiles<1>(s, g, k_fast);
}

}  // namespace

bool takes_pointwise(uint64_t images, uint64_t plane, uint64_t k, uint64_t m) {
  const uint64_t positions = images * plane;
  return ((256 - 1) / plane + 2) * k * plane * 4 < kMaxBytes && m * k * 4 < kMaxBytes &&
         positions < (1ull << 31) - 512 &&
         (positions + 31) / 32 * ((m + kRows - 1) / kRows) < (1ull << 23);
}

void pointwise(hipStream_t s, uint32_t images, uint32_t plane, uint32_t k, uint32_t m,
               bool transposed, const float *x, const float *weight, const float *bias,
               const float *addend, float *y) {
  PointArgs g{};
  g.x = x, g.w = weight, g.bias = bias, g.addend = addend, g.y = y;
  g.K = k, g.M = m, g.N = images * plane, g.plane = plane, g.images = images;
  g.w_m = transposed ? 1 : k, g.w_k = transposed ? m : 1;
  launch_point(s, g, !transposed);
}

}  // namespace conv_mfma
}  // namespace oxh
