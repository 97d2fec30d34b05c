// conv_depthwise.hip -- depthwise 3 x 3 and 5 x 5 convolutions over planes beyond the fused
// depthwise + BatchNorm kernels (conv_mfma.h declares them; CPU semantics: evaluation.rs:334-445,
// autograd.rs:412-527).
//
// These layers move about as many bytes as they add products, so they are bound by memory once
// loads stop repeating: a thread per output reads its K * K inputs one by one.  Here a thread takes
// a tile of outputs and reads each row of inputs under it once, four values per load at any
// alignment.  64 images of 192 x 28 x 28, 5 x 5: forward 124 -> 21 us, input gradient 140 -> 21 us
// (both tensors once, at the 6.24 TB/s of a large copy: 12.4 us); 32 of 32 x 112 x 112, 3 x 3:
// 44 -> 19 and 76 -> 19 us (16.5 us).
// Sums keep the CPU path's order (bias, then taps by row and column; the input gradient by output
// row and column), one multiplication and one addition per tap: bit-identical.  An input outside
// the plane is a +0 operand in place of a skipped tap: the same sum while the weights are finite
// and the sum does not start at -0.  A tile at the plane's edge is taken again where they are not
// or where it does, with -0, which no sum notices, in place of the products outside.
//
// The weight gradient gives a channel one block; each thread reads four outputs' gradients and
// the rows of inputs under them and keeps one sum per tap, by fused multiply-adds.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "conv_mfma.h"

namespace oxh {
namespace conv_mfma {
namespace {

constexpr uint64_t kMaxElements = 1ull << 31;

struct DepthArgs {
  const float *x, *w, *bias, *addend;
  float *y;
  uint32_t C, H, W, OH, OW, items, tiles_y, tiles_x;
  int pad, last;  // last: the last offset of four values in x
  FastDiv tiles_x_div, tiles_y_div, c_div;
};

typedef float float4_any __attribute__((ext_vector_type(4), aligned(4)));

// Q * 4 neighbouring values from offset `at` of x, those whose mask is off +0.  Values outside the
// row are its neighbours' (masked); only a load past an end of the tensor moves into it.
template <int Q>
__device__ __forceinline__ void load_row(const float *x, int last, int at, bool row,
                                         const bool (&mask)[4 * Q], float (&v)[4 * Q]) {
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int want = at + 4 * q, from = want < 0 ? 0 : want > last ? last : want;
    const float4_any u = *reinterpret_cast<const float4_any *>(x + from);
    float got[4] = {u.x, u.y, u.z, u.w};
    if (want != from) {
      const int move = want - from;  // wanted value i is value i + move of the load
      const float all[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        got[i] = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) got[i] = k == i + move ? all[k] : got[i];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[4 * q + i] = row && mask[4 * q + i] ? got[i] : 0.0f;
  }
}

template <int N>
__device__ __forceinline__ void column_masks(int ix, uint32_t W, bool (&mask)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) mask[i] = static_cast<uint32_t>(ix + i) < W;
}

template <int N>
__device__ __forceinline__ bool not_finite(const float (&v)[N]) {
  float z = 0.0f;
#pragma unroll
  for (int i = 0; i < N; ++i) z = __builtin_fmaf(v[i], 0.0f, z);
  return !(z == 0.0f);
}

__device__ __forceinline__ void store4(float *y, const float *addend, uint64_t at, uint32_t count,
                                       const float (&v)[4]) {
  if (count >= 4) {
    float4_any o = {v[0], v[1], v[2], v[3]};
    if (addend != nullptr) o += *reinterpret_cast<const float4_any *>(addend + at);
    *reinterpret_cast<float4_any *>(y + at) = o;
  } else {
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
      if (j < count) y[at + j] = addend != nullptr ? v[j] + addend[at + j] : v[j];
  }
}

// Forward, and (Flip) the input gradient of a stride-1 convolution: source = the output's
// gradient, pad = K - 1 - the convolution's, weights turned round.  A thread: TY x 4 outputs.
template <int K, int S, bool Flip>
__global__ __launch_bounds__(256, 4) void depthwise_kernel(DepthArgs a) {
  constexpr int T = K * K, TX = 4, TY = S == 1 ? 4 : 2;
  constexpr int RY = (TY - 1) * S + K, Q = ((TX - 1) * S + K + 3) / 4;
  const uint32_t item = blockIdx.x * 256 + threadIdx.x;
  if (item >= a.items) return;
  const uint32_t t0 = fast_div(item, a.tiles_x_div), tx = item - t0 * a.tiles_x;
  const uint32_t plane = fast_div(t0, a.tiles_y_div), ty = t0 - plane * a.tiles_y;
  const uint32_t c = plane - fast_div(plane, a.c_div) * a.C;
  const uint32_t oy0 = ty * TY, ox0 = tx * TX;
  const int iy0 = static_cast<int>(oy0 * S) - a.pad, ix0 = static_cast<int>(ox0 * S) - a.pad;
  const uint32_t first = plane * a.H * a.W;
  float w[T];
#pragma unroll
  for (int t = 0; t < T; ++t) w[t] = a.w[c * T + t];
  const float b = a.bias != nullptr ? a.bias[c] : 0.0f;
  float acc[TY][TX];
  auto sum = [&](auto skip, int y0, int x0) {  // Skip: products outside the plane are -0
    bool mask[4 * Q];
    column_masks(x0, a.W, mask);
#pragma unroll
    for (int i = 0; i < TY; ++i)
#pragma unroll
      for (int j = 0; j < TX; ++j) acc[i][j] = b;
#pragma unroll
    for (int r = 0; r < RY; ++r) {
      const int iy = y0 + r;
      const bool in = static_cast<uint32_t>(iy) < a.H;
      float row[4 * Q];
      load_row<Q>(a.x, a.last, static_cast<int>(first + (in ? iy : 0) * a.W) + x0, in, mask, row);
#pragma unroll
      for (int i = 0; i < TY; ++i) {
        const int ky = r - i * S;
        if (ky < 0 || ky >= K) continue;
#pragma unroll
        for (int kx = 0; kx < K; ++kx)
#pragma unroll
          for (int j = 0; j < TX; ++j) {
            const float p = row[j * S + kx] * w[Flip ? T - 1 - (ky * K + kx) : ky * K + kx];
            acc[i][j] += !decltype(skip)::value || (in && mask[j * S + kx]) ? p : -0.0f;
          }
      }
    }
  };
  sum(std::false_type{}, iy0, ix0);
  const bool inside = iy0 >= 0 && ix0 >= 0 && iy0 + RY <= static_cast<int>(a.H) &&
                      ix0 + (TX - 1) * S + K <= static_cast<int>(a.W);
  if (!inside && (not_finite(w) || __float_as_uint(b) == 0x80000000u)) {
    int y0 = iy0, x0 = ix0;
    asm volatile("" : "+v"(y0), "+v"(x0));  // loaded again, not held in registers
    sum(std::true_type{}, y0, x0);
  }
  const uint64_t out = static_cast<uint64_t>(plane) * a.OH * a.OW;
#pragma unroll
  for (int i = 0; i < TY; ++i) {
    if (oy0 + i >= a.OH) break;
    store4(a.y, a.addend, out + (oy0 + i) * a.OW + ox0, a.OW - ox0, acc[i]);
  }
}

// Input gradient of a stride-2 convolution: with y + pad = 2 a + py, inputs (a, py) meet outputs
// oy = a - i through ky = py + 2 i.  A thread: a in {a0, a0 + 1}, b in {b0, b0 + 1}, so 4 x 4
// inputs under (M2 + 1) x (M2 + 1) outputs, M2 = ceil(K / 2).  x: the gradient (H x W), y: the
// input's (OH x OW).
template <int K>
__global__ __launch_bounds__(256, 4) void depthwise_input_s2_kernel(DepthArgs a, uint32_t start) {
  constexpr int T = K * K, M2 = (K + 1) / 2, R = M2 + 1;
  const uint32_t item = blockIdx.x * 256 + threadIdx.x;
  if (item >= a.items) return;
  const uint32_t t0 = fast_div(item, a.tiles_x_div), tx = item - t0 * a.tiles_x;
  const uint32_t plane = fast_div(t0, a.tiles_y_div), ty = t0 - plane * a.tiles_y;
  const uint32_t c = plane - fast_div(plane, a.c_div) * a.C;
  const int a0 = static_cast<int>(start + 2 * ty), b0 = static_cast<int>(start + 2 * tx);
  const uint32_t first = plane * a.H * a.W;
  float w[T], acc[4][4];
#pragma unroll
  for (int t = 0; t < T; ++t) w[t] = a.w[c * T + t];
  auto sum = [&](auto skip, int oy0, int ox0) {  // as in depthwise_kernel
    float rows[R][4];  // rows[r][q]: output (oy0 + r, ox0 + q)
    bool mask[4], in[R];
    column_masks(ox0, a.W, mask);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      in[r] = static_cast<uint32_t>(oy0 + r) < a.H;
      load_row<1>(a.x, a.last, static_cast<int>(first + (in[r] ? oy0 + r : 0) * a.W) + ox0, in[r],
                  mask, rows[r]);
    }
#pragma unroll
    for (int ry = 0; ry < 4; ++ry)
#pragma unroll
      for (int rx = 0; rx < 4; ++rx) {
        float v = 0.0f;
#pragma unroll
        for (int i = M2 - 1; i >= 0; --i) {  // oy ascending
          const int ky = ry % 2 + 2 * i;
          if (ky >= K) continue;
#pragma unroll
          for (int j = M2 - 1; j >= 0; --j) {
            const int kx = rx % 2 + 2 * j, r = ry / 2 - i + M2 - 1, q = rx / 2 - j + M2 - 1;
            if (kx >= K) continue;
            const float p = rows[r][q] * w[ky * K + kx];
            v += !decltype(skip)::value || (in[r] && mask[q]) ? p : -0.0f;
          }
        }
        acc[ry][rx] = v;
      }
  };
  int oy0 = a0 - (M2 - 1), ox0 = b0 - (M2 - 1);
  sum(std::false_type{}, oy0, ox0);
  const bool inside = oy0 >= 0 && ox0 >= 0 && a0 + 1 < static_cast<int>(a.H) &&
                      b0 + 1 < static_cast<int>(a.W);
  if (!inside && not_finite(w)) {
    asm volatile("" : "+v"(oy0), "+v"(ox0));
    sum(std::true_type{}, oy0, ox0);
  }
  const int x0 = 2 * b0 - a.pad;  // -1 where the padding is odd
  const uint64_t out = static_cast<uint64_t>(plane) * a.OH * a.OW;
#pragma unroll
  for (int ry = 0; ry < 4; ++ry) {
    const int y = 2 * a0 + ry - a.pad;
    if (static_cast<uint32_t>(y) >= a.OH) continue;
    const uint64_t at = out + static_cast<uint32_t>(y) * a.OW;
    if (x0 >= 0) {
      if (static_cast<uint32_t>(x0) < a.OW) store4(a.y, a.addend, at + x0, a.OW - x0, acc[ry]);
    } else {
#pragma unroll
      for (int rx = 0; rx < 4; ++rx)
        if (static_cast<uint32_t>(x0 + rx) < a.OW) {
          const uint64_t o = at + (x0 + rx);
          a.y[o] = a.addend != nullptr ? acc[ry][rx] + a.addend[o] : acc[ry][rx];
        }
    }
  }
}

// Weight gradient: block per channel and chunk of images; a thread item is a TY x 4 tile of
// outputs, whose products go to one sum per tap by fused multiply-adds; wave sums in a fixed order,
// waves in order.  Operands outside are +0; a thread that ends with a sum that is not finite walks
// its items again, skipping them.  Bound by the loads a CU issues: the tile shares each row of
// inputs among its outputs' rows.  64 images of 192 x 28 x 28, 5 x 5: 157 -> 29 us; 32 of 64 x 28 x
// 28, 5 x 5: 51 -> 14.5 us; 32 of 32 x 112 x 112, 3 x 3: 305 -> 29 us.  5 x 5 kernels are bound to
// three waves per SIMD (bound to four, their rows spilled: 14 against 18 us for 192 x 28 x 28 at
// stride 2).
struct DepthWeightArgs {
  const float *g, *x;
  float *dw;
  uint32_t C, H, W, OH, OW, items, per_chunk, tiles_x, tiles_y;  // per_chunk, items: per channel
  int pad, g_last, x_last;
  FastDiv tiles_x_div, tiles_y_div;
};
template <int K, int S, int Threads>
__global__ __launch_bounds__(Threads, K == 5 ? 3 : 4) void depthwise_weight_kernel(
    DepthWeightArgs a) {
  constexpr int T = K * K, Q = (3 * S + K + 3) / 4, TY = S == 1 ? 4 : 2, RY = (TY - 1) * S + K;
  __shared__ float sums[Threads / 64][T];
  const uint32_t c = blockIdx.x, begin = blockIdx.y * a.per_chunk;
  const uint32_t end = begin + a.per_chunk < a.items ? begin + a.per_chunk : a.items;
  float acc[T];
  auto walk = [&](auto skip) {  // Skip: products outside either plane are left out
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = 0.0f;
    for (uint32_t item = begin + threadIdx.x; item < end; item += Threads) {
      const uint32_t t0 = fast_div(item, a.tiles_x_div), ox0 = 4 * (item - t0 * a.tiles_x);
      const uint32_t n = fast_div(t0, a.tiles_y_div), oy0 = TY * (t0 - n * a.tiles_y);
      const uint32_t plane = n * a.C + c;
      const int iy0 = static_cast<int>(oy0 * S) - a.pad, ix0 = static_cast<int>(ox0 * S) - a.pad;
      float gv[TY][4];
      bool gmask[4], mask[4 * Q];
      column_masks(static_cast<int>(ox0), a.OW, gmask);
      column_masks(ix0, a.W, mask);
#pragma unroll
      for (int i = 0; i < TY; ++i) {
        const bool in = oy0 + i < a.OH;
        load_row<1>(a.g, a.g_last,
                    static_cast<int>((plane * a.OH + (in ? oy0 + i : 0)) * a.OW + ox0), in, gmask,
                    gv[i]);
      }
#pragma unroll
      for (int r = 0; r < RY; ++r) {
        const int iy = iy0 + r;
        const bool in = static_cast<uint32_t>(iy) < a.H;
        float row[4 * Q];
        load_row<Q>(a.x, a.x_last, static_cast<int>((plane * a.H + (in ? iy : 0)) * a.W) + ix0, in,
                    mask, row);
#pragma unroll
        for (int i = 0; i < TY; ++i) {
          const int ky = r - i * S;
          if (ky < 0 || ky >= K) continue;
#pragma unroll
          for (int kx = 0; kx < K; ++kx)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int t = ky * K + kx;
              const float v = __builtin_fmaf(gv[i][j], row[j * S + kx], acc[t]);
              const bool at = oy0 + i < a.OH && gmask[j] && in && mask[j * S + kx];
              acc[t] = !decltype(skip)::value || at ? v : acc[t];
            }
        }
      }
    }
  };
  walk(std::false_type{});
  if (not_finite(acc)) walk(std::true_type{});
  wave_sums_rows(acc);
  if (threadIdx.x % 64 == 0) {
#pragma unroll
    for (int t = 0; t < T; ++t) sums[threadIdx.x / 64][t] = acc[t];
  }
  __syncthreads();
  if (threadIdx.x < T) {
    float v = sums[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < Threads / 64; ++w) v += sums[w][threadIdx.x];
    a.dw[(blockIdx.y * a.C + c) * T + threadIdx.x] = v;
  }
}

template <int K, int S, bool Flip>
void launch_depthwise(hipStream_t s, DepthArgs a, uint32_t planes) {
  constexpr uint32_t TY = S == 1 ? 4 : 2;
  a.tiles_x = (a.OW + 3) / 4, a.tiles_y = (a.OH + TY - 1) / TY;
  a.items = planes * a.tiles_x * a.tiles_y;
  a.tiles_x_div = make_fastdiv(a.tiles_x), a.tiles_y_div = make_fastdiv(a.tiles_y);
  launch(depthwise_kernel<K, S, Flip>, dim3((a.items + 255) / 256), dim3(256), 0, s, a);
}

struct WeightSplit {
  uint32_t tiles_x, tiles_y, items, per_chunk, chunks;
};
// A channel's tiles (TY x 4 outputs each) go to several blocks where there are enough for two of
// kWeightItems, up to the blocks that fill the chip (three waves per SIMD); fewer tiles cost less
// than the launch that adds the chunks.
constexpr uint32_t kWeightItems = 1024;
WeightSplit weight_split(const Dims &d) {
  WeightSplit w{};
  const uint32_t ty = d.stride == 1 ? 4 : 2;
  w.tiles_x = (d.ow + 3) / 4, w.tiles_y = (d.oh + ty - 1) / ty;
  w.items = d.batch * w.tiles_x * w.tiles_y;
  const uint32_t fill = (768 + d.in_c - 1) / d.in_c, most = w.items / kWeightItems;
  const uint32_t chunks = most < 2 ? 1 : most < fill ? most : fill;
  const uint32_t rounds = (w.items + 255) / 256;
  w.per_chunk = 256 * ((rounds + chunks - 1) / chunks);
  w.chunks = (w.items + w.per_chunk - 1) / w.per_chunk;
  return w;
}

template <int Threads>
void launch_weight(hipStream_t s, const Dims &d, const DepthWeightArgs &a, uint32_t chunks) {
  const dim3 grid(d.in_c, chunks), block(Threads);
  if constexpr (Threads > 64) {  // 3 x 3 layers of so few tiles take another kernel (conv.hip)
    if (d.k == 3 && d.stride == 1)
      launch(depthwise_weight_kernel<3, 1, Threads>, grid, block, 0, s, a);
    else if (d.k == 3)
      launch(depthwise_weight_kernel<3, 2, Threads>, grid, block, 0, s, a);
    if (d.k == 3) return;
  }
  if (d.stride == 1) launch(depthwise_weight_kernel<5, 1, Threads>, grid, block, 0, s, a);
  else launch(depthwise_weight_kernel<5, 2, Threads>, grid, block, 0, s, a);
}

}  // namespace

bool takes_depthwise(const Dims &d) {
  return d.in_c == d.out_c && (d.k == 3 || d.k == 5) && (d.stride == 1 || d.stride == 2) &&
         d.w >= 4 && d.ow >= 4 && d.pad < 4 * d.k &&
         static_cast<uint64_t>(d.batch) * d.in_c * (d.h + 2 * d.pad + 4) *
                 (d.w + 2 * d.pad + 4) <
             kMaxElements;
}

void depthwise_forward(hipStream_t s, const Dims &d, const float *x, const float *weight,
                       const float *bias, float *y) {
  DepthArgs a{};
  a.x = x, a.w = weight, a.bias = bias, a.y = y;
  a.C = d.in_c, a.H = d.h, a.W = d.w, a.OH = d.oh, a.OW = d.ow, a.pad = static_cast<int>(d.pad);
  a.c_div = make_fastdiv(d.in_c);
  const uint32_t planes = d.batch * d.in_c;
  a.last = static_cast<int>(planes * d.h * d.w) - 4;
  if (d.k == 3 && d.stride == 1) launch_depthwise<3, 1, false>(s, a, planes);
  else if (d.k == 3) launch_depthwise<3, 2, false>(s, a, planes);
  else if (d.stride == 1) launch_depthwise<5, 1, false>(s, a, planes);
  else launch_depthwise<5, 2, false>(s, a, planes);
}

void depthwise_input_backward(hipStream_t s, const Dims &d, const float *gradient,
                              const float *weight, const float *addend, float *dx) {
  DepthArgs a{};
  a.x = gradient, a.w = weight, a.addend = addend, a.y = dx;
  a.C = d.in_c, a.H = d.oh, a.W = d.ow, a.OH = d.h, a.OW = d.w;
  a.c_div = make_fastdiv(d.in_c);
  const uint32_t planes = d.batch * d.in_c;
  a.last = static_cast<int>(planes * d.oh * d.ow) - 4;
  if (d.stride == 1) {
    a.pad = static_cast<int>(d.k) - 1 - static_cast<int>(d.pad);
    if (d.k == 3) launch_depthwise<3, 1, true>(s, a, planes);
    else launch_depthwise<5, 1, true>(s, a, planes);
    return;
  }
  a.pad = static_cast<int>(d.pad);
  const uint32_t start = d.pad / 2;
  a.tiles_y = ((d.h - 1 + d.pad) / 2 - start) / 2 + 1;
  a.tiles_x = ((d.w - 1 + d.pad) / 2 - start) / 2 + 1;
  a.items = planes * a.tiles_y * a.tiles_x;
  a.tiles_x_div = make_fastdiv(a.tiles_x), a.tiles_y_div = make_fastdiv(a.tiles_y);
  const dim3 grid((a.items + 255) / 256), block(256);
  if (d.k == 3) launch(depthwise_input_s2_kernel<3>, grid, block, 0, s, a, start);
  else launch(depthwise_input_s2_kernel<5>, grid, block, 0, s, a, start);
}

uint32_t depthwise_weight_partials(const Dims &d) { return weight_split(d).chunks; }

void depthwise_weight_backward(hipStream_t s, const Dims &d, const float *gradient,
                               const float *x, float *dw) {
  DepthWeightArgs a{};
  a.g = gradient, a.x = x, a.dw = dw;
  a.C = d.in_c, a.H = d.h, a.W = d.w, a.OH = d.oh, a.OW = d.ow, a.pad = static_cast<int>(d.pad);
  a.g_last = static_cast<int>(d.batch * d.in_c * d.oh * d.ow) - 4;
  a.x_last = static_cast<int>(d.batch * d.in_c * d.h * d.w) - 4;
  const WeightSplit w = weight_split(d);
  a.tiles_x = w.tiles_x, a.tiles_y = w.tiles_y, a.items = w.items, a.per_chunk = w.per_chunk;
  a.tiles_x_div = make_fastdiv(w.tiles_x), a.tiles_y_div = make_fastdiv(w.tiles_y);
  // a wave or four where that is about a tile per thread; eight where channels leave CUs idle
  if (w.items <= 128 && d.k == 5) launch_weight<64>(s, d, a, w.chunks);
  else if (w.items <= 512 || d.in_c * w.chunks > 256) launch_weight<256>(s, d, a, w.chunks);
  else launch_weight<512>(s, d, a, w.chunks);
}

}  // namespace conv_mfma
}  // namespace oxh
