// a14 loop filters (Gaborish 3x3, EPF passes 1 and 2) and a15 XYB -> linear
// RGB on the unpadded reconstruction, as EvaluateQuantization applies them
// (src/codec/adaptive_quantization.cpp:972-1000): the padded reconstruction
// is cropped to the source extent and every filter mirrors at that extent.
#include <cmath>

#include "common.h"
#include "tile_mirror.h"

namespace gjxl_amd {
namespace {

__device__ __forceinline__ int MirrorInt(int c, int size) {
  if (c >= 0 && c < size) return c;
  const long long period = 2LL * size;
  long long phase;
  if (c >= 0) {
    phase = c % period;
  } else {
    const long long mag = -(static_cast<long long>(c) + 1) + 1;
    const long long rem = mag % period;
    phase = rem == 0 ? 0 : period - rem;
  }
  return static_cast<int>(phase < size ? phase : period - 1 - phase);
}

struct GaborishWeights {
  float center, axis, diagonal;
};

// ApplyGaborish (src/codec/gaborish.cpp:101-190) and ApplyEpfPass
// (src/codec/epf.cpp:61-205, pass 1 plus-patch SAD, pass 2 pixel SAD, four
// cardinal neighbours, default options) are evaluated in LoopFilterKernel.
struct InverseOpsin {
  float m[3][3];
  float scale;       // 255 / intensity
  float bias_cbrt;   // host cbrtf(bias)
};

// OpsinToLinearRgb (src/codec/color_transform.cpp:433-471) of one pixel.
__device__ __forceinline__ void OpsinToLinearPixel(float x, float y, float b,
                                                   const InverseOpsin& p, float out[3]) {
  constexpr float kOpsinBias = 0.0037930732552754493f;
  const float gamma[3] = {y + x + p.bias_cbrt, y - x + p.bias_cbrt, b + p.bias_cbrt};
  float mixed[3];
  for (int c = 0; c < 3; ++c) mixed[c] = gamma[c] * gamma[c] * gamma[c] - kOpsinBias;
  for (int row = 0; row < 3; ++row) {
    float v = p.scale * p.m[row][0] * mixed[0];
    v = __builtin_fmaf(p.scale * p.m[row][1], mixed[1], v);
    v = __builtin_fmaf(p.scale * p.m[row][2], mixed[2], v);
    out[row] = v;
  }
}


// The three loop filters and XYB -> linear fused: one work group per 64x16
// output tile.  LDS holds the mirrored input with a 4-pixel halo, Gaborish on
// the tile plus 3, EPF pass 1 on the tile plus 1, and pass 2 on the tile.
// Each filter's samples outside the image are its own values at the
// mirrored coordinate (every filter mirrors its input at the image extent),
// copied from the slot of that coordinate, which lies within the same region.
constexpr int kLfTileW = 64, kLfTileH = 16;
constexpr int kRawW = kLfTileW + 8, kRawH = kLfTileH + 8;  // halo 4
constexpr int kGabW = kLfTileW + 6, kGabH = kLfTileH + 6;  // halo 3
constexpr int kE1W = kLfTileW + 2, kE1H = kLfTileH + 2;    // halo 1
static_assert(kE1W * kE1H <= kRawW * kRawH, "pass 1 reuses the input tile's space");

template <int kPass, typename Sample>
__device__ __forceinline__ void EpfPixel(Sample S, float bis, int x, int y,
                                         float out[3]) {
  constexpr float kMinInverseSigma = -1.1715728752538099024f / 0.3f;
  constexpr float kSigmaScale = 1.65f * (kPass == 2 ? 6.5f : 1.0f);
  constexpr int kCard[4][2] = {{0, -1}, {-1, 0}, {1, 0}, {0, 1}};
  constexpr int kPlus[5][2] = {{0, 0}, {0, -1}, {-1, 0}, {0, 1}, {1, 0}};
  constexpr float kScale[3] = {40.0f, 5.0f, 3.5f};
  if (bis < kMinInverseSigma) {
    for (int c = 0; c < 3; ++c) out[c] = S(c, 0, 0);
    return;
  }
  const bool border = x % 8 == 0 || x % 8 == 7 || y % 8 == 0 || y % 8 == 7;
  const float sis = bis * kSigmaScale * (border ? 2.0f / 3.0f : 1.0f);
  float sum[3] = {S(0, 0, 0), S(1, 0, 0), S(2, 0, 0)};
  float weight_sum = 1.0f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int dx = kCard[k][0], dy = kCard[k][1];
    float sad = 0.0f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if constexpr (kPass == 1) {
        float cs = 0.0f;
#pragma unroll
        for (int o = 0; o < 5; ++o) {
          cs += fabsf(S(c, kPlus[o][0], kPlus[o][1]) -
                      S(c, dx + kPlus[o][0], dy + kPlus[o][1]));
        }
        sad = __builtin_fmaf(cs, kScale[c], sad);
      } else {
        sad = __builtin_fmaf(fabsf(S(c, 0, 0) - S(c, dx, dy)), kScale[c], sad);
      }
    }
    float weight = __builtin_fmaf(sad, sis, 1.0f);
    weight = 0.0f < weight ? weight : 0.0f;
    weight_sum += weight;
#pragma unroll
    for (int c = 0; c < 3; ++c) sum[c] = __builtin_fmaf(weight, S(c, dx, dy), sum[c]);
  }
  for (int c = 0; c < 3; ++c) out[c] = sum[c] / weight_sum;
}

// kOnce: w and h are at least 4, so every coordinate that an output needs (at
// most 4 outside the image) needs one reflection; what a lane reads further
// outside, in an image narrower than 34 or lower than 10, lies inside it
// (TileMirror) and is never used.
template <bool kOnce>
__global__ __launch_bounds__(256) void LoopFilterKernel(
  const float* __restrict__ in, int in_stride, size_t in_plane, int w, int h,
  GaborishWeights g, const float* __restrict__ inverse_sigma, InverseOpsin p,
  float* __restrict__ filtered, float* __restrict__ linear) {
  // the input tile is dead once Gaborish is done: pass 1 reuses its space
  __shared__ float raw_e1[3 * kRawH * kRawW];
  __shared__ float gab[3][kGabH][kGabW];
  auto raw = reinterpret_cast<float (*)[kRawH][kRawW]>(raw_e1);
  auto e1 = reinterpret_cast<float (*)[kE1H][kE1W]>(raw_e1);
  const TileIndex tile_index = XcdTile();
  const int x0 = tile_index.x * kLfTileW, y0 = tile_index.y * kLfTileH;
  const int bw = (w + 7) / 8;
  const size_t plane = static_cast<size_t>(w) * h;
  auto mirror = [](int c, int size) { return kOnce ? TileMirror(c, size) : MirrorInt(c, size); };
  // The tile's 3 x kRawH rows of kRawW = 64 + 8 columns: each wave reads
  // kWaveRows whole rows, one lane per column of the first 64, with the row
  // address uniform (scalar arithmetic); the last 8 columns of every row are
  // three reads per thread.  Every read issues before the first store.
  static_assert(kRawW == 64 + 8 && (3 * kRawH) % 4 == 0, "tile rows split over four waves");
  constexpr int kWaveRows = 3 * kRawH / 4;
  constexpr int kStripCount = 3 * kRawH * 8;
  constexpr int kStripLoads = (kStripCount + 255) / 256;
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64));
  const int sx = mirror(x0 - 4 + lane, w);
  float rows[kWaveRows];
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) {
    const int row = wave * kWaveRows + i;
    const int c = row / kRawH, r = row % kRawH;
    const float* src = in + c * in_plane + static_cast<size_t>(mirror(y0 - 4 + r, h)) * in_stride;
    rows[i] = src[sx];
  }
  float strip[kStripLoads];
#pragma unroll
  for (int k = 0; k < kStripLoads; ++k) {
    const int e = min(static_cast<int>(threadIdx.x) + k * 256, kStripCount - 1);
    const int row = e / 8, c = row / kRawH, r = row % kRawH;
    const int sy = mirror(y0 - 4 + r, h), sxs = mirror(x0 - 4 + 64 + e % 8, w);
    strip[k] = in[c * in_plane + static_cast<size_t>(sy) * in_stride + sxs];
  }
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) {
    raw_e1[(wave * kWaveRows + i) * kRawW + lane] = rows[i];
  }
#pragma unroll
  for (int k = 0; k < kStripLoads; ++k) {
    const int e = threadIdx.x + k * 256;
    if (e < kStripCount) raw_e1[(e / 8) * kRawW + 64 + e % 8] = strip[k];
  }
  __syncthreads();
  // Gaborish (gaborish.cpp:101-190) at the in-image slots of its region
  for (int e = threadIdx.x; e < kGabH * kGabW; e += blockDim.x) {
    const int r = e / kGabW, col = e % kGabW;
    const int gx = x0 - 3 + col, gy = y0 - 3 + r;
    if (gx < 0 || gy < 0 || gx >= w || gy >= h) continue;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      auto S = [&](int dx, int dy) { return raw[c][r + 1 + dy][col + 1 + dx]; };
      const float axes = (S(-1, 0) + S(1, 0)) + (S(0, -1) + S(0, 1));
      const float diagonals = (S(-1, -1) + S(1, -1)) + (S(-1, 1) + S(1, 1));
      gab[c][r][col] = g.center * S(0, 0) + g.axis * axes + g.diagonal * diagonals;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kGabH * kGabW; e += blockDim.x) {
    const int r = e / kGabW, col = e % kGabW;
    const int gx = x0 - 3 + col, gy = y0 - 3 + r;
    if (gx >= 0 && gy >= 0 && gx < w && gy < h) continue;
    const int mr = mirror(gy, h) - (y0 - 3), mc = mirror(gx, w) - (x0 - 3);
    if (mr < 0 || mc < 0 || mr >= kGabH || mc >= kGabW) continue;  // never read
#pragma unroll
    for (int c = 0; c < 3; ++c) gab[c][r][col] = gab[c][mr][mc];
  }
  __syncthreads();
  // EPF pass 1 at the in-image slots of its region
  for (int e = threadIdx.x; e < kE1H * kE1W; e += blockDim.x) {
    const int r = e / kE1W, col = e % kE1W;
    const int x = x0 - 1 + col, y = y0 - 1 + r;
    if (x < 0 || y < 0 || x >= w || y >= h) continue;
    auto S = [&](int c, int dx, int dy) { return gab[c][r + 2 + dy][col + 2 + dx]; };
    float v[3];
    EpfPixel<1>(S, inverse_sigma[static_cast<size_t>(y / 8) * bw + x / 8], x, y, v);
#pragma unroll
    for (int c = 0; c < 3; ++c) e1[c][r][col] = v[c];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kE1H * kE1W; e += blockDim.x) {
    const int r = e / kE1W, col = e % kE1W;
    const int x = x0 - 1 + col, y = y0 - 1 + r;
    if (x >= 0 && y >= 0 && x < w && y < h) continue;
    const int mr = mirror(y, h) - (y0 - 1), mc = mirror(x, w) - (x0 - 1);
    if (mr < 0 || mc < 0 || mr >= kE1H || mc >= kE1W) continue;  // never read
#pragma unroll
    for (int c = 0; c < 3; ++c) e1[c][r][col] = e1[c][mr][mc];
  }
  __syncthreads();
  // EPF pass 2 on the tile, then XYB -> linear
  const int tx = threadIdx.x % kLfTileW;
  for (int ty = threadIdx.x / kLfTileW; ty < kLfTileH; ty += blockDim.x / kLfTileW) {
    const int x = x0 + tx, y = y0 + ty;
    if (x >= w || y >= h) continue;
    auto S = [&](int c, int dx, int dy) { return e1[c][ty + 1 + dy][tx + 1 + dx]; };
    float v[3];
    EpfPixel<2>(S, inverse_sigma[static_cast<size_t>(y / 8) * bw + x / 8], x, y, v);
    const size_t i = static_cast<size_t>(y) * w + x;
    for (int c = 0; c < 3; ++c) filtered[c * plane + i] = v[c];
    float rgb[3];
    OpsinToLinearPixel(v[0], v[1], v[2], p, rgb);
    for (int c = 0; c < 3; ++c) linear[c * plane + i] = rgb[c];
  }
}

}  // namespace

// Gaborish, EPF passes 1 and 2 of the padded reconstruction (stride pw,
// plane pw*ph) into filtered, and XYB -> linear into linear.  Both outputs
// are unpadded w x h planes.
GJXLResult LaunchLoopFiltersAndColor(hipStream_t s, const float* reconstructed,
                                     int pw, int ph, int w, int h,
                                     const float* inverse_sigma, float* filtered,
                                     float* linear, float intensity_target) {
  const float w1 = 1.1f * 0.104699568f, w2 = 1.1f * 0.055680538f;
  const float divisor = 1.0f + 4.0f * (w1 + w2);
  const GaborishWeights g{1.0f / divisor, w1 / divisor, w2 / divisor};
  // The host libm's cbrtf, as the reference evaluates it; the volatile keeps
  // the compiler from folding it with a different method.
  volatile float bias = 0.0037930732552754493f;
  InverseOpsin p{{{11.031566901960783f, -9.866943921568629f, -0.16462299647058826f},
                  {-3.254147380392157f, 4.418770392156863f, -0.16462299647058826f},
                  {-3.6588512862745097f, 2.7129230470588235f, 1.9459282392156863f}},
                 255.0f / intensity_target,
                 cbrtf(bias)};
  const dim3 grid(CeilDiv(w, kLfTileW), CeilDiv(h, kLfTileH));
  if (w >= 4 && h >= 4) {
    hipLaunchKernelGGL(LoopFilterKernel<true>, grid, dim3(256), 0, s, reconstructed, pw,
                       static_cast<size_t>(pw) * ph, w, h, g, inverse_sigma, p, filtered,
                       linear);
  } else {
    hipLaunchKernelGGL(LoopFilterKernel<false>, grid, dim3(256), 0, s, reconstructed, pw,
                       static_cast<size_t>(pw) * ph, w, h, g, inverse_sigma, p, filtered,
                       linear);
  }
  return CheckLaunch("LoopFilterKernel");
}

}  // namespace gjxl_amd
