// a16-a17: Butteraugli on the device and the per-transform 16-norm
// reduction of its map.
//
//   OpsinDynamicsKernel   5x5 mirrored blur + opsin dynamics (Gamma via the
//                         unfused FastLog2), butteraugli_internal.cpp:622-700
//   BlurKernel            separable Gaussian of radius 16, 7, 3 or 6 with the
//                         reference's interior summation order and its
//                         renormalised border columns (:245-620), both passes
//                         in one kernel; SeparateFrequencies (:702-846) and
//                         the masking activity are the blurs' epilogues
//   MaskKernel            fuzzy erosion, MaskY/MaskDcY
//   DifferencesKernel     MaltaDiffMap of the six stages (butteraugli_
//                         distance_internal.cpp:482-577, zero outside the
//                         image), their accumulation (UHF, HF, MF), the L2
//                         terms, masked AC Y and the final composition
//                         (:657-870), per tile
//   Expand/ComposeKernel  the two-scale map and its maximum (:872-1003); the
//                         half-scale image is formed where the opsin kernel
//                         reads it
//   ReduceKernel          ReduceButteraugliDistanceMap (butteraugli.cpp:
//                         116-222)
//
// Every output is computed by one thread in the reference's own operation
// order (binary32, no contraction; binary64 where the reference promotes), so
// the maps equal the CPU's bit for bit.  The reference image's planes and
// masking terms are computed once per prepare and stay resident.
//
// Every launch covers both scales: the work groups of the half scale follow
// those of the full one.  An image has some fifty kernels' worth of stages,
// and below about two megapixels each of them is over before the next launch
// could have filled the chip (a 512x512 preparation and comparison took 43 and
// 45 launches of 4 to 16 us each; now 6 and 7).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>

#include "butteraugli.h"
#include "libm_port.h"
#include "tables.h"
#include "tile_mirror.h"

namespace gjxl_amd {
namespace {

constexpr int kThreads = 256;
// A blur's taps travel in its kernel's arguments: read through a pointer they
// were vector loads at every use, since the planes a kernel writes may alias
// them as far as the compiler knows.
struct Taps {
  float k[33], sk[17];
};
constexpr float kSigmas[kSigmaCount] = {1.2f, 7.15593339443f, 3.22489901262f,
                                        1.56416327805f, 2.7f};

__device__ __forceinline__ float BMax(float a, float b) { return a < b ? b : a; }

// ---- Gaussian blurs --------------------------------------------------------

// An interior output of ConvolutionWithTranspose from the 2R + 1 samples
// s[0 .. 2R] around it (s[R] is the centre): mirrored pairs times the scaled
// taps, accumulated into four interleaved partial sums, in the reference's
// order.
template <int R>
__device__ __forceinline__ float ConvolveInterior(const float* s, const float* sk) {
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const float pair = (s[i] + s[2 * R - i]) * sk[i];
    acc[i % 4] = i < 4 ? pair : acc[i % 4] + pair;
  }
  float r = s[R] * sk[R];
#pragma unroll
  for (int i = 0; i < 4 && i < R; ++i) r = r + acc[i];
  return r;
}

// 1 / the weight of the taps that fall inside a line of `len` samples around
// the border position of index `i`: positions 0 .. R - 1 have the indexes 0 ..
// R - 1, those of the other end R .. 2R - 1 (BorderPosition).  Every tap is
// visited in ascending order and the ones outside are skipped by selects, so
// the sum is the reference's.
template <int R>
__device__ __forceinline__ int BorderPosition(int i, int len) {
  return i < R ? i : max(R, len - R) + i - R;
}
template <int R>
__device__ __forceinline__ int BorderIndex(int pos, int len) {
  return pos < R ? pos : R + pos - max(R, len - R);
}
template <int R>
__device__ __forceinline__ float BorderScale(int i, int len, const float* k) {
  const int pos = BorderPosition<R>(i, len);
  float weight = 0.0f;
#pragma unroll
  for (int t = 0; t <= 2 * R; ++t) {
    const int sx = pos - R + t;
    const float next = weight + k[t];
    weight = sx >= 0 && sx < len ? next : weight;
  }
  return 1.0f / weight;
}

// A border output of ConvolutionWithTranspose (fewer than R samples on one
// side): the taps that fall inside the line, in ascending order, renormalised
// by `scale`; sample(t) is the sample under tap t (any value outside),
// inside(t) whether it lies in the line.
template <int R, typename Sample, typename Inside>
__device__ __forceinline__ float ConvolveBorder(Sample sample, Inside inside, float scale,
                                                const float* k) {
  float sum = 0.0f;
#pragma unroll
  for (int t = 0; t <= 2 * R; ++t) {
    const float next = sum + sample(t) * k[t];
    sum = inside(t) ? next : sum;
  }
  return sum * scale;
}

// ---- the fused blur ---------------------------------------------------------
//
// A work group blurs a strip of kStripW columns by a segment of rows, both
// passes, without writing the row pass to memory.  It walks down the segment
// kBandH input rows at a time: the rows and their halo columns go to LDS
// (`stage`, fetched into registers while the previous band is computed), the
// row pass leaves them blurred in a ring of the last kGroups bands, and the
// column pass takes kBandH output rows from the ring.
//   * Row pass: a lane makes four adjacent outputs from one window of 16-byte
//     LDS reads (conflict-free).
//   * Column pass: a lane makes kOut outputs down one column from one window
//     of kOut + 2R ring rows; the epilogue consumes them (Load(row, x, in)
//     reads what the split of a pixel needs, Store(row, x, v, in) writes its
//     results; row, the offset of a whole row, is uniform, so the addresses
//     are scalar; a lane reads everything before its first store, which may
//     alias its reads as far as the compiler knows).
//   * Border rows and columns take the renormalised border convolution, with
//     the 2R reciprocal weights of each axis computed once per work group.
// What bounds it: at 12 megapixels the two passes' arithmetic, 2 (3R + 5)
// operations per output in the reference's order, and the latencies between
// a band's two barriers; below about two megapixels those latencies alone,
// which is why 512 lanes share a band (four outputs each) and not 256 (eight):
// radius 16 at 77x45 34 to 23 us, at 1537x1153 75 to 66, at 4032x3024 250 to
// 230.  The separate row and column kernels that this replaces wrote and read
// a plane more per pass, re-read 8 + 2R rows for every eight outputs of a
// column, and took 36 launches per image and scale pair where this takes
// four (all four radii at 4032x3024, reference image: 830 to 540 us; whole
// preparation and comparison at 1537x1153: 1063 to 490).
constexpr int kStripW = 128, kBandH = 16;
constexpr int kBlurThreads = 512;

template <int R>
struct BlurShape {
  // samples x - R .. x + 3 + R of a lane's outputs x .. x + 3, whole float4s
  static constexpr int kWindow = (2 * R + 4 + 3) / 4 * 4;
  static constexpr int kStageW = kStripW - 4 + kWindow;
  // bands of rows that an output band needs
  static constexpr int kGroups = (kBandH + 2 * R + kBandH - 1) / kBandH;
};

template <int R>
struct BlurShared {
  __align__(16) float stage[kBandH][BlurShape<R>::kStageW];
  __align__(16) float ring[BlurShape<R>::kGroups * kBandH][kStripW];
  float xscale[2 * R], yscale[2 * R];  // BorderScale of each border index
  // the unscaled taps, for the border outputs (in scalar registers beside the
  // scaled ones they spill)
  float taps[2 * R + 1];
};

// Fills the border scales; the first barrier of BlurSegment orders them.
template <int R>
__device__ __forceinline__ void BlurBegin(BlurShared<R>& sh, int w, int h,
                                          const Taps& taps) {
  const int t = threadIdx.x;
  if (t <= 2 * R) sh.taps[t] = taps.k[t];
  if (t < 4 * R) {
    const bool rows = t >= 2 * R;
    const float scale = BorderScale<R>(rows ? t - 2 * R : t, rows ? h : w, taps.k);
    (rows ? sh.yscale : sh.xscale)[rows ? t - 2 * R : t] = scale;
  }
}

// Rows y0 .. y1 - 1 (y1 - y0 a multiple of kBandH unless y1 is h) of the
// columns x0 .. of the planes that `epilogue` names: plane k of its order is
// epilogue.Input(k), and epilogue.Visit(k, f) calls f with that plane's split.
//
// The code is kept small: a work group runs each part of it a few times only,
// and straight-line code that no wave has run yet comes in at the latency of
// the instruction fetch.  So the planes share one copy (a uniform switch picks
// the split), interior outputs are computed for every row and lane, and
// the border outputs of a column are one rolled loop over the taps.  (Unrolled
// per plane and output, the 110 KB of the radius-16 kernel made the work groups
// at an image's border 2.5 times as long as the others.)
template <int R, int kT, typename Epilogue>
__device__ __forceinline__ void BlurSegment(BlurShared<R>& sh, int w, int h, int x0, int y0,
                                            int y1, const Taps& taps, int first_plane,
                                            int planes, const Epilogue& epilogue) {
  using S = BlurShape<R>;
  const float* sk = taps.sk;
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  constexpr int kWaveRows = kBandH / (kT / 64);
  constexpr int kOut = kStripW * kBandH / kT;  // outputs per lane and pass
  constexpr int kRowSets = kOut / 4;           // quads of outputs in the row pass
  constexpr int kRowStep = kBandH / kRowSets;
  constexpr int kLoads = (S::kStageW + 63) / 64;
  const int first_x = min(w, R), last_x = max(w - R, 0);
  const int first_y = min(h, R), last_y = max(h - R, 0);
  // stage column c holds sample x0 - R + c (clamped into the row: what lies
  // outside is never used)
  unsigned column[kLoads];
#pragma unroll
  for (int k = 0; k < kLoads; ++k) {
    column[k] = min(max(x0 - R + min(lane + 64 * k, S::kStageW - 1), 0), w - 1);
  }
  const int bands = (y1 - y0 + kBandH - 1) / kBandH;
  const int groups = bands + S::kGroups - 1;
  float next[kWaveRows][kLoads];
  // group g of plane k; past a plane's last group, the next plane's first
  auto fetch = [&](int k, int g) {
    if (g == groups) {
      ++k;
      g = 0;
    }
    if (k == planes) return;
    const float* in = epilogue.Input(k);
#pragma unroll
    for (int r = 0; r < kWaveRows; ++r) {
      const int y = min(max(y0 - R + kBandH * g + wave * kWaveRows + r, 0), h - 1);
      const float* row = in + static_cast<size_t>(y) * w;
#pragma unroll
      for (int c = 0; c < kLoads; ++c) next[r][c] = row[column[c]];
    }
  };
  // the strip's border columns: `left` from x0, then `right` from right_begin
  const int left = min(max(first_x - x0, 0), kStripW);
  const int right_begin = max(max(last_x, first_x), x0);
  const int border = left + max(min(w, x0 + kStripW) - right_begin, 0);
  // column pass: this lane's column and its kOut rows of a band
  const int col = tid % kStripW, part = wave / (kStripW / 64);
  const unsigned x = x0 + col;
  fetch(first_plane, 0);
#pragma unroll 1
  for (int k = first_plane; k < planes; ++k) {
    int slot = 0;  // ring band of group g: g % kGroups
#pragma unroll 1
    for (int g = 0; g < groups; ++g) {
#pragma unroll
      for (int r = 0; r < kWaveRows; ++r) {
#pragma unroll
        for (int c = 0; c < kLoads; ++c) {
          const int at = lane + 64 * c;
          if (at < S::kStageW) sh.stage[wave * kWaveRows + r][at] = next[r][c];
        }
      }
      __syncthreads();
      fetch(k, g + 1);
      {
        const int q = tid % (kStripW / 4);
#pragma unroll 1
        for (int m = 0; m < kRowSets; ++m) {
          const int row = tid / (kStripW / 4) + m * kRowStep;
          float window[S::kWindow];
          const float4* s4 = reinterpret_cast<const float4*>(&sh.stage[row][4 * q]);
#pragma unroll
          for (int j = 0; j < S::kWindow / 4; ++j) {
            const float4 v = s4[j];
            window[4 * j] = v.x;
            window[4 * j + 1] = v.y;
            window[4 * j + 2] = v.z;
            window[4 * j + 3] = v.w;
          }
          float r[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) r[j] = ConvolveInterior<R>(window + j, sk);
          // (a border column's lane writes its own output after this one)
          float* ring = &sh.ring[slot * kBandH + row][0];
          *reinterpret_cast<float4*>(ring + 4 * q) = make_float4(r[0], r[1], r[2], r[3]);
        }
      }
      if (border > 0) {
        // at most 2R <= 32 border columns, all rows: one lane per output, in
        // the wave that has written the interior form of the same rows
        const int b = tid % 32;
        const int xb = b < left ? x0 + b : right_begin + (b - left);
        const float scale = sh.xscale[b < border ? BorderIndex<R>(xb, w) : 0];
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (int m = 0; m < kRowSets; ++m) {
          const int row = tid / 32 + m * kRowStep;
          if (b < border) {
            const float* line = &sh.stage[row][xb - x0];
            sh.ring[slot * kBandH + row][xb - x0] =
              ConvolveBorder<R>([&](int t) { return line[t]; },
                                [&](int t) {
                                  return static_cast<unsigned>(xb - R + t) <
                                         static_cast<unsigned>(w);
                                },
                                scale, sh.taps);
          }
        }
      }
      __syncthreads();
      const int next_slot = slot + 1 == S::kGroups ? 0 : slot + 1;
      const int yb = y0 + kBandH * (g - (S::kGroups - 1)) + kOut * part;  // wave-uniform
      if (g >= S::kGroups - 1 && yb < y1 && x < static_cast<unsigned>(w)) {
        float split[kOut][Epilogue::kLoads];
        epilogue.Visit(k, [&](auto s) {
#pragma unroll
          for (int p = 0; p < kOut; ++p) {
            s.Load(static_cast<size_t>(min(yb + p, h - 1)) * w, x, split[p]);
          }
        });
        // the oldest band of the ring is the first that this band needs
        constexpr int kBlocks = (2 * R) / kOut + 1 + ((2 * R) % kOut != 0);
        constexpr int kBandBlocks = kBandH / kOut;
        float window[kOut * kBlocks];
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) {
          int block = kBandBlocks * next_slot + part + j;  // ring rows in blocks of kOut
          block = block >= kBandBlocks * S::kGroups ? block - kBandBlocks * S::kGroups : block;
#pragma unroll
          for (int i = 0; i < kOut; ++i) {
            if (kOut * j + i < kOut + 2 * R) window[kOut * j + i] = sh.ring[kOut * block + i][col];
          }
        }
        float v[kOut];
#pragma unroll
        for (int p = 0; p < kOut; ++p) v[p] = ConvolveInterior<R>(window + p, sk);
        if (yb < first_y || yb + kOut - 1 >= last_y) {
          // the taps of all outputs one after another: at tap t output p
          // needs ring row p + t of the window
          float sum[kOut] = {}, samples[kOut];
          auto ring_row = [&](int i) {
            int r = kBandH * next_slot + kOut * part + i;
            r = r >= S::kGroups * kBandH ? r - S::kGroups * kBandH : r;
            return sh.ring[r][col];
          };
#pragma unroll
          for (int p = 0; p < kOut; ++p) samples[p] = ring_row(p);
#pragma unroll 1
          for (int t = 0; t <= 2 * R; ++t) {
            const float after = ring_row(min(kOut + t, kOut - 1 + 2 * R));
            const float tap = sh.taps[t];
#pragma unroll
            for (int p = 0; p < kOut; ++p) {
              const float moved = sum[p] + samples[p] * tap;
              const bool inside = static_cast<unsigned>(yb + p - R + t) < static_cast<unsigned>(h);
              sum[p] = inside ? moved : sum[p];
              samples[p] = p + 1 < kOut ? samples[p + 1 < kOut ? p + 1 : p] : after;
            }
          }
#pragma unroll
          for (int p = 0; p < kOut; ++p) {
            const int y = yb + p;
            const bool interior = y >= first_y && y < last_y;
            const float scale = sh.yscale[interior ? 0 : BorderIndex<R>(min(y, h - 1), h)];
            v[p] = interior ? v[p] : sum[p] * scale;
          }
        }
        epilogue.Visit(k, [&](auto s) {
#pragma unroll
          for (int p = 0; p < kOut; ++p) {
            if (yb + p < y1) s.Store(static_cast<size_t>(yb + p) * w, x, v[p], split[p]);
          }
        });
      }
      slot = next_slot;
    }
  }
}

// ---- launches over both scales ------------------------------------------------

// The tiles of the full scale, then those of the half scale, in one
// one-dimensional grid; within a scale in the XCD-aware order (XcdTile).
struct ScaleTile {
  int scale, x, y, unit;
};
struct ScaleBlocks {
  unsigned tiles_w[2] = {1, 1}, count[2] = {0, 0};
  unsigned units = 1;  // work groups per tile, consecutive
  dim3 Grid() const { return dim3(count[0] + count[1]); }
  __device__ __forceinline__ ScaleTile Tile() const {
    constexpr unsigned kXcds = 8;
    const int scale = blockIdx.x >= count[0] ? 1 : 0;
    const unsigned i = blockIdx.x - (scale ? count[0] : 0);
    const unsigned per = count[scale] / kXcds;
    const unsigned t = i < per * kXcds ? (i % kXcds) * per + i / kXcds : i;
    const unsigned tile = t / units;
    return {scale, static_cast<int>(tile % tiles_w[scale]), static_cast<int>(tile / tiles_w[scale]),
            static_cast<int>(t % units)};
  }
};

// ---- opsin dynamics ---------------------------------------------------------

__device__ __forceinline__ float ButteraugliFastLog2(float v) {
  const uint32_t bits = __float_as_uint(v);
  const int32_t e = static_cast<int32_t>(bits - 0x3f2aaaabu) >> 23;
  const float x = __uint_as_float(bits - (static_cast<uint32_t>(e) << 23)) - 1.0f;
  float num = 0.74245873327820566f * x + 1.4287160470083755f;
  num = num * x + -1.8503833400518310e-06f;
  float den = 0.17409343003366853f * x + 1.0096718572241148f;
  den = den * x + 0.99032814277590719f;
  return num / den + static_cast<float>(e);
}

__device__ __forceinline__ float ButteraugliGamma(float v) {
  constexpr float kRetMul = 19.245013259874995f * 0.6931471805599453f;
  v = BMax(v, 0.0f);
  return kRetMul * ButteraugliFastLog2(v + 9.9710635769299145f) + -23.16046239805755f;
}

__device__ __forceinline__ void Absorbance(float r, float g, float b, bool clamp,
                                           float out[3]) {
  out[0] = 0.29956550340058319f * r +
           (0.63373087833825936f * g + (0.077705617820981968f * b + 1.7557483643287353f));
  out[1] = 0.22158691104574774f * r +
           (0.69391388044116142f * g + (0.0987313588422f * b + 1.7557483643287353f));
  out[2] = 0.02f * r + (0.02f * g + (0.20480129041026129f * b + 12.226454707163354f));
  if (clamp) {
    out[0] = BMax(out[0], 1.7557483643287353f);
    out[1] = BMax(out[1], 1.7557483643287353f);
    out[2] = BMax(out[2], 12.226454707163354f);
  }
}

// One work group per 64x16 tile: the three planes' tile with a mirrored
// 2-pixel halo in LDS, then per pixel the 5-tap horizontal sums of the five
// rows it needs and their vertical combination, in the reference's order.
// The half scale's image (SubSample2x of the linear one) is formed as its
// tiles are read: four reads per sample of an image that the full scale has
// just pulled into the caches, instead of a launch that wrote and re-read
// three planes.
// Both scales are at least 8 pixels a side, and every lane of a tile reads: in
// a plane narrower than 33 pixels or lower than 9 also further outside it than
// one reflection reaches (TileMirror holds those reads inside the image).
constexpr int kOpsinTileW = 64, kOpsinTileH = 16;
constexpr int kOpsinRows = kOpsinTileH / (kThreads / kOpsinTileW);  // per thread

struct OpsinArgs {
  ScaleBlocks blocks;
  const float* rgb;  // the full scale's image
  int w[2], h[2];
  float* xyb[2];
  float intensity;
  Taps taps;
  uint32_t* score;  // cleared for the comparison that follows, or null
};

__global__ __launch_bounds__(kThreads) void OpsinDynamicsKernel(OpsinArgs args) {
  constexpr int TW = kOpsinTileW + 4, TH = kOpsinTileH + 4;
  __shared__ float tile[3][TH][TW];
  const ScaleTile at = args.blocks.Tile();
  const int x0 = at.x * kOpsinTileW, y0 = at.y * kOpsinTileH;
  const int w = args.w[at.scale], h = args.h[at.scale];
  const size_t n = static_cast<size_t>(w) * h;
  const float intensity = args.intensity;
  const float* __restrict__ rgb = args.rgb;
  float* __restrict__ xyb = args.xyb[at.scale];
  if (args.score != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *args.score = 0;
  // The tile's 3 x TH rows of TW = 64 + 4 columns: each wave reads kWaveRows
  // whole rows, one lane per column of the first 64, with the row address
  // uniform (scalar arithmetic); the last 4 columns of every row are one
  // read per thread.  Every read issues before the first store.
  static_assert(TW == 64 + 4 && (3 * TH) % (kThreads / 64) == 0 && 3 * TH * 4 <= kThreads,
                "tile rows split over the waves");
  constexpr int kWaveRows = 3 * TH / (kThreads / 64);
  constexpr int kStripCount = 3 * TH * 4;
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64));
  const int sx = TileMirror(x0 - 2 + lane, w);
  const int e = min(static_cast<int>(threadIdx.x), kStripCount - 1);
  const int strip_c = e / 4 / TH;
  const int strip_y = TileMirror(y0 - 2 + e / 4 % TH, h);
  const int strip_x = TileMirror(x0 - 2 + 64 + e % 4, w);
  float rows[kWaveRows];
  float strip;
  if (at.scale == 0) {
#pragma unroll
    for (int i = 0; i < kWaveRows; ++i) {
      const int row = wave * kWaveRows + i;
      const int c = row / TH, r = row % TH;
      rows[i] = rgb[c * n + static_cast<size_t>(TileMirror(y0 - 2 + r, h)) * w + sx];
    }
    strip = rgb[strip_c * n + static_cast<size_t>(strip_y) * w + strip_x];
  } else {
    const int fw = args.w[0], fh = args.h[0];
    const size_t fn = static_cast<size_t>(fw) * fh;
    // the four samples under half-scale sample (x, y) of plane c, clamped
    // into the image
    struct Quad {
      float a, b, d, e;
    };
    auto read = [&](int c, int x, int y) {
      const int x1 = 2 * x + 1 < fw ? 2 * x + 1 : 2 * x;
      const float* r0 = rgb + c * fn + static_cast<size_t>(2 * y) * fw;
      const float* r1 = rgb + c * fn + static_cast<size_t>(min(2 * y + 1, fh - 1)) * fw;
      return Quad{r0[2 * x], r0[x1], r1[2 * x], r1[x1]};
    };
    // their sum over the in-image ones, in the reference's order
    auto sum = [&](Quad q, int x, int y) {
      // (the empty asm keeps the compiler from moving a read under its select)
      asm volatile("" : "+v"(q.a), "+v"(q.b), "+v"(q.d), "+v"(q.e));
      const bool right = 2 * x + 1 < fw, below = 2 * y + 1 < fh;
      float v = 0.0f + 0.25f * q.a;
      v = right ? v + 0.25f * q.b : v;
      const float lower = v + 0.25f * q.d;
      v = below ? (right ? lower + 0.25f * q.e : lower) : v;
      if ((fw & 1) && x == w - 1) v *= 2.0f;
      if ((fh & 1) && y == h - 1) v *= 2.0f;
      return v;
    };
    Quad quads[kWaveRows];
#pragma unroll
    for (int i = 0; i < kWaveRows; ++i) {
      const int row = wave * kWaveRows + i;
      quads[i] = read(row / TH, sx, TileMirror(y0 - 2 + row % TH, h));
    }
    const Quad strip_quad = read(strip_c, strip_x, strip_y);
#pragma unroll
    for (int i = 0; i < kWaveRows; ++i) {
      rows[i] = sum(quads[i], sx, TileMirror(y0 - 2 + (wave * kWaveRows + i) % TH, h));
    }
    strip = sum(strip_quad, strip_x, strip_y);
  }
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) {
    (&tile[0][0][0])[(wave * kWaveRows + i) * TW + lane] = rows[i];
  }
  if (threadIdx.x < kStripCount) {
    (&tile[0][0][0])[(threadIdx.x / 4) * TW + 64 + threadIdx.x % 4] = strip;
  }
  __syncthreads();
  const float w0 = args.taps.sk[2], w1 = args.taps.sk[1], w2 = args.taps.sk[0];
  const int lx = threadIdx.x % kOpsinTileW;
  const int ly0 = (threadIdx.x / kOpsinTileW) * kOpsinRows;
  const int x = x0 + lx;
  if (x >= w) return;
  // horizontal sums of tile rows ly0 .. ly0 + kOpsinRows + 3, per channel
  float hz[3][kOpsinRows + 4];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
#pragma unroll
    for (int r = 0; r < kOpsinRows + 4; ++r) {
      const float* row = &tile[c][ly0 + r][lx + 2];
      float v = row[0] * w0;
      v = (row[-1] + row[1]) * w1 + v;
      v = (row[-2] + row[2]) * w2 + v;
      hz[c][r] = v;
    }
  }
#pragma unroll
  for (int j = 0; j < kOpsinRows; ++j) {
    const int y = y0 + ly0 + j;
    if (y >= h) break;
    float blurred[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      float r = hz[c][j + 2] * w0;
      r = (hz[c][j + 1] + hz[c][j + 3]) * w1 + r;
      r = (hz[c][j] + hz[c][j + 4]) * w2 + r;
      blurred[c] = r;
    }
    const size_t i = static_cast<size_t>(y) * w + x;
    float pre[3], cur[3], sens[3];
    Absorbance(blurred[0] * intensity, blurred[1] * intensity, blurred[2] * intensity,
               true, pre);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      pre[c] = BMax(pre[c], 1.0e-4f);
      sens[c] = BMax(ButteraugliGamma(pre[c]) / pre[c], 1.0e-4f);
    }
    const int ly = ly0 + j + 2, tx = lx + 2;
    Absorbance(tile[0][ly][tx] * intensity, tile[1][ly][tx] * intensity,
               tile[2][ly][tx] * intensity, false, cur);
    cur[0] = BMax(cur[0] * sens[0], 1.7557483643287353f);
    cur[1] = BMax(cur[1] * sens[1], 1.7557483643287353f);
    cur[2] = BMax(cur[2] * sens[2], 12.226454707163354f);
    xyb[i] = cur[0] - cur[1];
    xyb[n + i] = cur[0] + cur[1];
    xyb[2 * n + i] = cur[2];
  }
}

// ---- frequency separation ---------------------------------------------------

__device__ __forceinline__ float MaximumClamp(float v, float maximum) {
  constexpr float k = 0.724216145665f;
  if (v >= maximum) return (v - maximum) * k + maximum;
  if (v < -maximum) return (v + maximum) * k + -maximum;
  return v;
}
__device__ __forceinline__ float RemoveRange(float v, float width) {
  if (v > width) return v - width;
  if (v < -width) return v + width;
  return 0.0f;
}
__device__ __forceinline__ float AmplifyRange(float v, float width) {
  if (v > width) return v + width;
  if (v < -width) return v - width;
  return v + v;
}

// The blurs of SeparateFrequencies and their splits.  A blur reads its whole
// neighbourhood, so no split writes the plane that its blur reads: the MF
// planes before their blur, the HF planes before theirs and the masking
// activity before its own are scratch planes.  A split reads kLoads values
// per pixel; where the second plane of a work group needs the first one's
// result at the same pixel, the same lane has written it.

struct StoreBlur {
  float* out;
  __device__ __forceinline__ void Load(size_t, unsigned, float* in) const { in[0] = 0.0f; }
  __device__ __forceinline__ void Store(size_t row, unsigned x, float v, const float*) const {
    (out + row)[x] = v;
  }
};

// The LF blur v of channel C: MF = XYB - LF, then the LF plane scaled.  Y's
// LF stays raw until B's pass, which needs it and then scales it.
template <int C>
struct LowSplit {
  const float* xyb;
  float* lf;
  float* mf;
  size_t n;
  __device__ __forceinline__ void Load(size_t row, unsigned x, float* in) const {
    in[0] = (xyb + C * n + row)[x];
    if constexpr (C == 2) in[1] = (lf + n + row)[x];
  }
  __device__ __forceinline__ void Store(size_t row, unsigned x, float v, const float* in) const {
    (mf + C * n + row)[x] = in[0] - v;
    if constexpr (C == 0) {
      (lf + row)[x] = v * 33.832837186260f;
    } else if constexpr (C == 1) {
      (lf + n + row)[x] = v;
    } else {
      const float ly = in[1];
      (lf + 2 * n + row)[x] = (-0.362267051518f * ly + v) * 49.87984651440f;
      (lf + n + row)[x] = ly * 14.458268100570f;
    }
  }
};

// The 3.22 blur v of MF channel C: HF and MF of channel C; channel 1 also
// applies SuppressXByY to HF X.
template <int C>
struct HighSplit {
  const float* raw;  // the MF planes before the blur
  float* mf;
  float* hf;
  size_t n;
  __device__ __forceinline__ void Load(size_t row, unsigned x, float* in) const {
    in[0] = C == 2 ? 0.0f : (raw + C * n + row)[x];
    if constexpr (C == 1) in[1] = (hf + row)[x];
  }
  __device__ __forceinline__ void Store(size_t row, unsigned x, float v, const float* in) const {
    if constexpr (C == 2) {
      (mf + 2 * n + row)[x] = v;
      return;
    }
    const float high = in[0] - v;
    (hf + C * n + row)[x] = high;
    (mf + C * n + row)[x] = C == 0 ? RemoveRange(v, 0.29f) : AmplifyRange(v, 0.1f);
    if constexpr (C == 1) {
      constexpr float kS = 46.0f, kMin = 0.653020556257f;
      const float scaler = (kS / (high * high + kS)) * (1.0f - kMin) + kMin;
      (hf + row)[x] = scaler * in[1];
    }
  }
};

// The 1.56 blur v of HF channel C: UHF and HF of channel C; channel 1 also
// forms the masking activity (CombineChannelsForMasking + DiffPrecompute).
template <int C>
struct UltraSplit {
  const float* raw;  // the HF planes before the blur
  float* hf;
  float* uhf;
  float* activity;
  size_t n;
  __device__ __forceinline__ void Load(size_t row, unsigned x, float* in) const {
    in[0] = (raw + C * n + row)[x];
    if constexpr (C == 1) {
      in[1] = (uhf + row)[x];
      in[2] = (hf + row)[x];
    }
  }
  __device__ __forceinline__ void Store(size_t row, unsigned x, float v, const float* in) const {
    const float original = in[0];
    float hv = v;
    if constexpr (C == 0) {
      (uhf + row)[x] = RemoveRange(original - hv, 0.04f);
      (hf + row)[x] = RemoveRange(hv, 1.5f);
    } else {
      hv = MaximumClamp(hv, 28.4691806922f);
      float uv = original - hv;
      uv = MaximumClamp(uv, 5.19175294647f);
      const float uhf_y = uv * 2.69313763794f;
      const float hf_y = AmplifyRange(hv * 2.155f, 0.132f);
      (uhf + n + row)[x] = uhf_y;
      (hf + n + row)[x] = hf_y;
      constexpr float kMul = 6.19424080439f;
      const float bias = kMul * 12.61050594197f;
      const float sqrt_bias = sqrtf(bias);
      const float xd = (in[1] + in[2]) * 2.5f;
      const float yd = uhf_y * 0.4f + hf_y * 0.4f;
      const float a = sqrtf(xd * xd + yd * yd);
      (activity + row)[x] = sqrtf(kMul * fabsf(a) + bias) - sqrt_bias;
    }
  }
};

// One scale of a blur: the planes it reads, the psycho image it writes and
// the scratch planes that the next blur reads.
struct BlurScale {
  const float* in;
  float* psycho;
  float* scratch;
  int w, h;
  size_t n;
};
struct BlurArgs {
  ScaleBlocks blocks;  // tiles of kStripW columns by `rows` rows
  BlurScale scale[2];
  Taps taps;
  int rows;
};

// The planes of each blur in the order a work group takes them: the one that
// stands alone, then the two of which the second needs the first one's result.
// With two units in the grid, unit 1 takes the first plane and unit 0 the
// others.

// in: XYB; scratch: the raw MF planes.  X, Y, B.
struct LowPlanes {
  static constexpr int kLoads = 2;
  const BlurScale& s;
  __device__ __forceinline__ const float* Input(int k) const { return s.in + k * s.n; }
  template <typename F>
  __device__ __forceinline__ void Visit(int k, F&& f) const {
    if (k == 0) f(LowSplit<0>{s.in, s.psycho, s.scratch, s.n});
    else if (k == 1) f(LowSplit<1>{s.in, s.psycho, s.scratch, s.n});
    else f(LowSplit<2>{s.in, s.psycho, s.scratch, s.n});
  }
};

// in: the raw MF planes; scratch: the raw HF planes.  B, X, Y.
struct HighPlanes {
  static constexpr int kLoads = 2;
  const BlurScale& s;
  __device__ __forceinline__ const float* Input(int k) const {
    return s.in + (k == 0 ? 2 : k - 1) * s.n;
  }
  template <typename F>
  __device__ __forceinline__ void Visit(int k, F&& f) const {
    float* mf = s.psycho + 3 * s.n;
    if (k == 0) f(HighSplit<2>{s.in, mf, s.scratch, s.n});
    else if (k == 1) f(HighSplit<0>{s.in, mf, s.scratch, s.n});
    else f(HighSplit<1>{s.in, mf, s.scratch, s.n});
  }
};

// in: the raw HF planes; scratch: the masking activity.  X, Y.
struct UltraPlanes {
  static constexpr int kLoads = 3;
  const BlurScale& s;
  __device__ __forceinline__ const float* Input(int k) const { return s.in + k * s.n; }
  template <typename F>
  __device__ __forceinline__ void Visit(int k, F&& f) const {
    float* hf = s.psycho + 6 * s.n;
    float* uhf = s.psycho + 8 * s.n;
    if (k == 0) f(UltraSplit<0>{s.in, hf, uhf, s.scratch, s.n});
    else f(UltraSplit<1>{s.in, hf, uhf, s.scratch, s.n});
  }
};

// in: the masking activity; scratch: the blurred activity.
struct MaskPlanes {
  static constexpr int kLoads = 1;
  const BlurScale& s;
  __device__ __forceinline__ const float* Input(int) const { return s.in; }
  template <typename F>
  __device__ __forceinline__ void Visit(int, F&& f) const {
    f(StoreBlur{s.scratch});
  }
};

template <int R, int kT, typename Planes, int kPlanes>
__global__ __launch_bounds__(kT, 4) void BlurKernel(BlurArgs a) {
  __shared__ BlurShared<R> sh;
  const ScaleTile t = a.blocks.Tile();
  const BlurScale s = a.scale[t.scale];
  const int x0 = t.x * kStripW, y0 = t.y * a.rows;
  const bool split = a.blocks.units == 2;
  BlurBegin<R>(sh, s.w, s.h, a.taps);
  BlurSegment<R, kT>(sh, s.w, s.h, x0, y0, min(y0 + a.rows, s.h), a.taps, split && t.unit == 0 ? 1 : 0,
                 split && t.unit == 1 ? 1 : kPlanes, Planes{s});
}

// ---- difference stages -------------------------------------------------------

struct MaltaScale {
  double gt;   // norm2_0_gt_1, a binary32 value
  double lt;   // norm2_0_lt_1, a binary32 value
  float norm;  // (float)norm
};

// The scaled difference MaltaDiffMap feeds its lines (butteraugli_distance_
// internal.cpp:512-555).
//
// The two binary32 quotients gt / den and lt / den come from one binary64
// reciprocal: r = 1 / den to within 2^-52 relative (hardware estimate and two
// Newton steps), then the binary64 product rounded to binary32.  A quotient
// of two binary32 values is never a binary32 rounding midpoint and lies at
// least 2^-49 (relative) from every midpoint, so a binary64 value within
// 2^-51 of it rounds to the same binary32 value: the correctly rounded
// quotient, as binary32 division gives.
//
// The four corrections s -/+ ds2 * (...) are one s +/- ds2 * (u - k) with
// u = |v1| mirrored by the sign of v0 and k = too_small or too_big picked by
// selects: negation is exact and rounding is symmetric, so -(x + y) is
// (-x) + (-y) and x - y is x + (-y), and the result is the reference's.
__device__ __forceinline__ float MaltaScaledDiff(float v0, float v1, const MaltaScale& m) {
  const float absolute = 0.5f * (fabsf(v0) + fabsf(v1));
  const float diff = v0 - v1;
  const double den = m.norm + absolute;
  double r = __builtin_amdgcn_rcp(den);
  r = fma(fma(-den, r, 1.0), r, r);
  r = fma(fma(-den, r, 1.0), r, r);
  const float scaler = static_cast<float>(m.gt * r);
  const float s = scaler * diff;
  const double ds2 = static_cast<float>(m.lt * r);
  const double magnitude = fabs(static_cast<double>(v0));
  const double too_small = 0.55 * magnitude, too_big = 1.05 * magnitude;
  // v0 < 0: dv1 > -too_small: s - ds2 * (dv1 + too_small)
  //         dv1 < -too_big:   s + ds2 * (-dv1 - too_big)
  // v0 >= 0: dv1 < too_small: s + ds2 * (too_small - dv1)
  //          dv1 > too_big:   s - ds2 * (dv1 - too_big)
  const bool negative = v0 < 0.0f;
  const double u = negative ? -v1 : v1;
  const bool near = u < too_small;
  const bool far = u > too_big;
  const double k = near ? too_small : too_big;
  const double w = ds2 * (u - k);
  const double ds = s;
  const float corrected = static_cast<float>(negative ? ds + w : ds - w);
  return near || far ? corrected : s;
}

// Keeps one Malta window's responses computed before the next window's LDS
// reads: an empty asm statement that takes the four values and orders
// memory, so that the compiler neither sinks their arithmetic below it nor
// hoists the next reads above it (with all windows live at once the kernel
// would need over 400 registers).
__device__ __forceinline__ void Settle(const float (&v)[4]) {
  asm volatile("" : : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]) : "memory");
}

__device__ __forceinline__ float Sum4(float a, float b, float c, float d) {
  return (a + b) + (c + d);
}

// The 16 Malta lines (MaltaUnitLf / MaltaUnitFull).  Offsets as (dx, dy).
struct MaltaTap {
  signed char dx, dy;
};
constexpr MaltaTap kLfLines[16][5] = {
  {{-4, 0}, {-2, 0}, {0, 0}, {2, 0}, {4, 0}},
  {{0, -4}, {0, -2}, {0, 0}, {0, 2}, {0, 4}},
  {{-3, -3}, {-2, -2}, {0, 0}, {2, 2}, {3, 3}},
  {{3, -3}, {2, -2}, {0, 0}, {-2, 2}, {-3, 3}},
  {{1, -4}, {1, -2}, {0, 0}, {-1, 2}, {-1, 4}},
  {{-1, -4}, {-1, -2}, {0, 0}, {1, 2}, {1, 4}},
  {{-4, -1}, {-2, -1}, {0, 0}, {2, 1}, {4, 1}},
  {{-4, 1}, {-2, 1}, {0, 0}, {2, -1}, {4, -1}},
  {{-2, -3}, {-1, -2}, {0, 0}, {1, 2}, {2, 3}},
  {{2, -3}, {1, -2}, {0, 0}, {-1, 2}, {-2, 3}},
  {{-3, -2}, {-2, -1}, {0, 0}, {2, 1}, {3, 2}},
  {{3, -2}, {2, -1}, {0, 0}, {-2, 1}, {-3, 2}},
  {{-4, 2}, {-2, 1}, {0, 0}, {2, -1}, {4, -2}},
  {{-4, -2}, {-2, -1}, {0, 0}, {2, 1}, {4, 2}},
  {{-2, -4}, {-1, -2}, {0, 0}, {1, 2}, {2, 4}},
  {{2, -4}, {1, -2}, {0, 0}, {-1, 2}, {-2, 4}},
};
constexpr int kFullTaps[16] = {9, 9, 7, 7, 9, 9, 9, 9, 7, 7, 7, 7, 9, 9, 9, 9};
constexpr MaltaTap kFullLines[16][9] = {
  {{-4, 0}, {-3, 0}, {-2, 0}, {-1, 0}, {0, 0}, {1, 0}, {2, 0}, {3, 0}, {4, 0}},
  {{0, -4}, {0, -3}, {0, -2}, {0, -1}, {0, 0}, {0, 1}, {0, 2}, {0, 3}, {0, 4}},
  {{-3, -3}, {-2, -2}, {-1, -1}, {0, 0}, {1, 1}, {2, 2}, {3, 3}},
  {{3, -3}, {2, -2}, {1, -1}, {0, 0}, {-1, 1}, {-2, 2}, {-3, 3}},
  {{1, -4}, {1, -3}, {1, -2}, {0, -1}, {0, 0}, {0, 1}, {-1, 2}, {-1, 3}, {-1, 4}},
  {{-1, -4}, {-1, -3}, {-1, -2}, {0, -1}, {0, 0}, {0, 1}, {1, 2}, {1, 3}, {1, 4}},
  {{-4, -1}, {-3, -1}, {-2, -1}, {-1, 0}, {0, 0}, {1, 0}, {2, 1}, {3, 1}, {4, 1}},
  {{-4, 1}, {-3, 1}, {-2, 1}, {-1, 0}, {0, 0}, {1, 0}, {2, -1}, {3, -1}, {4, -1}},
  {{-2, -3}, {-1, -2}, {-1, -1}, {0, 0}, {1, 1}, {1, 2}, {2, 3}},
  {{2, -3}, {1, -2}, {1, -1}, {0, 0}, {-1, 1}, {-1, 2}, {-2, 3}},
  {{-3, -2}, {-2, -1}, {-1, -1}, {0, 0}, {1, 1}, {2, 1}, {3, 2}},
  {{3, -2}, {2, -1}, {1, -1}, {0, 0}, {-1, 1}, {-2, 1}, {-3, 2}},
  {{-4, 1}, {-3, 1}, {-2, 1}, {-1, 0}, {0, 0}, {1, 0}, {2, -1}, {3, -1}, {4, -1}},
  {{-4, -1}, {-3, -1}, {-2, -1}, {-1, 0}, {0, 0}, {1, 0}, {2, 1}, {3, 1}, {4, 1}},
  {{-1, -4}, {-1, -3}, {-1, -2}, {0, -1}, {0, 0}, {0, 1}, {1, 2}, {1, 3}, {1, 4}},
  {{1, -4}, {1, -3}, {1, -2}, {0, -1}, {0, 0}, {0, 1}, {-1, 2}, {-1, 3}, {-1, 4}},
};

// Tiles of the difference stages: 64x32 outputs, a 4-pixel halo.
constexpr int kMaltaTileW = 64, kMaltaTileH = 32, kMaltaHalo = 4;
constexpr int kMaltaLw = kMaltaTileW + 2 * kMaltaHalo, kMaltaLh = kMaltaTileH + 2 * kMaltaHalo;
constexpr int kMaltaQuads = kMaltaTileW / 4;
constexpr int kMaltaWinW = 4 + 2 * kMaltaHalo, kMaltaWinH = 1 + 2 * kMaltaHalo;
constexpr int kMaltaRowsPerPass = kThreads / kMaltaQuads;
static_assert(kMaltaTileH == 2 * kMaltaRowsPerPass, "two rows of four outputs per thread");
static_assert(kMaltaLw % 4 == 0, "16-byte aligned LDS rows");

struct L2Weights {
  float asym_gt[2];  // weight_0_gt_1 * 0.8 for HF X, Y
  float asym_lt[2];  // weight_0_lt_1 * 0.8
  bool asym_on[2];
  float mf[3];
  float lf[3];
};

// The 16 Malta lines of one pixel (MaltaUnitLf / MaltaUnitFull) from a
// register window P(dx, dy), summed in the reference's order, 0 + response.
template <bool kLowFrequency, typename Window>
__device__ __forceinline__ float MaltaResponse(Window P) {
  float result = 0.0f;
#pragma unroll
  for (int l = 0; l < 16; ++l) {
    float s;
    if constexpr (kLowFrequency) {
      const MaltaTap* t = kLfLines[l];
      s = Sum4(P(t[0].dx, t[0].dy), P(t[1].dx, t[1].dy), P(t[2].dx, t[2].dy),
               P(t[3].dx, t[3].dy) + P(t[4].dx, t[4].dy));
    } else {
      const MaltaTap* t = kFullLines[l];
      float v[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) v[k] = k < kFullTaps[l] ? P(t[k].dx, t[k].dy) : 0.0f;
      s = kFullTaps[l] == 9
            ? (Sum4(v[0], v[1], v[2], v[3]) + Sum4(v[4], v[5], v[6], v[7])) + v[8]
            : Sum4(v[0], v[1], v[2], Sum4(v[3], v[4], v[5], v[6]));
    }
    result = l == 0 ? s * s : s * s + result;
  }
  return 0.0f + result;
}

// The psycho plane of Malta stage k (MF Y, MF X, HF Y, HF X, UHF Y, UHF X)
// and its line set (low-frequency lines for the first four).
constexpr int kMaltaPlanes[6] = {4, 3, 7, 6, 9, 8};
struct MaltaScales {
  MaltaScale m[6];
};

// The difference stages of one scale, fused per 64x32 tile:
// * MaltaDiffMap of the six stages, three at a time: the scaled differences
//   of the tile and its 4-pixel halo for each of three stages go to LDS
//   (zero outside the image, as the reference's ReadWithZeroBorder), the
//   reads of one stage issued before the previous stage's differences; each
//   thread then evaluates four adjacent outputs of a row, for two rows, from
//   9 x 12 register windows of 16-byte LDS reads, and stores the stage;
// * the Malta accumulation in the reference's order (UHF, HF, MF per
//   channel): the first three stages are UHF Y, HF Y and UHF X, and their
//   partial sums ((0 + UHF Y) + HF Y, 0 + UHF X) go to planes 0 and 1 of
//   `stages`, which the same thread reads back after the last three (HF X,
//   MF X, MF Y);
// * then the asymmetric HF and symmetric MF L2 terms, the DC differences
//   from LF, the Y blurred-activity term, masking and the final map
//   (MaskPsychoImage / CombineChannelsToDiffmap): stage 8.
// kKeepStages stores the six Malta maps (stages 0-5) and the masked Y term
// (stage 7) for inspection instead, and forms the partial sums from the
// first three maps read back; without it only the partial sums and the
// final map are written.
// Three stages of LDS (34.6 KB) let four work groups share a CU.
struct DifferencesScale {
  const float* ps0;
  const float* ps1;
  const float* ref_blurred;
  const float* dist_blurred;
  const float* mask_y;
  const float* mask_dc;
  float* stages;
  int w, h;
};
struct DifferencesArgs {
  ScaleBlocks blocks;
  DifferencesScale scale[2];
  MaltaScales ms;
  L2Weights lw;
  float x_multiplier;
};
template <bool kKeepStages>
__global__ __launch_bounds__(kThreads) void DifferencesKernel(DifferencesArgs args) {
  __shared__ __align__(16) float tile[3][kMaltaLh][kMaltaLw];
  const ScaleTile at = args.blocks.Tile();
  const DifferencesScale& sc = args.scale[at.scale];
  const float* __restrict__ ps0 = sc.ps0;
  const float* __restrict__ ps1 = sc.ps1;
  const float* __restrict__ ref_blurred = sc.ref_blurred;
  const float* __restrict__ dist_blurred = sc.dist_blurred;
  const float* __restrict__ mask_y = sc.mask_y;
  const float* __restrict__ mask_dc = sc.mask_dc;
  float* __restrict__ stages = sc.stages;
  const int w = sc.w, h = sc.h;
  const MaltaScales& ms = args.ms;
  const L2Weights& lw = args.lw;
  const float x_multiplier = args.x_multiplier;
  const TileIndex tile_index{at.x, at.y};
  const int x0 = tile_index.x * kMaltaTileW, y0 = tile_index.y * kMaltaTileH;
  const size_t n = static_cast<size_t>(w) * h;
  const int tid = threadIdx.x;
  // A stage's tile is kMaltaLh rows of kMaltaLw = 64 + 8 columns.  Each wave
  // forms kFormRows whole rows, one lane per column of the first 64, with
  // the row's address and its inside test uniform (scalar arithmetic); the
  // last 8 columns of every row are kFormStrip elements per thread.  Reads
  // are clamped to the image (32-bit byte offsets: a plane is under 4 GiB)
  // and elements outside it are zero.
  static_assert(kMaltaLw == 64 + 8 && kMaltaLh % (kThreads / 64) == 0, "rows split over the waves");
  constexpr int kFormRows = kMaltaLh / (kThreads / 64);
  constexpr int kStripCount = kMaltaLh * 8;
  constexpr int kFormStrip = (kStripCount + kThreads - 1) / kThreads;
  constexpr int kFormSlots = kFormRows + kFormStrip;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  // The index arithmetic of a formation is recomputed each time from an
  // opaque copy of the thread index: shared with the first formation, its
  // results would stay live through the first Malta phase and cost the
  // registers of a fourth wave per SIMD.
  struct FormIndex {
    uint32_t offset[kFormSlots];  // byte offset within a plane
    bool inside[kFormSlots];
    int lds[kFormStrip];          // tile index of the strip elements
  };
  auto index = [&](FormIndex& f) {
    int t = tid;
    asm volatile("" : "+v"(t));
    const int lane = t % 64;
    const int sx = x0 + lane - kMaltaHalo;
    const uint32_t sx4 = 4u * static_cast<uint32_t>(min(max(sx, 0), w - 1));
    const bool col_in = sx >= 0 && sx < w;
#pragma unroll
    for (int j = 0; j < kFormRows; ++j) {
      const int sy = y0 + wave * kFormRows + j - kMaltaHalo;
      f.offset[j] = 4u * static_cast<uint32_t>(min(max(sy, 0), h - 1) * w) + sx4;
      f.inside[j] = col_in && sy >= 0 && sy < h;
    }
#pragma unroll
    for (int j = 0; j < kFormStrip; ++j) {
      const int e = min(t + j * kThreads, kStripCount - 1);
      const int r = e / 8, col = 64 + e % 8;
      const int sy = y0 + r - kMaltaHalo, sxs = x0 + col - kMaltaHalo;
      f.offset[kFormRows + j] =
        4u * static_cast<uint32_t>(min(max(sy, 0), h - 1) * w + min(max(sxs, 0), w - 1));
      f.inside[kFormRows + j] = sxs >= 0 && sy >= 0 && sxs < w && sy < h;
      f.lds[j] = t + j * kThreads < kStripCount ? r * kMaltaLw + col : -1;
    }
  };
  auto load = [&](int k, const FormIndex& f, float (&v0)[kFormSlots], float (&v1)[kFormSlots]) {
    const char* p0 = reinterpret_cast<const char*>(ps0 + kMaltaPlanes[k] * n);
    const char* p1 = reinterpret_cast<const char*>(ps1 + kMaltaPlanes[k] * n);
#pragma unroll
    for (int j = 0; j < kFormSlots; ++j) {
      v0[j] = *reinterpret_cast<const float*>(p0 + f.offset[j]);
      v1[j] = *reinterpret_cast<const float*>(p1 + f.offset[j]);
    }
  };
  auto store = [&](int k, int slot, const FormIndex& f, const float (&v0)[kFormSlots],
                   const float (&v1)[kFormSlots]) {
    float* stage = &tile[slot][0][0];
    const int lane = tid % 64;
#pragma unroll
    for (int j = 0; j < kFormRows; ++j) {
      stage[(wave * kFormRows + j) * kMaltaLw + lane] =
        f.inside[j] ? MaltaScaledDiff(v0[j], v1[j], ms.m[k]) : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < kFormStrip; ++j) {
      if (f.lds[j] >= 0) {
        stage[f.lds[j]] = f.inside[kFormRows + j]
                            ? MaltaScaledDiff(v0[kFormRows + j], v1[kFormRows + j], ms.m[k])
                            : 0.0f;
      }
    }
  };
  // stages k0, k1, k2 into LDS slots 0, 1, 2
  auto form = [&](int k0, int k1, int k2) {
    FormIndex f;
    index(f);
    float a0[kFormSlots], a1[kFormSlots], b0[kFormSlots], b1[kFormSlots];
    load(k0, f, a0, a1);
    load(k1, f, b0, b1);
    store(k0, 0, f, a0, a1);
    load(k2, f, a0, a1);
    store(k1, 1, f, b0, b1);
    store(k2, 2, f, a0, a1);
  };
  const int q = tid % kMaltaQuads;
  const int x = x0 + 4 * q;
  // a thread past the right edge still takes part in forming the stages
  const bool active = x < w;
  // four consecutive pixels of a plane: one 16-byte access when rows start
  // on 16-byte boundaries (then x + 3 < w), else one access per pixel
  // (32-bit byte offsets from the plane's base: a plane is under 4 GiB)
  const bool vector = (w & 3) == 0;
  auto load4 = [&](const float* plane, size_t i, float (&out)[4]) {
    const char* at = reinterpret_cast<const char*>(plane) + 4u * static_cast<uint32_t>(i);
    if (vector) {
      const float4 v = *reinterpret_cast<const float4*>(at);
      out[0] = v.x;
      out[1] = v.y;
      out[2] = v.z;
      out[3] = v.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        out[j] = x + j < w ? reinterpret_cast<const float*>(at)[j] : 0.0f;
      }
    }
  };
  auto store4 = [&](float* plane, size_t i, const float (&v)[4]) {
    char* at = reinterpret_cast<char*>(plane) + 4u * static_cast<uint32_t>(i);
    if (vector) {
      *reinterpret_cast<float4*>(at) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (x + j < w) reinterpret_cast<float*>(at)[j] = v[j];
      }
    }
  };
  // Malta of stage k (in LDS slot `slot`) for the four outputs of row ty
  auto malta = [&](auto stage, int slot, int ty, float (&out)[4]) {
    constexpr int k = decltype(stage)::value;
    // win[r][c] = tile[slot][ty + r][4q + c]: rows y - 4 .. y + 4, columns
    // x - 4 .. x + 7
    float win[kMaltaWinH][kMaltaWinW];
#pragma unroll
    for (int r = 0; r < kMaltaWinH; ++r) {
      const float4* s4 = reinterpret_cast<const float4*>(&tile[slot][ty + r][4 * q]);
#pragma unroll
      for (int c4 = 0; c4 < kMaltaWinW / 4; ++c4) {
        const float4 v = s4[c4];
        win[r][4 * c4] = v.x;
        win[r][4 * c4 + 1] = v.y;
        win[r][4 * c4 + 2] = v.z;
        win[r][4 * c4 + 3] = v.w;
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      auto P = [&](int dx, int dy) -> float {
        return win[kMaltaHalo + dy][j + kMaltaHalo + dx];
      };
      out[j] = MaltaResponse<(k < 4)>(P);
    }
  };
  form(4, 2, 5);
  __syncthreads();
  if (active) {
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
      const int ty = tid / kMaltaQuads + pass * kMaltaRowsPerPass;
      const int y = y0 + ty;
      if (y >= h) break;
      const size_t base = static_cast<size_t>(y) * w + x;
      float sv[3][4];
      // one Malta window live at a time: the scheduling barriers stand where
      // the stores of the inspected stages keep the windows apart
      malta(std::integral_constant<int, 4>{}, 0, ty, sv[0]);
      if constexpr (kKeepStages) store4(stages + 4 * n, base, sv[0]);
      Settle(sv[0]);
      malta(std::integral_constant<int, 2>{}, 1, ty, sv[1]);
      if constexpr (kKeepStages) store4(stages + 2 * n, base, sv[1]);
      Settle(sv[1]);
      malta(std::integral_constant<int, 5>{}, 2, ty, sv[2]);
      if constexpr (kKeepStages) {
        store4(stages + 5 * n, base, sv[2]);
      } else {
        float acc_y[4], acc_x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc_y[j] = 0.0f;
          acc_y[j] += sv[0][j];
          acc_y[j] += sv[1][j];
          acc_x[j] = 0.0f;
          acc_x[j] += sv[2][j];
        }
        store4(stages, base, acc_y);
        store4(stages + n, base, acc_x);
      }
    }
  }
  __syncthreads();
  form(3, 1, 0);
  __syncthreads();
  if (!active) return;
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    const int ty = tid / kMaltaQuads + pass * kMaltaRowsPerPass;
    const int y = y0 + ty;
    if (y >= h) return;
    const size_t base = static_cast<size_t>(y) * w + x;
    float sv[6][4];
    malta(std::integral_constant<int, 3>{}, 0, ty, sv[3]);
    if constexpr (kKeepStages) store4(stages + 3 * n, base, sv[3]);
    Settle(sv[3]);
    malta(std::integral_constant<int, 1>{}, 1, ty, sv[1]);
    if constexpr (kKeepStages) store4(stages + 1 * n, base, sv[1]);
    Settle(sv[1]);
    malta(std::integral_constant<int, 0>{}, 2, ty, sv[0]);
    if constexpr (kKeepStages) store4(stages, base, sv[0]);
    Settle(sv[0]);
    // the first half's partial sums as this thread stored them (or its
    // stages 4, 2, 5)
    float acc_y[4], acc_x[4];
    if constexpr (kKeepStages) {
      load4(stages + 4 * n, base, sv[4]);
      load4(stages + 2 * n, base, sv[2]);
      load4(stages + 5 * n, base, sv[5]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc_y[j] = 0.0f;
        acc_y[j] += sv[4][j];
        acc_y[j] += sv[2][j];
        acc_x[j] = 0.0f;
        acc_x[j] += sv[5][j];
      }
    } else {
      load4(stages, base, acc_y);
      load4(stages + n, base, acc_x);
    }
    // the per-pixel inputs of the L2 terms and the final map
    float p0[8][4], p1[8][4];  // planes LF 0-2, MF 3-5, HF 6-7
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      load4(ps0 + c * n, base, p0[c]);
      load4(ps1 + c * n, base, p1[c]);
    }
    float rb[4], db[4], my[4], mdc[4];
    load4(ref_blurred, base, rb);
    load4(dist_blurred, base, db);
    load4(mask_y, base, my);
    load4(mask_dc, base, mdc);
    float masked_y[4], final_map[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float a[3], dcv[3];
      // Y: (UHF + HF) + MF; X: (UHF + HF) + MF, from 0 as the reference sums
      a[1] = acc_y[j];
      a[1] += sv[0][j];
      a[0] = acc_x[j];
      a[0] += sv[3][j];
      a[0] += sv[1][j];
      a[2] = 0.0f;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (c < 2 && lw.asym_on[c]) {
          const float v0 = p0[6 + c][j], v1 = p1[6 + c][j];
          const float d = v0 - v1;
          const float total = (d * d) * lw.asym_gt[c] + a[c];
          const float mag = fabsf(v0);
          const float small = 0.4f * mag;
          // v0 < 0:  v1 > -small: v1 + small;  else v1 < -mag: -v1 - mag
          // v0 >= 0: v1 < small:  small - v1;  else v1 > mag:  v1 - mag
          // (else 0), as selects on the same comparisons
          const float below = v0 < 0.0f ? (v1 > -small ? v1 + small : (v1 < -mag ? -v1 - mag : 0.0f))
                                        : 0.0f;
          const float above = v1 < small ? small - v1 : (v1 > mag ? v1 - mag : 0.0f);
          const float sec = v0 < 0.0f ? below : above;
          a[c] = lw.asym_lt[c] * (sec * sec) + total;
        }
        if (lw.mf[c] != 0.0f) {
          const float d = p0[3 + c][j] - p1[3 + c][j];
          a[c] = (d * d) * lw.mf[c] + a[c];
        }
        const float e = p0[c][j] - p1[c][j];
        dcv[c] = lw.lf[c] == 0.0f ? 0.0f : e * e * lw.lf[c];
      }
      const float d = rb[j] - db[j];
      const float ay = a[1] + 10.0f * d * d;
      masked_y[j] = ay;
      const float dc0 = dcv[0] * x_multiplier;
      const float ac0 = a[0] * x_multiplier;
      const float masked_dc = dc0 * mdc[j] + dcv[1] * mdc[j] + dcv[2] * mdc[j];
      const float masked_ac = ac0 * my[j] + ay * my[j] + a[2] * my[j];
      final_map[j] = sqrtf(masked_dc + masked_ac);
    }
    if constexpr (kKeepStages) store4(stages + 7 * n, base, masked_y);
    store4(stages + 8 * n, base, final_map);
  }
}

// StoreMin3 of the reference as selects: the same comparisons decide the
// same moves, also when m0 <= m1 <= m2 does not hold.
__device__ __forceinline__ void StoreMin3(float v, float& m0, float& m1, float& m2) {
  const bool below2 = v < m2, below0 = v < m0, below1 = v < m1;
  // if (v < m2) { if (v < m0) {m2 = m1; m1 = m0; m0 = v;}
  //               else if (v < m1) {m2 = m1; m1 = v;} else {m2 = v;} }
  const float n2 = below0 || below1 ? m1 : v;
  const float n1 = below0 ? m0 : (below1 ? v : m1);
  const float n0 = below0 ? v : m0;
  m2 = below2 ? n2 : m2;
  m1 = below2 ? n1 : m1;
  m0 = below2 ? n0 : m0;
}

// FuzzyErosion of the reference's blurred activity, and MaskY / MaskDcY of
// the result.
struct MaskScale {
  const float* in;
  float* mask;
  float* mask_y;
  float* mask_dc;
  int w, h;
};
struct MaskArgs {
  ScaleBlocks blocks;  // tiles of kThreads pixels of a row
  MaskScale scale[2];
};
__global__ __launch_bounds__(kThreads) void MaskKernel(MaskArgs args) {
  const ScaleTile tile = args.blocks.Tile();
  const MaskScale& sc = args.scale[tile.scale];
  const float* __restrict__ in = sc.in;
  float* __restrict__ mask = sc.mask;
  float* __restrict__ mask_y = sc.mask_y;
  float* __restrict__ mask_dc = sc.mask_dc;
  const int w = sc.w, h = sc.h;
  const int x = tile.x * kThreads + threadIdx.x, y = tile.y;
  if (x >= w) return;
  constexpr int s = 3;
  // every neighbour is read (at clamped positions) before the selection,
  // which then takes the ones inside the image in the reference's order
  const int xl = max(x - s, 0), xr = min(x + s, w - 1);
  const int yu = max(y - s, 0), yd = min(y + s, h - 1);
  auto at = [&](int xx, int yy) { return in[static_cast<size_t>(yy) * w + xx]; };
  const float c0 = at(x, y);
  const float l0 = at(xl, y), lu = at(xl, yu), ld = at(xl, yd);
  const float r0 = at(xr, y), ru = at(xr, yu), rd = at(xr, yd);
  const float u0 = at(x, yu), d0 = at(x, yd);
  const bool left = x >= s, right = x + s < w, up = y >= s, down = y + s < h;
  // a neighbour outside the image is +inf, which no StoreMin3 comparison
  // lets in (v < m2 is false for every m2), as the reference skips it
  constexpr float kSkip = __builtin_inff();
  float m0 = c0;
  float m1 = 2.0f * m0, m2 = m1;
  StoreMin3(left ? l0 : kSkip, m0, m1, m2);
  StoreMin3(left && up ? lu : kSkip, m0, m1, m2);
  StoreMin3(left && down ? ld : kSkip, m0, m1, m2);
  StoreMin3(right ? r0 : kSkip, m0, m1, m2);
  StoreMin3(right && up ? ru : kSkip, m0, m1, m2);
  StoreMin3(right && down ? rd : kSkip, m0, m1, m2);
  StoreMin3(up ? u0 : kSkip, m0, m1, m2);
  StoreMin3(down ? d0 : kSkip, m0, m1, m2);
  const float m = 0.45f * m0 + 0.3f * m1 + 0.25f * m2;
  const size_t i = static_cast<size_t>(y) * w + x;
  mask[i] = m;
  constexpr double kGlobal = 1.0 / (17.83 * 0.79079917404);
  const double vy = kGlobal * (1.0 + 2.5485944793 / (0.451936922203 * m + 0.829591754942));
  const double vd = kGlobal * (1.0 + 0.505054525019 / (3.87449418804 * m + 0.20025578522));
  mask_y[i] = static_cast<float>(vy * vy);
  mask_dc[i] = static_cast<float>(vd * vd);
}

// ---- scales ------------------------------------------------------------------

// ExpandImage for extents below 8: edge-replicated into ew x eh.
__global__ __launch_bounds__(kThreads) void ExpandKernel(
  const float* __restrict__ in, int w, int h, int xb, int yb, int ew, int eh,
  float* __restrict__ out) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  const int c = blockIdx.z;
  if (x >= ew) return;
  int sy = y > yb ? y - yb : 0;
  sy = sy < h - 1 ? sy : h - 1;
  int sx = x > xb ? x - xb : 0;
  sx = sx < w - 1 ? sx : w - 1;
  out[static_cast<size_t>(c) * ew * eh + static_cast<size_t>(y) * ew + x] =
    in[static_cast<size_t>(c) * w * h + static_cast<size_t>(sy) * w + sx];
}

// The requested-extent map: 0.85 main + 0.5 sub (two scales), the main map
// cropped from the expanded extent, or the main map alone; and its maximum
// (non-negative floats compare as their bit patterns), one atomic per group.
__global__ __launch_bounds__(kThreads) void ComposeKernel(
  const float* __restrict__ main_map, int mw, const float* __restrict__ sub_map,
  int sw, int w, int h, int xb, int yb, float* __restrict__ map,
  float* __restrict__ map_out, uint32_t* __restrict__ score_bits) {
  uint32_t best[1] = {0u};
  // rows strided over the groups, columns over the threads (no division)
  for (int y = blockIdx.x; y < h; y += gridDim.x) {
    const float* main_row = main_map + static_cast<size_t>(y + yb) * mw + xb;
    const float* sub_row = sub_map != nullptr ? sub_map + static_cast<size_t>(y / 2) * sw : nullptr;
    const size_t row = static_cast<size_t>(y) * w;
    for (int x = threadIdx.x; x < w; x += blockDim.x) {
      const float m = main_row[x];
      const float v = sub_row != nullptr ? m * 0.85f + 0.5f * sub_row[x / 2] : m;
      map[row + x] = v;
      if (map_out != nullptr) map_out[row + x] = v;
      const uint32_t bits = __float_as_uint(v);
      best[0] = bits > best[0] ? bits : best[0];
    }
  }
  BlockReduceU32(best, U32Max());
  if (threadIdx.x == 0) atomicMax(score_bits, best[0]);
}

// ---- a17 reduction ------------------------------------------------------------

// std::pow(x, 1.0f / 16.0f) as the reference's libm evaluates it.
__device__ __forceinline__ float Root16(float x) { return GlibcPowf(x, 1.0f / 16.0f); }

// One work group per 64x64 tile of the map: the 16th powers of its pixels go
// to LDS, read whole rows at a time, and lane i of the first wave adds up the
// transform anchored at block i in raster order.  Pixels outside the image are
// zeros, which change no non-negative sum.  (With one thread per block and its
// reads along the transform's rows, the ordered adds waited for memory: 37 us
// at 512x512 and 58 at 4032x3024, now 9 and 26.)  A footprint that leaves the
// tile, which the strategy search never makes, is summed from memory.
// The first work group also keeps the comparison's score where `score` says.
constexpr int kReduceTile = 64;
constexpr int kReduceStride = kReduceTile + 4;  // 16-byte rows on shifted banks

__device__ __forceinline__ float Power16(float v) {
  v *= v;
  v *= v;
  v *= v;
  return v * v;
}

__global__ __launch_bounds__(kThreads) void ReduceKernel(
  const float* __restrict__ map, int w, int h, const uint8_t* __restrict__ cells,
  int bw, int bh, float* __restrict__ out, const uint32_t* __restrict__ score,
  uint32_t* __restrict__ score_out) {
  __shared__ __align__(16) float tile[kReduceTile][kReduceStride];
  if (score != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    *score_out = *score;
  }
  const int tx0 = blockIdx.x * kReduceTile, ty0 = blockIdx.y * kReduceTile;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  constexpr int kRows = kReduceTile / (kThreads / 64);
  float v[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const int y = ty0 + wave * kRows + r, x = tx0 + lane;
    v[r] = map[static_cast<size_t>(min(y, h - 1)) * w + min(x, w - 1)];
  }
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const int y = ty0 + wave * kRows + r;
    tile[wave * kRows + r][lane] = y < h && tx0 + lane < w ? Power16(v[r]) : 0.0f;
  }
  __syncthreads();
  if (wave != 0) return;
  const int lx = lane % 8, ly = lane / 8;
  const int bx = tx0 / 8 + lx, by = ty0 / 8 + ly;
  if (bx >= bw || by >= bh) return;
  const uint8_t c = cells[static_cast<size_t>(by) * bw + bx];
  if (!(c & 1)) return;
  const int cw = CoveredW(c >> 1), ch = CoveredH(c >> 1);
  // a footprint past the grid is not a valid transform: nothing is written
  if (bx + cw > bw || by + ch > bh) return;
  const int x0 = bx * 8, y0 = by * 8;
  const int x1 = min(w, x0 + cw * 8), y1 = min(h, y0 + ch * 8);
  const int count = (x1 - x0) * max(y1 - y0, 0);
  if (count <= 0) return;
  float norm = 0.0f;
  if (lx + cw <= 8 && ly + ch <= 8) {
    // 32 pixels at a time (four runs of eight along the rows; every transform
    // holds whole 64s), read one step ahead of their adds: the adds of a step
    // take as long as the reads of the next
    constexpr int kRuns = 4;
    const int shift = cw == 1 ? 0 : cw == 2 ? 1 : 2;
    const int steps = cw * ch * 8 / kRuns;
    auto read = [&](int step, float4 (&v)[2 * kRuns]) {
#pragma unroll
      for (int j = 0; j < kRuns; ++j) {
        const int run = step * kRuns + j;
        const float4* p = reinterpret_cast<const float4*>(
          &tile[8 * ly + (run >> shift)][8 * (lx + (run & (cw - 1)))]);
        v[2 * j] = p[0];
        v[2 * j + 1] = p[1];
      }
    };
    float4 next[2 * kRuns];
    read(0, next);
    for (int step = 0; step < steps; ++step) {
      float4 v[2 * kRuns];
#pragma unroll
      for (int j = 0; j < 2 * kRuns; ++j) v[j] = next[j];
      read(min(step + 1, steps - 1), next);
#pragma unroll
      for (int j = 0; j < 2 * kRuns; ++j) {
        norm = norm + v[j].x;
        norm = norm + v[j].y;
        norm = norm + v[j].z;
        norm = norm + v[j].w;
      }
    }
  } else {
    for (int y = y0; y < y1; ++y)
      for (int x = x0; x < x1; ++x) norm = norm + Power16(map[static_cast<size_t>(y) * w + x]);
  }
  const float d = 1.2f * Root16(norm / static_cast<float>(count));
  for (int dy = 0; dy < ch; ++dy)
    for (int dx = 0; dx < cw; ++dx) out[static_cast<size_t>(by + dy) * bw + bx + dx] = d;
}

// ---- host side -------------------------------------------------------------------

Taps HostTaps(float sigma) {
  Taps out{};
  const float scaled = 2.25f * std::fabs(sigma);
  int radius = static_cast<int>(scaled);
  radius = radius < 1 ? 1 : radius;
  const int size = 2 * radius + 1;
  // the host libm's exp, as the reference evaluates it; volatile keeps the
  // compiler from folding it
  volatile double exponent_scale = -1.0 / (2.0 * sigma * sigma);
  for (int i = -radius; i <= radius; ++i) {
    out.k[i + radius] = static_cast<float>(std::exp(exponent_scale * i * i));
  }
  float full = 0.0f;
  for (int i = 0; i < size; ++i) full += out.k[i];
  const float scale = 1.0f / full;
  for (int i = 0; i <= radius; ++i) out.sk[i] = out.k[i] * scale;
  return out;
}

inline dim3 Grid2(int w, int h, int z = 1) {
  return dim3(CeilDiv(static_cast<uint32_t>(w), kThreads), h, z);
}

const Taps& TapsOf(ButteraugliSigma s) {
  static const struct Table {
    Taps taps[kSigmaCount];
    Table() {
      for (int k = 0; k < kSigmaCount; ++k) taps[k] = HostTaps(kSigmas[k]);
    }
  } table;
  return table.taps[s];
}

int Scales(const GJXLAmdButteraugli* b) { return b->has_subscale ? 2 : 1; }

ScaleBlocks Blocks(const GJXLAmdButteraugli* b, uint32_t tile_w, uint32_t tile_h,
                   unsigned units = 1) {
  ScaleBlocks r;
  r.units = units;
  for (int k = 0; k < Scales(b); ++k) {
    r.tiles_w[k] = CeilDiv(static_cast<uint32_t>(b->scale[k].width), tile_w);
    r.count[k] = r.tiles_w[k] * CeilDiv(static_cast<uint32_t>(b->scale[k].height), tile_h) * units;
  }
  return r;
}

// The grid of a blur of radius R.  A segment of n bands filters n + kGroups - 1
// of them by rows and n by columns, so tall segments filter fewer halo rows;
// but the work groups of a CU end one after another (the oldest is served
// first) and the last one runs alone, so there must be enough of them:
// 4-band segments once the image leaves kWorkGroups of those, shorter ones
// below.  Where even single bands leave CUs idle the planes are split over two
// work groups (`split`).  Measured, radius 16, us with 1 / 2 / 3 / 4 bands:
// 1537x1153 75 / 70 / 66 / 76, 4032x3024 319 / 260 / 252 / 230; one and two
// units at 77x45 32 and 23, at 512x512 33 and 32, at 1537x1153 75 and 80.
template <int R>
BlurArgs BlurGrid(const GJXLAmdButteraugli* b, ButteraugliSigma sigma, bool split) {
  constexpr uint32_t kWorkGroups = BlurShape<R>::kGroups > 2 ? 400 : 700;
  uint32_t bands = 0;
  for (int k = 0; k < Scales(b); ++k) {
    bands += CeilDiv(static_cast<uint32_t>(b->scale[k].width), kStripW) *
             CeilDiv(static_cast<uint32_t>(b->scale[k].height), kBandH);
  }
  const uint32_t per = std::min(4u, std::max(1u, (bands + kWorkGroups / 2) / kWorkGroups));
  BlurArgs a{};
  a.rows = static_cast<int>(per * kBandH);
  a.blocks = Blocks(b, kStripW, per * kBandH, split && bands <= 256 ? 2 : 1);
  a.taps = TapsOf(sigma);
  return a;
}

float* PsychoPlanes(const ButteraugliScale& s, bool reference) {
  return reference ? s.ref_psycho : s.dist_psycho;
}
// Scratch of one pass over an image, in planes that hold nothing then: the
// raw MF planes, the raw HF planes and the masking activity (the half
// scale's image is never stored, the full scale's only when it is expanded,
// and then the opsin kernel has consumed it).
float* RawMf(const ButteraugliScale& s) { return s.tmp[0]; }
float* RawHf(const ButteraugliScale& s) { return s.input; }
float* Activity(const ButteraugliScale& s) { return s.input + 2 * s.n; }
// The compared image's blurred activity (after the raw MF planes).
float* DistortedBlurred(const ButteraugliScale& s) { return s.tmp[2]; }

// Opsin dynamics and frequency separation of `in` at both scales into the
// reference's or the compared image's psycho planes, and their masking
// activity.
GJXLResult Psycho(GJXLAmdButteraugli* b, const float* in, bool reference) {
  hipStream_t st = b->device->stream;
  OpsinArgs o{};
  o.blocks = Blocks(b, kOpsinTileW, kOpsinTileH);
  o.rgb = in;
  for (int k = 0; k < Scales(b); ++k) {
    o.w[k] = b->scale[k].width;
    o.h[k] = b->scale[k].height;
    o.xyb[k] = b->scale[k].xyb;
  }
  o.intensity = b->params.intensity_target;
  o.taps = TapsOf(kSigmaOpsin);
  o.score = reference ? nullptr : b->score_bits;
  hipLaunchKernelGGL(OpsinDynamicsKernel, o.blocks.Grid(), dim3(kThreads), 0, st, o);
  GJXL_AMD_TRY(CheckLaunch("OpsinDynamicsKernel"));
  auto scales = [&](BlurArgs& a, auto in_of, auto scratch_of) {
    for (int k = 0; k < Scales(b); ++k) {
      const ButteraugliScale& s = b->scale[k];
      a.scale[k] = BlurScale{in_of(s), PsychoPlanes(s, reference), scratch_of(s), s.width,
                             s.height, s.n};
    }
  };
  BlurArgs low = BlurGrid<16>(b, kSigmaLow, true);
  scales(low, [](const ButteraugliScale& s) { return s.xyb; }, RawMf);
  hipLaunchKernelGGL((BlurKernel<16, kBlurThreads, LowPlanes, 3>), low.blocks.Grid(), dim3(kBlurThreads), 0, st, low);
  GJXL_AMD_TRY(CheckLaunch("LowBlurKernel"));
  BlurArgs high = BlurGrid<7>(b, kSigmaHigh, true);
  scales(high, RawMf, RawHf);
  hipLaunchKernelGGL((BlurKernel<7, kBlurThreads, HighPlanes, 3>), high.blocks.Grid(), dim3(kBlurThreads), 0, st, high);
  GJXL_AMD_TRY(CheckLaunch("HighBlurKernel"));
  BlurArgs ultra = BlurGrid<3>(b, kSigmaUltra, false);
  scales(ultra, RawHf, Activity);
  hipLaunchKernelGGL((BlurKernel<3, kBlurThreads, UltraPlanes, 2>), ultra.blocks.Grid(), dim3(kBlurThreads), 0, st, ultra);
  return CheckLaunch("UltraBlurKernel");
}

// The blurred masking activity of the image that Psycho has just separated.
GJXLResult MaskActivity(GJXLAmdButteraugli* b, bool reference) {
  BlurArgs a = BlurGrid<6>(b, kSigmaMask, false);
  for (int k = 0; k < Scales(b); ++k) {
    const ButteraugliScale& s = b->scale[k];
    a.scale[k] = BlurScale{Activity(s), nullptr, reference ? s.ref_blurred : DistortedBlurred(s),
                           s.width, s.height, s.n};
  }
  hipLaunchKernelGGL((BlurKernel<6, kBlurThreads, MaskPlanes, 1>), a.blocks.Grid(), dim3(kBlurThreads), 0, b->device->stream, a);
  return CheckLaunch("MaskBlurKernel");
}

constexpr double kMaltaWeights[6] = {37.0819870399, 8246.75321353, 18.7237414387,
                                     6923.99476109, 1.10039032555, 173.5};
constexpr double kMaltaNorms[6] = {130262059.556, 1009002.70582, 4498534.45232,
                                   8051.15833247, 71.7800275169, 5.0};
constexpr float kL2[9] = {400.0f, 1.50815703118f, 0.0f, 2150.0f, 10.6195433239f,
                          16.2176043152f, 29.2353797994f, 0.844626970982f,
                          0.703646627719f};

GJXLResult Differences(GJXLAmdButteraugli* b, bool keep_stages) {
  hipStream_t st = b->device->stream;
  const float asym = b->params.hf_asymmetry;
  const float sqrt_asym = std::sqrt(asym);
  const double up[6] = {kMaltaWeights[0], kMaltaWeights[1], kMaltaWeights[2] * sqrt_asym,
                        kMaltaWeights[3] * sqrt_asym, kMaltaWeights[4] * asym,
                        kMaltaWeights[5] * asym};
  const double down[6] = {kMaltaWeights[0], kMaltaWeights[1], kMaltaWeights[2] / sqrt_asym,
                          kMaltaWeights[3] / sqrt_asym, kMaltaWeights[4] / asym,
                          kMaltaWeights[5] / asym};
  MaltaScales ms;
  for (int k = 0; k < 6; ++k) {
    const bool lf = k < 4;
    const double multiplier = lf ? 0.611612573796 : 0.39905817637;
    const double pre_gt = multiplier * std::sqrt(0.5f * up[k]) / (3.75 * 2.0 + 1.0);
    const double pre_lt = multiplier * std::sqrt(0.33f * down[k]) / (3.75 * 2.0 + 1.0);
    ms.m[k] = MaltaScale{static_cast<float>(pre_gt * kMaltaNorms[k]),
                         static_cast<float>(pre_lt * kMaltaNorms[k]),
                         static_cast<float>(kMaltaNorms[k])};  // gt, lt: binary32 values
  }
  L2Weights lw{};
  for (int c = 0; c < 2; ++c) {
    const float gt = kL2[c] * asym, lt = kL2[c] / asym;
    lw.asym_on[c] = !(gt == 0.0f && lt == 0.0f);
    lw.asym_gt[c] = gt * 0.8f;
    lw.asym_lt[c] = lt * 0.8f;
  }
  for (int c = 0; c < 3; ++c) {
    lw.mf[c] = kL2[3 + c];
    lw.lf[c] = kL2[6 + c];
  }
  DifferencesArgs args{};
  args.blocks = Blocks(b, kMaltaTileW, kMaltaTileH);
  for (int k = 0; k < Scales(b); ++k) {
    const ButteraugliScale& s = b->scale[k];
    args.scale[k] = DifferencesScale{s.ref_psycho, s.dist_psycho, s.ref_blurred,
                                     DistortedBlurred(s), s.mask_y, s.mask_dc, s.stages,
                                     s.width, s.height};
  }
  args.ms = ms;
  args.lw = lw;
  args.x_multiplier = b->params.x_multiplier;
  const bool probed = ProbeBegin(b->device, GJXL_AMD_KERNEL_BUTTERAUGLI_DIFFERENCES);
  if (keep_stages) {
    hipLaunchKernelGGL(DifferencesKernel<true>, args.blocks.Grid(), dim3(kThreads), 0, st, args);
  } else {
    hipLaunchKernelGGL(DifferencesKernel<false>, args.blocks.Grid(), dim3(kThreads), 0, st, args);
  }
  ProbeEnd(b->device, probed);
  return CheckLaunch("DifferencesKernel");
}

constexpr int kScalePlanes = 3 + 3 + 10 + 10 + 3 + 9 + 3;

}  // namespace

GJXLResult ButteraugliCompare(GJXLAmdButteraugli* b, const float* distorted,
                              float* map_out, bool keep_stages) {
  hipStream_t st = b->device->stream;
  // the difference kernel addresses a plane with 32-bit byte offsets
  if (static_cast<uint64_t>(b->scale[0].width) * b->scale[0].height >= (uint64_t{1} << 30)) {
    return Fail(GJXL_ERROR_UNSUPPORTED, "Butteraugli differences: plane of 2^30 or more pixels");
  }
  ButteraugliScale& m = b->scale[0];
  const float* main_in = distorted;
  if (b->expanded) {
    hipLaunchKernelGGL(ExpandKernel, Grid2(m.width, m.height, 3), dim3(kThreads), 0, st,
                       distorted, b->width, b->height, b->xborder, b->yborder, m.width,
                       m.height, m.input);
    GJXL_AMD_TRY(CheckLaunch("ExpandKernel"));
    main_in = m.input;
  }
  GJXL_AMD_TRY(Psycho(b, main_in, false));
  GJXL_AMD_TRY(MaskActivity(b, false));
  GJXL_AMD_TRY(Differences(b, keep_stages));
  const float* sub_map = nullptr;
  int sw = 0;
  if (b->has_subscale) {
    sub_map = b->scale[1].stages + 8 * b->scale[1].n;
    sw = b->scale[1].width;
  }
  hipLaunchKernelGGL(ComposeKernel,
                     dim3(ReductionGroups(static_cast<size_t>(b->width) * b->height)),
                     dim3(kThreads), 0, st,
                     m.stages + 8 * m.n, m.width, sub_map, sw, b->width, b->height,
                     b->xborder, b->yborder, b->map, map_out, b->score_bits);
  return CheckLaunch("ComposeKernel");
}

GJXLResult LaunchReduceDistanceMap(hipStream_t s, const float* map, int width,
                                   int height, const uint8_t* cells, int bw,
                                   int bh, float* out, const uint32_t* score,
                                   uint32_t* score_out) {
  hipLaunchKernelGGL(ReduceKernel,
                     dim3(CeilDiv(static_cast<uint32_t>(bw), kReduceTile / 8),
                          CeilDiv(static_cast<uint32_t>(bh), kReduceTile / 8)),
                     dim3(kThreads), 0, s, map, width, height, cells, bw, bh, out, score,
                     score_out);
  return CheckLaunch("ReduceKernel");
}

size_t ButteraugliGeometry(GJXLAmdButteraugli* b, uint32_t width, uint32_t height) {
  b->width = static_cast<int>(width);
  b->height = static_cast<int>(height);
  b->expanded = width < 8 || height < 8;
  b->has_subscale = !b->expanded && width >= 15 && height >= 15;
  b->xborder = width < 8 ? (8 - static_cast<int>(width)) / 2 : 0;
  b->yborder = height < 8 ? (8 - static_cast<int>(height)) / 2 : 0;
  const int mw = width < 8 ? 8 : static_cast<int>(width);
  const int mh = height < 8 ? 8 : static_cast<int>(height);
  b->scale[0].width = mw;
  b->scale[0].height = mh;
  b->scale[1].width = (static_cast<int>(width) + 1) / 2;
  b->scale[1].height = (static_cast<int>(height) + 1) / 2;
  size_t floats = static_cast<size_t>(width) * height + 64;
  const int scales = b->has_subscale ? 2 : 1;
  for (int k = 0; k < scales; ++k) {
    auto& s = b->scale[k];
    s.n = static_cast<size_t>(s.width) * s.height;
    floats += kScalePlanes * s.n;
  }
  return floats;
}

void CarveButteraugli(GJXLAmdButteraugli* b) {
  float* p = static_cast<float*>(b->allocation);
  b->score_bits = reinterpret_cast<uint32_t*>(p);
  p += 64;
  b->map = p;
  p += static_cast<size_t>(b->width) * b->height;
  const int scales = b->has_subscale ? 2 : 1;
  for (int k = 0; k < scales; ++k) {
    auto& s = b->scale[k];
    const size_t n = s.n;
    s.input = p; p += 3 * n;
    s.xyb = p; p += 3 * n;
    s.ref_psycho = p; p += 10 * n;
    s.dist_psycho = p; p += 10 * n;
    s.ref_blurred = p; p += n;
    s.mask_y = p; p += n;
    s.mask_dc = p; p += n;
    s.stages = p; p += 9 * n;
    for (auto& t : s.tmp) { t = p; p += n; }
  }
}

GJXLResult ResizeButteraugli(GJXLAmdButteraugli* b, uint32_t width, uint32_t height) {
  if (width == 0 || height == 0 || width > 65535 || height > 65535) {
    return Fail(GJXL_ERROR_INVALID_ARGUMENT, "Butteraugli geometry is invalid");
  }
  GJXLAmdButteraugli probe;
  if (ButteraugliGeometry(&probe, width, height) > b->capacity_floats) {
    return Fail(GJXL_ERROR_INVALID_ARGUMENT, "extent exceeds the Butteraugli capacity");
  }
  (void)ButteraugliGeometry(b, width, height);
  CarveButteraugli(b);
  b->prepared = false;
  return GJXL_OK;
}

}  // namespace gjxl_amd

using gjxl_amd::Check;
using gjxl_amd::Fail;

extern "C" {

GJXLResult gjxl_amd_butteraugli_create(GJXLAmdDevice* device, uint32_t width,
                                       uint32_t height, float hf_asymmetry,
                                       float x_multiplier, float intensity_target,
                                       GJXLAmdButteraugli** out) {
  GJXL_AMD_TRY(gjxl_amd::ValidateDevice(device));
  if (out == nullptr || *out != nullptr || width == 0 || height == 0 ||
      width > 65535 || height > 65535 || !std::isfinite(hf_asymmetry) ||
      hf_asymmetry <= 0.0f || !std::isfinite(x_multiplier) || x_multiplier <= 0.0f ||
      !std::isfinite(intensity_target) || intensity_target <= 0.0f) {
    return Fail(GJXL_ERROR_INVALID_ARGUMENT, "Butteraugli geometry or options are invalid");
  }
  auto* b = new (std::nothrow) GJXLAmdButteraugli;
  if (b == nullptr) return Fail(GJXL_ERROR_OUT_OF_MEMORY, "Butteraugli allocation failed");
  b->device = device;
  b->params = {hf_asymmetry, x_multiplier, intensity_target};
  const size_t floats = gjxl_amd::ButteraugliGeometry(b, width, height);
  GJXLResult r = Check(hipSetDevice(device->ordinal), "hipSetDevice");
  if (r == GJXL_OK) r = gjxl_amd::DeviceAlloc(device, floats * sizeof(float), &b->allocation);
  if (r != GJXL_OK) {
    delete b;
    return r;
  }
  b->capacity_floats = floats;
  gjxl_amd::CarveButteraugli(b);
  *out = b;
  return GJXL_OK;
}

void gjxl_amd_butteraugli_destroy(GJXLAmdButteraugli* b) {
  if (b == nullptr) return;
  if (b->device != nullptr) {
    (void)hipSetDevice(b->device->ordinal);
    (void)hipStreamSynchronize(b->device->stream);
  }
  if (b->device != nullptr) gjxl_amd::DeviceFree(b->device, b->allocation);
  delete b;
}

GJXLResult gjxl_amd_butteraugli_prepare(GJXLAmdButteraugli* b,
                                        const float* reference_linear) {
  if (b == nullptr || reference_linear == nullptr) {
    return Fail(GJXL_ERROR_INVALID_ARGUMENT, "Butteraugli prepare arguments are null");
  }
  GJXL_AMD_TRY(gjxl_amd::ValidateDevice(b->device));
  using namespace gjxl_amd;
  b->prepared = false;
  hipStream_t st = b->device->stream;
  ButteraugliScale& m = b->scale[0];
  const float* in = reference_linear;
  if (b->expanded) {
    hipLaunchKernelGGL(ExpandKernel, Grid2(m.width, m.height, 3), dim3(kThreads), 0, st,
                       reference_linear, b->width, b->height, b->xborder, b->yborder, m.width,
                       m.height, m.input);
    GJXL_AMD_TRY(CheckLaunch("ExpandKernel"));
    in = m.input;
  }
  GJXL_AMD_TRY(Psycho(b, in, true));
  GJXL_AMD_TRY(MaskActivity(b, true));
  MaskArgs args{};
  args.blocks = Blocks(b, kThreads, 1);
  for (int k = 0; k < Scales(b); ++k) {
    const ButteraugliScale& s = b->scale[k];
    args.scale[k] = MaskScale{s.ref_blurred, s.stages + 6 * s.n, s.mask_y, s.mask_dc, s.width,
                              s.height};
  }
  hipLaunchKernelGGL(MaskKernel, args.blocks.Grid(), dim3(kThreads), 0, st, args);
  GJXL_AMD_TRY(CheckLaunch("MaskKernel"));
  b->prepared = true;
  return GJXL_OK;
}

GJXLResult gjxl_amd_butteraugli_compare(GJXLAmdButteraugli* b,
                                        const float* distorted_linear,
                                        float* distance_map) {
  if (b == nullptr || distorted_linear == nullptr) {
    return Fail(GJXL_ERROR_INVALID_ARGUMENT, "Butteraugli compare arguments are null");
  }
  GJXL_AMD_TRY(gjxl_amd::ValidateDevice(b->device));
  if (!b->prepared) {
    return Fail(GJXL_ERROR_INVALID_ARGUMENT, "Butteraugli reference has not been prepared");
  }
  return gjxl_amd::ButteraugliCompare(b, distorted_linear, distance_map, true);
}

GJXLResult gjxl_amd_butteraugli_score(GJXLAmdButteraugli* b, double* score) {
  if (b == nullptr || score == nullptr) {
    return Fail(GJXL_ERROR_INVALID_ARGUMENT, "Butteraugli score arguments are null");
  }
  GJXL_AMD_TRY(gjxl_amd::ValidateDevice(b->device));
  uint32_t bits = 0;
  GJXL_AMD_TRY(Check(hipMemcpyAsync(&bits, b->score_bits, 4, hipMemcpyDeviceToHost,
                                    b->device->stream), "hipMemcpyAsync(score)"));
  GJXL_AMD_TRY(Check(hipStreamSynchronize(b->device->stream), "hipStreamSynchronize"));
  float v;
  std::memcpy(&v, &bits, 4);
  *score = v;
  return GJXL_OK;
}

GJXLResult gjxl_amd_butteraugli_buffer(GJXLAmdButteraugli* b, int32_t scale,
                                       int32_t id, void** pointer, size_t* bytes) {
  if (b == nullptr || pointer == nullptr || scale < 0 || scale > 1 ||
      (scale == 1 && !b->has_subscale)) {
    return Fail(GJXL_ERROR_INVALID_ARGUMENT, "Butteraugli buffer request is invalid");
  }
  const gjxl_amd::ButteraugliScale& s = b->scale[scale];
  const size_t plane = s.n * sizeof(float);
  void* p = nullptr;
  size_t z = 0;
  switch (id) {
    case GJXL_AMD_BUTTERAUGLI_MAP: p = b->map; z = sizeof(float) * b->width * b->height; break;
    case GJXL_AMD_BUTTERAUGLI_REFERENCE_PSYCHO: p = s.ref_psycho; z = 10 * plane; break;
    case GJXL_AMD_BUTTERAUGLI_DISTORTED_PSYCHO: p = s.dist_psycho; z = 10 * plane; break;
    case GJXL_AMD_BUTTERAUGLI_STAGES: p = s.stages; z = 9 * plane; break;
    case GJXL_AMD_BUTTERAUGLI_XYB: p = s.xyb; z = 3 * plane; break;
    case GJXL_AMD_BUTTERAUGLI_SCORE: p = b->score_bits; z = 4; break;
    default: return Fail(GJXL_ERROR_INVALID_ARGUMENT, "Butteraugli buffer id is invalid");
  }
  *pointer = p;
  if (bytes) *bytes = z;
  return GJXL_OK;
}

GJXLResult gjxl_amd_reduce_distance_map(GJXLAmdDevice* device, const float* map,
                                        uint32_t width, uint32_t height,
                                        const uint8_t* cells, float* block_distance) {
  GJXL_AMD_TRY(gjxl_amd::ValidateDevice(device));
  if (map == nullptr || cells == nullptr || block_distance == nullptr || width == 0 ||
      height == 0) {
    return Fail(GJXL_ERROR_INVALID_ARGUMENT, "Distance-map reduction arguments are invalid");
  }
  const int bw = static_cast<int>(gjxl_amd::CeilDiv(width, 8));
  const int bh = static_cast<int>(gjxl_amd::CeilDiv(height, 8));
  return gjxl_amd::LaunchReduceDistanceMap(device->stream, map, width, height, cells, bw,
                                           bh, block_distance);
}

}  // extern "C"
