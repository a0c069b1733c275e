// Image preprocessing of the data path on gfx950: decoded uint8 RGB images ->
// the encoder's normalised float32 planes, bit-identical to the reference's
// evaluation transform (models/backbone/open_clip/transform.py:118-133: Resize((S,
// S), BICUBIC) on a PIL image, CenterCrop, ToTensor, Normalize), which torchvision
// runs per image on the CPU inside the dataset item (datasets/mvtec.py:101-103).
//
// The resize is Pillow's 8-bit resampling (Pillow pinned at 11.1.0 by the
// reference, requirements.txt:13): per axis a table of 22-bit fixed-point bicubic
// coefficients (a = -0.5, support 2 stretched by max(in/out, 1)), then a horizontal
// pass over the source rows the vertical pass reads, rounding to uint8, then a
// vertical pass rounding to uint8 again; an axis that keeps its size is not
// resampled.  The coefficient tables are computed on the device with the same IEEE
// double operations in the same order as Pillow's C code (FP contraction off, so no
// fused multiply-add changes a rounding), which makes the fixed-point tables, and
// hence the integer passes, identical.  ToTensor (u8 / 255) and Normalize ((x -
// mean) / std) are fused into the vertical pass as correctly rounded float32
// division and subtraction, the operations torch performs on the CPU.
#include <type_traits>

#include "common.hpp"

namespace musc {
namespace prep {

constexpr int kPrecisionBits = 22;
constexpr int kMaxTaps = 64;     // taps = 2*ceil(2*max(in/out, 1)) + 1, so in/out <= 15.5
constexpr int kThreads = 256;

struct Norm {
  float mean[3];
  float stdv[3];
};

// FP contraction is off in the coefficient code: a fused multiply-add would round
// differently from Pillow's separate multiply and add.
__host__ __device__ inline double bicubic(double x) {
#pragma clang fp contract(off)
  const double a = -0.5;
  if (x < 0.0) x = -x;
  if (x < 1.0) return ((a + 2.0) * x - (a + 3.0)) * x * x + 1;
  if (x < 2.0) return (((x - 5) * x + 8) * x - 4) * a;
  return 0.0;
}

struct AxisGeom {
  double scale, support, ss;
  int taps;
};

__host__ __device__ inline AxisGeom axis_geom(int in_size, int out_size) {
#pragma clang fp contract(off)
  AxisGeom g;
  g.scale = (double)in_size / out_size;
  const double filterscale = g.scale < 1.0 ? 1.0 : g.scale;
  g.support = 2.0 * filterscale;
  g.ss = 1.0 / filterscale;
  g.taps = (int)ceil(g.support) * 2 + 1;
  return g;
}

// Source window [xmin, xmin + count) of output index xx and its center.
__host__ __device__ inline int2 window(const AxisGeom& g, int in_size, int xx, double* center_out) {
#pragma clang fp contract(off)
  const double center = 0.0 + (xx + 0.5) * g.scale;
  int xmin = (int)(center - g.support + 0.5);
  if (xmin < 0) xmin = 0;
  int xmax = (int)(center + g.support + 0.5);
  if (xmax > in_size) xmax = in_size;
  if (center_out) *center_out = center;
  return make_int2(xmin, xmax - xmin);
}

// One axis of the coefficient launch.  identity: the axis keeps its size and is not
// resampled (window {xx, 1}, coefficient 1.0, which reproduces the byte exactly).
struct AxisTable {
  AxisGeom g;
  int in_size, out_size, shift, identity;
  int2* bounds;
  int* kk;
};

// Both axes' tables in one launch (3.3 us at 1024 -> 518), kLanes lanes per output index: bounds (xmin - shift,
// count) and a row of `width` <= kLanes fixed-point coefficients (zero past the window).
// Bound by latency: a lane forms one bicubic value and one quotient where a thread per
// output index formed all of them one after the other.  The sum over the window stays in
// Pillow's order (each lane adds the group's values in turn), so its rounding does too.
template <int kLanes>
__global__ __launch_bounds__(kThreads) void coeff_kernel(AxisTable h, AxisTable v, int width) {
#pragma clang fp contract(off)
  const int unit = (blockIdx.x * kThreads + threadIdx.x) / kLanes, x = threadIdx.x % kLanes;
  if (unit >= h.out_size + v.out_size) return;
  const bool second = unit >= h.out_size;
  const int xx = second ? unit - h.out_size : unit;
  const AxisTable t = second ? v : h;
  int2 w = make_int2(xx, 1);
  int q = x == 0 ? 1 << kPrecisionBits : 0;
  if (!t.identity) {
    double center;
    w = window(t.g, t.in_size, xx, &center);
    double k = x < w.y ? bicubic((x + w.x - center + 0.5) * t.g.ss) : 0.0;
    double ww = 0.0;
    for (int i = 0; i < w.y; ++i) ww += __shfl(k, i, kLanes);
    if (ww != 0.0) k /= ww;
    q = k < 0 ? (int)(-0.5 + k * (1 << kPrecisionBits)) : (int)(0.5 + k * (1 << kPrecisionBits));
    if (x >= w.y) q = 0;
  }
  if (x < width) t.kk[(long long)xx * width + x] = q;
  if (x == 0) t.bounds[xx] = make_int2(w.x - t.shift, w.y);
}

__device__ inline int clip8(int acc) {
  if (acc >= (1 << kPrecisionBits << 8)) return 255;
  if (acc <= 0) return 0;
  return acc >> kPrecisionBits;
}

// Coefficient rows are kW ints wide (kW a multiple of 4, zero past the window), so
// a thread fetches its whole row with kW/4 independent 16-byte loads and the tap
// loops have a compile-time trip count: every load of a pixel is in flight at once.
// Taps past the window carry weight 0; their source index is clamped into the image.
template <int kW>
__device__ inline void load_coeffs(const int* __restrict__ k, int (&c)[kW]) {
  const int4* k4 = reinterpret_cast<const int4*>(k);
#pragma unroll
  for (int i = 0; i < kW / 4; ++i) {
    const int4 v = k4[i];
    c[4 * i + 0] = v.x;
    c[4 * i + 1] = v.y;
    c[4 * i + 2] = v.z;
    c[4 * i + 3] = v.w;
  }
}

// 22-bit fixed-point sums of kW taps of interleaved RGB bytes: tap x reads
// base + min(first + x, last) * stride.
template <int kW>
__device__ inline int3 tap_sums(const uint8_t* __restrict__ base, int first, int last, long long stride,
                                const int (&c)[kW]) {
  int s0 = 1 << (kPrecisionBits - 1), s1 = s0, s2 = s0;
#pragma unroll
  for (int x = 0; x < kW; ++x) {
    const int i = first + x < last ? first + x : last;
    const uint8_t* q = base + i * stride;
    s0 += (int)q[0] * c[x];
    s1 += (int)q[1] * c[x];
    s2 += (int)q[2] * c[x];
  }
  return make_int3(s0, s1, s2);
}

__device__ inline void store_normalised(float* __restrict__ o, long long plane, int3 s, const Norm& nrm) {
  const int u[3] = {clip8(s.x), clip8(s.y), clip8(s.z)};
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float t = (float)u[c] / 255.0f;
    o[c * plane] = (t - nrm.mean[c]) / nrm.stdv[c];
  }
}

// Horizontal pass: tmp (batch, rows, out_w, 3) uint8 from source rows row0 .. row0+rows-1.
template <int kW>
__global__ __launch_bounds__(kThreads) void hpass_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ tmp,
                                                         int in_h, int in_w, int row0, int rows, int out_w,
                                                         const int2* __restrict__ bounds, const int* __restrict__ kk) {
  const int xx = blockIdx.x * kThreads + threadIdx.x;
  if (xx >= out_w) return;
  const int r = blockIdx.y, b = blockIdx.z;
  const uint8_t* row = src + (((long long)b * in_h + row0 + r) * in_w) * 3;
  const int2 bd = bounds[xx];
  int c[kW];
  load_coeffs<kW>(kk + (long long)xx * kW, c);
  const int3 s = tap_sums<kW>(row, bd.x, in_w - 1, 3, c);
  uint8_t* o = tmp + (((long long)b * rows + r) * out_w + xx) * 3;
  o[0] = (uint8_t)clip8(s.x);
  o[1] = (uint8_t)clip8(s.y);
  o[2] = (uint8_t)clip8(s.z);
}

// Vertical pass + ToTensor + Normalize: out (batch, 3, out_h, w) float32 from an
// interleaved uint8 (batch, rows, w, 3) image (the horizontal pass's output, or the
// source when the width is kept).
template <int kW>
__global__ __launch_bounds__(kThreads) void vpass_kernel(const uint8_t* __restrict__ img, int rows, int w, int out_h,
                                                         const int2* __restrict__ bounds, const int* __restrict__ kk,
                                                         Norm nrm, float* __restrict__ out) {
  const int xx = blockIdx.x * kThreads + threadIdx.x;
  if (xx >= w) return;
  const int yy = blockIdx.y, b = blockIdx.z;
  const int2 bd = bounds[yy];
  int c[kW];
  load_coeffs<kW>(kk + (long long)yy * kW, c);
  const int3 s = tap_sums<kW>(img + ((long long)b * rows * w + xx) * 3, bd.x, rows - 1, (long long)w * 3, c);
  const long long plane = (long long)out_h * w;
  store_normalised(out + (long long)b * 3 * plane + (long long)yy * w + xx, plane, s, nrm);
}

// Fused resize: one workgroup per (image, band of output rows, up to 64 output columns).
// The source rectangle under the tile's windows goes into LDS as aligned 4-byte words, all
// its loads in flight at once; a wave then resamples one source row at a time (a lane owns
// one output column and keeps its coefficients in registers) into an LDS block of one word
// (R | G << 8 | B << 16) per pixel, and the vertical pass walks the output rows of the tile
// the same way (coefficients uniform in the wave).  (u / 255 - mean) / std has 256 values
// per channel: a table in LDS, formed with the same two divisions.  Two barriers in all,
// and the uint8 intermediate never reaches HBM.  Any in_w and image alignment: a row's
// words start at its address rounded down to 4, the remainder joins the window's offset.
// Bound by instruction issue (a byte extraction and a 24-bit multiply-add per tap and
// channel: the VALU is busy for 96 % of the cycles) and, up to four images, by the host and the
// launches.  Whole call, 1024 x 1024 ->
// 518: one image 48.9 -> 18.2 us, 4 51.9 -> 18.6, 16 97.1 -> 42.9 against a band of 8 whole rows per
// workgroup, its source rows staged one at a time with a barrier each; 4 of 1023 x 1023, whose
// width took two passes through HBM, 56.9 -> 18.6.  With a test of every word
// against the batch's ends, which put each load behind its own branch and wait, 16 images took
// 52.5 us; tiles away from the ends now go without.
constexpr int kTileCols = kWave;      // output columns per tile at most: one per lane
constexpr int kTileMaxBand = 16;
constexpr int kTileMaxTaps = 31;
constexpr int kWaves = kThreads / kWave;
constexpr int kLoadRows = 5, kLoadWords = 2;  // rows x words of 64 lanes a wave loads at once

// 24-bit products: bytes times coefficients below 2 in 22-bit fixed point
__device__ inline int mad24(uint32_t byte, int coeff, int acc) { return __mul24((int)byte, coeff) + acc; }

// Horizontal tap sums of one output pixel from an LDS row: the window's 3*kT bytes
// (kT = the axis' tap count, <= kW) start at byte a; they are read as aligned 4-byte
// words, realigned by a % 4 with v_alignbyte, and each byte is then at a
// compile-time position.
template <int kW, int kT>
__device__ inline int3 hsum_words(const uint8_t* __restrict__ row, int a, const int (&c)[kW]) {
  constexpr int kE = (3 * kT + 3) / 4;           // realigned words holding the 3*kT window bytes
  constexpr int kD = kE + 1;                      // words read: the window at any offset a % 4
  const uint32_t* w = reinterpret_cast<const uint32_t*>(row + (a & ~3));
  uint32_t d[kD];
#pragma unroll
  for (int i = 0; i < kD; ++i) d[i] = w[i];
  const uint32_t sh = (uint32_t)(a & 3);
  uint32_t e[kE];
#pragma unroll
  for (int i = 0; i < kE; ++i) e[i] = __builtin_amdgcn_alignbyte(d[i + 1], d[i], sh);
  int s0 = 1 << (kPrecisionBits - 1), s1 = s0, s2 = s0;
#pragma unroll
  for (int x = 0; x < kT; ++x) {
    const int j = 3 * x;
    s0 = mad24((e[j >> 2] >> (8 * (j & 3))) & 0xffu, c[x], s0);
    s1 = mad24((e[(j + 1) >> 2] >> (8 * ((j + 1) & 3))) & 0xffu, c[x], s1);
    s2 = mad24((e[(j + 2) >> 2] >> (8 * ((j + 2) & 3))) & 0xffu, c[x], s2);
  }
  return make_int3(s0, s1, s2);
}

// The word at p, which lies on a 4-byte boundary and may stick out of [first, end) at the
// first or last bytes of the batch: bytes outside are not read.
__device__ inline uint32_t image_word(const uint8_t* p, const uint8_t* first, const uint8_t* end) {
  if (p >= first && p + 4 <= end) return *reinterpret_cast<const uint32_t*>(p);
  uint32_t v = 0;
  for (int i = 0; i < 4; ++i)
    if (p + i >= first && p + i < end) v |= (uint32_t)p[i] << (8 * i);
  return v;
}

template <int kW, int kT>
__global__ __launch_bounds__(kThreads) void tile_kernel(const uint8_t* __restrict__ src, int batch, int in_h,
                                                        int in_w, int out_h, int out_w, int band, int cols,
                                                        int max_rows, int pitch, const int2* __restrict__ bh,
                                                        const int* __restrict__ kh, const int2* __restrict__ bv,
                                                        const int* __restrict__ kv, Norm nrm,
                                                        float* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];  // [max_rows][pitch] bytes | [max_rows][64] words
  __shared__ float lut[3][256];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int x0 = blockIdx.x * cols, x1 = min(x0 + cols, out_w);
  const int y0 = blockIdx.y * band, y1 = min(y0 + band, out_h);
  const int r0 = bv[y0].x, nrows = bv[y1 - 1].x + bv[y1 - 1].y - r0;
  const int c0 = bh[x0].x, c1 = bh[x1 - 1].x + bh[x1 - 1].y;
  // the host sized the LDS with the same window arithmetic
  if (nrows > max_rows || 3 * (c1 - c0) + 3 * kT + 16 > pitch) return;
  uint32_t* const blk = reinterpret_cast<uint32_t*>(smem + max_rows * pitch);

  const long long row_bytes = (long long)in_w * 3;
  const uint8_t* const end = src + (long long)batch * in_h * row_bytes;
  const uint8_t* const first = src + ((long long)blockIdx.z * in_h + r0) * row_bytes + 3 * c0;
  const int mis0 = (int)(reinterpret_cast<uintptr_t>(first) & 3), row_mis = (int)(row_bytes & 3);
  const int seg = 3 * (c1 - c0);  // bytes of a row
  auto row_word = [&](int rr) {   // the boundary below the row's first byte
    return first + rr * row_bytes - ((mis0 + rr * row_mis) & 3);
  };
  auto stage = [&](auto whole) {
    for (int r = wave; r < nrows; r += kWaves * kLoadRows) {
      for (int w0 = 0; 4 * w0 < seg + 3; w0 += kWave * kLoadWords) {
        uint32_t v[kLoadRows][kLoadWords];
#pragma unroll
        for (int i = 0; i < kLoadRows; ++i) {
          // past the rectangle its last row and word are loaded again, never stored
          const int rr = min(r + i * kWaves, nrows - 1);
          const int last = (((mis0 + rr * row_mis) & 3) + seg - 1) / 4;
          const uint8_t* p = row_word(rr);
#pragma unroll
          for (int j = 0; j < kLoadWords; ++j) {
            const uint32_t at = 4 * (uint32_t)min(w0 + j * kWave + lane, last);
            if constexpr (decltype(whole)::value) {
              v[i][j] = *reinterpret_cast<const uint32_t*>(p + at);
            } else {
              v[i][j] = image_word(p + at, src, end);
            }
          }
        }
        // every load before the first wait (the compiler sinks one into its store's branch)
#pragma unroll
        for (int i = 0; i < kLoadRows; ++i)
#pragma unroll
          for (int j = 0; j < kLoadWords; ++j) asm volatile("" : "+v"(v[i][j]));
#pragma unroll
        for (int i = 0; i < kLoadRows; ++i)
#pragma unroll
          for (int j = 0; j < kLoadWords; ++j) {
            const int rr = r + i * kWaves, w = w0 + j * kWave + lane;
            if (rr < nrows && 4 * w < seg + 3) *reinterpret_cast<uint32_t*>(smem + rr * pitch + 4 * w) = v[i][j];
          }
      }
    }
  };
  // a rectangle whose words all lie inside the batch needs no test per word
  if (row_word(0) >= src && row_word(nrows - 1) + seg + 6 <= end) {
    stage(std::true_type{});
  } else {
    stage(std::false_type{});
  }
  const bool active = x0 + lane < x1;
  const int xx = active ? x0 + lane : x1 - 1;
  int hc[kW];
  load_coeffs<kW>(kh + (long long)xx * kW, hc);
  const int off = 3 * (bh[xx].x - c0);
#pragma unroll
  for (int c = 0; c < 3; ++c) lut[c][tid] = ((float)tid / 255.0f - nrm.mean[c]) / nrm.stdv[c];
  __syncthreads();

  for (int r = wave; r < nrows; r += kWaves) {
    // taps past the window carry weight 0; they read the row's slack bytes
    const int3 s = hsum_words<kW, kT>(smem + r * pitch, off + ((mis0 + r * row_mis) & 3), hc);
    blk[r * kWave + lane] = clip8(s.x) | clip8(s.y) << 8 | clip8(s.z) << 16;
  }
  __syncthreads();

  const long long plane = (long long)out_h * out_w;
  float* o = out + (long long)blockIdx.z * 3 * plane + x0 + lane;
  for (int y = y0 + wave; y < y1; y += kWaves) {
    const int top = bv[y].x - r0;
    int s0 = 1 << (kPrecisionBits - 1), s1 = s0, s2 = s0;
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      const int c = kv[(long long)y * kW + t];
      const uint32_t u = blk[min(top + t, nrows - 1) * kWave + lane];  // weight 0 past the window
      s0 = mad24(u & 0xffu, c, s0);
      s1 = mad24((u >> 8) & 0xffu, c, s1);
      s2 = mad24((u >> 16) & 0xffu, c, s2);
    }
    if (active) {
      o[(long long)y * out_w] = lut[0][clip8(s0)];
      o[(long long)y * out_w + plane] = lut[1][clip8(s1)];
      o[(long long)y * out_w + 2 * plane] = lut[2][clip8(s2)];
    }
  }
}

// Tile of the fused kernel, or band 0 when it does not apply (more than 31 taps; there the
// passes through HBM read each source row once, a tile several times).  Up to 31 taps the
// tile is ahead throughout: 1400 x 1365 -> 224 (27 taps, 3 images) 69.4 -> 34.5 us, 1000 x
// 777 -> 224 (6 images) 75.8 -> 23.3, 300 x 300 -> 224 (1) 55.1 -> 17.9.  Columns:
// equal tiles of at most 64.  Band: the more output rows share a source row, the fewer
// source rows are resampled twice, but the rectangle must leave room for several
// workgroups per CU, and the grid must fill the chip.
constexpr size_t kTileLds = 32 * 1024, kTileLdsMax = 60 * 1024;
constexpr long long kTileGrid = 1024;

struct TilePlan {
  int band, cols, max_rows, pitch;
  size_t lds;
};

inline TilePlan tile_plan(int batch, int in_h, int in_w, int out_h, int out_w, const AxisGeom& gh, const AxisGeom& gv,
                          int taps) {
  TilePlan best{0, 0, 0, 0, 0};
  if (taps > kTileMaxTaps) return best;
  const int tiles = (out_w + kTileCols - 1) / kTileCols;
  best.cols = ((out_w + tiles - 1) / tiles + 3) & ~3;
  auto extent = [](const AxisGeom& g, int in_size, int out_size, int step) {  // most source rows or columns of a tile
    int worst = 0;
    for (int i = 0; i < out_size; i += step) {
      const int j = i + step < out_size ? i + step : out_size;
      const int2 a = window(g, in_size, i, nullptr), z = window(g, in_size, j - 1, nullptr);
      worst = worst > z.x + z.y - a.x ? worst : z.x + z.y - a.x;
    }
    return worst;
  };
  // a row: its words, and what the widest instantiated window reads past them
  best.pitch = (3 * extent(gh, in_w, out_w, best.cols) + 3 * kTileMaxTaps + 16 + 3) & ~3;
  for (int band = kTileMaxBand; band >= 1; band /= 2) {
    best.max_rows = extent(gv, in_h, out_h, band);
    best.lds = (size_t)best.max_rows * (best.pitch + 4 * kWave);
    const long long grid = (long long)batch * tiles * ((out_h + band - 1) / band);
    if (band > 4 ? best.lds <= kTileLds && grid >= kTileGrid : best.lds <= kTileLdsMax) {
      best.band = band;
      return best;
    }
  }
  return best;
}

// Coefficient row widths the kernels are instantiated for.
inline int table_width(int taps) {
  const int widths[] = {4, 8, 12, 16, 24, 32, 48, 64};
  for (int w : widths)
    if (taps <= w) return w;
  return 0;
}

// Workspace: h-axis bounds + coefficients | v-axis bounds + coefficients | uint8 intermediate.
struct Plan {
  AxisGeom gh, gv;
  bool need_h, need_v;
  TilePlan tile;             // fused kernel, when tile.band > 0
  bool words;                // the interface asks for 4-byte aligned images and reserves no uint8 intermediate
  int width;                 // coefficient row width (both axes): a bucket >= the taps of either axis
  int taps;                  // the larger of the two axes' tap counts
  int row0, rows;            // source rows the vertical pass reads (horizontal pass extent)
  size_t off_bh, off_kh, off_bv, off_kv, off_tmp, total;
};

inline Plan plan(int batch, int in_h, int in_w, int out_h, int out_w) {
  Plan p;
  p.gh = axis_geom(in_w, out_w);
  p.gv = axis_geom(in_h, out_h);
  p.need_h = out_w != in_w;
  p.need_v = out_h != in_h;
  if (!p.need_h) p.gh.taps = 1;
  if (!p.need_v) p.gv.taps = 1;
  p.taps = p.gh.taps > p.gv.taps ? p.gh.taps : p.gv.taps;
  p.width = table_width(p.taps);
  const bool both = p.need_h && p.need_v;
  p.tile = both ? tile_plan(batch, in_h, in_w, out_h, out_w, p.gh, p.gv, p.taps) : TilePlan{0, 0, 0, 0, 0};
  // the terms of the interface, which callers size and align their buffers by; the fused kernel
  // itself takes other widths, alignments and tap counts too and then leaves the room unused
  p.words = both && in_w % 4 == 0 && out_w <= 768 && p.taps <= 15;
  if (p.need_h && p.need_v) {
    const int2 first = window(p.gv, in_h, 0, nullptr);
    const int2 last = window(p.gv, in_h, out_h - 1, nullptr);
    p.row0 = first.x;
    p.rows = last.x + last.y - first.x;
  } else {
    p.row0 = 0;
    p.rows = in_h;
  }
  size_t off = 0;
  p.off_bh = off;
  off = align_up(off + (size_t)out_w * sizeof(int2), 256);
  p.off_kh = off;
  off = align_up(off + (size_t)out_w * p.width * sizeof(int), 256);
  p.off_bv = off;
  off = align_up(off + (size_t)out_h * sizeof(int2), 256);
  p.off_kv = off;
  off = align_up(off + (size_t)out_h * p.width * sizeof(int), 256);
  p.off_tmp = off;
  // the two passes write an intermediate: whoever takes them has room for it
  if (p.need_h && (!p.words || p.tile.band == 0)) off = align_up(off + (size_t)batch * p.rows * out_w * 3, 256);
  p.total = off;
  return p;
}

inline int validate(int batch, int in_h, int in_w, int out_h, int out_w) {
  if (batch < 1 || in_h < 1 || in_w < 1 || out_h < 1 || out_w < 1) return MUSC_ERR_INVALID_ARG;
  if (batch > 65535 || out_h > 65535 || in_h > 65535) return MUSC_ERR_UNSUPPORTED;  // grid y / z limits
  if ((long long)in_h * in_w * 3 > (1LL << 31)) return MUSC_ERR_UNSUPPORTED;
  const AxisGeom gh = axis_geom(in_w, out_w), gv = axis_geom(in_h, out_h);
  if (gh.taps > kMaxTaps || gv.taps > kMaxTaps) return MUSC_ERR_UNSUPPORTED;
  return MUSC_OK;
}

}  // namespace prep
}  // namespace musc

using namespace musc;

extern "C" int musc_preprocess_workspace_bytes(int batch, int in_h, int in_w, int out_h, int out_w, size_t* out) {
  if (!out) return MUSC_ERR_INVALID_ARG;
  const int rc = prep::validate(batch, in_h, in_w, out_h, out_w);
  if (rc) return rc;
  *out = prep::plan(batch, in_h, in_w, out_h, out_w).total;
  return MUSC_OK;
}

extern "C" int musc_preprocess_u8(const uint8_t* images, int batch, int in_h, int in_w, int out_h, int out_w,
                                  const float* mean3, const float* std3, float* out, void* workspace,
                                  size_t workspace_bytes, hipStream_t stream) {
  if (!images || !mean3 || !std3 || !out) return MUSC_ERR_INVALID_ARG;
  int rc = prep::validate(batch, in_h, in_w, out_h, out_w);
  if (rc) return rc;
  const prep::Plan p = prep::plan(batch, in_h, in_w, out_h, out_w);
  if (p.words && (reinterpret_cast<uintptr_t>(images) & 3) != 0) return MUSC_ERR_INVALID_ARG;
  if (!workspace || workspace_bytes < p.total) return MUSC_ERR_WORKSPACE;
  prep::Norm nrm;
  for (int c = 0; c < 3; ++c) {
    if (!(std3[c] != 0.0f)) return MUSC_ERR_INVALID_ARG;
    nrm.mean[c] = mean3[c];
    nrm.stdv[c] = std3[c];
  }
  char* ws = static_cast<char*>(workspace);
  auto* bh = reinterpret_cast<int2*>(ws + p.off_bh);
  auto* kh = reinterpret_cast<int*>(ws + p.off_kh);
  auto* bv = reinterpret_cast<int2*>(ws + p.off_bv);
  auto* kv = reinterpret_cast<int*>(ws + p.off_kv);
  auto* tmp = reinterpret_cast<uint8_t*>(ws + p.off_tmp);
  const int T = prep::kThreads;
  // the two-pass path reads the horizontal pass's rows from 0; the fused kernel reads source rows
  const int vshift = (p.need_h && p.tile.band == 0) ? p.row0 : 0;
  const prep::AxisTable th{p.gh, in_w, out_w, 0, p.need_h ? 0 : 1, bh, kh};
  const prep::AxisTable tv{p.gv, in_h, out_h, vshift, p.need_v ? 0 : 1, bv, kv};
#define MUSC_PREP_COEFF(L)                                                                                         \
  hipLaunchKernelGGL(prep::coeff_kernel<L>, dim3((unsigned)(((long long)(out_w + out_h) * L + T - 1) / T)), dim3(T), \
                     0, stream, th, tv, p.width)
  if (p.width <= 16) {
    MUSC_PREP_COEFF(16);
  } else if (p.width <= 32) {
    MUSC_PREP_COEFF(32);
  } else {
    MUSC_PREP_COEFF(64);
  }
#undef MUSC_PREP_COEFF
  const prep::TilePlan& tp = p.tile;
  if (tp.band > 0) {
#define MUSC_PREP_TILE(W, TAPS)                                                                                    \
  hipLaunchKernelGGL((prep::tile_kernel<W, TAPS>),                                                                 \
                     dim3((out_w + tp.cols - 1) / tp.cols, (out_h + tp.band - 1) / tp.band, batch), dim3(T), tp.lds, \
                     stream, images, batch, in_h, in_w, out_h, out_w, tp.band, tp.cols, tp.max_rows, tp.pitch, bh,  \
                     kh, bv, kv, nrm, out)
    switch (p.taps) {  // odd, at least 5 when an axis is resampled
      case 5: MUSC_PREP_TILE(8, 5); break;
      case 7: MUSC_PREP_TILE(8, 7); break;
      case 9: MUSC_PREP_TILE(12, 9); break;
      case 11: MUSC_PREP_TILE(12, 11); break;
      case 13: MUSC_PREP_TILE(16, 13); break;
      case 15: MUSC_PREP_TILE(16, 15); break;
      case 17: case 19: MUSC_PREP_TILE(24, 19); break;
      case 21: case 23: MUSC_PREP_TILE(24, 23); break;
      case 25: case 27: MUSC_PREP_TILE(32, 27); break;
      case 29: case 31: MUSC_PREP_TILE(32, 31); break;
      default: return MUSC_ERR_UNSUPPORTED;
    }
#undef MUSC_PREP_TILE
    return check_launch();
  }
#define MUSC_PREP_LAUNCH(W)                                                                                        \
  if (p.need_h) {                                                                                                  \
    hipLaunchKernelGGL(prep::hpass_kernel<W>, dim3((out_w + T - 1) / T, p.rows, batch), dim3(T), 0, stream,       \
                       images, tmp, in_h, in_w, p.row0, p.rows, out_w, bh, kh);                                     \
    hipLaunchKernelGGL(prep::vpass_kernel<W>, dim3((out_w + T - 1) / T, out_h, batch), dim3(T), 0, stream, tmp,   \
                       p.rows, out_w, out_h, bv, kv, nrm, out);                                                    \
  } else {                                                                                                         \
    hipLaunchKernelGGL(prep::vpass_kernel<W>, dim3((out_w + T - 1) / T, out_h, batch), dim3(T), 0, stream, images,\
                       in_h, in_w, out_h, bv, kv, nrm, out);                                                       \
  }
  switch (p.width) {
    case 4: MUSC_PREP_LAUNCH(4); break;
    case 8: MUSC_PREP_LAUNCH(8); break;
    case 12: MUSC_PREP_LAUNCH(12); break;
    case 16: MUSC_PREP_LAUNCH(16); break;
    case 24: MUSC_PREP_LAUNCH(24); break;
    case 32: MUSC_PREP_LAUNCH(32); break;
    case 48: MUSC_PREP_LAUNCH(48); break;
    case 64: MUSC_PREP_LAUNCH(64); break;
    default: return MUSC_ERR_UNSUPPORTED;
  }
#undef MUSC_PREP_LAUNCH
  return check_launch();
}
