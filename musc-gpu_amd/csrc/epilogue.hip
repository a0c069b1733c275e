// Score-map epilogue for gfx950: layer/radius means, bilinear upsampling with
// align_corners=True, and the per-image maximum.
//
// Reference (models/musc.py:259-288): mean over the layers' (N, P) float64 maps,
// mean over radii, view (N, 1, side, side), F.interpolate(size=S, bilinear,
// align_corners=True), image score = max of each S x S map.
//
// One workgroup per (image, band of output rows: up to kRows, fewer when the bands
// would not fill the chip or a strong downsampling would make them span more than
// kMaxGridRows grid rows).  A band touches a few grid rows, so the workgroup averages
// only those rows of the n_radii * n_layers score maps into LDS.  Thread t owns output
// column t (t + blockDim.x, ...) and walks down the band: the horizontal
// interpolants of the two grid rows around an output row change only when the output
// row passes a grid row, so a pixel costs the vertical interpolation and one store of a
// whole coalesced row.  The band maximum is merged into image_scores with a 64-bit
// atomicMax on the bit pattern (all scores are non-negative distances, whose
// IEEE bits order like the values).  The maximum propagates NaN, as numpy's max
// at models/musc.py:288 does: NaN bit patterns (either sign) compare above every
// non-negative number as unsigned integers, so the atomic keeps them too.
//
// Bound by the float64 map writes: N = 83, 3 x 4 maps, 37 -> 518 (178 MB written, 11 MB
// read) in 37.8 us = 5.0 TB/s, the rate of a large copy; 62.5 us when every pixel formed
// its own coordinates and both horizontal interpolants in 8-row bands.
#include "common.hpp"

namespace musc {
namespace epi {

constexpr int kRows = 32;          // output rows per band at most
constexpr int kMaxThreads = 1024;
constexpr int kMaxSide = 128;
constexpr int kMaxGridRows = 16;   // grid rows one band may touch
constexpr int kFillBlocks = 256;   // workgroups wanted before bands grow (one per CU)

__device__ inline double nmax(double a, double b) { return __builtin_elementwise_maximum(a, b); }

// kGroups > 1 (rows narrower than a workgroup): that many groups of blockDim.x / kGroups
// threads, each with a column per thread, walk equal runs of the band's rows.
template <int kGroups>
__global__ __launch_bounds__(kMaxThreads) void maps_kernel(const double* __restrict__ scores, int n_radii,
                                                           int n_layers, int n, int side, int out_size, int rows,
                                                           double* __restrict__ maps,
                                                           unsigned long long* __restrict__ image_bits) {
  const int bands = (out_size + rows - 1) / rows;
  const int img = blockIdx.x / bands, band = blockIdx.x % bands;
  const int y0 = band * rows;
  const int y1 = min(out_size, y0 + rows);
  const int P = side * side;
  const double scale = out_size > 1 ? (double)(side - 1) / (double)(out_size - 1) : 0.0;
  // grid rows touched by output rows y0..y1-1
  const int g0 = (int)(scale * y0);
  int g1 = (int)(scale * (y1 - 1));
  g1 = min(g1 + 1, side - 1);
  const int ng = g1 - g0 + 1;

  __shared__ double avg[kMaxGridRows][kMaxSide];
  __shared__ double s_lh1[kRows];
  __shared__ int s_h0[kRows];
  for (int t = threadIdx.x; t < ng * side; t += blockDim.x) {
    const int gr = g0 + t / side, gc = t % side;
    const long long pix = (long long)gr * side + gc;
    double rsum = 0.0;
    for (int r = 0; r < n_radii; ++r) {
      double lsum = 0.0;
      for (int l = 0; l < n_layers; ++l) lsum += scores[(((long long)r * n_layers + l) * n + img) * P + pix];
      rsum += lsum / (double)n_layers;
    }
    avg[t / side][gc] = rsum / (double)n_radii;
  }
  if (kGroups == 1 && threadIdx.x < y1 - y0) {
    const double sy = scale * (y0 + (int)threadIdx.x);
    const int h0 = (int)sy;
    s_h0[threadIdx.x] = h0;
    s_lh1[threadIdx.x] = sy - h0;
  }
  __syncthreads();

  constexpr int kCols = 4 * kWave / kGroups;  // columns of a group
  const int per = (y1 - y0 + kGroups - 1) / kGroups;
  const int yb = kGroups > 1 ? (int)threadIdx.x / kCols * per : 0, ye = kGroups > 1 ? min(yb + per, y1 - y0) : y1 - y0;
  const int first = kGroups > 1 ? (yb < ye ? (int)threadIdx.x % kCols : out_size) : (int)threadIdx.x;
  double vmax = 0.0;
  for (int x = first; x < out_size; x += blockDim.x) {
    const double sx = scale * x;
    const int w0 = (int)sx;
    const int w1 = w0 < side - 1 ? w0 + 1 : w0;
    const double lw1 = sx - w0, lw0 = 1.0 - lw1;
    auto across = [&](int g) { return lw0 * avg[g - g0][w0] + lw1 * avg[g - g0][w1]; };
    double* dst = maps ? maps + ((long long)img * out_size + y0) * out_size + x : nullptr;
    // a group's few rows form their coordinates themselves, a whole band reads the table
    int h = kGroups > 1 ? (int)(scale * (y0 + yb)) : s_h0[0];  // grid row of `top`; the same throughout a group
    double top = across(h), bottom = across(min(h + 1, side - 1));
    int next_h0 = h;                      // the next output row's table entries, read one row ahead
    double next_lh1 = kGroups > 1 ? 0.0 : s_lh1[0];
    for (int y = yb; y < ye; ++y) {
      int h0 = next_h0;
      double lh1 = next_lh1;
      if constexpr (kGroups > 1) {
        const double yy = y0 + y;
        h0 = (int)(scale * yy);
        lh1 = __builtin_fma(scale, yy, -(double)h0);  // rounded once, as the table's difference is
      } else {
        const int yn = min(y + 1, ye - 1);
        next_h0 = s_h0[yn];
        next_lh1 = s_lh1[yn];
      }
      const double lh0 = 1.0 - lh1;
      if (h0 != h) {
        top = h0 == h + 1 ? bottom : across(h0);
        bottom = across(min(h0 + 1, side - 1));
        h = h0;
      }
      const double v = lh0 * top + lh1 * bottom;
      if (dst) dst[(long long)y * out_size] = v;
      vmax = nmax(vmax, v);
    }
  }
  if (image_bits) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) vmax = nmax(vmax, __shfl_xor(vmax, off, kWave));
    __shared__ double wmax[kMaxThreads / kWave];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (lane == 0) wmax[wave] = vmax;
    __syncthreads();
    if (threadIdx.x == 0) {
      double m = wmax[0];
      for (int w = 1; w < (kGroups > 1 ? 4 : (int)(blockDim.x / kWave)); ++w) m = nmax(m, wmax[w]);
      atomicMax(image_bits + img, (unsigned long long)__double_as_longlong(m));
    }
  }
}

}  // namespace epi
}  // namespace musc

using namespace musc;

extern "C" int musc_maps_f64(const double* scores, int n_radii, int n_layers, int n, int side, int out_size,
                             double* maps, double* image_scores, hipStream_t stream) {
  if (!scores || n_radii < 1 || n_layers < 1 || n < 1 || side < 1 || out_size < 1) return MUSC_ERR_INVALID_ARG;
  if (!maps && !image_scores) return MUSC_ERR_INVALID_ARG;
  if (side > epi::kMaxSide) return MUSC_ERR_UNSUPPORTED;
  // a band of R output rows starting at y0 touches grid rows floor(scale y0) ..
  // floor(scale (y0 + R - 1)) + 1, at most floor(scale (R - 1)) + 3 of them: take the
  // largest R <= kRows within kMaxGridRows (R = 1 always is: 3 rows)
  const double scale = out_size > 1 ? (double)(side - 1) / (double)(out_size - 1) : 0.0;
  int rows = epi::kRows;
  while (rows > 1 && (int)(scale * (rows - 1)) + 3 > epi::kMaxGridRows) --rows;
  // 32-row bands repeat less of the averaging of the grid rows shared with their
  // neighbours; 16-row bands only where 32 would leave CUs idle (3 x 4 maps, 37 -> 518, by
  // N, 16 against 32 rows: N = 8 12.0 / 12.8 us, 16 15.9 / 15.7, 83 42.5 / 37.8)
  // (upsampling less than four times, where the averaging is most of the work, four times the
  // workgroups before 32 rows, eight before 16: 25 maps 125 -> 140 10.9 us without, 9.5 so)
  const bool wide = scale < 0.25;
  auto blocks = [&](int r) { return (long long)n * ((out_size + r - 1) / r); };
  if (rows > 16 && blocks(rows) < (wide ? 1 : 4) * epi::kFillBlocks) rows = 16;
  // a handful of small maps: the walk down a band is all the time there is (one image, 3 x 4 maps,
  // 37 -> 518, 8 against 16 rows: 7.4 / 8.1 us; 8 images 64 -> 64 5.8 / 6.3; 14 -> 100 5.9 / 5.7)
  if (rows > 8 && blocks(rows) < (wide ? epi::kFillBlocks / 4 : 2 * epi::kFillBlocks)) rows = 8;
  const int bands = (out_size + rows - 1) / rows;
  // a column per thread; at least four waves, for the averaging and, on rows of up to 128 columns,
  // in groups that share the band's rows (one map, 83 images 64 -> 64: 8.4 us with three of four
  // waves idle, 7.1 so; 16 -> 128: 9.9 / 8.2; 500 of 8 -> 16: 7.0 / 5.4).  A last turn of few
  // columns past 1024 stays: equal turns, with fewer waves, take 188 us for 1030 where it takes 166
  const int threads = min(max((out_size + kWave - 1) / kWave * kWave, 4 * kWave), epi::kMaxThreads);
  if ((long long)n * bands > 0x7fffffffLL) return MUSC_ERR_UNSUPPORTED;
  unsigned long long* bits = reinterpret_cast<unsigned long long*>(image_scores);
  if (bits) launch_fill_u32(reinterpret_cast<uint32_t*>(bits), (size_t)n * 2, 0u, stream);
  auto kernel = epi::maps_kernel<1>;
  if (out_size <= kWave / 2) kernel = epi::maps_kernel<8>;
  else if (out_size <= kWave) kernel = epi::maps_kernel<4>;
  else if (out_size <= 2 * kWave) kernel = epi::maps_kernel<2>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(n * bands)), dim3(threads), 0, stream, scores, n_radii, n_layers, n, side,
                     out_size, rows, maps, bits);
  return check_launch();
}
