// RsCIN image-score refinement for gfx950.
//
// Reference (models/modules/_RsCIN.py:5-32): scores are min-max normalised, the
// class-token similarity W = X X^T is formed, and for every k in k_list each row
// keeps only its k largest similarities (torch.topk zeroes the N-k smallest,
// :8-11); the refined score of image i is sum_j W_ij s_j / sum_j W_ij over the
// kept entries (the row-normalised D^-1 W times s, :12-18), averaged over k_list
// (:20).  One workgroup per image i: similarities of row i into LDS, each kept
// set found by rank counting (ties broken by column index), sums in fp64.  The
// similarities are accumulated in fp64, so the kept set is the one exact arithmetic
// selects: where two similarities lie closer together than fp32 rounding can
// resolve, the reference's own fp32 product keeps one or the other depending on its
// summation order, and no fp32 ordering could reproduce that choice in general.  The
// min-max normalisation propagates NaN like numpy's min/max (:27): one NaN raw
// score makes every refined score NaN, as in the reference.
#include "common.hpp"

namespace musc {
namespace rscin {

constexpr int kRowsAtOnce = 4;   // similarities a wave forms together
constexpr int kSteps = 3;        // 64-vector steps whose loads are in flight together
constexpr int kMaxN = 4096;
constexpr int kMaxK = 16;

__device__ inline double nmin(double a, double b) { return __builtin_elementwise_minimum(a, b); }
__device__ inline double nmax(double a, double b) { return __builtin_elementwise_maximum(a, b); }

struct KList {
  int k[kMaxK];
  int n, most;
};

// wave_sum of several values, their exchanges in flight together.
template <int kCount>
__device__ inline void wave_sums(double (&v)[kCount]) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    double t[kCount];
#pragma unroll
    for (int r = 0; r < kCount; ++r) t[r] = __shfl_xor(v[r], off, kWave);
#pragma unroll
    for (int r = 0; r < kCount; ++r) v[r] += t[r];
  }
}

// Latency-bound: n workgroups of a few microseconds of work each.  A wave forms four
// similarities at a time, all loads of up to 768 channels in flight together, where one
// row at a time waited for memory once per 64 channels; 16 waves share the row; each
// entry's rank is counted once for all of k_list, by several lanes.  N = 83, d = 768,
// k = 1, 2, 3, right after the map kernel: 12.1 us, against 88.7 us with 4 waves, one
// similarity at a time, scalar loads and a rank count per k.  From N = 513 on the n^2
// comparisons of a row are most of it and n rows fill the chip: 4 waves, more workgroups on
// a CU; up to N = 16 4 waves form every similarity at once (N = 1600, d = 512:
// 1.02 ms; 2.10 with 16 waves and both comparisons for every entry; 83 images 11.6 us).
template <int kVec, int kThreads>  // floats per load: 4 when every row is 16-byte aligned, else 1
__global__ __launch_bounds__(kThreads) void rscin_kernel(const float* __restrict__ x, const double* __restrict__ raw,
                                                         int n, int d, int share, KList ks, float* __restrict__ out) {
  typedef float vec __attribute__((ext_vector_type(kVec)));
  constexpr int kWaves = kThreads / kWave;
  extern __shared__ double w[];  // n similarities of row i
  __shared__ double s_range[2][kWaves];
  __shared__ double s_part[kMaxK][2][kWaves];
  __shared__ double s_ratio[kMaxK];
  const int i = blockIdx.x, tid = threadIdx.x;
  const int wave = tid / kWave, lane = tid % kWave;
  // min / max of the raw scores
  double mn = INFINITY, mx = -INFINITY;
  for (int j = tid; j < n; j += kThreads) {
    mn = nmin(mn, raw[j]);
    mx = nmax(mx, raw[j]);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    mn = nmin(mn, __shfl_xor(mn, off, kWave));
    mx = nmax(mx, __shfl_xor(mx, off, kWave));
  }
  if (lane == 0) {
    s_range[0][wave] = mn;
    s_range[1][wave] = mx;
  }
  // similarities W[i][j] = x_i . x_j (fp64 accumulation of the fp32 tokens): the loads of
  // kSteps steps of 64 vectors, of this row and of kRowsAtOnce others, before the first use
  const vec* xi = reinterpret_cast<const vec*>(x + (long long)i * d);
  const int dv = d / kVec;
  for (int j0 = wave * kRowsAtOnce; j0 < n; j0 += kWaves * kRowsAtOnce) {
    const vec* xj[kRowsAtOnce];
    double acc[kRowsAtOnce];
#pragma unroll
    for (int r = 0; r < kRowsAtOnce; ++r) {
      xj[r] = reinterpret_cast<const vec*>(x + (long long)min(j0 + r, n - 1) * d);
      acc[r] = 0.0;
    }
    for (int c0 = 0; c0 < dv; c0 += kSteps * kWave) {
      vec a[kSteps], b[kSteps][kRowsAtOnce];
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        const int c = c0 + u * kWave + lane;
        const bool ok = c < dv;  // vectors past the row add 0 x 0
        const int cc = ok ? c : dv - 1;
        a[u] = xi[cc];
#pragma unroll
        for (int r = 0; r < kRowsAtOnce; ++r) b[u][r] = xj[r][cc];
        if (!ok) {
          a[u] = vec{};
#pragma unroll
          for (int r = 0; r < kRowsAtOnce; ++r) b[u][r] = vec{};
        }
      }
#pragma unroll
      for (int u = 0; u < kSteps; ++u)
#pragma unroll
        for (int e = 0; e < kVec; ++e)
#pragma unroll
          for (int r = 0; r < kRowsAtOnce; ++r) acc[r] = fma((double)a[u][e], (double)b[u][r][e], acc[r]);
    }
    wave_sums(acc);
#pragma unroll
    for (int r = 0; r < kRowsAtOnce; ++r)
      if (lane == 0 && j0 + r < n) w[j0 + r] = acc[r];
  }
  __syncthreads();
  double lo = s_range[0][0], hi = s_range[1][0];
#pragma unroll
  for (int q = 1; q < kWaves; ++q) {
    lo = nmin(lo, s_range[0][q]);
    hi = nmax(hi, s_range[1][q]);
  }
  const double span = hi - lo;
  double num[kMaxK], den[kMaxK];
#pragma unroll
  for (int q = 0; q < kMaxK; ++q) num[q] = den[q] = 0.0;
  // an entry's rank is counted by `share` neighbouring lanes, each over every share-th entry
  for (int t0 = 0; t0 < n * share; t0 += kThreads) {
    if (t0 + wave * kWave >= n * share) break;  // a wave past the last entry counts nothing
    const int j = (t0 + tid) / share, m0 = (t0 + tid) % share;
    const bool own = j < n && m0 == 0;
    const double v = w[min(j, n - 1)];
    // entries strictly before j in descending order: those above, and equal ones with a lower
    // index; only within the wave's own entries does a comparison depend on the lane's index
    int rank = 0, m = m0;
    const int lowest = (t0 + wave * kWave) / share, past = min((t0 + wave * kWave + kWave - 1) / share + 1, n);
#pragma unroll 4
    for (; m < lowest; m += share) rank += w[m] >= v;
    for (; m < past; m += share) {
      const double u = w[m];
      rank += (u > v) | ((u == v) & (m < j));
    }
#pragma unroll 4
    for (; m < n; m += share) rank += w[m] > v;
    for (int off = share / 2; off >= 1; off >>= 1) rank += __shfl_xor(rank, off, kWave);
    if (own && rank < ks.most) {
      const double s01 = (double)(float)((raw[j] - lo) / span);
#pragma unroll
      for (int q = 0; q < kMaxK; ++q)
        if (q < ks.n && rank < ks.k[q]) {
          num[q] += v * s01;
          den[q] += v;
        }
    }
  }
#pragma unroll
  for (int q = 0; q < kMaxK; ++q)
    if (q < ks.n) {
      double part[2] = {num[q], den[q]};
      if (wave * kWave < n * share) wave_sums(part);  // waves past the last entry hold zeros
      if (lane == 0) {
        s_part[q][0][wave] = part[0];
        s_part[q][1][wave] = part[1];
      }
    }
  __syncthreads();
  if (tid < ks.n) {
    double a = 0.0, b = 0.0;
#pragma unroll
    for (int r = 0; r < kWaves; ++r) {
      a += s_part[tid][0][r];
      b += s_part[tid][1][r];
    }
    s_ratio[tid] = a / b;
  }
  __syncthreads();
  if (tid == 0) {
    double total = 0.0;
    for (int q = 0; q < ks.n; ++q) total += s_ratio[q];
    out[i] = (float)(total / ks.n);
  }
}

}  // namespace rscin
}  // namespace musc

using namespace musc;

extern "C" int musc_rscin_f32(const float* cls_tokens, const double* image_scores, int n, int d, const int* k_list,
                              int n_k, float* out, hipStream_t stream) {
  if (!cls_tokens || !image_scores || !out || !k_list || n < 1 || d < 1 || n_k < 1) return MUSC_ERR_INVALID_ARG;
  if (n > rscin::kMaxN || n_k > rscin::kMaxK) return MUSC_ERR_UNSUPPORTED;
  rscin::KList ks{};
  ks.n = n_k;
  for (int q = 0; q < n_k; ++q) {
    if (k_list[q] < 1 || k_list[q] > n) return MUSC_ERR_INVALID_ARG;
    ks.k[q] = k_list[q];
    ks.most = ks.most > k_list[q] ? ks.most : k_list[q];
  }
  const int threads = n <= 16 || n > 512 ? 256 : 1024;
  int share = 1;  // lanes per entry of the rank count
  while (share < 16 && n * share * 2 <= threads) share *= 2;
  const bool vec4 = d % 4 == 0 && (reinterpret_cast<uintptr_t>(cls_tokens) & 15) == 0;
  auto kernel = threads == 256 ? (vec4 ? rscin::rscin_kernel<4, 256> : rscin::rscin_kernel<1, 256>)
                               : (vec4 ? rscin::rscin_kernel<4, 1024> : rscin::rscin_kernel<1, 1024>);
  hipLaunchKernelGGL(kernel, dim3(n), dim3(threads), (size_t)n * sizeof(double), stream, cls_tokens, image_scores, n, d,
                     share, ks, out);
  return check_launch();
}
