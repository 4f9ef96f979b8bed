// Fully connected layers of one to four images, forward: y[k, n] = sum over the volume of f[., k] x[., n].
//
// What bounds them is reading the bank once (2048 -> 1000: 8 MB, under 2 us); as a product of one pixel they ran on tiles made for
// 32 and more, behind a bank packed for those.  Here a workgroup has one or two filters: its 256 threads read them where they lie,
// 16 bytes each, multiply them with every image's values (small, from the caches) and meet in LDS.  A sum is FV / 256 products per
// thread, then a tree, whatever the number of filters.  Against the tiles with a packed bank in hand, in captured graphs over cold
// banks, one image / four: 2048 -> 1000 14.5 -> 3.6 / 15.0 -> 4.7 us, 512 -> 100 41 -> 2.3 / 2.9, 7x7x512 -> 1000 82 -> 22 / 26,
// 4096 -> 4096 28 -> 13 / 18, 6x6x256 -> 4096 45 -> 29 / 38, 7x7x512 -> 4096 103 -> 74 / 96; packing it took 3 to 165 us more.  Error
// against 64 bits 2.6e-7 -> 0.9e-7, 7.4e-7 -> 2.0e-7 (7x7x512).
#include "conv_common.hpp"

namespace mcn {
namespace {

constexpr int kThreads = 256;

template <int IMAGES, int FILTERS, bool VEC>
__global__ __launch_bounds__(kThreads) void conv_dot(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ f,
                                                     const float* __restrict__ bias, int FV, int K, float alpha, float beta) {
  __shared__ float lds[FILTERS][IMAGES][kThreads / kWave];
  const int k0 = blockIdx.x * FILTERS, lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const float* row[FILTERS];
  float sum[FILTERS][IMAGES];
#pragma unroll
  for (int j = 0; j < FILTERS; ++j) {
    row[j] = f + (size_t)min(k0 + j, K - 1) * FV;
#pragma unroll
    for (int n = 0; n < IMAGES; ++n) sum[j][n] = 0.f;
  }
  if (VEC) {
#pragma unroll 4
    for (int i = threadIdx.x; i < FV / 4; i += kThreads) {
      v4f w[FILTERS];
#pragma unroll
      for (int j = 0; j < FILTERS; ++j) w[j] = ((const v4f*)row[j])[i];
#pragma unroll
      for (int n = 0; n < IMAGES; ++n) {
        const v4f v = ((const v4f*)(x + (size_t)n * FV))[i];
#pragma unroll
        for (int j = 0; j < FILTERS; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[j][n] = fmaf(w[j][e], v[e], sum[j][n]);
      }
    }
  } else {
#pragma unroll 4
    for (int i = threadIdx.x; i < FV; i += kThreads)
#pragma unroll
      for (int n = 0; n < IMAGES; ++n) {
        const float v = x[(size_t)n * FV + i];
#pragma unroll
        for (int j = 0; j < FILTERS; ++j) sum[j][n] = fmaf(row[j][i], v, sum[j][n]);
      }
  }
#pragma unroll
  for (int j = 0; j < FILTERS; ++j)
#pragma unroll
    for (int n = 0; n < IMAGES; ++n) {
#pragma unroll
      for (int lanes = kWave / 2; lanes > 0; lanes >>= 1) sum[j][n] += __shfl_xor(sum[j][n], lanes);
      if (lane == 0) lds[j][n][wave] = sum[j][n];
    }
  __syncthreads();
  const int j = threadIdx.x / IMAGES, n = threadIdx.x % IMAGES;
  if (j < FILTERS && k0 + j < K) {
    float* o = y + (size_t)n * K + k0 + j;
    float v = alpha * ((lds[j][n][0] + lds[j][n][1]) + (lds[j][n][2] + lds[j][n][3]));
    if (beta != 0.f) v = fmaf(beta, *o, v);
    if (bias) v += bias[k0 + j];
    *o = v;
  }
}

}  // namespace

bool conv_dot_takes(const PixP& p) {
  return p.IH * p.IW == 1 && p.OH * p.OW == 1 && p.T == 1 && p.dhBase == 0 && p.dwBase == 0 && p.N >= 1 && p.N <= 4 && p.Cin > 0 &&
         p.inImg == p.Cin && p.outImg == p.Cout && !tunable("conv_no_dot", 0);
}

// Two filters to a workgroup halve what it reads of the images beside the bank: where the bank is large, several images, and still
// two workgroups to a CU.  One / two filters, four images: 7x7x512 -> 4096 132 / 96 us, 6x6x256 -> 4096 50 / 38.5, 7x7x512 -> 1000
// 36 / 26.5, 4096 -> 1000 8.3 / 7.4; 2048 -> 1000 4.7 / 5.0, 7x7x2048 -> 100 38 / 47.
int conv_dot_launch(hipStream_t s, const char* who, const PixP& p, float* y, const float* x, const float* f, const float* bias) {
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  const bool two = p.N >= 2 && (double)p.Cin * p.Cout >= 4e6 && p.Cout >= 2 * cus;
  const bool vec = p.Cin % 4 == 0 && aligned16(x) && aligned16(f);
  const dim3 grid((unsigned)(two ? (p.Cout + 1) / 2 : p.Cout)), block(kThreads);
  KernelTimer timer("conv_dot", s);
#define DOT_GO(N, FILTERS)                                                                                                            \
  if (vec) hipLaunchKernelGGL((conv_dot<N, FILTERS, true>), grid, block, 0, s, y, x, f, bias, p.Cin, p.Cout, p.alpha, p.beta);         \
  else hipLaunchKernelGGL((conv_dot<N, FILTERS, false>), grid, block, 0, s, y, x, f, bias, p.Cin, p.Cout, p.alpha, p.beta)
  switch (p.N) {
    case 1: DOT_GO(1, 1); break;
    case 2: if (two) { DOT_GO(2, 2); } else { DOT_GO(2, 1); } break;
    case 3: if (two) { DOT_GO(3, 2); } else { DOT_GO(3, 1); } break;
    default: if (two) { DOT_GO(4, 2); } else { DOT_GO(4, 1); } break;
  }
#undef DOT_GO
  return check_launch(who);
}

}  // namespace mcn
