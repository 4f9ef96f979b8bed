// Fully connected layers of one to four images, forward: y[k, n] = sum over the volume of f[., k] x[., n].
//
// What bounds them is reading the bank once (2048 -> 1000: 8 MB, under 2 us); as a product of one pixel they ran on tiles made for
// 32 and more, behind a bank packed for those.  Here a workgroup has one filter: its 256 threads read the filter where it lies, 16
// bytes each, multiply it with every image's values (small, from the caches) and meet in LDS.  A sum is FV / 256 products per thread, then
// a tree.  Bank in hand, one image
// / four: 2048 -> 1000 18.7 -> 6.2 / 18.4 -> 6.6 us, 512 -> 100 41 -> 6.4 / 6.1, 7x7x512 -> 1000 64 -> 17.6 / 67 -> 25, 4096 -> 4096
// 25.5 -> 13.3 / 18, 6x6x256 -> 4096 42.3 -> 28.2; packing it took 7 to 55 us more.  Error against 64 bits 2.6e-7 -> 0.9e-7, 7.4e-7 ->
// 2.0e-7 (7x7x512).
#include "conv_common.hpp"

namespace mcn {
namespace {

constexpr int kThreads = 256;

template <int IMAGES, bool VEC>
__global__ __launch_bounds__(kThreads) void conv_dot(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ f,
                                                     const float* __restrict__ bias, int FV, int K, float alpha, float beta) {
  __shared__ float lds[IMAGES][kThreads / kWave];
  const int k = blockIdx.x, lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const float* row = f + (size_t)k * FV;
  float sum[IMAGES];
#pragma unroll
  for (int n = 0; n < IMAGES; ++n) sum[n] = 0.f;
  if (VEC) {
#pragma unroll 4
    for (int i = threadIdx.x; i < FV / 4; i += kThreads) {
      const v4f w = ((const v4f*)row)[i];
#pragma unroll
      for (int n = 0; n < IMAGES; ++n) {
        const v4f v = ((const v4f*)(x + (size_t)n * FV))[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[n] = fmaf(w[e], v[e], sum[n]);
      }
    }
  } else {
#pragma unroll 4
    for (int i = threadIdx.x; i < FV; i += kThreads)
#pragma unroll
      for (int n = 0; n < IMAGES; ++n) sum[n] = fmaf(row[i], x[(size_t)n * FV + i], sum[n]);
  }
#pragma unroll
  for (int n = 0; n < IMAGES; ++n) {
#pragma unroll
    for (int lanes = kWave / 2; lanes > 0; lanes >>= 1) sum[n] += __shfl_xor(sum[n], lanes);
    if (lane == 0) lds[n][wave] = sum[n];
  }
  __syncthreads();
  if (threadIdx.x < IMAGES) {
    const int n = threadIdx.x;
    float* o = y + (size_t)n * K + k;
    float v = alpha * ((lds[n][0] + lds[n][1]) + (lds[n][2] + lds[n][3]));
    if (beta != 0.f) v = fmaf(beta, *o, v);
    if (bias) v += bias[k];
    *o = v;
  }
}

}  // namespace

// From some 1.1e8 products on reading the images' values once per filter costs what the tiles cost that read a packed bank
// (6x6x256x4096, 3 images 43.4 -> 43.3, 4 images 44.3 -> 50.4): not taken where one is in hand.  Else packing alone takes longer.
bool conv_dot_takes(const ConvP& p, bool packed) {
  if (packed && (double)p.N * p.FC * p.K > 1.1e8) return false;
  return p.H * p.W == 1 && p.FH * p.FW == 1 && p.pt == 0 && p.pl == 0 && p.outH * p.outW == 1 && p.groups == 1 && p.N >= 1 && p.N <= 4 && p.FC > 0 &&
         !tunable("conv_no_dot", 0);
}

int conv_dot_launch(hipStream_t s, const char* who, const ConvP& p, float* y, float outMult, const float* x, float inMult, const float* f,
                    const float* bias) {
  const bool vec = p.FC % 4 == 0 && aligned16(x) && aligned16(f);
  const dim3 grid((unsigned)p.K), block(kThreads);
  KernelTimer timer("conv_dot", s);
#define DOT_GO(N)                                                                                                                  \
  case N:                                                                                                                          \
    if (vec) hipLaunchKernelGGL((conv_dot<N, true>), grid, block, 0, s, y, x, f, bias, p.FC, p.K, inMult, outMult);                  \
    else hipLaunchKernelGGL((conv_dot<N, false>), grid, block, 0, s, y, x, f, bias, p.FC, p.K, inMult, outMult);                     \
    break
  switch (p.N) {
    DOT_GO(1);
    DOT_GO(2);
    DOT_GO(3);
    DOT_GO(4);
  }
#undef DOT_GO
  return check_launch(who);
}

}  // namespace mcn
