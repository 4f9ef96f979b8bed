// Filter gradient in double precision on v_mfma_f64_16x16x4_f64:  dF[R, k] = sum over the output pixels m of all images of
// xg[R, m] dzdy[k, m], xg = the (never materialised) patch matrix.
//
// What bounds it is the matrix instruction (16 of them, 1024 cycles, per wavefront and step); the general kernel
// (conv64_mfma) fetched with a lane per row, each lane in a cache line of its own, and waited for that: 0.35 of the
// instruction's rate.  Here the operands go from global memory straight into LDS the way they lie: a load holds 16 neighbouring
// pixels of two rows (64 lanes x 4 bytes), 8 rows apart in a half-block of 16, and such pairs lie 272 bytes apart, so that
// the 32 lanes of a fragment read (16 rows x 2 pixels) fall into 64 banks.
//   * A workgroup makes 64 filters x 64 rows, four wavefronts of 32 x 32; rows are tap-major in half-blocks of 16 channels, so
//     a half-block has one tap and its inside-the-image test is one per lane and step.  Where 16 does not divide the channels
//     (filters), the last half-block starts 16 before the end and computes some rows twice, to the same bits.
//   * Three buffers, loads two steps ahead, one between every two matrix instructions; three workgroups to a CU.
//   * A lane's pixel advances by carries, its offsets with it: no divisions in the loop.
// 3x3x64x64 on 56x56x64x32: 270 -> 145 us (51 TFLOP/s of the 77 that instruction reaches).
#include "conv_common.hpp"

#include <algorithm>

namespace mcn {
namespace {

typedef double doublex4 __attribute__((ext_vector_type(4)));

constexpr int kPairFloats = 68;                  // 272 bytes
constexpr int kHalfFloats = 8 * kPairFloats;     // a half-block: 16 rows x 16 pixels
constexpr int kBuffers = 3;
constexpr int kBufFloats = 8 * kHalfFloats;      // four half-blocks of each operand

struct Wg64P {
  int H, W, C, K, OH, OW, FH;
  int sy, sx, pt, pl, dly, dlx;
  int FV, M, chunk, halves;
  int xImg, dyImg;             // elements between images
  unsigned xBytes, dyBytes;    // < 2 GiB
  int stepW, stepH;            // 16 pixels on (after whole images): columns, rows
  int advX, carryH, carryW;  // bytes of x: 16 pixels on; on a carry out of a column; out of an image
  int advY, carryY;                // bytes of dzdy likewise
  FastDiv byQ, byOH, byFH, byTilesK, byHalves;
};

__global__ __launch_bounds__(256, 3) void conv64_wgrad_mfma(double* __restrict__ out, const double* __restrict__ x,
                                                            const double* __restrict__ dy, Wg64P p) {
  __shared__ float smem[kBuffers * kBufFloats];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave >> 1, wr = wave & 1;
  const int split = blockIdx.y;
  int rt, kt;
  p.byTilesK.divmod((int)blockIdx.x, &rt, &kt);
  const int HW8 = p.H * p.W * 8, Q8 = p.OH * p.OW * 8;
  const int mBegin = split * p.chunk, mEnd = min(mBegin + p.chunk, p.M);
  const int nSteps = mEnd > mBegin ? (mEnd - mBegin + 15) / 16 : 0;

  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, (int)p.xBytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc((void*)dy, 0, (int)p.dyBytes, 0x00020000);
  auto half_block = [&](int h, int* dh, int* dw, int* t, int* cb) {
    int j, i, part;
    p.byHalves.divmod(h < p.halves ? h : 0, t, &part);
    p.byFH.divmod(*t, &j, &i);
    *dh = i * p.dly - p.pt;
    *dw = j * p.dlx - p.pl;
    *cb = min(16 * part, p.C - 16);
  };
  // four half-blocks of rows: tap and first channel (uniform)
  int hbDh[4], hbDw[4], hbShift[4], hbRow[4], hbK[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int h = 4 * rt + b;
    int dh, dw, t, cb;
    half_block(h, &dh, &dw, &t, &cb);
    hbDh[b] = h < p.halves ? dh : -0x40000000;  // absent: never inside the image
    hbDw[b] = dw;
    hbShift[b] = (dh + p.H * dw) * 8;
    hbRow[b] = cb * HW8;
    hbK[b] = min(16 * (4 * kt + b), p.K - 16) * Q8;
  }

  // ---- this lane's pixel
  int mL = mBegin + ((lane & 31) >> 1), ih, iw;
  unsigned pixX, pixY;
  {
    int n, q, ow, oh;
    p.byQ.divmod(mL < p.M ? mL : 0, &n, &q);
    p.byOH.divmod(q, &ow, &oh);
    ih = oh * p.sy;
    iw = ow * p.sx;
    const unsigned part = (lane & 1) * 4u;
    pixX = (unsigned)(n * p.xImg + ih + p.H * iw) * 8u + (lane >> 5) * 8u * (unsigned)HW8 + part;
    pixY = (unsigned)(n * p.dyImg + q) * 8u + (lane >> 5) * 8u * (unsigned)Q8 + part;
  }
  const int endH = p.OH * p.sy, endW = p.OW * p.sx, stepIh = p.stepH * p.sy, stepIw = p.stepW * p.sx;

  unsigned voX[4], voY = kOutside;
  int bufL = 0;
  float* dst = smem;
  auto prep = [&]() {  // offsets of the next step; then on by 16 pixels (a step past the split's end fetches nothing)
    const bool valid = mL < mEnd;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const bool ok = valid && (unsigned)(ih + hbDh[b]) < (unsigned)p.H && (unsigned)(iw + hbDw[b]) < (unsigned)p.W;
      voX[b] = ok ? pixX + (unsigned)hbShift[b] : kOutside;
    }
    voY = valid ? pixY : kOutside;
    mL += 16;
    ih += stepIh;
    pixX += (unsigned)p.advX;
    pixY += (unsigned)p.advY;
    const bool cH = ih >= endH;
    ih -= cH ? endH : 0;
    iw += stepIw + (cH ? p.sx : 0);
    pixX += cH ? (unsigned)p.carryH : 0u;
    const bool cW = iw >= endW;
    iw -= cW ? endW : 0;
    pixX += cW ? (unsigned)p.carryW : 0u;
    pixY += cW ? (unsigned)p.carryY : 0u;
    dst = smem + bufL * kBufFloats;
    bufL = bufL == kBuffers - 1 ? 0 : bufL + 1;
  };
  auto issue = [&](int t) {  // load t of 16: pair wave + 4 (t & 1) of half-block t / 2 (dzdy's behind x's)
    typedef __attribute__((address_space(3))) void* lds_ptr;
    const int b = t >> 1, q = wave + 4 * (t & 1);
    float* at = dst + b * kHalfFloats + q * kPairFloats;
    if (b < 4) __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)at, 4, (int)voX[b], hbRow[b] + q * HW8, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(yr, (lds_ptr)at, 4, (int)voY, hbK[b - 4] + q * Q8, 0, 0);
  };

  doublex4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (doublex4){0.0, 0.0, 0.0, 0.0};

  const int l16 = lane & 15, lk = lane >> 4;
  const int laneAt = (l16 & 7) * kPairFloats + (l16 >> 3) * 32 + 2 * lk;
#pragma unroll
  for (int s = 0; s < kBuffers - 1; ++s) {
    prep();
#pragma unroll
    for (int t = 0; t < 16; ++t) issue(t);
  }
  asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" ::: "memory");
  int buf = 0;
#pragma unroll 1
  for (int step = 0; step < nSteps; ++step) {
    prep();
    const float* Ab = smem + buf * kBufFloats + (4 + 2 * wk) * kHalfFloats + laneAt;
    const float* Bb = smem + buf * kBufFloats + 2 * wr * kHalfFloats + laneAt;
    double a[2][2], b[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      a[0][i] = *(const double*)(Ab + i * kHalfFloats);
      b[0][i] = *(const double*)(Bb + i * kHalfFloats);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int cur = s & 1, nxt = cur ^ 1;
      if (s < 3) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a[nxt][i] = *(const double*)(Ab + i * kHalfFloats + 8 * (s + 1));
          b[nxt][i] = *(const double*)(Bb + i * kHalfFloats + 8 * (s + 1));
        }
      }
#pragma unroll
      for (int t = 4 * s; t < 4 * s + 4; ++t) issue(t);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[cur][i], b[cur][j], acc[i][j], 0, 0, 0);
    }
    // the next step's loads have landed (this step's sixteen may be in flight), this wavefront's reads are done
    asm volatile("s_waitcnt vmcnt(16)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    buf = buf == kBuffers - 1 ? 0 : buf + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- acc[i][j][e]: filter (lane / 16) + 4 e of half-block i, row lane % 16 of half-block j; stored c + C t + FV k
  double* bank = out + (size_t)split * p.FV * p.K;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int h = 4 * rt + 2 * wr + j;
    int dh, dw, t, cb;
    half_block(h, &dh, &dw, &t, &cb);
    if (h >= p.halves) continue;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int hk = 4 * kt + 2 * wk + i;
      if (16 * hk >= p.K) continue;  // (copies only)
      const int kb = min(16 * hk, p.K - 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) bank[(size_t)p.FV * (kb + lk + 4 * e) + cb + l16 + (size_t)p.C * t] = acc[i][j][e];
    }
  }
}

}  // namespace

// One filter group: its channels and filters in `p`, the image strides of the whole layer.  Offsets into both tensors stay
// below the one that loads nothing.
bool conv64_wgrad_takes(const ConvP& p, long long xLayerElements, long long yLayerElements) {
  return !tunable("conv64_no_mfma", 0) && !tunable("conv64_no_wgrad", 0) && p.FC >= 16 && p.Kg >= 16 && xLayerElements * 8 < (long long)kOutside &&
         yLayerElements * 8 < (long long)kOutside && (long long)p.outH * p.outW * p.N < (1ll << 30) &&
         (long long)p.FH * p.FW * p.FC * p.Kg < (1ll << 31) &&
         // under 512 pixels the general kernel on the matrix instruction (one group) needs one launch, no partial banks and no
         // second pass over a bank that is large beside the work (5x5x130 -> 2303 over 5 pixels 20 us, 187 here; 3x3x256 ->
         // 256 over 64 / 256 / 512 pixels 10 / 25 / 55, here 35 / 36 / 43)
         (p.groups != 1 || (long long)p.outH * p.outW * p.N >= 512 || tunable("conv_any_size", 0)) &&
         // taps whose last half-block would be mostly copies: the general kernel
         (p.FH * p.FW == 1 || 3 * ((p.FC + 15) / 16 * 16) <= 5 * p.FC);
}

// Splits of the pixels: three workgroups to a CU (3x3x64x64 on 56x56x64x32, 9 tiles: 85), at least four steps each.
int conv64_wgrad_splits(const ConvP& p) {
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  const int halves = p.FH * p.FW * ((p.FC + 15) / 16);
  const long long tiles = (long long)((halves + 3) / 4) * ((p.Kg + 63) / 64), M = (long long)p.outH * p.outW * p.N;
  long long s = std::max(1ll, std::min<long long>(3ll * cus / tiles, M / 64));
  s = std::min(s, 4096ll);
  const long long chunk = ((M + s - 1) / s + 15) / 16 * 16;
  return (int)((M + chunk - 1) / chunk);
}

int conv64_wgrad_launch(hipStream_t s, const ConvP& p, double* out, const double* x, const double* dy) {
  Wg64P q;
  q.H = p.H; q.W = p.W; q.C = p.FC; q.K = p.Kg;
  q.OH = p.outH; q.OW = p.outW; q.FH = p.FH;
  q.sy = p.sy; q.sx = p.sx; q.pt = p.pt; q.pl = p.pl; q.dly = p.dy; q.dlx = p.dx;
  q.FV = p.FH * p.FW * p.FC;
  const int Q = p.outH * p.outW;
  q.M = Q * p.N;
  const int splits = conv64_wgrad_splits(p);
  q.chunk = ((q.M + splits - 1) / splits + 15) / 16 * 16;
  const int perTap = (p.FC + 15) / 16;
  q.halves = p.FH * p.FW * perTap;
  const int tilesK = (p.Kg + 63) / 64, tilesR = (q.halves + 3) / 4;
  q.xImg = p.C * p.H * p.W;
  q.dyImg = p.K * Q;
  q.xBytes = (unsigned)(((long long)(p.N - 1) * q.xImg + (long long)p.FC * p.H * p.W) * 8);
  q.dyBytes = (unsigned)(((long long)(p.N - 1) * q.dyImg + (long long)p.Kg * Q) * 8);
  const int stepN = 16 / Q;
  const int rest = 16 % Q;
  q.stepW = rest / p.outH;
  q.stepH = rest % p.outH;
  q.advX = (int)(8u * ((unsigned)stepN * q.xImg + (unsigned)(q.stepH * p.sy) + (unsigned)p.H * (q.stepW * p.sx)));
  q.carryH = (int)(8u * ((unsigned)p.H * p.sx - (unsigned)p.outH * p.sy));
  q.carryW = (int)(8u * ((unsigned)q.xImg - (unsigned)p.H * (p.outW * p.sx)));
  q.advY = (int)(8u * ((unsigned)stepN * q.dyImg + (unsigned)rest));
  q.carryY = (int)(8u * ((unsigned)q.dyImg - (unsigned)Q));
  q.byQ = FastDiv(Q);
  q.byOH = FastDiv(p.outH);
  q.byFH = FastDiv(p.FH);
  q.byTilesK = FastDiv(tilesK);
  q.byHalves = FastDiv(perTap);
  KernelTimer timer("conv64_wgrad_mfma", s);
  hipLaunchKernelGGL(conv64_wgrad_mfma, dim3((unsigned)(tilesK * tilesR), (unsigned)splits), dim3(256), 0, s, out, x, dy, q);
  return check_launch("mcn_conv_backward_filter_f64");
}

}  // namespace mcn
