// Forward and (unit strides) backward-data product in double precision on v_mfma_f64_16x16x4_f64:
//   out[co, m] = sum over taps t and channels ci of w[co, ci, t] in[ci, pixel(m) + shift(t)]
//
// What bounds it is the matrix instruction (16 of them, 1024 cycles, per wavefront and stage of 16 channels of a tap).  The
// general kernel (conv64_mfma) works out an address per element and stage and reads the bank with a lane per row; here
//   * the bank is packed first, [chunk of 16 channels][tap][16 channels][64 output channels]: a stage of it is 8 KB that lie
//     together and come straight into LDS, 256 bytes per load;
//   * a lane's pixel never changes: a stage's tap is one test and one addition for it, the channel is a scalar offset; 32
//     pixels of a channel (64 lanes x 4 bytes) come straight into LDS with a load;
//   * rows of 64 pixels lie 640 bytes apart, rows of 64 channels 640 likewise: the 32 lanes of a fragment read (2 rows x 16
//     values) fall into 64 banks;
//   * two buffers of 20 KB, the next stage's loads between this one's matrix instructions, three workgroups to a CU.
// Channels past the last of a ragged chunk are zeros in both operands (a zero weight beside an infinity would be a NaN).
// 3x3x64x64 on 56x56x64x32, backward-data: 230 -> 165 us with the packing (45 TFLOP/s of the 77 that instruction reaches).
#include "conv_common.hpp"

#include <algorithm>

namespace mcn {
namespace {

typedef double doublex4 __attribute__((ext_vector_type(4)));

constexpr int kRowFloats = 160;                    // 640 bytes: 64 doubles and the gap
constexpr int kOperandFloats = 16 * kRowFloats;    // 16 rows
constexpr int kStageFloats = 2 * kOperandFloats;   // pixels, then the bank
constexpr int kStageDoubles = 16 * 64;             // of the packed bank

struct Pix64P {
  int IH, IW, Cin, OH, OW, Cout, T, FH;
  int sy, sx, dhBase, dhStep, dwBase, dwStep;
  int M, stages;               // pixels of all images; stages of 16 channels of a tap
  int inImg, outImg;
  unsigned inBytes, bankBytes;
  double alpha, beta;
  FastDiv byQ, byOH, byTilesC;
};

template <bool RAGGED>  // channels that are no multiple of 16
__global__ __launch_bounds__(256, 3) void conv64_pix_mfma(double* __restrict__ out, const double* __restrict__ in,
                                                          const double* __restrict__ bank, const double* __restrict__ bias, Pix64P p) {
  __shared__ float smem[2 * kStageFloats];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = wave >> 1, wp = wave & 1;
  int mt, ct;
  p.byTilesC.divmod(xcd_contiguous_id((int)blockIdx.x, (int)gridDim.x), &mt, &ct);
  const int plane8 = p.IH * p.IW * 8;
  const __amdgpu_buffer_rsrc_t ir = __builtin_amdgcn_make_buffer_rsrc((void*)in, 0, (int)p.inBytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc((void*)bank, 0, (int)p.bankBytes, 0x00020000);

  // ---- loader: wavefront w fetches pixels 32 (w & 1) ... of channels (w >> 1), (w >> 1) + 2, ...; its pixel is lane / 2
  int ih0, iw0;
  unsigned pix;
  {
    const int m = mt * 64 + 32 * (wave & 1) + (lane >> 1);
    int n, q, ow, oh;
    p.byQ.divmod(m < p.M ? m : 0, &n, &q);
    p.byOH.divmod(q, &ow, &oh);
    ih0 = m < p.M ? oh * p.sy : -0x40000000;  // (never inside)
    iw0 = ow * p.sx;
    pix = (unsigned)(n * p.inImg + oh * p.sy + p.IH * iw0) * 8u + (lane & 1) * 4u;
  }
  int stageL = 0, chunkL = 0, tapL = 0, rowL = 0, dh = p.dhBase, dw = p.dwBase;
  unsigned vo = kOutside;
  float* dst = smem;
  int firstRow = 0, bankAt = 0;
  auto prep = [&]() {  // offsets of the next stage, then on to the one after it (past the last one nothing is fetched)
    const bool live = stageL < p.stages;
    const bool ok = live && (unsigned)(ih0 + dh) < (unsigned)p.IH && (unsigned)(iw0 + dw) < (unsigned)p.IW;
    vo = ok ? pix + (unsigned)((dh + p.IH * dw) * 8) : kOutside;
    firstRow = chunkL * 16;
    bankAt = live ? (ct * p.stages + stageL) * (kStageDoubles * 8) : (int)kOutside;
    dst = smem + (stageL & 1) * kStageFloats;
    ++stageL;
    dh += p.dhStep;
    if (++rowL == p.FH) {
      rowL = 0;
      dh = p.dhBase;
      dw += p.dwStep;
    }
    if (++tapL == p.T) {
      tapL = rowL = 0;
      dh = p.dhBase;
      dw = p.dwBase;
      ++chunkL;
    }
  };
  auto issue = [&](int t) {  // loads 0 ... 7: pixels; 8 ... 15: the bank, half a row of 64 channels each
    typedef __attribute__((address_space(3))) void* lds_ptr;
    const int r = 2 * (t & 7) + (wave >> 1), half = wave & 1;
    if (t < 8) {
      const int row = firstRow + r;
      const bool present = !RAGGED || row < p.Cin;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ir, (lds_ptr)(dst + r * kRowFloats + 64 * half), 4, present ? (int)vo : (int)kOutside,
                                               min(row, p.Cin - 1) * plane8, 0, 0);
    } else {
      const int voB = bankAt < 0 ? (int)kOutside : lane * 4;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(br, (lds_ptr)(dst + kOperandFloats + r * kRowFloats + 64 * half), 4, voB,
                                               bankAt < 0 ? 0 : bankAt + (r * 64 + 32 * half) * 8, 0, 0);
    }
  };

  doublex4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (doublex4){0.0, 0.0, 0.0, 0.0};
  const int l16 = lane & 15, lk = lane >> 4;
  prep();
#pragma unroll
  for (int t = 0; t < 16; ++t) issue(t);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll 1
  for (int s = 0; s < p.stages; ++s) {
    prep();
    const float* at = smem + (s & 1) * kStageFloats;
    const float* Ab = at + kOperandFloats + lk * kRowFloats + (32 * wc + l16) * 2;
    const float* Bb = at + lk * kRowFloats + (32 * wp + l16) * 2;
    double a[2][2], b[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      a[0][i] = *(const double*)(Ab + 32 * i);
      b[0][i] = *(const double*)(Bb + 32 * i);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int cur = k & 1, nxt = cur ^ 1;
      if (k < 3) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a[nxt][i] = *(const double*)(Ab + 32 * i + 4 * (k + 1) * kRowFloats);
          b[nxt][i] = *(const double*)(Bb + 32 * i + 4 * (k + 1) * kRowFloats);
        }
      }
      // (all out in the first half of the stage: they have the second to land in)
#pragma unroll
      for (int t = 8 * k; t < 8 * k + 8 && t < 16; ++t) issue(t);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[cur][i], b[cur][j], acc[i][j], 0, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }

  // ---- acc[i][j][e]: channel lane / 16 + 4 e of block i, pixel lane % 16 of block j
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int m = mt * 64 + 32 * wp + 16 * j + l16;
    if (m >= p.M) continue;
    int n, q;
    p.byQ.divmod(m, &n, &q);
    double* o = out + (size_t)n * p.outImg + q;
    const int Q = p.OH * p.OW;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int co = ct * 64 + 32 * wc + 16 * i + lk + 4 * e;
        if (co >= p.Cout) continue;
        const size_t at = (size_t)co * Q;
        double v = p.alpha * acc[i][j][e];
        if (p.beta != 0.0) v = fma(p.beta, o[at], v);
        if (bias) v += bias[co];
        o[at] = v;
      }
  }
}

// The bank: a workgroup per stage and tile of 64 output channels.  forward: w[co, ci, t] = f[t + T (ci + C co)], C channels in;
// backward: the filter is the channel in, f[t + T (co + C ci)], C channels out.
__global__ __launch_bounds__(256) void conv64_pack(double* __restrict__ bank, const double* __restrict__ f, int Cin, int Cout, int T, int stages,
                                                   int backward) {
  const int ct = blockIdx.x / stages, stage = blockIdx.x - ct * stages;
  const int chunk = stage / T, t = stage - chunk * T;
  for (int i = threadIdx.x; i < kStageDoubles; i += 256) {
    const int co = ct * 64 + (i & 63), ci = chunk * 16 + (i >> 6);
    double v = 0.0;
    if (co < Cout && ci < Cin) v = f[(size_t)t + (size_t)T * (backward ? (size_t)co + (size_t)Cout * ci : (size_t)ci + (size_t)Cin * co)];
    bank[(size_t)blockIdx.x * kStageDoubles + i] = v;
  }
}

}  // namespace

size_t conv64_pix_bank_bytes(const ConvP& p, bool backward) {
  const int Cin = backward ? p.Kg : p.FC, Cout = backward ? p.FC : p.Kg;
  return (size_t)((Cin + 15) / 16) * p.FH * p.FW * ((Cout + 63) / 64) * kStageDoubles * sizeof(double);
}

// Enough work that the bank's launch does not show (about 5 us), at least 16 channels either way (fewer leave most of a chunk or
// a tile to zeros), tensors and bank below the offset that loads nothing.  Where the general kernel takes a group with unit
// strides it is the faster one for reductions that a quarter of padding rows lengthens (3x3x34 -> 96 on 28x28x8 31 us, 35 here;
// 24 -> 64 on 56x56x8 34 and 38; 66 -> 256 214 and 209), and while it takes less than a call that gets its bank from the pool
// costs the host (1x1x96 -> 64 on 56x56x8 19 us, 38 here; 256 -> 98 on 28x28x8 26 and 38, on 56x56x8 59 and 50): its time is
// about 0.07 us per row of the reduction and 0.0002 per row and tile.  With strides or dilation it is slower, half of padding
// rows are too many (5x5x17 -> 83, dilated, on 60x60x2 40 us, 53 here).
bool conv64_pix_takes(const ConvP& p, bool backward) {
  const long long in = backward ? (long long)p.outH * p.outW * p.K * p.N : (long long)p.H * p.W * p.C * p.N;
  const long long pixels = backward ? (long long)p.H * p.W * p.N : (long long)p.outH * p.outW * p.N;
  if (tunable("conv64_no_mfma", 0) || tunable("conv64_no_pix", 0) || (backward && (p.sy != 1 || p.sx != 1))) return false;
  if (p.FC < 16 || p.Kg < 16 || in * 8 >= (long long)kOutside || pixels >= (1ll << 30) || conv64_pix_bank_bytes(p, backward) >= (size_t)kOutside) return false;
  if (p.outH * p.outW == 0 || 2.0 * pixels * p.FH * p.FW * p.FC * p.K < 2e8) return false;
  if (p.groups != 1 || tunable("conv_any_size", 0)) return true;
  const int Cin = backward ? p.Kg : p.FC, Cout = backward ? p.FC : p.Kg;
  if (p.sy != 1 || p.sx != 1 || p.dy != 1 || p.dx != 1) return (Cin + 15) / 16 * 16 * 2 <= 3 * Cin;
  const double tiles = (double)((pixels + 63) / 64) * ((Cout + 63) / 64), rows = (double)p.FH * p.FW * Cin;
  return (Cin + 15) / 16 * 16 * 4 <= 5 * Cin && rows * (0.07 + 0.0002 * tiles) >= 40.0;
}

// One filter group: pointers at the group's first channel; the bank is packed here.
int conv64_pix_launch(hipStream_t s, const char* who, const ConvP& p, bool backward, double* out, const double* in, const double* f,
                      const double* bias, double alpha, double beta, double* bank) {
  Pix64P q;
  q.IH = backward ? p.outH : p.H; q.IW = backward ? p.outW : p.W; q.Cin = backward ? p.Kg : p.FC;
  q.OH = backward ? p.H : p.outH; q.OW = backward ? p.W : p.outW; q.Cout = backward ? p.FC : p.Kg;
  q.T = p.FH * p.FW; q.FH = p.FH;
  q.sy = backward ? 1 : p.sy; q.sx = backward ? 1 : p.sx;
  q.dhBase = backward ? p.pt : -p.pt; q.dhStep = backward ? -p.dy : p.dy;
  q.dwBase = backward ? p.pl : -p.pl; q.dwStep = backward ? -p.dx : p.dx;
  const int Q = q.OH * q.OW;
  q.M = Q * p.N;
  q.stages = (q.Cin + 15) / 16 * q.T;
  q.inImg = (backward ? p.K : p.C) * q.IH * q.IW;
  q.outImg = (backward ? p.C : p.K) * Q;
  q.inBytes = (unsigned)(((long long)(p.N - 1) * q.inImg + (long long)q.Cin * q.IH * q.IW) * 8);
  q.bankBytes = (unsigned)conv64_pix_bank_bytes(p, backward);
  q.alpha = alpha; q.beta = beta;
  const int tilesC = (q.Cout + 63) / 64;
  q.byQ = FastDiv(Q);
  q.byOH = FastDiv(q.OH);
  q.byTilesC = FastDiv(tilesC);
  {
    KernelTimer timer("conv64_pack", s);
    hipLaunchKernelGGL(conv64_pack, dim3((unsigned)(tilesC * q.stages)), dim3(256), 0, s, bank, f, q.Cin, q.Cout, q.T, q.stages, backward ? 1 : 0);
  }
  KernelTimer timer("conv64_pix_mfma", s);
  const dim3 grid((unsigned)((q.M + 63) / 64 * tilesC));
  if (q.Cin % 16) hipLaunchKernelGGL(conv64_pix_mfma<true>, grid, dim3(256), 0, s, out, in, bank, bias, q);
  else hipLaunchKernelGGL(conv64_pix_mfma<false>, grid, dim3(256), 0, s, out, in, bank, bias, q);
  return check_launch(who);
}

}  // namespace mcn
