// Filter-gradient product on the bf16 matrix instruction with operands split in three:
//   dF[R, k] = sum_m xg[R, m] * dzdy[k, m],  xg = the (never materialised) patch matrix, m = the output pixels of all images.
//
// The numbers are those of conv_split.hip: a float is the sum of three bf16 numbers, six of the nine products of two floats
// reach the last place of fp32, the five small ones have accumulators of their own (the same time: two workgroups to a CU as
// with one set), and a workgroup that finds an accumulator that is not finite does its tile again on the
// fp32 instruction.  What differs is where the operands come from: both have the reduction (pixels) contiguous in memory,
// which is what a lane of the matrix instruction wants (eight reduction steps of one row).
//   * Loads go straight into LDS, a row of 32 pixels per half-wave: 32 neighbouring pixels are one to three runs of memory
//     whatever the tap, the stride or the image's edges do to their addresses.  A load holds rows r and r + 16 of a block of
//     32; they lie side by side, such pairs 68 floats apart, so that the 16-byte reads of eight lanes fall into 32 banks.
//   * A lane reads eight pixels of its row from there and splits them in registers.  In a 64 x 64 block per wavefront that is
//     208 vector instructions beside 24 matrix instructions per 16 pixels: the vector unit is busy 832 cycles to the matrix
//     pipe's 768.  Two workgroups to a CU overlap the two; inside a wavefront the second half of a step is split between
//     the matrix instructions of the first half, the next step's loads stand between those of the second.
//   * Rows are tap-major in half-blocks of 16 channels.  Where 16 does not divide the channels (or the filters), the last
//     half-block starts 16 before the end: its first rows are computed twice, and stored from the half-block before (the
//     two may lie in different workgroups, of which one may have taken the fp32 instruction).
// What bounds it: the matrix pipe and the power it draws (conv_split.hip).
#include "conv_common.hpp"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace mcn {
namespace {

constexpr int kPair = 68;               // floats from one pair of rows to the next
constexpr int kBlockFloats = 16 * kPair;  // 32 rows x 32 pixels
constexpr int kStep = 32;               // pixels of a step

struct WsP {
  int H, W, C, K;
  int OH, OW, FH;
  int sy, sx, pt, pl, dly, dlx;
  int FV;
  int M;                       // output pixels of all images (< 2^31)
  int halves;                  // half-blocks of 16 rows: taps x ceil(C / 16)
  int chunkSpan;               // pixels per split (a multiple of 32)
  int xImg, dyImg;             // elements between images of x and of dzdy
  unsigned xBytes, dyBytes;    // bytes this product may read of each (< 2 GiB)
  unsigned outBytes;           // size of the partial banks, or 0 when they do not fit a 2 GiB buffer descriptor
  FastDiv byQ, byOH, byFH, byTiles, byTilesK, byHalves;  // byHalves: half-blocks per tap
};

constexpr int wsplit_buffers(int blocks, bool deep) { return blocks <= 6 || deep ? 3 : 2; }

template <int WA, int WB, int NWA, int NWB, bool DEEP>
__global__ __launch_bounds__(256, 2) void conv_wgrad_mfma_split(float* __restrict__ out, const float* __restrict__ x,
                                                           const float* __restrict__ dy, WsP p) {
  static_assert(NWA * NWB == 4, "four wavefronts per workgroup");
  constexpr int ABLK = WA * NWA, BBLK = WB * NWB;  // blocks of 32 filters, of 32 filter-volume rows
  constexpr int NBUF = wsplit_buffers(ABLK + BBLK, DEEP);
  constexpr int BUF = (ABLK + BBLK) * kBlockFloats;
  constexpr int NLOADS = 4 * (ABLK + BBLK);        // per wavefront and step
  constexpr int FR = WA + WB;
  extern __shared__ float smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, kh = lane >> 5;
  const int wa = wave / NWB, wb = wave - wa * NWB;

  const int logical = xcd_contiguous_id(blockIdx.x, gridDim.x);
  int split, tile, rt, kt;
  p.byTiles.divmod(logical, &split, &tile);
  p.byTilesK.divmod(tile, &rt, &kt);
  const int HW = p.H * p.W, Q = p.OH * p.OW;
  const int mBegin = split * p.chunkSpan;
  const int mEnd = min(mBegin + p.chunkSpan, p.M);
  const int nSteps = mEnd > mBegin ? (mEnd - mBegin + kStep - 1) / kStep : 0;

  // ---- the loader: this lane's pixel, and per block of 32 rows the half-block (lane / 32) it fetches from
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, (int)p.xBytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc((void*)dy, 0, (int)p.dyBytes, 0x00020000);
  // tap and first channel of half-block h of the volume
  auto half_block = [&](int h, int* dh, int* dw, int* t, int* cb) {
    int j, i, part;
    p.byHalves.divmod(h < p.halves ? h : 0, t, &part);
    p.byFH.divmod(*t, &j, &i);
    *dh = i * p.dly - p.pt;
    *dw = j * p.dlx - p.pl;
    *cb = min(16 * part, p.C - 16);
  };
  auto filter_base = [&](int h) { return min(16 * h, p.K - 16); };
  int blkDh[BBLK], blkDw[BBLK];
  unsigned blkX[BBLK], blkY[ABLK];
#pragma unroll
  for (int b = 0; b < BBLK; ++b) {
    const int h = 2 * (rt * BBLK + b) + kh;
    int dh, dw, t, cb;
    half_block(h, &dh, &dw, &t, &cb);
    blkDh[b] = h < p.halves ? dh : -0x40000000;  // absent: never inside the image
    blkDw[b] = dw;
    blkX[b] = (unsigned)((cb * HW + dh + p.H * dw) * 4);
  }
#pragma unroll
  for (int a = 0; a < ABLK; ++a) blkY[a] = (unsigned)(filter_base(2 * (kt * ABLK + a) + kh) * Q) * 4u;

  unsigned voX[BBLK], voY[ABLK];
  int bufL = 0, bufAt = 0;
  auto prep = [&](int step) {  // (a step that does not exist fetches nothing: the counts of loads in flight stay exact)
    const int m = mBegin + step * kStep + (lane & 31);
    const bool valid = m < mEnd;
    int n, q, ow, oh;
    p.byQ.divmod(valid ? m : mBegin, &n, &q);
    p.byOH.divmod(q, &ow, &oh);
    const int ihB = oh * p.sy, iwB = ow * p.sx;
    const unsigned pixX = (unsigned)(n * p.xImg + ihB + p.H * iwB) * 4u;
    const unsigned pixY = (unsigned)(n * p.dyImg + q) * 4u;
#pragma unroll
    for (int b = 0; b < BBLK; ++b) {
      const bool ok = valid && (unsigned)(ihB + blkDh[b]) < (unsigned)p.H && (unsigned)(iwB + blkDw[b]) < (unsigned)p.W;
      voX[b] = ok ? pixX + blkX[b] : kOutside;
    }
#pragma unroll
    for (int a = 0; a < ABLK; ++a) voY[a] = valid ? pixY + blkY[a] : kOutside;
    bufAt = bufL * BUF;
    bufL = bufL == NBUF - 1 ? 0 : bufL + 1;
  };
  auto issue = [&](int t) {  // load t of a step: pair wave + 4 (t % 4) of block t / 4 (dzdy's blocks behind x's)
    typedef __attribute__((address_space(3))) void* lds_ptr;
    const int b = t / 4, row = wave + 4 * (t % 4);
    float* dst = smem + bufAt + b * kBlockFloats + row * kPair;
    if (b < BBLK) __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)dst, 4, (int)voX[b], row * HW * 4, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(yr, (lds_ptr)dst, 4, (int)voY[b - BBLK], row * Q * 4, 0, 0);
  };

  floatx16 acc[WA][WB], low[WA][WB];  // the products h h; the other five
  typedef union { uintx4 u; bf16x8 v; } frag;
  struct Parts { frag h, m, l; };
  typedef float v8f __attribute__((ext_vector_type(8)));

  const int laneAt = (l32 & 15) * kPair + (l32 >> 4) * 32 + 8 * kh;
  // fragment f (filters first) of half-step s: eight pixels of this lane's row
  auto read_raw = [&](int buf, int s, int f) -> v8f {
    const int b = f < WA ? BBLK + wa * WA + f : wb * WB + (f - WA);
    const float* at = smem + buf * BUF + b * kBlockFloats + laneAt + 16 * s;
    const v4f lo = *(const v4f*)at, hi = *(const v4f*)(at + 4);
    return (v8f){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto split8 = [&](const v8f& v) {
    Parts o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned h, m, l;
      split_pair(v[2 * j] * kSplitScale, v[2 * j + 1] * kSplitScale, &h, &m, &l);
      o.h.u[j] = h;
      o.m.u[j] = m;
      o.l.u[j] = l;
    }
    return o;
  };
  // One product of a half-step: i counts the 6 WA WB matrix instructions, small products first
  auto multiply = [&](int i, const Parts (&c)[FR]) {
    const int term = i / (WA * WB), a = (i % (WA * WB)) / WB, b = i % WB;
    const Parts &A = c[a], &B = c[WA + b];
    switch (term) {
      case 0: low[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.l.v, B.h.v, low[a][b], 0, 0, 0); break;
      case 1: low[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.h.v, B.l.v, low[a][b], 0, 0, 0); break;
      case 2: low[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.m.v, B.m.v, low[a][b], 0, 0, 0); break;
      case 3: low[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.m.v, B.h.v, low[a][b], 0, 0, 0); break;
      case 4: low[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.h.v, B.m.v, low[a][b], 0, 0, 0); break;
      default: acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.h.v, B.h.v, acc[a][b], 0, 0, 0); break;
    }
    if (term < 5) asm volatile("" : "+v"(low[a][b]));
    else asm volatile("" : "+v"(acc[a][b]));
  };

  auto pass = [&](auto fp32C) {
    constexpr bool FP32 = decltype(fp32C)::value;
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = low[a][b][r] = 0.f;
    bufL = 0;
#pragma unroll
    for (int s = 0; s < NBUF - 1; ++s) {
      prep(s);
#pragma unroll
      for (int t = 0; t < NLOADS; ++t) issue(t);
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NLOADS * (NBUF - 2)) : "memory");
    int buf = 0;
#pragma unroll 1
    for (int step = 0; step < nSteps; ++step) {
      prep(step + NBUF - 1);
      if constexpr (FP32) {
#pragma unroll
        for (int t = 0; t < NLOADS; ++t) issue(t);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          v8f raw[FR];
#pragma unroll
          for (int f = 0; f < FR; ++f) raw[f] = read_raw(buf, s, f);
#pragma unroll
          for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int a = 0; a < WA; ++a)
#pragma unroll
              for (int b = 0; b < WB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(raw[a][j], raw[WA + b][j], acc[a][b], 0, 0, 0);
        }
      } else {
        constexpr int MM = 6 * WA * WB, STAGES = 28 * FR;
        Parts cur[FR], next[FR];
        v8f raw[FR];
#pragma unroll
        for (int f = 0; f < FR; ++f) raw[f] = read_raw(buf, 0, f);
#pragma unroll
        for (int f = 0; f < FR; ++f) cur[f] = split8(raw[f]);
#pragma unroll
        for (int f = 0; f < FR; ++f) raw[f] = read_raw(buf, 1, f);
        __builtin_amdgcn_sched_barrier(0);
        float r0 = 0.f, r1 = 0.f;
        auto stage = [&](int k) {  // a seventh of the splitting of two numbers (see conv_split.hip)
          const int f = k / 28, j = k / 7 % 4;
          Parts& n = next[f];
          const float u = raw[f][2 * j], v = raw[f][2 * j + 1];
          switch (k % 7) {
            case 0: n.h.u[j] = round_pair(u * kSplitScale, v * kSplitScale); asm volatile("" : "+v"(n.h.u[j])); break;
            case 1: r0 = fmaf(u, kSplitScale, -__builtin_bit_cast(float, n.h.u[j] << 16)); asm volatile("" : "+v"(r0)); break;
            case 2: r1 = fmaf(v, kSplitScale, -__builtin_bit_cast(float, n.h.u[j] & 0xffff0000u)); asm volatile("" : "+v"(r1)); break;
            case 3: n.m.u[j] = round_pair(r0, r1); asm volatile("" : "+v"(n.m.u[j])); break;
            case 4: r0 -= __builtin_bit_cast(float, n.m.u[j] << 16); asm volatile("" : "+v"(r0)); break;
            case 5: r1 -= __builtin_bit_cast(float, n.m.u[j] & 0xffff0000u); asm volatile("" : "+v"(r1)); break;
            default: n.l.u[j] = round_pair(r0, r1); asm volatile("" : "+v"(n.l.u[j])); break;
          }
        };
#pragma unroll
        for (int i = 0; i < MM; ++i) {
          multiply(i, cur);
#pragma unroll
          for (int k = i * STAGES / MM; k < (i + 1) * STAGES / MM; ++k) stage(k);
#pragma unroll
          for (int t = i * NLOADS / MM; t < (i + 1) * NLOADS / MM; ++t) issue(t);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < MM; ++i) multiply(i, next);
      }
      // the next step's loads have landed (with three buffers those issued in this step may be in flight), this
      // wavefront's own reads are done
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"(NLOADS * (NBUF - 2)) : "memory");
      buf = buf == NBUF - 1 ? 0 : buf + 1;
    }
    if constexpr (!FP32) {
#pragma unroll
      for (int a = 0; a < WA; ++a)
#pragma unroll
        for (int b = 0; b < WB; ++b) acc[a][b] = (acc[a][b] + low[a][b]) * kSplitUnscale;
    }
  };
  pass(std::false_type());
  {
    float t = 0.f;
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) t = fmaf(acc[a][b][r], 0.f, t);
    // (every load into LDS has landed before the next pass's first one is issued)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (__builtin_expect(__syncthreads_or(!(t == 0.f)), 0)) pass(std::true_type());
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  // ---- epilogue: lane = row of the volume, register = filter
  const size_t bank = (size_t)split * p.FV * p.K;
#pragma unroll
  for (int b = 0; b < WB; ++b) {
    const int h = 2 * (rt * BBLK + wb * WB + b) + (l32 >> 4);
    int dh, dw, t, cb;
    half_block(h, &dh, &dw, &t, &cb);
    const int R = cb + (l32 & 15) + p.C * t;
    const int part = h - p.byHalves.div(h < p.halves ? h : 0) * p.byHalves.d;
    const bool present = h < p.halves && cb + (l32 & 15) >= 16 * part;  // (the half-block before stores the others)
#pragma unroll
    for (int a = 0; a < WA; ++a) {
      const int hk = 2 * (kt * ABLK + wa * WA + a);
      if (16 * hk >= p.K) continue;  // (a block of copies only)
      const int kb[2] = {filter_base(hk), filter_base(hk + 1)};
      auto stored = [&](int r) { return kb[r / 8] + 8 * (r / 4 % 2) + 4 * kh + r % 4 >= 16 * (hk + r / 8); };  // (likewise)
      if (p.outBytes != 0) {
        const bufrsrc rsrc = make_bufrsrc(out, p.outBytes);
        const int plane = p.FV * 4;
        const unsigned vo = present ? (unsigned)(R + 4 * kh * p.FV) * 4u : kOutside;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          buffer_store_untracked(acc[a][b][r], stored(r) ? vo : kOutside, rsrc, (split * p.K + kb[r / 8] + 8 * (r / 4 % 2) + r % 4) * plane);
      } else if (present) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (stored(r)) out[bank + (size_t)p.FV * (kb[r / 8] + 8 * (r / 4 % 2) + 4 * kh + r % 4) + R] = acc[a][b][r];
      }
    }
  }
}

template <int WA, int WB, int NWA, int NWB, bool DEEP>
int launch(hipStream_t s, unsigned blocks, float* out, const float* x, const float* dy, const WsP& p) {
  constexpr int BLK = WA * NWA + WB * NWB;
  constexpr size_t lds = (size_t)wsplit_buffers(BLK, DEEP) * BLK * kBlockFloats * sizeof(float);
  // Beside another stream's kernels the launch asks for more local memory than it uses, so that a CU holds one of its
  // workgroups and the other stream keeps the rest (see launch_wgrad).
  const size_t ask = stream_beside(s) ? std::max(lds, (size_t)84 * 1024) : lds;
  if (ask > 64 * 1024) {
    static std::atomic<bool> raisedOn[kMaxDevices];  // opt-in to more than 64 KB of LDS per workgroup, once per device
    const int dev = current_device();
    const bool known = dev >= 0 && dev < kMaxDevices;
    if (!known || !raisedOn[dev].load(std::memory_order_acquire)) {
      if (hipFuncSetAttribute((const void*)conv_wgrad_mfma_split<WA, WB, NWA, NWB, DEEP>, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024) !=
          hipSuccess) {
        (void)hipGetLastError();
        return fail(MCN_DEVICE_ERROR, "mcn_conv_backward_filter: cannot reserve %zu bytes of LDS", ask);
      }
      if (known) raisedOn[dev].store(true, std::memory_order_release);
    }
  }
  KernelTimer timer("conv_wgrad_mfma_split", s);
  hipLaunchKernelGGL((conv_wgrad_mfma_split<WA, WB, NWA, NWB, DEEP>), dim3(blocks), dim3(256), ask, s, out, x, dy, p);
  return MCN_SUCCESS;
}

// Tile (blocks of 32 filters x blocks of 32 rows) and splits of the pixels.
struct Plan { int blkA, blkB, tilesA, tilesB, splits; };

Plan plan_wsplit(const ConvP& p) {
  const int halves = p.FH * p.FW * ((p.FC + 15) / 16), rowBlocks = (halves + 1) / 2, kBlocks = (p.K + 31) / 32;
  Plan q;
  q.blkA = kBlocks > 2 ? 4 : (kBlocks > 1 ? 2 : 1);
  q.blkB = 4;
  if (rowBlocks <= 2 && q.blkA >= 2) q.blkB = 2;
  // a volume that tiles of six blocks cover and tiles of four do not (3x3x64: 18 blocks, three tiles instead of five)
  else if (q.blkA == 2 && (rowBlocks + 5) / 6 * 6 < (rowBlocks + 3) / 4 * 4) q.blkB = 6;
  q.tilesA = (kBlocks + q.blkA - 1) / q.blkA;
  q.tilesB = (rowBlocks + q.blkB - 1) / q.blkB;
  const int tiles = q.tilesA * q.tilesB;
  const long long steps = ((long long)p.outH * p.outW * p.N + kStep - 1) / kStep;
  // two workgroups to a CU; one where its share of a 1x1 layer would be small with several banks to write (see wgrad_splits)
  const double flops = 2.0 * p.outH * p.outW * p.N * (double)p.FH * p.FW * p.FC * p.K;
  const bool small = p.FH * p.FW == 1 && flops < 5e9 && (tiles >= 4 || tiles == 1);
  long long s = std::max<long long>(1, (small ? 256 : 512) / tiles);
  s = std::min<long long>(s, std::max<long long>(1, steps / 4));
  q.splits = (int)s;
  return q;
}

}  // namespace

bool conv_wsplit_takes(const ConvP& p, long long xLayerElements, long long yLayerElements) {
  if (tunable("conv_no_ws", 0) || tunable("conv_no_uniform_tap", 0) || tunable("conv_wgrad_no_split", 0)) return false;
  if (p.FC < 16 || p.K < 16 || xLayerElements >= (1ll << 29) || yLayerElements >= (1ll << 29)) return false;
  if (p.outH * p.outW == 1 && p.H * p.W == 1) return false;  // (fully connected: its pixels are not neighbours in memory)
  // channels that leave more than a third of the half-blocks' rows twice computed: not worth it
  return 3 * ((p.FC + 15) / 16 * 16) <= 4 * p.FC || p.FH * p.FW == 1;
}

int conv_wsplit_splits(const ConvP& p) { return plan_wsplit(p).splits; }

int conv_wsplit_launch(hipStream_t s, const ConvP& p, int xImg, int dyImg, float* out, const float* x, const float* dy) {
  const Plan plan = plan_wsplit(p);
  WsP q;
  q.H = p.H; q.W = p.W; q.C = p.C; q.K = p.K;
  q.OH = p.outH; q.OW = p.outW; q.FH = p.FH;
  q.sy = p.sy; q.sx = p.sx; q.pt = p.pt; q.pl = p.pl; q.dly = p.dy; q.dlx = p.dx;
  q.FV = p.FH * p.FW * p.C;
  q.M = p.outH * p.outW * p.N;
  const int perTap = (p.C + 15) / 16;
  q.halves = p.FH * p.FW * perTap;
  const int steps = (q.M + kStep - 1) / kStep;
  q.chunkSpan = (steps + plan.splits - 1) / plan.splits * kStep;
  q.xImg = xImg;
  q.dyImg = dyImg;
  q.xBytes = (unsigned)(((long long)(p.N - 1) * xImg + (long long)p.C * p.H * p.W) * 4);
  q.dyBytes = (unsigned)(((long long)(p.N - 1) * dyImg + (long long)p.K * p.outH * p.outW) * 4);
  const unsigned long long ob = (unsigned long long)plan.splits * q.FV * p.K * sizeof(float);
  q.outBytes = ob < (1ull << 31) ? (unsigned)ob : 0u;
  const int tiles = plan.tilesA * plan.tilesB;
  q.byQ = FastDiv(p.outH * p.outW);
  q.byOH = FastDiv(p.outH);
  q.byFH = FastDiv(p.FH);
  q.byTiles = FastDiv(tiles);
  q.byTilesK = FastDiv(plan.tilesA);
  q.byHalves = FastDiv(perTap);
  const unsigned blocks = (unsigned)(tiles * plan.splits);
  const bool deep = (long long)blocks <= device_compute_units();
  if (plan.blkA == 4) {
    if (plan.blkB == 2) return launch<2, 1, 2, 2, false>(s, blocks, out, x, dy, q);
    return deep ? launch<2, 2, 2, 2, true>(s, blocks, out, x, dy, q) : launch<2, 2, 2, 2, false>(s, blocks, out, x, dy, q);
  }
  if (plan.blkA == 2) {
    if (plan.blkB == 2) return launch<1, 1, 2, 2, false>(s, blocks, out, x, dy, q);
    if (plan.blkB == 6) return launch<1, 3, 2, 2, false>(s, blocks, out, x, dy, q);
    return launch<2, 1, 1, 4, false>(s, blocks, out, x, dy, q);
  }
  return launch<1, 1, 1, 4, false>(s, blocks, out, x, dy, q);
}

}  // namespace mcn
