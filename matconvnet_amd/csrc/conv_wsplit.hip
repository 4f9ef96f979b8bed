// Filter-gradient product on the bf16 matrix instruction with operands split in three:
//   dF[R, k] = sum_m xg[R, m] * dzdy[k, m],  xg = the (never materialised) patch matrix, m = the output pixels of all images.
//
// The numbers are those of conv_split.hip: a float is the sum of three bf16 numbers, six of the nine products of two floats
// reach the last place of fp32, the five small ones have accumulators of their own, and a workgroup that finds an accumulator
// that is not finite does its tile again on the fp32 instruction.  What differs is where the operands come from: both have
// the reduction (pixels) contiguous in memory, which is what a lane of the matrix instruction wants (eight reduction steps
// of one row).  Rows are tap-major in half-blocks of 16 channels.  Where 16 does not divide the channels (or the filters), the
// last half-block starts 16 before the end: its first rows are computed twice, and stored from the half-block before (the two
// may lie in different workgroups, of which one may have taken the fp32 instruction).
//
// Both operands have to be split, and the splitting is what bounds the product: 52 vector instructions for a lane's eight
// floats, 208 beside the 24 matrix instructions of a 64 x 64 block.  A SIMD takes up to six vector instructions behind a matrix
// instruction for next to nothing and some four cycles for each further one.
//
// conv_wgrad_mfma_split_shared splits every operand once per workgroup (eight wavefronts) instead of once per wavefront.
//   * Pixels come from global memory straight into registers, lane = pixel (32 of them), half-wave = 8 of the 16 rows of a
//     unit, and are split there: 3.3 vector instructions to a matrix instruction in tiles of 128 x 256 instead of 8.7.  The
//     parts go to LDS, eight rows of a pixel in 16 bytes, and are read back transposed by ds_read_b64_tr_b16: 16 lanes read
//     four pixels of 16 rows and get four pixels of a row each.
//   * LDS holds two steps of 32 pixels.  Everything stands between the matrix instructions of the step before: the
//     fragments' reads a few products ahead, the splitting, its loads (into the registers that the splitting leaves: a step
//     ahead) and their offsets.  One barrier per step, before the last products: what they leave to read is the next step's.
//   * 3x3x256x256 over 56x56x256x64: 1.69 -> 1.17 ms (202 TFLOP/s), 5x5x48x128 over 27x27x128 197 -> 156 us, layers of
//     ResNet-50 at 32 images 35-64 -> 29-54 us.  The tile is part of what the bits depend on: the largest one sums as the kernel below
//     for the same splits of the pixels, the others set their sums aside every eight steps.
//     The matrix pipe is busy 0.65 of the time at 1.67 GHz (0.43 at 1.87 before): power, and waits at the barrier.
// conv_wgrad_mfma_split has every wavefront split the fragments it multiplies (four wavefronts).  It stays for tiles where
// the former would keep too few wavefronts busy (up to 32 filters, 64 x 64) or waste rows (3x3 over 64 channels: 18 blocks of
// rows are three tiles of six; 63 against 68 us over 56x56x64x32).
//   * Loads go straight into LDS, a row of 32 pixels per half-wave: 32 neighbouring pixels are one to three runs of memory
//     whatever the tap, the stride or the image's edges do to their addresses.  A load holds rows r and r + 16 of a block of
//     32; they lie side by side, such pairs 68 floats apart.
//   * A half-step's splitting stands between the matrix instructions of the half-step before it, the loads of a later step
//     between those of every other half-step; the barrier of a step stands in its middle.
#include "conv_common.hpp"

#include <algorithm>
#include <atomic>
#include <iterator>
#include <type_traits>
#include <utility>

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

// f(0), f(1) ... f(N - 1) as constants (a loop of this size is unrolled too late for arrays it indexes to stay in registers)
template <typename F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  each_of(static_cast<F&&>(f), std::make_integer_sequence<int, N>());
}

constexpr int wsplit_buffers(int blocks) { return blocks <= 6 ? 3 : 2; }

template <int WA, int WB, int NWA, int NWB>
__global__ __launch_bounds__(256, 2) void conv_wgrad_mfma_split(float* __restrict__ out, const float* __restrict__ x,
                                                           const float* __restrict__ dy, WsP p) {
  static_assert(NWA * NWB == 4, "four wavefronts per workgroup");
  constexpr int ABLK = WA * NWA, BBLK = WB * NWB;  // blocks of 32 filters, of 32 filter-volume rows
  constexpr int NBUF = wsplit_buffers(ABLK + BBLK);
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
  // Offsets of a step's loads, in PREP stages (a few instructions each, without branches: they stand between matrix
  // instructions).  A step that does not exist fetches nothing: the counts of loads in flight stay exact.
  constexpr int PREP = 4 + BBLK + ABLK;
  int mL = 0, qL = 0, ihL = 0, iwL = 0;
  bool validL = false;
  unsigned pixX = 0, pixY = 0;
  auto prep_stage = [&](int k, int step) {
    if (k == 0) {
      mL = mBegin + step * kStep + (lane & 31);
      validL = mL < mEnd;
      mL = validL ? mL : mBegin;
    } else if (k == 1) {
      int n;
      p.byQ.divmod(mL, &n, &qL);
      pixX = (unsigned)(n * p.xImg);
      pixY = (unsigned)(n * p.dyImg + qL) * 4u;
    } else if (k == 2) {
      int ow, oh;
      p.byOH.divmod(qL, &ow, &oh);
      ihL = oh * p.sy;
      iwL = ow * p.sx;
    } else if (k == 3) {
      pixX = (pixX + (unsigned)(ihL + p.H * iwL)) * 4u;
    } else if (k < 4 + BBLK) {
      const int b = k - 4;
      const bool ok = validL & ((unsigned)(ihL + blkDh[b]) < (unsigned)p.H) & ((unsigned)(iwL + blkDw[b]) < (unsigned)p.W);
      voX[b] = ok ? pixX + blkX[b] : kOutside;
    } else {
      const int a = k - 4 - BBLK;
      voY[a] = validL ? pixY + blkY[a] : kOutside;
    }
  };
  auto next_buffer = [&]() {
    bufAt = bufL * BUF;
    bufL = bufL == NBUF - 1 ? 0 : bufL + 1;
  };
  auto prep = [&](int step) {
#pragma unroll
    for (int k = 0; k < PREP; ++k) prep_stage(k, step);
    next_buffer();
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

  // The row of a block that a lane multiplies: row rowP of half-block rowQ.  A 16-byte read goes through the banks by quads of
  // lanes, 0, 3, 5, 6 of a half-wave first, then 1, 2, 4, 7: each four quads read one half-block, whose rows of 68 floats
  // fall into all 64 banks (in plain order every read took its cycles twice).
  const int rowP = (l32 >> 3) * 4 + (l32 & 3), rowQ = (l32 >> 2 ^ l32 >> 3 ^ l32 >> 4) & 1;
  const int laneAt = rowP * kPair + rowQ * 32 + 8 * kh;
  // fragment f (filters first) of half-step s: eight pixels of this lane's row
  auto read_raw = [&](int buf, int s, int f) -> v8f {
    const int b = f < WA ? BBLK + wa * WA + f : wb * WB + (f - WA);
    const float* at = smem + buf * BUF + b * kBlockFloats + laneAt + 16 * s;
    const v4f lo = *(const v4f*)at, hi = *(const v4f*)(at + 4);
    return (v8f){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto split8 = [&](const v8f& v, Parts& o) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned h, m, l;
      split_pair(v[2 * j] * kSplitScale, v[2 * j + 1] * kSplitScale, &h, &m, &l);
      o.h.u[j] = h;
      o.m.u[j] = m;
      o.l.u[j] = l;
    }
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

  // A half-step: the products of `c`, and between them the splitting of half-step `half` of buffer `buf` into `n`: its first
  // fragment is in `raw` already (LEAD = 0) or read now and split from matrix instruction LEAD on, the others are read a
  // fragment ahead.  Between the matrix instructions too: ISSUE: the loads of the step that was prepared; else the offsets of
  // the loads of step `loads`.
  constexpr int MM = 6 * WA * WB, STAGES = kSplitStages * FR;
  SplitStages stages;
  auto half_step = [&](const Parts (&c)[FR], Parts (&n)[FR], v8f (&raw)[2], int buf, int loads, auto halfC, auto leadC, auto issueC) __attribute__((always_inline)) {
    constexpr int HALF = decltype(halfC)::value, LEAD = decltype(leadC)::value;
    constexpr bool ISSUE = decltype(issueC)::value;
    if (LEAD) {
      raw[0] = read_raw(buf, HALF, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    auto stage = [&](int k) {
      const int f = k / kSplitStages;
      if (k % kSplitStages == 0 && f + 1 < FR) raw[(f + 1) & 1] = read_raw(buf, HALF, f + 1);
      stages.stage(k % kSplitStages, raw[f & 1], n[f].h.u, n[f].m.u, n[f].l.u, [](int) {});
    };
    each<MM>([&](auto iC) __attribute__((always_inline)) {
      constexpr int i = decltype(iC)::value;
      multiply(i, c);
      __builtin_amdgcn_sched_barrier(0);
      if (i >= LEAD) {
#pragma unroll
        for (int k = (i - LEAD) * STAGES / (MM - LEAD); k < (i - LEAD + 1) * STAGES / (MM - LEAD); ++k) stage(k);
      }
      if (ISSUE) {
#pragma unroll
        for (int t = i * NLOADS / MM; t < (i + 1) * NLOADS / MM; ++t) issue(t);
      } else {
#pragma unroll
        for (int k = i * PREP / MM; k < (i + 1) * PREP / MM; ++k) prep_stage(k, loads);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  auto pass = [&](auto fp32C) __attribute__((always_inline)) {
    constexpr bool FP32 = decltype(fp32C)::value;
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = low[a][b][r] = 0.f;
    bufL = 0;
    if constexpr (FP32) {  // (rare: a step at a time)
#pragma unroll 1
      for (int step = 0; step < nSteps; ++step) {
        bufL = 0;
        prep(step);
#pragma unroll
        for (int t = 0; t < NLOADS; ++t) issue(t);
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          v8f raw[FR];
#pragma unroll
          for (int f = 0; f < FR; ++f) raw[f] = read_raw(0, s, f);
#pragma unroll
          for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int a = 0; a < WA; ++a)
#pragma unroll
              for (int b = 0; b < WB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(raw[a][j], raw[WA + b][j], acc[a][b], 0, 0, 0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      }
    } else {
#pragma unroll
      for (int s = 0; s < NBUF; ++s) {
        prep(s);
#pragma unroll
        for (int t = 0; t < NLOADS; ++t) issue(t);
      }
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(std::min(63, NLOADS * (NBUF - 1))) : "memory");
      typedef std::integral_constant<int, 0> zero;
      typedef std::integral_constant<int, 1> one;
      typedef std::integral_constant<int, 2> two;
      Parts cur[FR], next[FR];
      v8f raw[2];
      each<FR>([&](auto f) { split8(read_raw(0, 0, f), cur[f]); });
      raw[0] = read_raw(0, 1, 0);
      int buf = 0;
#pragma unroll 1
      for (int step = 0; step < nSteps; ++step) {
        half_step(cur, next, raw, buf, step + NBUF, one(), zero(), std::false_type());
        // The next step's loads have landed (with three buffers those of the step behind it may be in flight), and every
        // wavefront is done with this step's buffer: the loads of the step NBUF ahead go there.
        next_buffer();
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"(NLOADS * (NBUF - 2)) : "memory");
        buf = buf == NBUF - 1 ? 0 : buf + 1;
        half_step(next, cur, raw, buf, 0, zero(), two(), std::true_type());
        raw[0] = read_raw(buf, 1, 0);
      }
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
  }

  // ---- epilogue: lane = row of the volume, register = filter
  const size_t bank = (size_t)split * p.FV * p.K;
#pragma unroll
  for (int b = 0; b < WB; ++b) {
    const int h = 2 * (rt * BBLK + wb * WB + b) + rowQ;
    int dh, dw, t, cb;
    half_block(h, &dh, &dw, &t, &cb);
    const int R = cb + rowP + p.C * t;
    const int part = h - p.byHalves.div(h < p.halves ? h : 0) * p.byHalves.d;
    const bool present = h < p.halves && cb + rowP >= 16 * part;  // (the half-block before stores the others)
#pragma unroll
    for (int a = 0; a < WA; ++a) {
      const int hk = 2 * (kt * ABLK + wa * WA + a);
      if (16 * hk >= p.K) continue;  // (a block of copies only)
      // register r: filter r of half-block kh, of the other one in the two quads of odd parity (rowP, rowQ of its row)
      auto filters = [&](int r) { return hk + (kh ^ (r / 4 == 1 || r / 4 == 2)); };
      auto stored = [&](int r) { return filter_base(filters(r)) + r >= 16 * filters(r); };  // (likewise)
      if (p.outBytes != 0) {
        const bufrsrc rsrc = make_bufrsrc(out, p.outBytes);
        const int plane = p.FV * 4;
        const unsigned vo[2] = {(unsigned)(R + filter_base(hk + kh) * p.FV) * 4u, (unsigned)(R + filter_base(hk + (kh ^ 1)) * p.FV) * 4u};
#pragma unroll
        for (int r = 0; r < 16; ++r)
          buffer_store_untracked(acc[a][b][r], present && stored(r) ? vo[r / 4 == 1 || r / 4 == 2] : kOutside, rsrc, (split * p.K + r) * plane);
      } else if (present) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (stored(r)) out[bank + (size_t)p.FV * (filter_base(filters(r)) + r) + R] = acc[a][b][r];
      }
    }
  }
}

// The product with every operand split once per workgroup.
template <int WA, int WB, int NWA, int NWB>
__global__ __launch_bounds__(64 * NWA * NWB, NWA * NWB / 4) void conv_wgrad_mfma_split_shared(float* __restrict__ out, const float* __restrict__ x,
                                                                    const float* __restrict__ dy, WsP p) {
  constexpr int NW = NWA * NWB;                    // wavefronts
  constexpr int ABLK = WA * NWA, BBLK = WB * NWB;  // blocks of 32 filters, of 32 filter-volume rows
  constexpr int UA = 2 * ABLK, UB = 2 * BBLK, UNITS = UA + UB;  // units of 16 rows: the filters' first
  // Units that a wavefront splits: USA of the filters, then those of the rows.  Where there are fewer units than wavefronts,
  // two wavefronts split and store the same one.
  constexpr int USA = (UA + NW - 1) / NW, US = USA + (UB + NW - 1) / NW;
  static_assert((UA % NW == 0 || NW % UA == 0) && (UB % NW == 0 || NW % UB == 0), "whole units per wavefront");
  constexpr int kPart = 1024, kUnit = 3 * kPart;   // bytes: 32 pixels x 16 rows of bf16; the three parts
  constexpr int BUF = UNITS * kUnit;
  constexpr int MM = 6 * WA * WB;                  // matrix instructions of a half-step
  extern __shared__ char parts[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, kh = lane >> 5;
  const int wa = wave / NWB, wb = wave - wa * NWB;
  const int firstA = wave % UA, firstB = wave % UB;  // this wavefront's first units, the others NW apart

  const int logical = xcd_contiguous_id(blockIdx.x, gridDim.x);
  int split, tile, rt, kt;
  p.byTiles.divmod(logical, &split, &tile);
  p.byTilesK.divmod(tile, &rt, &kt);
  const int HW = p.H * p.W, Q = p.OH * p.OW;
  const int mBegin = split * p.chunkSpan;
  const int mEnd = min(mBegin + p.chunkSpan, p.M);
  const int nSteps = mEnd > mBegin ? (mEnd - mBegin + kStep - 1) / kStep : 0;

  // ---- the loader: lane = pixel, half-wave = 8 rows of the unit
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, (int)p.xBytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc((void*)dy, 0, (int)p.dyBytes, 0x00020000);
  auto half_block = [&](int h, int* dh, int* dw, int* t, int* cb) __attribute__((always_inline)) {  // tap and first channel of half-block h of the volume
    int j, i, part;
    p.byHalves.divmod(h < p.halves ? h : 0, t, &part);
    p.byFH.divmod(*t, &j, &i);
    *dh = i * p.dly - p.pt;
    *dw = j * p.dlx - p.pl;
    *cb = min(16 * part, p.C - 16);
  };
  auto filter_base = [&](int h) __attribute__((always_inline)) { return min(16 * h, p.K - 16); };
  int unitDh[US], unitDw[US];  // (uniform)
  unsigned unitAt[US];
  each<US>([&](auto uC) __attribute__((always_inline)) {
    constexpr int u = decltype(uC)::value;
    if constexpr (u < USA) {
      unitAt[u] = (unsigned)((filter_base(2 * kt * ABLK + firstA + u * NW) + 8 * kh) * Q) * 4u;
    } else {
      const int h = 2 * rt * BBLK + firstB + (u - USA) * NW;
      int dh, dw, t, cb;
      half_block(h, &dh, &dw, &t, &cb);
      unitDh[u] = h < p.halves ? dh : -0x40000000;  // absent: never inside the image
      unitDw[u] = dw;
      unitAt[u] = (unsigned)(((cb + 8 * kh) * HW + dh + p.H * dw) * 4);
    }
  });
  // Offsets of a step's loads, in PREP stages of a few instructions (a step that does not exist fetches nothing)
  constexpr int PREP = 4;
  int mL = 0, qL = 0, ihL = 0, iwL = 0;
  bool validL = false;
  unsigned pixX = 0, pixY = 0, vo[US];
  auto prep_pixel = [&](auto kC, int step) __attribute__((always_inline)) {
    constexpr int k = decltype(kC)::value;
    if constexpr (k == 0) {
      mL = mBegin + step * kStep + l32;
      validL = mL < mEnd;
      mL = validL ? mL : mBegin;
    } else if constexpr (k == 1) {
      int n;
      p.byQ.divmod(mL, &n, &qL);
      pixX = (unsigned)(n * p.xImg);
      pixY = (unsigned)(n * p.dyImg + qL) * 4u;
    } else if constexpr (k == 2) {
      int ow, oh;
      p.byOH.divmod(qL, &ow, &oh);
      ihL = oh * p.sy;
      iwL = ow * p.sx;
    } else {
      pixX = (pixX + (unsigned)(ihL + p.H * iwL)) * 4u;
    }
  };
  auto prep_unit = [&](auto uC) __attribute__((always_inline)) {
    constexpr int u = decltype(uC)::value;
    if constexpr (u < USA) {
      vo[u] = validL ? pixY + unitAt[u] : kOutside;
    } else {
      const bool ok = validL & ((unsigned)(ihL + unitDh[u]) < (unsigned)p.H) & ((unsigned)(iwL + unitDw[u]) < (unsigned)p.W);
      vo[u] = ok ? pixX + unitAt[u] : kOutside;
    }
  };
  auto prep = [&](int step) __attribute__((always_inline)) {
    each<PREP>([&](auto k) __attribute__((always_inline)) { prep_pixel(k, step); });
    each<US>(prep_unit);
  };
  typedef float v8f __attribute__((ext_vector_type(8)));
  v8f raw[US];
  auto load_row = [&](auto uC, int j) __attribute__((always_inline)) -> float {
    constexpr int u = decltype(uC)::value;
    if constexpr (u < USA) return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(yr, (int)vo[u], j * Q * 4, 0));
    else return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, (int)vo[u], j * HW * 4, 0));
  };

  // The products h h; the other five.  An accumulator's error grows with the root of the pixels it has taken: where there are
  // registers for it, the sums of ASIDE steps go to `done` (tiles of 64 x 64 per wavefront have none: see plan_wsplit).
  constexpr bool ASIDE = WA * WB <= 2;
  constexpr int kAsideSteps = 8;
  floatx16 acc[WA][WB], low[WA][WB], done[ASIDE ? WA : 1][ASIDE ? WB : 1];
  typedef union { uintx4 u; bf16x8 v; } frag;
  struct Parts { frag h, m, l; };

  // ---- split operands in LDS.  Of each unit and part: rows 0-7 of 32 pixels, 16 bytes a pixel, then rows 8-15 with groups of
  // four pixels exchanged, in odd units groups of eight too: 16 lanes read 8 bytes each (four pixels' four quads of rows), 32
  // lanes of two neighbouring units all banks; eight lanes write 128 bytes side by side.
  const int odd = wave & 1;  // (of all this wavefront's units)
  const int putLane = kh * 512 + (l32 ^ (4 * kh) ^ (8 * odd)) * 16;
  const int putA = firstA * kUnit + putLane, putB = (UA + firstB) * kUnit + putLane;
  auto put = [&](int b, auto uC, const Parts& s) __attribute__((always_inline)) {
    constexpr int u = decltype(uC)::value;
    char* at = parts + b * BUF + (u < USA ? putA + u * (NW * kUnit) : putB + (u - USA) * (NW * kUnit));
    *(uintx4*)at = s.h.u;
    *(uintx4*)(at + kPart) = s.m.u;
    *(uintx4*)(at + 2 * kPart) = s.l.u;
  };
  const int getUnit = lane >> 4 & 1, getHalf = lane >> 1 & 1;
  const int getAt = getUnit * kUnit + getHalf * 512 + ((8 * kh + (lane >> 2 & 3)) ^ (4 * getHalf) ^ (8 * getUnit)) * 16 + (lane & 1) * 8;
  const int getAt2 = getAt ^ 64;  // the next four pixels
  typedef short short4v __attribute__((ext_vector_type(4)));
  typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
  // half `e` of the fragment of block `blk` (filters first) and part, half-step s
  auto get = [&](int b, int s, int blk, int part, int e, frag& f) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) short4v* lds_ptr;
    const char* at = parts + b * BUF + blk * (2 * kUnit) + part * kPart + s * 256 + (e ? getAt2 : getAt);
    const uintx2 v = __builtin_bit_cast(uintx2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)at));
    f.u[2 * e] = v[0];
    f.u[2 * e + 1] = v[1];
  };

  // One product of a half-step: i counts the matrix instructions, small products first
  struct Frags { frag Al[WA], Am[WA], Ah[WA], Bl[WB], Bm[WB], Bh[2][WB]; };
  auto multiply = [&](auto iC, const Frags& f, auto sC) __attribute__((always_inline)) {
    constexpr int i = decltype(iC)::value, s = decltype(sC)::value;
    constexpr int term = i / (WA * WB), a = (i % (WA * WB)) / WB, b = i % WB;
    floatx16& sum = term < 5 ? low[a][b] : acc[a][b];
    const bf16x8 A = term == 0 ? f.Al[a].v : term == 2 || term == 3 ? f.Am[a].v : f.Ah[a].v;
    const bf16x8 B = term == 1 ? f.Bl[b].v : term == 2 || term == 4 ? f.Bm[b].v : f.Bh[s][b].v;
    sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, B, sum, 0, 0, 0);
    asm volatile("" : "+v"(sum));
    __builtin_amdgcn_sched_barrier(0);
  };
  const int blkA = wa * WA, blkB = ABLK + wb * WB;
  // reads in the order they are needed, half a fragment each: l of the filters, h of the rows (before the half-step begins);
  // h and l (during its first products); m
  constexpr int READS = 2 * (WA + WB);
  auto read_first = [&](int r, int b, int s, Frags& f) __attribute__((always_inline)) {
    if (r < 2 * WA) get(b, s, blkA + r / 2, 2, r & 1, f.Al[r / 2]);
    else get(b, s, blkB + (r / 2 - WA), 0, r & 1, f.Bh[s][r / 2 - WA]);
  };
  auto read_second = [&](int r, int b, int s, Frags& f) __attribute__((always_inline)) {
    if (r < 2 * WA) get(b, s, blkA + r / 2, 0, r & 1, f.Ah[r / 2]);
    else get(b, s, blkB + (r / 2 - WA), 2, r & 1, f.Bl[r / 2 - WA]);
  };
  auto read_third = [&](int r, int b, int s, Frags& f) __attribute__((always_inline)) {
    if (r < 2 * WA) get(b, s, blkA + r / 2, 1, r & 1, f.Am[r / 2]);
    else get(b, s, blkB + (r / 2 - WA), 1, r & 1, f.Bm[r / 2 - WA]);
  };

#pragma unroll
  for (int a = 0; a < WA; ++a)
#pragma unroll
    for (int b = 0; b < WB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[a][b][r] = low[a][b][r] = 0.f;
        if (ASIDE) done[a][b][r] = 0.f;
      }
  auto set_aside = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int b = 0; b < WB; ++b) {
        if constexpr (ASIDE) {
          done[a][b] += acc[a][b];
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
        }
      }
  };
  {
    Frags f;
    SplitStages stages;
    Parts now[2];
    prep(0);
    each<US>([&](auto uC) __attribute__((always_inline)) {
      constexpr int u = decltype(uC)::value;
#pragma unroll
      for (int j = 0; j < 8; ++j) raw[u][j] = load_row(uC, j);
    });
    prep(1);
    each<US>([&](auto uC) __attribute__((always_inline)) {
      constexpr int u = decltype(uC)::value;
      Parts s;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        unsigned h, m, l;
        split_pair(raw[u][2 * j] * kSplitScale, raw[u][2 * j + 1] * kSplitScale, &h, &m, &l);
        s.h.u[j] = h;
        s.m.u[j] = m;
        s.l.u[j] = l;
        raw[u][2 * j] = load_row(uC, 2 * j);
        raw[u][2 * j + 1] = load_row(uC, 2 * j + 1);
      }
      put(0, uC, s);
    });
    prep(2);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int r = 0; r < READS; ++r) read_first(r, 0, 0, f);
    int buf = 0;
    // where the stages of splitting end, and the barrier stands, in a step's 2 MM matrix instructions
    constexpr int SPLIT_END = 2 * MM - 2 * WA * WB;
#pragma unroll 1
    for (int step = 0, stop = 0; step < nSteps;) {
    stop = ASIDE ? min(step + kAsideSteps, nSteps) : nSteps;
#pragma unroll 1
    for (; step < stop; ++step) {
      each<2 * MM>([&](auto iC) __attribute__((always_inline)) {
        constexpr int i = decltype(iC)::value, s = i / MM, k = i % MM, T = WA * WB;
        multiply(std::integral_constant<int, k>(), f, std::integral_constant<int, s>());
        // the fragments
        if constexpr (k < T) {
#pragma unroll
          for (int r = k * READS / T; r < (k + 1) * READS / T; ++r) read_second(r, buf, s, f);
        } else if constexpr (k < 2 * T) {
#pragma unroll
          for (int r = (k - T) * READS / T; r < (k - T + 1) * READS / T; ++r) read_third(r, buf, s, f);
        } else if constexpr (k >= 4 * T) {
#pragma unroll
          for (int r = (k - 4 * T) * READS / (2 * T); r < (k - 4 * T + 1) * READS / (2 * T); ++r) read_first(r, s ? buf ^ 1 : buf, s ^ 1, f);
        }
        // the next step's operands
        if constexpr (i < SPLIT_END) {
          each<(i + 1) * US * kSplitStages / SPLIT_END - i * US * kSplitStages / SPLIT_END>([&](auto gC) __attribute__((always_inline)) {
            constexpr int g = i * US * kSplitStages / SPLIT_END + decltype(gC)::value, u = g / kSplitStages, at = g % kSplitStages;
            constexpr auto uC = std::integral_constant<int, u>();
            stages.stage(at, raw[u], now[u & 1].h.u, now[u & 1].m.u, now[u & 1].l.u, [&](int j) __attribute__((always_inline)) {
              raw[u][2 * j] = load_row(uC, 2 * j);
              raw[u][2 * j + 1] = load_row(uC, 2 * j + 1);
            });
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (at == kSplitStages - 1) put(buf ^ 1, uC, now[u & 1]);
            // (offsets of the step after that: the pixel beside the first unit, a unit's as soon as its loads are issued)
            if constexpr (u == 0 && at >= 20 && at % 3 == 2 && at < 20 + 3 * PREP) prep_pixel(std::integral_constant<int, (at - 20) / 3>(), step + 3);
            if constexpr (u > 0 && at == 4) prep_unit(std::integral_constant<int, u - 1>());
            if constexpr (u == US - 1 && at == 24) prep_unit(uC);
          });
        }
        if constexpr (i == SPLIT_END - 1) {
          // the next step's operands are in LDS, and every wavefront has read all of this one's
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      buf ^= 1;
    }
    set_aside();
    }
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int b = 0; b < WB; ++b) {
        if constexpr (ASIDE) acc[a][b] += done[a][b];
        acc[a][b] = (acc[a][b] + low[a][b]) * kSplitUnscale;
      }
  }
  {
    float t = 0.f;
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) t = fmaf(acc[a][b][r], 0.f, t);
    if (__builtin_expect(__syncthreads_or(!(t == 0.f)), 0)) {
      // the tile again on the fp32 instruction, a step at a time: floats in the units' places, rows of 32 pixels
#pragma unroll
      for (int a = 0; a < WA; ++a)
#pragma unroll
        for (int b = 0; b < WB; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
#pragma unroll 1
      for (int step = 0; step < nSteps; ++step) {
        prep(step);
        each<US>([&](auto uC) __attribute__((always_inline)) {
          constexpr int u = decltype(uC)::value;
          float* at = (float*)(parts + (u < USA ? firstA + u * NW : UA + firstB + (u - USA) * NW) * kUnit) + 8 * kh * 32 + l32;
#pragma unroll
          for (int j = 0; j < 8; ++j) at[j * 32] = load_row(uC, j);
        });
        __syncthreads();
        auto row = [&](int blk) __attribute__((always_inline)) { return (const float*)(parts + (2 * blk + (l32 >> 4)) * kUnit) + (l32 & 15) * 32 + 8 * kh; };
#pragma unroll 1
        for (int k = 0; k < 16; ++k) {
          const int at = k / 8 * 16 + k % 8;
#pragma unroll
          for (int a = 0; a < WA; ++a)
#pragma unroll
            for (int b = 0; b < WB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(row(blkA + a)[at], row(blkB + b)[at], acc[a][b], 0, 0, 0);
        }
        __syncthreads();
      }
    }
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
      auto stored = [&](int r) __attribute__((always_inline)) { return kb[r / 8] + 8 * (r / 4 % 2) + 4 * kh + r % 4 >= 16 * (hk + r / 8); };  // (likewise)
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

template <int WA, int WB, int NWA, int NWB>
int launch(hipStream_t s, unsigned blocks, float* out, const float* x, const float* dy, const WsP& p) {
  constexpr int BLK = WA * NWA + WB * NWB;
  constexpr size_t lds = (size_t)wsplit_buffers(BLK) * BLK * kBlockFloats * sizeof(float);
  // Beside another stream's kernels the launch asks for more local memory than it uses, so that a CU holds one of its
  // workgroups and the other stream keeps the rest (see launch_wgrad).
  const size_t ask = stream_beside(s) ? std::max(lds, (size_t)84 * 1024) : lds;
  if (ask > 64 * 1024) {
    static std::atomic<bool> raisedOn[kMaxDevices];  // opt-in to more than 64 KB of LDS per workgroup, once per device
    const int dev = current_device();
    const bool known = dev >= 0 && dev < kMaxDevices;
    if (!known || !raisedOn[dev].load(std::memory_order_acquire)) {
      if (hipFuncSetAttribute((const void*)conv_wgrad_mfma_split<WA, WB, NWA, NWB>, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024) !=
          hipSuccess) {
        (void)hipGetLastError();
        return fail(MCN_DEVICE_ERROR, "mcn_conv_backward_filter: cannot reserve %zu bytes of LDS", ask);
      }
      if (known) raisedOn[dev].store(true, std::memory_order_release);
    }
  }
  KernelTimer timer(ask > lds ? "conv_wgrad_mfma_split_beside" : "conv_wgrad_mfma_split", s);
  hipLaunchKernelGGL((conv_wgrad_mfma_split<WA, WB, NWA, NWB>), dim3(blocks), dim3(256), ask, s, out, x, dy, p);
  return MCN_SUCCESS;
}

template <int WA, int WB, int NWA, int NWB>
int launch_shared(hipStream_t s, unsigned blocks, float* out, const float* x, const float* dy, const WsP& p) {
  constexpr size_t lds = (size_t)2 * 2 * (WA * NWA + WB * NWB) * 3072;
  // (beside another stream's kernels one workgroup to a CU, as above; the larger tiles have no room for a second anyway)
  constexpr size_t most = std::max(lds, (size_t)84 * 1024);
  const size_t ask = stream_beside(s) ? most : lds;
  static std::atomic<bool> raisedOn[kMaxDevices];  // opt-in to more than 64 KB of LDS per workgroup, once per device
  const int dev = current_device();
  const bool known = dev >= 0 && dev < kMaxDevices;
  if (!known || !raisedOn[dev].load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute((const void*)conv_wgrad_mfma_split_shared<WA, WB, NWA, NWB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most) !=
        hipSuccess) {
      (void)hipGetLastError();
      return fail(MCN_DEVICE_ERROR, "mcn_conv_backward_filter: cannot reserve %zu bytes of LDS", most);
    }
    if (known) raisedOn[dev].store(true, std::memory_order_release);
  }
  KernelTimer timer(ask > lds ? "conv_wgrad_mfma_split_shared_beside" : "conv_wgrad_mfma_split_shared", s);
  hipLaunchKernelGGL((conv_wgrad_mfma_split_shared<WA, WB, NWA, NWB>), dim3(blocks), dim3(64 * NWA * NWB), ask, s, out, x, dy, p);
  return MCN_SUCCESS;
}

// Tile (blocks of 32 filters x blocks of 32 rows) and splits of the pixels: those with the least modelled time.  The times are
// those of the layers of ResNet-50 at 32 images and of 3x3x256x256 over 56x56 at 64 in each tile (the model is mostly within
// 10 % of them): 4 x 4 is the best up to some 30 steps, 4 x 8 from there on.  Against the rule before (4 x 4 of wavefronts that
// split for themselves, two workgroups to a CU), with the sum of the partial banks: 1x1x256x1024 over 14x14x32 37 -> 31 us,
// 3x3x128x128 over 28x28x32 63 -> 55, 3x3x256x256 over 14x14x4 28 -> 23, 3x3x100x90 over 33x33x7 32 -> 24.
struct Tile {
  int a, b;
  bool shared;
  double start, one, full;  // us: a launch without its steps; a step of a workgroup alone on its CU, and of each of several
};
struct Plan { Tile tile; int tilesA, tilesB, splits; };

Plan plan_wsplit(const ConvP& p) {
  static const Tile tiles[] = {
      {4, 8, true, 12.5, 2.51, 2.51}, {4, 4, true, 9.5, 1.48, 1.48}, {8, 2, true, 11.0, 1.73, 1.73}, {4, 2, true, 8.5, 1.15, 1.12},
      {2, 8, true, 11.0, 1.73, 1.73}, {2, 4, true, 8.5, 1.10, 1.03}, {2, 6, false, 10.5, 2.20, 1.40},  {2, 2, false, 10.0, 0.75, 0.70},
      {1, 4, false, 8.5, 0.80, 0.48},
  };
  const int halves = p.FH * p.FW * ((p.FC + 15) / 16), rowBlocks = (halves + 1) / 2, kBlocks = (p.K + 31) / 32;
  const long long steps = ((long long)p.outH * p.outW * p.N + kStep - 1) / kStep;
  const double bankMB = 4e-6 * p.FH * p.FW * p.FC * p.K;
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  // Tiles whose sums are not set aside on the way (conv_wgrad_mfma_split_shared) keep their chains of pixels, and with them
  // their error, at what 128 x 128 tiles, two workgroups to a CU, have (one for small 1x1 layers with several banks to write).
  const int a0 = std::min(kBlocks > 2 ? 4 : kBlocks, 4);
  const int b0 = rowBlocks <= 2 && a0 >= 2 ? 2 : (a0 == 2 && (rowBlocks + 5) / 6 * 6 < (rowBlocks + 3) / 4 * 4 ? 6 : 4);
  const long long n0 = (long long)((kBlocks + a0 - 1) / a0) * ((rowBlocks + b0 - 1) / b0);
  const double flops = 2.0 * p.outH * p.outW * p.N * (double)p.FH * p.FW * p.FC * p.K;
  const bool small = p.FH * p.FW == 1 && flops < 5e9 && (n0 >= 4 || n0 == 1);
  const long long least = std::min(std::max(1ll, (small ? 256 : 512) / n0), std::max(1ll, steps / 4));
  int forced = tunable("conv_wsplit_tile", 0);
  if (std::none_of(std::begin(tiles), std::end(tiles), [&](const Tile& t) { return t.a * 10 + t.b == forced; })) forced = 0;
  Plan best;
  best.splits = 0;
  double bestUs = 0;
  for (const Tile& t : tiles) {
    const bool fits = (t.a == 8 ? kBlocks > 4 : t.a == (kBlocks > 2 ? 4 : kBlocks)) && (t.a == 1 || (rowBlocks <= 2) == (t.b == 2));
    if (forced ? t.a * 10 + t.b != forced : !fits) continue;
    Plan q;
    q.tile = t;
    q.tilesA = (kBlocks + t.a - 1) / t.a;
    q.tilesB = (rowBlocks + t.b - 1) / t.b;
    const long long n = (long long)q.tilesA * q.tilesB;
    for (int perCu = 1; perCu <= (t.shared ? 3 : 2); ++perCu) {
      long long s = std::max(1ll, std::min(perCu * (long long)cus / n, steps / 4));
      if (!t.shared || t.a * t.b > 16) s = std::max(s, least);
      const long long per = (steps + s - 1) / s;
      s = (steps + per - 1) / per;
      const long long busiest = (n * s + cus - 1) / cus;
      double us = t.start + (double)per * (busiest == 1 ? t.one : busiest * t.full);
      if (s > 1 || p.FH * p.FW > 1) us += 5.5 + 0.14 * bankMB * s;
      if (best.splits == 0 || us < bestUs) {
        bestUs = us;
        best = q;
        best.splits = (int)s;
      }
    }
  }
  return best;
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
  switch (plan.tile.a * 10 + plan.tile.b) {
    case 48: return launch_shared<2, 2, 2, 4>(s, blocks, out, x, dy, q);
    case 44: return launch_shared<2, 1, 2, 4>(s, blocks, out, x, dy, q);
    case 82: return launch_shared<2, 1, 4, 2>(s, blocks, out, x, dy, q);
    case 42: return launch_shared<1, 1, 4, 2>(s, blocks, out, x, dy, q);
    case 28: return launch_shared<1, 2, 2, 4>(s, blocks, out, x, dy, q);
    case 24: return launch_shared<1, 1, 2, 4>(s, blocks, out, x, dy, q);
    case 26: return launch<1, 3, 2, 2>(s, blocks, out, x, dy, q);
    case 22: return launch<1, 1, 2, 2>(s, blocks, out, x, dy, q);
    default: return launch<1, 1, 1, 4>(s, blocks, out, x, dy, q);
  }
}

}  // namespace mcn
