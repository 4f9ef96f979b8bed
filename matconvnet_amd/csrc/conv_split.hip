// Implicit-GEMM convolution on the bf16 matrix instruction with operands split in three (forward and backward-data).
//
// What bounds these products is the matrix pipe, and v_mfma_f32_32x32x2_f32 gives it 157 TFLOP/s, a sixteenth of what
// v_mfma_f32_32x32x16_bf16 does.  A float is the sum of three bf16 numbers, x = h + m + l, each the rounding of what
// the ones before leave: 24 bits of significand in three times 8, nothing is lost.  The product of two bf16 numbers is
// exact in fp32, so a b is the sum of nine exact products; the three smallest (m l, l m, l l) are together below 2^-26 of a b,
// under a quarter of a unit in the last place of one fp32 rounding, and are left out.  The other six go through the bf16 instruction
// with fp32 accumulators: 6 x 32 cycles of matrix time per 16 reduction rows of a 32 x 32 block instead of 8 x 64.
// The instruction adds eight products and its addend on a grid set by the largest of them and rounds ties down, so what
// counts is how often the large sum passes through it: the products h h have accumulators of their own, the five small ones
// (2^-8 and below of the sum) another set, added once at the end.  In one set all six rounded at the sum's last place, and
// with a bias: errors up to 1.3 times the fp32 instruction's where an operand is behind a ReLU, and channel means 12 sigma
// off zero.  Dot products of N(0,1) numbers against double, relative error (2-norm) over 64 / 576 / 2304 / 8192 rows: 0.50 /
// 0.86 / 1.10 / 1.49 e-7 here, 1.44 / 4.31 / 3.10 / 4.13 e-7 on the fp32 instruction; one operand behind a ReLU: 0.41 / 0.71 /
// 0.94 / 1.25 and 1.04 / 3.04 / 2.23 / 2.99 e-7; channel means within 1.1 sigma.  The second set costs a workgroup per CU
// where tiles are 128 wide (two left): 2 % of the time of ResNet-50's layers at 32 images, nothing for the large ones.
// Operands are scaled by 2^24 before they are split (kSplitScale), so that the parts of the smallest floats are numbers of
// bf16 too (unscaled, those below 2^-110 lost bits of l: error 2e-6 at 2^-116, all of it at 2^-140; two multiplications per
// pair, 2 to 4 % of the time).  Infinities, NaNs and magnitudes that scaling takes beyond bf16 (2^104) leave accumulators
// that are not finite: a wavefront that finds one does its block again on the fp32 instruction, which gives what fp32 gives.
//
// What bounds the large ones is power: a stream of the six products from registers alone reaches 298 TFLOP/s of fp32 work on
// N(0,1) operands and 408 on zeros (the fp32 instruction: 155), with the splitting of one operand beside it 299 and 281
// (8 floats to 24 and to 12 products).  3x3x256x256 on 56x56x256x64 on this kernel: 1.69 -> 1.04 ms (228 TFLOP/s), clock at 1.6 GHz;
// pixels staged for all taps (conv_staged.hpp), as that product runs, 0.94.
//
//   * a workgroup of four wavefronts owns 32 WA output channels x 128 pixels; each wavefront multiplies its own 32
//     pixels against all 32 WA channels, so the pixels are split once per wavefront and 16 rows (52 vector instructions
//     beside 24 matrix instructions for WA = 4);
//   * the pixel operand (lane = pixel, half-wave = 8 rows) comes from global memory straight into registers: eight buffer
//     loads of 32 consecutive pixels per half-wave, a slab (GPS groups of 16 rows) ahead; out-of-image lanes use an
//     offset beyond the tensor and get 0;
//   * the bank is split when it is packed (conv_pack_split) and lies in the order the fragments are read: 1 KB per
//     16 rows x 32 channels x part, lane by lane.  A slab of it goes from global memory straight into one of two LDS
//     buffers; a fragment read is 64 lanes x 16 consecutive bytes (no bank conflicts), half of the LDS bandwidth;
//   * one barrier per slab, behind a counted wait: the pixel loads of the next slab stay in flight across it.  It stands where
//     the slab's last fragments have been read, half a group of matrix instructions before its end: behind it the next slab's
//     first fragments are read and the slab after that is asked for while those products run, and a wavefront alone on its SIMD
//     does not stand before an empty matrix pipe at the head of each slab;
//   * where a lane's pixel lies under each tap is a table in LDS: worked out for every group, it was a row of 20 scalar
//     instructions, of which four are free behind a matrix instruction and each other costs 8 cycles.  Both together, one
//     workgroup to a CU: 72 groups of 3x3x256x256 over 14x14, 32 images 45.4 -> 40 us (1217 -> 1097 cycles each);
//   * what is not a matrix instruction stands between matrix instructions, pinned there (see `group`): products of few
//     workgroups, alone on their SIMDs, spend their time in what the compiler puts in front of the first one otherwise
//     (3x3x512x512 on 7x7x512x32, unsplit: 204 -> 147 us).
// Reduction order: chunks of 16 channels, the taps inside a chunk.
#include "conv_split.hpp"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace mcn {
namespace {

constexpr int kMaxMulti = 4;

__host__ __device__ constexpr int groups_per_slab(int WA) { return WA == 1 ? 4 : 2; }

// TAPS: where a pixel's offsets under the taps come from: there is one, unshifted; a table in LDS, worked out once per
// workgroup (its lanes' offsets, kFarOfTable outside the image; one row more of that for what follows the last group); worked out
// for every group (banks of more taps than the table has room for beside two slabs in 64 KB)
enum { kPoint = 0, kTable = 1, kWorked = 2 };
constexpr int kTableTaps = 31;
// What a lane whose tap lies outside the image has in the table: a half-wave adds eight planes to it.  Where channels 8 and on
// exist these are below 2^31 (nine planes are inside a descriptor), so that the sum stays out of range; where they do not,
// nothing of that half is loaded at all (lastOr).
constexpr unsigned kFarOfTable = kOutside;
static_assert(kFarOfTable >= kOutside && (unsigned long long)kFarOfTable + 8ull * ((kOutside - 1) / 9) < (1ull << 32), "");

constexpr size_t kLds[5] = {0, 2 * groups_per_slab(1) * 1 * kBlockBytes, 2 * groups_per_slab(2) * 2 * kBlockBytes, 0,
                            2 * groups_per_slab(4) * 4 * kBlockBytes};

// of a workgroup without its table, which lies behind
constexpr size_t lds_bytes(int WA, int epi) {
  const size_t stats = stats_lds_bytes(32 * WA);
  return epi == kStats && stats > kLds[WA] ? stats : kLds[WA];
}
constexpr size_t table_bytes(int taps, int T) { return taps == kTable ? (size_t)(T + 1) * 128 * sizeof(unsigned) : 0; }

template <int WA, int TAPS, bool RAGGED, int EPI>
__device__ __forceinline__ void split_body(float* __restrict__ out, const float* __restrict__ in, const void* __restrict__ bank,
                                           const float* __restrict__ bias, const PixP& p, const SplitP& w, const unsigned block,
                                           const unsigned blocks, const int firstTile = 0) {
  constexpr int GPS = groups_per_slab(WA);
  constexpr int SLAB = GPS * WA * kBlockBytes;       // bytes of a slab in LDS
  constexpr int DMA = SLAB / 1024 / 4;               // 1 KB loads per wavefront and slab
  constexpr int CT = 32 * WA;
  extern __shared__ char slabs[];
  unsigned* const table = (unsigned*)(slabs + lds_bytes(WA, EPI));  // [wavefront][T + 1][32]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, kh = lane >> 5;
  const int IHW = p.IH * p.IW;

  // (channel tiles of one pixel tile are neighbours, numbered XCD by XCD: they and the neighbouring pixel tiles read the
  // same pixels behind one L2)
  int logical = xcd_contiguous_id((int)block, (int)blocks);
  int split = 0;
  if (EPI == kTail) {
    split = logical / w.tailTiles;
    logical -= split * w.tailTiles;
    out += ((size_t)split * w.tailTiles + logical) * (size_t)(CT * 128);
    logical += w.tileBase;
  } else if (p.rSplits > 1) {
    const int tiles = (int)blocks / p.rSplits;
    split = logical / tiles;
    logical -= split * tiles;
    out += (size_t)split * p.partStride;
  }
  logical += firstTile;
  const int mt = logical / w.tilesC;
  const int ct = logical - mt * w.tilesC;
  const int slabBegin = split * w.slabsPerSplit;
  const int slabEnd = min(w.slabs, slabBegin + w.slabsPerSplit);
  if (slabBegin >= slabEnd) return;  // (uniform)

  // ---- the pixel loader
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)in, 0, (int)w.inBytes, 0x00020000);
  const int planeBytes = IHW * 4;
  const int m = mt * 128 + wave * 32 + l32;
  const bool mvalid = m < p.M;
  const unsigned halfOff = (unsigned)(kh * 8 * planeBytes);
  unsigned voff;  // (kPoint: with halfOff)
  int ihB, iwB;
  {
    int n, q, ow, oh;
    p.byQ.divmod(mvalid ? m : 0, &n, &q);
    p.byOH.divmod(q, &ow, &oh);
    ihB = mvalid ? oh * p.sy : -0x40000000;
    iwB = ow * p.sx;
    voff = mvalid ? (unsigned)(n * p.inImg + oh * p.sy + p.IH * iwB) * 4u + (TAPS == kTable ? 0u : halfOff) : kFar;
  }
  // RAGGED: rows of the last chunk beyond the last channel fetch nothing: what makes a lane's offset kFar for each of its
  // eight rows
  unsigned lastOr[RAGGED ? 8 : 1];
  if (RAGGED) {
    const int rem = p.Cin - (w.chunks - 1) * 16;
#pragma unroll
    for (int j = 0; j < 8; ++j) lastOr[j] = 8 * kh + j < rem ? 0u : kFar;
  }
  int chunkL, tapL, tapRow, dhL, dwL, groupsLeft;
  unsigned voTap;
  auto shifted = [&](int dh, int dw, bool present) -> unsigned {
    const bool ok = present & ((unsigned)(ihB + dh) < (unsigned)p.IH) & ((unsigned)(iwB + dw) < (unsigned)p.IW);
    const unsigned at = voff + (unsigned)((dh + p.IH * dw) * 4);
    return ok ? at : TAPS == kTable ? kFarOfTable : kFar;
  };
  const unsigned* const myTable = table + wave * ((p.T + 1) * 32) + l32;
  auto tap_offset = [&]() -> unsigned {
    if (TAPS == kPoint) return groupsLeft > 0 ? voff : kFar;
    if (TAPS == kTable) return myTable[(groupsLeft > 0 ? tapL : p.T) * 32] + halfOff;
    return shifted(dhL, dwL, groupsLeft > 0);
  };
  // (a wavefront's rows of the table: its halves take the taps in turn)
  auto fill_table = [&]() {
    if (TAPS != kTable) return;
    unsigned* row = table + wave * ((p.T + 1) * 32) + l32;
    int i = kh % p.FH, j = kh / p.FH;
    for (int t = kh; t <= p.T; t += 2) {
      row[t * 32] = shifted(p.dhBase + i * p.dhStep, p.dwBase + j * p.dwStep, t < p.T);
      i += 2;
      while (i >= p.FH) {
        i -= p.FH;
        ++j;
      }
    }
  };
  auto rewind = [&]() {
    const int g0 = slabBegin * GPS;
    chunkL = g0 / p.T;
    tapL = g0 - chunkL * p.T;
    if (TAPS == kWorked) {
      tapRow = tapL % p.FH;
      dhL = p.dhBase + tapRow * p.dhStep;
      dwL = p.dwBase + (tapL / p.FH) * p.dwStep;
    }
    groupsLeft = min(slabEnd * GPS, w.groups) - g0;  // (a last slab's padding groups and what follows it fetch nothing)
    voTap = tap_offset();
  };
  typedef float vbuf __attribute__((ext_vector_type(8)));
  // row j of the group the loader stands at (offset vo: voTap; c: its chunk, or the last one when it is past the end: the
  // scalar offset stays inside the tensor whatever the lanes' offsets say)
  auto load_row = [&](int j, unsigned vo, int c, bool last) -> float {
    const int row = RAGGED ? min(c * 16 + j, p.Cin - 1) : c * 16 + j;
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(RAGGED ? vo | (last ? lastOr[j] : 0u) : vo), row * planeBytes, 0));
  };
  auto chunk_at = [&]() { return min(chunkL, w.chunks - 1); };
  auto last_chunk = [&]() { return RAGGED && chunkL >= w.chunks - 1; };
  // (selects throughout: a branch here would end the block in which the matrix instructions are interleaved with this)
  auto advance = [&]() {
    --groupsLeft;
    if (TAPS == kWorked) {
      const bool endRow = tapRow + 1 == p.FH;
      tapRow = endRow ? 0 : tapRow + 1;
      dhL = endRow ? p.dhBase : dhL + p.dhStep;
      dwL += endRow ? p.dwStep : 0;
    }
    const bool endTaps = tapL + 1 == p.T;
    tapL = endTaps ? 0 : tapL + 1;
    if (TAPS == kWorked) dwL = endTaps ? p.dwBase : dwL;
    chunkL += endTaps ? 1 : 0;
    voTap = tap_offset();
  };
  // loads the next group of 16 rows and advances
  auto load_next = [&](vbuf& dst) {
#pragma unroll
    for (int j = 0; j < 8; ++j) dst[j] = load_row(j, voTap, chunk_at(), last_chunk());
    advance();
  };

  // ---- the bank: slab s into LDS buffer b
  const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc((void*)bank, 0, (int)w.bankBytes, 0x00020000);
  const int groupPitch = w.blocksC * kBlockBytes;  // bytes of a group of the bank
  // (a wavefront's pieces of a slab's GPS x WA x 3 follow one another, in LDS and in the bank: they are of one group)
  static_assert((3 * WA) % DMA == 0, "");
  const int dmaAt = (wave * DMA) / (3 * WA) * groupPitch + ct * (WA * kBlockBytes) + (wave * DMA) % (3 * WA) * 1024;
  auto dma = [&](int s, int b) {
    typedef __attribute__((address_space(3))) void* lds_ptr;
    const int vo = lane * 16, from = s * (GPS * groupPitch) + dmaAt;
    char* const to = slabs + b * SLAB + wave * (DMA * 1024);
#define SPLIT_DMA(I) \
  if (I < DMA) __builtin_amdgcn_raw_ptr_buffer_load_lds(brsrc, (lds_ptr)(to + I / 4 * 4096), 16, vo, from + I / 4 * 4096, I % 4 * 1024, 0)
    SPLIT_DMA(0);
    SPLIT_DMA(1);
    SPLIT_DMA(2);
    SPLIT_DMA(3);
    SPLIT_DMA(4);
    SPLIT_DMA(5);
#undef SPLIT_DMA
    static_assert(DMA <= 6, "");
  };

  floatx16 acc[WA], low[WA];  // the products h h; the other five
#pragma unroll
  for (int a = 0; a < WA; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[a][r] = low[a][r] = 0.f;

  typedef union { uintx4 u; bf16x8 v; } frag;
  vbuf px[GPS];
  struct Pix { frag h, m, l; };
  auto split_px = [&](const vbuf& v) {
    Pix o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned h, mm, l;
      split_pair(v[2 * j] * kSplitScale, v[2 * j + 1] * kSplitScale, &h, &mm, &l);
      o.h.u[j] = h;
      o.m.u[j] = mm;
      o.l.u[j] = l;
    }
    return o;
  };
  // Multiplies a group (its pixels split in `b`): the parts of the bank one after the other (l, m, h: the small products
  // first).  Everything else of the loop is dealt out behind the matrix instructions and pinned there: the fragment reads a
  // row of WA matrix instructions ahead, the splitting of the next group's pixels (28 stages of one or two instructions),
  // the loads of the group a slab ahead into the registers the splitting leaves, the loader's step.  So a wavefront
  // alone on its SIMD does not leave the matrix pipe waiting for them.
  // al: the l fragments of this group, and on return those of the next one, which lies at `then`.  LAST (of a slab): `turn` is
  // called where the slab's last fragments have been read and half of the group's products are still to come.
  auto group = [&](Pix& b, frag (&al)[WA], const char* at, const char* then, vbuf& next, auto lastC, auto&& turn) {
    constexpr bool LAST = decltype(lastC)::value;
    frag am[WA], ah[WA];
    Pix n;
    float r0[4], r1[4];
    const unsigned vo = voTap;
    const int chunk = chunk_at();
    const bool last = last_chunk();
    auto stage = [&](int k) {
      const int j = k / 7;
      const float x = next[2 * j], y = next[2 * j + 1];
      switch (k % 7) {
        case 0: n.h.u[j] = round_pair(x * kSplitScale, y * kSplitScale); break;
        case 1: r0[j] = fmaf(x, kSplitScale, -__builtin_bit_cast(float, n.h.u[j] << 16)); break;
        case 2:
          r1[j] = fmaf(y, kSplitScale, -__builtin_bit_cast(float, n.h.u[j] & 0xffff0000u));
          next[2 * j] = load_row(2 * j, vo, chunk, last);
          next[2 * j + 1] = load_row(2 * j + 1, vo, chunk, last);
          break;
        case 3: n.m.u[j] = round_pair(r0[j], r1[j]); break;
        case 4: r0[j] -= __builtin_bit_cast(float, n.m.u[j] << 16); break;
        case 5: r1[j] -= __builtin_bit_cast(float, n.m.u[j] & 0xffff0000u); break;
        default: n.l.u[j] = round_pair(r0[j], r1[j]); break;
      }
      // (needed here, these say: otherwise the compiler moves the splitting behind the matrix instructions)
      switch (k % 7) {
        case 0: asm volatile("" : "+v"(n.h.u[j])); break;
        case 1: asm volatile("" : "+v"(r0[j])); break;
        case 2: asm volatile("" : "+v"(r1[j])); break;
        case 3: asm volatile("" : "+v"(n.m.u[j])); break;
        case 4: asm volatile("" : "+v"(r0[j])); break;
        case 5: asm volatile("" : "+v"(r1[j])); break;
        default: asm volatile("" : "+v"(n.l.u[j])); break;
      }
    };
    // (a row of matrix instructions ahead, except where a row is one instruction)
    if (WA == 1) {
      am[0].u = *(const uintx4*)(at + kFragBytes);
      ah[0].u = *(const uintx4*)at;
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 6 * WA; ++i) {
      const int a = i % WA;
      switch (i / WA) {
        case 0: low[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[a].v, b.h.v, low[a], 0, 0, 0); break;
        case 1: low[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am[a].v, b.m.v, low[a], 0, 0, 0); break;
        case 2: low[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am[a].v, b.h.v, low[a], 0, 0, 0); break;
        case 3: low[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a].v, b.l.v, low[a], 0, 0, 0); break;
        case 4: low[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a].v, b.m.v, low[a], 0, 0, 0); break;
        default: acc[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a].v, b.h.v, acc[a], 0, 0, 0); break;
      }
      if (i < 5 * WA) asm volatile("" : "+v"(low[a]));
      else asm volatile("" : "+v"(acc[a]));
      if (WA > 1 && i < WA) am[a].u = *(const uintx4*)(at + a * kBlockBytes + kFragBytes);
      if (WA > 1 && i >= WA && i < 2 * WA) ah[a].u = *(const uintx4*)(at + a * kBlockBytes);
      if (i >= 4 * WA && i < 5 * WA) al[a].u = *(const uintx4*)(then + a * kBlockBytes + 2 * kFragBytes);
      if (i == 1) {
        // (not before: the loader's step would else be worked out ahead of the first matrix instruction)
        asm volatile("" : "+s"(groupsLeft), "+s"(chunkL), "+s"(tapL));
        if (TAPS == kWorked) asm volatile("" : "+s"(tapRow), "+s"(dhL), "+s"(dwL));
        advance();
      }
      if (LAST && i == 3 * WA) {
        __builtin_amdgcn_sched_barrier(0);
        turn();
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int k = i * 28 / (6 * WA); k < (i + 1) * 28 / (6 * WA); ++k) stage(k);
      __builtin_amdgcn_sched_barrier(0);
    }
    b = n;
  };
  dma(slabBegin, 0);
  __builtin_amdgcn_sched_barrier(0);
  fill_table();
  rewind();
#pragma unroll
  for (int g = 0; g < GPS; ++g) load_next(px[g]);
  __builtin_amdgcn_sched_barrier(0);
  if (slabBegin + 1 < slabEnd) dma(slabBegin + 1, 1);
  __builtin_amdgcn_sched_barrier(0);
  Pix cur = split_px(px[0]);
  load_next(px[0]);
  // (the first slab is in LDS: its loads are older than the pixels just split; what may be under way is younger than those)
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(GPS * 8 + DMA) : "memory");
  int buf = 0;
  frag al[WA];
#pragma unroll
  for (int a = 0; a < WA; ++a) al[a].u = *(const uintx4*)(slabs + lane * 16 + a * kBlockBytes + 2 * kFragBytes);
  for (int s = slabBegin; s < slabEnd; ++s) {
    const char* at = slabs + buf * SLAB + lane * 16;
    const char* after = slabs + (buf ^ 1) * SLAB + lane * 16;
    typedef std::integral_constant<bool, true> yes;
    typedef std::integral_constant<bool, false> no;
    // Before the slab's last products: this wavefront's loads of the next slab into LDS have landed, its fragment reads of
    // this one are done; the pixels of the next slab (GPS x 8 younger loads: since then a group's eight each, the first time
    // four less and the eight before the loop) may be in flight.  Behind the barrier the slab after the next one goes where this
    // one was, and the next one's first fragments are read, beside the products left.
    // (Past the split's end pixel loads fetch nothing and loads into LDS are left out: none is under way behind the loop.)
    auto turn = [&]() {
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"(GPS * 8) : "memory");
      if (s + 2 < slabEnd) dma(s + 2, buf);
    };
    auto stay = [] {};
#pragma unroll
    for (int g = 0; g < GPS - 1; ++g) group(cur, al, at + g * (WA * kBlockBytes), at + (g + 1) * (WA * kBlockBytes), px[(g + 1) % GPS], no(), stay);
    group(cur, al, at + (GPS - 1) * (WA * kBlockBytes), after, px[0], yes(), turn);
    buf ^= 1;
  }
#pragma unroll
  for (int a = 0; a < WA; ++a) acc[a] = (acc[a] + low[a]) * kSplitUnscale;

  // ---- an accumulator that is not finite: the block again on the fp32 instruction
  {
    float t = 0.f;
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) t = fmaf(acc[a][r], 0.f, t);
    if (__builtin_expect(__any(!(t == 0.f)), 0)) {
#pragma unroll
      for (int a = 0; a < WA; ++a)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][r] = 0.f;
      rewind();
      const int gEnd = min(slabEnd * GPS, w.groups);
#pragma unroll 1
      for (int g = slabBegin * GPS; g < gEnd; ++g) {
        const int rows = RAGGED ? p.Cin - chunkL * 16 - 8 * kh : 8;  // rows of this half that exist
        vbuf v;
        load_next(v);
#pragma unroll
        for (int a = 0; a < WA; ++a) {
          const char* at = (const char*)bank + (size_t)g * groupPitch + (ct * WA + a) * kBlockBytes + lane * 16;
          const uintx4 h = *(const uintx4*)at, mm = *(const uintx4*)(at + kFragBytes), l = *(const uintx4*)(at + 2 * kFragBytes);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            auto part = [&](const uintx4& u) { return j & 1 ? u[j / 2] >> 16 : u[j / 2] & 0xffffu; };
            const float wv = split_weight(part(h), part(mm), part(l));
            acc[a] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv, j < rows ? v[j] : 0.f, acc[a], 0, 0, 0);
          }
        }
      }
    }
  }

  // ---- epilogue: lane = pixel, register = channel
  const int coW = ct * CT;
  if (EPI == kTail) {
    split_store_tail<WA>(acc, out, CT, 0, wave * 32 + l32, kh);
    return;
  }
  if (EPI == kNormalise) {
    // (whole blocks of channels; the slabs are free: the channels' coefficients go there, read back four to a load)
    BnCoef* coefs = (BnCoef*)slabs;
    if (tid < CT && coW + tid < p.Cout) coefs[tid] = bn_coefficients(p, coW + tid);
    __syncthreads();
    split_store_normalised<WA>(acc, out, p, coefs, coW, m, mvalid, kh);
    return;
  }
  split_store<WA, EPI>(acc, out, bias, p, coW, m, mvalid, kh);
  if (EPI == kStats) {
    split_sums<WA>(acc, slabs, wave, wave, CT, 0, l32, kh);
    __syncthreads();
    split_sums_out(slabs, p, CT, coW, mt, tid);
  }
}

template <int WA, int TAPS, bool RAGGED, int EPI>
__global__ __launch_bounds__(256, WA == 4 ? 2 : WA == 2 && RAGGED ? 3 : 4) void conv_split_mfma(float* __restrict__ out, const float* __restrict__ in,
                                                          const void* __restrict__ bank, const float* __restrict__ bias, PixP p,
                                                          SplitP w) {
  split_body<WA, TAPS, RAGGED, EPI>(out, in, bank, bias, p, w, blockIdx.x, gridDim.x);
}

// The same with what is left over after whole rounds of tiles in tiles of 32 channels, v.tileBase the first of them: blocks
// from `whole` on.  (See plan_ends.  Same bits where the accumulators are finite: a channel's products follow one another as in the
// wider tile.  A tile with one that is not is done again on the fp32 instruction, all its channels: of the narrower tile fewer.)
template <int WA, int TAPS, int EPI>
__global__ __launch_bounds__(256, WA == 4 ? 2 : 4) void conv_split_mfma_ends(float* __restrict__ out, const float* __restrict__ in,
                                                                             const void* __restrict__ bank, const float* __restrict__ bias, PixP p,
                                                                             SplitP w, SplitP v, unsigned whole) {
  if (blockIdx.x < whole) split_body<WA, TAPS, false, EPI>(out, in, bank, bias, p, w, blockIdx.x, whole);
  else split_body<1, TAPS, false, EPI>(out, in, bank, bias, p, v, blockIdx.x - whole, gridDim.x - whole, v.tileBase);
}

// Up to four products over the same two tensors in one launch: the stride classes of a strided layer's backward-data
// product, the longest reductions first (see conv_pix_multi).
struct SplitMulti {
  PixP p[kMaxMulti];
  SplitP w[kMaxMulti];
  const void* bank[kMaxMulti];
  unsigned first[kMaxMulti + 1];
  int n;
};

template <int WA, int TAPS, bool RAGGED>
__global__ __launch_bounds__(256, WA == 4 ? 2 : WA == 2 && RAGGED ? 3 : 4) void conv_split_multi(float* __restrict__ out, const float* __restrict__ in, SplitMulti m) {
  int i = 0;
#pragma unroll
  for (int j = 1; j < kMaxMulti; ++j)
    if (j < m.n && blockIdx.x >= m.first[j]) i = j;
  split_body<WA, TAPS, RAGGED, kStore>(out, in, m.bank[i], nullptr, m.p[i], m.w[i], blockIdx.x - m.first[i], m.first[i + 1] - m.first[i]);
}

// out[tile of the tail] = alpha * (sum over the splits, in their order) (+ beta * out) (+ bias), or what the launch of the other
// tiles does with its accumulators (PixP::bnMoments, stats, addend): one thread per (tile, channel, pixel), pixels fastest
__global__ __launch_bounds__(256) void conv_split_tail_reduce(float* __restrict__ out, const float* __restrict__ partials,
                                                              const float* __restrict__ bias, PixP p, SplitP w, int splits, int CT) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const int pxl = (int)(idx & 127);
  const long long rest = idx >> 7;
  const int c = (int)(rest % CT), tl = (int)(rest / CT);
  const int tile = w.tileBase + tl;
  const int mt = tile / w.tilesC, ct = tile - mt * w.tilesC;
  const long long m = (long long)mt * 128 + pxl;
  const int co = ct * CT + c;
  const bool present = tl < w.tailTiles && m < p.M && co < p.Cout;
  float sum = 0.f;
  if (present) {
    const size_t tileFloats = (size_t)CT * 128;
    const float* src = partials + (size_t)tl * tileFloats + (size_t)c * 128 + pxl;
    for (int k = 0; k < splits; ++k) sum += src[(size_t)k * w.tailTiles * tileFloats];
    int n, q;
    p.byQ.divmod((int)m, &n, &q);
    float* o = out + (size_t)n * p.outImg + out_pixel_offset(p, q) + (size_t)co * p.outPlane;
    const size_t at = o - out;
    if (p.bnMoments) {
      *o = bn_apply(bn_coefficients(p, co), sum, p.bnResidual != nullptr, p.bnResidual ? p.bnResidual[at] : 0.f, p.bnRelu != 0);
    } else if (p.addend) {
      *o = fmaf(p.addend[at], (float)(p.addBits[at >> 5] >> (at & 31) & 1u), sum);  // (as store_block_masked_add)
    } else {
      float v = p.alpha * sum;
      if (p.beta != 0.f) v = fmaf(p.beta, *o, v);
      if (bias) v += bias[co];
      *o = v;
    }
  }
  if (p.stats) {  // (uniform; alpha = 1, beta = 0, no bias: `sum` is what was stored)
    __shared__ double part[4][2];
    double t1 = (double)sum, t2 = t1 * t1;
#pragma unroll
    for (int lanes = 32; lanes > 0; lanes >>= 1) {
      t1 += __shfl_xor(t1, lanes);
      t2 += __shfl_xor(t2, lanes);
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
      part[wave][0] = t1;
      part[wave][1] = t2;
    }
    __syncthreads();
    if ((threadIdx.x & 127) == 0 && tl < w.tailTiles && co < p.Cout) {
      double* o = p.stats + ((size_t)co * p.statGroups + mt) * 2;
      o[0] = part[wave][0] + part[wave + 1][0];
      o[1] = part[wave][1] + part[wave + 1][1];
    }
  }
}

template <int WA, int TAPS, bool RAGGED>
void launch_epi(hipStream_t s, int epi, unsigned blocks, float* out, const float* in, const void* bank, const float* bias, const PixP& p,
                const SplitP& w) {
  KernelTimer timer(epi == kTail ? "conv_split_mfma_tail" : "conv_split_mfma", s);
  const dim3 grid(blocks), block(256);
  const size_t table = table_bytes(TAPS, p.T);
#define EPI_GO(EPI) \
  hipLaunchKernelGGL((conv_split_mfma<WA, TAPS, RAGGED, EPI>), grid, block, lds_bytes(WA, EPI) + table, s, out, in, bank, bias, p, w)
  if constexpr (!RAGGED) {  // (whole chunks only: conv_split_stat_groups, conv_split_adds, conv_split_normalises)
    if (epi == kStats) {
      EPI_GO(kStats);
      return;
    }
    if (epi == kNormalise) {
      EPI_GO(kNormalise);
      return;
    }
    if (epi == kMaskedAdd) {
      EPI_GO(kMaskedAdd);
      return;
    }
  }
  if (epi == kTail) EPI_GO(kTail);
  else EPI_GO(kStore);
#undef EPI_GO
}

void launch(hipStream_t s, int WA, int taps, bool ragged, int epi, unsigned blocks, float* out, const float* in, const void* bank,
            const float* bias, const PixP& p, const SplitP& w) {
#define SPLIT_TAPS(W, TAPS)                                                                   \
  do {                                                                                        \
    if (ragged) launch_epi<W, TAPS, true>(s, epi, blocks, out, in, bank, bias, p, w);         \
    else launch_epi<W, TAPS, false>(s, epi, blocks, out, in, bank, bias, p, w);               \
  } while (0)
#define SPLIT_GO(W)                                \
  do {                                             \
    if (taps == kTable) SPLIT_TAPS(W, kTable);     \
    else if (taps == kPoint) SPLIT_TAPS(W, kPoint); \
    else SPLIT_TAPS(W, kWorked);                   \
  } while (0)
  if (WA == 4) SPLIT_GO(4);
  else if (WA == 2) SPLIT_GO(2);
  else SPLIT_GO(1);
#undef SPLIT_GO
#undef SPLIT_TAPS
}

int chunks_of(int Cin) { return (Cin + 15) / 16; }

// groups of 16 rows of the packed bank: whole slabs of four, whatever the width of the tiles that read it
int bank_groups(int Cin, int T) { return (chunks_of(Cin) * T + 3) / 4 * 4; }
int bank_blocks(int Cout) { return Cout > 64 ? (Cout + 127) / 128 * 4 : (Cout > 32 ? 2 : 1); }

void fill_geometry(const PixP& p, int WA, SplitP* w) {
  const int GPS = groups_per_slab(WA);
  w->blocksC = bank_blocks(p.Cout);
  w->tilesC = (p.Cout + 32 * WA - 1) / (32 * WA);
  w->chunks = chunks_of(p.Cin);
  w->groups = w->chunks * p.T;
  w->slabs = (w->groups + GPS - 1) / GPS;
  w->slabsPerSplit = w->slabs;
  w->inBytes = (unsigned)(((long long)(p.N - 1) * p.inImg + (long long)p.Cin * p.IH * p.IW) * 4);
  w->bankBytes = (unsigned)conv_split_bank_bytes(p.Cin, p.T, p.Cout);
  w->tileBase = w->tailTiles = 0;
}

int taps_of(const PixP& p) {
  if (p.T == 1 && p.dhBase == 0 && p.dwBase == 0 && p.sy == 1 && p.sx == 1 && p.IH == p.OH && p.IW == p.OW) return kPoint;
  return p.T <= kTableTaps ? kTable : kWorked;
}

// Width of the tiles and reduction splits of a product: the pair with the least modelled time.  A group of 16 rows of a tile
// of 128, 64, 32 channels takes a workgroup alone on its CU 0.50, 0.385, 0.28 us and a CU full of them 0.55, 0.30, 0.20 us
// per workgroup (3x3x512x512 on 7x7, 3x3x256x256 on 14x14, 3x3x128x128 on 28x28, 32 images each); what counts is the busiest
// CU.  Partial results are written and read back once per split, and adding them up is a launch.
struct Plan { int WA, splits, slabsPerSplit; double us; };
// of `groups` groups to a split
double modelled_us(int WA, int groups, int splits, long long tiles, long long M, int Cout, int cus) {
  static const double alone[5] = {0, 0.28, 0.385, 0, 0.50}, full[5] = {0, 0.20, 0.30, 0, 0.55};
  const long long perCu = (tiles * splits + cus - 1) / cus;
  double us = groups * std::max(alone[WA], (double)perCu * full[WA]) + 2.0;
  if (splits > 1) us += 2.0 * splits * (double)M * Cout * 4.0 / 5e6 + 5.0;
  return us;
}
Plan plan_split(int Cin, int T, int Cout, long long M) {
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  const int groups = chunks_of(Cin) * T;
  const long long mTiles = (M + 127) / 128;
  int forced = tunable("conv_split_wa", 0);
  if (forced > bank_blocks(Cout)) forced = 0;
  // (a split count the slabs cannot be cut into: the next smaller one)
  const int forcedSplits = tunable("conv_split_splits", 0);
  const int most = tunable("conv_no_split", 0) ? 1 : 32;
  Plan best = {0, 1, 0, 0};
  for (int WA : {4, 2, 1}) {
    if (32 * WA > bank_blocks(Cout) * 32 || (forced && forced != WA)) continue;
    const int GPS = groups_per_slab(WA), slabs = (groups + GPS - 1) / GPS;
    const long long tiles = mTiles * ((Cout + 32 * WA - 1) / (32 * WA));
    for (int s = 1; s <= most; ++s) {
      const int per = (slabs + s - 1) / s;
      if (s > 1 && per * GPS < 8) break;
      if ((slabs + per - 1) / per != s) continue;
      if (forcedSplits && s > forcedSplits) continue;
      if (forcedSplits) { best = {WA, s, per, 0}; continue; }
      const double us = modelled_us(WA, per * GPS, s, tiles, M, Cout, cus);
      if (best.WA == 0 || us < best.us) best = {WA, s, per, us};
    }
  }
  return best;
}

// The tiles left over after the last full round of workgroups get a launch of their own that splits their reduction over the
// chip (see conv_sb.hip).  Depends on the extents only.  Rounds are counted with one workgroup to a CU more than stay resident
// in tiles of 128: tiles follow one another as they end, and at the resident count 56x56 layers at 32 images would get a tail
// that costs more than it saves (1x1 256 -> 64 25.9 -> 32.0 us, 64 -> 256 28.8 -> 32.2).
struct Tail { int tiles, splits, slabsPerSplit; size_t bytes; };
Tail plan_tail(const Plan& plan, int Cin, int T, int Cout, long long M) {
  Tail t = {0, 0, 0, 0};
  if (plan.splits != 1 || !tunable("conv_sb_tail", 1)) return t;
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  const int WA = plan.WA, GPS = groups_per_slab(WA);
  const long long tiles = (M + 127) / 128 * ((Cout + 32 * WA - 1) / (32 * WA));
  const long long slots = (long long)cus * (WA == 4 ? 3 : 4);
  const long long rem = tiles % slots;
  if (tiles <= slots || rem == 0 || 2 * rem > slots) return t;
  const int slabs = (chunks_of(Cin) * T + GPS - 1) / GPS;
  int s = (int)std::min<long long>(slots / rem, slabs / 4);
  s = std::min(s, 16);
  if (s < 2) return t;
  const int per = (slabs + s - 1) / s;
  s = (slabs + per - 1) / per;
  if (s < 2) return t;
  t.tiles = (int)rem;
  t.splits = s;
  t.slabsPerSplit = per;
  t.bytes = (size_t)s * (size_t)rem * 32 * WA * 128 * sizeof(float);
  return t;
}

// Tiles beyond whole rounds of one to a CU, where a launch of their own does not pay: 784 tiles (56x56 over 32 images) leave 16
// CUs with four and the others with three, and the four are what the launch takes.  Those 16 go in tiles of 32 channels, each
// to a CU of its own, in the same launch; 0: none.  (More than a CU each: the narrow tiles split every pixel again, WA times.)
// Without and with, 32 images unless said: 56x56 3x3x64x64 53.3 -> 50.3 us (36 images, 114 tiles left: 55.1 -> 53.7; 64: 91.0 ->
// 89.4), 1x1x256x64 31.3 -> 29.7, 1x1x64x256 36.2 -> 34.0, 3x3x128x128 169 -> 166, 28x28 1x1x128x512 32.2 -> 30.8, 64x64x96x9
// 3x3x96x64 38.7 -> 35.3; of 28 such products none is slower by more than the runs differ (1 %; 3x3 ones read per tap then, before
// conv_staged.hpp).  From 16 rounds on a round more is not seen.
int plan_ends(const Plan& plan, int Cout, long long M) {
  const int WA = plan.WA;
  if (plan.splits != 1 || WA == 1 || Cout % (32 * WA) != 0 || !tunable("conv_split_ends", 1)) return 0;
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  const long long tiles = (M + 127) / 128 * (Cout / (32 * WA)), rem = tiles % cus;
  return tiles > cus && tiles < 16ll * cus && rem * WA <= cus ? (int)rem : 0;
}

template <int WA, int TAPS>
void launch_ends(hipStream_t s, int epi, unsigned whole, unsigned blocks, float* out, const float* in, const void* bank, const float* bias,
                 const PixP& p, const SplitP& w, const SplitP& v) {
  KernelTimer timer("conv_split_mfma_ends", s);
  const dim3 grid(blocks), block(256);
  const size_t table = table_bytes(TAPS, p.T);
  static_assert(lds_bytes(WA, kStore) >= lds_bytes(1, kStore) && lds_bytes(WA, kStats) >= lds_bytes(1, kStats), "");
#define ENDS_GO(EPI) \
  hipLaunchKernelGGL((conv_split_mfma_ends<WA, TAPS, EPI>), grid, block, lds_bytes(WA, EPI) + table, s, out, in, bank, bias, p, w, v, whole)
  if (epi == kStats) ENDS_GO(kStats);
  else if (epi == kNormalise) ENDS_GO(kNormalise);
  else if (epi == kMaskedAdd) ENDS_GO(kMaskedAdd);
  else ENDS_GO(kStore);
#undef ENDS_GO
}

// A reduction in so many splits, cut at whole chunks as the staged pixels are: chunks to a split, and splits.
struct ChunkCut { int per, splits; };
ChunkCut cut_chunks(int chunks, int splits) {
  const int per = (chunks + splits - 1) / splits;
  return {per, (chunks + per - 1) / per};
}

// A split reduction cut at whole chunks has a longer longest split and fewer of them; false: in the model that costs more than
// staging gives (tiles of 64 channels have more to gain).  Of 220 split products of nine and 25 taps, staged against
// conv_split_mfma: tiles of 64 channels, 25 % less to 3 % more time up to 1.3 times the modelled one, 5 % less to 6 % more beyond;
// tiles of 128, 14 % less to 7 % more up to 1.15, 6 % less to 23 % more beyond; behind the better of both by 0.4 % on average
// (always staged 1.8, never 5).  us, before staging -> staged -> now: 5x5x96x128 over 56x56, 4 images 55.7 -> 66.8 -> 54.4,
// 5x5x192x64 over 27x27, 8 images 38.8 -> 39.1 -> 37.7, 3x3x192x192 over 24x24, 4 images 27.3 -> 25.6 -> 25.6.  What counts against
// the CUs is the number planned: where fewer workgroups are left it is the partial results not written that show (5x5x512x192
// over 24x24, one image, 240 workgroups of 465: 45.0 -> 36.9).
bool cut_holds(const Plan& plan, const ChunkCut& cut, int T, long long tiles, long long M, int Cout) {
  if (cut.splits < 2) return false;  // (whoever adds them up expects partial results)
  if (tunable("conv_staged", 0) > 0) return true;
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  return modelled_us(plan.WA, cut.per * T, cut.splits, tiles, M, Cout, cus) <=
         (plan.WA == 4 ? 1.15 : 1.3) * modelled_us(plan.WA, plan.slabsPerSplit * groups_per_slab(plan.WA), plan.splits, tiles, M, Cout, cus);
}

__global__ __launch_bounds__(256) void conv_pack_split(PackJob j) { conv_pack_split_block(j, blockIdx.x); }

}  // namespace

void conv_split_pack_job(PackJob* j, void* bank, const float* f, const TapSet& taps, int Cin, int Cout, int backward) {
  const int T = taps.nI * taps.nJ;
  j->wt = (float*)bank;
  j->f = f;
  j->taps = taps;
  j->Cin = Cin;
  j->Cout = Cout;
  j->rPad = bank_groups(Cin, T) * 16;
  j->coutPad = bank_blocks(Cout) * 32;
  j->backward = backward;
  j->tapMajor = kPackSplit;
  j->firstBlock = 0;
  // Few chunks and blocks: a workgroup takes four taps (with the padding groups of the last chunk) instead of all of them one
  // after the other (5x5 x 16 -> 64: 12.4 -> 6.5 us).  From 128 workgroups on the taps stay together.
  const unsigned blocks = (unsigned)(chunks_of(Cin) * bank_blocks(Cout));
  j->blocks = blocks < 128 ? blocks * (unsigned)((T + 3 + 3) / 4) : blocks;
}

int conv_split_pack(hipStream_t s, const char* who, const PackJob& j) {
  KernelTimer timer("conv_pack_split", s);
  hipLaunchKernelGGL(conv_pack_split, dim3(j.blocks), dim3(256), 0, s, j);
  return check_launch(who);
}

double conv_split_modelled_us(int Cin, int T, int Cout, long long M) { return plan_split(Cin, T, Cout, M).us; }

int conv_split_bank_blocks(int Cout) { return bank_blocks(Cout); }

size_t conv_split_bank_bytes(int Cin, int T, int Cout) {
  return (size_t)bank_groups(Cin, T) * bank_blocks(Cout) * kBlockBytes;
}

bool conv_split_takes(const PixP& p) {
  if (tunable("conv_no_ws", 0) || tunable("conv_ws_min_units", 0) > 0 || tunable("conv_no_uniform_tap", 0)) return false;
  if (p.Cout <= 4 || p.Cin < 6) return false;
  // fully connected: a few pixels per filter bank, which would be read, written out in three parts and read again for them
  if (p.OH * p.OW == 1 && p.IH * p.IW == 1) return false;
  const long long inBytes = ((long long)(p.N - 1) * p.inImg + (long long)p.Cin * p.IH * p.IW) * 4;
  if (inBytes >= (long long)kOutside || conv_split_bank_bytes(p.Cin, p.T, p.Cout) >= (size_t)kOutside) return false;
  return ((long long)p.M / 128 + 1) * bank_blocks(p.Cout) < (1ll << 26);
}

size_t conv_split_workspace_bytes(int Cin, int T, int Cout, long long M) {
  const size_t bank = (conv_split_bank_bytes(Cin, T, Cout) + 255) / 256 * 256;
  const Plan plan = plan_split(Cin, T, Cout, M);
  const size_t parts = plan.splits > 1 ? (size_t)plan.splits * (size_t)M * Cout * sizeof(float) : (size_t)0;
  return bank + std::max(parts, plan_tail(plan, Cin, T, Cout, M).bytes);
}

int conv_split_stat_groups(const PixP& p) {
  if (p.Cin % 16 != 0 || p.Cout % 32 != 0 || p.outBytes == 0 || p.beta != 0.f || p.alpha != 1.f) return 0;
  if (conv_short_plan(p).wa) return conv_short_stat_groups(p.M);
  if (plan_split(p.Cin, p.T, p.Cout, p.M).splits != 1) return 0;
  return (int)(((long long)p.M + 127) / 128);
}

bool conv_split_adds(const PixP& p) {
  if (p.Cin % 16 != 0 || p.alpha != 1.f || p.beta != 0.f || !p.dense || p.outBytes == 0 || p.Cout % 32 != 0 || p.outPlane % 32 != 0 || p.outImg % 32 != 0) return false;
  return conv_short_plan(p).wa || plan_split(p.Cin, p.T, p.Cout, p.M).splits == 1;
}

bool conv_split_normalises(const PixP& p) {
  return p.Cin % 16 == 0 && p.Cout % 32 == 0 && p.alpha == 1.f && p.beta == 0.f && p.dense && p.outBytes != 0;
}

int conv_split_launch(hipStream_t s, const char* who, float* out, const float* in, const void* bank, const float* bias, PixP p, void* scratch,
                      size_t scratchBytes, PixP* reduce) {
  const ShortPlan few = conv_short_plan(p);
  if (few.wa) {
    reduce->rSplits = 1;
    return conv_short_launch(s, who, few, out, in, bank, bias, p);
  }
  const Plan plan = plan_split(p.Cin, p.T, p.Cout, p.M);
  SplitP w;
  fill_geometry(p, plan.WA, &w);
  const int taps = taps_of(p);
  const bool ragged = p.Cin % 16 != 0;
  const long long mTiles = ((long long)p.M + 127) / 128, tiles = mTiles * w.tilesC;
  p.rSplits = 1;
  reduce->rSplits = 1;
  if (plan.splits > 1) {
    const size_t nOut = (size_t)p.M * p.Cout;
    if (!scratch || scratchBytes < (size_t)plan.splits * nOut * sizeof(float))
      return fail(MCN_ILLEGAL_ARGUMENT, "%s: workspace too small for %d partial results", who, plan.splits);
    w.slabsPerSplit = plan.slabsPerSplit;
    p.rSplits = plan.splits;
    p.partStride = (long long)nOut;
    reduce->rSplits = plan.splits;
    reduce->partStride = p.partStride;
    p.alpha = 1.f;
    p.beta = 0.f;
    p.outPlane = p.OH * p.OW;
    p.outImg = p.Cout * p.outPlane;
    p.outOff = 0; p.outSH = 1; p.outSW = p.OH; p.dense = 1;
    p.outBytes = nOut * 4 < (1ull << 31) ? (unsigned)(nOut * 4) : 0u;
    const ChunkCut cut = cut_chunks(w.chunks, plan.splits);
    if (conv_staged_takes(p, plan.WA, tiles * plan.splits) && cut_holds(plan, cut, p.T, tiles, p.M, p.Cout)) {
      p.rSplits = reduce->rSplits = cut.splits;
      return conv_staged_launch(s, who, plan.WA, kStore, (unsigned)(tiles * cut.splits), 0, cut.per, 0, 0, (float*)scratch, in, bank, nullptr, p);
    }
    launch(s, plan.WA, taps, ragged, kStore, (unsigned)(tiles * plan.splits), (float*)scratch, in, bank, nullptr, p, w);
    return check_launch(who);
  }
  const int whole = p.stats ? kStats : p.addend ? kMaskedAdd : p.bnMoments ? kNormalise : kStore;
  const bool staged = conv_staged_takes(p, plan.WA, tiles);
  const Tail tail = plan_tail(plan, p.Cin, p.T, p.Cout, p.M);
  if (tail.tiles && scratch && scratchBytes >= tail.bytes) {
    SplitP t = w;
    t.tileBase = (int)(tiles - tail.tiles);
    t.tailTiles = tail.tiles;
    t.slabsPerSplit = tail.slabsPerSplit;
    int splits = tail.splits;
    if (staged) {
      // (Whole chunks, however few splits are left: the tail runs beside the end of the whole tiles.  Its launch staged and on
      // conv_split_mfma: 3x3x256x256 over 56x56, 64 images, 18 groups for 12, 963 and 966 us; 5x5x96x256 over 56x56, 32 images, 25 for
      // 10, 514 and 515; 3x3x128x512 over 40x40, 32 images, 9 for 8, 272 and 277.)
      const ChunkCut cut = cut_chunks(w.chunks, splits);
      splits = cut.splits;
      int rc = conv_staged_launch(s, who, plan.WA, whole, (unsigned)t.tileBase, 0, w.chunks, 0, 0, out, in, bank, bias, p);
      if (!rc) rc = conv_staged_launch(s, who, plan.WA, kTail, (unsigned)(tail.tiles * splits), 0, cut.per, t.tileBase, t.tailTiles, (float*)scratch, in, bank, nullptr, p);
      if (rc) return rc;
    } else {
      launch(s, plan.WA, taps, ragged, whole, (unsigned)t.tileBase, out, in, bank, bias, p, w);
      launch(s, plan.WA, taps, ragged, kTail, (unsigned)(tail.tiles * splits), (float*)scratch, in, bank, nullptr, p, t);
    }
    KernelTimer timer("conv_split_tail_reduce", s);
    const long long threads = (long long)tail.tiles * 32 * plan.WA * 128;
    hipLaunchKernelGGL(conv_split_tail_reduce, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, out, (const float*)scratch, bias, p, t,
                       splits, 32 * plan.WA);
    return check_launch(who);
  }
  const int ends = ragged || (staged && p.T != 9) ? 0 : plan_ends(plan, p.Cout, p.M);
  if (staged) return conv_staged_launch(s, who, plan.WA, whole, (unsigned)(tiles - ends), ends, w.chunks, 0, 0, out, in, bank, bias, p);
  if (ends) {
    SplitP v;
    fill_geometry(p, 1, &v);
    v.tileBase = (int)(tiles - ends) * plan.WA;
    const unsigned first = (unsigned)(tiles - ends), blocks = first + (unsigned)(ends * plan.WA);
#define ENDS_GO(W)                                                                                              \
  do {                                                                                                          \
    if (taps == kTable) launch_ends<W, kTable>(s, whole, first, blocks, out, in, bank, bias, p, w, v);          \
    else if (taps == kPoint) launch_ends<W, kPoint>(s, whole, first, blocks, out, in, bank, bias, p, w, v);     \
    else launch_ends<W, kWorked>(s, whole, first, blocks, out, in, bank, bias, p, w, v);                        \
  } while (0)
    if (plan.WA == 4) ENDS_GO(4);
    else ENDS_GO(2);
#undef ENDS_GO
    return check_launch(who);
  }
  launch(s, plan.WA, taps, ragged, whole, (unsigned)tiles, out, in, bank, bias, p, w);
  return check_launch(who);
}

int conv_split_launch_multi(hipStream_t s, const char* who, float* out, const float* in, const PixP* products, const void* const* banks, int n) {
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  long long mTiles = 0;
  for (int i = 0; i < n; ++i) mTiles += ((long long)products[i].M + 127) / 128;
  const int Cout = products[0].Cout;
  // the widest tiles that still leave two to a CU
  int WA = bank_blocks(Cout) >= 4 ? 4 : bank_blocks(Cout);
  while (WA > 1 && mTiles * ((Cout + 32 * WA - 1) / (32 * WA)) < 2 * cus) WA /= 2;
  SplitMulti m;
  m.n = n;
  unsigned at = 0;
  for (int i = 0; i < kMaxMulti; ++i) {
    m.first[i] = at;
    if (i >= n) continue;
    m.p[i] = products[i];
    m.p[i].rSplits = 1;
    m.bank[i] = banks[i];
    fill_geometry(products[i], WA, &m.w[i]);
    at += (unsigned)((((long long)products[i].M + 127) / 128) * m.w[i].tilesC);
  }
  m.first[kMaxMulti] = at;
  for (int i = n; i <= kMaxMulti; ++i) m.first[i] = at;
  KernelTimer timer("conv_split_multi", s);
  const bool ragged = products[0].Cin % 16 != 0;
  int mostTaps = 0;
  for (int i = 0; i < n; ++i) mostTaps = std::max(mostTaps, products[i].T);
#define SPLIT_TAPS(W, TAPS, RAGGED) \
  hipLaunchKernelGGL((conv_split_multi<W, TAPS, RAGGED>), dim3(at), dim3(256), lds_bytes(W, kStore) + table_bytes(TAPS, mostTaps), s, out, in, m)
#define SPLIT_GO(W)                                                       \
  do {                                                                    \
    if (mostTaps <= kTableTaps && ragged) SPLIT_TAPS(W, kTable, true);    \
    else if (mostTaps <= kTableTaps) SPLIT_TAPS(W, kTable, false);        \
    else if (ragged) SPLIT_TAPS(W, kWorked, true);                        \
    else SPLIT_TAPS(W, kWorked, false);                                   \
  } while (0)
  if (WA == 4) SPLIT_GO(4);
  else if (WA == 2) SPLIT_GO(2);
  else SPLIT_GO(1);
#undef SPLIT_TAPS
#undef SPLIT_GO
  return check_launch(who);
}

}  // namespace mcn
