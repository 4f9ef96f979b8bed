// Implicit-GEMM convolution on the bf16 matrix instruction with operands split in three, for filters with taps whose output
// lies on the grid of their input (forward, and backward-data at unit stride): 3x3 and 5x5 layers.
//
// conv_split.hip reads and splits a pixel once for every tap: 62 vector instructions beside 24 matrix instructions, each some 3
// cycles of matrix time, and power; its matrix pipe is busy 0.73 of the time.  Here the pixels under a tile of 128 and its
// taps are split once per 16 channels into LDS, and every tap reads them from there: 21 vector instructions, matrix pipe busy
// 0.82 to 0.86 of the time (by card) at 1.6 GHz: what bounds the large products is power (3x3x256x256 over 56x56, 64 images: 228 ->
// 252 TFLOP/s, of the 298 that the six products reach from registers).
//   * Pixels are numbered on through columns and images, so a tap is a constant distance.  Of `slots` of them (the tile, what
//     its taps reach on both sides, and zeros for lanes whose tap lies outside the image) LDS holds both halves of 8 channels,
//     48 bytes each: the parts h, m, l of 8 channels, a fragment read is 16 bytes a lane at a distance of 48 (every bank once).
//   * A chunk of 16 channels is T groups, unrolled.  While it is multiplied, the pixels of the next chunk are loaded, split and
//     written to a second buffer, a unit of 64 half-slots to a wavefront at a time, 28 stages dealt out behind the matrix
//     instructions of one group; where a lane's pixel lies under each tap is a table in LDS, worked out once.  (A loop over
//     groups, for any T, is a fifth of the code and slower: 3x3x256x256 1.048 instead of 1.057, the 5x5 layer 1.08 instead of 1.12
//     times as fast as before: its branches and the scalars' steps cost a wavefront 8 cycles each where they come in a row.)
//   * The bank passes through a ring of R groups in LDS, filled straight from global memory R - 1 groups ahead.  One barrier a
//     group stands behind its last fragment reads, with half of its matrix instructions still to come.  (R: 2 to 6 measured
//     the same but where the bank comes cold and R is 2; what lets two workgroups be on a CU.)
//   * 128 channels to a workgroup: a wavefront has 64 pixels x 64 channels (12 KB of fragments per 24 matrix instructions);
//     64 channels: 32 pixels x 64.
// The numbers are conv_split.hip's, bit for bit, where a reduction is not split: the same products in the same order.  Split ones
// and tails are cut at whole chunks here (2e-8 apart); beside an accumulator that is not finite as many channels are done again on
// the fp32 instruction as the wavefront has, 64 here (a rounding apart).
#pragma once

#include "conv_split.hpp"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace mcn {

constexpr int kSlotBytes = 48;  // of a half-slot: 8 channels, three parts
constexpr int most_units(int T, int WA) { return T == 9 || WA < 4 ? 2 : 3; }  // of a wavefront (see conv_staged_takes)

struct StagedP {
  int tilesC, blocksC, chunks, chunksPerSplit;
  unsigned inBytes, bankBytes;
  int tileBase, tailTiles;  // kTail (see SplitP)
  int first, span, slots;   // pixels from the tile's first + `first` on, `span` of them; slots: with zeros, whole 64s
  FastDiv byIHW;
};

namespace {

// Of the T groups of a chunk, the one beside which unit u (of U) of the next chunk's pixels is split: -1 .. U of them by group.
// Behind it the unit that follows is loaded.
constexpr int split_group(int T, int U, int u) { return (u + 1) * T / (U + 1); }
constexpr int unit_split(int T, int U, int t) {
  for (int u = 0; u < U; ++u)
    if (split_group(T, U, u) == t) return u;
  return -1;
}
// pixels asked for behind one of the R - 1 groups before group t
constexpr bool unit_loaded(int T, int U, int R, int t) {
  for (int u = 0; u < U; ++u)
    if (split_group(T, U, u) < t && split_group(T, U, u) > t - R) return true;
  return false;
}

constexpr int ring_bytes(int CT, int R) { return R * (CT / 32) * kBlockBytes; }
__host__ __device__ constexpr int patch_bytes(int slots) { return 2 * slots * kSlotBytes; }
// what loads of a wavefront without pieces of its own write (zeros; of 128 channels every one has)
__host__ __device__ constexpr int spare_bytes(int CT) { return CT == 128 ? 0 : 2048; }
__host__ __device__ constexpr int table_at(int CT, int R, int slots) { return ring_bytes(CT, R) + 2 * patch_bytes(slots) + spare_bytes(CT); }

template <int N, typename F>
__device__ __forceinline__ void unrolled(F&& f) {
  if constexpr (N > 0) {
    unrolled<N - 1>(f);
    f(std::integral_constant<int, N - 1>());
  }
}

// PB x CB blocks of 32 pixels x 32 channels to a wavefront, WPX wavefronts side by side along the tile's 128 pixels
template <int PB, int CB, int WPX, int T, int U, int R, int EPI>
__device__ __forceinline__ void staged_body(float* __restrict__ out, const float* __restrict__ in, const void* __restrict__ bank,
                                            const float* __restrict__ bias, const PixP& p, const StagedP& w, const unsigned block,
                                            const unsigned blocks, const int firstTile = 0) {
  static_assert(PB * WPX == 4, "");
  static_assert(split_group(T, U, 0) >= 2 && split_group(T, U, U - 1) <= T - R, "");
  constexpr int WCH = 4 / WPX, CT = 32 * CB * WCH;
  constexpr int NB = CT / 32, GROUP = NB * kBlockBytes;
  constexpr int PIECES = 3 * NB, DMA = (PIECES + 3) / 4;  // 1 KB loads of a group, and of a wavefront
  constexpr int NP = PB * CB;
  extern __shared__ __attribute__((aligned(16))) char lds[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, kh = lane >> 5;
  const int wpx = wave % WPX, wch = wave / WPX;
  const int IHW = p.IH * p.IW, planeBytes = IHW * 4;

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
  const int chunkBegin = split * w.chunksPerSplit;
  const int chunkEnd = min(w.chunks, chunkBegin + w.chunksPerSplit);
  if (chunkBegin >= chunkEnd) return;  // (uniform)

  // ---- the pixels' loader: this wavefront's units, the same in every chunk
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)in, 0, (int)w.inBytes, 0x00020000);
  char* const patches = lds + ring_bytes(CT, R);
  const int patchBytes = patch_bytes(w.slots), halfBytes = w.slots * kSlotBytes;
  unsigned unitFrom[U];
  int unitTo[U];
  const int perHalf = w.slots / 64, units = 2 * perHalf;
  {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int unit = min(wave + 4 * u, units - 1);  // (more wavefronts than units: the last one twice, the same numbers)
      const int half = unit >= perHalf ? 1 : 0, slot = (unit - half * perHalf) * 64 + lane;
      const int L = mt * 128 + w.first + slot;
      const bool ok = (slot < w.span) & ((unsigned)L < (unsigned)(p.N * IHW));
      int n, q;
      w.byIHW.divmod(ok ? L : 0, &n, &q);
      unitFrom[u] = ok ? (unsigned)(n * p.inImg + q + half * 8 * IHW) * 4u : kFar;
      unitTo[u] = half * halfBytes + slot * kSlotBytes;
    }
  }
  auto load_row = [&](unsigned from, int chunk, int j) -> float {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)from, (chunk * 16 + j) * planeBytes, 0));
  };

  // ---- the bank: the group at byte `from` of it into slot r of the ring
  const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc((void*)bank, 0, (int)w.bankBytes, 0x00020000);
  const int groupPitch = w.blocksC * kBlockBytes;
  // (a wavefront's pieces follow one another; one without pieces of its own loads nothing into the spare bytes)
  const bool own = wave * DMA < PIECES;
  static_assert(PIECES % DMA == 0 && (PIECES == 4 * DMA || DMA * 1024 <= spare_bytes(CT)), "");
  const int dmaOff = own ? lane * 16 : (int)kOutside;
  const int dmaTo = own ? wave * DMA * 1024 : ring_bytes(CT, R) + 2 * patchBytes;
  auto dma_piece = [&](int from, int to, int i) __attribute__((always_inline)) {  // (i of DMA: a constant)
    typedef __attribute__((address_space(3))) void* lds_ptr;
    lds_ptr at = (lds_ptr)(lds + to);
    if (i == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(brsrc, at, 16, dmaOff, from, 0, 0);
    else if (i == 1) __builtin_amdgcn_raw_ptr_buffer_load_lds(brsrc, at, 16, dmaOff, from, 1024, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(brsrc, at, 16, dmaOff, from, 2048, 0);
  };
  static_assert(DMA <= 3, "");
  const int bankMine = ct * GROUP + (own ? wave * DMA * 1024 : 0);
  const int lastGroup = (chunkEnd * T - 1) * groupPitch + bankMine;
  int bankAt = chunkBegin * T * groupPitch + bankMine;  // of the group that goes to the ring next

  // ---- before the first chunk
  typedef float vbuf __attribute__((ext_vector_type(8)));
  typedef union { uintx4 u; bf16x8 v; } frag;
  vbuf px;
  {
    vbuf first[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 8; ++j) first[u][j] = load_row(unitFrom[u], chunkBegin, j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < DMA; ++i) dma_piece(bankAt, dmaTo, i);
    bankAt = min(bankAt + groupPitch, lastGroup);
    __builtin_amdgcn_sched_barrier(0);
    const int next = min(chunkBegin + 1, chunkEnd - 1);
#pragma unroll
    for (int j = 0; j < 8; ++j) px[j] = load_row(unitFrom[0], next, j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 1; r < R; ++r) {
#pragma unroll
      for (int i = 0; i < DMA; ++i) dma_piece(bankAt, dmaTo + (own ? r * GROUP : 0), i);
      bankAt = min(bankAt + groupPitch, lastGroup);
    }
    __builtin_amdgcn_sched_barrier(0);
    // the table: where pixel `at` of the tile lies under each tap, in bytes from its half of a patch
    unsigned short* table = (unsigned short*)(lds + table_at(CT, R, w.slots));
    const int at = tid & 127, m = mt * 128 + at;
    int n, q, ow, oh;
    p.byQ.divmod(m < p.M ? m : 0, &n, &q);
    p.byOH.divmod(q, &ow, &oh);
    if (m >= p.M) oh = -0x40000000;
    int i = (tid >> 7) % p.FH, j = (tid >> 7) / p.FH;
    for (int t = tid >> 7; t < T; t += 2) {
      const int dh = p.dhBase + i * p.dhStep, dw = p.dwBase + j * p.dwStep;
      const bool ok = ((unsigned)(oh + dh) < (unsigned)p.IH) & ((unsigned)(ow + dw) < (unsigned)p.IW);
      table[t * 128 + at] = (unsigned short)((ok ? at + dh + p.IH * dw - w.first : w.span) * kSlotBytes);
      i += 2;
      while (i >= p.FH) {
        i -= p.FH;
        ++j;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      frag h, mm, l;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        unsigned a, b, c;
        split_pair(first[u][2 * k] * kSplitScale, first[u][2 * k + 1] * kSplitScale, &a, &b, &c);
        h.u[k] = a;
        mm.u[k] = b;
        l.u[k] = c;
      }
      char* to = patches + unitTo[u];
      *(uintx4*)to = h.u;
      *(uintx4*)(to + 16) = mm.u;
      *(uintx4*)(to + 32) = l.u;
    }
  }
  // (the first group's bank is older than these pixels and the other groups')
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"(8 + (R - 1) * DMA) : "memory");

  // ---- the products
  floatx16 acc[PB][CB], low[PB][CB];
#pragma unroll
  for (int b = 0; b < PB; ++b)
#pragma unroll
    for (int a = 0; a < CB; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[b][a][r] = low[b][a][r] = 0.f;

  const int myTable = table_at(CT, R, w.slots) + (wpx * PB * 32 + l32) * 2;
  const int ringMine = wch * (CB * kBlockBytes) + lane * 16;
  const int myHalf = ring_bytes(CT, R) + kh * halfBytes;
  // (all in bytes: the ring's slot and the patch at hand)
  int slotAt = 0, patchAt = 0;

  frag al[CB], am[CB], ah[CB], bh[PB], bm[PB], bl[PB];
  int bAt[PB], at = ringMine;
#pragma unroll
  for (int b = 0; b < PB; ++b) {
    bAt[b] = myHalf + *(const unsigned short*)(lds + myTable + b * 64);
    bh[b].u = *(const uintx4*)(lds + bAt[b]);
    bm[b].u = *(const uintx4*)(lds + bAt[b] + 16);
  }
#pragma unroll
  for (int a = 0; a < CB; ++a) {
    al[a].u = *(const uintx4*)(lds + at + a * kBlockBytes + 2 * kFragBytes);
    am[a].u = *(const uintx4*)(lds + at + a * kBlockBytes + kFragBytes);
  }

  // Group t of a chunk.  SPLIT: this wavefront's unit of the next chunk's pixels that is split beside the first half of the
  // products and written to the other patch, the one behind it loaded.
  auto group = [&](auto tC, const int chunk) __attribute__((always_inline)) {
    constexpr int t = decltype(tC)::value, then = t + 1 == T ? 0 : t + 1, SPLIT = unit_split(T, U, t), UNIT = SPLIT < 0 ? 0 : SPLIT;
    constexpr bool LOADED = unit_loaded(T, U, R, t);
    int atThen = 0, dmaAt = 0;
    int off[PB];
    frag nh, nm, nl, bmNext[PB];
    float r0[4], r1[4];
    auto stage = [&](int k) __attribute__((always_inline)) {
      const int j = k / 7;
      switch (k % 7) {
        case 0: nh.u[j] = round_pair(px[2 * j] * kSplitScale, px[2 * j + 1] * kSplitScale); asm volatile("" : "+v"(nh.u[j])); break;
        case 1: r0[j] = fmaf(px[2 * j], kSplitScale, -__builtin_bit_cast(float, nh.u[j] << 16)); asm volatile("" : "+v"(r0[j])); break;
        case 2: r1[j] = fmaf(px[2 * j + 1], kSplitScale, -__builtin_bit_cast(float, nh.u[j] & 0xffff0000u)); asm volatile("" : "+v"(r1[j])); break;
        case 3: nm.u[j] = round_pair(r0[j], r1[j]); asm volatile("" : "+v"(nm.u[j])); break;
        case 4: r0[j] -= __builtin_bit_cast(float, nm.u[j] << 16); asm volatile("" : "+v"(r0[j])); break;
        case 5: r1[j] -= __builtin_bit_cast(float, nm.u[j] & 0xffff0000u); asm volatile("" : "+v"(r1[j])); break;
        default: nl.u[j] = round_pair(r0[j], r1[j]); asm volatile("" : "+v"(nl.u[j])); break;
      }
    };
    constexpr int TURN = 3 * NP;
#pragma unroll
    for (int i = 0; i < 6 * NP; ++i) {
      const int row = i / NP, b = i % NP / CB, a = i % CB;
      floatx16& to = row == 3 ? acc[b][a] : low[b][a];
      switch (row) {  // (the small products l h, m m, m h, h l, h m one after the other; h h apart, where its operands are free early)
        case 0: to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[a].v, bh[b].v, to, 0, 0, 0); break;
        case 1: to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am[a].v, bm[b].v, to, 0, 0, 0); break;
        case 2: to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am[a].v, bh[b].v, to, 0, 0, 0); break;
        case 3: to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a].v, bh[b].v, to, 0, 0, 0); break;
        case 4: to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a].v, bl[b].v, to, 0, 0, 0); break;
        default: to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a].v, bm[b].v, to, 0, 0, 0); break;
      }
      asm volatile("" : "+v"(to));
      // this group's other fragments, and where the next group's pixels lie
      if (row == 0) {
#pragma unroll
        for (int e = i * CB / NP; e < (i + 1) * CB / NP; ++e) ah[e].u = *(const uintx4*)(lds + at + e * kBlockBytes);
      }
      if (row == 1) {
#pragma unroll
        for (int e = (i - NP) * PB / NP; e < (i - NP + 1) * PB / NP; ++e) bl[e].u = *(const uintx4*)(lds + bAt[e] + 32);
      }
      if (i == 2 * NP - 1) {
#pragma unroll
        for (int e = 0; e < PB; ++e) off[e] = *(const unsigned short*)(lds + myTable + then * 256 + e * 64);
      }
      // the scalars' steps, a few behind each matrix instruction (a wavefront alone on its SIMD has 32 cycles behind each for
      // four of these; more of them cost 8 cycles each)
      if (i == 0 && then == 0) patchAt = patchBytes - patchAt;
      if (i == NP) {
        asm volatile("" : "+s"(slotAt));
        dmaAt = dmaTo + (own ? slotAt : 0);
        slotAt += GROUP;
        slotAt = slotAt == R * GROUP ? 0 : slotAt;
        asm volatile("" : "+s"(slotAt), "+s"(dmaAt));
        atThen = ringMine + slotAt;
      }
      if (SPLIT >= 0 && i < TURN) {
#pragma unroll
        for (int k = i * 28 / TURN; k < (i + 1) * 28 / TURN; ++k) stage(k);
      }
      if (i == TURN) {
        // This wavefront has read what it needs of the group; the next one's bank has landed (DMA loads for each of the R - 2
        // groups behind it and the pixels asked for since may be under way); what it wrote of the next chunk's pixels is in
        // LDS.  Behind the barrier the group R ahead goes where this one was.
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"((R - 2) * DMA + (LOADED ? 8 : 0)) : "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < PB; ++e) bAt[e] = myHalf + patchAt + off[e];
      }
      if (i > TURN && i <= TURN + DMA) dma_piece(bankAt, dmaAt, i - TURN - 1);
      if (i == 5 * NP - 1) {
        asm volatile("" : "+s"(bankAt));
        bankAt = min(bankAt + groupPitch, lastGroup);
        asm volatile("" : "+s"(bankAt));
      }
      if (i == 4 * NP) {
#pragma unroll
        for (int e = 0; e < CB; ++e) al[e].u = *(const uintx4*)(lds + atThen + e * kBlockBytes + 2 * kFragBytes);
      }
      if (i == 4 * NP + NP / 2) {
#pragma unroll
        for (int e = 0; e < PB; ++e) bh[e].u = *(const uintx4*)(lds + bAt[e]);
      }
      if (i == 4 * NP + NP / 2 && PB == 1) bmNext[0].u = *(const uintx4*)(lds + bAt[0] + 16);
      if (i == 5 * NP) {
#pragma unroll
        for (int e = 0; e < CB; ++e) am[e].u = *(const uintx4*)(lds + atThen + e * kBlockBytes + kFragBytes);
      }
      if (PB > 1 && row == 5 && a == CB - 1) bm[b].u = *(const uintx4*)(lds + bAt[b] + 16);
      if (SPLIT >= 0 && i == 5 * NP - 1) {
        char* write = patches + (patchBytes - patchAt) + unitTo[UNIT];
        *(uintx4*)write = nh.u;
        *(uintx4*)(write + 16) = nm.u;
        *(uintx4*)(write + 32) = nl.u;
      }
      if (i == 6 * NP - 1) {
        at = atThen;
        if (PB == 1) bm[0] = bmNext[0];
        if (SPLIT >= 0) {
          constexpr int next = UNIT + 1 == U ? 0 : UNIT + 1;
          const int from = min(next == 0 ? chunk + 2 : chunk + 1, chunkEnd - 1);  // (behind the last one: that again, for nothing)
#pragma unroll
          for (int j = 0; j < 8; ++j) px[j] = load_row(unitFrom[next], from, j);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int chunk = chunkBegin; chunk < chunkEnd; ++chunk)
    unrolled<T>([&](auto t) __attribute__((always_inline)) { group(t, chunk); });
  // (what was loaded into LDS for groups behind the last one must not land in memory that is used again)
  asm volatile("s_waitcnt vmcnt(0)\n\ts_waitcnt lgkmcnt(0)" ::: "memory");
  if (EPI == kStats || EPI == kNormalise) __syncthreads();

#pragma unroll
  for (int b = 0; b < PB; ++b)
#pragma unroll
    for (int a = 0; a < CB; ++a) acc[b][a] = (acc[b][a] + low[b][a]) * kSplitUnscale;

  // ---- an accumulator that is not finite: its pixels' blocks of the wavefront again on the fp32 instruction
#pragma unroll
  for (int b = 0; b < PB; ++b) {
    float sum = 0.f;
#pragma unroll
    for (int a = 0; a < CB; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum = fmaf(acc[b][a][r], 0.f, sum);
    if (__builtin_expect(!__any(!(sum == 0.f)), 1)) continue;
    const int m = mt * 128 + (wpx * PB + b) * 32 + l32;
    int n, q, ow, oh;
    p.byQ.divmod(m < p.M ? m : 0, &n, &q);
    p.byOH.divmod(q, &ow, &oh);
    const unsigned from = (unsigned)(n * p.inImg + q + kh * 8 * IHW) * 4u;
    if (m >= p.M) oh = -0x40000000;
#pragma unroll
    for (int a = 0; a < CB; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[b][a][r] = 0.f;
#pragma unroll 1
    for (int g = chunkBegin * T; g < chunkEnd * T; ++g) {
      const int chunk = g / T, tap = g - chunk * T, j = tap / p.FH, i = tap - j * p.FH;
      const int dh = p.dhBase + i * p.dhStep, dw = p.dwBase + j * p.dwStep;
      const bool ok = ((unsigned)(oh + dh) < (unsigned)p.IH) & ((unsigned)(ow + dw) < (unsigned)p.IW);
      const unsigned vo = ok ? from + (unsigned)((dh + p.IH * dw) * 4) : kFar;
      vbuf v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = load_row(vo, chunk, e);
#pragma unroll
      for (int a = 0; a < CB; ++a) {
        const char* at = (const char*)bank + (size_t)g * groupPitch + ((ct * WCH + wch) * CB + a) * kBlockBytes + lane * 16;
        const uintx4 h = *(const uintx4*)at, mm = *(const uintx4*)(at + kFragBytes), l = *(const uintx4*)(at + 2 * kFragBytes);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          auto part = [&](const uintx4& u) { return e & 1 ? u[e / 2] >> 16 : u[e / 2] & 0xffffu; };
          acc[b][a] = __builtin_amdgcn_mfma_f32_32x32x2f32(split_weight(part(h), part(mm), part(l)), v[e], acc[b][a], 0, 0, 0);
        }
      }
    }
  }

  // ---- epilogue
  const int coW = ct * CT;
  if (EPI == kNormalise) {
    BnCoef* coefs = (BnCoef*)lds;
    if (tid < CT && coW + tid < p.Cout) coefs[tid] = bn_coefficients(p, coW + tid);
    __syncthreads();
  }
#pragma unroll
  for (int b = 0; b < PB; ++b) {
    const int row = wpx * PB + b, m = mt * 128 + row * 32 + l32, cOff = wch * CB * 32;
    if (EPI == kTail) split_store_tail<CB>(acc[b], out, CT, cOff, row * 32 + l32, kh);
    else if (EPI == kNormalise) split_store_normalised<CB>(acc[b], out, p, (const BnCoef*)lds + cOff, coW + cOff, m, m < p.M, kh);
    else split_store<CB, EPI>(acc[b], out, bias, p, coW + cOff, m, m < p.M, kh);
    if (EPI == kStats) split_sums<CB>(acc[b], lds, wave, row, CT, cOff, l32, kh);
  }
  if (EPI == kStats) {
    __syncthreads();
    split_sums_out(lds, p, CT, coW, mt, tid);
  }
}

// CT channels x 128 pixels to a workgroup
template <int CT, int T, int U, int R, int EPI>
__global__ __launch_bounds__(256, 2) void conv_staged_mfma(float* __restrict__ out, const float* __restrict__ in,
                                                           const void* __restrict__ bank, const float* __restrict__ bias, PixP p,
                                                           StagedP w) {
  if constexpr (CT == 128) staged_body<2, 2, 2, T, U, R, EPI>(out, in, bank, bias, p, w, blockIdx.x, gridDim.x);
  else staged_body<1, 2, 4, T, U, R, EPI>(out, in, bank, bias, p, w, blockIdx.x, gridDim.x);
}

// The same with the tiles from w.tileBase on, left over after whole rounds, in tiles of 32 channels: blocks from `whole` on
// (see plan_ends of conv_split.hip)
template <int CT, int T, int U, int R, int EPI>
__global__ __launch_bounds__(256, 2) void conv_staged_ends(float* __restrict__ out, const float* __restrict__ in,
                                                           const void* __restrict__ bank, const float* __restrict__ bias, PixP p,
                                                           StagedP w, StagedP v, unsigned whole) {
  if (blockIdx.x >= whole) staged_body<1, 1, 4, T, U, R, EPI>(out, in, bank, bias, p, v, blockIdx.x - whole, gridDim.x - whole, v.tileBase);
  else if constexpr (CT == 128) staged_body<2, 2, 2, T, U, R, EPI>(out, in, bank, bias, p, w, blockIdx.x, whole);
  else staged_body<1, 2, 4, T, U, R, EPI>(out, in, bank, bias, p, w, blockIdx.x, whole);
}

constexpr size_t kLdsMost = 160 * 1024;

size_t lds_bytes(int CT, int T, int R, int slots, int epi) {
  const size_t loop = (size_t)table_at(CT, R, slots) + (size_t)T * 128 * sizeof(unsigned short);
  return epi == kStats ? std::max(loop, stats_lds_bytes(CT)) : loop;
}

// ends: this many blocks more in tiles of 32 channels, of geometry v
template <int CT, int T, int U, int R, int EPI>
int go(hipStream_t s, unsigned blocks, unsigned ends, float* out, const float* in, const void* bank, const float* bias, const PixP& p,
       const StagedP& w, const StagedP& v) {
  const size_t lds = lds_bytes(CT, p.T, R, w.slots, EPI);
  constexpr bool ENDS = EPI != kTail && T == 9;
  const void* kernels[2] = {(const void*)conv_staged_mfma<CT, T, U, R, EPI>, nullptr};
  if constexpr (ENDS) kernels[1] = (const void*)conv_staged_ends<CT, T, U, R, EPI>;
  if (lds > 64 * 1024) {
    static std::atomic<bool> raisedOn[2][kMaxDevices];  // opt-in to more than 64 KB of LDS per workgroup, once per device
    const int dev = current_device(), k = ends ? 1 : 0;
    const bool known = dev >= 0 && dev < kMaxDevices;
    if (!known || !raisedOn[k][dev].load(std::memory_order_acquire)) {
      if (hipFuncSetAttribute(kernels[k], hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMost) != hipSuccess) {
        (void)hipGetLastError();
        return fail(MCN_DEVICE_ERROR, "convolution: cannot reserve %zu bytes of LDS", lds);
      }
      if (known) raisedOn[k][dev].store(true, std::memory_order_release);
    }
  }
  KernelTimer timer(EPI == kTail ? "conv_split_mfma_staged_tail" : ends ? "conv_split_mfma_ends_staged" : "conv_split_mfma_staged", s);
  if constexpr (ENDS) {
    if (ends) {
      hipLaunchKernelGGL((conv_staged_ends<CT, T, U, R, EPI>), dim3(blocks + ends), dim3(256), lds, s, out, in, bank, bias, p, w, v, blocks);
      return MCN_SUCCESS;
    }
  }
  hipLaunchKernelGGL((conv_staged_mfma<CT, T, U, R, EPI>), dim3(blocks), dim3(256), lds, s, out, in, bank, bias, p, w);
  return MCN_SUCCESS;
}

template <int CT, int T, int U, int R>
int go_epi(hipStream_t s, int epi, unsigned blocks, unsigned ends, float* out, const float* in, const void* bank, const float* bias, const PixP& p,
           const StagedP& w, const StagedP& v) {
  if constexpr (T == 9) {
    if (epi == kStats) return go<CT, T, U, R, kStats>(s, blocks, ends, out, in, bank, bias, p, w, v);
    if (epi == kNormalise) return go<CT, T, U, R, kNormalise>(s, blocks, ends, out, in, bank, bias, p, w, v);
    if (epi == kMaskedAdd) return go<CT, T, U, R, kMaskedAdd>(s, blocks, ends, out, in, bank, bias, p, w, v);
  }
  if (epi == kTail) return go<CT, T, U, R, kTail>(s, blocks, ends, out, in, bank, bias, p, w, v);
  return go<CT, T, U, R, kStore>(s, blocks, ends, out, in, bank, bias, p, w, v);
}

// in tiles of 32 WA channels; two workgroups to a CU have the LDS where the pixels leave it
template <int T>
int go_taps(hipStream_t s, int WA, int epi, unsigned blocks, unsigned ends, float* out, const float* in, const void* bank, const float* bias,
            const PixP& p, const StagedP& w, const StagedP& v) {
  if (WA == 2) return go_epi<64, T, 2, 3>(s, epi, blocks, ends, out, in, bank, bias, p, w, v);
  const int units = (w.slots / 64 * 2 + 3) / 4;  // of a wavefront
  if constexpr (most_units(T, 4) > 2) {
    if (units > 2) return go_epi<128, T, 3, 2>(s, epi, blocks, ends, out, in, bank, bias, p, w, v);
  }
  if (2 * lds_bytes(128, T, 3, w.slots, epi) <= kLdsMost) return go_epi<128, T, 2, 3>(s, epi, blocks, ends, out, in, bank, bias, p, w, v);
  return go_epi<128, T, 2, 2>(s, epi, blocks, ends, out, in, bank, bias, p, w, v);
}

}  // namespace

int conv_staged_launch_25(hipStream_t s, int WA, int epi, unsigned blocks, unsigned ends, float* out, const float* in, const void* bank,
                          const float* bias, const PixP& p, const StagedP& w, const StagedP& v);

}  // namespace mcn
