// Convolution (forward and backward-data) over few pixels, on the bf16 matrix instruction with operands split in three.
//
// conv_split.hip's tiles of 128 pixels leave such products a handful of workgroups: their reductions are cut over the chip and
// a second launch adds the partial results up.  What bounds them is neither rate but the chain of one launch: start, addresses,
// first loads, as many groups of 16 rows one after the other as a wavefront has, sum, store (some 7 us), and again for the
// second launch (4 us; 33 of the 53 products of ResNet-50 over one image had one).
//
// Here a workgroup owns a small tile, 16 WA channels x 32 pixels, and its wavefronts share the reduction: wavefront w
// multiplies pairs of groups w, w + NW, ... and the partial results meet in LDS, where they are added two by two and
// stored with whatever is behind the product.  One launch, no partial results in memory, NW short chains in flight per tile.
//   * v_mfma_f32_16x16x32_bf16: the 32 rows are two groups of conv_split.hip's bank (lane quarter kq: group kq / 2, rows
//     8 (kq % 2) ...), whose fragments a lane reads straight into registers, 16 bytes a part; a group's pixels are read as
//     there, eight rows of a pixel to a lane, and split in registers.  Nothing is shared between wavefronts before the sum, so
//     there is no barrier before it.
//   * 1x1 filters: both operands of a wavefront's next pair are loaded before this one's are multiplied.
//   * Filters with taps: read from memory for every tap, pixels were two thirds of what a CU's 64 bytes per clock had to
//     bring (3x3x256x256 over 14x14: 15 us, 11 staged).  The pixels under the tile and its taps are split once into LDS, all
//     channels of them (a barrier), and the loop reads only the bank, four pairs ahead.
//   * Neighbouring workgroups, behind one L2, share what is larger, their part of the bank or the pixels.
// The numbers are conv_split.hip's: six products, accumulators of their own for the product h h, the fp32 instruction where one
// is not finite.
#include "conv_common.hpp"

#include <algorithm>
#include <atomic>

namespace mcn {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kPixels = 32;
constexpr size_t kStagedMost = 152 * 1024;  // LDS of a workgroup for staged pixels
constexpr int kPitch = 36;  // floats from one channel of a partial result to the next (four rows of lanes: all banks)

struct ShortP {
  int pixelsInner;  // neighbouring workgroups have the same channels (else the same pixels)
  int blocksC;   // 32-channel blocks of the bank
  int groups;    // chunks x taps
  int pairs;     // of groups (the bank is padded to whole slabs of four)
  unsigned inBytes, bankBytes;
  FastDiv byInner, byFH;
  // kStaged: pixels from `first` before a tile's first one on, `span` of them, in rows of `slots`
  int first, span, slots;
  FastDiv bySlots, byIHW;
};

// Where a wavefront's pixels come from: memory (1x1 filters), or LDS, where they were split once for all taps
enum { kPoint = 0, kStaged = 1 };

template <int WA, int NW, int MODE>
__global__ __launch_bounds__(64 * NW, NW / 4) void conv_split_short(float* __restrict__ out, const float* __restrict__ in,
                                                                    const void* __restrict__ bank, const float* __restrict__ bias,
                                                                    PixP p, ShortP w) {
  constexpr bool TAPS = MODE == kStaged;
  constexpr int CT = 16 * WA;
  constexpr int TILE = CT * kPitch;  // floats of a partial result
  extern __shared__ __attribute__((aligned(16))) float sums[];  // [NW][TILE]; before that the staged pixels

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kq = lane >> 4, kh = kq & 1;
  const int IHW = p.IH * p.IW;

  // (neighbours, behind one L2, share what is the larger of the two: a pixel tile's pixels or a channel tile's part of the bank)
  const int logical = xcd_contiguous_id((int)blockIdx.x, (int)gridDim.x);
  int outer, inner;
  w.byInner.divmod(logical, &outer, &inner);
  const int mt = w.pixelsInner ? inner : outer, ct = w.pixelsInner ? outer : inner;

  // ---- where this lane's operands lie
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)in, 0, (int)w.inBytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc((void*)bank, 0, (int)w.bankBytes, 0x00020000);
  int ihB[2], iwB[2], pix[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int m = mt * kPixels + 16 * b + l16;
    const bool valid = m < p.M;
    int n, q, ow, oh;
    p.byQ.divmod(valid ? m : 0, &n, &q);
    p.byOH.divmod(q, &ow, &oh);
    ihB[b] = valid ? oh * p.sy : -0x40000000;  // (never inside the image)
    iwB[b] = ow * p.sx;
    pix[b] = n * p.inImg + oh * p.sy + p.IH * iwB[b] + kh * 8 * IHW;
  }
  const int groupPitch = w.blocksC * kBlockBytes;
  unsigned bankAt[WA];
#pragma unroll
  for (int a = 0; a < WA; ++a) {
    const int c = ct * CT + 16 * a;
    bankAt[a] = (unsigned)((kq >> 1) * groupPitch + (c / 32) * kBlockBytes + (kh * 32 + c % 32 + l16) * 16);
  }

  struct Weights { uintx4 h[WA], m[WA], l[WA]; };
  struct Operands : Weights { float px[2][8]; };
  struct Tap { int chunk, dh, dw, shift; bool present; };
  auto tap_of = [&](int pair) __attribute__((always_inline)) -> Tap {  // this lane's group of a pair
    const int g = 2 * pair + (kq >> 1);
    Tap t = {g, p.dhBase, p.dwBase, 0, g < w.groups};
    if (TAPS) {
      int k, i, j;
      p.byT.divmod(g, &t.chunk, &k);
      w.byFH.divmod(k, &j, &i);
      t.dh += i * p.dhStep;
      t.dw += j * p.dwStep;
      t.shift = t.dh + p.IH * t.dw;
    }
    return t;
  };
  auto inside = [&](const Tap& t, int b) __attribute__((always_inline)) -> bool {
    if (!TAPS) return t.present & (ihB[b] >= 0);
    return t.present & ((unsigned)(ihB[b] + t.dh) < (unsigned)p.IH) & ((unsigned)(iwB[b] + t.dw) < (unsigned)p.IW);
  };
  auto load_weights = [&](int pair, Weights& o) __attribute__((always_inline)) {
    const int so = 2 * pair * groupPitch;
#pragma unroll
    for (int a = 0; a < WA; ++a) {
      o.h[a] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(brsrc, (int)bankAt[a], so, 0));
      o.m[a] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(brsrc, (int)bankAt[a], so + kFragBytes, 0));
      o.l[a] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(brsrc, (int)bankAt[a], so + 2 * kFragBytes, 0));
    }
  };
  auto load = [&](int pair, Operands& o) __attribute__((always_inline)) {
    const Tap t = tap_of(pair);
    const int shift = t.chunk * 16 * IHW + t.shift;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const unsigned vo = inside(t, b) ? (unsigned)(pix[b] + shift) * 4u : kOutside;
#pragma unroll
      for (int j = 0; j < 8; ++j) o.px[b][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)vo, j * IHW * 4, 0));
    }
    load_weights(pair, o);
  };

  // The products h h of a few pairs, and of those before; the other five.  (An accumulator's error grows with the root of the
  // rows it has taken, 1.0e-7 of the result over 128, 1.4e-7 over 576: none takes more than four pairs.)
  floatx4 acc[WA][2], done[WA][2], low[WA][2];
#pragma unroll
  for (int a = 0; a < WA; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[a][b][r] = done[a][b][r] = low[a][b][r] = 0.f;
  auto set_aside = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        done[a][b] += acc[a][b];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[a][b][r] = 0.f;
      }
  };
  auto products = [&](const Weights& o, int b, const uintx4& h, const uintx4& m, const uintx4& l) __attribute__((always_inline)) {
    auto mfma = [](const uintx4& x, const uintx4& y, floatx4 c) __attribute__((always_inline)) {
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), c, 0, 0, 0);
    };
#pragma unroll
    for (int a = 0; a < WA; ++a) low[a][b] = mfma(o.l[a], h, low[a][b]);
#pragma unroll
    for (int a = 0; a < WA; ++a) acc[a][b] = mfma(o.h[a], h, acc[a][b]);
#pragma unroll
    for (int a = 0; a < WA; ++a) low[a][b] = mfma(o.m[a], m, low[a][b]);
#pragma unroll
    for (int a = 0; a < WA; ++a) low[a][b] = mfma(o.m[a], h, low[a][b]);
#pragma unroll
    for (int a = 0; a < WA; ++a) low[a][b] = mfma(o.h[a], l, low[a][b]);
#pragma unroll
    for (int a = 0; a < WA; ++a) low[a][b] = mfma(o.h[a], m, low[a][b]);
  };
  auto split8 = [&](const float (&v)[8], uintx4* h, uintx4* m, uintx4* l) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned uh, um, ul;
      split_pair(v[2 * j] * kSplitScale, v[2 * j + 1] * kSplitScale, &uh, &um, &ul);
      (*h)[j] = uh;
      (*m)[j] = um;
      (*l)[j] = ul;
    }
  };
  if constexpr (MODE == kStaged) {
    // All channels of the pixels under the tile and its taps, split: of each half-chunk (8 channels) and part a row of
    // `slots` pixels, 16 bytes each.  In one image and the next pixels are numbered on; what lies before the first or
    // behind the last image is never asked for.
    constexpr int AHEAD = 4;
    Weights ring[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD - 1; ++i)
      if (wave + i * NW < w.pairs) load_weights(wave + i * NW, ring[i]);
    const int items = w.groups / p.T * 2 * w.slots;
    const int firstPixel = mt * kPixels + w.first, allPixels = p.N * IHW;
    char* const stage = (char*)sums;
    const int rowBytes = w.slots * 16, zeros = w.groups / p.T * 6 * rowBytes;  // (16 bytes behind them, for what lies outside)
    if (tid == 0) *(uintx4*)(stage + zeros) = (uintx4){0u, 0u, 0u, 0u};
    constexpr int BATCH = 2;
    for (int i0 = tid; i0 < items; i0 += BATCH * 64 * NW) {
      float v[BATCH][8];
      int half[BATCH], slot[BATCH];
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
        const int i = i0 + u * 64 * NW;
        w.bySlots.divmod(min(i, items - 1), &half[u], &slot[u]);
        const int L = firstPixel + slot[u];
        const bool ok = i < items & slot[u] < w.span & (unsigned)L < (unsigned)allPixels;
        int n, q;
        w.byIHW.divmod(ok ? L : 0, &n, &q);
        const unsigned vo = ok ? (unsigned)(n * p.inImg + q + half[u] * 8 * IHW) * 4u : kOutside;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[u][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)vo, j * IHW * 4, 0));
      }
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
        uintx4 h, m, l;
        split8(v[u], &h, &m, &l);
        if (i0 + u * 64 * NW < items) {
          char* at = stage + (size_t)half[u] * 3 * rowBytes + slot[u] * 16;
          *(uintx4*)at = h;
          *(uintx4*)(at + rowBytes) = m;
          *(uintx4*)(at + 2 * rowBytes) = l;
        }
      }
    }
    __syncthreads();
    auto step = [&](int pair, const Weights& o) __attribute__((always_inline)) {
      const Tap t = tap_of(pair);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const bool ok = inside(t, b);
        const int pitch = ok ? rowBytes : 0;
        const char* at = stage + (ok ? (2 * t.chunk + kh) * 3 * rowBytes + (16 * b + l16 + t.shift - w.first) * 16 : zeros);
        products(o, b, *(const uintx4*)at, *(const uintx4*)(at + pitch), *(const uintx4*)(at + 2 * pitch));
      }
    };
    int pair = wave;
    for (; pair < w.pairs; pair += AHEAD * NW) {
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        if (pair + (i + AHEAD - 1) * NW < w.pairs) load_weights(pair + (i + AHEAD - 1) * NW, ring[(i + AHEAD - 1) % AHEAD]);
        if (pair + i * NW < w.pairs) step(pair + i * NW, ring[i]);
      }
      set_aside();
    }
    __syncthreads();  // (the partial results take the staged pixels' place)
  } else if (wave < w.pairs) {
    auto multiply = [&](const Operands& o) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        uintx4 h, m, l;
        split8(o.px[b], &h, &m, &l);
        products(o, b, h, m, l);
      }
    };
    Operands x, y;
    load(wave, x);
    for (int pair = wave; pair < w.pairs; pair += 2 * NW) {
      if (pair + NW < w.pairs) load(pair + NW, y);
      multiply(x);
      if (pair + NW < w.pairs) {
        if (pair + 2 * NW < w.pairs) load(pair + 2 * NW, x);
        multiply(y);
      }
      set_aside();
    }
  }

  // ---- the outputs of this thread: what is behind the product is read while the partial results are on their way
  constexpr int PER = CT * kPixels / (64 * NW) > 0 ? CT * kPixels / (64 * NW) : 1;
  auto element = [&](int e, int* c, int* px) {  // element e of the tile: pixels fastest
    *c = e / kPixels;
    *px = e % kPixels;
  };
  auto put = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) sums[wave * TILE + (16 * a + 4 * kq + r) * kPitch + 16 * b + l16] = acc[a][b][r];
  };
  float t = 0.f;
#pragma unroll
  for (int a = 0; a < WA; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      acc[a][b] = (done[a][b] + low[a][b]) * kSplitUnscale;
#pragma unroll
      for (int r = 0; r < 4; ++r) t = fmaf(acc[a][b][r], 0.f, t);
    }
  put();
  if (__builtin_expect(__syncthreads_or(!(t == 0.f)), 0)) {
    // an accumulator that is not finite: the tile again on the fp32 instruction
#pragma unroll
    for (int a = 0; a < WA; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[a][b][r] = 0.f;
#pragma unroll 1
    for (int pair = wave; pair < w.pairs; pair += NW) {
      Operands o;
      load(pair, o);
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int a = 0; a < WA; ++a) {
          auto part = [&](const uintx4& u) { return j & 1 ? u[j / 2] >> 16 : u[j / 2] & 0xffffu; };
          const float wv = split_weight(part(o.h[a]), part(o.m[a]), part(o.l[a]));
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv, o.px[b][j], acc[a][b], 0, 0, 0);
        }
    }
    put();
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = i * 64 * NW + tid;
    int c, px;
    element(e, &c, &px);
    const int co = ct * CT + c, m = mt * kPixels + px;
    const bool inTile = CT * kPixels >= 64 * NW || e < CT * kPixels;
    const bool present = inTile && co < p.Cout && m < p.M;
    float sum = 0.f;
    if (inTile) {
      float v[NW];
#pragma unroll
      for (int k = 0; k < NW; ++k) v[k] = sums[k * TILE + c * kPitch + px];
#pragma unroll
      for (int half = NW / 2; half > 0; half /= 2)
#pragma unroll
        for (int k = 0; k < half; ++k) v[k] += v[k + half];
      sum = v[0];
    }
    if (present) {
      int n, q;
      p.byQ.divmod(m, &n, &q);
      const size_t at = (size_t)n * p.outImg + out_pixel_offset(p, q) + (size_t)co * p.outPlane;
      float* o = out + at;
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
    if (p.stats) {  // (uniform; alpha = 1, beta = 0, no bias, whole blocks of channels: `sum` is what was stored, 0 past the last pixel)
      double t1 = (double)sum, t2 = t1 * t1;
#pragma unroll
      for (int lanes = 16; lanes > 0; lanes >>= 1) {
        t1 += __shfl_xor(t1, lanes);
        t2 += __shfl_xor(t2, lanes);
      }
      if (px == 0 && inTile && co < p.Cout) {
        double* o = p.stats + ((size_t)co * p.statGroups + mt) * 2;
        o[0] = t1;
        o[1] = t2;
      }
    }
  }
}

// 1x1 filters without padding, any stride
bool point(const PixP& p) {
  return p.T == 1 && p.dhBase == 0 && p.dwBase == 0 && (p.OH - 1) * p.sy < p.IH && (p.OW - 1) * p.sx < p.IW;
}

// The pixels under a tile of 32 and its taps, all channels, in LDS: for products whose output lies on the grid of their input.
// 0: too many, or none such.
size_t staged_bytes(const PixP& p, ShortP* w) {
  if (p.T == 1 || p.sy != 1 || p.sx != 1 || p.OH != p.IH || p.OW != p.IW) return 0;
  const int FW = p.T / p.FH;
  const int lastH = p.dhBase + (p.FH - 1) * p.dhStep, lastW = p.dwBase + (FW - 1) * p.dwStep;
  const long long first = std::min(p.dhBase, lastH) + (long long)p.IH * std::min(p.dwBase, lastW);
  const long long span = kPixels + std::max(p.dhBase, lastH) + (long long)p.IH * std::max(p.dwBase, lastW) - first;
  const long long slots = (span + 15) / 16 * 16, bytes = p.Cin / 8 * 3 * slots * 16 + 16;
  if (bytes > (long long)kStagedMost) return 0;
  w->first = (int)first;
  w->span = (int)span;
  w->slots = (int)slots;
  return (size_t)bytes;
}

template <int WA, int NW, int MODE>
int go(hipStream_t s, unsigned blocks, size_t staged, float* out, const float* in, const void* bank, const float* bias, const PixP& p, const ShortP& w) {
  const size_t lds = std::max((size_t)NW * 16 * WA * kPitch * sizeof(float), staged);
  if (lds > 64 * 1024) {
    static std::atomic<bool> raisedOn[kMaxDevices];  // opt-in to more than 64 KB of LDS per workgroup, once per device
    const int dev = current_device();
    const bool known = dev >= 0 && dev < kMaxDevices;
    if (!known || !raisedOn[dev].load(std::memory_order_acquire)) {
      if (hipFuncSetAttribute((const void*)conv_split_short<WA, NW, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kStagedMost) != hipSuccess) {
        (void)hipGetLastError();
        return fail(MCN_DEVICE_ERROR, "convolution: cannot reserve %zu bytes of LDS", lds);
      }
      if (known) raisedOn[dev].store(true, std::memory_order_release);
    }
  }
  KernelTimer timer("conv_split_short", s);
  hipLaunchKernelGGL((conv_split_short<WA, NW, MODE>), dim3(blocks), dim3(64 * NW), lds, s, out, in, bank, bias, p, w);
  return MCN_SUCCESS;
}

}  // namespace

// Channels per workgroup and wavefronts, or none: whichever of the three kinds and conv_split.hip's launches (`others`: their
// modelled time, with the sum of partial results) takes the least modelled time.  The times are fitted to 220 products of 16
// to 8000 pixels and up to 1e9 operations in captured graphs, cold banks (within 8 to 15 % of them): a launch, a wavefront's pairs, what all
// workgroups on a CU have to multiply, their start, and the pixels they stage.  Over those products the time falls by a factor
// of 1.31 (1.35 if the better kernel were always known), at most 4 % is lost: 3x3x256x256 over 14x14 14.1 -> 9.2 us, 3x3x512x512
// over 7x7 18.8 -> 12.8, 1x1x512x128 over 28x28 9.1 -> 5.5, 1x1x64x256 over 56x56 5.4 (6.9 here), 1x1x1024x256 over 14x14x8
// 16.3 -> 13.2.
ShortPlan conv_short_plan(const PixP& p) {
  struct Kind { int wa, waves; double pointUs[4], stagedUs[5]; };
  static const Kind kinds[] = {
      {1, 8, {2.66, 0.82, 0.078, 0.71}, {3.15, 0.45, 0.028, 0.91, 0.94}},
      {1, 16, {1.85, 1.60, 0.091, 1.61}, {2.70, 0.90, 0.001, 2.49, 1.35}},
      {2, 4, {3.51, 0.54, 0.091, 0.70}, {3.51, 0.52, 0.020, 0.81, 1.81}},
  };
  const ShortPlan none = {0, 0};
  const int forced = tunable("conv_short", 0);
  if (p.Cin % 16 != 0 || forced < 0 || tunable("conv_split_wa", 0) || tunable("conv_split_splits", 0)) return none;
  if (!forced && (p.M > 8192 || 2.0 * p.M * p.R * p.Cout > 1e9)) return none;  // (what the times were fitted to)
  ShortP w;
  const bool isPoint = point(p);
  if (!isPoint && !staged_bytes(p, &w)) return none;
  if (forced) return {forced / 100, forced % 100};
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  const int pairs = (p.Cin / 16 * p.T + 1) / 2;
  ShortPlan best = none;
  double bestUs = 0.95 * (2.15 + 0.98 * conv_split_modelled_us(p.Cin, p.T, p.Cout, p.M));
  for (const Kind& k : kinds) {
    const double perCu = (double)((p.M + kPixels - 1) / kPixels) * ((p.Cout + 16 * k.wa - 1) / (16 * k.wa)) / cus;
    const double* c = isPoint ? k.pointUs : k.stagedUs;
    double us = c[0] + c[1] * ((pairs + k.waves - 1) / k.waves) + c[2] * perCu * pairs + c[3] * perCu;
    if (!isPoint) us += c[4] * perCu * (p.Cin / 8 * w.slots / 1024.0);
    if (us < bestUs) {
      bestUs = us;
      best = {k.wa, k.waves};
    }
  }
  return best;
}

int conv_short_stat_groups(long long M) { return (int)((M + kPixels - 1) / kPixels); }

int conv_short_launch(hipStream_t s, const char* who, const ShortPlan& plan, float* out, const float* in, const void* bank, const float* bias,
                      const PixP& p) {
  ShortP w;
  w.blocksC = conv_split_bank_blocks(p.Cout);
  w.groups = p.Cin / 16 * p.T;
  w.pairs = (w.groups + 1) / 2;
  w.inBytes = (unsigned)(((long long)(p.N - 1) * p.inImg + (long long)p.Cin * p.IH * p.IW) * 4);
  w.bankBytes = (unsigned)conv_split_bank_bytes(p.Cin, p.T, p.Cout);
  const int tilesC = (p.Cout + 16 * plan.wa - 1) / (16 * plan.wa), tilesM = (p.M + kPixels - 1) / kPixels;
  w.pixelsInner = w.bankBytes > w.inBytes;
  w.byInner = FastDiv(w.pixelsInner ? tilesM : tilesC);
  w.byFH = FastDiv(p.FH);
  w.first = w.span = w.slots = 0;
  const size_t staged = staged_bytes(p, &w);
  w.bySlots = FastDiv(w.slots);
  w.byIHW = FastDiv(p.IH * p.IW);
  const unsigned blocks = (unsigned)tilesM * (unsigned)tilesC;
  int rc;
#define SHORT_GO(WA, NW)                                                                          \
  rc = staged ? go<WA, NW, kStaged>(s, blocks, staged, out, in, bank, bias, p, w) : go<WA, NW, kPoint>(s, blocks, 0, out, in, bank, bias, p, w)
  if (plan.wa == 2) SHORT_GO(2, 4);
  else if (plan.waves == 16) SHORT_GO(1, 16);
  else SHORT_GO(1, 8);
#undef SHORT_GO
  return rc ? rc : check_launch(who);
}

}  // namespace mcn
