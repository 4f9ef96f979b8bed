// Geometry shared by the convolution kernels.
#pragma once

#include "mcn_internal.hpp"

#include <vector>

namespace mcn {

struct ConvP {
  int H, W, C, N;
  int FH, FW, FC, K;
  int sy, sx, pt, pl, dy, dx;
  int outH, outW;
  int groups, Kg;  // Kg = filters per group
};

// Validates like the MEX driver (vl_nnconv.cu:269-342) and fills the derived fields.
int conv_setup(const mcn_conv_geom* g, const char* who, ConvP* p);

// direct (one accumulator per output element) kernels: any stride / dilation / padding / groups
int conv_forward_direct(hipStream_t s, const ConvP& p, float* y, float outMult, const float* x, float inMult,
                        const float* f, const float* b);
int conv_backward_data_direct(hipStream_t s, const ConvP& p, float* dx, float dxMult, const float* f, const float* dy);
int conv_backward_filter_direct(hipStream_t s, const ConvP& p, float* df, const float* x, const float* dy);

// The taps of a stored FH x FW filter that take part in one product: (i0 + a*iStep, j0 + b*jStep), a < nI, b < nJ
// (all of them for a plain layer; one stride class for the backward-data product of a strided layer).
struct TapSet {
  int FH, FW;            // the filter as stored
  int i0, iStep, nI;
  int j0, jStep, nJ;
};

// One re-laying of (part of) a filter bank into the order the MFMA kernels read: a launch of conv_pack_weights, or
// one entry of a batched launch.  Plain data: it crosses the C ABI as mcn_conv_pack_job.
struct PackJob {
  float* wt;
  const float* f;
  TapSet taps;
  int Cin, Cout, rPad, coutPad, backward, tapMajor;
  unsigned firstBlock, blocks;  // workgroups [firstBlock, firstBlock + blocks) of a batched launch
};

// Filter banks packed ahead of the calls that use them.  The products of a layer visit their banks in a fixed
// order (groups, then stride classes); every bank takes a 256-byte aligned slot of the caller's buffer in that
// order, so planning, packing and using agree on where each one lies.
struct PackCtx {
  enum Mode { kPlan, kPack, kUse };
  Mode mode;
  char* base;                  // the caller's buffer (null when only the size is wanted)
  size_t capacity, offset;
  std::vector<PackJob>* jobs;  // kPlan: the jobs are appended here instead of being launched
};

// The sum over reduction splits that finishes a filter gradient (conv_wgrad_reduce), as data: one entry of a batched
// launch.  Plain data: it crosses the C ABI as mcn_conv_reduce_job.
struct ReduceJob {
  float* df;
  const float* partials;
  size_t n;               // elements of the bank
  int splits, tapMajor, C, T;
  unsigned firstBlock, blocks;
};

// Filter gradients whose final sum is deferred: the matrix kernel leaves its partial banks in the caller's buffer
// (one 256-byte aligned slot per filter group, in group order) and the sums of many layers run in one launch later.
struct ReduceCtx {
  char* base;
  size_t capacity, offset;
  std::vector<ReduceJob>* jobs;  // not null: the jobs are appended here
  bool launch;                   // false: plan only (sizes and jobs), nothing is launched
};

// MFMA implicit-GEMM kernels (groups == 1).  *_supported says whether the fast path covers `p`.
bool conv_mfma_forward_supported(const ConvP& p);
bool conv_mfma_backward_data_supported(const ConvP& p);
bool conv_mfma_backward_filter_supported(const ConvP& p);
// first layers (few input channels, 32 or 64 filters): filter gradient and, from the same pass, bias gradient
// (conv_first.hip); dB may be null
bool conv_first_backward_filter_supported(const ConvP& p);
size_t conv_first_workspace_bytes(const ConvP& p);
// (their forward product; and their input gradient at stride 1, on vector FMAs: at most four channels come out)
bool conv_first_forward_supported(const ConvP& p);
struct BnAfter;
int conv_first_forward(hipStream_t s, const ConvP& p, float* y, const float* x, const float* f, const float* bias, const BnAfter* bn = nullptr);
bool conv_first_backward_data_supported(const ConvP& p);
int conv_first_backward_data(hipStream_t s, const ConvP& p, float* dx, const float* f, const float* dy);
int conv_first_backward_filter(hipStream_t s, const ConvP& p, float* dF, float* dB, const float* x, const float* dy, void* ws,
                               size_t wsBytes);
size_t conv_mfma_workspace_bytes(const ConvP& p, int product);
// bn: a batch normalisation with given moments behind the product (see PixP::bnMoments); bnQuery: plan only
// (conv: where the product's own output goes, of first layers only; may be null)
struct BnAfter { const float *moments, *mult, *bias, *residual; int relu; float* conv; };
// stats / statGroups: also write per-channel partial sums of y and y^2 (see PixP::stats); statQuery: plan only
int conv_forward_mfma(hipStream_t s, const ConvP& p, float* y, float outMult, const float* x, float inMult,
                      const float* f, const float* b, void* ws, size_t wsBytes, PackCtx* pk = nullptr,
                      double* stats = nullptr, int statGroups = 0, int* statQuery = nullptr, const BnAfter* bn = nullptr,
                      int* bnQuery = nullptr);
// addend / addBits: a masked second term added in the epilogue (see PixP::addend); addQuery: plan only
int conv_backward_data_mfma(hipStream_t s, const ConvP& p, float* dx, float dxMult, const float* f, const float* dy,
                            void* ws, size_t wsBytes, PackCtx* pk = nullptr, const float* addend = nullptr,
                            const unsigned* addBits = nullptr, int* addQuery = nullptr);
int conv_pack_batch(hipStream_t s, const PackJob* deviceJobs, int nJobs, unsigned totalBlocks);
int conv_backward_filter_mfma(hipStream_t s, const ConvP& p, float* df, const float* x, const float* dy, void* ws,
                              size_t wsBytes, ReduceCtx* deferred = nullptr);
int conv_reduce_batch(hipStream_t s, const ReduceJob* deviceJobs, int nJobs, unsigned totalBlocks);

// Parameters of the pixel-major products (forward / backward-data): out[co, m] = sum_R wt[R][co] * in[ci(R), pixel(m) + tap(R)]
struct PixP {
  int IH, IW, Cin;    // grid and channels of the gathered tensor
  int OH, OW, Cout;   // grid and channels of the produced tensor
  int N;
  int FH, T;          // filter height, taps = FH*FW
  int sy, sx;         // gathered row = oh*sy + dh(tap)
  int dhBase, dhStep, dwBase, dwStep;
  int R;              // reduction length = T*Cin
  int coutPad;        // row pitch of wt
  int M;              // OH*OW*N (< 2^31)
  float alpha, beta;
  FastDiv byQ, byOH, byT;  // Q = OH*OW; T = taps
  int advC, advT;          // 16 = advC*T + advT (reduction rows per step)
  unsigned outBytes;       // bytes from `out` to the end of the produced tensor, or 0 when >= 2 GiB (no buffer descriptor)
  // tiled kernel, loads straight into LDS: bytes of the gathered tensor and of the packed bank (both < 2 GiB), else 0
  unsigned inBytes = 0, wtBytes = 0;
  // Where things lie, in elements.  The gathered tensor: image n, channel ci at in + n*inImg + ci*IH*IW.  The produced
  // tensor: pixel (oh, ow) of image n, channel co at out + n*outImg + co*outPlane + outOff + oh*outSH + ow*outSW.
  // A plain layer has inImg = Cin*IH*IW, outImg = Cout*OH*OW, outPlane = OH*OW, outOff = 0, outSH = 1, outSW = OH
  // (dense = 1: the pixel offset is the pixel index itself); a filter group sees a slice of the channels of a
  // wider tensor, a stride class of a strided layer's backward-data product a sub-grid of the pixels.
  int inImg, outImg, outPlane, outOff, outSH, outSW, dense;
  // Split reduction (tiled kernel only; 1 = none): workgroup `split` multiplies steps [split*stepsPerSplit, ...) of
  // 16 rows and writes its partial result to out + split*partStride (dense layout, alpha = 1, beta = 0, no bias);
  // conv_pix_reduce then adds the partials up.  For layers with few output pixels and a long reduction
  // (fully-connected layers above all), which would otherwise keep a handful of workgroups busy for a long time.
  int rSplits, stepsPerSplit;
  long long partStride;
  // Per-channel sums of the produced tensor taken in the same launch (weights-stationary kernel only): where the
  // partial sums go, and how many of them each channel gets.  statQuery (host only): no launch, just report that
  // number (0: this product has no such form).
  double* stats = nullptr;
  int statGroups = 0;
  int* statQuery = nullptr;
  // A second term added in the epilogue (weights-stationary kernel only, dense whole 32-channel blocks, planes of a
  // multiple of 32 elements, alpha = 1, beta = 0, no bias): out = acc + (bit ? addend : addend*0), addend a tensor of
  // the produced tensor's layout, bit = bit e % 32 of word e / 32 of addBits for element e.  addQuery (host only): no
  // launch, just report whether the product has this form.
  const float* addend = nullptr;
  const unsigned* addBits = nullptr;
  int* addQuery = nullptr;
  // A batch normalisation with given moments (mean, sigma: Cout of each), an optional second term of the produced
  // tensor's layout and an optional ReLU behind the product, in its epilogue or in the pass that adds up a split
  // reduction (conv_split.hip only; alpha = 1, beta = 0, no bias, dense).  bnQuery (host only) as addQuery.
  const float* bnMoments = nullptr;
  const float *bnMult = nullptr, *bnBias = nullptr, *bnResidual = nullptr;
  int bnRelu = 0;
  int* bnQuery = nullptr;
};

// y = a (x - s) + k of a channel, and what follows it, with the roundings of mcn_bnorm_forward_fused (bnorm.hip):
// subtract, multiply-add, add, maximum
struct BnCoef { float a, k, s, unused; };
__device__ __forceinline__ BnCoef bn_coefficients(const float* moments, const float* mult, const float* bias, int channels, int co) {
  const double mean = (double)moments[co], coef = (double)mult[co] / (double)moments[co + channels];
  BnCoef c;
  c.s = (float)mean;
  c.a = (float)coef;
  c.k = (float)((double)bias[co] - coef * (mean - (double)c.s));
  c.unused = 0.f;
  return c;
}
__device__ __forceinline__ BnCoef bn_coefficients(const PixP& p, int co) {
  return bn_coefficients(p.bnMoments, p.bnMult, p.bnBias, p.Cout, co);
}
__device__ __forceinline__ float bn_apply(const BnCoef& c, float x, bool residual, float r, bool relu) {
  float v = fmaf(c.a, x - c.s, c.k);
  if (residual) v = v + r;
  return relu ? (v > 0.f ? v : 0.f) : v;
}

// the pixel's element offset inside its channel plane of the produced tensor
__device__ __forceinline__ int out_pixel_offset(const PixP& p, int q) {
  if (p.dense) return q;
  int ow, oh;
  p.byOH.divmod(q, &ow, &oh);
  return p.outOff + oh * p.outSH + ow * p.outSW;
}

// ------------------------------------------------------------------------------------------------
// Epilogue shared by the pixel-major MFMA kernels
// ------------------------------------------------------------------------------------------------
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef int bufrsrc __attribute__((ext_vector_type(4)));

constexpr unsigned kOutside = 0x80000000u;  // buffer offset no tensor handled here reaches (they are < 2 GiB)

// Raw buffer descriptor over `bytes` bytes at `base` (uniform): accesses at offsets >= bytes are dropped (stores)
// or return 0 (loads).
__device__ __forceinline__ bufrsrc make_bufrsrc(const void* base, unsigned bytes) {
  const unsigned long long a = (unsigned long long)base;
  bufrsrc r;
  r.x = (int)(unsigned)(a & 0xffffffffull);
  r.y = (int)(unsigned)((a >> 32) & 0xffffull);
  r.z = (int)bytes;
  r.w = 0x00020000;
  return r;
}

// A store the compiler's memory-wait bookkeeping does not see.  With ordinary stores in flight beside loads it
// can no longer tell which of them the hardware counter is counting and waits for everything at every use of a
// loaded value.  The hardware counter still counts these stores; that only makes the compiler's waits for older
// loads (which return in order among themselves) longer, never shorter.  Store data is read when the
// instruction issues, so the registers can be reused right after.
__device__ __forceinline__ void buffer_store_untracked(float v, unsigned voffset, bufrsrc rsrc, int soffset) {
  asm volatile("buffer_store_dword %0, %1, %2, %3 offen" ::"v"(v), "v"(voffset), "s"(rsrc), "s"(soffset) : "memory");
}

// Writes one wavefront's 32 channels x 32 pixels accumulator block of v_mfma_f32_32x32x2_f32 (register r of lane
// l holds channel 8(r/4) + 4(l/32) + r%4 of pixel l%32):  out = alpha*acc (+ beta*out) (+ bias).
//   rsrc     descriptor of the whole output tensor
//   voffset  byte offset of this lane's pixel in channel 4(l/32) of the block's image (kOutside: lane writes nothing)
//   sblock   byte offset of the block's first channel plane (uniform)
//   plane    bytes per channel plane (uniform)
//   biasBlk  bias of the block's first channel, or null (uniform)
// Straight-line: 16 stores at "lane offset + scalar offset", no per-store address arithmetic in vector registers,
// no per-store branches.
template <bool BETA, bool BIAS>
__device__ __forceinline__ void store_block_as(floatx16 acc, bufrsrc rsrc, unsigned voffset, int sblock, int plane,
                                               float alpha, float beta, const float* biasBlk, int kh) {
  float old[16], bv[16];
  if (BETA) {
    const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(((unsigned long long)(unsigned)rsrc.x) | ((unsigned long long)(unsigned)rsrc.y << 32)), 0, rsrc.z, rsrc.w);
#pragma unroll
    for (int r = 0; r < 16; ++r)
      old[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rr, (int)voffset, sblock + (8 * (r / 4) + r % 4) * plane, 0));
  }
  if (BIAS) {
#pragma unroll
    for (int r = 0; r < 16; ++r) bv[r] = biasBlk[8 * (r / 4) + 4 * kh + r % 4];
  }
  if (!BETA && !BIAS && alpha == 1.f) {
    // the plain product: the accumulators as they are (1 * x = x: sixteen multiplies less per block, which short
    // reductions -- 32 MFMAs per block with 64 input channels -- notice)
#pragma unroll
    for (int r = 0; r < 16; ++r) buffer_store_untracked(acc[r], voffset, rsrc, sblock + (8 * (r / 4) + r % 4) * plane);
    return;
  }
  // (alpha made opaque here: left visible, the compiler forms the sixteen products before it tests alpha == 1 and the
  // plain product above pays for them as well)
  asm volatile("" : "+s"(alpha));
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    float v = alpha * acc[r];
    if (BETA) v = fmaf(beta, old[r], v);
    if (BIAS) v += bv[r];
    buffer_store_untracked(v, voffset, rsrc, sblock + (8 * (r / 4) + r % 4) * plane);
  }
}

__device__ __forceinline__ void store_block(floatx16 acc, bufrsrc rsrc, unsigned voffset, int sblock, int plane,
                                            float alpha, float beta, const float* biasBlk, int kh) {
  if (beta != 0.f) {
    if (biasBlk) store_block_as<true, true>(acc, rsrc, voffset, sblock, plane, alpha, beta, biasBlk, kh);
    else store_block_as<true, false>(acc, rsrc, voffset, sblock, plane, alpha, beta, biasBlk, kh);
  } else if (biasBlk) {
    store_block_as<false, true>(acc, rsrc, voffset, sblock, plane, alpha, beta, biasBlk, kh);
  } else {
    store_block_as<false, false>(acc, rsrc, voffset, sblock, plane, alpha, beta, biasBlk, kh);
  }
}

// out = acc + (bit ? addend : addend*0): the block of store_block with a second term from a tensor of the same layout,
// gated by one bit per element (see PixP::addend).  arsrc / brsrc: descriptors of the addend and of the bit words;
// voffset and sblock as in store_block (plane bytes a multiple of 128, so a lane's bit position is the same for all 16
// channels and the word offset splits into a lane part and a scalar part).
__device__ __forceinline__ void store_block_masked_add(floatx16 acc, bufrsrc rsrc, bufrsrc arsrc, bufrsrc brsrc, unsigned voffset,
                                                       int sblock, int plane) {
  const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(((unsigned long long)(unsigned)arsrc.x) | ((unsigned long long)(unsigned)arsrc.y << 32)), 0, arsrc.z, arsrc.w);
  const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(((unsigned long long)(unsigned)brsrc.x) | ((unsigned long long)(unsigned)brsrc.y << 32)), 0, brsrc.z, brsrc.w);
  const unsigned vword = voffset == kOutside ? kOutside : (voffset >> 7) << 2;  // byte offset of the lane's word at scalar offset 0
  const unsigned bit = (voffset >> 2) & 31u;
  float add[16];
  unsigned wd[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int so = sblock + (8 * (r / 4) + r % 4) * plane;
    add[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ar, (int)voffset, so, 0));
    wd[r] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(br, (int)vword, so >> 5, 0);
  }
  // acc + addend * (0 or 1): the product is exact (the addend itself, or the zero, or the NaN, that addend * 0 is), so one
  // fused multiply-add gives the bits of "bit ? addend : addend * 0" added to acc -- three vector instructions per
  // element (bit field, conversion, multiply-add) instead of six
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float gate = (float)__builtin_amdgcn_ubfe(wd[r], bit, 1u);
    buffer_store_untracked(__builtin_fmaf(add[r], gate, acc[r]), voffset, rsrc, sblock + (8 * (r / 4) + r % 4) * plane);
  }
}

// Weights-stationary variant (conv_ws.hip) for filter banks that fit in LDS: wt is the packed bank in the
// 16-channel-chunk order of conv_pack_weights.  Sets *handled when it took the work.
int conv_ws_launch(hipStream_t s, const char* who, float* out, const float* in, const float* wt, const float* bias,
                   const PixP& p, int* handled);
// partial sums per channel it would write when asked to sum its output (PixP::stats); 0: it would not take `p` that way
int conv_ws_stat_groups(const PixP& p);

// Streamed-bank variant (conv_sb.hip) for banks too large for LDS, same packed order.  conv_sb_splits: the reduction
// splits it would use for a product of these extents (0: it does not take them; depends on nothing else, so that the
// workspace can be sized ahead); conv_sb_plan: the same, with the layout conditions checked.  conv_sb_launch: `p` laid
// out as for the tiled kernel (with splits > 1: the partial tensors' dense layout, alpha = 1, beta = 0, no bias).
// conv_sb_tail_bytes: scratch memory an unsplit launch of these extents wants for the tiles of its last, partly
// filled round (0: none); conv_sb_launch takes it as tailWs (nullptr: every tile by one workgroup).
int conv_sb_splits(int Cout, long long M, int R);
size_t conv_sb_tail_bytes(int Cout, long long M, int R);
bool conv_sb_plan(const PixP& p, int* splits);
int conv_sb_launch(hipStream_t s, float* out, const float* in, const float* wt, const float* bias, PixP p, int splits,
                   float* tailWs);

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

constexpr int kFragBytes = 1024;        // one part of 16 rows x 32 channels
constexpr int kBlockBytes = 3 * kFragBytes;

constexpr int kPackSplit = 4;  // PackJob::tapMajor of a bank for those products

// Operands of the split products are multiplied by this first: a float's last bit lies at 2^-149 or above and bf16's at
// 2^-133, scaled every float's three parts are normal bf16 numbers, down to the subnormal ones.  What the scale lifts over
// bf16's largest ends in an accumulator that is not finite, like infinities.
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;  // of an operand; of a product

// Two (scaled) floats as three packed pairs of bf16, x = h + m + l (conv_split.hip)
__device__ __forceinline__ unsigned round_pair(float x, float y) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2){x, y}, bf16x2));
}
__device__ __forceinline__ void split_pair(float x, float y, unsigned* h, unsigned* m, unsigned* l) {
  *h = round_pair(x, y);
  const float rx = x - __builtin_bit_cast(float, *h << 16), ry = y - __builtin_bit_cast(float, *h & 0xffff0000u);
  *m = round_pair(rx, ry);
  *l = round_pair(rx - __builtin_bit_cast(float, *m << 16), ry - __builtin_bit_cast(float, *m & 0xffff0000u));
}

// The splitting of eight floats in kSplitStages stages of one or two instructions, for interleaving with matrix instructions.
// Two pairs go side by side: no stage reads what the one before it wrote, which would cost a wait (the empty asm that keeps
// a stage where it is looks to the compiler like an instruction whose result is late: a quarter of the loop were s_nop).
constexpr int kSplitStages = 32;
struct SplitStages {
  float r[4];
  // taken(j): the floats of pair j are in `r`, those in `v` may be overwritten
  template <typename Vec, typename Taken>
  __device__ __forceinline__ void stage(int k, const Vec& v, uintx4& h, uintx4& m, uintx4& l, Taken taken) {
    const int s = k % 16;
    if (s < 4 || s == 8 || s == 9 || s >= 14) {  // a pair at a time
      const int j = k / 16 * 2 + s % 2;
      float &x = r[s % 2 * 2], &y = r[s % 2 * 2 + 1];
      if (s < 2) {
        x = v[2 * j] * kSplitScale;
        y = v[2 * j + 1] * kSplitScale;
        asm volatile("" : "+v"(x), "+v"(y));
        taken(j);
        return;
      }
      unsigned pair = round_pair(x, y);
      asm volatile("" : "+v"(pair));
      (s < 4 ? h : s < 10 ? m : l)[j] = pair;
    } else {  // a float at a time
      const int i = (s - (s < 8 ? 4 : 10)), j = k / 16 * 2 + i / 2;
      const unsigned pair = (s < 8 ? h : m)[j];
      r[i] -= __builtin_bit_cast(float, i % 2 ? pair & 0xffff0000u : pair << 16);
      asm volatile("" : "+v"(r[i]));
    }
  }
};

// A stored weight from the parts conv_pack_split_block makes of it: exact
__device__ __forceinline__ float split_weight(unsigned h, unsigned m, unsigned l) {
  if ((h & 0x7f80u) == 0x7f80u) return __builtin_bit_cast(float, m << 16 | l);
  auto value = [](unsigned u) { return __builtin_bit_cast(float, u << 16); };
  return ((value(h) + value(m)) + value(l)) * (1.f / kSplitScale);
}

// One fragment lane of the bank: eight rows (channels 8 kh ... of a chunk) of one tap, one output channel, split in three.
// A block of 256 threads packs a chunk of 16 channels of a block of 32 output channels: all taps, so that the 32 (forward)
// or 16 (backward) runs of the stored filters that it reads are shared in L1, or four taps (see conv_split_pack_job).
__device__ inline void conv_pack_split_block(const PackJob& j, unsigned block) {
  const int T = j.taps.nI * j.taps.nJ, blocksC = j.coutPad / 32;
  const int chunks = (j.Cin + 15) / 16;
  const int slices = (int)(j.blocks / (unsigned)(chunks * blocksC)), slice = (int)(block / (unsigned)(chunks * blocksC));
  block -= (unsigned)(slice * chunks * blocksC);
  const int chunk = (int)(block / blocksC), cb = (int)(block - (unsigned)chunk * blocksC);
  const int gBegin = chunk * T, gEnd = chunk == chunks - 1 ? j.rPad / 16 : gBegin + T;  // (the last chunk: with the padding)
  const size_t Tf = (size_t)j.taps.FH * j.taps.FW;
  for (int i = slice * 256 + threadIdx.x; i < (gEnd - gBegin) * 64; i += slices * 256) {
    const int t = i >> 6, lane = i & 63, kh = lane >> 5;
    const int co = cb * 32 + (lane & 31);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
    if (t < T && co < j.Cout) {
      const int b = t / j.taps.nI, a = t - b * j.taps.nI;
      const float* src = j.f + (size_t)(j.taps.i0 + a * j.taps.iStep) + (size_t)j.taps.FH * (j.taps.j0 + b * j.taps.jStep) +
                         (j.backward ? Tf * co : Tf * j.Cin * co);
      const size_t step = j.backward ? Tf * j.Cout : Tf;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int ci = chunk * 16 + 8 * kh + e;
        if (ci < j.Cin) v[e] = src[step * ci];
      }
    }
    uintx4 part[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      unsigned q[3] = {0, 0, 0};
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const float x = v[2 * e + half];
        unsigned h, m, l;
        split_pair(x * kSplitScale, 0.f, &h, &m, &l);
        if ((h & 0x7f80u) == 0x7f80u) {
          // not finite, or not below bf16's infinity when scaled: an infinity, and the number itself in the other two parts
          // (whatever it is multiplied by, the accumulator is not finite, and the repeat on the fp32 instruction takes it from there: split_weight)
          const unsigned u = __builtin_bit_cast(unsigned, x);
          h = 0x7f80u;
          m = u >> 16;
          l = u & 0xffffu;
        }
        q[0] |= (h & 0xffffu) << (16 * half);
        q[1] |= (m & 0xffffu) << (16 * half);
        q[2] |= (l & 0xffffu) << (16 * half);
      }
      part[0][e] = q[0];
      part[1][e] = q[1];
      part[2][e] = q[2];
    }
    uintx4* dst = (uintx4*)((char*)j.wt + ((size_t)(gBegin + t) * blocksC + cb) * kBlockBytes) + lane;
    dst[0] = part[0];
    dst[kFragBytes / 16] = part[1];
    dst[2 * kFragBytes / 16] = part[2];
  }
}

// The products on the bf16 matrix instruction with operands split in three (conv_split.hip).  conv_split_takes: whether it
// covers a product of these extents; conv_split_bank_bytes: its bank as conv_pack_split lays it out; conv_split_workspace_
// bytes: that bank and the partial results behind it.  conv_split_stat_groups / conv_split_adds: the partial sums per
// channel it writes (PixP::stats), whether it adds a masked second term (PixP::addend), whether it normalises its output
// (PixP::bnMoments).  conv_split_launch: with a split
// reduction the partial results are left in `scratch` and *reduce gets their number and distance (else 1): the caller
// adds them up.
bool conv_split_takes(const PixP& p);
void conv_split_pack_job(PackJob* j, void* bank, const float* f, const TapSet& taps, int Cin, int Cout, int backward);
int conv_split_pack(hipStream_t s, const char* who, const PackJob& j);
size_t conv_split_bank_bytes(int Cin, int T, int Cout);
size_t conv_split_workspace_bytes(int Cin, int T, int Cout, long long M);
int conv_split_stat_groups(const PixP& p);
bool conv_split_adds(const PixP& p);
bool conv_split_normalises(const PixP& p);
int conv_split_launch(hipStream_t s, const char* who, float* out, const float* in, const void* bank, const float* bias, PixP p,
                      void* scratch, size_t scratchBytes, PixP* reduce);
int conv_split_bank_blocks(int Cout);  // 32-channel blocks of a bank
// The same product over few pixels (conv_short.hip): channels per workgroup in units of 16 and wavefronts that share the
// reduction, or none.  Takes every form that conv_split_launch takes; sums per channel come in conv_short_stat_groups(M) parts.
struct ShortPlan { int wa, waves; };
ShortPlan conv_short_plan(const PixP& p);
double conv_split_modelled_us(int Cin, int T, int Cout, long long M);  // of conv_split.hip's launches, the sum of partial results included
int conv_short_stat_groups(long long M);
int conv_short_launch(hipStream_t s, const char* who, const ShortPlan& plan, float* out, const float* in, const void* bank,
                      const float* bias, const PixP& p);
// Products of filters with taps over pixels staged in LDS (conv_staged.hip), in tiles of 32 WA channels; conv_split_launch calls it.
// ends: tiles behind the `blocks` whole ones that go in tiles of 32 channels, in the same launch.
bool conv_staged_takes(const PixP& p, int WA, long long blocks);
int conv_staged_launch(hipStream_t s, const char* who, int WA, int epi, unsigned blocks, int ends, int chunksPerSplit, int tileBase, int tailTiles,
                       float* out, const float* in, const void* bank, const float* bias, const PixP& p);
int conv_split_launch_multi(hipStream_t s, const char* who, float* out, const float* in, const PixP* products,
                            const void* const* banks, int n);

// The filter gradient on the same instruction (conv_wsplit.hip), of one filter group `p`; the elements of x and dzdy are the
// whole layer's.  The partial banks (conv_wsplit_splits of them, after one another at `out`) are indexed c + C t + FV k.
bool conv_wsplit_takes(const ConvP& p, long long xLayerElements, long long yLayerElements);
int conv_wsplit_splits(const ConvP& p);
int conv_wsplit_launch(hipStream_t s, const ConvP& p, int xImg, int dyImg, float* out, const float* x, const float* dy);

// The filter gradient in double precision (f64_wgrad.hip), of one filter group (FC channels, Kg filters of layer `p`; the
// tensors begin at the group's first channel).  Partial banks as for conv_wsplit_launch.
bool conv64_wgrad_takes(const ConvP& p, long long xLayerElements, long long yLayerElements);
int conv64_wgrad_splits(const ConvP& p);
int conv64_wgrad_launch(hipStream_t s, const ConvP& p, double* out, const double* x, const double* dy);

// Forward and unit-stride backward-data in double precision (f64_pix.hip), likewise; `bank`: device memory for the packed bank.
bool conv64_pix_takes(const ConvP& p, bool backward);
size_t conv64_pix_bank_bytes(const ConvP& p, bool backward);
int conv64_pix_launch(hipStream_t s, const char* who, const ConvP& p, bool backward, double* out, const double* in, const double* f,
                      const double* bias, double alpha, double beta, double* bank);

// Fully connected layers (as 1x1 filters on 1x1 images, one group) of one to four images, forward (conv_dot.hip): the filters are
// read where they lie
bool conv_dot_takes(const PixP& p);
int conv_dot_launch(hipStream_t s, const char* who, const PixP& p, float* y, const float* x, const float* f, const float* bias);

// Products with at most four output channels (conv_few.hip): wt is the packed bank (tapMajor: its row order, see
// conv_pack_weights).  Sets *handled when it took the work.
int conv_few_launch(hipStream_t s, const char* who, float* out, const float* in, const float* wt, const float* bias,
                    const PixP& p, bool tapMajor, int* handled);

}  // namespace mcn
