// What the kernels with operands split in three over tiles of 128 pixels share (conv_split.hip, conv_staged.hip): the
// geometry, and what is done with a finished block of 32 channels x 32 pixels (lane = pixel, register = channel).
#pragma once

#include "conv_common.hpp"

namespace mcn {

struct SplitP {
  int tilesC;         // channel tiles of 32 WA
  int blocksC;        // 32-channel blocks of the bank
  int chunks;         // chunks of 16 reduction channels
  int groups;         // chunks x taps
  int slabs;          // the bank's groups (padded to whole slabs) / GPS
  int slabsPerSplit;
  unsigned inBytes, bankBytes;
  int tileBase, tailTiles;  // kTail: the launch covers tiles [tileBase, tileBase + tailTiles)
};

constexpr unsigned kFar = 0xC0000000u;  // like kOutside; any offset inside a tensor becomes one like it by OR
// EPI: what the epilogue does with a finished block
enum { kStore = 0, kStats = 1, kMaskedAdd = 2, kTail = 3, kNormalise = 4 };

constexpr int kTurnPitch = 36;  // floats between the channels of a block turned in LDS (16-byte reads of 8 lanes: all 32 banks)


// The LDS of a workgroup that sums its output per channel: a block turned by each wavefront, and the partial sums
constexpr size_t stats_lds_bytes(int CT) { return 4 * 32 * kTurnPitch * sizeof(float) + 8 * CT * 2 * sizeof(double); }

// In what follows `acc` holds NB blocks of 32 channels, from channel c0 on, of this lane's pixel m.

// ... into the partial result of a tile of CT channels, block cOff of it first; px: the pixel inside the tile
template <int NB>
__device__ __forceinline__ void split_store_tail(floatx16 (&acc)[NB], float* out, int CT, int cOff, int px, int kh) {
  const bufrsrc orsrc = make_bufrsrc(out, (unsigned)(CT * 128 * 4));
  const unsigned vo = (unsigned)(px + 4 * kh * 128) * 4u;
#pragma unroll
  for (int a = 0; a < NB; ++a) store_block(acc[a], orsrc, vo, (cOff + a * 32) * 512, 512, 1.f, 0.f, nullptr, kh);
}

// ... normalised (PixP::bnMoments); coefs: of channel c0 first
template <int NB>
__device__ __forceinline__ void split_store_normalised(floatx16 (&acc)[NB], float* out, const PixP& p, const BnCoef* coefs, int c0, int m,
                                                       bool mvalid, int kh) {
  const bufrsrc orsrc = make_bufrsrc(out, p.outBytes);
  const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.bnResidual ? p.bnResidual : out), 0, (int)p.outBytes, 0x00020000);
  const int plane = p.outPlane * 4;
  int n, q;
  p.byQ.divmod(mvalid ? m : 0, &n, &q);
  const unsigned vo = mvalid ? (unsigned)(n * p.outImg + q + 4 * kh * p.outPlane) * 4u : kOutside;
  const bool residual = p.bnResidual != nullptr, relu = p.bnRelu != 0;
  // (the second term of all blocks first: loads and stores in turn would leave a wavefront waiting for memory once per block.
  // Blocks past the last channel read nothing.)
  float add[NB][16];
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) add[a][r] = 0.f;
  __builtin_amdgcn_sched_barrier(0);
  if (residual) {
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int c = c0 + a * 32;
        add[a][r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rr, c < p.Cout ? (int)vo : (int)kOutside, (min(c, p.Cout - 32) + 8 * (r / 4) + r % 4) * plane, 0));
      }
  }
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    const int c = c0 + a * 32;
    if (c >= p.Cout) continue;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int k = 8 * (r / 4) + r % 4;
      buffer_store_untracked(bn_apply(coefs[a * 32 + k + 4 * kh], acc[a][r], residual, add[a][r], relu), vo, orsrc, (c + k) * plane);
    }
  }
}

// ... alpha * acc (+ beta * out) (+ bias), or with a masked second term (kMaskedAdd)
template <int NB, int EPI>
__device__ __forceinline__ void split_store(floatx16 (&acc)[NB], float* out, const float* bias, const PixP& p, int cFirst, int m, bool mvalid,
                                            int kh) {
  if (EPI == kStats || EPI == kMaskedAdd || p.outBytes != 0) {
    const bufrsrc orsrc = make_bufrsrc(out, p.outBytes);
    const int plane = p.outPlane * 4;
    int n, q;
    p.byQ.divmod(mvalid ? m : 0, &n, &q);
    const unsigned vo = mvalid ? (unsigned)(n * p.outImg + out_pixel_offset(p, q) + 4 * kh * p.outPlane) * 4u : kOutside;
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      const int c0 = cFirst + a * 32;
      if (c0 + 32 <= p.Cout) {
        if (EPI == kMaskedAdd)
          store_block_masked_add(acc[a], orsrc, make_bufrsrc(p.addend, p.outBytes), make_bufrsrc(p.addBits, p.outBytes >> 5), vo, c0 * plane, plane);
        else
          store_block(acc[a], orsrc, vo, c0 * plane, plane, p.alpha, p.beta, bias ? bias + c0 : nullptr, kh);
      } else if (EPI == kStore && c0 < p.Cout && mvalid) {
        float* o = out + (size_t)n * p.outImg + out_pixel_offset(p, q);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int co = c0 + 8 * (r / 4) + 4 * kh + (r % 4);
          if (co < p.Cout) {
            float v = p.alpha * acc[a][r];
            if (p.beta != 0.f) v = fmaf(p.beta, o[(size_t)co * p.outPlane], v);
            if (bias) v += bias[co];
            o[(size_t)co * p.outPlane] = v;
          }
        }
      }
    }
    return;
  }
  if (!mvalid) return;
  int n, q;
  p.byQ.divmod(m, &n, &q);
  float* o = out + (size_t)n * p.outImg + out_pixel_offset(p, q);
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int co = cFirst + a * 32 + 8 * (r / 4) + 4 * kh + (r % 4);
      if (co < p.Cout) {
        float v = p.alpha * acc[a][r];
        if (p.beta != 0.f) v = fmaf(p.beta, o[(size_t)co * p.outPlane], v);
        if (bias) v += bias[co];
        o[(size_t)co * p.outPlane] = v;
      }
    }
}

// Per-channel sums of what was stored (alpha = 1; lanes past the last pixel hold zeros), in double: what they miss must
// not show in the moments, whose last bit decides which side of zero a ReLU's argument next to zero falls on.  A
// wavefront turns each 32 x 32 block in LDS so that a lane holds 16 pixels of one channel (16 writes, 4 reads and 48
// vector instructions per lane; adding across the lanes takes 144 in fp32), the eight half-rows of the workgroup meet
// there in a fixed order, and the workgroup writes one partial per channel.  row: the block's 32 pixels of the tile's 128.
template <int NB>
__device__ __forceinline__ void split_sums(floatx16 (&acc)[NB], char* lds, int wave, int row, int CT, int cOff, int l32, int kh) {
  float* turn = (float*)lds + wave * (32 * kTurnPitch);
  double* sums = (double*)(lds + 4 * 32 * kTurnPitch * sizeof(float));  // [8][CT][2]
#pragma unroll
  for (int a = 0; a < NB; ++a) {
#pragma unroll
    for (int r = 0; r < 16; ++r) turn[(8 * (r / 4) + 4 * kh + r % 4) * kTurnPitch + l32] = acc[a][r];
    double t1 = 0.0, t2 = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const v4f v = *(const v4f*)&turn[l32 * kTurnPitch + 16 * kh + 4 * i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double d = (double)v[e];
        t1 += d;
        t2 = fma(d, d, t2);
      }
    }
    double* o = sums + ((row * 2 + kh) * CT + cOff + a * 32 + l32) * 2;
    o[0] = t1;
    o[1] = t2;
  }
}
// (behind a barrier) one partial per channel of pixel tile mt
__device__ __forceinline__ void split_sums_out(const char* lds, const PixP& p, int CT, int coW, int mt, int tid) {
  if (tid >= CT || coW + tid >= p.Cout) return;
  const double* sums = (const double*)(lds + 4 * 32 * kTurnPitch * sizeof(float));
  double t1 = 0.0, t2 = 0.0;
#pragma unroll
  for (int row = 0; row < 8; ++row) {
    t1 += sums[(row * CT + tid) * 2];
    t2 += sums[(row * CT + tid) * 2 + 1];
  }
  double* o = p.stats + ((size_t)(coW + tid) * p.statGroups + mt) * 2;
  o[0] = t1;
  o[1] = t2;
}

}  // namespace mcn
