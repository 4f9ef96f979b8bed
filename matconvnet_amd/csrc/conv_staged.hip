// Which products go over staged pixels (conv_staged.hpp), and those with nine taps.
#include "conv_staged.hpp"

namespace mcn {
namespace {

// The pixels under a tile of 128 and its taps; false: not a product of this kind, or too many
bool staged_span(const PixP& p, int WA, StagedP* w) {
  if ((p.T != 9 && p.T != 25) || p.sy != 1 || p.sx != 1 || p.OH != p.IH || p.OW != p.IW || p.Cin % 16 != 0) return false;
  const int FW = p.T / p.FH;
  const long long lastH = p.dhBase + (long long)(p.FH - 1) * p.dhStep, lastW = p.dwBase + (long long)(FW - 1) * p.dwStep;
  const long long first = std::min<long long>(p.dhBase, lastH) + p.IH * std::min<long long>(p.dwBase, lastW);
  const long long span = 128 + std::max<long long>(p.dhBase, lastH) + p.IH * std::max<long long>(p.dwBase, lastW) - first;
  if (span >= 128 * most_units(p.T, WA)) return false;
  w->first = (int)first;
  w->span = (int)span;
  w->slots = (int)(span + 1 + 63) / 64 * 64;
  return true;
}

}  // namespace

// Products of one workgroup to a CU stay on conv_split.hip's kernel: alone on its SIMD a wavefront waits here for each barrier
// (one a group there too, but a fifth of the code): cold, after other launches, 3x3x256x256 over 14x14, 32 images (196
// workgroups) takes 52 us here and 49 there.  With two to a CU, that kernel -> this one: 3x3x64x64 over 56x56, 32 images, forward
// 49.5 -> 48.4, backward-data 48.8 -> 46.0, 3x3x256x256 over 56x56, 64 images 1037 -> 938, two groups of 5x5x48x128 over 27x27, 128
// images, forward and backward-data 690 -> 575 us.
// Nine taps read at most 255 pixels under a tile: three units to a wavefront, 257 to 383 pixels for 128, are split for too few
// products (8 images, that kernel -> this one: 3x3x64x128 over 112x112 88 -> 102 us, 3x3x128x128 162 -> 178, 80x80 83 -> 93).
// So do 25 taps under tiles of 64 channels, where these are one or two to a CU (5x5x64x64 over 48x48, 16 images 58.5 -> 62.3,
// 5x5x32x64 over 62x62, 12 images 36.2 -> 37.8; with three, 5x5x64x128 over 62x62, 104 -> 96, which the simpler rule leaves).
// 25 taps under tiles of 128 keep three units: 5x5x96x256 over 32x32, 32 images 179 -> 163, over 56x56 553 -> 503, 5x5x64x128 over
// 40x40 107 -> 100, 5x5x48x128 over 62x62, 24 images 135 -> 125.  One chunk has nothing to stage ahead of: 5x5x16x128 over 62x62,
// 16 images 40.5 -> 42.0.
bool conv_staged_takes(const PixP& p, int WA, long long blocks) {
  StagedP w;
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  const int forced = tunable("conv_staged", 0);
  if (p.T != 9 && (p.stats || p.addend || p.bnMoments)) return false;  // (those are compiled for nine taps)
  return (WA == 2 || WA == 4) && forced >= 0 && ((blocks > cus && p.Cin > 16) || forced > 0) && staged_span(p, WA, &w);
}

int conv_staged_launch(hipStream_t s, const char* who, int WA, int epi, unsigned blocks, int ends, int chunksPerSplit, int tileBase, int tailTiles,
                       float* out, const float* in, const void* bank, const float* bias, const PixP& p) {
  StagedP w;
  if (!staged_span(p, WA, &w)) return fail(MCN_ILLEGAL_ARGUMENT, "%s: not a product over staged pixels", who);
  w.blocksC = conv_split_bank_blocks(p.Cout);
  w.tilesC = (p.Cout + 32 * WA - 1) / (32 * WA);
  w.chunks = p.Cin / 16;
  w.chunksPerSplit = chunksPerSplit;
  w.inBytes = (unsigned)(((long long)(p.N - 1) * p.inImg + (long long)p.Cin * p.IH * p.IW) * 4);
  w.bankBytes = (unsigned)conv_split_bank_bytes(p.Cin, p.T, p.Cout);
  w.tileBase = tileBase;
  w.tailTiles = tailTiles;
  w.byIHW = FastDiv(p.IH * p.IW);
  StagedP v = w;
  v.tilesC = (p.Cout + 31) / 32;
  v.tileBase = (int)blocks * WA;
  const unsigned narrow = (unsigned)(ends * WA);
  const int rc = p.T == 9 ? go_taps<9>(s, WA, epi, blocks, narrow, out, in, bank, bias, p, w, v)
                          : conv_staged_launch_25(s, WA, epi, blocks, narrow, out, in, bank, bias, p, w, v);
  return rc ? rc : check_launch(who);
}

}  // namespace mcn
