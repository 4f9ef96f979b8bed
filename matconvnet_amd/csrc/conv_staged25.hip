// The products over staged pixels with 25 taps (conv_staged.hpp), compiled apart: 25 groups unrolled take as long as all others.
#include "conv_staged.hpp"

namespace mcn {

int conv_staged_launch_25(hipStream_t s, int WA, int epi, unsigned blocks, unsigned ends, float* out, const float* in, const void* bank,
                          const float* bias, const PixP& p, const StagedP& w, const StagedP& v) {
  return go_taps<25>(s, WA, epi, blocks, ends, out, in, bank, bias, p, w, v);
}

}  // namespace mcn
