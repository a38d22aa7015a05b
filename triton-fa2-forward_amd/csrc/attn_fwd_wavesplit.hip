// attn_fwd_wavesplit.hip - the wave-split kernel's instances (attn_fwd_wavesplit.hpp). The
// measurement library compiles it again with FA2_WAVE_SPLIT_VARIANT for its masking variant.
#include "attn_fwd_wavesplit.hpp"

#include "attn_fwd_launch.hpp"

#ifndef FA2_WAVE_SPLIT_VARIANT
#define FA2_WAVE_SPLIT_VARIANT 0
#endif

namespace fa2 {

namespace {

template <int DT, int D, bool CAUSAL>
int launch_shape(const Params& p, int row_waves, unsigned grid, hipStream_t s) {
  constexpr int V = FA2_WAVE_SPLIT_VARIANT;
  constexpr int BN1 = wave_split_block_n(D, 1, CAUSAL), BN2 = wave_split_block_n(D, 2, CAUSAL);
  if (row_waves == 1)
    hipLaunchKernelGGL((attn_wave_split_kernel<DT, D, 1, BN1, CAUSAL, V>), dim3(grid), dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((attn_wave_split_kernel<DT, D, 2, BN2, CAUSAL, V>), dim3(grid), dim3(256), 0, s, p);
  return (int)hipGetLastError();
}

template <int DT, int D>
int launch_d(const Params& p, int row_waves, bool causal, unsigned grid, hipStream_t s) {
  return causal ? launch_shape<DT, D, true>(p, row_waves, grid, s)
                : launch_shape<DT, D, false>(p, row_waves, grid, s);
}

}  // namespace

template <>
int launch_wave_split<FA2_WAVE_SPLIT_VARIANT>(int dtype, int head_dim, const Params& p,
                                              int row_waves, bool causal, unsigned grid,
                                              hipStream_t s) {
  switch (dtype * 4 + (head_dim == 16 ? 0 : head_dim == 32 ? 1 : head_dim == 64 ? 2 : 3)) {
    case 0: return launch_d<0, 16>(p, row_waves, causal, grid, s);
    case 1: return launch_d<0, 32>(p, row_waves, causal, grid, s);
    case 2: return launch_d<0, 64>(p, row_waves, causal, grid, s);
    case 3: return launch_d<0, 128>(p, row_waves, causal, grid, s);
    case 4: return launch_d<1, 16>(p, row_waves, causal, grid, s);
    case 5: return launch_d<1, 32>(p, row_waves, causal, grid, s);
    case 6: return launch_d<1, 64>(p, row_waves, causal, grid, s);
    default: return launch_d<1, 128>(p, row_waves, causal, grid, s);
  }
}

}  // namespace fa2
