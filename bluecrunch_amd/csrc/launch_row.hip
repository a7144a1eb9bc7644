// Innermost pass kernels of transforms that stand alone, every length class.
#include "launch_impl.h"

namespace bcg {

// Blocks per workgroup: whole waves (L / 8 threads each), as mid_blocks.
constexpr int row_blocks(int L) {
  return L % 3 == 0 ? (L < 1536 ? 1536 / L : 1) : (L < 512 ? 512 / L : 1);
}

// grid = number of contiguous blocks of L points.
template <int L>
int launch_row(bool inverse, int grid, hipStream_t s, const PassArgs &a) {
  constexpr int T = Row<L, 8>::T, BPW = row_blocks(L);
  if (BPW > 1 && grid % BPW == 0) {
    if (inverse)
      BCG_LAUNCH2((k_row<L, true, BPW>), grid / BPW, 1, T * BPW, s, a);
    else
      BCG_LAUNCH2((k_row<L, false, BPW>), grid / BPW, 1, T * BPW, s, a);
  } else {
    if (inverse)
      BCG_LAUNCH2((k_row<L, true>), grid, 1, T, s, a);
    else
      BCG_LAUNCH2((k_row<L, false>), grid, 1, T, s, a);
  }
  return 0;
}

row_fn pick_row(int L) {
  switch (L) {
    case 64: return &launch_row<64>;
    case 128: return &launch_row<128>;
    case 256: return &launch_row<256>;
    case 512: return &launch_row<512>;
    case 1024: return &launch_row<1024>;
    case 2048: return &launch_row<2048>;
    case 4096: return &launch_row<4096>;
    case 8192: return &launch_row<8192>;
    case 96: return &launch_row<96>;
    case 192: return &launch_row<192>;
    case 384: return &launch_row<384>;
    case 768: return &launch_row<768>;
    case 1536: return &launch_row<1536>;
    case 3072: return &launch_row<3072>;
    case 6144: return &launch_row<6144>;
  }
  return nullptr;
}

// Loads this unit's code object now; the runtime otherwise loads it at the
// first launch of one of its kernels, inside a caller's first transform.
int preload_row() {
  hipFuncAttributes fa;
  return hipFuncGetAttributes(&fa, reinterpret_cast<const void *>(&(k_row<1024, false>))) == hipSuccess ? 0 : -1;
}

}  // namespace bcg
