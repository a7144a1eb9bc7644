// Launcher templates shared by the launch_*.hip translation units.
#pragma once
#include "launch.h"

namespace bcg {

#define BCG_LAUNCH2(kern, gx, gy, block, stream, ...) \
  hipLaunchKernelGGL(kern, dim3(gx, gy), dim3(block), 0, stream, __VA_ARGS__)

// Blocks of L points one workgroup of a middle pass holds: enough to fill whole
// waves (L / 8 threads each: eight blocks of 64 points make one wave, two of 768
// three), a power of two because the block counts are.
constexpr int mid_blocks(int L) {
  const int wave = 64 * mid_points(L);
  return L % 3 == 0 ? (L < 1536 ? 1536 / L : 1) : (L < wave ? wave / L : 1);
}

// The packing and unpacking passes of single products take eight points per thread
// (k_fwd8, k_inv8) up to this many tiles of eight columns in a launch, two a CU: 12000
// by 12000 words 38.3 -> 35.1 us, 2^17 by 2^17 49.6 -> 48.8 us; twice as many make no
// difference. Strided passes between points of transforms are slower so (2^20 points
// through the transform calls 123 -> 125 us), and a batched product keeps its class's
// kernel however many share the launch.
constexpr int STRIP_TILES = 512;
template <int L, int C>
constexpr bool has_strip() {
  return C == 8 && (L == 64 || L == 128 || L == 256);
}

// Strided passes are powers of two (the 3 * 2^k factor sits in the innermost pass).
template <int L, int C>
int launch_fwd(bool pack, int grid, int gy, hipStream_t s, const PassArgs &a) {
  if constexpr (has_strip<L, C>()) {
    if (pack && !a.desc && grid * gy <= STRIP_TILES) {
      if (a.lower)
        BCG_LAUNCH2((k_fwd8<L, true>), grid, gy, L, s, a);
      else
        BCG_LAUNCH2((k_fwd8<L, false>), grid, gy, L, s, a);
      return 0;
    }
  }
  if (pack && a.lower)
    BCG_LAUNCH2((k_fwd<L, C, true, 0, true>), grid, gy, (Tile<L, C>::T), s, a);
  else if (pack)
    BCG_LAUNCH2((k_fwd<L, C, true>), grid, gy, (Tile<L, C>::T), s, a);
  else
    BCG_LAUNCH2((k_fwd<L, C, false>), grid, gy, (Tile<L, C>::T), s, a);
  return 0;
}

// Unpacking into group sums (a.ybuf) exists for 8- and 16-column tiles.
template <int L, int C>
int launch_inv(bool unpack, int grid, int gy, hipStream_t s, const PassArgs &a) {
  if constexpr (has_strip<L, C>()) {
    if (unpack && !a.desc && grid * gy <= STRIP_TILES) {
      if (a.ybuf)
        BCG_LAUNCH2((k_inv8<L, true>), grid, gy, L, s, a);
      else
        BCG_LAUNCH2((k_inv8<L, false>), grid, gy, L, s, a);
      return 0;
    }
  }
  if (unpack && a.ybuf) {
    if constexpr (C == 8 || C == 16)
      BCG_LAUNCH2((k_inv<L, C, 2>), grid, gy, (Tile<L, C>::T), s, a);
    else
      return -2;
  } else if (unpack) {
    BCG_LAUNCH2((k_inv<L, C, 1>), grid, gy, (Tile<L, C>::T), s, a);
  } else {
    BCG_LAUNCH2((k_inv<L, C, 0>), grid, gy, (Tile<L, C>::T), s, a);
  }
  return 0;
}

// Column counts with L * C <= 8192 elements per tile (32 columns only for the
// middle inverse pass of 256-point tiles, see inv_cols).
template <int L, template <int, int> class F>
struct ByC {
  static fwd_fn pick(int C) {
    switch (C) {
      case 1: return &F<L, 1>::run;
      case 2: return (L * 2 <= 8192) ? &F<L, (L * 2 <= 8192 ? 2 : 1)>::run : nullptr;
      case 4: return (L * 4 <= 8192) ? &F<L, (L * 4 <= 8192 ? 4 : 1)>::run : nullptr;
      case 8: return (L * 8 <= 8192) ? &F<L, (L * 8 <= 8192 ? 8 : 1)>::run : nullptr;
      case 16: return (L * 16 <= 8192) ? &F<L, (L * 16 <= 8192 ? 16 : 1)>::run : nullptr;
      case 32: return (L == 256) ? &F<L, (L == 256 ? 32 : 1)>::run : nullptr;
    }
    return nullptr;
  }
};

template <int L, int C>
struct FwdL {
  static int run(bool f, int gx, int gy, hipStream_t s, const PassArgs &a) { return launch_fwd<L, C>(f, gx, gy, s, a); }
};
template <int L, int C>
struct InvL {
  static int run(bool f, int gx, int gy, hipStream_t s, const PassArgs &a) { return launch_inv<L, C>(f, gx, gy, s, a); }
};

}  // namespace bcg
