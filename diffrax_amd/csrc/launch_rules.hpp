// launch_rules.hpp -- which build and launch shape a solve takes on the device at hand: the
// rules that count its compute units (256 on a whole MI355X, fewer on a partition of one).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace dfx {

constexpr int kSimdsPerCu = 4;
constexpr int64_t kLdsPerCu = 160 << 10, kLdsPerBlock = 64 << 10;

// Compute units of the current device.  Asked for at every launch (0.1 us): the current device
// may change between two.
inline int device_cus() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1)
    return 256;
  return n;
}

// Whether a small-system batch's waves get a SIMD each, and so the builds that allow one wave
// per SIMD: the dispatcher pairs waves on some SIMDs while others are empty
// (erk_small_kernel).  A larger batch would wait for its last waves in those builds.
inline bool waves_alone(int64_t batch, int cus) {
  return batch <= (int64_t)64 * kSimdsPerCu * cus;
}

// Whether the save times of the waves that a CU holds at once (by the batch; 8 by registers)
// fit in its LDS, wave_bytes each, in workgroups of `block` threads: with fewer resident
// 131,072 instances with 64 saves take 2.2 ms, in the build without them 1.9 ms.
inline bool save_times_fit(int64_t wave_bytes, int64_t batch, int block, int cus) {
  const int64_t per_cu = (batch + 64 * cus - 1) / (64 * cus);
  const int64_t waves = std::min<int64_t>(8, std::max<int64_t>(per_cu, block / 64));
  return wave_bytes * (block / 64) <= kLdsPerBlock && wave_bytes * waves <= kLdsPerCu;
}

// Waves per tile of a neural-ODE solve (MlpWaves): eight, two per SIMD, for the three-piece
// form (its registers at four waves leave one wave per SIMD) and for float32 batches of at most
// one tile per CU; larger float32 batches take four, of which two workgroups share a CU and
// fill each other's barriers (256 CUs: solves of 8,192, 10,007 and 16,384 trajectories 416,
// 776 and 785 us at eight, 427, 743 and 756 us at four).
inline int mlp_tile_waves(bool pieces, int64_t tiles, int cus) {
  return pieces || tiles <= cus ? 8 : 4;
}

}  // namespace dfx
