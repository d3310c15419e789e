// Which large products take 256 x 256 tiles, and in how many slices of k. Plain arithmetic on
// sizes, so that a host program can ask which kernel a product runs on.
#pragma once

#include <algorithm>
#include <cstdint>

namespace tnh {
namespace gs {

// prec: 0 FP64, 1 FP32, 2 split-BF16x3; cu: compute units
// The number of k slices of a large product whose tiles leave part of the last round of
// workgroups idle (1: no split). The estimate is in rounds of the mode's usual tile at the rate
// the kernel reaches when the chip is full, plus the slices' traffic; a split has to win 5%.
// It depends on the shape and mode only, not on the tuned tile, so that tiles still never
// change a result. Measured, whole matvecs, unsplit / split, us: FP64 701 x 593, D = 5 645 / 585,
// 1100 x 1200, D = 3 1806 / 1638; FP32 1100 x 1000 1125 / 1040; split-BF16x3 1536 1460 / 1325;
// where rounds come out even a split only costs (FP32 2048, 8 rounds: 5883 / 6541 in two).
inline int ksplit_wanted(int64_t cu, int prec, int64_t M, int64_t N, int64_t K, double *seconds = nullptr) {
  const double rate[3] = {53e12, 122e12, 290e12}, mem = 8e12;  // flop/s of the full chip, bytes/s (mostly cache)
  const int side = prec == 0 ? 64 : 128, per_cu = prec == 0 ? 3 : 2;
  const int64_t tiles = ((M + side - 1) / side) * ((N + side - 1) / side), slots = per_cu * cu;
  const double round = double(slots) * 2 * side * side * double(K) / rate[prec];
  auto cost = [&](int s) {
    const double t = double((tiles * s + slots - 1) / slots) / s * round;
    return s == 1 ? t : t + 2.0 * s * double(M) * N * (prec == 0 ? 8 : 4) / mem + 4e-6;
  };
  int best = 1;
  double tb = 0.95 * cost(1);
  for (int s = 2; s <= 4 && K / s >= 512 && K >= 2048; ++s)
    if (cost(s) < tb) {
      best = s;
      tb = cost(s);
    }
  if (seconds) *seconds = best == 1 ? cost(1) : tb;
  return best;
}

// Whether an FP32 or split-BF16x3 product of at least 256 k takes the 256 x 256 tiles of gemm_wide.hip /
// gemm_wide_bf16.hip (one workgroup per CU), and then in how many k slices (0: it does not):
// when whole rounds of these tiles at the kernel's full rate, and the slices' traffic, cost 4%
// less than the other tiles are expected to. Those cost the rounds of ksplit_wanted, but reach
// 105 (270) TF whatever the rounds (the tuner then finds a smaller tile). Measured, other tiles /
// these, us, FP32: 8192 x 2048 x 6144 1698 / 1452; 9000 x 6800 x 1800 2036 / 1732; 7680 x 5600 x
// 1536 1180 / 1103; 6000 x 4400 x 1200 656 / 616; in five slices 7200 x 1700 x 8500 2084 / 1824,
// 5120 x 1280 x 5120 716 / 608. Beyond the line: 5120 x 5120 x 1280 630 / 645; 8000 x 6400 x 1600
// 1487 / 1555; 6144 x 4000 x 2048 in two slices 854 / 936; at K 64 124 / 132 (K 256: 94 / 87).
// Split-BF16x3, operand splits included: 4096 x 4096 x 1024 153 / 107, 6000 x 4400 x 1200 305 /
// 220, 8192 x 2048 x 6144 827 / 653, 4096 x 4096 x 256 56 / 49.
inline int wide_slices(int64_t cu, int prec, int64_t M, int64_t N, int64_t K, bool may_split) {
  if (prec == 0 || K < 256) return 0;
  const double rate = prec == 1 ? 140e12 : 380e12, other_rate = prec == 1 ? 105e12 : 270e12;
  const double mem = 2.5e12, flops = 2.0 * M * N * double(K);
  const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
  double others = 0;
  ksplit_wanted(cu, prec, M, N, K, &others);
  double tb = 0.96 * std::min(others, flops / other_rate);
  int best = 0;
  for (int s = 1; s <= (may_split ? 6 : 1) && (s == 1 || K / s >= 512); ++s) {
    double t = double((tiles * s + cu - 1) / cu * cu) / s * 2 * 65536 * double(K) / rate;
    if (s > 1) t += 2.0 * s * double(M) * N * 4 / mem + 4e-6;
    if (t < tb) {
      best = s;
      tb = 0.95 * t;  // another slice has to win 5%
    }
  }
  return best;
}

// k of a slice: whole k-steps and vectors. The last slice is shorter; none is empty, since a
// slice has at least 512 k and there are at most six.
inline int slice_width(int K, int slices) { return ((K + slices - 1) / slices + 63) / 64 * 64; }

}  // namespace gs
}  // namespace tnh
