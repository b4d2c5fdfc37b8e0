// Arithmetic of the FP32 precision modes (host code, no GPU types).
#pragma once
#include <stdint.h>

namespace ccqk {

// Products that precision modes 1 and 2 compute in FP64: one side of at most 64
// and either a summed range of at most 32, a side of less than 16 (both bound by
// memory in FP64 too) or at most 2^26 multiply-adds (2 us of the chip in FP64, about
// a launch's latency).  A rule of the shape alone, so that neither the planner's
// cost model nor a measured plan decides the arithmetic.  It takes in every
// product that the planner has given to the register-direct kernel, which
// computes in FP64 only.  Its price: FP32-storage sweeps of CCSD 61 orbitals 347 ->
// 362 us, CCSDT 31 1087 -> 1131 us.
constexpr bool fp64_in_mixed(int64_t M, int64_t N, int64_t K) {
  const int64_t side = M < N ? M : N;
  return side <= 64 && (K <= 32 || side < 16 || M * N <= ((int64_t)1 << 26) / K);
}

}  // namespace ccqk
