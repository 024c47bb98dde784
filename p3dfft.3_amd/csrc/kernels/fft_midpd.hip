// Single-buffer mixed-radix kernels with a prime radix above 16, FP64.
#include "mid_kernels.h"

namespace p3e {

int launch_mid_prime_d(const PassArgs *a, size_t lds_bytes, int threads, unsigned int nblocks, hipStream_t st) {
  if (a->mid_prime <= 23) return launch_mid<double, 23, P3E_MID_MANY>(a, nullptr, nullptr, 0, lds_bytes, threads, nblocks, st);
  if (a->mid_prime == 29) return launch_mid<double, 29, P3E_MID_MANY>(a, nullptr, nullptr, 0, lds_bytes, threads, nblocks, st);
  return (int)hipErrorInvalidValue;
}

}  // namespace p3e
