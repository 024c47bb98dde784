// Single-buffer mixed-radix kernels with a prime radix above 16, FP32: one
// kernel per range of primes, so that the registers of the larger butterflies
// are allocated only where needed.
#include "mid_kernels.h"

namespace p3e {

int launch_mid_prime_s(const PassArgs *a, size_t lds_bytes, int threads, unsigned int nblocks, hipStream_t st) {
  if (a->mid_prime <= 23) return launch_mid<float, 23, P3E_MID_MANY>(a, nullptr, nullptr, 0, lds_bytes, threads, nblocks, st);
  if (a->mid_prime <= 31) return launch_mid<float, 31, P3E_MID_MANY>(a, nullptr, nullptr, 0, lds_bytes, threads, nblocks, st);
  if (a->mid_prime <= 47) return launch_mid<float, 47, P3E_MID_MANY>(a, nullptr, nullptr, 0, lds_bytes, threads, nblocks, st);
  return (int)hipErrorInvalidValue;
}

}  // namespace p3e
