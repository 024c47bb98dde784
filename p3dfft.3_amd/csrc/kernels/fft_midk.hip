// Single-buffer mixed-radix kernels without a prime radix above 16, FP32, and
// the launchers of that path.
#include "mid_kernels.h"

namespace p3e {

// fft_midd.hip: FP64 without a prime above 16; fft_midp.hip and
// fft_midpd.hip: with one, FP32 and FP64.
int launch_mid_base_d(const PassArgs *a, const PassArgs *tab, const uint32_t *start, int n, size_t lds_bytes,
                      int threads, unsigned int nblocks, hipStream_t st);
int launch_mid_prime_s(const PassArgs *a, size_t lds_bytes, int threads, unsigned int nblocks, hipStream_t st);
int launch_mid_prime_d(const PassArgs *a, size_t lds_bytes, int threads, unsigned int nblocks, hipStream_t st);

// A grouped launch of passes without a prime radix above 16, all of the
// class and route of a; tab and start in device memory.
int launch_mid_group(const PassArgs *a, const PassArgs *tab, const uint32_t *start, int n, int prec, size_t lds_bytes,
                     int threads, unsigned int nblocks, hipStream_t st) {
  return prec == 8 ? launch_mid_base_d(a, tab, start, n, lds_bytes, threads, nblocks, st)
                   : launch_mid<float, 0>(a, tab, start, n, lds_bytes, threads, nblocks, st);
}

int launch_mid_pass(const PassArgs *a, int prec, size_t lds_bytes, int threads, unsigned int nblocks,
                    hipStream_t st) {
  if (a->mid_prime > 16)
    return prec == 8 ? launch_mid_prime_d(a, lds_bytes, threads, nblocks, st)
                     : launch_mid_prime_s(a, lds_bytes, threads, nblocks, st);
  return prec == 8 ? launch_mid_base_d(a, nullptr, nullptr, 0, lds_bytes, threads, nblocks, st)
                   : launch_mid<float, 0>(a, nullptr, nullptr, 0, lds_bytes, threads, nblocks, st);
}

}  // namespace p3e
