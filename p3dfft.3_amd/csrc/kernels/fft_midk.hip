// Single-buffer mixed-radix kernels without a prime radix above 16, FP32 with
// few values per thread, and the launchers of that path.
#include "mid_kernels.h"

namespace p3e {

// fft_midw.hip, fft_midd.hip and fft_midwd.hip: FP32 with many values per
// thread, FP64 with few and many; fft_midp.hip and fft_midpd.hip: with a
// prime radix above 16, FP32 and FP64.
int launch_mid_many_s(const PassArgs *a, const PassArgs *tab, const uint32_t *start, int n, size_t lds_bytes,
                      int threads, unsigned int nblocks, hipStream_t st);
int launch_mid_few_d(const PassArgs *a, const PassArgs *tab, const uint32_t *start, int n, size_t lds_bytes,
                     int threads, unsigned int nblocks, hipStream_t st);
int launch_mid_many_d(const PassArgs *a, const PassArgs *tab, const uint32_t *start, int n, size_t lds_bytes,
                      int threads, unsigned int nblocks, hipStream_t st);
int launch_mid_prime_s(const PassArgs *a, size_t lds_bytes, int threads, unsigned int nblocks, hipStream_t st);
int launch_mid_prime_d(const PassArgs *a, size_t lds_bytes, int threads, unsigned int nblocks, hipStream_t st);

// A grouped launch of passes without a prime radix above 16, all of the
// class, route and values per thread of a; tab and start in device memory.
// (tab null: the pass a alone.)
int launch_mid_group(const PassArgs *a, const PassArgs *tab, const uint32_t *start, int n, int prec, size_t lds_bytes,
                     int threads, unsigned int nblocks, hipStream_t st) {
  if (a->mid_e == P3E_MID_FEW)
    return prec == 8 ? launch_mid_few_d(a, tab, start, n, lds_bytes, threads, nblocks, st)
                     : launch_mid<float, 0, P3E_MID_FEW>(a, tab, start, n, lds_bytes, threads, nblocks, st);
  return prec == 8 ? launch_mid_many_d(a, tab, start, n, lds_bytes, threads, nblocks, st)
                   : launch_mid_many_s(a, tab, start, n, lds_bytes, threads, nblocks, st);
}

int launch_mid_pass(const PassArgs *a, int prec, size_t lds_bytes, int threads, unsigned int nblocks,
                    hipStream_t st) {
  if (a->mid_prime > 16)
    return prec == 8 ? launch_mid_prime_d(a, lds_bytes, threads, nblocks, st)
                     : launch_mid_prime_s(a, lds_bytes, threads, nblocks, st);
  return launch_mid_group(a, nullptr, nullptr, 0, prec, lds_bytes, threads, nblocks, st);
}

}  // namespace p3e
