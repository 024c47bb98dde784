// Single-buffer mixed-radix kernels without a prime radix above 16, FP32 with many values per thread.
#include "mid_kernels.h"

namespace p3e {

int launch_mid_many_s(const PassArgs *a, const PassArgs *tab, const uint32_t *start, int n, size_t lds_bytes,
                      int threads, unsigned int nblocks, hipStream_t st) {
  return launch_mid<float, 0, P3E_MID_MANY>(a, tab, start, n, lds_bytes, threads, nblocks, st);
}

}  // namespace p3e
