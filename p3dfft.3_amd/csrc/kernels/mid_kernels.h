// Single-buffer mixed-radix pass kernels (fft_mid.h): the kernel templates
// and launchers that the translation units fft_mid*.hip instantiate (split so
// that they compile in parallel).
#pragma once
#include <hip/hip_runtime.h>

#include "fft_core.h"
#include "fft_mid.h"
#include "pass_dev.h"

namespace p3e {

// The tile in LDS, then the twiddles.
template <typename T, int P, int E, int CLS, int IN, int OUT, bool BLUE>
__device__ __forceinline__ void mid_body(const PassArgs &p, uint32_t tile) {
  extern __shared__ unsigned char smem_raw[];
  cx<T> *buf = reinterpret_cast<cx<T> *>(smem_raw);
  const cx<T> *tw = reinterpret_cast<const cx<T> *>(p.tw);
  const int tid = threadIdx.x, nth = p.nthreads;
  cx<T> *ltw = buf + p.L * p.pit;
  for (int i = tid; i < p.ntw; i += blockDim.x) ltw[i] = tw[i];
  DevMidRun<T> run{tid, nth};
  DevEach each{tid};
  mid_tile_as<T, P, E, CLS, IN, OUT, BLUE>(p, tile, buf, nth, run, each, ltw);
}

template <typename T, int P, int E, int CLS, int IN, int OUT, bool BLUE>
__global__ void __launch_bounds__(P3E_MID_MAXTH) pass_kernel_mid(PassArgs p) {
  mid_body<T, P, E, CLS, IN, OUT, BLUE>(p, xcd_tile(blockIdx.x, gridDim.x));
}

// The same pass of many transforms in one launch (see pass_kernel_pow2_grp):
// passes of one class and route.
template <typename T, int P, int E, int CLS, int IN, int OUT, bool BLUE>
__global__ void __launch_bounds__(P3E_MID_MAXTH)
    pass_kernel_mid_grp(const PassArgs *__restrict__ tab, const uint32_t *__restrict__ start, int n) {
  const uint32_t i = group_item(start, n, blockIdx.x);
  mid_body<T, P, E, CLS, IN, OUT, BLUE>(tab[i], blockIdx.x - start[i]);
}

static inline int mid_lds_limit(const void *fn, size_t lds_bytes) {
  if (lds_bytes <= 65536) return 0;
  return (int)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
}

// The pass a, or the grouped launch (tab, start, n) of passes of a's class
// and route.
template <typename T, int P, int E>
static int launch_mid(const PassArgs *a, const PassArgs *tab, const uint32_t *start, int n, size_t lds_bytes,
                      int threads, unsigned int nblocks, hipStream_t st) {
  mid_dispatch<P>(*a, [&](auto c, auto in, auto out, auto blue) {
    if (tab) {
      if constexpr (P <= 16) {
        const auto fn = pass_kernel_mid_grp<T, P, E, c.v, in.v, out.v, blue.v>;
        (void)mid_lds_limit((const void *)fn, lds_bytes);
        hipLaunchKernelGGL(fn, dim3(nblocks), dim3(threads), lds_bytes, st, tab, start, n);
      }
    } else {
      const auto fn = pass_kernel_mid<T, P, E, c.v, in.v, out.v, blue.v>;
      (void)mid_lds_limit((const void *)fn, lds_bytes);
      hipLaunchKernelGGL(fn, dim3(nblocks), dim3(threads), lds_bytes, st, *a);
    }
  });
  return (int)hipGetLastError();
}

}  // namespace p3e
