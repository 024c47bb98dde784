// Kernels of the compile-time-length path (fft_fast.h) and their
// single-length launchers, instantiated by fft_pow2.hip (powers of two) and
// fft_pow2x.hip (3 and 5 times a power of two).
#pragma once
#include <hip/hip_runtime.h>

#include "fft_core.h"
#include "fft_fast.h"
#include "pass_dev.h"

namespace p3e {

// Compile-time-length path: complex length M at compile time, one LDS buffer for
// the tile, followed in LDS by the twiddle table (ntw entries) and, for
// R2C/C2R, the split factors (M + 1 entries): the radix passes and the
// split/merge read them from LDS instead of issuing global loads (which
// would compete with the tile's stream for the memory pipeline).
template <typename T> struct FixedStage {
  static constexpr bool staged = true;
  TabStage<T> tw, wn;
  bool has_wn, wait;
  __device__ __forceinline__ void operator()(int tid) const {
    tw.store(tid);
    if (has_wn) wn.store(tid);
    if (wait) __syncthreads();
  }
};

template <typename T, int M>
__device__ __forceinline__ void pow2_body(const PassArgs &p, uint32_t tile) {
  extern __shared__ unsigned char smem_raw[];
  cx<T> *buf = reinterpret_cast<cx<T> *>(smem_raw);
  cx<T> *ltw = buf + p.tab_off;
  cx<T> *lwn = ltw + p.ntw;
  const cx<T> *gtw = reinterpret_cast<const cx<T> *>(p.tw);
  const cx<T> *gwn = reinterpret_cast<const cx<T> *>(p.wN);
  const int tid = threadIdx.x, nth = p.nthreads, step = (int)blockDim.x;
  const bool r2c = p.cls == CLS_R2C, c2r = p.cls == CLS_C2R;
  // R2C and the split DCT-I have the longest tables for their tiles: those
  // are loaded before the tile and written to LDS once the tile's loads are
  // issued, so that the two latencies overlap (512^3 FP64 R2C pass 0.651 ->
  // 0.62 ms, 513-point FP32 DCT-I 0.60 -> 0.575 ms; the DCT-I load phase also
  // reads its pre-twiddles and has to wait for all threads' copies).  The
  // other passes copy them first, which measured faster (512^3 FP32: C2C y
  // 0.201 against 0.206 ms, C2R 0.235 against 0.250 ms, which needs the merge
  // factors before its first value anyway).
  FixedStage<T> stage{{gtw, ltw, p.ntw, step, {}}, {gwn, lwn, M + 1, step, {}}, r2c, (bool)p.dct_split};
  if (r2c || p.dct_split) {
    stage.tw.load(tid);
    if (r2c) stage.wn.load(tid);
  } else {
    for (int i = tid; i < p.ntw; i += step) ltw[i] = gtw[i];
    if (c2r) {
      for (int i = tid; i <= M; i += step) lwn[i] = gwn[i];
      // the C2R load phase merges (X_k, X_{M-k}) with the split factors, so
      // they must be in LDS before any thread's load phase
      __syncthreads();
    }
  }
  DevPassRun<T> run{tid, nth};
  DevEach each{tid};
  fast_tile<T, M, DevPassRun<T>, DevEach, true, FixedStage<T>>(p, tile, buf, nth, run, each, ltw, lwn, stage);
}

template <typename T, int M>
__global__ void __launch_bounds__(P3E_FAST_MAX_THREADS) pass_kernel_pow2(PassArgs p) {
  pow2_body<T, M>(p, p.xcd_map ? xcd_tile(blockIdx.x, gridDim.x) : blockIdx.x);
}

// The same pass of many transforms in one launch (a batch stage): item i
// owns workgroups start[i] .. start[i+1] - 1 and runs with tab[i]; the
// workgroup size is the largest nthreads of the items (the others idle).
template <typename T, int M>
__global__ void __launch_bounds__(P3E_FAST_MAX_THREADS)
    pass_kernel_pow2_grp(const PassArgs *__restrict__ tab, const uint32_t *__restrict__ start, int n) {
  const uint32_t i = group_item(start, n, blockIdx.x);
  pow2_body<T, M>(tab[i], blockIdx.x - start[i]);
}

template <typename T, int M>
static inline int launch_pow2(const PassArgs *a, size_t lds_bytes, int threads, unsigned int nblocks, hipStream_t st) {
  if (lds_bytes > 65536)
    (void)hipFuncSetAttribute((const void *)pass_kernel_pow2<T, M>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds_bytes);
  hipLaunchKernelGGL((pass_kernel_pow2<T, M>), dim3(nblocks), dim3(threads), lds_bytes, st, *a);
  return (int)hipGetLastError();
}

template <typename T, int M>
static inline int launch_pow2_grp(const PassArgs *tab, const uint32_t *start, int n, size_t lds_bytes, int threads,
                           unsigned int nblocks, hipStream_t st) {
  if (lds_bytes > 65536)
    (void)hipFuncSetAttribute((const void *)pass_kernel_pow2_grp<T, M>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds_bytes);
  hipLaunchKernelGGL((pass_kernel_pow2_grp<T, M>), dim3(nblocks), dim3(threads), lds_bytes, st, tab, start, n);
  return (int)hipGetLastError();
}

}  // namespace p3e
