// Single-buffer mixed-radix path of the fused reorder + 1D transform pass:
// any work length L that is a product of the radices 2..10 and 12..16 (with
// 7, 11 and 13 as primes) and, in a kernel of its own, one odd prime P from
// 17 to 47; runtime L, radices and strides.
//
// The tile lives in LDS position-major: element m of line t at m pit + t,
// pit the (odd) number of lines plus one, and consecutive threads take
// consecutive lines.  Then
//   - a thread's addresses within a radix pass are one base plus multiples
//     of a workgroup-uniform step, whatever L is: no padding arithmetic and
//     one division per butterfly (j mod Ns) instead of several per element;
//   - LDS accesses of a pass touch consecutive elements, and a phase that
//     walks along a line touches elements an odd distance apart: few bank
//     conflicts for any radix;
//   - a pass that reads or writes the array across lines (tile order) is
//     coalesced as it is, so the first radix pass reads its operands from
//     global memory and the last one writes its results there (the load
//     and store phases, their LDS round trips and barriers are only needed
//     on a side that runs along lines, or whose elements mix: R2C splits,
//     C2R merges, DCT/DST).
// Real transforms (R2C, C2R, real DCT/DST) put two real lines in one complex
// line, z = x_{2t} + i x_{2t+1}: every transform is complex-linear, so one
// complex FFT serves both.  DCT/DST-II and -III of N points run an N-point
// FFT (Makhoul's reordering) instead of the 2N-point one of the extension.
// Bound by instruction issue and latency rather than by HBM: 3.5-4.5 TB/s of
// a pass's bytes on MI355X where its arrays fit the 256 MiB cache (copies
// reach 7 TB/s).  Against line-major padded lines with every pass through
// LDS, radices 2, 3, 4, 5, 8, 16 and 2N-point DCTs (FP32 unless stated): a
// 360-point C2C pass of 360^3 0.151 -> 0.091 ms (4.1 TB/s), its R2C pass 0.210
// -> 0.098 ms, a 376-point (8 47) pass 0.350 -> 0.154 ms, a 1024-point pass at
// 8 MiB strides, which only the two-buffer path took, 7.2 -> 1.8-2.2 ms, a
// one 256-point DCT-II call of 320x256x300 0.219 -> 0.113 ms, the FP64 DST-I
// pass of 129x255x200 0.117 -> 0.070 ms, an FP64 Bluestein pass of 131 points
// 0.245 -> 0.104 ms (0.165 through LDS on both sides and a product phase of its
// own, 0.131 with 20 values per thread).
// Shared by the HIP kernels and the host build used by the CPU tests.
#pragma once
#include "fft_core.h"

namespace p3e {

// What one tile's phases share: its coordinates and the tile in LDS.
template <typename T> struct MidTile {
  const PassArgs &p;
  cx<T> *buf;
  uint32_t f;
  int e0, nb, nl;  // first line, array lines and LDS lines of the tile
};

// Lines of LDS a tile of nb lines occupies.
P3E_HD P3E_INL int tile_lines(const PassArgs &p, int nb) { return p.pair ? (nb + 1) / 2 : nb; }

template <typename T> P3E_HD P3E_INL const char *tile_in(const MidTile<T> &t) {
  const long long esz = t.p.in_cplx ? 2 * sizeof(T) : sizeof(T);
  return reinterpret_cast<const char *>(t.p.in) + ((long long)t.e0 * t.p.is_e + (long long)t.f * t.p.is_f) * esz;
}
template <typename T> P3E_HD P3E_INL char *tile_out(const MidTile<T> &t) {
  const long long esz = t.p.out_cplx ? 2 * sizeof(T) : sizeof(T);
  return reinterpret_cast<char *>(t.p.out) + ((long long)t.e0 * t.p.os_e + (long long)t.f * t.p.os_f) * esz;
}

// y with its sign flipped where the mask is 1 << 31 (0: unchanged): the
// conjugation around a DFT of sign +1, without a branch.
template <typename T> P3E_HD P3E_INL T flip(T y, uint32_t mask) {
  if constexpr (sizeof(T) == 4) {
    union { T f; uint32_t u; } v = {y};
    v.u ^= mask;
    return v.f;
  } else {
    union { T f; uint64_t u; } v = {y};
    v.u ^= (uint64_t)mask << 32;
    return v.f;
  }
}
P3E_HD P3E_INL uint32_t sign_mask(const PassArgs &p) { return p.sign > 0 ? 0x80000000u : 0u; }

// Radix-R pass at input stride Ns of the DFT with sign -1 (a DFT with sign +1
// is the conjugate of this one of the conjugate; mask: the conjugation at a
// global side).  IN: MidIn, OUT: MidOut; a prime above 16 writes to LDS only.
template <typename T, int R, int E, int IN, int OUT> struct MPass {
  static constexpr int NB = mid_butterflies(R, E);  // butterflies per thread
  static constexpr int SLOTS = NB * R;
  static constexpr uint32_t RS = sizeof(T), CS = 2 * sizeof(T);
  const MidTile<T> &t;
  int L, lgl, pit;  // p.L, p.lgl, p.pit
  int Ns;
  FastDiv dns;
  const cx<T> *tw;  // w^(k r), w = e^(-2 pi i / (Ns R)), at k (R - 1) + r - 1
  char *gl;         // the tile's first element in global memory (IN or OUT)
  uint32_t mask;

  // Butterflies past the tile's last one read that one's operands (no
  // branch: every load of the thread is issued before the first is used).
  // Offsets: L / R rows and the tile's width stay below 2^32 bytes (the
  // planner's condition), the R operands are uniform 64-bit steps apart.
  P3E_HD P3E_INL void read(int tid, int nth, cx<T> *v) const {
    const PassArgs &p = t.p;
    const int nbf = L / R, last = (nbf << lgl) - 1, lines = (1 << lgl) - 1;
#pragma unroll
    for (int m = 0; m < NB; m++) {
      int b = tid + m * nth;
      b = b < last ? b : last;
      const int line = b & lines, j = b >> lgl;
      cx<T> *w = v + m * R;
      if constexpr (IN == MID_IN_LDS) {
        const cx<T> *q = t.buf + j * pit + line;
        const int step = nbf * pit;
#pragma unroll
        for (int r = 0; r < R; r++) w[r] = q[r * step];
      } else {
        const uint32_t l = line < t.nl ? (uint32_t)line : 0u;
        if constexpr (IN == MID_IN_CPLX) {
          const uint32_t off = ((uint32_t)j * (uint32_t)p.is_d + l * (uint32_t)p.is_e) * CS;
          const long long step = (long long)nbf * p.is_d * CS;
#pragma unroll
          for (int r = 0; r < R; r++) w[r] = ldg<cx<T>>(gl + r * step, off);
        } else if constexpr (IN == MID_IN_BLUE) {
          // rows of the line only: past it, a row that is in the line (the
          // value is dropped), from a base that is in it too
          const uint32_t lo = l * (uint32_t)p.is_e * CS, off = (uint32_t)j * (uint32_t)p.is_d * CS + lo;
          const long long step = (long long)nbf * p.is_d * CS;
#pragma unroll
          for (int r = 0; r < R; r++)
            w[r] = ldg<cx<T>>(r * nbf < p.W ? gl + r * step : gl, j + r * nbf < p.W ? off : lo);
        } else {
          // lines 2l and 2l + 1 of a real array, adjacent in memory
          const uint32_t off = ((uint32_t)j * (uint32_t)p.is_d + 2 * l) * RS;
          const long long step = (long long)nbf * p.is_d * RS;
#pragma unroll
          for (int r = 0; r < R; r++) {
            const RealPair<T> x = ldg<RealPair<T>>(gl + r * step, off);
            w[r] = mk(x.a, x.b);
          }
        }
      }
    }
  }

  P3E_HD P3E_INL void write(int tid, int nth, cx<T> *v) const {
    const PassArgs &p = t.p;
    const int nbf = L / R, total = nbf << lgl, lines = (1 << lgl) - 1;
#pragma unroll
    for (int m = 0; m < NB; m++) {
      const int b = tid + m * nth;
      if (b >= total) continue;
      const int line = b & lines, j = b >> lgl;
      int k = 0;
      cx<T> *w = v + m * R;
      if constexpr (IN == MID_IN_CPLX) {
#pragma unroll
        for (int r = 0; r < R; r++) w[r].y = flip(w[r].y, mask);
      }
      if constexpr (IN == MID_IN_BLUE) {
        const cx<T> *ch = reinterpret_cast<const cx<T> *>(p.chirp);
#pragma unroll
        for (int r = 0; r < R; r++) {
          const int n = j + r * nbf;
          const cx<T> x = mul(w[r], ch[n < p.W ? n : 0]);
          w[r] = n < p.W ? x : mk((T)0, (T)0);
        }
      }
      if (IN == MID_IN_LDS && Ns > 1) {
        k = j - (int)fdiv((uint32_t)j, dns) * Ns;
        const cx<T> *tk = tw + k * (R - 1);
#pragma unroll
        for (int r = 1; r < R; r++) w[r] = mul(w[r], tk[r - 1]);
      }
      if constexpr (OUT == MID_OUT_LDS) {
        cx<T> *d = t.buf + ((j - k) * R + k) * pit + line;
        const int step = Ns * pit;
        if constexpr (R > 16) {
          // each output leaves its registers as soon as it is formed
          bf_prime<T, R>(w, -1, [&](int r, cx<T> x) P3E_LAMBDA_INL { d[r * step] = x; });
        } else {
          bfly<T, R>(w, -1);
#pragma unroll
          for (int r = 0; r < R; r++) d[r * step] = w[r];
        }
      } else if constexpr (OUT == MID_OUT_HAT) {
        // last pass of the forward FFT of a convolution: conjugated, so that
        // the inverse FFT is another forward one
        const cx<T> *hat = reinterpret_cast<const cx<T> *>(p.chirp_hat);
        cx<T> *d = t.buf + j * pit + line;
        bfly<T, R>(w, -1);
#pragma unroll
        for (int r = 0; r < R; r++) d[r * nbf * pit] = conj(mul(w[r], hat[j + r * nbf]));
      } else if constexpr (OUT == MID_OUT_BLUE) {
        const cx<T> *ch = reinterpret_cast<const cx<T> *>(p.chirp);
        bfly<T, R>(w, -1);
        if (line >= t.nl) continue;
        const uint32_t off = ((uint32_t)j * (uint32_t)p.os_d + (uint32_t)line * (uint32_t)p.os_e) * CS;
        const long long step = (long long)nbf * p.os_d * CS;
#pragma unroll
        for (int r = 0; r < R; r++) {
          const int k = j + r * nbf;
          if (k >= p.N) continue;
          stg(gl + r * step, off, out_rule(p, mul(conj(w[r]), ch[k]), k, t.e0 + line, t.f));
        }
      } else {
        // last pass: Ns = L / R, output positions j + r Ns
        bfly<T, R>(w, -1);
#pragma unroll
        for (int r = 0; r < R; r++) w[r].y = flip(w[r].y, mask);
        if (line >= t.nl) continue;
        if constexpr (OUT == MID_OUT_PAIR) {
          const uint32_t off = ((uint32_t)j * (uint32_t)p.os_d + 2u * (uint32_t)line) * RS;
          const long long step = (long long)nbf * p.os_d * RS;
#pragma unroll
          for (int r = 0; r < R; r++) stg(gl + r * step, off, RealPair<T>{w[r].x, w[r].y});
        } else {
          const uint32_t off = ((uint32_t)j * (uint32_t)p.os_d + (uint32_t)line * (uint32_t)p.os_e) * CS;
          const long long step = (long long)nbf * p.os_d * CS;
#pragma unroll
          for (int r = 0; r < R; r++) {
            if constexpr (OUT == MID_OUT_RULE) w[r] = out_rule(p, w[r], j + r * nbf, t.e0 + line, t.f);
            stg(gl + r * step, off, w[r]);
          }
        }
      }
    }
  }
};

// FFT of length L in place (Bluestein: both FFTs of the convolution and the
// spectrum product between them); `run` executes one pass (read half, barrier,
// write half, barrier).  tw: the twiddles of the passes after the first,
// pass by pass.  P: the largest prime radix of the instantiation (0: none
// above 16; 23, 31 and 47 also run the smaller primes above 16, 23 and 31;
// any other prime only itself).
template <typename T, int P, int E, int IN, int OUT, typename Run>
P3E_HD P3E_INL void mid_pass(Run &run, const MidTile<T> &t, int R, int L, int lgl, int pit, int Ns, const FastDiv &dns,
                             const cx<T> *tw, char *gl, uint32_t mask) {
#define P3E_MID_CASE(RR)                                                   \
  case RR: {                                                               \
    MPass<T, RR, E, IN, OUT> ps{t, L, lgl, pit, Ns, dns, tw, gl, mask};       \
    run(ps);                                                               \
  } break;
  switch (R) {
    P3E_MID_CASE(2)
    P3E_MID_CASE(3)
    P3E_MID_CASE(4)
    P3E_MID_CASE(5)
    P3E_MID_CASE(6)
    P3E_MID_CASE(7)
    P3E_MID_CASE(8)
    P3E_MID_CASE(9)
    P3E_MID_CASE(10)
    P3E_MID_CASE(12)
    P3E_MID_CASE(16)
    default:
      // the planner admits no other radix to the instantiation
      if constexpr (P <= 16) {
        switch (R) {
          P3E_MID_CASE(11)
          P3E_MID_CASE(13)
          P3E_MID_CASE(14)
          P3E_MID_CASE(15)
        }
      } else if constexpr (OUT == MID_OUT_LDS) {
        if constexpr (P == 23) {
          switch (R) {
            P3E_MID_CASE(17)
            P3E_MID_CASE(19)
            P3E_MID_CASE(23)
          }
        } else if constexpr (P == 31) {
          switch (R) {
            P3E_MID_CASE(29)
            P3E_MID_CASE(31)
          }
        } else if constexpr (P == 47) {
          switch (R) {
            P3E_MID_CASE(37)
            P3E_MID_CASE(41)
            P3E_MID_CASE(43)
            P3E_MID_CASE(47)
          }
        } else {
          switch (R) { P3E_MID_CASE(P) }
        }
      }
      break;
  }
#undef P3E_MID_CASE
}

template <typename T, int P, int E, int IN, int OUT, bool BLUE, typename Run>
P3E_HD P3E_INL void mid_fft(Run &run, const MidTile<T> &t, const cx<T> *tw0, char *src, char *dst, uint32_t mask) {
  const PassArgs &p = t.p;
  const cx<T> *tw = tw0;
  const int np = BLUE ? 2 * p.nrad : p.nrad;
  int Ns = 1;
  for (int q = 0; q < np; q++) {
    const int i = BLUE && q >= p.nrad ? q - p.nrad : q;
    if (i == 0) {
      Ns = 1;
      tw = tw0;
    }
    const int R = p.radix[i];
    const FastDiv ds = p.div_ns[i];
    int L = p.L, lgl = p.lgl, pit = p.pit;
    // opaque per pass: the address arithmetic of every radix is invariant
    // over this loop, and the compiler would hoist all of it (256 VGPRs and
    // 2.3 KiB of scratch per lane)
    P3E_OPAQUE_S(L);
    P3E_OPAQUE_S(lgl);
    P3E_OPAQUE_S(pit);
    if (IN != MID_IN_LDS && q == 0)
      mid_pass<T, P, E, IN, MID_OUT_LDS>(run, t, R, L, lgl, pit, Ns, ds, tw, src, mask);
    else if (BLUE && q == p.nrad - 1)
      mid_pass<T, P, E, MID_IN_LDS, BLUE ? MID_OUT_HAT : MID_OUT_LDS>(run, t, R, L, lgl, pit, Ns, ds, tw, nullptr, 0u);
    else if (OUT != MID_OUT_LDS && q == np - 1)
      mid_pass<T, P, E, MID_IN_LDS, OUT>(run, t, R, L, lgl, pit, Ns, ds, tw, dst, mask);
    else
      mid_pass<T, P, E, MID_IN_LDS, MID_OUT_LDS>(run, t, R, L, lgl, pit, Ns, ds, tw, nullptr, 0u);
    if (Ns > 1) tw += Ns * (R - 1);
    Ns *= R;
  }
}

// ---------------------------------------------------------------- load phase
// Into LDS, in groups of U entries per thread: the loads of a group are all
// issued before its LDS writes.  Out-of-tile entries load the tile's first
// element (always valid) and are not written.

// (line, element) of entry i: along lines of len elements, or across the
// tile's 2^lgl LDS lines.
P3E_HD P3E_INL void mid_index(const PassArgs &p, bool along, int i, int len, const FastDiv &dlen, int *line, int *n) {
  if (along) {
    *line = (int)fdiv((uint32_t)i, dlen);
    *n = i - *line * len;
  } else {
    *line = i & ((1 << p.lgl) - 1);
    *n = i >> p.lgl;
  }
}

// Element m of a line's work sequence: chirped (Bluestein) or conjugated (a
// DFT of sign +1).
template <typename T, bool BLUE> P3E_HD P3E_INL void mid_put(const PassArgs &p, cx<T> *line, int m, cx<T> v) {
  if (BLUE) v = mul(v, reinterpret_cast<const cx<T> *>(p.chirp)[m]);
  else v.y = flip(v.y, sign_mask(p));
  line[m * p.pit] = v;
}

// Input element n of a line into the work sequence (DCT/DST extensions and
// the reordering of the short forms of type II).
template <typename T, int CLS, bool BLUE> P3E_HD P3E_INL void mid_scatter(const PassArgs &p, cx<T> *line, int n, cx<T> x) {
  const int N = p.N, W = p.W;
  const cx<T> y = mk(-x.x, -x.y);
  if constexpr (CLS != CLS_R2R) {
    mid_put<T, BLUE>(p, line, n, x);
    return;
  }
  const cx<T> *pre = reinterpret_cast<const cx<T> *>(p.pre);
  switch (p.r2r_kind) {
    case REDFT00:
      mid_put<T, BLUE>(p, line, n, x);
      if (n >= 1 && n <= N - 2) mid_put<T, BLUE>(p, line, W - n, x);
      break;
    case RODFT00:
      mid_put<T, BLUE>(p, line, n + 1, x);
      mid_put<T, BLUE>(p, line, W - n - 1, y);
      break;
    case REDFT10:
    case RODFT10: {
      const cx<T> z = (p.r2r_kind == RODFT10 && (n & 1)) ? y : x;
      if (p.dct_short) {
        mid_put<T, BLUE>(p, line, (n & 1) ? N - 1 - (n >> 1) : n >> 1, z);
      } else {
        mid_put<T, BLUE>(p, line, n, x);
        mid_put<T, BLUE>(p, line, 2 * N - 1 - n, p.r2r_kind == RODFT10 ? y : x);
      }
      break;
    }
    case REDFT01:
      mid_put<T, BLUE>(p, line, n, mul(x, pre[n]));
      if (n >= 1) mid_put<T, BLUE>(p, line, 2 * N - n, mul(y, pre[2 * N - n]));
      break;
    case RODFT01:
      mid_put<T, BLUE>(p, line, n + 1, mul(x, pre[n + 1]));
      if (n <= N - 2) mid_put<T, BLUE>(p, line, 2 * N - n - 1, mul(x, pre[2 * N - n - 1]));
      break;
    case REDFT11:
      mid_put<T, BLUE>(p, line, n, mul(x, pre[n]));
      mid_put<T, BLUE>(p, line, 2 * N - 1 - n, mul(y, pre[2 * N - 1 - n]));
      break;
    case RODFT11:
      mid_put<T, BLUE>(p, line, n, mul(x, pre[n]));
      mid_put<T, BLUE>(p, line, 2 * N - 1 - n, mul(x, pre[2 * N - 1 - n]));
      break;
  }
}

// Element n of LDS line l: the complex element, or the real elements of
// lines 2l and 2l + 1 (0 for an absent line) as one complex value.
template <typename T> P3E_HD P3E_INL cx<T> mid_fetch(const MidTile<T> &t, const char *tin, int l, int n, bool ok) {
  const PassArgs &p = t.p;
  if (p.in_cplx) {
    const unsigned long long o = (unsigned long long)(uint32_t)n * (uint32_t)p.is_d + (uint32_t)l * (uint32_t)p.is_e;
    return *reinterpret_cast<const cx<T> *>(tin + (ok ? o * (2 * sizeof(T)) : 0));
  }
  const unsigned long long o = (unsigned long long)(uint32_t)n * (uint32_t)p.is_d + 2u * (uint32_t)l * (uint32_t)p.is_e;
  const T *q = reinterpret_cast<const T *>(tin + (ok ? o * sizeof(T) : 0));
  const bool two = ok && 2 * l + 1 < t.nb;
  const T a = q[0], b = q[two ? p.is_e : 0];
  return mk(a, two ? b : (T)0);
}

template <typename T, int CLS, bool BLUE> P3E_HD P3E_INL void mid_load(const MidTile<T> &t, int tid, int nth) {
  constexpr uint32_t RS = sizeof(T), CS = 2 * sizeof(T);
  constexpr int U = 32 / sizeof(T);  // complex values in flight per thread
  const PassArgs &p = t.p;
  const char *tin = tile_in(t);
  const bool along = p.load_order == ORD_LINE;
  const int N = p.N, nl = t.nl, rows = along ? nl : 1 << p.lgl;
  const int ise = (int)p.is_e;
  if constexpr (BLUE) {
    const int tail = (p.L - p.W) << p.lgl;
    for (int i = tid; i < tail; i += nth)
      t.buf[(p.W + (i >> p.lgl)) * p.pit + (i & ((1 << p.lgl) - 1))] = mk((T)0, (T)0);
  }
  if constexpr (CLS == CLS_C2R) {
    // Z_k = Y_{2l,k} + i Y_{2l+1,k} over the Hermitian extension of both half
    // spectra; the imaginary parts of the DC and (even N) Nyquist inputs are
    // dropped first, as a real inverse transform ignores them
    const int tot = rows * p.nin;
    const unsigned long long isd = (unsigned long long)p.is_d;
    for (int i0 = tid; i0 < tot; i0 += (U / 2) * nth) {
      T v[2 * U];
#pragma unroll
      for (int u = 0; u < U / 2; u++) {
        const int i = i0 + u * nth;
        int l, n;
        mid_index(p, along, i, p.nin, p.div_nin, &l, &n);
        const bool ok = i < tot && l < nl, two = ok && 2 * l + 1 < t.nb;
        const char *q = tin + (ok ? ((uint32_t)n * isd + 2u * (uint32_t)l * (uint32_t)ise) * CS : 0);
        if (p.vec2) {
          const CxPair<T> y = *reinterpret_cast<const CxPair<T> *>(q);
          v[4 * u] = y.ar;
          v[4 * u + 1] = y.ai;
          v[4 * u + 2] = y.br;
          v[4 * u + 3] = y.bi;
        } else {
          const cx<T> a = *reinterpret_cast<const cx<T> *>(q);
          const cx<T> b = *reinterpret_cast<const cx<T> *>(q + (two ? (size_t)ise * CS : 0));
          v[4 * u] = a.x;
          v[4 * u + 1] = a.y;
          v[4 * u + 2] = two ? b.x : (T)0;
          v[4 * u + 3] = two ? b.y : (T)0;
        }
      }
#pragma unroll
      for (int u = 0; u < U / 2; u++) {
        const int i = i0 + u * nth;
        int l, n;
        mid_index(p, along, i, p.nin, p.div_nin, &l, &n);
        if (!(i < tot && l < nl)) continue;
        cx<T> a = mk(v[4 * u], v[4 * u + 1]), b = mk(v[4 * u + 2], v[4 * u + 3]);
        if (n == 0 || 2 * n == N) {
          a.y = (T)0;
          b.y = (T)0;
        }
        cx<T> *line = t.buf + l;
        mid_put<T, BLUE>(p, line, n, mk(a.x - b.y, a.y + b.x));
        if (n >= 1 && n < (N + 1) / 2) mid_put<T, BLUE>(p, line, N - n, mk(a.x + b.y, b.x - a.y));
      }
    }
    return;
  }
  if (CLS == CLS_R2R && p.dct_short && (p.r2r_kind == REDFT01 || p.r2r_kind == RODFT01)) {
    // type III: V_n = (x_n - i x_{N-n}) e^{i pi n / 2N} (x_N = 0), both ends of
    // a pair in one thread; DST-III is the DCT-III of the reversed line
    const cx<T> *pre = reinterpret_cast<const cx<T> *>(p.pre);
    const bool rev = p.r2r_kind == RODFT01;
    const int H = N / 2 + 1, tot = rows * H;
    for (int i0 = tid; i0 < tot; i0 += (U / 2) * nth) {
      T v[2 * U];
#pragma unroll
      for (int u = 0; u < U / 2; u++) {
        const int i = i0 + u * nth;
        int l, n;
        mid_index(p, along, i, H, p.div_pairs, &l, &n);
        const bool ok = i < tot && l < nl;
        const int n2 = n ? N - n : 0;
        const cx<T> a = mid_fetch(t, tin, l, rev ? N - 1 - n : n, ok), b = mid_fetch(t, tin, l, rev ? N - 1 - n2 : n2, ok);
        v[4 * u] = a.x;
        v[4 * u + 1] = a.y;
        v[4 * u + 2] = n ? b.x : (T)0;
        v[4 * u + 3] = n ? b.y : (T)0;
      }
#pragma unroll
      for (int u = 0; u < U / 2; u++) {
        const int i = i0 + u * nth;
        int l, n;
        mid_index(p, along, i, H, p.div_pairs, &l, &n);
        if (!(i < tot && l < nl)) continue;
        const cx<T> a = mk(v[4 * u], v[4 * u + 1]), b = mk(v[4 * u + 2], v[4 * u + 3]), w = pre[n];
        cx<T> *line = t.buf + l;
        mid_put<T, BLUE>(p, line, n, mul(add(a, rot(b, -1)), w));
        if (n && 2 * n != N) mid_put<T, BLUE>(p, line, N - n, mul(add(a, rot(b, 1)), conj(w)));
      }
    }
    return;
  }
  if (CLS != CLS_R2R && p.vec2 && along) {
    // elements n = 2 m and n + 1 of a line per load (p.div_pairs divides by
    // nin / 2)
    const int half = p.nin / 2, tot = nl * half;
    for (int i0 = tid; i0 < tot; i0 += (U / 2) * nth) {
      T v[2 * U];
#pragma unroll
      for (int u = 0; u < U / 2; u++) {
        const int i = i0 + u * nth;
        const int l = (int)fdiv((uint32_t)i, p.div_pairs), n = 2 * (i - l * half);
        const bool ok = i < tot;
        if constexpr (CLS == CLS_R2C) {
          const uint32_t off = ok ? (uint32_t)(n + 2 * l * ise) * RS : 0u;
          const bool two = ok && 2 * l + 1 < t.nb;
          const RealPair<T> a = ldg_nt<RealPair<T>>(tin, off);
          const RealPair<T> b = ldg_nt<RealPair<T>>(tin, two ? off + (uint32_t)ise * RS : off);
          v[4 * u] = a.a;
          v[4 * u + 1] = two ? b.a : (T)0;
          v[4 * u + 2] = a.b;
          v[4 * u + 3] = two ? b.b : (T)0;
        } else {
          const CxPair<T> a = ldg_nt<CxPair<T>>(tin, ok ? (uint32_t)(n + l * ise) * CS : 0u);
          v[4 * u] = a.ar;
          v[4 * u + 1] = a.ai;
          v[4 * u + 2] = a.br;
          v[4 * u + 3] = a.bi;
        }
      }
#pragma unroll
      for (int u = 0; u < U / 2; u++) {
        const int i = i0 + u * nth;
        if (i >= tot) continue;
        const int l = (int)fdiv((uint32_t)i, p.div_pairs), n = 2 * (i - l * half);
        mid_put<T, BLUE>(p, t.buf + l, n, mk(v[4 * u], v[4 * u + 1]));
        mid_put<T, BLUE>(p, t.buf + l, n + 1, mk(v[4 * u + 2], v[4 * u + 3]));
      }
    }
    return;
  }
  const int tot = rows * p.nin;
  for (int i0 = tid; i0 < tot; i0 += U * nth) {
    T v[2 * U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * nth;
      int l, n;
      mid_index(p, along, i, p.nin, p.div_nin, &l, &n);
      const cx<T> x = mid_fetch(t, tin, l, n, i < tot && l < nl);
      v[2 * u] = x.x;
      v[2 * u + 1] = x.y;
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * nth;
      int l, n;
      mid_index(p, along, i, p.nin, p.div_nin, &l, &n);
      if (i < tot && l < nl) mid_scatter<T, CLS, BLUE>(p, t.buf + l, n, mk(v[2 * u], v[2 * u + 1]));
    }
  }
}

// ---------------------------------------------------------------- store phase

// Work element m of a line after the FFT.
template <typename T, bool BLUE> P3E_HD P3E_INL cx<T> mid_get(const PassArgs &p, const cx<T> *line, int m) {
  const cx<T> z = line[m * p.pit];
  return BLUE ? mul(conj(z), reinterpret_cast<const cx<T> *>(p.chirp)[m]) : mk(z.x, flip(z.y, sign_mask(p)));
}

// Output k of a line, before the output rule (every class but R2C).
template <typename T, int CLS, bool BLUE> P3E_HD P3E_INL cx<T> mid_result(const PassArgs &p, const cx<T> *line, int k) {
  if constexpr (CLS != CLS_R2R) return mid_get<T, BLUE>(p, line, k);
  const cx<T> *post = reinterpret_cast<const cx<T> *>(p.post);
  const int N = p.N;
  if (p.dct_short) {
    // type III (type II: mid_store)
    const cx<T> z = mid_get<T, BLUE>(p, line, (k & 1) ? N - 1 - (k >> 1) : k >> 1);
    return (p.r2r_kind == RODFT01 && (k & 1)) ? mk(-z.x, -z.y) : z;
  }
  const cx<T> z = mid_get<T, BLUE>(p, line, k + p.post_off);
  return p.post_mode ? mul(z, post[k]) : z;
}

template <typename T, int CLS, bool BLUE> P3E_HD P3E_INL void mid_store(const MidTile<T> &t, int tid, int nth) {
  constexpr uint32_t RS = sizeof(T), CS = 2 * sizeof(T);
  const PassArgs &p = t.p;
  char *tout = tile_out(t);
  const bool along = p.store_order == ORD_LINE;
  const int N = p.N, nl = t.nl, rows = along ? nl : 1 << p.lgl;
  const int ose = (int)p.os_e;
  const unsigned long long osd = (unsigned long long)p.os_d;
  if constexpr (CLS == CLS_R2C) {
    // X_{2l,k} = (Z_k + conj Z_{N-k}) / 2, X_{2l+1,k} = (Z_k - conj Z_{N-k}) / 2i
    const int tot = rows * p.nout;
#pragma unroll 2
    for (int i = tid; i < tot; i += nth) {
      int l, k;
      mid_index(p, along, i, p.nout, p.div_nout, &l, &k);
      if (l >= nl) continue;
      const cx<T> z = mid_get<T, BLUE>(p, t.buf + l, k), zm = mid_get<T, BLUE>(p, t.buf + l, k ? N - k : 0);
      cx<T> y0 = mk((T)0.5 * (z.x + zm.x), (T)0.5 * (z.y - zm.y));
      cx<T> y1 = mk((T)0.5 * (z.y + zm.y), (T)0.5 * (zm.x - z.x));
      if (p.deriv | p.spec_op | p.has_scale) {
        y0 = out_rule(p, y0, k, t.e0 + 2 * l, t.f);
        y1 = out_rule(p, y1, k, t.e0 + 2 * l + 1, t.f);
      }
      char *q = tout + ((uint32_t)k * osd + 2u * (uint32_t)l * (uint32_t)ose) * CS;
      if (p.vec2s) {
        CxPair<T> v;
        v.ar = y0.x;
        v.ai = y0.y;
        v.br = y1.x;
        v.bi = y1.y;
        *reinterpret_cast<CxPair<T> *>(q) = v;
      } else {
        *reinterpret_cast<cx<T> *>(q) = y0;
        if (2 * l + 1 < t.nb) *reinterpret_cast<cx<T> *>(q + (size_t)ose * CS) = y1;
      }
    }
    return;
  }
  if (CLS != CLS_R2R && p.vec2s && along) {
    // outputs k = 2 m and k + 1 of a line per store (p.div_pairs2 divides by
    // nout / 2)
    const int half = p.nout / 2, tot = nl * half;
#pragma unroll 2
    for (int i = tid; i < tot; i += nth) {
      const int l = (int)fdiv((uint32_t)i, p.div_pairs2), k = 2 * (i - l * half);
      cx<T> a = mid_get<T, BLUE>(p, t.buf + l, k), b = mid_get<T, BLUE>(p, t.buf + l, k + 1);
      if constexpr (CLS == CLS_C2R) {
        if (p.has_scale) {
          a = scl(a, (T)p.scale);
          b = scl(b, (T)p.scale);
        }
        const uint32_t off = (uint32_t)(k + 2 * l * ose) * RS;
        RealPair<T> v;
        v.a = a.x;
        v.b = b.x;
        stg_nt(tout, off, v);
        if (2 * l + 1 < t.nb) {
          v.a = a.y;
          v.b = b.y;
          stg_nt(tout, off + (uint32_t)ose * RS, v);
        }
      } else {
        a = out_rule(p, a, k, t.e0 + l, t.f);
        b = out_rule(p, b, k + 1, t.e0 + l, t.f);
        CxPair<T> v;
        v.ar = a.x;
        v.ai = a.y;
        v.br = b.x;
        v.bi = b.y;
        stg_nt(tout, (uint32_t)(k + l * ose) * CS, v);
      }
    }
    return;
  }
  const auto emit = [&](int l, int k, cx<T> y) P3E_LAMBDA_INL {
    if (p.out_cplx) {
      y = out_rule(p, y, k, t.e0 + l, t.f);
      *reinterpret_cast<cx<T> *>(tout + ((uint32_t)k * osd + (uint32_t)l * (uint32_t)ose) * CS) = y;
    } else {
      if (p.has_scale) y = scl(y, (T)p.scale);
      char *q = tout + ((uint32_t)k * osd + 2u * (uint32_t)l * (uint32_t)ose) * RS;
      if (p.vec2s && !along) {
        RealPair<T> v;
        v.a = y.x;
        v.b = y.y;
        *reinterpret_cast<RealPair<T> *>(q) = v;
      } else {
        *reinterpret_cast<T *>(q) = y.x;
        if (2 * l + 1 < t.nb) *reinterpret_cast<T *>(q + (size_t)ose * RS) = y.y;
      }
    }
  };
  // groups of G values per thread: the table and LDS reads of a group are all
  // issued before its stores (which the compiler cannot move reads across; one
  // 256-point DCT-II call of 320x256x300 FP32 0.121 -> 0.113 ms with both outputs
  // of a pair in one thread).  The classes without a table are slower so
  // (300x250x360 FP32 round trip 0.314 -> 0.325 ms)
  constexpr int G = 16 / sizeof(T);
  if (CLS == CLS_R2R && p.dct_short && (p.r2r_kind == REDFT10 || p.r2r_kind == RODFT10)) {
    // a = w^k V_k, b = conj(w^k) V_{N-k}, w = e^{-i pi / 2N}: Y_k = a + b and
    // Y_{N-k} = i (a - b), both outputs in one thread; DST-II is the DCT-II of
    // (-1)^n x_n with its outputs reversed
    const cx<T> *post = reinterpret_cast<const cx<T> *>(p.post);
    const bool rev = p.r2r_kind == RODFT10;
    const int H = N / 2 + 1, tot = rows * H;
    for (int i0 = tid; i0 < tot; i0 += G * nth) {
      T v[4 * G];
#pragma unroll
      for (int u = 0; u < G; u++) {
        const int i = i0 + u * nth;
        int l, k;
        mid_index(p, along, i < tot ? i : 0, H, p.div_pairs, &l, &k);
        const cx<T> w = post[k];
        const cx<T> a = mul(w, mid_get<T, BLUE>(p, t.buf + l, k));
        const cx<T> b = mul(conj(w), mid_get<T, BLUE>(p, t.buf + l, k ? N - k : 0));
        v[4 * u] = a.x;
        v[4 * u + 1] = a.y;
        v[4 * u + 2] = b.x;
        v[4 * u + 3] = b.y;
      }
#pragma unroll
      for (int u = 0; u < G; u++) {
        const int i = i0 + u * nth;
        int l, k;
        mid_index(p, along, i, H, p.div_pairs, &l, &k);
        if (!(i < tot && l < nl)) continue;
        const cx<T> a = mk(v[4 * u], v[4 * u + 1]), b = mk(v[4 * u + 2], v[4 * u + 3]);
        emit(l, rev ? N - 1 - k : k, add(a, b));
        if (k && 2 * k != N) emit(l, rev ? k - 1 : N - k, mk(b.y - a.y, a.x - b.x));
      }
    }
    return;
  }
  const int tot = rows * p.nout;
  if constexpr (CLS != CLS_R2R) {
    // (no table)
#pragma unroll 2
    for (int i = tid; i < tot; i += nth) {
      int l, k;
      mid_index(p, along, i, p.nout, p.div_nout, &l, &k);
      if (l < nl) emit(l, k, mid_result<T, CLS, BLUE>(p, t.buf + l, k));
    }
    return;
  }
  for (int i0 = tid; i0 < tot; i0 += G * nth) {
    T v[2 * G];
#pragma unroll
    for (int u = 0; u < G; u++) {
      const int i = i0 + u * nth;
      int l, k;
      mid_index(p, along, i < tot ? i : 0, p.nout, p.div_nout, &l, &k);
      const cx<T> y = mid_result<T, CLS, BLUE>(p, t.buf + l, k);
      v[2 * u] = y.x;
      v[2 * u + 1] = y.y;
    }
#pragma unroll
    for (int u = 0; u < G; u++) {
      const int i = i0 + u * nth;
      int l, k;
      mid_index(p, along, i, p.nout, p.div_nout, &l, &k);
      if (i < tot && l < nl) emit(l, k, mk(v[2 * u], v[2 * u + 1]));
    }
  }
}

// Whole tile of a pass of class CLS by the given routes.  `each(f)` runs
// phase f for the calling thread and ends with a barrier (device), or runs
// it for every thread in turn (host build).  Only threads tid < nth work;
// the others take part in the barriers.
template <typename T, int P, int E, int CLS, int IN, int OUT, bool BLUE, typename Run, typename Each>
P3E_HD P3E_INL void mid_tile_as(const PassArgs &p, uint32_t tile, cx<T> *buf, int nth, Run &run, Each &each,
                                const cx<T> *tw) {
  uint32_t f;
  int e0, nb;
  generic_tile_coords(p, tile, &f, &e0, &nb);
  const MidTile<T> t{p, buf, f, e0, nb, tile_lines(p, nb)};
  if constexpr (IN == MID_IN_LDS) {
    if ((CLS == CLS_R2R) && p.zero_fill)
      each([&](int tid) P3E_LAMBDA_INL {
        if (tid < nth)
          for (int i = tid; i < p.L << p.lgl; i += nth)
            buf[(i >> p.lgl) * p.pit + (i & ((1 << p.lgl) - 1))] = mk((T)0, (T)0);
      });
    each([&](int tid) P3E_LAMBDA_INL {
      if (tid < nth) mid_load<T, CLS, BLUE>(t, tid, nth);
    });
  }
  char *src = const_cast<char *>(tile_in(t)), *dst = tile_out(t);
  // Bluestein: the store conjugates back and applies the output chirp
  mid_fft<T, P, E, IN, OUT, BLUE>(run, t, tw, src, dst, BLUE ? 0u : sign_mask(p));
  if constexpr (OUT == MID_OUT_LDS)
    each([&](int tid) P3E_LAMBDA_INL {
      if (tid < nth) mid_store<T, CLS, BLUE>(t, tid, nth);
    });
}

// The instantiation that pass p takes: f(class, in route, out route,
// Bluestein) with compile-time values (std::integral_constant-like tags).
template <int V> struct MidC {
  static constexpr int v = V;
};
template <int P, typename F> P3E_HD P3E_INL void mid_dispatch(const PassArgs &p, F f) {
  const int in = mid_in_route(p), out = mid_out_route(p);
  if (P <= 16 && p.bluestein) {
    switch (p.cls) {
      case CLS_C2C:
        if (in == MID_IN_LDS) {
          if (out == MID_OUT_LDS) return f(MidC<CLS_C2C>{}, MidC<0>{}, MidC<0>{}, MidC<P <= 16>{});
          return f(MidC<CLS_C2C>{}, MidC<0>{}, MidC<MID_OUT_BLUE>{}, MidC<P <= 16>{});
        }
        if (out == MID_OUT_LDS) return f(MidC<CLS_C2C>{}, MidC<MID_IN_BLUE>{}, MidC<0>{}, MidC<P <= 16>{});
        return f(MidC<CLS_C2C>{}, MidC<MID_IN_BLUE>{}, MidC<MID_OUT_BLUE>{}, MidC<P <= 16>{});
      case CLS_R2C: return f(MidC<CLS_R2C>{}, MidC<0>{}, MidC<0>{}, MidC<P <= 16>{});
      case CLS_C2R: return f(MidC<CLS_C2R>{}, MidC<0>{}, MidC<0>{}, MidC<P <= 16>{});
      default: return f(MidC<CLS_R2R>{}, MidC<0>{}, MidC<0>{}, MidC<P <= 16>{});
    }
  }
  switch (p.cls) {
    case CLS_C2C:
      if (in == MID_IN_LDS) {
        if (out == MID_OUT_LDS) return f(MidC<CLS_C2C>{}, MidC<0>{}, MidC<0>{}, MidC<0>{});
        if (out == MID_OUT_CPLX) return f(MidC<CLS_C2C>{}, MidC<0>{}, MidC<MID_OUT_CPLX>{}, MidC<0>{});
        return f(MidC<CLS_C2C>{}, MidC<0>{}, MidC<MID_OUT_RULE>{}, MidC<0>{});
      }
      if (out == MID_OUT_LDS) return f(MidC<CLS_C2C>{}, MidC<MID_IN_CPLX>{}, MidC<0>{}, MidC<0>{});
      if (out == MID_OUT_CPLX) return f(MidC<CLS_C2C>{}, MidC<MID_IN_CPLX>{}, MidC<MID_OUT_CPLX>{}, MidC<0>{});
      return f(MidC<CLS_C2C>{}, MidC<MID_IN_CPLX>{}, MidC<MID_OUT_RULE>{}, MidC<0>{});
    case CLS_R2C:
      if (in == MID_IN_LDS) return f(MidC<CLS_R2C>{}, MidC<0>{}, MidC<0>{}, MidC<0>{});
      return f(MidC<CLS_R2C>{}, MidC<MID_IN_PAIR>{}, MidC<0>{}, MidC<0>{});
    case CLS_C2R:
      if (out == MID_OUT_LDS) return f(MidC<CLS_C2R>{}, MidC<0>{}, MidC<0>{}, MidC<0>{});
      return f(MidC<CLS_C2R>{}, MidC<0>{}, MidC<MID_OUT_PAIR>{}, MidC<0>{});
    default: return f(MidC<CLS_R2R>{}, MidC<0>{}, MidC<0>{}, MidC<0>{});
  }
}

// Whole tile, any class and route (the host build).
template <typename T, int P, typename Run, typename Each>
P3E_HD P3E_INL void mid_tile(const PassArgs &p, uint32_t tile, cx<T> *buf, int nth, Run &run, Each &each,
                             const cx<T> *tw) {
  mid_dispatch<P>(p, [&](auto c, auto in, auto out, auto blue) {
    if constexpr (P <= 16) {
      if (p.mid_e == P3E_MID_FEW)
        return mid_tile_as<T, P, P3E_MID_FEW, c.v, in.v, out.v, blue.v>(p, tile, buf, nth, run, each, tw);
    }
    mid_tile_as<T, P, P3E_MID_MANY, c.v, in.v, out.v, blue.v>(p, tile, buf, nth, run, each, tw);
  });
}

}  // namespace p3e
