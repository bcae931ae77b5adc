// In-LDS FFTs of a length known at run time: Stockham autosort stages over V interleaved lines in a
// ping-pong pair of LDS buffers, with the radix of each stage (2..16) chosen on the host.  Each butterfly
// is transformed in registers, so a length costs one LDS round trip and one barrier per radix: 225 = 15 * 15
// takes two, 1000 = 10 * 10 * 10 three.  Forward only; an inverse transform swaps real and imaginary parts
// of its input and of its output (gx_swap).
//
// Position p of line v lives at slot i + i / 16, i = p V + v: the lanes of one position move V consecutive
// slots, and one slot of padding per 16 spreads strided accesses (the first stages' writes, walks along a
// line) over the banks.  (Slots p (V + 1) + v gave the same for 16 lines, but left a radix-8 stage of two
// lines on a quarter of the banks: 301-point rows, two at a time, 69 us against 39.)
#pragma once
#include "fft_core.hpp"
#include "gfft.hpp"

namespace tfsm {

// exp(-2 pi i m / N) tables for the fixed-size butterflies, from the Taylor series of cosine and sine
constexpr double gx_cosine(double x) {
  double t = 1.0, s = 1.0;
  for (int i = 1; i < 24; ++i) {
    t *= -x * x / ((2.0 * i - 1.0) * (2.0 * i));
    s += t;
  }
  return s;
}
constexpr double gx_sine(double x) {
  double t = x, s = x;
  for (int i = 1; i < 24; ++i) {
    t *= -x * x / ((2.0 * i) * (2.0 * i + 1.0));
    s += t;
  }
  return s;
}
// angle 2 pi m / N reduced to [-pi, pi]
constexpr double gx_angle(int m, int n) { return 6.283185307179586476925 * (2 * m > n ? m - n : m) / n; }
template <int N>
struct GxTable {
  float c[N], s[N];
  constexpr GxTable() : c(), s() {
    for (int m = 0; m < N; ++m) {
      c[m] = (float)gx_cosine(gx_angle(m, N));
      s[m] = (float)gx_sine(gx_angle(m, N));
    }
  }
};
template <int N>
struct GxRoots {
  static constexpr GxTable<N> T = GxTable<N>();
};

// odd prime radix from its definition, folded over the conjugate pairs (dft_odd in fft_core.hpp)
template <int R>
__device__ __forceinline__ void gx_odd(float2* x) {
  constexpr int H = (R - 1) / 2;
  float2 t[H + 1], d[H + 1];
  float2 s0 = x[0];
#pragma unroll
  for (int n = 1; n <= H; ++n) {
    t[n] = cadd(x[n], x[R - n]);
    d[n] = csub(x[n], x[R - n]);
    s0 = cadd(s0, t[n]);
  }
  float2 out[R];
  out[0] = s0;
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    float2 a = x[0], b = make_float2(0.f, 0.f);
#pragma unroll
    for (int n = 1; n <= H; ++n) {
      const float c = GxRoots<R>::T.c[(n * k) % R], sn = GxRoots<R>::T.s[(n * k) % R];
      a = make_float2(a.x + c * t[n].x, a.y + c * t[n].y);
      b = make_float2(b.x + sn * d[n].x, b.y + sn * d[n].y);
    }
    out[k] = make_float2(a.x + b.y, a.y - b.x);      // a - i b
    out[R - k] = make_float2(a.x - b.y, a.y + b.x);  // a + i b
  }
#pragma unroll
  for (int r = 0; r < R; ++r) x[r] = out[r];
}

template <int R>
__device__ __forceinline__ void gx_dft(float2* x);

// P * Q points: P-point transforms of the Q interleaved subsequences, twiddles, Q-point transforms
template <int P, int Q>
__device__ __forceinline__ void gx_comp(float2* x) {
  constexpr int N = P * Q;
  float2 y[Q][P];
#pragma unroll
  for (int b = 0; b < Q; ++b) {
#pragma unroll
    for (int a = 0; a < P; ++a) y[b][a] = x[Q * a + b];
    gx_dft<P>(y[b]);
#pragma unroll
    for (int k = 1; k < P; ++k) {
      if (b > 0) {
        const float c = GxRoots<N>::T.c[(b * k) % N], s = GxRoots<N>::T.s[(b * k) % N];
        const float2 z = y[b][k];
        y[b][k] = make_float2(z.x * c + z.y * s, z.y * c - z.x * s);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < P; ++k) {
    float2 z[Q];
#pragma unroll
    for (int b = 0; b < Q; ++b) z[b] = y[b][k];
    gx_dft<Q>(z);
#pragma unroll
    for (int m = 0; m < Q; ++m) x[k + P * m] = z[m];
  }
}

template <int R>
__device__ __forceinline__ void gx_dft(float2* x) {
  if constexpr (R == 6) gx_comp<2, 3>(x);
  else if constexpr (R == 9) gx_comp<3, 3>(x);
  else if constexpr (R == 10) gx_comp<2, 5>(x);
  else if constexpr (R == 12) gx_comp<4, 3>(x);
  else if constexpr (R == 15) gx_comp<3, 5>(x);
  else if constexpr (R == 11 || R == 13) gx_odd<R>(x);
  else dft<R, -1>(x);
}

#define GX_RADICES(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(15) X(16)

// layout of a workgroup's V interleaved lines: a power of two (GxLines) or any number (GxLinesN)
struct GxLines {
  int vl, V;
  __device__ __forceinline__ int slot(int p, int v) const {
    const int i = (p << vl) + v;
    return i + (i >> 4);
  }
  __device__ __forceinline__ int total(int n) const { return n << vl; }
  __device__ __forceinline__ void split(int i, int& b, int& v) const {
    v = i & (V - 1);
    b = i >> vl;
  }
};
struct GxLinesN {
  int V;
  unsigned mg;  // ceil(2^32 / V), V > 1
  __device__ __forceinline__ void set(int lines) {
    V = lines;
    mg = lines > 1 ? 0xffffffffu / (unsigned)lines + 1u : 0u;
  }
  __device__ __forceinline__ int slot(int p, int v) const {
    const int i = (int)__umul24(p, V) + v;
    return i + (i >> 4);
  }
  __device__ __forceinline__ int total(int n) const { return n * V; }
  __device__ __forceinline__ void split(int i, int& b, int& v) const {
    b = V > 1 ? (int)__umulhi((unsigned)i, mg) : i;
    v = i - (int)__umul24(b, V);
  }
};
// LDS slots of one buffer of V lines
__host__ __device__ inline int gx_slots(int L, int V) { return L * V + (L * V >> 4) + 1; }

template <int R, class LN>
__device__ __forceinline__ void gx_stage(const float2* src, float2* dst, const float2* tw, const GRadix& g, int s,
                                         const LN& ln, int tid, int nth) {
  const int nb = g.nb[s], Ns = g.ns[s], span = g.span[s], total = ln.total(nb);
  const unsigned mg = g.mg[s];
  for (int i = tid; i < total; i += nth) {
    int b, v;
    ln.split(i, b, v);
    float2 x[R];
#pragma unroll
    for (int q = 0; q < R; ++q) x[q] = src[ln.slot(b + q * nb, v)];
    int grp = b, k = 0;
    if (s > 0) {
      grp = (int)__umulhi((unsigned)b, mg);  // b / Ns
      k = b - grp * Ns;
      const int step = k * span;
#pragma unroll
      for (int q = 1; q < R; ++q) x[q] = cmul(x[q], tw[q * step]);
    }
    gx_dft<R>(x);
    const int d0 = grp * Ns * R + k;
#pragma unroll
    for (int q = 0; q < R; ++q) dst[ln.slot(d0 + q * Ns, v)] = x[q];
  }
  __syncthreads();
}

// every stage; the input is in `cur` (complete, behind a barrier), the result ends in `cur`
template <class LN>
__device__ __forceinline__ void gx_fft(const GRadix& g, const float2* tw, float2*& cur, float2*& alt, const LN& ln,
                                       int tid, int nth) {
#pragma unroll 1
  for (int s = 0; s < g.nr; ++s) {
    switch (g.r[s]) {
#define GX_CASE(R) \
  case R: gx_stage<R>(cur, alt, tw, g, s, ln, tid, nth); break;
      GX_RADICES(GX_CASE)
#undef GX_CASE
      default: break;
    }
    float2* t = cur;
    cur = alt;
    alt = t;
  }
}

__device__ __forceinline__ float2 gx_swap(float2 z) { return make_float2(z.y, z.x); }

}  // namespace tfsm
