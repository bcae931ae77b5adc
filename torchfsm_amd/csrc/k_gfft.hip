// General-length batched FFTs (declarations and conventions in gfft.hpp, the in-LDS stages in gx_core.hpp).
//
// One workgroup transforms V lines that are consecutive in the batch's fastest index (V a power of two, up to
// 16, so that two buffers of V lines fit LDS and the launch still fills the GPU).  The lines are gathered
// from their strided layout into LDS (real inputs promoted, Hermitian halves mirrored, Bluestein chirp
// applied), transformed, and scattered with the output's own index map (first n/2 + 1 values for R2C,
// real parts for C2R).  Threads walk the lines interleaved where adjacent lines are adjacent in memory
// (strided columns, four-step passes), one line after the other otherwise (rows), so that both coalesce; a
// run of lines that V does not divide ends in a partly filled workgroup.  Four-step and long Bluestein
// transforms chain these launches through a scratch buffer.
//
// Bound by latency and instruction issue, not bandwidth.  Forward transforms, us, before (radices 2..7, one
// element's load at a time, 16 adjacent lines or one) and now: 65536 points, B = 16 58 -> 27; 225 x 301,
// B = 16 65 -> 43; 1000^2, B = 4 94 -> 60; 120^3, B = 3 119 -> 90; 84 x 76 x 96, B = 3 69 -> 51.
#include <cmath>
#include <complex>
#include <vector>

#include "gfft.hpp"
#include "gx_core.hpp"

namespace tfsm {
namespace {

// One launch: line index = (o * n_i + i) * n_s + s.  Loaded element j of a line is logical input
// index q = j * qj + s * qs; stored element k is logical output index r = k * rk + s * rs.
struct GLaunch {
  GRadix g;
  int dir;               // sign of the exponent of the (first) FFT
  const float2* bmid;    // one-pass Bluestein: multiply by bmid, then the +1 FFT of the same length
  long long n_o, n_i, n_s;
  const void* in;
  long long ios, iis, ies, qj, qs;
  int in_mode;           // 0 complex, 1 real, 2 Hermitian half (hbins values of an nfull-point line)
  long long nload, nfull, hbins;
  const float2* pre;     // input multiplier per logical q (Bluestein chirp)
  void* out;
  long long oos, ois, oes, rk, rs;
  int out_mode;          // 0 complex, 1 real part
  long long nstore;      // logical outputs r < nstore are stored
  const float2* post;    // output multiplier per logical r (Bluestein chirp or kernel spectrum)
  long long twn;         // four-step twiddle exp(twdir 2 pi i k s / twn) (0: none)
  int twdir;
  const float2* twt;     // its table exp(-2 pi i t / twn), t < twn (null: computed in float64)
  float scale;
  // set by launch_g: V = 1 << vl lines per workgroup, consecutive in the fastest index with more than one
  // value (fd: 0 o, 1 i, 2 s); threads walk them interleaved on input / output where they are adjacent
  int vl, fd, ilv_in, ilv_out;
  unsigned mgL;          // ceil(2^32 / L)
  int twlds;             // the stage twiddles are staged in LDS
};

__device__ __forceinline__ float2 gmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ float2 gtw(const float2* tw, int t, int dir) {
  const float2 w = tw[t];
  return dir < 0 ? w : make_float2(w.x, -w.y);
}

__global__ void __launch_bounds__(1024) k_gfft(GLaunch a) {
  extern __shared__ float2 g_lds[];
  const int L = a.g.L, nth = blockDim.x, tid = threadIdx.x;
  GxLines ln;
  ln.vl = a.vl;
  ln.V = 1 << a.vl;
  const int slots = gx_slots(L, 1 << a.vl);
  float2* cur = g_lds;
  float2* alt = g_lds + slots;
  const float2* tw = a.g.tw;
  if (a.twlds) {
    float2* t = g_lds + 2 * slots;
    for (int i = tid; i < L; i += nth) t[i] = a.g.tw[i];
    tw = t;
  }
  // the workgroup's first line, and how many of its V lines exist
  const long long nf = a.fd == 0 ? a.n_o : (a.fd == 1 ? a.n_i : a.n_s);
  const long long groups = (nf + ln.V - 1) >> a.vl;
  const long long f0 = ((long long)blockIdx.x % groups) << a.vl, rest = (long long)blockIdx.x / groups;
  const int nv = (int)(nf - f0 < ln.V ? nf - f0 : ln.V);
  const long long o0 = a.fd == 0 ? f0 : (a.fd == 1 ? rest : rest / a.n_i);
  const long long i0 = a.fd == 0 ? 0 : (a.fd == 1 ? f0 : rest % a.n_i);
  const long long s0 = a.fd == 2 ? f0 : 0;
  const long long ib0 = o0 * a.ios + i0 * a.iis, ob0 = o0 * a.oos + i0 * a.ois;
  const long long dib = a.fd == 0 ? a.ios : (a.fd == 1 ? a.iis : 0), dob = a.fd == 0 ? a.oos : (a.fd == 1 ? a.ois : 0);
  const int ds = a.fd == 2 ? 1 : 0;
  const int total = L << a.vl;
  const bool inv = a.dir > 0;
  // loads in batches of GB per thread, issued before the first of them is used (one element at a time, a
  // workgroup paid a memory latency per element of its longest thread)
  constexpr int GB = 4;
  for (int e0 = tid; e0 < total; e0 += GB * nth) {
    float2 z[GB], c[GB];
    int vv[GB], jj[GB];
    bool ok[GB], cj[GB];
#pragma unroll
    for (int u = 0; u < GB; ++u) {
      const int e = e0 + u * nth;
      if (a.ilv_in) {
        vv[u] = e & (ln.V - 1);
        jj[u] = e >> a.vl;
      } else {
        vv[u] = (int)__umulhi((unsigned)e, a.mgL);
        jj[u] = e - vv[u] * L;
      }
      long long q = (long long)jj[u] * a.qj + (s0 + ds * vv[u]) * a.qs;
      ok[u] = e < total && vv[u] < nv && q < a.nload;
      if (!ok[u]) q = 0;
      const long long ib = ib0 + (ok[u] ? vv[u] : 0) * dib;
      cj[u] = a.in_mode == 2 && q >= a.hbins;
      const long long o = ib + (cj[u] ? a.nfull - q : q) * a.ies;
      if (a.in_mode == 1) z[u] = make_float2(((const float*)a.in)[o], 0.f);
      else z[u] = ((const float2*)a.in)[o];
      if (a.in_mode == 2 && (q == 0 || 2 * q == a.nfull)) z[u].y = 0.f;
      c[u] = a.pre ? a.pre[q] : make_float2(1.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < GB; ++u) {
      if (e0 + u * nth >= total) continue;
      float2 x = cj[u] ? make_float2(z[u].x, -z[u].y) : z[u];
      if (a.pre) x = gmul(x, c[u]);
      if (!ok[u]) x = make_float2(0.f, 0.f);
      cur[ln.slot(jj[u], vv[u])] = inv ? gx_swap(x) : x;
    }
  }
  __syncthreads();
  bool swapped = inv;
#pragma unroll 1
  for (int pass = 0;; ++pass) {
    gx_fft(a.g, tw, cur, alt, ln, tid, nth);
    if (!a.bmid || pass == 1) break;
    for (int e = tid; e < total; e += nth) {
      const int v = e & (ln.V - 1), k = e >> a.vl, sl = ln.slot(k, v);
      const float2 z = cur[sl];
      cur[sl] = gx_swap(gmul(swapped ? gx_swap(z) : z, a.bmid[k]));
    }
    swapped = true;
    __syncthreads();
  }
  for (int e = tid; e < total; e += nth) {
    int v, k;
    if (a.ilv_out) {
      v = e & (ln.V - 1);
      k = e >> a.vl;
    } else {
      v = (int)__umulhi((unsigned)e, a.mgL);
      k = e - v * L;
    }
    const long long s = s0 + ds * v, r = (long long)k * a.rk + s * a.rs;
    if (v >= nv || r >= a.nstore) continue;
    float2 z = cur[ln.slot(k, v)];
    if (swapped) z = gx_swap(z);
    if (a.twn) {
      long long t = (long long)k * s;  // k < L1, s < L2: below twn = L1 L2
      if (t >= a.twn) t %= a.twn;
      if (a.twt) {
        z = gmul(z, gtw(a.twt, (int)t, a.twdir));
      } else {
        double sn, cs;
        sincos((double)a.twdir * 2.0 * M_PI * (double)t / (double)a.twn, &sn, &cs);
        z = gmul(z, make_float2((float)cs, (float)sn));
      }
    }
    if (a.post) z = gmul(z, a.post[r]);
    z.x *= a.scale;
    z.y *= a.scale;
    const long long ob = ob0 + v * dob;
    if (a.out_mode == 1)
      ((float*)a.out)[ob + r * a.oes] = z.x;
    else
      ((float2*)a.out)[ob + r * a.oes] = z;
  }
}

constexpr size_t GX_LDS_BYTES = 150 * 1024;  // of 160 KB
constexpr size_t GX_LDS_PAIR = 80 * 1024;    // two workgroups per CU

hipError_t launch_g(GLaunch a, hipStream_t st) {
  const long long nlines = a.n_o * a.n_i * a.n_s;
  if (nlines <= 0) return hipSuccess;
  a.fd = a.n_s > 1 ? 2 : (a.n_i > 1 ? 1 : 0);
  const long long nf = a.fd == 0 ? a.n_o : (a.fd == 1 ? a.n_i : a.n_s), outer = nlines / nf;
  const long long din = a.fd == 2 ? a.qs * a.ies : (a.fd == 1 ? a.iis : a.ios);
  const long long dout = a.fd == 2 ? a.rs * a.oes : (a.fd == 1 ? a.ois : a.oos);
  const bool adj = din == 1 || dout == 1;
  // lines per workgroup: about 4096 points, 16 lines at most, and two workgroups per CU (2048 points two lines at a
  // time, one workgroup per CU: 1015 points B = 2048 155 us there and back, 112 one line at a time); fewer while the
  // launch has under two workgroups per CU (but 8 where adjacent lines share cache lines)
  auto lds_of = [&](int v, bool tables) {
    return (2 * (size_t)gx_slots(a.g.L, 1 << v) + (tables ? a.g.L : 0)) * sizeof(float2);
  };
  int vl = 0;
  while (a.g.L > 1 && vl < 4 && ((long long)a.g.L << (vl + 1)) <= GFFT_LDS_MAX && (1 << vl) < nf &&
         lds_of(vl + 1, true) <= GX_LDS_PAIR)
    ++vl;
  const int least = adj ? 3 : 0;
  while (vl > least && outer * ((nf + (1 << vl) - 1) >> vl) < 512) --vl;
  a.vl = vl;
  a.ilv_in = vl && din == 1;
  a.ilv_out = vl && dout == 1;
  a.mgL = (unsigned)((0x100000000ULL + a.g.L - 1) / a.g.L);
  const long long blocks = outer * ((nf + (1 << vl) - 1) >> vl);
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  a.twlds = lds_of(vl, true) <= (blocks > 256 ? GX_LDS_PAIR : GX_LDS_BYTES) ? 1 : 0;
  const size_t lds = lds_of(vl, a.twlds);
  // one butterfly of about 4 values per thread, so that a stage is one round of butterflies (with 8 values radices 4
  // to 6 took two: 500^2 B = 1 there and back 52 us against 42, 57 x 246 57 against 43, 1D 496 points B = 64 35 against
  // 29), of 2 where a CU has one workgroup at most (unfused KSConvection 1000 points 117 us per step against 112), and
  // 1024 threads only there (505 x 576 B = 1 55 us against 61; B = 32 the reverse, 1.07)
  const long long most = blocks > 256 ? 512 : 1024;
  long long nth = ((((long long)a.g.L << vl) / (blocks > 256 ? 4 : 2) + 63) / 64) * 64;
  nth = nth < 64 ? 64 : (nth > most ? most : nth);
  hipLaunchKernelGGL(k_gfft, dim3((unsigned)blocks), dim3((unsigned)nth), lds, st, a);
  return hipGetLastError();
}

// (`extra` per stage: Bluestein's sequences take fewer, longer stages, 400 more each: two transforms and the chirps
// between them make a stage dearer there.  Vorticity 993 x 64 B = 1 SETDRK4 2606 us for 8 steps against 2350, 1D Burgers
// 767 points 709 against 650, conv 787 x 96 3302 against 2934; errors within 1 %.)
// The cheapest radix sequence by the time of one butterfly per thread, in cycles: a stage's barrier and LDS
// latency, plus its LDS traffic, twiddles and index arithmetic (64 per value) and its arithmetic.  The
// launches that matter are latency bound, so a few stages of radix 4 to 9 beat fewer of radix 15 and 16.
constexpr int kRadices[] = {2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 15, 16};
constexpr int kStageCost[] = {670, 760, 820, 1020, 1110, 1350, 1270, 1550, 1720, 2100, 1850, 2500, 2560, 2300};
void plan_radices(int n, int i, int cost, int extra, std::vector<int>& now, std::vector<int>& best, int& bestc) {
  if (!best.empty() && cost >= bestc) return;
  if (n == 1) {
    best = now;
    bestc = cost;
    return;
  }
  for (int k = i; k >= 0; --k)
    if (n % kRadices[k] == 0) {
      now.push_back(kRadices[k]);
      plan_radices(n / kRadices[k], k, cost + kStageCost[k] + extra, extra, now, best, bestc);
      now.pop_back();
    }
}

bool radices(int L, GRadix& g, int extra) {
  g = GRadix();
  g.L = L;
  std::vector<int> now, best;
  if (L > 1) {
    int bestc = 0;
    plan_radices(L, (int)(sizeof(kRadices) / sizeof(int)) - 1, 0, extra, now, best, bestc);
    if (best.empty() || (int)best.size() > GFFT_MAX_RADICES) return false;
  }
  int ns = 1;
  for (int r : best) {
    const int s = g.nr++;
    g.r[s] = r;
    g.ns[s] = ns;
    g.nb[s] = L / r;
    g.span[s] = L / (ns * r);
    g.mg[s] = ns > 1 ? (unsigned)((0x100000000ULL + ns - 1) / ns) : 0;
    ns *= r;
  }
  return true;
}

// L = L1 L2 with both at most GFFT_LDS_MAX, as square as possible (0: none).  Pass A's lines are strided by
// L2 and gathered up to 16 adjacent ones at a time: a long L1 would leave LDS for one line only
// (65536 points at 4096 * 16 and radices up to 7 57 us, at 256 * 256 30)
int split_four(int L) {
  for (int l1 = (int)std::ceil(std::sqrt((double)L)); l1 <= GFFT_LDS_MAX; ++l1)
    if (L % l1 == 0) return l1;
  return 0;
}

// circular length M >= 2n - 1 that one workgroup holds (0: none): the smallest of 2^a, 5 2^a and 15 2^a.  The last
// transform spreads the rounding errors of both over M points, of which n are kept, and the twiddle tables' own
// errors add up most where every radix is a power of two.  22 lengths from 53 to 1017, rms error against 64 bits (forward
// transform of white noise; diffusion; vorticity and velocity steps; pressure), powers of two / these / the shortest
// lengths with factors up to 13: 1.44 / 1.54 / 1.61e-7; 2.69 / 2.68 / 2.80e-7; 3.69 / 3.54 / 3.66e-7; 3.18 / 2.94 / 3.11e-7;
// 5.99 / 4.01 / 4.22e-7.  SETDRK4 step, us: vorticity 225 x 301 B = 8 991 / 850 / 855, 97^2 B = 8 319 / 313 / 317; 1D Burgers
// 767 points 71 / 71 / 69.
int bluestein_length(int n) {
  int best = 0;
  for (int f : {1, 5, 15})
    for (int m = f; m <= GFFT_LDS_MAX; m *= 2)
      if (m >= 2 * n - 1 && (!best || m < best)) best = m;
  return best;
}

hipError_t upload(const std::vector<float2>& h, const float2** out, std::vector<void*>& allocs) {
  void* d = nullptr;
  hipError_t e = hipMalloc(&d, h.size() * sizeof(float2));
  if (e != hipSuccess) return e;
  allocs.push_back(d);
  e = hipMemcpy(d, h.data(), h.size() * sizeof(float2), hipMemcpyHostToDevice);
  *out = (const float2*)d;
  return e;
}

hipError_t build_radix(GRadix& g, int L, std::vector<void*>& allocs, int extra = 0) {
  if (!radices(L, g, extra)) return hipErrorInvalidValue;
  std::vector<float2> h(L);
  for (int t = 0; t < L; ++t) {
    const double ang = -2.0 * M_PI * (double)t / (double)L;
    h[t] = make_float2((float)std::cos(ang), (float)std::sin(ang));
  }
  return upload(h, &g.tw, allocs);
}

// FFT in double (host), exponent sign -1, any smooth length, decimation in time by the smallest factor:
// x[i * step], i < n, into out[0..n); w: the roots of unity of the whole length, n * wstep of them
void host_fft(const std::complex<double>* x, size_t n, size_t step, std::complex<double>* out,
              const std::vector<std::complex<double>>& w, size_t wstep) {
  if (n == 1) {
    out[0] = x[0];
    return;
  }
  size_t p = 2;
  while (n % p) ++p;
  const size_t m = n / p;
  for (size_t q = 0; q < p; ++q) host_fft(x + q * step, m, step * p, out + q * m, w, wstep * p);
  std::complex<double> t[16];
  for (size_t k = 0; k < m; ++k) {
    for (size_t q = 0; q < p; ++q) t[q] = out[q * m + k];
    for (size_t h = 0; h < p; ++h) {
      const size_t f = k + h * m;
      std::complex<double> acc = t[0];
      for (size_t q = 1; q < p; ++q) acc += w[(q * f % n) * wstep] * t[q];
      out[f] = acc;
    }
  }
}

}  // namespace

bool gfft_smooth(int n) {
  if (n < 1) return false;
  for (int r : {2, 3, 5, 7, 11, 13})
    while (n % r == 0) n /= r;
  return n == 1;
}

hipError_t gaxis_build(GAxis& a, int n, std::vector<void*>& allocs) {
  if (n < 1) return hipErrorInvalidValue;
  a = GAxis();
  a.n = n;
  if (gfft_smooth(n) && (n <= GFFT_LDS_MAX || split_four(n))) {
    a.L = n;
  } else {
    long long m = bluestein_length(n);
    if (!m) {
      m = 1;
      while (m < 2LL * n - 1) m <<= 1;
    }
    if (m > (long long)GFFT_LDS_MAX * GFFT_LDS_MAX) return hipErrorInvalidValue;
    a.blu = true;
    a.L = (int)m;
  }
  hipError_t e;
  if (a.L <= GFFT_LDS_MAX) {
    e = build_radix(a.g, a.L, allocs, a.blu ? 400 : 0);
  } else {
    a.four = true;
    const int l1 = split_four(a.L);
    if (!l1) return hipErrorInvalidValue;
    e = build_radix(a.g1, l1, allocs);
    if (e == hipSuccess) e = build_radix(a.g2, a.L / l1, allocs);
    if (e == hipSuccess) {
      // the L-point twiddle table of the four-step (float32 of float64 values, 8 L bytes)
      std::vector<float2> h(a.L);
      for (int t = 0; t < a.L; ++t) {
        const double ang = -2.0 * M_PI * (double)t / (double)a.L;
        h[t] = make_float2((float)std::cos(ang), (float)std::sin(ang));
      }
      e = upload(h, &a.tw4, allocs);
    }
  }
  if (e != hipSuccess || !a.blu) return e;
  // chirp c_d[t] = exp(-/+ i pi (t^2 mod 2n) / n); kernel b[m] = conj(c_d[|m|]) for |m| < n on the
  // circle of M points; bhat = FFT_M(b) / M
  const int M = a.L;
  std::vector<std::complex<double>> c(n), b(M, 0.0), bf(M), w(M);
  for (int t = 0; t < n; ++t) {
    const long long q = ((long long)t * t) % (2LL * n);
    c[t] = std::polar(1.0, -M_PI * (double)q / (double)n);
    b[t] = std::conj(c[t]);
    if (t > 0) b[M - t] = b[t];
  }
  for (int t = 0; t < M; ++t) w[t] = std::polar(1.0, -2.0 * M_PI * (double)t / (double)M);
  host_fft(b.data(), M, 1, bf.data(), w, 1);
  // the inverse direction's chirp and kernel are the conjugates, and as the kernel is even so is its spectrum
  for (int d = 0; d < 2; ++d) {
    const double sg = d == 0 ? 1.0 : -1.0;
    std::vector<float2> ch(n), bh(M);
    for (int t = 0; t < n; ++t) ch[t] = make_float2((float)c[t].real(), (float)(sg * c[t].imag()));
    for (int k = 0; k < M; ++k) bh[k] = make_float2((float)(bf[k].real() / M), (float)(sg * bf[k].imag() / M));
    e = upload(ch, &a.chirp[d], allocs);
    if (e == hipSuccess) e = upload(bh, &a.bhat[d], allocs);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

size_t gfft_tmp_elems(const GAxis& a, size_t lines) { return a.four ? 2 * lines * (size_t)a.L : 0; }

hipError_t gfft_run(const GAxis& a, int mode, int dir, const void* in, const GLines& li, void* out, const GLines& lo,
                    float scale, float2* tmp, hipStream_t st) {
  if (a.n < 1 || (dir != -1 && dir != 1)) return hipErrorInvalidValue;
  if (li.n_o != lo.n_o || li.n_i != lo.n_i) return hipErrorInvalidValue;
  const int d = dir < 0 ? 0 : 1;
  const long long n = a.n, H = n / 2 + 1;
  GLaunch base{};
  base.n_o = (long long)li.n_o;
  base.n_i = (long long)li.n_i;
  base.n_s = 1;
  base.in = in;
  base.ios = (long long)li.os;
  base.iis = (long long)li.is;
  base.ies = (long long)li.es;
  base.qj = 1;
  base.qs = 0;
  base.in_mode = mode == GM_R2C ? 1 : (mode == GM_C2R ? 2 : 0);
  base.nload = n;
  base.nfull = n;
  base.hbins = H;
  base.pre = a.blu ? a.chirp[d] : nullptr;
  base.out = out;
  base.oos = (long long)lo.os;
  base.ois = (long long)lo.is;
  base.oes = (long long)lo.es;
  base.rk = 1;
  base.rs = 0;
  base.out_mode = mode == GM_C2R ? 1 : 0;
  base.nstore = mode == GM_R2C ? H : n;
  base.post = a.blu ? a.chirp[d] : nullptr;
  base.scale = scale;
  if (!a.four) {
    GLaunch x = base;
    x.g = a.g;
    x.dir = a.blu ? -1 : dir;
    x.bmid = a.blu ? a.bhat[d] : nullptr;
    return launch_g(x, st);
  }
  if (!tmp) return hipErrorInvalidValue;
  const long long L = a.L, L1 = a.g1.L, L2 = a.g2.L;
  const long long lines = base.n_o * base.n_i;
  float2* t1 = tmp;
  float2* t2 = tmp + (size_t)lines * L;
  // pass A: L1-point FFTs over j1 of x[j1 L2 + j2], twiddled by w_L^(k1 j2), into t1[line][k1 L2 + j2]
  GLaunch A = base;
  A.g = a.g1;
  A.dir = a.blu ? -1 : dir;
  A.n_s = L2;
  A.qj = L2;
  A.qs = 1;
  A.out = t1;
  A.oos = base.n_i * L;
  A.ois = L;
  A.oes = 1;
  A.rk = L2;
  A.rs = 1;
  A.out_mode = 0;
  A.nstore = L;
  A.post = nullptr;
  A.twn = L;
  A.twdir = A.dir;
  A.twt = a.tw4;
  A.scale = 1.0f;
  // pass B: L2-point FFTs over j2 of t1[k1 L2 + j2]; result X[k1 + L1 k2]
  GLaunch B = base;
  B.g = a.g2;
  B.dir = A.dir;
  B.n_s = L1;
  B.in = t1;
  B.ios = base.n_i * L;
  B.iis = L;
  B.ies = 1;
  B.qj = 1;
  B.qs = L2;
  B.in_mode = 0;
  B.nload = L;
  B.pre = nullptr;
  B.rk = L1;
  B.rs = 1;
  hipError_t e = launch_g(A, st);
  if (e != hipSuccess) return e;
  if (!a.blu) return launch_g(B, st);
  // Bluestein: X * bhat into t2 (natural order), then the inverse four-step into the output
  GLaunch B1 = B;
  B1.out = t2;
  B1.oos = base.n_i * L;
  B1.ois = L;
  B1.oes = 1;
  B1.out_mode = 0;
  B1.nstore = L;
  B1.post = a.bhat[d];
  B1.scale = 1.0f;
  e = launch_g(B1, st);
  if (e != hipSuccess) return e;
  GLaunch C = A;
  C.dir = +1;
  C.twdir = +1;
  C.in = t2;
  C.ios = base.n_i * L;
  C.iis = L;
  C.ies = 1;
  C.in_mode = 0;
  C.nload = L;
  C.pre = nullptr;
  e = launch_g(C, st);
  if (e != hipSuccess) return e;
  GLaunch D = B;
  D.dir = +1;
  return launch_g(D, st);
}

}  // namespace tfsm
