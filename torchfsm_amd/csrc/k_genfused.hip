// Fused evaluation and stepping on meshes of any size (run-time FFT lengths, gx_core.hpp), where an axis has
// no fixed-size kernel:
//   k_g2row, k_g2col  the row and column pass of k_step2d.hpp (same layouts of P and G, so either may be
//                     the fixed-size kernel of its axis), for VorticityConvection, Convection,
//                     NSPressureConvection and KSConvection
//   k_g1run           the persistent 1D stepper (k1_run): one workgroup per sample runs every step, the
//                     spectrum of the current stage in LDS
// An evaluation of the unfused path is seven launches that each move every field (2D), and each of them was
// as long as its chain of dependent loads; here it is two (2D) or none (1D, one launch per call).
//
// Bound by latency: a launch is about one round of workgroups, as long as one workgroup's chain of loads
// and FFT stages.  So loads are issued in batches ahead of their use, a stage is a butterfly of a
// few values per thread, a pass transforms several fields of its lines at once where LDS holds them, and the
// workgroups are kept small enough to fill the GPU.
// SETDRK4 step, us, on the unfused path and here: vorticity 225 x 301 B = 1 275 / 135, B = 4 421 / 224, B = 32
// 1330 / 937; 768^2 B = 4 755 / 585; 60 x 72 B = 64 319 / 117; Burgers 150^2 B = 8 328 / 133; NSP 172^2 B = 1
// 284 / 167; 1D Burgers 1000 B = 1 102 / 34, 767 B = 15 160 / 64, 3000 B = 8 161 / 48.  With one field at a time
// in its workgroup columns of 225 x 301 B = 4 took 32 us against 21, a step of 172^2 B = 1 350 against 185.
#include "engine.hpp"
#include "gx_core.hpp"
#include "k_step2d.hpp"

namespace tfsm {
namespace {

// one axis of run-time length in a kernel: Bluestein axes carry chirp and kernel spectrum
struct GxDev {
  GRadix g;
  int n = 0;
  const float2* chirp = nullptr;  // [n] (null: plain length L = n)
  const float2* bhat = nullptr;   // [L]
  int V = 1;                      // columns or rows per workgroup
  int fg = 1;                     // fields (or channels) transformed together: up to V * fg lines in LDS
  unsigned mgn = 0;               // ceil(2^32 / n)
};

// LDS state of a workgroup's transforms.  put() and get() take the logical points p < n of line v; inverse
// transforms swap real and imaginary parts on both sides, Bluestein's chirps are applied here too.
// TL: twiddles, chirp and kernel spectrum are staged in LDS (from global memory, each read in the element
// loops is a memory latency: 225 x 301, B = 4, one field at a time, columns 42 us against 32)
template <bool TL>
struct GxWork {
  const GxDev& ax;
  GxLinesN ln;
  float2 *cur, *alt, *end;
  const float2 *tw, *chirp, *bhat;
  int tid, nth;
  __device__ __forceinline__ GxWork(const GxDev& a, float2* lds) : ax(a), tid(threadIdx.x), nth(blockDim.x) {
    const int slots = gx_slots(a.g.L, a.V * a.fg);
    ln.set(a.V);
    cur = lds;
    alt = lds + slots;
    end = lds + 2 * slots;
    tw = a.g.tw;
    chirp = a.chirp;
    bhat = a.bhat;
    if constexpr (TL) {
      float2* t = end;
      for (int i = tid; i < a.g.L; i += nth) t[i] = a.g.tw[i];
      tw = t;
      end += a.g.L;
      if (a.chirp) {
        float2 *c = end, *h = end + a.n;
        for (int i = tid; i < a.n; i += nth) c[i] = a.chirp[i];
        for (int i = tid; i < a.g.L; i += nth) h[i] = a.bhat[i];
        chirp = c;
        bhat = h;
        end += a.n + a.g.L;
        __syncthreads();
      }
    }
  }
  // first LDS slot after the buffers and tables
  __device__ __forceinline__ float2* rest() const { return end; }
  // start a group of `lines` lines: put() then writes the buffer that get() of the last group does not read
  __device__ __forceinline__ void begin(int lines) {
    next.set(lines);
  }
  GxLinesN next;
  __device__ __forceinline__ void put(int p, int v, float2 z, bool inv) {
    if (inv) z = gx_swap(z);
    if (ax.chirp) z = cmul(z, chirp[p]);
    alt[next.slot(p, v)] = z;
  }
  __device__ __forceinline__ float2 get(int p, int v, bool inv) const {
    float2 z = cur[ln.slot(p, v)];
    if (ax.chirp) z = cmul(gx_swap(z), chirp[p]);
    return inv ? gx_swap(z) : z;
  }
  // the transforms of what put() wrote (with barriers on both sides)
  __device__ __forceinline__ void run() {
    float2* t = cur;
    cur = alt;
    alt = t;
    ln = next;
    if (ax.chirp)
      for (int e = tid; e < ln.total(ax.g.L - ax.n); e += nth) {
        int p, v;
        ln.split(e, p, v);
        cur[ln.slot(ax.n + p, v)] = make_float2(0.f, 0.f);
      }
    __syncthreads();
#pragma unroll 1
    for (int pass = 0;; ++pass) {
      gx_fft(ax.g, tw, cur, alt, ln, tid, nth);
      if (!ax.chirp || pass == 1) break;
      for (int e = tid; e < ln.total(ax.g.L); e += nth) {
        int k, v;
        ln.split(e, k, v);
        const int sl = ln.slot(k, v);
        cur[sl] = gx_swap(cmul(cur[sl], bhat[k]));
      }
      __syncthreads();
    }
  }
};

constexpr int GU = 4;  // elements per thread whose loads are in flight together

// ---------------------------------------------------------------- 2D columns
// Layouts and arithmetic of col2_tile (k_step2d.hpp).  s holds the NC spectra of the tile: the products'
// transforms, then the combined stage spectra; element e = p V + v belongs to thread e % nth throughout.
// Channels, then fields, are transformed in groups of up to fg (their lines side by side in LDS).
template <int TERM, bool TL>
__global__ void __launch_bounds__(1024) k_g2col(Col2Args a, GxDev ax, int stage) {
  constexpr int NC = Term2<TERM>::NC, NF = Term2<TERM>::NF;
  extern __shared__ float2 g_lds[];
  GxWork<TL> w(ax, g_lds);
  const int V = ax.V, N0 = ax.n, E = N0 * V;
  float2* s = w.rest();  // [NC][E]
  float* s_ax = reinterpret_cast<float*>(s + NC * E);  // [N0] x wavenumbers
  for (int i = threadIdx.x; i < N0; i += blockDim.x) s_ax[i] = a.ax[i];
  __syncthreads();
  GxLinesN ev;  // elements: (point, column)
  ev.set(V);
  const int ntiles = (a.H1 + V - 1) / V;
  const int tile = blockIdx.x % ntiles, b = a.b0 + blockIdx.x / ntiles;
  if (a.mask.skip(b)) return;
  const size_t plane = (size_t)N0 * a.P1;
  const int c0 = tile * V;
  const int tid = w.tid, nth = w.nth;
  // element -> point p, column v of the tile and ky (clamped to the last one); its offset within a channel
  auto at = [&](int e, int& p, int& v, int& ky) {
    ev.split(e, p, v);
    ky = c0 + v < a.H1 ? c0 + v : a.H1 - 1;
    return (unsigned)p * a.P1 + ky;
  };
  const int nfwd = stage == ST_PRO ? 0 : NC;
  if (stage == ST_PRO) {
#pragma unroll 1
    for (int c = 0; c < NC; ++c)
      for (int e0 = tid; e0 < E; e0 += GU * nth) {
        float2 z[GU];
#pragma unroll
        for (int u = 0; u < GU; ++u) {
          const int e = e0 + u * nth < E ? e0 + u * nth : e0;
          int p, v, ky;
          z[u] = a.U[((size_t)b * NC + c) * plane + at(e, p, v, ky)];
        }
#pragma unroll
        for (int u = 0; u < GU; ++u)
          if (e0 + u * nth < E) s[c * E + e0 + u * nth] = z[u];
      }
  }
  const bool fields = c0 <= a.kmax1;  // uniform: the tile has kept columns
  const int nt = nfwd + (fields && stage != ST_EVAL ? NF : 0);
#pragma unroll 1
  for (int t = 0; t < nt;) {
    const bool inv = t >= nfwd;
    const int lim = inv ? nt : nfwd, cnt = lim - t < ax.fg ? lim - t : ax.fg;
    w.begin(cnt * V);
    if (!inv) {
#pragma unroll 1
      for (int i = 0; i < cnt; ++i) {
        const float2* P = a.P + ((size_t)b * NC + t + i) * plane;
        for (int e0 = tid; e0 < E; e0 += GU * nth) {
          float2 z[GU];
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            const int e = e0 + u * nth < E ? e0 + u * nth : e0;
            int p, v, ky;
            z[u] = P[at(e, p, v, ky)];
          }
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            const int e = e0 + u * nth;
            if (e >= E) continue;
            int p, v;
            ev.split(e, p, v);
            w.put(p, i * V + v, z[u], false);
          }
        }
      }
    } else {
      const int f0 = t - nfwd;
      for (int e = tid; e < E; e += nth) {
        int x, v, kyl;
        at(e, x, v, kyl);
        const int ky = c0 + v, ks = x <= N0 / 2 ? x : N0 - x;
        const bool keep = ky <= a.kmax1 && ks <= a.kmax0;
        const float axv = s_ax[x];
        float2 z[NC], psi = make_float2(0.f, 0.f);
#pragma unroll
        for (int c = 0; c < NC; ++c) z[c] = s[c * E + e];
        if (TERM == TERM_VC && keep) {
          const float ay = a.ay[ky];
          const float lap = addr(-mulr(axv, axv), -mulr(ay, ay));
          const float il = (lap == 0.f) ? 1.0f : __fdiv_rn(1.0f, lap);
          psi = make_float2(mulr(-z[0].x, il), mulr(-z[0].y, il));
        }
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          if (f < f0 || f >= f0 + cnt) continue;
          float2 val = make_float2(0.f, 0.f);
          if (keep) {
            const bool dx = TERM == TERM_VC ? (f == 1 || f == 2) : (f & 1);  // the field times a_x
            val = TERM == TERM_VC ? (f < 2 ? psi : z[0]) : z[NC > 1 ? f >> 1 : 0];
            if (dx) val = make_float2(mulr(axv, val.x), mulr(axv, val.y));
            val = make_float2(val.x * a.scale, val.y * a.scale);
          }
          w.put(x, (f - f0) * V + v, val, true);
        }
      }
    }
    w.run();
    if (inv) {
      const int f0 = t - nfwd;
      for (int e = tid; e < E; e += nth) {
        int x, v;
        ev.split(e, x, v);
        if (c0 + v > a.kmax1) continue;
        float2* G = a.G + (((size_t)b * NF + f0) * N0 + x) * a.PF + c0 + v;
#pragma unroll 1
        for (int i = 0; i < cnt; ++i) G[(size_t)i * N0 * a.PF] = w.get(x, i * V + v, true);
      }
      t += cnt;
      continue;
    }
    for (int e = tid; e < E; e += nth) {
      int x, v;
      ev.split(e, x, v);
#pragma unroll 1
      for (int i = 0; i < cnt; ++i) {
        float2 z = w.get(x, i * V + v, false);
        // remove_mean: fft(p - mean(p)) differs from fft(p) only at k = 0, by the batch mean of the DC
        if constexpr (TERM == TERM_KS) {
          if (a.dc && e == 0 && c0 == 0) z = rsub(z, a.dc[0]);
        }
        s[(t + i) * E + e] = z;
      }
    }
    t += cnt;
    if (t < nfwd) continue;
    if constexpr (TERM == TERM_NSP) {
      for (int e = tid; e < E; e += nth) {
        int x, v, ky;
        at(e, x, v, ky);
        float2 cv[2] = {s[e], s[E + e]};
        const float av[2] = {s_ax[x], a.ay[ky]};
        const bool nyx = 2 * x == N0, nyy = 2 * ky == a.N1, own = (x == 0 || nyx) && (ky == 0 || nyy);
        const bool ny[2] = {nyx && !own, nyy && !own};
        nsp_project<2>(cv, av, ny);
        s[e] = cv[0];
        s[E + e] = cv[1];
      }
    }
    const bool rdu = stage_reads_u(stage), rd1 = stage_reads_a1(stage), rd2 = stage_reads_a2(stage);
    const bool rd5 = stage == ST_R4_E2;
    const int tgt = stage_target(stage), h16 = stage_coef_half(stage) << 4;
    const float4* cpk = a.cpk + (size_t)b * a.cpk_bstride;
    const float* c5t = a.c5t + (size_t)b * (a.cpk_bstride / 2);
#pragma unroll 1
    for (int c = 0; c < NC; ++c) {
      const size_t base = ((size_t)b * NC + c) * plane;
      const float2* U = a.U + base;
      const float2* A1 = a.A1 + base;
      const float2* A2 = a.A2 + base;
      float2* dst = (tgt == 0 ? a.U : (tgt == 1 ? a.A1 : a.A2)) + base;
      const float2* src = a.src ? a.src + (size_t)b * a.src_bstride + (size_t)c * a.src_cstride : nullptr;
      for (int e0 = tid; e0 < E; e0 += GU * nth) {
        float2 uu[GU], q1[GU], q2[GU], sv[GU];
        float4 cc[GU];
        float c5[GU];
        unsigned o[GU];
#pragma unroll
        for (int u = 0; u < GU; ++u) {
          const int e = e0 + u * nth < E ? e0 + u * nth : e0;
          int x, v, ky;
          o[u] = at(e, x, v, ky);
          cc[u] = cpk[2 * o[u] - (o[u] & 15) + h16];
          uu[u] = q1[u] = q2[u] = sv[u] = make_float2(0.f, 0.f);
          c5[u] = 0.f;
        }
#pragma unroll
        for (int u = 0; u < GU; ++u) {
          if (rdu) uu[u] = U[o[u]];
          if (rd1) q1[u] = A1[o[u]];
          if (rd2) q2[u] = A2[o[u]];
          if (src) sv[u] = src[o[u]];
          if (rd5) c5[u] = c5t[o[u]];
        }
#pragma unroll
        for (int u = 0; u < GU; ++u) {
          const int e = e0 + u * nth;
          if (e >= E) continue;
          int x, v;
          ev.split(e, x, v);
          float2 nv = rscale(a.coef_t, s[c * E + e]);
          if (src) nv = radd(nv, sv[u]);
          float2 st;
          s[c * E + e] = stage_combine_v(stage, nv, uu[u], q1[u], q2[u], cc[u], c5[u], &st);
          if (c0 + v < a.H1) dst[o[u]] = st;
        }
      }
    }
  }
}

// ---------------------------------------------------------------- 2D rows
// Layouts and arithmetic of row2_body (k_step2d.hpp); V rows of a.B samples * N0 per workgroup.
template <int TERM, bool TL>
__global__ void __launch_bounds__(1024) k_g2row(Row2Args a, GxDev ax) {
  constexpr int NF = Term2<TERM>::NF;
  constexpr int NI = TERM == TERM_CONV ? 3 : (TERM == TERM_VC ? 2 : 1);  // packed inverse transforms
  constexpr int NP = TERM == TERM_CONV ? 2 : 1;
  extern __shared__ float2 g_lds[];
  __shared__ int s_row[16];  // row of each line in [samples][N0], or -1
  GxWork<TL> w(ax, g_lds);
  const int V = ax.V, n = ax.n, E = n * V, tid = w.tid, nth = w.nth;
  float2* zs = w.rest();                  // [E] the first pair of fields
  float2* ps = NI > 1 ? zs + E : zs;      // [E] the real products
  if (tid < V) {
    const int r = blockIdx.x * V + tid;
    int row = -1;
    if (r < a.B * a.N0) {
      const int b = a.b0 + r / a.N0;
      if (!a.mask.skip(b)) row = b * a.N0 + r % a.N0;
    }
    s_row[tid] = row;
  }
  __syncthreads();
  const size_t fs = (size_t)a.N0 * a.PF;
  // element e = v n + p: threads walk along the rows
  auto at = [&](int e, int& v, int& p) {
    v = (int)__umulhi((unsigned)e, ax.mgn);
    p = e - v * n;
  };
#pragma unroll 1
  for (int h0 = 0; h0 <= NI;) {
    const bool inv = h0 < NI;
    const int cnt = inv ? (NI - h0 < ax.fg ? NI - h0 : ax.fg) : 1;
    w.begin(cnt * V);
    if (inv) {
#pragma unroll 1
      for (int i = 0; i < cnt; ++i) {
        const int h = h0 + i;
        // the two half-transformed fields packed into one complex inverse transform, and what multiplies
        // them: 0: 1, 1: i, 2: i a_y, 3: -i
        int fa, fb, ma, mb;
        if constexpr (TERM == TERM_VC) {
          fa = h == 0 ? 0 : 2;   // u_x = C2R(i a_y psi), u_y = C2R(-i kx psi); w_x = C2R(i kx w), w_y = C2R(i a_y w)
          fb = h == 0 ? 1 : 3;
          ma = h == 0 ? 2 : 1;
          mb = h == 0 ? 3 : 2;
        } else if constexpr (TERM == TERM_KS) {
          fa = 1;                // d_x phi, d_y phi
          fb = 0;
          ma = 1;
          mb = 2;
        } else {
          fa = h == 0 ? 0 : (h == 1 ? 1 : 3);  // (u0, u1), (d_x u0, d_y u0), (d_x u1, d_y u1)
          fb = h == 0 ? 2 : (h == 1 ? 0 : 2);
          ma = h == 0 ? 0 : 1;
          mb = h == 0 ? 0 : 2;
        }
        for (int e0 = tid; e0 < E; e0 += GU * nth) {
          float2 A[GU], Bv[GU];
          float ay[GU];
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            int v, p;
            at(e0 + u * nth < E ? e0 + u * nth : e0, v, p);
            const int k = p > n / 2 ? n - p : p, row = s_row[v];
            A[u] = Bv[u] = make_float2(0.f, 0.f);
            ay[u] = 0.f;
            if (row >= 0 && k <= a.kmax1) {
              const int b = row / a.N0, x = row - b * a.N0;
              const float2* g = a.G + (size_t)b * NF * fs + (size_t)x * a.PF + k;
              A[u] = g[(size_t)fa * fs];
              Bv[u] = g[(size_t)fb * fs];
              ay[u] = a.ay[k];
            }
          }
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            if (e0 + u * nth >= E) continue;
            int v, p;
            at(e0 + u * nth, v, p);
            const bool cj = p > n / 2;
            const int k = cj ? n - p : p;
            auto mul = [&](float2 z, int m) {
              const float y = m == 2 ? ay[u] : (m == 3 ? -1.f : 1.f);
              return m == 0 ? z : make_float2(-y * z.y, y * z.x);
            };
            w.put(p, i * V + v, pack_pair(mul(A[u], ma), mul(Bv[u], mb), cj, k == 0 || 2 * k == n), true);
          }
        }
      }
    } else {
      for (int e = tid; e < E; e += nth) {
        int v, p;
        at(e, v, p);
        w.put(p, v, ps[e], false);
      }
    }
    w.run();
    if (inv) {
      for (int e = tid; e < E; e += nth) {
        int v, p;
        at(e, v, p);
#pragma unroll 1
        for (int i = 0; i < cnt; ++i) {
          const int h = h0 + i;
          const float2 z = w.get(p, i * V + v, true);
          if constexpr (TERM == TERM_KS) {
            ps[e] = make_float2(mulr(0.5f, addr(mulr(z.x, z.x), mulr(z.y, z.y))), 0.f);
          } else {
            if (h == 0) zs[e] = z;
            else {
              const float pr = zs[e].x * z.x + zs[e].y * z.y;
              if (h == 1) ps[e] = make_float2(pr, 0.f);
              else ps[e].y = pr;
            }
          }
        }
      }
      h0 += cnt;
      continue;
    }
    for (int e = tid; e < E; e += nth) {
      int v, k;
      at(e, v, k);
      const int row = s_row[v];
      if (row < 0 || k > n / 2) continue;
      const float2 zk = w.get(k, v, false);
      if constexpr (NP == 1) {
        a.P[(size_t)row * a.P1 + k] = zk;
      } else {
        const float2 zm = w.get(k == 0 ? 0 : n - k, v, false);
        const int b = row / a.N0, x = row - b * a.N0;
        float2* p0 = a.P + ((size_t)2 * b * a.N0 + x) * a.P1 + k;
        p0[0] = make_float2(0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y));
        const float2 d = make_float2(zk.x - zm.x, zk.y + zm.y);
        p0[(size_t)a.N0 * a.P1] = make_float2(0.5f * d.y, -0.5f * d.x);
      }
    }
    return;
  }
}

// ---------------------------------------------------------------- 1D persistent stepper
// k1_run's arithmetic with a run-time length, one workgroup per sample; the current stage spectrum s, the
// state and the stage arrays stay in LDS (local = 1) or in global memory where they do not fit.
template <bool TL>
__global__ void __launch_bounds__(1024) k_g1run(Run1Args a, GxDev ax, int local) {
  extern __shared__ float2 g_lds[];
  GxWork<TL> w(ax, g_lds);
  const int n = ax.n, H = n / 2 + 1, tid = w.tid, nth = w.nth, smp = blockIdx.x;
  float2* s = w.rest();
  float2* Ug = a.U + (size_t)smp * a.P;
  float2* A1g = a.A1 + (size_t)smp * a.P;
  float2 *U = Ug, *A1 = A1g, *A2 = a.A2 + (size_t)smp * a.P;
  const float* axk = a.ax + (size_t)smp * a.ax_bstride;
  const float4* cpk = a.cpk + (size_t)smp * a.cpk_bstride;
  const float2* src = a.src ? a.src + (size_t)smp * a.src_bstride : nullptr;
  float4 *c0 = nullptr, *c1 = nullptr;
  if (local) {
    U = s + H;
    A1 = U + H;
    A2 = A1 + H;
    float2* v = A2 + H;
    c0 = reinterpret_cast<float4*>(v + ((v - g_lds) & 1));  // 16-byte aligned
    c1 = c0 + H;
    float* x = reinterpret_cast<float*>(c1 + H);
    for (int k = tid; k < H; k += nth) {
      c0[k] = cpk[cpk_index(k, 0)];
      c1[k] = cpk[cpk_index(k, 1)];
      x[k] = axk[k];
    }
    axk = x;
  }
  for (int k = tid; k < H; k += nth) {
    const float2 z = Ug[k];
    s[k] = z;
    if (local) U[k] = z;
  }
  const int nev = a.eval_only ? 1 : scheme_evals(a.scheme);
  const int nst = a.eval_only ? 1 : a.nsteps;
  // mode k belongs to thread k % nth throughout (U, A1, A2, s); s is read across threads, behind a barrier
  auto record = [&](int i) {
    const int sl = a.rec_slot[i];
    if (sl < 0 || sl >= a.T) return;
    float2* t = a.traj + ((size_t)smp * a.T + sl) * a.P;
    for (int k = tid; k < H; k += nth) t[k] = U[k];
  };
#pragma unroll 1
  for (int it = 0; it < nst * nev; ++it) {
    const int e = it % nev;
    if (e == 0 && a.rec_slot && !a.eval_only) record(it / nev);
    __syncthreads();
    const int stage = a.eval_only ? ST_EVAL : scheme_stage(a.scheme, e);
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
      w.begin(1);
      for (int p = tid; p < n; p += nth) {
        float2 z;
        if (h == 0) {
          const bool cj = p > n / 2;
          const int k = cj ? n - p : p;
          float2 A = make_float2(0.f, 0.f);
          float ak = 0.f;
          if (k <= a.kmax) {
            A = s[k];
            A = make_float2(A.x * a.scale, A.y * a.scale);
            ak = a.cons ? 0.f : axk[k];
          }
          z = pack_pair(A, make_float2(-ak * A.y, ak * A.x), cj, k == 0 || 2 * k == n);
        } else {
          z = w.get(p, 0, true);
          z = make_float2(a.cons ? z.x * z.x : z.x * z.y, 0.f);
        }
        w.put(p, 0, z, h == 0);
      }
      w.run();
    }
    const int half = stage_coef_half(stage);
    for (int k = tid; k < H; k += nth) {
      const float4 c = local ? (half ? c1[k] : c0[k]) : cpk[cpk_index(k, half)];
      const float c5 = stage == ST_R4_E2 ? (local ? c1[k].z : cpk[cpk_index(k, 1)].z) : 0.f;
      float2 f = w.get(k, 0, false);
      if (a.cons) {
        // (i a) fft(u u); on an even axis' Nyquist frequency as k1_run does
        const float ak = axk[k];
        f = make_float2(-mulr(ak, f.y), mulr(ak, f.x));
      }
      float2 nv = rscale(a.coef_t, f);
      if (src) nv = radd(nv, src[k]);
      const float2 u = stage_reads_u(stage) ? U[k] : make_float2(0.f, 0.f);
      const float2 q1 = stage_reads_a1(stage) ? A1[k] : make_float2(0.f, 0.f);
      const float2 q2 = stage_reads_a2(stage) ? A2[k] : make_float2(0.f, 0.f);
      float2 st;
      s[k] = stage_combine_v(stage, nv, u, q1, q2, c, c5, &st);
      const int tgt = stage_target(stage);
      if (tgt == 0) U[k] = st;
      else if (tgt == 1) A1[k] = st;
      else A2[k] = st;
    }
  }
  if (a.rec_slot && !a.eval_only) record(nst);
  if (!local) return;
  for (int k = tid; k < H; k += nth) {
    if (a.eval_only) A1g[k] = A1[k];
    else Ug[k] = U[k];
  }
}

constexpr size_t GF_LDS = 150 * 1024;  // of 160 KB

// LDS bytes of V lines times fg fields, with `extra` float2 values per logical element, `fixed` more, and the
// tables staged or not
size_t lds_bytes(const GAxis& ax, int V, int fg, int extra, size_t fixed, bool tables) {
  const size_t tab = tables ? (size_t)ax.g.L + (ax.blu ? (size_t)ax.n + ax.g.L : 0) : 0;
  return (2 * (size_t)gx_slots(ax.g.L, V * fg) + tab + (size_t)extra * ax.n * V + fixed) * sizeof(float2);
}

// launch shape of one pass: the workgroup's lines, fields at once, tables in LDS
struct GxShape {
  int V = 1, fg = 1;
  bool tl = false;
  size_t lds = 0;
  unsigned threads = 64;
};

// nfield transforms of `lines` lines: all fields at once if LDS holds them, as many lines as 8192 points in
// flight allow (16 at most), but no fewer than `least` (adjacent columns share cache lines) unless LDS forces
// it, and otherwise few enough for two workgroups per CU; about 4 values per thread.  Where that would leave fewer
// than 64 workgroups they take single lines with more fields at once (8 SETDRK4 steps, us, B = 1: 509 x 64 Burgers 2587
// -> 1185, vorticity 2163 -> 987, where the unfused path takes 1940 and 1861; 993 x 256 vorticity 2505 -> 1820; a line of
// 256 workgroups instead of 64 costs 500^2 B = 4 half again)
GxShape choose(const GAxis& ax, size_t lines, int nfield, int least, int extra, size_t fixed) {
  if (lines / least < 64) least = 1;
  GxShape s;
  auto fits = [&](int V, int fg) { return lds_bytes(ax, V, fg, extra, fixed, true) <= GF_LDS; };
  s.fg = nfield;
  while (s.fg > 1 && !fits(least, s.fg)) --s.fg;
  const int groups = (nfield + s.fg - 1) / s.fg;
  s.fg = (nfield + groups - 1) / groups;
  while (s.V < 16 && ax.g.L * 2 * s.V * s.fg <= 8192 && fits(2 * s.V, s.fg)) s.V *= 2;
  while (s.V > least && lines / s.V < 512) s.V /= 2;
  s.tl = fits(s.V, s.fg);
  s.lds = lds_bytes(ax, s.V, s.fg, extra, fixed, s.tl);
  const long long t = (((long long)ax.g.L * s.V * s.fg / 4 + 63) / 64) * 64;
  s.threads = (unsigned)(t < 64 ? 64 : (t > 1024 ? 1024 : t));
  return s;
}

GxDev gx_dev(const GAxis& ax, const GxShape& s) {
  GxDev d;
  d.g = ax.g;
  d.n = ax.n;
  d.chirp = ax.blu ? ax.chirp[0] : nullptr;
  d.bhat = ax.blu ? ax.bhat[0] : nullptr;
  d.V = s.V;
  d.fg = s.fg;
  d.mgn = (unsigned)((0x100000000ULL + ax.n - 1) / ax.n);
  return d;
}

}  // namespace

// an axis of the 2D passes (two product planes and the wavenumbers beside the buffers), and the 1D stepper's mesh
// (the stage spectrum beside them: smooth lengths up to 4096)
bool genfused_axis(const GAxis& ax) {
  return ax.n > 1 && !ax.four && ax.g.L > 1 && lds_bytes(ax, 1, 1, 2, ax.n, false) <= GF_LDS;
}
bool genfused_mesh1d(const GAxis& ax) {
  return ax.n > 1 && !ax.four && ax.g.L > 1 && lds_bytes(ax, 1, 1, 0, (size_t)ax.n / 2 + 1, false) <= GF_LDS;
}

#define GF_LAUNCH(K, T, ...)                                                            \
  if (s.tl) hipLaunchKernelGGL((K<T, true>), grid, block, s.lds, st, __VA_ARGS__);         \
  else hipLaunchKernelGGL((K<T, false>), grid, block, s.lds, st, __VA_ARGS__);          \
  break;

hipError_t launch_g2col(int term, const Col2Args& a, const GAxis& ax, int nb, int stage, hipStream_t st) {
  const bool two = term == TERM_CONV || term == TERM_NSP;
  const size_t fixed = (size_t)ax.n / 2 + 1;  // x wavenumbers
  const GxShape s = choose(ax, (size_t)a.H1 * nb, a.NF, 4, two ? 2 : 1, fixed);
  const GxDev d = gx_dev(ax, s);
  if (ax.n != a.N0 || s.lds > GF_LDS) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(((a.H1 + s.V - 1) / s.V) * nb)), block(s.threads);
  switch (term) {
    case TERM_VC: GF_LAUNCH(k_g2col, TERM_VC, a, d, stage)
    case TERM_CONV: GF_LAUNCH(k_g2col, TERM_CONV, a, d, stage)
    case TERM_NSP: GF_LAUNCH(k_g2col, TERM_NSP, a, d, stage)
    case TERM_KS: GF_LAUNCH(k_g2col, TERM_KS, a, d, stage)
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_g2row(int term, const Row2Args& a, const GAxis& ax, hipStream_t st) {
  const int ni = term == TERM_KS ? 1 : (term == TERM_VC ? 2 : 3);
  const GxShape s = choose(ax, (size_t)a.B * a.N0, ni, 1, term == TERM_KS ? 1 : 2, 0);
  const GxDev d = gx_dev(ax, s);
  if (ax.n != a.N1 || s.lds > GF_LDS) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((a.B * a.N0 + s.V - 1) / s.V)), block(s.threads);
  switch (term) {
    case TERM_VC: GF_LAUNCH(k_g2row, TERM_VC, a, d)
    case TERM_CONV: case TERM_NSP: GF_LAUNCH(k_g2row, TERM_CONV, a, d)
    case TERM_KS: GF_LAUNCH(k_g2row, TERM_KS, a, d)
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_g1run(const Run1Args& a, const GAxis& ax, hipStream_t st) {
  const size_t H = (size_t)ax.n / 2 + 1;
  // s alone, or s, U, A1, A2, both coefficient halves (and a slot to align them) and the wavenumbers
  const size_t all = 8 * H + 1 + H / 2 + 1;
  const GxShape s = choose(ax, 1, 1, 1, 0, H);
  const int local = lds_bytes(ax, 1, 1, 0, all, s.tl) <= GF_LDS ? 1 : 0;
  const size_t lds = lds_bytes(ax, 1, 1, 0, local ? all : H, s.tl);
  if (ax.n != a.N || s.V != 1 || lds > GF_LDS || a.nsteps_per || a.coefc) return hipErrorInvalidValue;
  const dim3 grid((unsigned)a.B), block(s.threads);
  if (s.tl) hipLaunchKernelGGL(k_g1run<true>, grid, block, lds, st, a, gx_dev(ax, s), local);
  else hipLaunchKernelGGL(k_g1run<false>, grid, block, lds, st, a, gx_dev(ax, s), local);
  return hipGetLastError();
}

}  // namespace tfsm
