// Fused ETD evaluation of long 1D meshes, N = L1 * L2 points beyond the persistent stepper's 4096
// (Convection and ConservativeConvection, C = 1, real L).
//
// With modes q = q2 + L2 q1 and points x = x1 + L1 x2, a transform of N points is a four-step one:
//   T(x1, q2) = exp(2 pi i q2 x1 / N) sum_q1 U(q2 + L2 q1) exp(2 pi i q1 x1 / L1)
//   u(x1 + L1 x2) = sum_q2 T(x1, q2) exp(2 pi i q2 x2 / L2)
// For a real u the sequence over x2 at a fixed x1 is real, so T(x1, .) is Hermitian and only the
// columns q2 = 0..L2/2 are kept.  One nonlinear evaluation is therefore the row and column pass of a
// 2D one, and the points never reach memory:
//   k1l_row  per x1: packed C2R of (u, u_x) over q2, product, R2C            -> P [B][L1][PG]
//   k1l_col  per tile of V columns q2: conjugate twiddles, forward FFT over x1, N^, stage combine,
//            the next stage's fields u^ and i a u^, inverse FFTs, twiddles    -> G [B][NF][L1][PG]
// The state keeps its natural order [B][P]: column q2 holds the modes q2 + L2 q1, and one beyond
// N/2 is the conjugate of mode N - q, so a tile's lanes read consecutive (or reversed) modes.
// Every mode belongs to one column, except in the columns 0 and L2/2, which hold both q and N - q:
// there both compute the mode (all loads of the workgroup come before its first store) and the
// lower one stores it.
//
// Bound by the latency of one round of workgroups and by cache traffic: N = 65536, B = 16 moves about
// 40 MB per evaluation, which stays in the last-level cache, in 16 us (columns) + 8 us (rows); with the
// combine's operands loaded after the forward transform the columns took 17.7 us, and with 4 values per
// thread 15.8 (rows 8.6).  Before, an evaluation was six general-length FFT passes of 17-63 us and three
// elementwise ones, 205 us together.
#include "engine.hpp"

namespace tfsm {
namespace {

// A + iB of two Hermitian half spectra (mirror positions conjugated; the zero and Nyquist terms real)
__device__ __forceinline__ float2 pack_herm(float2 A, float2 Bv, bool cj, bool edge) {
  if (edge) {
    A.y = 0.f;
    Bv.y = 0.f;
  }
  return cj ? make_float2(A.x + Bv.y, Bv.x - A.y) : make_float2(A.x - Bv.y, A.y + Bv.x);
}

template <int L1, int V, int VAR>
__global__ void __launch_bounds__((Fft<L1, VAR>::NT * V)) k1l_col(Long1Args a, int stage) {
  using F = Fft<L1, VAR>;
  constexpr int RMAX = F::RMAX, NT = F::NT;
  __shared__ float2 s_tw[Fft<L1, VAR>::tw_size()];
  __shared__ float2 s_buf[LdsSize<L1, V>::slots];
  const int vi = threadIdx.x % V, j = threadIdx.x / V;
  const int H2 = a.L2 / 2 + 1;
  const int ntiles = (H2 + V - 1) / V;
  const int tile = blockIdx.x % ntiles, b = blockIdx.x / ntiles;
  const int q2 = tile * V + vi;
  const bool colv = q2 < H2;
  const int ql = colv ? q2 : H2 - 1;  // lanes past the last column read it and store nothing
  const bool both = ql == 0 || 2 * ql == a.L2;  // the column holds q and N - q
  const int half = a.N / 2;
  float2* U = a.U + (size_t)b * a.P;
  const float* ax = a.ax + (size_t)b * a.ax_bstride;
  // mode of value m: k <= N/2, mirrored when the lane's own q lies beyond N/2
  auto mode = [&](int m, bool& mir) {
    const int q = ql + a.L2 * (j + m * NT);
    mir = q > half;
    return mir ? a.N - q : q;
  };
  auto cj = [](float2 z, bool mir) { return mir ? make_float2(z.x, -z.y) : z; };
  float2 w[RMAX], s[RMAX];  // w: exp(-2 pi i q2 x1 / N) of this lane's x1
#pragma unroll
  for (int m = 0; m < RMAX; ++m) w[m] = a.tw4[(size_t)(j + m * NT) * a.PG + ql];
  if (stage == ST_PRO) {
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      bool mir;
      const int k = mode(m, mir);
      s[m] = cj(U[k], mir);
    }
    load_twiddles<L1, VAR>(s_tw, a.tw1);
    __syncthreads();
  } else {
    // every operand of the tile is loaded before the forward transform, whose time then hides the
    // memory latency (a launch has about one workgroup per CU: no other wave does)
    float2 v[RMAX], uu[RMAX], o1[RMAX], o2[RMAX];
    float4 cc[RMAX];
    float c5[RMAX];
    const float2* Pb = a.Pr + (size_t)b * L1 * a.PG + ql;
#pragma unroll
    for (int m = 0; m < RMAX; ++m) v[m] = Pb[(size_t)(j + m * NT) * a.PG];
    const bool rdu = stage_reads_u(stage), rd1 = stage_reads_a1(stage), rd2 = stage_reads_a2(stage);
    const int tgt = stage_target(stage), h16 = stage_coef_half(stage) << 4;
    float2* A1 = a.A1 + (size_t)b * a.P;
    float2* A2 = a.A2 + (size_t)b * a.P;
    float2* dst = tgt == 0 ? U : (tgt == 1 ? A1 : A2);
    const float2* src = a.src ? a.src + (size_t)b * a.src_bstride : nullptr;
    const float4* cpk = a.cpk + (size_t)b * a.cpk_bstride;
    const float* c5t = a.c5t + (size_t)b * (a.cpk_bstride / 2);
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      bool mir;
      const int k = mode(m, mir);
      cc[m] = cpk[2 * k - (k & 15) + h16];
      uu[m] = o1[m] = o2[m] = make_float2(0.f, 0.f);
      c5[m] = 0.f;
      if (rdu) uu[m] = U[k];
      if (rd1) o1[m] = A1[k];
      if (rd2) o2[m] = A2[k];
      if (stage == ST_R4_E2) c5[m] = c5t[k];
    }
    load_twiddles<L1, VAR>(s_tw, a.tw1);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < RMAX; ++m) v[m] = cmul(v[m], w[m]);
    fft_wg<L1, -1, V, VAR>(v, s_buf, s_tw, j, vi);
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      bool mir;
      const int k = mode(m, mir);
      float2 f = v[m];
      if (a.cons) {
        const float ak = mir ? -ax[k] : ax[k];
        f = make_float2(-mulr(ak, f.y), mulr(ak, f.x));  // (i a) fft(u u)
      }
      float2 nv = rscale(a.coef_t, f);
      if (src) nv = radd(nv, cj(src[k], mir));
      float2 st;
      s[m] = stage_combine_v(stage, nv, cj(uu[m], mir), cj(o1[m], mir), cj(o2[m], mir), cc[m], c5[m], &st);
      v[m] = st;
    }
    __syncthreads();  // every load of the columns that hold a mode twice is done
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      bool mir;
      const int k = mode(m, mir);
      if (colv && !(both && mir)) dst[k] = cj(v[m], mir);
    }
    if (stage == ST_EVAL) return;  // a single evaluation needs no fields
  }
  const int nf = a.cons ? 1 : 2;
#pragma unroll 1
  for (int f = 0; f < nf; ++f) {
    float2 v[RMAX];
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      bool mir;
      const int k = mode(m, mir);
      float2 val = make_float2(0.f, 0.f);
      if (k <= a.kmax) {
        val = make_float2(s[m].x * a.scale, s[m].y * a.scale);
        if (f) {
          const float ak = mir ? -ax[k] : ax[k];
          val = make_float2(-ak * val.y, ak * val.x);  // i a u^
        }
      }
      v[m] = val;
    }
    fft_wg<L1, +1, V, VAR>(v, s_buf, s_tw, j, vi);
    if (colv) {
      float2* g = a.G + ((size_t)b * nf + f) * L1 * a.PG + ql;
#pragma unroll
      for (int m = 0; m < RMAX; ++m) g[(size_t)(j + m * NT) * a.PG] = cmulc(v[m], w[m]);
    }
  }
}

template <int L2, int ROWS, int VAR>
__global__ void __launch_bounds__((Fft<L2, VAR>::NT * ROWS)) k1l_row(Long1Args a) {
  using F = Fft<L2, VAR>;
  constexpr int RMAX = F::RMAX, NT = F::NT, SL = LdsSize<L2, 1>::slots;
  constexpr bool WS = RowSync<L2, VAR>::WS;
  __shared__ float2 s_tw[Fft<L2, VAR>::tw_size()];
  __shared__ float2 s_buf[ROWS * SL];
  const int g = threadIdx.x / NT, j = threadIdx.x % NT;
  const int row = blockIdx.x * ROWS + g;
  const bool rv = row < a.B * a.L1;
  const int b = rv ? row / a.L1 : 0, x1 = rv ? row % a.L1 : 0;
  const int nf = a.cons ? 1 : 2;
  const float2* G0 = a.G + ((size_t)b * nf * a.L1 + x1) * a.PG;
  const float2* G1 = G0 + (a.cons ? 0 : (size_t)a.L1 * a.PG);
  float2 v[RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) {
    const int pos = j + m * NT;
    const bool cj = pos > L2 / 2;
    const int k = cj ? L2 - pos : pos;
    const float2 A = G0[k];
    const float2 Bv = a.cons ? make_float2(0.f, 0.f) : G1[k];
    v[m] = pack_herm(A, Bv, cj, k == 0 || k == L2 / 2);
  }
  load_twiddles<L2, VAR>(s_tw, a.tw2);
  __syncthreads();
  float2* lds = s_buf + g * SL;
  fft_wg<L2, +1, 1, VAR, WS>(v, lds, s_tw, j, 0);
  // Convection u u_x, or ConservativeConvection's u u (its derivative follows the transform)
#pragma unroll
  for (int m = 0; m < RMAX; ++m) v[m] = make_float2(a.cons ? v[m].x * v[m].x : v[m].x * v[m].y, 0.f);
  fft_wg<L2, -1, 1, VAR, WS>(v, lds, s_tw, j, 0);
  if (rv) {
    float2* p = a.Pw + ((size_t)b * a.L1 + x1) * a.PG;
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      const int pos = j + m * NT;
      if (pos <= L2 / 2) p[pos] = v[m];
    }
  }
}

// radix-plan variant: 8 values per thread where the length has such a plan
constexpr int lvar(int n) { return n == 128 ? 2 : ((n == 256 || n == 1024) ? 1 : 0); }

template <int L1>
hipError_t launch_lcol_t(const Long1Args& a, int stage, hipStream_t st) {
  constexpr int V = 8, VR = lvar(L1);
  const int tiles = (a.L2 / 2 + 1 + V - 1) / V;
  hipLaunchKernelGGL((k1l_col<L1, V, VR>), dim3(tiles * a.B), dim3(Fft<L1, VR>::NT * V), 0, st, a, stage);
  return hipGetLastError();
}

template <int L2>
hipError_t launch_lrow_t(const Long1Args& a, hipStream_t st) {
  constexpr int VR = lvar(L2), NT = Fft<L2, VR>::NT, ROWS = NT >= 256 ? 1 : 256 / NT;
  hipLaunchKernelGGL((k1l_row<L2, ROWS, VR>), dim3((a.B * a.L1 + ROWS - 1) / ROWS), dim3(NT * ROWS), 0, st, a);
  return hipGetLastError();
}

#define TFSM_LONG_SIZES(X) \
  X(64) X(96) X(100) X(112) X(128) X(192) X(200) X(256) X(384) X(400) X(512) X(768) X(800) X(1024)

}  // namespace

int long1d_var(int n) { return lvar(n); }

// N = L1 L2 with both lengths among the instantiated ones, as square as possible with L1 <= L2
bool long1d_split(int n, int* l1, int* l2) {
  static const int sizes[] = {
#define TFSM_LONG_ITEM(M) M,
      TFSM_LONG_SIZES(TFSM_LONG_ITEM)
#undef TFSM_LONG_ITEM
  };
  bool found = false;
  for (int s : sizes)
    for (int t : sizes)
      if ((long long)s * t == n && s <= t && (!found || s > *l1)) {
        *l1 = s;
        *l2 = t;
        found = true;
      }
  return found;
}

hipError_t launch_long1d_col(const Long1Args& a, int stage, hipStream_t st) {
  switch (a.L1) {
#define TFSM_LONG_CASE(M) \
  case M: return launch_lcol_t<M>(a, stage, st);
    TFSM_LONG_SIZES(TFSM_LONG_CASE)
#undef TFSM_LONG_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_long1d_row(const Long1Args& a, hipStream_t st) {
  switch (a.L2) {
#define TFSM_LONG_CASE(M) \
  case M: return launch_lrow_t<M>(a, st);
    TFSM_LONG_SIZES(TFSM_LONG_CASE)
#undef TFSM_LONG_CASE
    default: return hipErrorInvalidValue;
  }
}

}  // namespace tfsm
