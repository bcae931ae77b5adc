// Fused adjoint of 2D Convection and VorticityConvection on power-of-two axes of 32 to 512 points (the
// step's adjoint is stated in k_adjoint.hip; the unfused kernels there serve every other shape).
//
// With v^ a stage adjoint and G the dealiased fields of the stage's state u after the x-inverse (the
// planes of k2_col), W = J_N(u)^T v^ takes two launches:
//   k2_adj_row  rows of G and of p = x-inverse of v^ (all columns: v^ is not dealiased) to physical
//               space, the products, and their forward rows: planes Q of the kept columns; NL: also the
//               forward rows of u's own product, as k2_row
//   k2_adj_col  forward columns of Q -> W, the stage algebra Y = W + sum s_k c_k X_k, and, for the next
//               stage down, v^ = s c Y + sum s_k c_k X_k and its x-inverse p; NL: N(u) as well
// Convection, one workgroup per channel in the column pass: with p_c the adjoint fields,
//   W_c = coef M (F[R_c] - i a_x F[S_c0] - i a_y F[S_c1]),  R_c = sum_j p_j d_c u_j,  S_ci = p_c u_i;
// a_y is constant along a column, so the row kernel stores the row transforms of R_c - i a_y S_c1 (planes
// 0, 1) and S_c0 (planes 2, 3).  VorticityConvection: planes p w_x, p w_y, p psi_y, p psi_x.
//
// Each launch is one or two rounds of workgroups, as long as one thread's chain of transforms: 4 values
// per thread (up to 256 points), 1 to 8 transforms.  Burgers 128^2, C = 2, B = 16, one ETDRK2 adjoint step with
// the gradient of the viscosity: 26 launches and copies, 179 us -> 10 launches, 70 us (rows 8.9 and 9.4 us, with the
// transforms one after the other 9.8 and 11.0; columns 4.8, 8.0 and 12.0; loading the column pass's operands before
// its first transform changes nothing).
#include "k_step2d.hpp"

namespace tfsm {

// K transforms: together (fft_wg_k) with 4 values per thread, otherwise one after the other
template <int N, int VAR>
struct Together {
  static constexpr bool value = Fft<N, VAR>::RMAX <= 4;
};
template <int K, int N, int DIR, int V, int VAR, bool WS>
__device__ __forceinline__ void fft_all(float2 (&z)[K][(Fft<N, VAR>::RMAX)], float2* lds, const float2* s_tw, int j,
                                        int vi) {
  if constexpr (Together<N, VAR>::value) {
    fft_wg_k<K, N, DIR, V, VAR, WS>(z, lds, LdsSize<N, V>::slots, s_tw, j, vi);
  } else {
#pragma unroll
    for (int l = 0; l < K; ++l) fft_wg<N, DIR, V, VAR, WS>(z[l], lds, s_tw, j, vi);
  }
}

// v holds forward row transforms of pairs of real fields: their half spectra, the first of pair l in v[l], the
// second in w[l] (this lane's positions, valid up to N1/2)
template <int K, int N1, int VAR>
__device__ __forceinline__ void unpack_pairs(float2 (&v)[K][(Fft<N1, VAR>::RMAX)],
                                             float2 (&w)[K][(Fft<N1, VAR>::RMAX)], float2* lds, int j) {
  using F = Fft<N1, VAR>;
  constexpr int RMAX = F::RMAX, NT = F::NT;
  constexpr bool WS = RowSync<N1, VAR>::WS;
  constexpr int KG = Together<N1, VAR>::value ? K : 1;  // pairs at once
#pragma unroll
  for (int l0 = 0; l0 < K; l0 += KG) {
#pragma unroll
    for (int l = 0; l < KG; ++l)
#pragma unroll
      for (int m = 0; m < RMAX; ++m) lds[l * LdsSize<N1, 1>::slots + lds_slot<1>(j + m * NT, 0)] = v[l0 + l][m];
    lds_sync<WS>();
#pragma unroll
    for (int l = 0; l < KG; ++l)
#pragma unroll
      for (int m = 0; m < RMAX; ++m) {
        const int pos = j + m * NT;
        const float2 zk = v[l0 + l][m];
        const float2 zm = lds[l * LdsSize<N1, 1>::slots + lds_slot<1>(pos == 0 ? 0 : N1 - pos, 0)];
        const float2 d = make_float2(zk.x - zm.x, zk.y + zm.y);
        v[l0 + l][m] = make_float2(0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y));
        w[l0 + l][m] = make_float2(0.5f * d.y, -0.5f * d.x);
      }
    lds_sync<WS>();
  }
}

template <int N1, int ROWS, int TERM, int VAR, bool NL>
__global__ void __launch_bounds__((Fft<N1, VAR>::NT * ROWS)) k2_adj_row(Adj2RowArgs a) {
  using F = Fft<N1, VAR>;
  constexpr int RMAX = F::RMAX, NT = F::NT;
  constexpr bool WS = RowSync<N1, VAR>::WS;
  constexpr int NC = Term2<TERM>::NC;
  constexpr int KI = Term2<TERM>::KR + 1, KF = (TERM == TERM_CONV ? 3 : 2) + (NL ? 1 : 0);  // transforms in, out
  constexpr int SL = (Together<N1, VAR>::value ? 4 : 1) * LdsSize<N1, 1>::slots;
  __shared__ float2 s_tw[F::tw_size()];
  __shared__ float2 s_buf[ROWS * SL];
  load_twiddles<N1, VAR>(s_tw, a.tw1);
  __syncthreads();
  const int g = threadIdx.x / NT, j = threadIdx.x % NT;
  float2* lds = s_buf + g * SL;
  const int row = blockIdx.x * ROWS + g;
  const bool rv = row < a.B * a.N0;
  const int b = rv ? row / a.N0 : 0, x = rv ? row % a.N0 : 0;
  const size_t fs = (size_t)a.N0 * a.PF, ps = (size_t)a.N0 * a.P1;
  const float2* gr = a.G + (size_t)b * 4 * fs + (size_t)x * a.PF;
  const float2* pr = a.GP + (size_t)b * NC * ps + (size_t)x * a.P1;
  float2 z[KI][RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) {
    const int pos = j + m * NT;
    const bool cj = pos > N1 / 2;
    const int k = cj ? N1 - pos : pos;
    const bool edge = (k == 0) || (k == N1 / 2);
    const float2 o = make_float2(0.f, 0.f);
    float2 f0 = o, f1 = o, f2 = o, f3 = o, p0 = o, p1 = o;
    float ay = 0.f;
    if (rv) {
      p0 = pr[k];
      if constexpr (NC == 2) p1 = pr[ps + k];
    }
    if (rv && k <= a.kmax1) {
      f0 = gr[k];
      f1 = gr[fs + k];
      f2 = gr[2 * fs + k];
      f3 = gr[3 * fs + k];
      ay = a.ay[k];
    }
    z[0][m] = pack_pair(p0, p1, cj, edge);
    if constexpr (TERM == TERM_VC) {  // fields psi, a_x psi, a_x w, w
      z[1][m] = pack_pair(make_float2(-ay * f0.y, ay * f0.x), make_float2(f1.y, -f1.x), cj, edge);  // psi_y, -psi_x
      z[2][m] = pack_pair(make_float2(-f2.y, f2.x), make_float2(-ay * f3.y, ay * f3.x), cj, edge);  // w_x, w_y
    } else {  // u0, a_x u0, u1, a_x u1
      z[1][m] = pack_pair(f0, f2, cj, edge);
      z[2][m] = pack_pair(make_float2(-f1.y, f1.x), make_float2(-ay * f0.y, ay * f0.x), cj, edge);  // d0u0, d1u0
      z[3][m] = pack_pair(make_float2(-f3.y, f3.x), make_float2(-ay * f2.y, ay * f2.x), cj, edge);  // d0u1, d1u1
    }
  }
  fft_all<KI, N1, +1, 1, VAR, WS>(z, lds, s_tw, j, 0);
  float2 v[KF][RMAX], w[KF][RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) {
    const float2 p = z[0][m], z1 = z[1][m], z2 = z[2][m];
    if constexpr (TERM == TERM_VC) {
      v[0][m] = make_float2(p.x * z2.x, p.x * z2.y);   // p w_x, p w_y
      v[1][m] = make_float2(p.x * z1.x, -p.x * z1.y);  // p psi_y, p psi_x
      if constexpr (NL) v[KF - 1][m] = make_float2(z1.x * z2.x + z1.y * z2.y, 0.f);
    } else {
      const float2 z3 = z[3][m];
      v[0][m] = make_float2(p.x * z2.x + p.y * z3.x, p.x * z2.y + p.y * z3.y);  // R_0, R_1
      v[1][m] = make_float2(p.x * z1.y, p.y * z1.y);                            // S_01, S_11
      v[2][m] = make_float2(p.x * z1.x, p.y * z1.x);                            // S_00, S_10
      if constexpr (NL) v[KF - 1][m] = make_float2(z1.x * z2.x + z1.y * z2.y, z1.x * z3.x + z1.y * z3.y);
    }
  }
  fft_all<KF, N1, -1, 1, VAR, WS>(v, lds, s_tw, j, 0);
  unpack_pairs<KF, N1, VAR>(v, w, lds, j);
  if (!rv) return;
  float2* q = a.Q + (size_t)b * 4 * fs + (size_t)x * a.PF;
  float2* p = a.P + (size_t)b * NC * ps + (size_t)x * a.P1;
#pragma unroll
  for (int m = 0; m < RMAX; ++m) {
    const int pos = j + m * NT;
    if (NL && pos <= N1 / 2) {
      p[pos] = v[KF - 1][m];
      if constexpr (NC == 2) p[ps + pos] = w[KF - 1][m];
    }
    if (pos <= a.kmax1) {
      if constexpr (TERM == TERM_VC) {
        q[pos] = v[0][m];
        q[fs + pos] = w[0][m];
        q[2 * fs + pos] = v[1][m];
        q[3 * fs + pos] = w[1][m];
      } else {
        const float ay = a.ay[pos];
        q[pos] = make_float2(v[0][m].x + ay * v[1][m].y, v[0][m].y - ay * v[1][m].x);
        q[fs + pos] = make_float2(w[0][m].x + ay * w[1][m].y, w[0][m].y - ay * w[1][m].x);
        q[2 * fs + pos] = v[2][m];
        q[3 * fs + pos] = w[2][m];
      }
    }
  }
}

// MODE 0: v^ -> p only; 1: W, Y and the next stage's v^ -> p; 2: W and Y
template <int N0, int V, int TERM, int VAR, int MODE>
__global__ void __launch_bounds__((Fft<N0, VAR>::NT * V)) k2_adj_col(Adj2ColArgs a) {
  using F = Fft<N0, VAR>;
  constexpr int RMAX = F::RMAX, NT = F::NT;
  constexpr int NC = Term2<TERM>::NC, NQ = TERM == TERM_CONV ? 2 : 4;  // channels, planes of Q per channel
  __shared__ float2 s_tw[F::tw_size()];
  __shared__ float2 s_buf[(MODE > 0 && Together<N0, VAR>::value ? NQ : 1) * LdsSize<N0, V>::slots];
  load_twiddles<N0, VAR>(s_tw, a.tw0);
  __syncthreads();
  const int vi = threadIdx.x % V, j = threadIdx.x / V;
  const int ntiles = a.P1 / V;
  const int tile = blockIdx.x % ntiles, bc = blockIdx.x / ntiles;
  const int b = bc / NC, c = bc % NC;
  const int ky = tile * V + vi;  // within the pitch: V divides it
  const bool colv = ky < a.H1;
  const size_t plane = (size_t)N0 * a.P1, fs = (size_t)N0 * a.PF;
  const size_t sb = (size_t)bc * plane + ky;  // this column of a state array
  const float* cf = a.coef + (size_t)b * a.coef_bstride + ky;
  const float2 z = make_float2(0.f, 0.f);
  float2 y[RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) y[m] = z;
  // acc += s c X (c: a coefficient table, slot < 0: 1)
  auto add = [&](float2 (&acc)[RMAX], const float2* X, int slot, float s) {
    float2 t[RMAX];
    float k[RMAX];
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      const size_t o = (size_t)(j + m * NT) * a.P1;
      t[m] = X[sb + o];
      k[m] = slot >= 0 ? cf[(size_t)slot * plane + o] : 1.f;
    }
#pragma unroll
    for (int m = 0; m < RMAX; ++m) acc[m] = make_float2(acc[m].x + s * k[m] * t[m].x, acc[m].y + s * k[m] * t[m].y);
  };
  constexpr int NX = MODE == 0 ? 0 : (MODE == 1 ? 1 : ADJ2_MAXT), NV = MODE == 2 ? 0 : 2;  // terms at most
  float yk[RMAX];
  if constexpr (MODE == 1) {
#pragma unroll
    for (int m = 0; m < RMAX; ++m) yk[m] = cf[(size_t)a.yslot * plane + (size_t)(j + m * NT) * a.P1];
  }
  if constexpr (MODE > 0) {
    const bool kept = tile * V <= a.kmax1;  // uniform: the tile has kept columns
    const bool kc = ky <= a.kmax1;
    float2 q[NQ][RMAX];
    if (kept) {
      const float2* qb = a.Q + (size_t)b * 4 * fs + ky;
#pragma unroll
      for (int l = 0; l < NQ; ++l) {
        const size_t pl = TERM == TERM_CONV ? 2 * l + c : l;
#pragma unroll
        for (int m = 0; m < RMAX; ++m) q[l][m] = kc ? qb[pl * fs + (size_t)(j + m * NT) * a.PF] : z;
      }
    }
    if (a.N) {  // uniform: N(u) = coef F(P) + S, from the product's rows
      float2 v[RMAX];
#pragma unroll
      for (int m = 0; m < RMAX; ++m) {
        const float2 t = a.P[sb + (size_t)(j + m * NT) * a.P1];
        v[m] = colv ? t : z;
      }
      fft_wg<N0, -1, V, VAR>(v, s_buf, s_tw, j, vi);
      const float2* src = a.src ? a.src + (size_t)b * a.src_bstride + (size_t)c * a.src_cstride + ky : nullptr;
#pragma unroll
      for (int m = 0; m < RMAX; ++m) {
        float2 n = make_float2(a.coef_t * v[m].x, a.coef_t * v[m].y);
        const size_t o = (size_t)(j + m * NT) * a.P1;
        if (src) {
          const float2 s = src[o];
          n = make_float2(n.x + s.x, n.y + s.y);
        }
        a.N[sb + o] = colv ? n : z;
      }
    }
    if (kept) {
      fft_all<NQ, N0, -1, V, VAR, false>(q, s_buf, s_tw, j, vi);
      const float ay = TERM == TERM_VC && colv ? a.ay[ky] : 0.f;
#pragma unroll
      for (int m = 0; m < RMAX; ++m) {
        const int kx = j + m * NT, ks = kx <= N0 / 2 ? kx : N0 - kx;
        const float ax = a.ax[kx];
        float2 w;
        if constexpr (TERM == TERM_CONV) {
          w = make_float2(q[0][m].x + ax * q[1][m].y, q[0][m].y - ax * q[1][m].x);
        } else {
          // coef M [invlap (i a_y R1 - i a_x R2) - i a_x R3 + i a_y R4]
          const float lap = -ax * ax - ay * ay;
          const float il = lap == 0.f ? 1.f : 1.f / lap;
          const float2 t = make_float2(-ay * q[0][m].y + ax * q[1][m].y, ay * q[0][m].x - ax * q[1][m].x);
          w = make_float2(il * t.x + ax * q[2][m].y - ay * q[3][m].y, il * t.y - ax * q[2][m].x + ay * q[3][m].x);
        }
        if (kc && ks <= a.kmax0) y[m] = make_float2(a.coef_t * w.x, a.coef_t * w.y);
      }
    }
#pragma unroll
    for (int k = 0; k < NX; ++k)
      if (k < a.nt) add(y, a.X[k], a.slot[k], a.s[k]);
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      if (!colv) y[m] = z;
      a.Y[sb + (size_t)(j + m * NT) * a.P1] = y[m];  // padded columns too: zero
    }
  }
  if constexpr (MODE < 2) {
    float2 v[RMAX];
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      v[m] = z;
      if constexpr (MODE == 1) v[m] = make_float2(a.ys * yk[m] * y[m].x, a.ys * yk[m] * y[m].y);
    }
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (k < a.nv) add(v, a.V[k], a.vslot[k], a.vs[k]);
#pragma unroll
    for (int m = 0; m < RMAX; ++m) v[m] = colv ? make_float2(v[m].x * a.scale, v[m].y * a.scale) : z;
    fft_wg<N0, +1, V, VAR>(v, s_buf, s_tw, j, vi);
    if (colv) {
#pragma unroll
      for (int m = 0; m < RMAX; ++m) a.GP[sb + (size_t)(j + m * NT) * a.P1] = v[m];
    }
  }
}

// ---------------------------------------------------------------- host launchers
// 4 values per thread up to 256 points, 8 at 512
int adj2d_var(int n) { return n == 512 ? 0 : 3; }
bool adj2d_size(int n) { return n == 32 || n == 64 || n == 128 || n == 256 || n == 512; }

#define TFSM_ADJ_SWITCH(n, ...)                                                    \
  switch (n) {                                                                     \
    case 32: { constexpr int NN = 32, VR = 3; __VA_ARGS__ }                        \
    case 64: { constexpr int NN = 64, VR = 3; __VA_ARGS__ }                        \
    case 128: { constexpr int NN = 128, VR = 3; __VA_ARGS__ }                      \
    case 256: { constexpr int NN = 256, VR = 3; __VA_ARGS__ }                      \
    case 512: { constexpr int NN = 512, VR = 0; __VA_ARGS__ }                      \
    default: return hipErrorInvalidValue;                                          \
  }

template <int NN, int VR, int TERM>
static hipError_t adj_row_t(const Adj2RowArgs& a, hipStream_t st) {
  constexpr int NT = Fft<NN, VR>::NT;
  constexpr int ROWS = NT >= 256 ? 1 : 256 / NT;
  const dim3 grid((a.B * a.N0 + ROWS - 1) / ROWS), block(NT * ROWS);
  if (a.P) hipLaunchKernelGGL((k2_adj_row<NN, ROWS, TERM, VR, true>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((k2_adj_row<NN, ROWS, TERM, VR, false>), grid, block, 0, st, a);
  return hipGetLastError();
}

template <int NN, int VR, int TERM>
static hipError_t adj_col_t(const Adj2ColArgs& a, hipStream_t st) {
  constexpr int V = 8;
  // (terms at most: the kernel's NX and NV)
  if (a.P1 % V != 0 || a.nt > (a.GP ? 1 : ADJ2_MAXT) || a.nv > (a.GP ? 2 : 0)) return hipErrorInvalidValue;
  const dim3 grid(a.P1 / V * a.B * Term2<TERM>::NC), block(Fft<NN, VR>::NT * V);
  if (!a.Q) hipLaunchKernelGGL((k2_adj_col<NN, V, TERM, VR, 0>), grid, block, 0, st, a);
  else if (a.GP) hipLaunchKernelGGL((k2_adj_col<NN, V, TERM, VR, 1>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((k2_adj_col<NN, V, TERM, VR, 2>), grid, block, 0, st, a);
  return hipGetLastError();
}

hipError_t launch_adj2d_row(int term, const Adj2RowArgs& a, hipStream_t st) {
  TFSM_ADJ_SWITCH(a.N1, {
    if (term == TERM_VC) return adj_row_t<NN, VR, TERM_VC>(a, st);
    return adj_row_t<NN, VR, TERM_CONV>(a, st);
  })
}

hipError_t launch_adj2d_col(int term, const Adj2ColArgs& a, hipStream_t st) {
  TFSM_ADJ_SWITCH(a.N0, {
    if (term == TERM_VC) return adj_col_t<NN, VR, TERM_VC>(a, st);
    return adj_col_t<NN, VR, TERM_CONV>(a, st);
  })
}

}  // namespace tfsm
