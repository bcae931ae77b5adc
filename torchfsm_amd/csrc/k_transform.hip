// Batched multi-dimensional FFT passes (FourierMesh.fft / .ifft, mesh.py:481-491), spectrum
// conversions at the API boundary, the exact linear stepper (ETDRK0, _etdrk.py:10-27) and the 1D
// persistent stepper.
#include "engine.hpp"

namespace tfsm {

// ---------------------------------------------------------------- contiguous rows
// real rows [nrows][in_ld] -> half spectrum rows [nrows][out_ld] (k = 0..N/2), times scale; the padded
// columns up to the pitch out_ld become zero (as far as the row's N positions reach)
template <int N, int ROWS>
__global__ void __launch_bounds__(Fft<N>::NT* ROWS)
    k_rows_r2c(const float* __restrict__ in, size_t in_ld, float2* __restrict__ out, size_t out_ld, int nrows,
               float scale, const float2* tw) {
  using F = Fft<N>;
  constexpr int RMAX = F::RMAX, NT = F::NT, SL = LdsSize<N, 1>::slots;
  __shared__ float2 s_tw[Fft<N>::tw_size()];
  __shared__ float2 s_buf[ROWS * SL];
  load_twiddles<N>(s_tw, tw);
  __syncthreads();
  const int g = threadIdx.x / NT, j = threadIdx.x % NT;
  const int row = blockIdx.x * ROWS + g;
  const bool rv = row < nrows;
  float2 v[RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) v[m] = make_float2(rv ? in[(size_t)row * in_ld + j + m * NT] : 0.f, 0.f);
  fft_wg<N, -1, 1, 0, RowSync<N, 0>::WS>(v, s_buf + g * SL, s_tw, j, 0);
  if (rv) {
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      const int pos = j + m * NT;
      if (pos < (int)out_ld)
        out[(size_t)row * out_ld + pos] = pos <= N / 2 ? make_float2(v[m].x * scale, v[m].y * scale) : make_float2(0.f, 0.f);
    }
  }
}

// half spectrum rows -> real rows, times scale (C2R: imaginary parts of k = 0 and N/2 ignored)
template <int N, int ROWS>
__global__ void __launch_bounds__(Fft<N>::NT* ROWS)
    k_rows_c2r(const float2* __restrict__ in, size_t in_ld, float* __restrict__ out, size_t out_ld, int nrows,
               float scale, const float2* tw) {
  using F = Fft<N>;
  constexpr int RMAX = F::RMAX, NT = F::NT, SL = LdsSize<N, 1>::slots;
  __shared__ float2 s_tw[Fft<N>::tw_size()];
  __shared__ float2 s_buf[ROWS * SL];
  load_twiddles<N>(s_tw, tw);
  __syncthreads();
  const int g = threadIdx.x / NT, j = threadIdx.x % NT;
  const int row = blockIdx.x * ROWS + g;
  const bool rv = row < nrows;
  float2 v[RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) {
    const int pos = j + m * NT;
    const bool cj = pos > N / 2;
    const int k = cj ? N - pos : pos;
    float2 x = rv ? in[(size_t)row * in_ld + k] : make_float2(0.f, 0.f);
    if (k == 0 || k == N / 2) x.y = 0.f;
    v[m] = cj ? make_float2(x.x, -x.y) : x;
  }
  fft_wg<N, +1, 1, 0, RowSync<N, 0>::WS>(v, s_buf + g * SL, s_tw, j, 0);
  if (rv) {
#pragma unroll
    for (int m = 0; m < RMAX; ++m) out[(size_t)row * out_ld + j + m * NT] = v[m].x * scale;
  }
}

// complex rows in place (length N, pitch ld)
template <int N, int ROWS, int DIR>
__global__ void __launch_bounds__(Fft<N>::NT* ROWS)
    k_rows_c2c(const float2* in, size_t in_ld, float2* out, size_t out_ld, int nrows, float scale,
               const float2* tw) {
  using F = Fft<N>;
  constexpr int RMAX = F::RMAX, NT = F::NT, SL = LdsSize<N, 1>::slots;
  __shared__ float2 s_tw[Fft<N>::tw_size()];
  __shared__ float2 s_buf[ROWS * SL];
  load_twiddles<N>(s_tw, tw);
  __syncthreads();
  const int g = threadIdx.x / NT, j = threadIdx.x % NT;
  const int row = blockIdx.x * ROWS + g;
  const bool rv = row < nrows;
  float2 v[RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) v[m] = rv ? in[(size_t)row * in_ld + j + m * NT] : make_float2(0.f, 0.f);
  fft_wg<N, DIR, 1, 0, RowSync<N, 0>::WS>(v, s_buf + g * SL, s_tw, j, 0);
  if (rv) {
#pragma unroll
    for (int m = 0; m < RMAX; ++m) out[(size_t)row * out_ld + j + m * NT] = make_float2(v[m].x * scale, v[m].y * scale);
  }
}

// ---------------------------------------------------------------- strided columns
// Element (o, p, i) at base + o*outer_stride + p*col_stride + i, p along the transformed axis,
// i in [0, ninner) contiguous.  A workgroup transforms V adjacent i of one o.  Out of place
// (in may equal out).
template <int N, int V, int DIR>
__global__ void __launch_bounds__(Fft<N>::NT* V)
    k_cols_c2c(const float2* in, float2* out, size_t outer_stride, size_t col_stride, int ninner, float scale,
               const float2* tw, StepMask mask, int b0, unsigned o0, unsigned outer_per_sample) {
  using F = Fft<N>;
  constexpr int RMAX = F::RMAX, NT = F::NT;
  __shared__ float2 s_tw[Fft<N>::tw_size()];
  __shared__ float2 s_buf[LdsSize<N, V>::slots];
  if (mask.act && mask.skip(b0 + (int)((o0 + blockIdx.y) / outer_per_sample))) return;
  load_twiddles<N>(s_tw, tw);
  __syncthreads();
  const int vi = threadIdx.x % V, j = threadIdx.x / V;
  const int i = blockIdx.x * V + vi;
  const bool iv = i < ninner;
  const size_t base = (size_t)blockIdx.y * outer_stride + i;
  float2 v[RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) v[m] = iv ? in[base + (size_t)(j + m * NT) * col_stride] : make_float2(0.f, 0.f);
  fft_wg<N, DIR, V>(v, s_buf, s_tw, j, vi);
  if (iv) {
#pragma unroll
    for (int m = 0; m < RMAX; ++m)
      out[base + (size_t)(j + m * NT) * col_stride] = make_float2(v[m].x * scale, v[m].y * scale);
  }
}

// U <- E^n U between the two directions of one axis, for the exact linear stepper (ETDRK0) of a call that
// starts and ends in physical space: the last forward pass, the steps and the first inverse pass of a column
// in one launch (heat equation 512^2, B = 16: forward 11.5, steps 13.3 and inverse 11.8 us as launches of their
// own, 15.5 here; the whole call 61 -> 33 us).  The steps multiply one at a time, as k_linear_steps does.  EV: float (real L) or float2.
__device__ __forceinline__ float2 lin_mul(float e, float2 u) { return rscale(e, u); }
__device__ __forceinline__ float2 lin_mul(float2 e, float2 u) { return cmulr(e, u); }
__device__ __forceinline__ float lin_conj(float e) { return e; }
__device__ __forceinline__ float2 lin_conj(float2 e) { return make_float2(e.x, -e.y); }

// strided columns (layout of k_cols_c2c), in place: block o = blockIdx.y belongs to sample (o0 + o) / C and its
// element (p, i) is mode p * col_stride + i
template <int N, int V, class EV>
__global__ void __launch_bounds__(Fft<N>::NT* V)
    k_cols_linear(float2* u, size_t outer_stride, size_t col_stride, int ninner, const float2* tw,
                  const EV* __restrict__ E, size_t e_bstride, int C, unsigned o0, int nsteps) {
  using F = Fft<N>;
  constexpr int RMAX = F::RMAX, NT = F::NT;
  __shared__ float2 s_tw[Fft<N>::tw_size()];
  __shared__ float2 s_buf[LdsSize<N, V>::slots];
  const int vi = threadIdx.x % V, j = threadIdx.x / V;
  const int i = blockIdx.x * V + vi;
  const bool iv = i < ninner;
  float2* ub = u + (size_t)blockIdx.y * outer_stride + (iv ? i : 0);
  const EV* Eb = E + (size_t)((o0 + blockIdx.y) / C) * e_bstride + (iv ? i : 0);
  float2 v[RMAX];
  EV e[RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) v[m] = ub[(size_t)(j + m * NT) * col_stride];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) e[m] = Eb[(size_t)(j + m * NT) * col_stride];
  load_twiddles<N>(s_tw, tw);
  __syncthreads();
  fft_wg<N, -1, V>(v, s_buf, s_tw, j, vi);
  for (int s = 0; s < nsteps; ++s)
#pragma unroll
    for (int m = 0; m < RMAX; ++m) v[m] = lin_mul(e[m], v[m]);
  fft_wg<N, +1, V>(v, s_buf, s_tw, j, vi);
  if (iv) {
#pragma unroll
    for (int m = 0; m < RMAX; ++m) ub[(size_t)(j + m * NT) * col_stride] = v[m];
  }
}

// 1D: whole real rows, mode k of row r in row r / C of E; a mirrored position takes the conjugate factor
template <int N, int ROWS, class EV>
__global__ void __launch_bounds__(Fft<N>::NT* ROWS)
    k_rows_linear(const float* __restrict__ in, float* __restrict__ out, int nrows, float scale, const float2* tw,
                  const EV* __restrict__ E, size_t e_bstride, int C, int nsteps) {
  using F = Fft<N>;
  constexpr int RMAX = F::RMAX, NT = F::NT, SL = LdsSize<N, 1>::slots;
  __shared__ float2 s_tw[Fft<N>::tw_size()];
  __shared__ float2 s_buf[ROWS * SL];
  const int g = threadIdx.x / NT, j = threadIdx.x % NT;
  const int row = blockIdx.x * ROWS + g;
  const bool rv = row < nrows;
  const EV* Er = E + (size_t)((rv ? row : 0) / C) * e_bstride;
  float2 v[RMAX];
  EV e[RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) {
    const int pos = j + m * NT;
    v[m] = make_float2(rv ? in[(size_t)row * N + pos] : 0.f, 0.f);
    e[m] = pos > N / 2 ? lin_conj(Er[N - pos]) : Er[pos];
  }
  load_twiddles<N>(s_tw, tw);
  __syncthreads();
  fft_wg<N, -1, 1, 0, RowSync<N, 0>::WS>(v, s_buf + g * SL, s_tw, j, 0);
#pragma unroll
  for (int m = 0; m < RMAX; ++m) {
    const int pos = j + m * NT;
    for (int s = 0; s < nsteps; ++s) v[m] = lin_mul(e[m], v[m]);
    if (pos == 0 || pos == N / 2) v[m].y = 0.f;
  }
  lds_sync<RowSync<N, 0>::WS>();
  fft_wg<N, +1, 1, 0, RowSync<N, 0>::WS>(v, s_buf + g * SL, s_tw, j, 0);
  if (rv) {
#pragma unroll
    for (int m = 0; m < RMAX; ++m) out[(size_t)row * N + j + m * NT] = v[m].x * scale;
  }
}

// ---------------------------------------------------------------- spectrum conversions


// full [nblk][N0..N_{D-1}] -> half [nblk][N0..][P]: Hermitian projection (x + conj(x_mirror)) / 2
__global__ void k_full_to_half(const float2* __restrict__ full, float2* __restrict__ half, ConvArgs a) {
  const int nl = a.n[a.D - 1];
  const size_t inner_half = (a.D == 1 ? 1 : (size_t)a.n[0] * (a.D == 3 ? a.n[1] : 1));
  const size_t total = a.nblk * inner_half * a.P;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const int k = (int)(e % a.P);
    size_t r = e / a.P;
    int i1 = 0, i0 = 0;
    if (a.D == 3) {
      i1 = (int)(r % a.n[1]);
      r /= a.n[1];
    }
    if (a.D >= 2) {
      i0 = (int)(r % a.n[0]);
      r /= a.n[0];
    }
    const size_t blk = r;
    float2 val = make_float2(0.f, 0.f);
    if (k < a.H) {
      size_t fb = blk;
      size_t fi = 0, fm = 0;
      const int mk = (nl - k) % nl;
      if (a.D == 1) {
        fi = fb * nl + k;
        fm = fb * nl + mk;
      } else if (a.D == 2) {
        const int m0 = (a.n[0] - i0) % a.n[0];
        fi = (fb * a.n[0] + i0) * nl + k;
        fm = (fb * a.n[0] + m0) * nl + mk;
      } else {
        const int m0 = (a.n[0] - i0) % a.n[0], m1 = (a.n[1] - i1) % a.n[1];
        fi = ((fb * a.n[0] + i0) * a.n[1] + i1) * nl + k;
        fm = ((fb * a.n[0] + m0) * a.n[1] + m1) * nl + mk;
      }
      const float2 x = full[fi], y = full[fm];
      val = make_float2(0.5f * (x.x + y.x), 0.5f * (x.y - y.y));
    }
    half[e] = val;
  }
}

// half -> full with Hermitian fill X[-i][-k] = conj(X[i][k])
__global__ void k_half_to_full(const float2* __restrict__ half, float2* __restrict__ full, ConvArgs a) {
  const int nl = a.n[a.D - 1];
  size_t cnt = a.nblk * nl;
  if (a.D >= 2) cnt *= a.n[0];
  if (a.D == 3) cnt *= a.n[1];
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < cnt; e += (size_t)gridDim.x * blockDim.x) {
    const int il = (int)(e % nl);
    size_t r = e / nl;
    int i1 = 0, i0 = 0;
    if (a.D == 3) {
      i1 = (int)(r % a.n[1]);
      r /= a.n[1];
    }
    if (a.D >= 2) {
      i0 = (int)(r % a.n[0]);
      r /= a.n[0];
    }
    const size_t blk = r;
    const bool cj = il > nl / 2;
    const int k = cj ? nl - il : il;
    const int j0 = (cj && a.D >= 2) ? (a.n[0] - i0) % a.n[0] : i0;
    const int j1 = (cj && a.D == 3) ? (a.n[1] - i1) % a.n[1] : i1;
    size_t hi;
    if (a.D == 1) hi = blk * a.P + k;
    else if (a.D == 2) hi = (blk * a.n[0] + j0) * a.P + k;
    else hi = ((blk * a.n[0] + j0) * a.n[1] + j1) * a.P + k;
    float2 x = half[hi];
    full[e] = cj ? make_float2(x.x, -x.y) : x;
  }
}

// ---------------------------------------------------------------- exact linear stepping (ETDRK0)
// U <- E U, nsteps times, recording frames before step i where rec_slot[i] is in [0, T) (and after).
__global__ void k_linear_steps(float2* __restrict__ U, const float* __restrict__ E, size_t coef_bstride,
                               size_t modes, int C, size_t total, int nsteps, const int* __restrict__ rec_slot,
                               float2* __restrict__ traj, int T) {
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const size_t mode = e % modes;
    const size_t bc = e / modes;
    const size_t b = bc / C, c = bc % C;
    const float ev = E[b * coef_bstride + mode];
    float2 u = U[e];
    for (int s = 0; s <= nsteps; ++s) {
      if (rec_slot) {
        const int sl = rec_slot[s];
        if (sl >= 0 && sl < T) traj[((b * T + sl) * C + c) * modes + mode] = u;
      }
      if (s < nsteps) u = rscale(ev, u);
    }
    U[e] = u;
  }
}


// complex-L plans: U <- E U with complex E (complex64 product)
__global__ void k_linear_steps_c(float2* __restrict__ U, const float2* __restrict__ E, size_t coef_bstride,
                                 size_t modes, int C, size_t total, int nsteps, const int* __restrict__ rec_slot,
                                 float2* __restrict__ traj, int T) {
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const size_t mode = e % modes;
    const size_t bc = e / modes;
    const size_t b = bc / C, c = bc % C;
    const float2 ev = E[b * coef_bstride + mode];
    float2 u = U[e];
    for (int s = 0; s <= nsteps; ++s) {
      if (rec_slot) {
        const int sl = rec_slot[s];
        if (sl >= 0 && sl < T) traj[((b * T + sl) * C + c) * modes + mode] = u;
      }
      if (s < nsteps) u = cmulr(ev, u);
    }
    U[e] = u;
  }
}

// copy the state U [B][per_sample] to traj[b][rec_slot[step]] when that slot is in [0, T)
// (_TrajRecorder.record before step i, traj_recorder.py:46-55); the schedule is read on the
// device so a captured step sequence does not depend on it.
__global__ void k_record(const float2* __restrict__ U, float2* __restrict__ traj, const int* __restrict__ rec_slot,
                         int step, int B, size_t per_sample, int T) {
  const int sl = rec_slot[step];
  if (sl < 0 || sl >= T) return;
  const size_t total = (size_t)B * per_sample;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const size_t b = e / per_sample, r = e % per_sample;
    traj[(b * T + sl) * per_sample + r] = U[e];
  }
}

// ---------------------------------------------------------------- 1D persistent stepper
// One launch runs every step of a call: NT = N / RMAX threads per sample, thread j owning the modes
// k = j + m NT (k <= N/2) with their state U, stage arrays A1, A2 and (real L) packed coefficients in
// registers for the whole run.  Convection (C = D = 1): N = coef_t * fft(u * u_x) [+ S], u from the
// dealiased stage spectrum; ConservativeConvection: N = coef_t * (i a) fft(u * u) [+ S].
// CPLX: complex-L plan (complex coefficient tables, stage_combine_c).
//
// Bound by one wavefront's serial chain: a few samples occupy a few CUs, so an evaluation takes as long
// as its instructions and LDS exchanges in a row.  The radix plans (var1) therefore hold 4 or 8 values
// per thread (up to 256 points 4, in one wavefront, without barriers; 512 and more 8, over two LDS
// buffers with one barrier per exchange).  One SETDRK4 step, in us, before (16 values per
// thread, state and coefficients in LDS or memory) and now: N = 128, B = 1 19.3 -> 5.2; 512, B = 8 12.1 ->
// 8.0; 2048, B = 8 28.5 -> 13.3; 4096, B = 16 33.1 -> 17.1; 100, B = 1 30.0 -> 17.7; several waves per SIMD
// gain as much (128, B = 4096 20.8 -> 7.5; 4096, B = 1024 133 -> 70).
template <int N>
struct Run1Shape {
  static constexpr int VAR = var1(N);
  using F = Fft<N, VAR>;
  static constexpr int NT = F::NT, RMAX = F::RMAX;
  static constexpr int G = NT >= 64 ? 1 : 64 / NT;  // samples per workgroup
  static constexpr bool WS = RowSync<N, VAR>::WS;   // a sample lives inside one wavefront
  static constexpr bool PP = NT > 64;               // two exchange buffers, workgroup barriers
  static constexpr int HM = RMAX / 2 + 1;           // modes per thread (the last one: k = N/2, j = 0 only)
};

template <int N, int DIR>
__device__ __forceinline__ void run1_fft(float2 (&v)[Run1Shape<N>::RMAX], float2* lds, const float2* tw, int j) {
  using S = Run1Shape<N>;
  if constexpr (S::PP) fft_wg_pp<N, DIR, 1, S::VAR>(v, lds, lds + LdsSize<N, 1>::slots, tw, j, 0);
  else fft_wg<N, DIR, 1, S::VAR, S::WS>(v, lds, tw, j, 0);
}

// the combine of one compile-time stage over a thread's modes; cf: packed coefficient halves
template <int N, bool CPLX, int ST>
__device__ __forceinline__ void run1_combine(const Run1Args& a, const float2 (&nv)[Run1Shape<N>::HM],
                                             float2 (&U)[Run1Shape<N>::HM], float2 (&A1)[Run1Shape<N>::HM],
                                             float2 (&A2)[Run1Shape<N>::HM],
                                             const float4 (&c0)[CPLX ? 1 : Run1Shape<N>::HM],
                                             const float4 (&c1)[CPLX ? 1 : Run1Shape<N>::HM], const float2* cfc,
                                             float2 (&s)[Run1Shape<N>::HM], int j) {
  using S = Run1Shape<N>;
#pragma unroll
  for (int i = 0; i < S::HM; ++i) {
    if constexpr (CPLX) {
      const int k = j + i * S::NT;
      s[i] = stage_combine_c(ST, nv[i], U, A1, A2, i, cfc, a.P, k <= N / 2 ? k : 0);
    } else {
      float2 w;
      s[i] = stage_combine_v(ST, nv[i], U[i], A1[i], A2[i], stage_coef_half(ST) ? c1[i] : c0[i], c1[i].z, &w);
      if constexpr (ST != ST_PRO) {
        if (stage_target(ST) == 0) U[i] = w;
        else if (stage_target(ST) == 1) A1[i] = w;
        else A2[i] = w;
      }
    }
  }
}

template <int N, bool CPLX>
__global__ void __launch_bounds__((Run1Shape<N>::NT * Run1Shape<N>::G)) k1_run(Run1Args a) {
  using S = Run1Shape<N>;
  using F = typename S::F;
  constexpr int RMAX = S::RMAX, NT = S::NT, HM = S::HM, SL = LdsSize<N, 1>::slots;
  __shared__ float2 s_tw[F::tw_size()];
  __shared__ float2 s_buf[S::G * (S::PP ? 2 : 1) * SL];
  __shared__ float2 s_mir[S::G * N];  // mirror positions N - k of the packed spectrum
  for (int i = threadIdx.x; i < F::tw_size(); i += NT * S::G) s_tw[i] = a.tw_run[i];
  const int g = threadIdx.x / NT, j = threadIdx.x % NT;
  const int smp = blockIdx.x * S::G + g;
  const bool valid = smp < a.B;
  const int sb = valid ? smp : 0;
  int nmax = 0;  // steps of the workgroup: every thread takes part in every transform
  for (int w = 0; w < S::G; ++w) {
    const int sw = blockIdx.x * S::G + w;
    if (sw < a.B) {
      const int ns = a.nsteps_per ? a.nsteps_per[sw] : a.nsteps;
      nmax = ns > nmax ? ns : nmax;
    }
  }
  const int nst = valid ? (a.nsteps_per ? a.nsteps_per[smp] : a.nsteps) : 0;
  float2* lds = s_buf + g * (S::PP ? 2 : 1) * SL;
  float2* mir = s_mir + g * N;
  float2* Ug = a.U + (size_t)sb * a.P;
  const float* ax = a.ax + (size_t)sb * a.ax_bstride;
  const float2* cfc = CPLX ? a.coefc + (size_t)sb * a.coef_bstride : nullptr;
  const float4* cpk = a.cpk + (size_t)sb * a.cpk_bstride;
  const float2* src = a.src ? a.src + (size_t)sb * a.src_bstride : nullptr;
  float2 U[HM], A1[HM], A2[HM], s[HM], sv[HM];
  float4 c0[CPLX ? 1 : HM], c1[CPLX ? 1 : HM];
  float axk[HM];
#pragma unroll
  for (int i = 0; i < HM; ++i) {
    const int k = j + i * NT, kc = k <= N / 2 ? k : 0;  // the last slot belongs to k = N/2 (j = 0)
    U[i] = Ug[kc];
    if (!valid) U[i] = make_float2(0.f, 0.f);
    A1[i] = A2[i] = make_float2(0.f, 0.f);
    s[i] = U[i];
    sv[i] = src ? src[kc] : make_float2(0.f, 0.f);
    axk[i] = ax[kc];
    if constexpr (!CPLX) {
      c0[i] = cpk[cpk_index(kc, 0)];
      c1[i] = cpk[cpk_index(kc, 1)];
    }
  }
  __syncthreads();
  const int nev = a.eval_only ? 1 : scheme_evals(a.scheme);
  const int nloop = a.eval_only ? 1 : nmax;
  const bool rec = a.rec_slot && valid && !a.eval_only;
  auto record = [&](int sl) {
    if (sl < 0 || sl >= a.T) return;
    float2* t = a.traj + ((size_t)smp * a.T + sl) * a.P;
#pragma unroll
    for (int i = 0; i < HM; ++i)
      if (j + i * NT <= N / 2) t[j + i * NT] = U[i];
  };
  int slot = rec ? a.rec_slot[0] : -1;
  for (int step = 0; step < nloop; ++step) {
    const bool active = valid && step < nst;
    if (rec && active) {
      record(slot);
      slot = a.rec_slot[step + 1];  // read a step ahead
    }
    for (int e = 0; e < nev; ++e) {
      const int stage = a.eval_only ? ST_EVAL : scheme_stage(a.scheme, e);
      float2 v[RMAX];
      // Z = A + i B of the Hermitian spectra A = u^ and B = i a u^ (B = 0 for ConservativeConvection:
      // u_x in the imaginary part would add its round-off to u): own positions k, and the mirrored
      // conj(A) + i conj(B) through LDS to the owner of position N - k
#pragma unroll
      for (int i = 0; i < HM; ++i) {
        const int k = j + i * NT;
        float2 A = make_float2(0.f, 0.f);
        float ak = 0.f;
        if (k <= a.kmax) {
          A = make_float2(s[i].x * a.scale, s[i].y * a.scale);
          ak = a.cons ? 0.f : axk[i];
        }
        float2 Bv = make_float2(-ak * A.y, ak * A.x);
        if (k == 0 || k == N / 2) {
          A.y = 0.f;
          Bv.y = 0.f;
        }
        if (i < RMAX / 2) {
          v[i] = make_float2(A.x - Bv.y, A.y + Bv.x);
          if (k > 0) mir[N - k] = make_float2(A.x + Bv.y, Bv.x - A.y);
        } else if (j == 0) {
          mir[N / 2] = make_float2(A.x - Bv.y, A.y + Bv.x);
        }
      }
      lds_sync<S::WS>();
#pragma unroll
      for (int m = RMAX / 2; m < RMAX; ++m) v[m] = mir[j + m * NT];
      run1_fft<N, +1>(v, lds, s_tw, j);
      // Convection u u_x, or ConservativeConvection's u u (its derivative follows the transform)
#pragma unroll
      for (int m = 0; m < RMAX; ++m) v[m] = make_float2(a.cons ? v[m].x * v[m].x : v[m].x * v[m].y, 0.f);
      run1_fft<N, -1>(v, lds, s_tw, j);
      if (!(active || (a.eval_only && valid))) continue;  // no barrier below
      float2 nv[HM];
#pragma unroll
      for (int i = 0; i < HM; ++i) {
        float2 f = v[i];
        if (a.cons) f = make_float2(-mulr(axk[i], f.y), mulr(axk[i], f.x));  // (i a) fft(u u)
        nv[i] = rscale(a.coef_t, f);
        if (src) nv[i] = radd(nv[i], sv[i]);
      }
      switch (stage) {
#define TFSM_RUN1_STAGE(X) \
  case X: run1_combine<N, CPLX, X>(a, nv, U, A1, A2, c0, c1, cfc, s, j); break;
        TFSM_RUN1_STAGE(ST_R1_E0)
        TFSM_RUN1_STAGE(ST_R2_E0)
        TFSM_RUN1_STAGE(ST_R2_E1)
        TFSM_RUN1_STAGE(ST_R3_E0)
        TFSM_RUN1_STAGE(ST_R3_E1)
        TFSM_RUN1_STAGE(ST_R3_E2)
        TFSM_RUN1_STAGE(ST_R4_E0)
        TFSM_RUN1_STAGE(ST_R4_E1)
        TFSM_RUN1_STAGE(ST_R4_E2)
        TFSM_RUN1_STAGE(ST_R4_E3)
        TFSM_RUN1_STAGE(ST_EVAL)
#undef TFSM_RUN1_STAGE
        default: break;
      }
    }
  }
  if (rec) record(slot);
  if (!valid) return;
  float2* out = a.eval_only ? a.A1 + (size_t)smp * a.P : Ug;
#pragma unroll
  for (int i = 0; i < HM; ++i) {
    // by component: a choice between the two arrays themselves would put both in scratch memory
    const float2 n = A1[i], u = U[i];
    if (j + i * NT <= N / 2) out[j + i * NT] = make_float2(a.eval_only ? n.x : u.x, a.eval_only ? n.y : u.y);
  }
}

// ---------------------------------------------------------------- 1D KSConvection, one stage per launch
// KSConvection's remove_mean subtracts the mean over the whole batch, so the stages of different
// samples are coupled through the DC mode: each stage is evaluated for every sample (raw product
// spectrum), the batch mean of the DC is reduced, then the stage combine runs.
// Nraw = fft(1/2 (d_x phi)^2) of the dealiased stage spectrum S (_ks_convection.py:27-38).
template <int N, int V>
__global__ void __launch_bounds__(Fft<N>::NT* V) k1_eval_ks(Run1Args a, const float2* S, float2* Nraw) {
  using F = Fft<N>;
  constexpr int RMAX = F::RMAX, NT = F::NT;
  __shared__ float2 s_tw[Fft<N>::tw_size()];
  __shared__ float2 s_buf[LdsSize<N, V>::slots];
  load_twiddles<N>(s_tw, a.tw);
  __syncthreads();
  const int vi = threadIdx.x % V, j = threadIdx.x / V;
  const int smp = blockIdx.x * V + vi;
  const bool valid = smp < a.B;
  const float2* Sb = S + (size_t)(valid ? smp : 0) * a.P;
  const float* ax = a.ax + (size_t)(valid ? smp : 0) * a.ax_bstride;
  float2 v[RMAX];
#pragma unroll
  for (int m = 0; m < RMAX; ++m) {
    const int pos = j + m * NT;
    const bool cj = pos > N / 2;
    const int k = cj ? N - pos : pos;
    float2 g = make_float2(0.f, 0.f);
    if (valid && k <= a.kmax) {
      const float2 val = make_float2(Sb[k].x * a.scale, Sb[k].y * a.scale);
      const float axk = ax[k];
      g = make_float2(-axk * val.y, axk * val.x);  // i a_k phi^
    }
    if (k == 0 || k == N / 2) g.y = 0.f;
    v[m] = cj ? make_float2(g.x, -g.y) : g;
  }
  fft_wg<N, +1, V>(v, s_buf, s_tw, j, vi);
#pragma unroll
  for (int m = 0; m < RMAX; ++m) v[m] = make_float2(mulr(0.5f, mulr(v[m].x, v[m].x)), 0.f);
  fft_wg<N, -1, V>(v, s_buf, s_tw, j, vi);
  if (valid) {
#pragma unroll
    for (int m = 0; m < RMAX; ++m) {
      const int pos = j + m * NT;
      if (pos <= N / 2) Nraw[(size_t)smp * a.P + pos] = v[m];
    }
  }
}

// stage combine of every (sample, k <= N/2): N = coef_t (Nraw - [k = 0] dc) + S_src, then the
// stage's update of U / A1 / A2; S receives the next stage spectrum
__global__ void k1_stage(Run1Args a, int stage, const float2* __restrict__ Nraw, const float2* __restrict__ dc,
                         float2* __restrict__ S) {
  const size_t total = (size_t)a.B * a.H;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const size_t smp = e / a.H;
    const int pos = (int)(e % a.H);
    const size_t so = smp * a.P;
    float2 v = Nraw[so + pos];
    if (pos == 0 && dc) v = rsub(v, dc[0]);
    const float2* src = a.src ? a.src + smp * a.src_bstride : nullptr;
    const float2 nv = nl_value(a.coef_t, v, src, pos);
    if (a.coefc)
      S[so + pos] = stage_combine_c(stage, nv, a.U + so, a.A1 + so, a.A2 + so, pos, a.coefc + smp * a.coef_bstride,
                                    a.P, pos);
    else
      S[so + pos] = stage_combine(stage, nv, a.U + so, a.A1 + so, a.A2 + so, pos, a.coef + smp * a.coef_bstride, a.P,
                                  pos, true);
  }
}

// ---------------------------------------------------------------- host launchers
template <int N>
static constexpr int rows_per_wg() {
  return Fft<N>::NT >= 256 ? 1 : 256 / Fft<N>::NT;
}

// lengths up to 512 points (rows and strided columns), and the longer ones (rows only)
#define TFSM_CASES_512(...) \
    case 16: { constexpr int NN = 16; __VA_ARGS__; } \
    case 32: { constexpr int NN = 32; __VA_ARGS__; } \
    case 64: { constexpr int NN = 64; __VA_ARGS__; } \
    case 128: { constexpr int NN = 128; __VA_ARGS__; } \
    case 256: { constexpr int NN = 256; __VA_ARGS__; } \
    case 512: { constexpr int NN = 512; __VA_ARGS__; } \
    case 48: { constexpr int NN = 48; __VA_ARGS__; } \
    case 96: { constexpr int NN = 96; __VA_ARGS__; } \
    case 100: { constexpr int NN = 100; __VA_ARGS__; } \
    case 112: { constexpr int NN = 112; __VA_ARGS__; } \
    case 192: { constexpr int NN = 192; __VA_ARGS__; } \
    case 200: { constexpr int NN = 200; __VA_ARGS__; } \
    case 384: { constexpr int NN = 384; __VA_ARGS__; } \
    case 400: { constexpr int NN = 400; __VA_ARGS__; }
#define TFSM_SWITCH_COLS(n, ...)  \
  switch (n) {                  \
    TFSM_CASES_512(__VA_ARGS__) \
    default: return hipErrorInvalidValue; \
  }
#define TFSM_SWITCH_N(n, ...)  \
  switch (n) {                  \
    TFSM_CASES_512(__VA_ARGS__) \
    case 1024: { constexpr int NN = 1024; __VA_ARGS__; } \
    case 2048: { constexpr int NN = 2048; __VA_ARGS__; } \
    case 4096: { constexpr int NN = 4096; __VA_ARGS__; } \
    case 768: { constexpr int NN = 768; __VA_ARGS__; } \
    case 800: { constexpr int NN = 800; __VA_ARGS__; } \
    default: return hipErrorInvalidValue; \
  }

hipError_t launch_rows_r2c(int n, const float* in, size_t in_ld, float2* out, size_t out_ld, int nrows, float scale,
                           const float2* tw, hipStream_t st) {
  if (nrows <= 0) return hipSuccess;
  TFSM_SWITCH_N(n, {
    constexpr int R = rows_per_wg<NN>();
    hipLaunchKernelGGL((k_rows_r2c<NN, R>), dim3((nrows + R - 1) / R), dim3(Fft<NN>::NT * R), 0, st, in, in_ld, out,
                       out_ld, nrows, scale, tw);
    return hipGetLastError();
  })
}

hipError_t launch_rows_c2r(int n, const float2* in, size_t in_ld, float* out, size_t out_ld, int nrows, float scale,
                           const float2* tw, hipStream_t st) {
  if (nrows <= 0) return hipSuccess;
  TFSM_SWITCH_N(n, {
    constexpr int R = rows_per_wg<NN>();
    hipLaunchKernelGGL((k_rows_c2r<NN, R>), dim3((nrows + R - 1) / R), dim3(Fft<NN>::NT * R), 0, st, in, in_ld, out,
                       out_ld, nrows, scale, tw);
    return hipGetLastError();
  })
}

hipError_t launch_rows_c2c(int n, int dir, const float2* in, size_t in_ld, float2* out, size_t out_ld, int nrows,
                           float scale, const float2* tw, hipStream_t st) {
  if (nrows <= 0) return hipSuccess;
  TFSM_SWITCH_N(n, {
    constexpr int R = rows_per_wg<NN>();
    if (dir < 0)
      hipLaunchKernelGGL((k_rows_c2c<NN, R, -1>), dim3((nrows + R - 1) / R), dim3(Fft<NN>::NT * R), 0, st, in, in_ld,
                         out, out_ld, nrows, scale, tw);
    else
      hipLaunchKernelGGL((k_rows_c2c<NN, R, 1>), dim3((nrows + R - 1) / R), dim3(Fft<NN>::NT * R), 0, st, in, in_ld,
                         out, out_ld, nrows, scale, tw);
    return hipGetLastError();
  })
}

hipError_t launch_cols_c2c(int n, int dir, const float2* in, float2* out, size_t nouter, size_t outer_stride,
                           size_t col_stride, int ninner, float scale, const float2* tw, hipStream_t st,
                           StepMask mask, int b0, size_t outer_per_sample) {
  if (nouter == 0 || ninner <= 0) return hipSuccess;
  if (mask.act && (outer_per_sample == 0 || nouter > 0xffffffffu)) return hipErrorInvalidValue;
  TFSM_SWITCH_COLS(n, {
    constexpr int V = Fft<NN>::NT * 16 <= 1024 ? 16 : 8;
    // grid.y is limited to 65535: launch the outer blocks in chunks
    for (size_t o0 = 0; o0 < nouter; o0 += 65535) {
      const size_t no = (nouter - o0) < 65535 ? (nouter - o0) : 65535;
      dim3 grid((ninner + V - 1) / V, (unsigned)no);
      const float2* ib = in + o0 * outer_stride;
      float2* ob = out + o0 * outer_stride;
      const unsigned ops = (unsigned)(outer_per_sample ? outer_per_sample : 1);
      if (dir < 0)
        TFSM_LAUNCH((k_cols_c2c<NN, V, -1>), grid, dim3(Fft<NN>::NT * V), 0, st, ib, ob, outer_stride,
                           col_stride, ninner, scale, tw, mask, b0, (unsigned)o0, ops);
      else
        TFSM_LAUNCH((k_cols_c2c<NN, V, 1>), grid, dim3(Fft<NN>::NT * V), 0, st, ib, ob, outer_stride,
                           col_stride, ninner, scale, tw, mask, b0, (unsigned)o0, ops);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  })
}

// the column passes around the exact linear steps (k_cols_linear); e_bstride in elements of E or Ec
hipError_t launch_cols_linear(int n, float2* u, size_t nouter, size_t outer_stride, size_t col_stride, int ninner,
                              const float2* tw, const float* E, const float2* Ec, size_t e_bstride, int C, int nsteps,
                              hipStream_t st) {
  if (nouter == 0 || ninner <= 0) return hipSuccess;
  TFSM_SWITCH_COLS(n, {
    constexpr int V = Fft<NN>::NT * 16 <= 1024 ? 16 : 8;
    for (size_t o0 = 0; o0 < nouter; o0 += 65535) {
      const size_t no = (nouter - o0) < 65535 ? (nouter - o0) : 65535;
      const dim3 grid((ninner + V - 1) / V, (unsigned)no);
      const dim3 block(Fft<NN>::NT * V);
      float2* ub = u + o0 * outer_stride;
      if (Ec)
        hipLaunchKernelGGL((k_cols_linear<NN, V, float2>), grid, block, 0, st, ub, outer_stride, col_stride, ninner, tw,
                           Ec, e_bstride, C, (unsigned)o0, nsteps);
      else
        hipLaunchKernelGGL((k_cols_linear<NN, V, float>), grid, block, 0, st, ub, outer_stride, col_stride, ninner, tw,
                           E, e_bstride, C, (unsigned)o0, nsteps);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  })
}

hipError_t launch_rows_linear(int n, const float* in, float* out, int nrows, float scale, const float2* tw,
                              const float* E, const float2* Ec, size_t e_bstride, int C, int nsteps, hipStream_t st) {
  if (nrows <= 0) return hipSuccess;
  TFSM_SWITCH_N(n, {
    constexpr int R = rows_per_wg<NN>();
    const dim3 grid((nrows + R - 1) / R);
    const dim3 block(Fft<NN>::NT * R);
    if (Ec)
      hipLaunchKernelGGL((k_rows_linear<NN, R, float2>), grid, block, 0, st, in, out, nrows, scale, tw, Ec, e_bstride,
                         C, nsteps);
    else
      hipLaunchKernelGGL((k_rows_linear<NN, R, float>), grid, block, 0, st, in, out, nrows, scale, tw, E, e_bstride, C,
                         nsteps);
    return hipGetLastError();
  })
}

hipError_t launch_full_to_half(const float2* full, float2* half, const ConvArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(k_full_to_half, dim3(1024), dim3(256), 0, st, full, half, a);
  return hipGetLastError();
}

hipError_t launch_half_to_full(const float2* half, float2* full, const ConvArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(k_half_to_full, dim3(1024), dim3(256), 0, st, half, full, a);
  return hipGetLastError();
}

hipError_t launch_linear_steps(float2* U, const float* E, size_t coef_bstride, size_t modes, int C, size_t total,
                               int nsteps, const int* rec_slot, float2* traj, int T, hipStream_t st) {
  unsigned blocks = (unsigned)((total + 255) / 256);
  if (blocks > 65535u * 4) blocks = 65535u * 4;
  hipLaunchKernelGGL(k_linear_steps, dim3(blocks), dim3(256), 0, st, U, E, coef_bstride, modes, C, total, nsteps,
                     rec_slot, traj, T);
  return hipGetLastError();
}

hipError_t launch_linear_steps_c(float2* U, const float2* E, size_t coef_bstride, size_t modes, int C, size_t total,
                                 int nsteps, const int* rec_slot, float2* traj, int T, hipStream_t st) {
  unsigned blocks = (unsigned)((total + 255) / 256);
  if (blocks > 65535u * 4) blocks = 65535u * 4;
  hipLaunchKernelGGL(k_linear_steps_c, dim3(blocks), dim3(256), 0, st, U, E, coef_bstride, modes, C, total, nsteps,
                     rec_slot, traj, T);
  return hipGetLastError();
}

hipError_t launch_record(const float2* U, float2* traj, const int* rec_slot, int step, int B, size_t per_sample,
                         int T, hipStream_t st) {
  size_t total = (size_t)B * per_sample;
  unsigned blocks = (unsigned)((total + 255) / 256);
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL(k_record, dim3(blocks), dim3(256), 0, st, U, traj, rec_slot, step, B, per_sample, T);
  return hipGetLastError();
}

template <int N>
static hipError_t launch_run1_t(const Run1Args& a, hipStream_t st) {
  using S = Run1Shape<N>;
  const dim3 grid((a.B + S::G - 1) / S::G), block(S::NT * S::G);
  if (a.coefc)
    hipLaunchKernelGGL((k1_run<N, true>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((k1_run<N, false>), grid, block, 0, st, a);
  return hipGetLastError();
}

template <int N>
static hipError_t launch_eval_ks_t(const Run1Args& a, const float2* S, float2* Nraw, hipStream_t st) {
  constexpr int NT = Fft<N>::NT;
  constexpr int V = NT >= 64 ? 1 : 64 / NT;
  hipLaunchKernelGGL((k1_eval_ks<N, V>), dim3((a.B + V - 1) / V), dim3(NT * V), 0, st, a, S, Nraw);
  return hipGetLastError();
}

hipError_t launch_k1_eval_ks(const Run1Args& a, const float2* S, float2* Nraw, hipStream_t st) {
  TFSM_SWITCH_N(a.N, { return launch_eval_ks_t<NN>(a, S, Nraw, st); })
}

hipError_t launch_k1_stage(const Run1Args& a, int stage, const float2* Nraw, const float2* dc, float2* S,
                           hipStream_t st) {
  const size_t total = (size_t)a.B * a.H;
  unsigned blocks = (unsigned)((total + 255) / 256);
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k1_stage, dim3(blocks), dim3(256), 0, st, a, stage, Nraw, dc, S);
  return hipGetLastError();
}

hipError_t launch_run1d(const Run1Args& a, hipStream_t st) {
  switch (a.N) {
    case 32: return launch_run1_t<32>(a, st);
    case 64: return launch_run1_t<64>(a, st);
    case 128: return launch_run1_t<128>(a, st);
    case 256: return launch_run1_t<256>(a, st);
    case 512: return launch_run1_t<512>(a, st);
    case 1024: return launch_run1_t<1024>(a, st);
    case 2048: return launch_run1_t<2048>(a, st);
    case 4096: return launch_run1_t<4096>(a, st);
    case 48: return launch_run1_t<48>(a, st);
    case 96: return launch_run1_t<96>(a, st);
    case 100: return launch_run1_t<100>(a, st);
    case 112: return launch_run1_t<112>(a, st);
    case 192: return launch_run1_t<192>(a, st);
    case 200: return launch_run1_t<200>(a, st);
    case 384: return launch_run1_t<384>(a, st);
    case 400: return launch_run1_t<400>(a, st);
    case 768: return launch_run1_t<768>(a, st);
    case 800: return launch_run1_t<800>(a, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace tfsm
